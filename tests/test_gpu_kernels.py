"""The edges of the kernels' launch rules and code paths, against the CPU oracle or a plain form of the same operation."""
import numpy as np
import pytest
import torch

from build_roms import rom_path

pytestmark = pytest.mark.gpu

ROM = open(rom_path("vanilla"), "rb").read()
WRAP = dict(sticky=0.25, noop_max=30, skip=4, maxpool=True, frame_stack=4, max_steps=2000)


@pytest.mark.parametrize("extra", [0, 1, 17, 4097])
def test_step_queue_edges(extra):
    """k_step with exactly as many envs as the GPU holds waves at once (a wave each), one and 17 more (the waves take
    envs from the queue, which some leave empty) and a whole second turn plus one: the first and the last envs step as the
    same envs do in a batch of their own, for 6 steps, twice as many as the two lists of the queue."""
    from fast_mario_env_amd import HipVecEnv
    n, m = 16 * torch.cuda.get_device_properties(0).multi_processor_count + extra, 24
    kw = dict(seed=5, rom=ROM, device="cuda:0", **WRAP)
    big = HipVecEnv("1-1", n, **kw)
    parts = [(k, HipVecEnv("1-1", m, env_offset=k, **kw)) for k in (0, n - m)]
    o = big.reset()
    for k, p in parts:
        assert torch.equal(p.reset(), o[k:k + m])
    acts = torch.from_numpy(np.random.default_rng(8).integers(0, 7, (6, n))).to("cuda:0")
    for t in range(6):
        f0 = big.frames
        got = [x.clone() for x in big.step(acts[t])[:4]] + [big.info_t.clone()]
        assert big.frames - f0 >= 4 * n - 3 * int((got[2] | got[3]).sum()), t     # every env ran
        for k, p in parts:
            want = [x.clone() for x in p.step(acts[t, k:k + m].contiguous())[:4]] + [p.info_t]
            for a, b in zip(got, want):
                assert torch.equal(a[k:k + m], b), (t, k)
    assert torch.equal(big.canon()[n - m:], parts[1][1].canon())
    for e in (big, parts[0][1], parts[1][1]):
        e.close()
