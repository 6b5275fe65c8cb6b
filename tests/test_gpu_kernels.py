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
    # a queue's two lists of 16 buckets are among an env's bytes (whole instances, padded to 64 envs, per env)
    own = 3 * (4384 + 160) + 144 + 2 * 61440 + 7056
    assert big.bytes_per_env() == (own + (128 if extra else 0)) * ((n + 63) // 64 * 64) // n
    assert parts[0][1].bytes_per_env() == own * 64 // m
    for e in (big, parts[0][1], parts[1][1]):
        e.close()


def _rollout(T, n, seed):
    g = torch.Generator().manual_seed(seed)
    rew, val = torch.randn(T, n, generator=g), torch.randn(T, n, generator=g) * 10
    start, cut = torch.rand(T, n, generator=g) < 0.1, torch.rand(n, generator=g) < 0.5
    val[-1, 0] = float("inf")             # a product of the recurrence, as in its row-by-row form: inf * 0 is NaN
    return rew, val, start, torch.randn(n, generator=g), cut


@pytest.mark.parametrize("T,n", [(1, 1), (15, 63), (16, 64), (17, 65), (33, 1000), (128, 257)])
def test_gae_kernel_is_the_row_by_row_form(T, n):
    """The kernel at the edges of its blocks of steps and envs, bit for bit the row-by-row form on the CPU (the same
    float32 operations in the same order); twice from a captured graph."""
    from fast_mario_env_amd.rollout import gae
    host = _rollout(T, n, T)
    dev = [x.cuda() for x in host]
    want = gae(*host)
    for a, b in zip(gae(*dev), want):
        assert torch.equal(a.cpu().nan_to_num(7e30), b.nan_to_num(7e30))
        assert torch.equal(a.cpu().isnan(), b.isnan())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = gae(*dev)
    for k in range(3):
        dev[0].add_(1.0)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, gae(*[x.cpu() for x in dev])):
            assert torch.equal(a.cpu().nan_to_num(7e30), b.nan_to_num(7e30)), k


def test_gae_calls_the_kernel_does_not_take():
    """Other strides, types, gradients, vmap and empty rollouts keep the row-by-row form and its results."""
    from fast_mario_env_amd import rollout
    host = _rollout(5, 40, 3)
    host[1][-1, 0] = 1.0
    dev = [x.cuda() for x in host]
    want = rollout.gae(*host)
    def same(got, rel=1e-6):
        for a, b in zip(got, want):
            assert torch.allclose(a.detach().cpu().float(), b, rtol=rel, atol=rel * 40)
    assert rollout._gae_kernel_takes(*dev, 0.99, 0.95)
    strided = [x.t().contiguous().t() if x.dim() == 2 else x for x in dev]
    wide = [x.double() if x.is_floating_point() else x for x in dev]
    flags = [x.float() if x.dtype == torch.bool else x for x in dev]
    for other in (strided, wide, flags):
        assert not rollout._gae_kernel_takes(*other, 0.99, 0.95)
        same(rollout.gae(*other))
    g = [x.clone().requires_grad_() if x.is_floating_point() else x for x in dev]
    out = rollout.gae(*g)
    same(out)
    out[0].sum().backward()
    assert g[0].grad is not None and g[3].grad is not None
    adv, ret = torch.vmap(rollout.gae, in_dims=(0, None, None, None, None), out_dims=0)(torch.stack([dev[0]] * 2), *dev[1:])
    same((adv[1], ret[1]))
    e = rollout.gae(*[x[:0] if x.dim() == 2 else x for x in dev])
    assert e[0].shape == (0, 40)


@pytest.mark.parametrize("extra", [-1, 0, 1, 3])
@pytest.mark.parametrize("layer", [1, 2, 3])
def test_policy_conv_batch_edges(layer, extra):
    """Each layer around the batch where a block starts taking several images (two or five per CU), and past what the
    blocks take in one turn: an image's activations are the bits that it has in a batch of its own (the same sums in the
    same order), also into an output that is aligned to 2 bytes only."""
    from fast_mario_env_amd._native import check, lib
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = {1: 2, 2: 2, 3: 5}[layer] * cus + extra
    ci, hi, co, ho, k = {1: (4, 84, 32, 20, 8), 2: (32, 20, 64, 9, 4), 3: (64, 9, 64, 7, 3)}[layer]
    g = torch.Generator(device="cuda").manual_seed(layer)
    w = (torch.randn(co, k * k * ci, generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    b = torch.randn(co, generator=g, device="cuda").to(torch.bfloat16)
    if layer == 1:
        x = torch.randint(0, 256, (n, ci, hi, hi), dtype=torch.uint8, device="cuda", generator=g)
    else:
        x = torch.randn(n, hi, hi, ci, generator=g, device="cuda").to(torch.bfloat16)

    def conv(x, out):
        args = (x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), x.shape[0])
        check(lib().mh_policy_conv1(*args, 0) if layer == 1 else lib().mh_policy_conv(*args, layer, 0), "conv")
        torch.cuda.synchronize()
        return out

    size = ho * ho * co
    y = conv(x, torch.zeros(n, size, dtype=torch.bfloat16, device="cuda"))
    for i in (0, 1, n // 2, n - 2, n - 1):
        one = conv(x[i:i + 1].clone(), torch.zeros(size, dtype=torch.bfloat16, device="cuda"))
        assert torch.equal(one, y[i]), i
    odd = torch.zeros(n * size + 2, dtype=torch.bfloat16, device="cuda")
    assert torch.equal(conv(x, odd[1:-1]).view(n, size), y) and odd[0] == 0 and odd[-1] == 0


@pytest.mark.parametrize("turns,extra", [(0, 1), (0, 2), (1, -1), (1, 0), (1, 1), (2, 1), (3, 0)])
def test_policy_first_two_layers_in_one_pass(turns, extra):
    """Around whole turns of one image per CU: the bits of the two layers' own kernels, and nothing past the output."""
    from fast_mario_env_amd._native import check, lib
    n = turns * torch.cuda.get_device_properties(0).multi_processor_count + extra
    g = torch.Generator(device="cuda").manual_seed(n)
    w1, w2 = ((torch.randn(s, generator=g, device="cuda") * 0.05).to(torch.bfloat16) for s in ((32, 256), (64, 512)))
    b1, b2 = (torch.randn(s, generator=g, device="cuda").to(torch.bfloat16) for s in (32, 64))
    x = torch.randint(0, 256, (n, 4, 84, 84), dtype=torch.uint8, device="cuda", generator=g)
    y1 = torch.empty(n, 20, 20, 32, dtype=torch.bfloat16, device="cuda")
    want = torch.empty(n * 5184, dtype=torch.bfloat16, device="cuda")
    got = torch.zeros(n * 5184 + 4, dtype=torch.bfloat16, device="cuda")
    check(lib().mh_policy_conv1(x.data_ptr(), w1.data_ptr(), b1.data_ptr(), y1.data_ptr(), n, 0), "conv1")
    check(lib().mh_policy_conv(y1.data_ptr(), w2.data_ptr(), b2.data_ptr(), want.data_ptr(), n, 2, 0), "conv")
    check(lib().mh_policy_conv12(x.data_ptr(), w1.data_ptr(), b1.data_ptr(), w2.data_ptr(), b2.data_ptr(), got.data_ptr(), n, 0),
          "conv12")
    assert torch.equal(got[:-4], want) and not got[-4:].any()


@pytest.mark.parametrize("channels_last", [False, True])
def test_policy_pack_is_the_cast_and_permuted_parameters(channels_last):
    from fast_mario_env_amd.rollout import _packed_params, make_net
    net = make_net(seed=3)
    for p in net.parameters():
        p.data += 0.01 * torch.randn_like(p)
    net = net.to(memory_format=torch.channels_last if channels_last else torch.contiguous_format)
    obs = torch.zeros(2, 4, 84, 84, dtype=torch.uint8, device="cuda")
    got = _packed_params(list(net.convs), net.fc, obs)
    parts = [net.convs[0].weight] + [c.weight.permute(0, 2, 3, 1) for c in net.convs[1:]] + [c.bias for c in net.convs]
    parts += [net.fc.bias, net.fc.weight.view(512, 64, 49).permute(0, 2, 1)]
    assert torch.equal(got, torch.cat([p.detach().reshape(-1) for p in parts]).to(torch.bfloat16))
    assert _packed_params(list(net.convs), net.fc.double(), obs) is None


@pytest.mark.parametrize("n,actions", [(1, 7), (3, 1), (300, 7), (8197, 7), (5, 8), (6, 12), (4, 15), (4, 16)])
def test_policy_heads_against_64_bits(n, actions):
    """512 products summed in float32: the error is below 512 units in the last place of the sum of their sizes, and not
    above that of torch's float32 layers."""
    from fast_mario_env_amd.rollout import _packed_heads, _plain_heads
    torch.manual_seed(n + actions)
    pi, vf = torch.nn.Linear(512, actions).cuda(), torch.nn.Linear(512, 1).cuda()
    h = torch.randn(n, 512, device="cuda").to(torch.bfloat16)
    assert _plain_heads(pi, vf, h)
    with torch.no_grad():
        x = h.float().relu()
        for got, m, plain in zip(_packed_heads(pi, vf, h), (pi, vf), (pi(x), vf(x).squeeze(-1))):
            want = (x.double() @ m.weight.double().T + m.bias.double()).reshape(got.shape)
            size = (x.double() @ m.weight.double().abs().T + m.bias.double().abs()).reshape(got.shape)
            assert ((got.double() - want).abs() <= 512 * 2.0 ** -24 * size).all()
            assert (got.double() - want).abs().max() <= 2 * (plain.double() - want).abs().max() + 2.0 ** -24 * size.max()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not _plain_heads(pi, vf, h)
    pi.register_forward_hook(lambda *a: None)
    assert not _plain_heads(pi, vf, h)


def test_policy_transforms_take_the_layers():
    """What follows the tensor operations (tangents, vmap over head weights, dispatch and function modes) sees them without
    autograd too."""
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    from fast_mario_env_amd.rollout import gae, make_net
    net = make_net(seed=4)
    called = []

    class Names(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            called.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    obs = torch.randint(0, 256, (3, 4, 84, 84), dtype=torch.uint8, device="cuda")
    w, b = net.pi.weight.detach().clone(), net.pi.bias.detach()
    def logits(weight):
        return torch.func.functional_call(net, {"pi.weight": weight}, (obs,))[0]
    with torch.no_grad():
        want = logits(w)
        both = torch.vmap(logits)(torch.stack([w, 2 * w]))
        # float32 sums of 512 products in another order
        assert torch.allclose(both[0], want, rtol=1e-4, atol=1e-5)
        assert torch.allclose(both[1] - b, 2 * (want - b), rtol=1e-4, atol=1e-5)
        with forward_ad.dual_level():
            out = logits(forward_ad.make_dual(w, torch.ones_like(w)))
            assert forward_ad.unpack_dual(out).tangent is not None
        with FlopCounterMode(display=False) as count:
            net(obs)
        with Names():
            net(obs)
            gae(*[x.cuda() for x in _rollout(3, 5, 1)])
    assert count.get_total_flops() >= 2 * 3 * 512 * (3136 + 8)
    assert called.count("linear") == 3 and "zeros_like" in called


def _draw_by_tensor_operations(rb, batch, n_step):
    C, d = rb.C, rb.dev
    lo = torch.clamp(rb._ptr - C + rb.k - 1, min=0)
    hi = rb._ptr - 1 - n_step
    cand = torch.nonzero(hi >= lo).flatten()
    env, pos = (torch.empty(batch, dtype=torch.long, device=d) for _ in range(2))
    rows = torch.arange(batch, device=d)
    while True:
        ee = cand[torch.randint(len(cand), (len(rows),), device=d, generator=rb.g)]
        width = (hi[ee] - lo[ee] + 1).double()
        pp = lo[ee] + (torch.rand(len(rows), device=d, generator=rb.g, dtype=torch.float64) * width).long()
        ok = (rb.flags[ee, pp % C] & 1).bool()
        env[rows[ok]], pos[rows[ok]] = ee[ok], pp[ok]
        rows = rows[~ok]
        if len(rows) == 0:
            return env, pos


@pytest.mark.parametrize("n_envs,batch,n_step", [(1, 1, 1), (70, 1023, 3), (1025, 1025, 1), (2600, 70001, 2), (5, 0, 1)])
def test_replay_draw_is_the_tensor_operations(n_envs, batch, n_step):
    """The same (env, pos) from the same generator as drawing with tensor operations, over rings at every stage of
    filling (some envs without a window), about a third of the slots no start, several rounds."""
    from fast_mario_env_amd.replay import FrameReplay
    rb = FrameReplay(9, n_envs, 4, hw=(4, 4), seed=7)
    g = torch.Generator(device="cuda").manual_seed(n_envs)
    rb._ptr.copy_(torch.randint(0, 40, (n_envs,), device="cuda", generator=g))
    rb._ptr[-1] = 30
    rb.flags.copy_(torch.randint(0, 3, (n_envs, 9), device="cuda", generator=g) > 0)
    rb.flags[-1] = 1
    state = rb.g.get_state()
    env, pos = rb.draw(batch, n_step)
    after = rb.g.get_state()
    rb.g.set_state(state)
    e2, p2 = _draw_by_tensor_operations(rb, batch, n_step)
    assert torch.equal(env, e2) and torch.equal(pos, p2) and torch.equal(after, rb.g.get_state())
    assert batch == 0 or bool((rb.flags[env, pos % 9] == 1).all())
    rb._ptr.zero_()
    with pytest.raises(ValueError):
        rb.draw(4, n_step)


@pytest.mark.parametrize("n", [1, 3, 65])
def test_console_outputs_at_any_alignment(n):
    """RAM, machine state and RGB of consoles in slots other than their env's, into outputs of every alignment: what the
    console's own dump and its palette screen hold, and nothing past the output."""
    from fast_mario_env_amd import HipRawNES, HipVecEnv, palette_rgb
    from fast_mario_env_amd._native import check, lib
    names = ["4-1", "1-1", "8-4"] * (n // 3) + ["1-1"] * (n % 3)
    env, raw = HipVecEnv(names, n, seed=1, rom=ROM, device="cuda:0", **WRAP), HipRawNES(ROM, n, device="cuda:0")
    env.reset()
    for t in range(3):
        env.step(torch.arange(n, device="cuda:0") % 7)
    for f in range(45):
        raw.frame(torch.tensor([(8 if f % 2 == 0 else i) & 255 for i in range(n)], dtype=torch.uint8, device="cuda:0"))
    pal = torch.from_numpy(palette_rgb().reshape(-1).copy()).to("cuda:0")
    rgb = torch.from_numpy(palette_rgb()).to("cuda:0")[(raw.screen & 63).long()]

    def out(call, size, offset):
        buf = torch.full((size + 32,), 0xa5, dtype=torch.uint8, device="cuda:0")
        check(call(buf.data_ptr() + offset), "out")
        torch.cuda.synchronize()
        assert bool((buf[:offset] == 0xa5).all()) and bool((buf[offset + size:] == 0xa5).all())
        return buf[offset:offset + size]

    for off in (0, 1, 4, 8):
        for con, ram, canon in ((env, lib().mh_env_ram, lib().mh_env_canon), (raw, lib().mh_raw_ram, lib().mh_raw_canon)):
            state = out(lambda p: canon(con.h, p, 0), n * 4464, off).view(n, 4464)
            assert torch.equal(out(lambda p: ram(con.h, p, 0), n * 2048, off).view(n, 2048), state[:, 2416:])
        got = out(lambda p: lib().mh_raw_screen_rgb(raw.h, pal.data_ptr(), p, 0), n * 61440 * 3, off)
        assert torch.equal(got, rgb.reshape(-1))
    env.close()
