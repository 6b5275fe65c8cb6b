"""The work that is timed to judge this framework's speed, through its public entry points.

kinds of case
  step    HipVecEnv.step on the GPU: one agent step of every env (the training loop's call)
  fast    FastVecEnv.step, numpy in and out: a few steps of a handful of envs (evaluation, a quick look, SB3)
  raw     HipRawNES / RawNES: one or more raw frames with their picture and RAM
  add     FrameReplay.add: one transition of every env into the ring
  sample  FrameReplay.sample: an n-step batch out of the ring
  policy  the rollout's Nature CNN forward (logits and values) of an observation batch
  gae     generalized advantage estimation over a rollout

The envs of a `step`, `fast` or `raw` case are carried past their start before the first pass, so that deaths,
resets and level loads are among what is timed, as in any run longer than a few seconds. The ROM is the synthetic
NROM program of tests/golden/roms.
"""
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "fast-mario-env_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "fast-mario-env_amd"))

from fast_mario_env_amd import ALL_LEVELS, FastVecEnv, HipRawNES, HipVecEnv, RawNES  # noqa: E402
from fast_mario_env_amd.replay import FrameReplay  # noqa: E402
from fast_mario_env_amd.rollout import gae, make_net  # noqa: E402

DEV = "cuda:0"
MODES = ("vanilla", "downsample", "pixel", "rectangle")
BUTTONS = (0x00, 0x80, 0x81, 0x82, 0x83, 0x01, 0x40)   # SIMPLE_MOVEMENT
FRAME = 84 * 84
ROWS = 64      # rows of actions or buttons made beforehand; a longer run goes round


def listed():
    return [
        # a person or an evaluation script with the class's default of 8 envs, over numpy
        dict(name="fast_8", kind="fast", n=8, steps=8, preroll=90),
        # the reference's own throughput sweep goes from 256 envs over all levels to 65,536; without max-pooling,
        # which its GPU class does not have
        dict(name="step_256_mixed", kind="step", n=256, levels="mixed", modes=1, maxpool=False, preroll=90),
        # an ordinary training batch over all levels, with the whole wrapper stack
        dict(name="step_4096_mixed", kind="step", n=4096, levels="mixed", modes=1, maxpool=True, preroll=90),
        # the headline benchmark's configuration
        dict(name="step_32768", kind="step", n=32768, levels="1-1", modes=1, maxpool=True, preroll=120),
        # the divergence-stress benchmark's configuration: every level, four ROM variants, biased actions
        dict(name="step_65536_stress", kind="step", n=65536, levels="mixed", modes=4, maxpool=False, preroll=40),
        # one console, picture and RAM to the host every frame: a viewer, a search, a recording
        dict(name="raw_1", kind="raw", n=1, frames=16, preroll=150),
        # the raw-emulator benchmark's configuration: RGB24 and RAM of every frame on the GPU
        dict(name="raw_4096", kind="raw", n=4096, frames=1, preroll=200),
        # the replay benchmark's two calls (the ring of the add is shorter: its depth costs nothing)
        dict(name="replay_add_32768", kind="add", n=32768, capacity=16, k=4),
        dict(name="replay_sample_4096", kind="sample", n=32768, capacity=64, k=4, batch=4096, n_step=3),
        # the rollout's policy: at the headline's batch, and at that of a small run or of bootstrapped final frames
        dict(name="policy_32768", kind="policy", n=32768),
        dict(name="policy_300", kind="policy", n=300),
        # the end of a PPO rollout of the headline envs
        dict(name="gae_128x32768", kind="gae", n=32768, steps=128),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(("step", "step", "step", "fast", "raw", "add", "sample", "policy", "policy", "gae"))
    if kind == "step":
        n = _log_int(rng, 1, 49152)
        return dict(kind=kind, n=n, levels=rng.choice(("mixed", "1-1", "4-2")), modes=rng.choice((1, 4)),
                    maxpool=rng.random() < 0.5, preroll=rng.randint(40, 100))
    if kind == "fast":
        return dict(kind=kind, n=_log_int(rng, 1, 128), steps=rng.randint(2, 8), preroll=rng.randint(40, 90))
    if kind == "raw":
        n = _log_int(rng, 1, 4096)
        return dict(kind=kind, n=n, frames=rng.randint(4, 16) if n == 1 else 1, preroll=rng.randint(100, 200))
    if kind == "add":
        return dict(kind=kind, n=_log_int(rng, 64, 32768), capacity=rng.randint(8, 16), k=rng.choice((1, 2, 4, 4)))
    if kind == "sample":
        return dict(kind=kind, n=_log_int(rng, 64, 32768), capacity=rng.randint(24, 64), k=rng.choice((1, 2, 4, 4)),
                    batch=_log_int(rng, 32, 4096), n_step=rng.randint(1, 5))
    if kind == "policy":
        return dict(kind=kind, n=_log_int(rng, 1, 32768))
    return dict(kind=kind, n=_log_int(rng, 64, 32768), steps=rng.randint(16, 128))


# ---------------------------------------------------------------- what a program has in hand before the call
def _rom(mode="vanilla"):
    with open(os.path.join(ROOT, "tests", "golden", "roms", f"mini_smb_{mode}.nes"), "rb") as f:
        return f.read()


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _levels(case, n):
    if case["levels"] != "mixed":
        return case["levels"]
    return [ALL_LEVELS[k] for k in np.random.default_rng(7).integers(0, len(ALL_LEVELS), n)]


def _actions(n, seed, biased):
    """(ROWS, n) actions; biased: right + jump half of the time, as the stress benchmark draws them."""
    g = _gen(seed)
    a = torch.randint(0, 7, (ROWS, n), generator=g, device=DEV)
    if biased:
        a = torch.where(torch.rand(ROWS, n, generator=g, device=DEV) < 0.5, torch.full_like(a, 2), a)
    return a


def _observations(n, seed, k=4):
    """(n, k, 84, 84) pictures of flat areas with edges and some noise, as the games' gray frames are."""
    g = _gen(seed)
    x = torch.randint(0, 256, (n, k, 21, 21), generator=g, device=DEV, dtype=torch.uint8)
    x = x.repeat_interleave(4, 2).repeat_interleave(4, 3)
    return x ^ torch.randint(0, 4, (n, k, 84, 84), generator=g, device=DEV, dtype=torch.uint8)


def _transitions(case, seed):
    """A few transitions of every env; the replay cases go round them."""
    n, g = case["n"], _gen(seed)
    out = []
    for j in range(3):
        done = torch.rand(n, generator=g, device=DEV) < 0.012
        out.append(dict(obs=_observations(n, seed * 8 + 2 * j, case["k"]),
                        next_obs=_observations(n, seed * 8 + 2 * j + 1, case["k"]),
                        action=torch.randint(0, 7, (n,), generator=g, device=DEV),
                        reward=torch.randint(-15, 16, (n,), generator=g, device=DEV).float(),
                        done=done, truncated=done & (torch.rand(n, generator=g, device=DEV) < 0.2)))
    return out


def _rollout(case, seed):
    T, n, g = case["steps"], case["n"], _gen(seed)
    return dict(rew=torch.randint(-15, 16, (T, n), generator=g, device=DEV).float(),
                val=torch.randn(T, n, generator=g, device=DEV) * 10,
                start=torch.rand(T, n, generator=g, device=DEV) < 0.012,
                next_val=torch.randn(n, generator=g, device=DEV) * 10,
                next_start=torch.rand(n, generator=g, device=DEV) < 0.012)


def _net(seed):
    net = make_net(seed=seed, device=DEV)
    g = _gen(seed)
    with torch.no_grad():   # the biases of a network that has been trained are not zero
        for m in list(net.convs) + [net.fc, net.pi, net.vf]:
            m.bias.copy_(torch.randn(m.bias.shape, generator=g, device=DEV) * 0.05)
    return net


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "step":
        roms = {m: _rom(m) for m in MODES[:case["modes"]]}
        env = HipVecEnv(_levels(case, n), n, seed=seed, sticky=0.25, noop_max=30, max_steps=2000, skip=4,
                        frame_stack=4, maxpool=case["maxpool"], rom=roms,
                        rom_mode=[MODES[i % case["modes"]] for i in range(n)], device=DEV)
        acts = _actions(n, seed, case["levels"] == "mixed")
        env.reset()
        for i in range(case["preroll"]):
            env.step(acts[i % ROWS])
        return dict(kind=kind, env=env, acts=acts, at=case["preroll"])
    if kind == "fast":
        env = FastVecEnv("1-1", n, seed=seed, sticky=0.25, noop_max=30, maxpool=True, rom=_rom(), device=DEV)
        acts = np.random.default_rng(seed).integers(0, 7, (ROWS, n))
        env.reset()
        for i in range(case["preroll"]):
            env.step(acts[i % ROWS])
        return dict(kind=kind, env=env, acts=acts, steps=case["steps"], at=case["preroll"])
    if kind == "raw":
        table = np.array(BUTTONS, np.uint8)
        acts = table[np.random.default_rng(seed).integers(0, 7, (ROWS, n))]
        if n == 1:
            con, buttons = RawNES(_rom(), device=DEV), acts[:, 0].tolist()
        else:
            con, buttons = HipRawNES(_rom(), n, device=DEV), torch.from_numpy(acts).to(DEV)
        for f in range(40):                       # start / nothing in turn: from the title into the first level
            con.frame(8 if f % 2 == 0 else 0)
        for f in range(case["preroll"]):
            con.frame(buttons[f % ROWS])
        return dict(kind=kind, con=con, buttons=buttons, n=n, frames=case["frames"], at=case["preroll"])
    if kind in ("add", "sample"):
        rb = FrameReplay(case["capacity"], n, case["k"], device=DEV, seed=seed)
        trans = _transitions(case, seed)
        for i in range(case["capacity"] + 5):     # once round the ring
            rb.add(**trans[i % 3])
        return dict(kind=kind, rb=rb, trans=trans, at=case["capacity"] + 5, **{k: case.get(k) for k in ("batch", "n_step")})
    if kind == "policy":
        return dict(kind=kind, net=_net(seed), obs=_observations(n, seed))
    return dict(kind=kind, **_rollout(case, seed))


# ---------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "step":
        env = s["env"]
        env.step(s["acts"][s["at"] % ROWS])
        s["at"] += 1
        return dict(obs=env.obs, rew=env.rew, term=env.term, trunc=env.trunc, info=env.info_t,
                    final_obs=env.final_obs, ep_ret=env.ep_ret, ep_len=env.ep_len)
    if kind == "fast":
        out = []
        for _ in range(s["steps"]):
            out.append(s["env"].step(s["acts"][s["at"] % ROWS])[:4])
            s["at"] += 1
        return out
    if kind == "raw":
        con, out = s["con"], []
        for _ in range(s["frames"]):
            con.frame(s["buttons"][s["at"] % ROWS])
            s["at"] += 1
            out.append((con.screen if s["n"] == 1 else con.screen_rgb, con.ram))
        return out
    if kind == "add":
        rb = s["rb"]
        rb.add(**s["trans"][s["at"] % 3])
        s["at"] += 1
        return dict(frames=rb.frames, age=rb.age, act=rb.act, rew=rb.rew, flags=rb.flags)
    if kind == "sample":
        return s["rb"].sample(s["batch"], s["n_step"], 0.99)
    if kind == "policy":
        with torch.no_grad():
            return s["net"](s["obs"])
    return gae(s["rew"], s["val"], s["start"], s["next_val"], s["next_start"], 0.99, 0.95)


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind, n = case["kind"], case["n"]
    if kind in ("step", "fast"):
        # per env: console state and env words in and out, action, reward / term / trunc / info, three frames of the
        # stack read and four written; the area filter's multiplies and adds
        times = case.get("steps", 1)
        return dict(bytes=times * n * (2 * 4548 + 2 * 144 + 8 + 46 + 7 * FRAME), flops=times * n * 2 * 106848)
    if kind == "raw":
        pixels = 256 * 240 * (1 if n == 1 else 3)
        return dict(bytes=case["frames"] * n * (2 * 4548 + pixels + 2048 + 1), flops=0)
    if kind == "add":
        return dict(bytes=n * (2 * FRAME + 40), flops=0)
    if kind == "sample":
        return dict(bytes=case["batch"] * (2 * case["k"] * 2 * FRAME + case["n_step"] * 6 + 60), flops=0)
    if kind == "policy":
        macs = 400 * 32 * 256 + 81 * 64 * 512 + 49 * 64 * 576 + 3136 * 512 + 512 * 8
        weights = 4 * (32 * 256 + 64 * 512 + 64 * 576 + 3136 * 512 + 512 * 8)
        return dict(bytes=n * (4 * FRAME + 4 * 8) + weights, flops=2 * n * macs)
    return dict(bytes=case["steps"] * n * (4 + 4 + 1 + 4 + 4) + 5 * n, flops=case["steps"] * n * 9)


def tolerance(case):
    # pictures, RAM, counters, copies and sums of a stated order are the same, bit for bit
    if case["kind"] == "policy":
        return dict(rel=0.02)      # bf16 weights and activations through four layers
    if case["kind"] == "gae":
        return dict(rel=1e-6)      # float32 recurrence
    return "exact"


# ---------------------------------------------------------------- the same in 64 bits, without the framework
def exact(case, seed):
    if case["kind"] == "policy":
        net, obs = _net(seed), _observations(case["n"], seed)
        F, d = torch.nn.functional, {k: v.detach().double() for k, v in net.state_dict().items()}
        logits, value = [], []
        for x in obs.split(1024):
            x = x.double() / 255.0
            for i, stride in enumerate((4, 2, 1)):
                x = F.relu(F.conv2d(x, d[f"convs.{i}.weight"], d[f"convs.{i}.bias"], stride))
            h = F.relu(F.linear(x.flatten(1), d["fc.weight"], d["fc.bias"]))
            logits.append(F.linear(h, d["pi.weight"], d["pi.bias"]))
            value.append(F.linear(h, d["vf.weight"], d["vf.bias"]).squeeze(-1))
        return torch.cat(logits), torch.cat(value)
    if case["kind"] == "gae":
        r = _rollout(case, seed)
        rew, val = r["rew"].double(), r["val"].double()
        adv, last = torch.zeros_like(rew), torch.zeros(case["n"], dtype=torch.float64, device=DEV)
        after, cut = r["next_val"].double(), r["next_start"]
        for t in reversed(range(case["steps"])):
            keep = 1.0 - cut.double()
            last = rew[t] + 0.99 * after * keep - val[t] + 0.99 * 0.95 * keep * last
            adv[t] = last
            after, cut = val[t], r["start"][t]
        return adv, adv + val
    return None   # emulated consoles, copies of frames: no computed floats but sums of whole rewards
