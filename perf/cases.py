"""Performance cases: the simulation work a program has this backend do, through
the package's public interface (Network, Configuration, Simulation, run_batch).

A case is a dict of plain values:

  kind      "step" (one nemo_step call), "run" (a multi-cycle run and its
            raster), "stdp" (runs with applyStdp between them), "kuramoto"
            (a run of phase oscillators and their phases), "batch" (many
            networks in one batched run)
  model     "iz" (the 80/20 Izhikevich network of the benchmark) or "if"
            (IF_curr_exp_noise, which fires at 333 Hz under this drive)
  n, m      neurons and synapses per neuron; targets are uniform
  dmax      delays are uniform in 1..dmax
  cycles    1 ms cycles per run
  stim      neurons forced to fire, and as many given a current, in every
            cycle of a run (or in each step)
  epochs    runs per pass, each followed by applyStdp ("stdp")
  nets      networks of a batch, sizes log-uniform in n_lo..n

Networks are synthetic: drawn from the seed on the device and handed to the
backend as host arrays, as a program that builds or loads a network would.
"""
import math

import numpy as np
import torch

import nemosim_amd
from nemosim_amd import examples

TWO_PI = 6.283185307179586


def listed():
    return [
        # closed-loop use, a robot or an experiment in real time: one call per
        # cycle with fresh stimulus, its spikes read back. The smallest network
        # of the benchmark, and a mid-size one.
        {"name": "step_1k", "kind": "step", "model": "iz", "n": 1000, "m": 100, "dmax": 20, "stim": 8},
        {"name": "step_100k", "kind": "step", "model": "iz", "n": 100000, "m": 300, "dmax": 20, "stim": 32},
        # one simulated second of a small network, with a stimulus schedule
        {"name": "run_1k", "kind": "run", "model": "iz", "n": 1000, "m": 100, "dmax": 20, "cycles": 1000, "stim": 4},
        # a ragged mid-size network: odd sizes, delays up to 33
        {"name": "run_10k", "kind": "run", "model": "iz", "n": 10007, "m": 313, "dmax": 33, "cycles": 500, "stim": 0},
        # the headline: 200k x 1000, one simulated second per launch
        {"name": "run_200k", "kind": "run", "model": "iz", "n": 200000, "m": 1000, "dmax": 20, "cycles": 1000, "stim": 0},
        # short launches between which a program looks at the spikes
        {"name": "short_100k", "kind": "run", "model": "iz", "n": 100000, "m": 100, "dmax": 20, "cycles": 20, "stim": 0},
        # plasticity: the STDP benchmark, one second and a reward
        {"name": "stdp_50k", "kind": "stdp", "model": "iz", "n": 50000, "m": 1000, "dmax": 20, "cycles": 1000, "epochs": 1},
        # reinforcement learning: rewards every 100 ms on a small network
        {"name": "stdp_3k", "kind": "stdp", "model": "iz", "n": 3001, "m": 300, "dmax": 20, "cycles": 100, "epochs": 5},
        # a densely firing network, as in the serving mix
        {"name": "if_12k", "kind": "run", "model": "if", "n": 12000, "m": 550, "dmax": 20, "cycles": 200, "stim": 0},
        # more neurons than the persistent kernel holds
        {"name": "large_300k", "kind": "run", "model": "iz", "n": 300000, "m": 100, "dmax": 20, "cycles": 200, "stim": 0},
        # densely coupled oscillators: every phase is read after the run
        {"name": "kuramoto_1k", "kind": "kuramoto", "n": 1000, "m": 1000, "dmax": 31, "cycles": 1000},
        # many independent networks at once: parameter sweeps, serving
        {"name": "batch_48", "kind": "batch", "model": "iz", "n": 20000, "n_lo": 1000, "m": 100, "dmax": 20,
         "cycles": 200, "nets": 48},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "run", "run", "run", "stdp", "kuramoto", "batch"])
    if kind == "kuramoto":
        n = _log(rng, 300, 4000)
        return {"kind": kind, "n": n, "m": max(1, min(_log(rng, 20, 1000), n)), "dmax": rng.randint(1, 31),
                "cycles": _log(rng, 200, 1000)}
    model = "iz" if kind == "step" else rng.choice(["iz", "iz", "iz", "if"])
    if kind == "batch":
        lo = _log(rng, 500, 2000)
        return {"kind": kind, "model": model, "n": _log(rng, 2 * lo, 12000), "n_lo": lo, "m": _log(rng, 50, 200),
                "dmax": rng.randint(5, 30), "cycles": _log(rng, 50, 300), "nets": rng.randint(4, 40)}
    # up to 2e7 synapses (4e6 where every neuron fires every third cycle)
    cap = 4000000 if model == "if" else 20000000
    n = _log(rng, 500, 50000 if (model == "if" or kind == "stdp") else 300000)
    m = max(20, min(_log(rng, 50, 1000), cap // n))
    case = {"kind": kind, "model": model, "n": n, "m": m, "dmax": rng.randint(2, 40)}
    if kind == "step":
        case["stim"] = rng.randint(0, 40)
    elif kind == "run":
        case["cycles"] = _log(rng, 10, 1000 if model == "iz" else 200)
        case["stim"] = rng.choice([0, 0, 1, 16])
    else:
        case["cycles"] = _log(rng, 50, 500 if model == "iz" else 100)
        case["epochs"] = rng.randint(1, 4)
    return case


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _neurons(net, model, n, rng):
    """The neuron populations of the benchmark: 80 % excitatory, 20 % inhibitory."""
    exc = np.arange(n) < (n * 4) // 5
    r = rng.random(n, dtype=np.float32)
    if model == "if":
        args = np.tile(np.array([-65.0, -65.0, 1.0, 20.0, 2.0, 5.0, 5.0, -50.0, 0.0, 3.0,
                                 -65.0, 0.0, 0.0, 1000.0], np.float32), (n, 1))
        args[:, 9] += r                     # the noise amplitude
        kind = net.add_neuron_type(examples.IF_CURR_EXP_NOISE)
    else:
        one = np.ones(n, np.float32)
        b = np.where(exc, 0.2 * one, 0.25 - 0.05 * r).astype(np.float32)
        args = np.stack([np.where(exc, 0.02 * one, 0.02 + 0.08 * r), b, np.where(exc, -65.0 + 15.0 * r * r, -65.0 * one),
                         np.where(exc, 8.0 - 6.0 * r * r, 2.0 * one), np.where(exc, 5.0 * one, 2.0 * one),
                         b * np.float32(-65.0), -65.0 * one], axis=1).astype(np.float32)
        kind = net.add_neuron_type(examples.IZHIKEVICH)
    net.add_neurons(kind, np.arange(n, dtype=np.uint32), args)


def _synapses(n, m, dmax, gen):
    """targets, delays, uniform [0,1) weights as host arrays, in source order"""
    dev = _device()
    t = torch.randint(0, n, (n * m,), generator=gen, device=dev, dtype=torch.int32)
    d = torch.randint(1, dmax + 1, (n * m,), generator=gen, device=dev, dtype=torch.uint8)
    u = torch.rand(n * m, generator=gen, device=dev)
    return t.cpu().numpy().view(np.uint32), d.cpu().numpy(), u


def _network(case, n, seed, plastic=False):
    gen = torch.Generator(device=_device())
    gen.manual_seed(seed)
    m = case["m"]
    t, d, u = _synapses(n, m, case["dmax"], gen)
    ne = ((n * 4) // 5) * m                # excitatory synapses come first
    u[:ne] *= 0.5
    u[ne:] *= -1.0
    pl = None
    if plastic:
        pl = np.zeros(n * m, np.uint8)
        pl[:ne] = 1
    net = nemosim_amd.Network()
    _neurons(net, case["model"], n, np.random.default_rng(seed))
    net.add_synapses_csr(np.arange(n + 1, dtype=np.uint64) * m, t, d, u.cpu().numpy(), pl)
    return net


def _simulation(net, stdp=False, queries=False):
    conf = nemosim_amd.Configuration()
    conf.set_cuda_backend(0)
    if not queries:
        conf.set_write_only_synapses()
    if stdp:
        pre, post = examples.stdp_window()
        conf.set_stdp_function(pre, post, min_e=0.0, max_e=1.0, min_i=0.0, max_i=-1.0)
    return nemosim_amd.Simulation(net, conf)


def _couplings(case, seed):
    gen = torch.Generator(device=_device())
    gen.manual_seed(seed)
    n, m = case["n"], case["m"]
    t, d, u = _synapses(n, m, case["dmax"], gen)
    w = (u * (0.5 / m)).cpu().numpy()      # enough to pull most of them together
    rng = np.random.default_rng(seed)
    args = np.stack([rng.uniform(0.0, 0.2, n), rng.uniform(0.0, TWO_PI, n)], axis=1).astype(np.float32)
    return t, d, w, args


def prepare(case, seed):
    kind = case["kind"]
    if kind == "kuramoto":
        t, d, w, args = _couplings(case, seed)
        n = case["n"]
        net = nemosim_amd.Network()
        net.add_neurons(net.add_neuron_type("Kuramoto"), np.arange(n, dtype=np.uint32), args)
        net.add_synapses_csr(np.arange(n + 1, dtype=np.uint64) * case["m"], t, d, w)
        return {"case": case, "sim": _simulation(net)}
    if kind == "batch":
        rng = np.random.default_rng(seed)
        sizes = np.exp(rng.uniform(math.log(case["n_lo"]), math.log(case["n"]), case["nets"])).astype(int)
        sims = [_simulation(_network(case, int(k), seed * 1000 + i)) for i, k in enumerate(sizes)]
        return {"case": case, "sims": sims, "steps": [case["cycles"]] * len(sims)}
    stdp = kind == "stdp"
    sim = _simulation(_network(case, case["n"], seed, plastic=stdp), stdp=stdp, queries=stdp and case["n"] <= 5000)
    state = {"case": case, "sim": sim}
    stim, n = case.get("stim", 0), case["n"]
    if stim:
        rng = np.random.default_rng(seed + 1)
        k = case.get("cycles", 64)          # "step": the stimuli of 64 calls, used in turn
        state["f"] = [rng.integers(0, n, stim).tolist() for _ in range(k)]
        state["i"] = [list(zip(rng.integers(0, n, stim).tolist(), rng.uniform(2.0, 20.0, stim).tolist())) for _ in range(k)]
    state["at"] = 0
    return state


def _record(case, ids):
    """The spikes in the program's own record: a buffer of fixed size, their
    number first, room for one spike per neuron and 40 ms (Izhikevich) or
    2.5 ms (IF_curr_exp_noise), and for one volley of all neurons."""
    n = case["n"] * case.get("nets", 1)
    buf = np.zeros(1 + n + int(n * case.get("cycles", 1) * (0.4 if case["model"] == "if" else 0.025)), np.uint32)
    buf[0] = len(ids)
    buf[1:len(ids) + 1] = ids
    return buf


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        k = state["at"]
        state["at"] = (k + 1) % 64
        sim = state["sim"]
        fired = sim.step(state["f"][k], state["i"][k]) if "f" in state else sim.step()
        return {"fired": _record(case, fired)}
    if kind == "run":
        sim = state["sim"]
        events = sim.run(case["cycles"], state.get("f"), state.get("i"))
        counts, ids = sim.read_fired()
        return {"events": events, "counts": counts, "ids": _record(case, ids)}
    if kind == "stdp":
        # rewards of either sign, small enough that the network keeps firing;
        # the spikes of every run after the first, and of the next pass, come
        # of the changed weights
        sim, out = state["sim"], {}
        for e in range(case["epochs"]):
            out["events%d" % e] = sim.run(case["cycles"])
            out["counts%d" % e], ids = sim.read_fired()
            out["ids%d" % e] = _record(case, ids)
            sim.apply_stdp(0.05 if e % 2 == 0 else -0.05)
        if case["n"] <= 5000:
            # what a learning experiment watches: the afferents of its output
            out["weights"] = np.array([sim.get_synapse_weight(s) for s in sim.get_synapses_from(0)[:16]], np.float32)
        return out
    if kind == "kuramoto":
        sim = state["sim"]
        sim.run(case["cycles"])
        return {"phase": np.array([sim.get_neuron_state(i, 0) for i in range(case["n"])], np.float32)}
    events = nemosim_amd.run_batch(state["sims"], state["steps"])
    fired = [s.read_fired() for s in state["sims"]]
    return {"events": np.asarray(events), "counts": np.concatenate([c for c, _ in fired]),
            "ids": _record(case, np.concatenate([i for _, i in fired]))}


def exact(case, seed):
    """Phases of the oscillators in 64 bits. Spikes, their counts and the
    fixed-point weights have no such value: they are whole numbers of a chaotic
    system and have to be equal."""
    if case["kind"] != "kuramoto":
        return None
    t, d, w, args = _couplings(case, seed)
    dev = _device()
    n, m = case["n"], case["m"]
    tgt = torch.from_numpy(t.view(np.int32)).to(dev).long()
    src = torch.arange(n, device=dev).repeat_interleave(m)
    lag = torch.from_numpy(d).to(dev).long() - 1
    wt = torch.from_numpy(w).to(dev).double()
    f = torch.from_numpy(args[:, 0].copy()).to(dev).double()
    order = torch.argsort(tgt, stable=True)
    tgt, src, lag, wt = tgt[order], src[order], lag[order], wt[order]
    ptr = torch.searchsorted(tgt, torch.arange(n + 1, device=dev))
    hist = torch.zeros(32, n, dtype=torch.float64, device=dev)      # plane c % 32: the phases of cycle c
    hist[0] = torch.from_numpy(args[:, 1].copy()).to(dev).double()
    for k in range(31):                                             # uncoupled before the start
        hist[(-k - 1) % 32] = torch.remainder(hist[(-k) % 32] - f, TWO_PI)

    def rate(x, theta):
        s = torch.cumsum(wt * torch.sin(theta - x[tgt]), 0)
        s = torch.cat([torch.zeros(1, dtype=s.dtype, device=dev), s])
        return f + s[ptr[1:]] - s[ptr[:-1]]

    for c in range(case["cycles"]):
        theta = hist[(c - lag) % 32, src]
        x = hist[c % 32]
        k0 = rate(x, theta)
        k1 = rate(x + 0.5 * k0, theta)
        k2 = rate(x + 0.5 * k1, theta)
        k3 = rate(x + k2, theta)
        hist[(c + 1) % 32] = torch.remainder(x + (k0 + 2.0 * k1 + 2.0 * k2 + k3) / 6.0, TWO_PI)
    return {"phase": hist[case["cycles"] % 32].cpu().numpy()}


def work(case):
    """Bytes: per cycle the neuron parameters and state read and written once
    (Izhikevich 68, IF_curr_exp_noise 104), 8 per synapse delivered and, with
    STDP, 20 per plastic in-synapse of a neuron that fired (its source, the
    source's history, the accumulator read and written); applyStdp 20 per
    plastic synapse. The rates are the networks' own, 8 and 333 Hz."""
    kind, m = case["kind"], case["m"]
    if kind == "kuramoto":
        n, c = case["n"], case["cycles"]
        # source, delay, weight and the source's phase; a sine, a product and
        # a sum in each of the four stages (the sine counted as 20 operations)
        return {"bytes": (16.0 * n * m + 12.0 * n) * c, "flops": 4.0 * n * m * 22.0 * c}
    rate, nbytes, nflops = (0.008, 68.0, 100.0) if case["model"] == "iz" else (0.333, 104.0, 80.0)
    n, c = float(case["n"]), case.get("cycles", 1) * case.get("epochs", 1)
    if kind == "batch":
        n = case["nets"] * (case["n"] - case["n_lo"]) / math.log(case["n"] / case["n_lo"])
    events = n * rate * m
    b, f = (nbytes * n + 8.0 * events) * c, (nflops * n + events) * c
    if kind == "stdp":
        b += 0.8 * events * 20.0 * c + case["epochs"] * 0.8 * n * m * 20.0
        f += 0.8 * events * 10.0 * c
    return {"bytes": b, "flops": f}
