"""Timed workloads of the connectivity update, the neuron step and the plasticity period.

Every case goes through the C ABI of include/relearn_bh.h on caller-owned buffers (page-locked host
arrays or device tensors), as a simulator that links the library does.  Five kinds of pass:

  update   one plasticity update of a network or an ensemble: vacancies handed over (from the host or
           from device memory), leaf fill and upward pass, target search, commit, and everything the
           caller needs to store the synapses: requests, accept flags, vacancies.
  period   one captured plasticity period: `steps` neuron steps over a connected network, the element
           commit with synapse deletion, the update, the append to the network graph; then the state.
  steps    `steps` calls of the neuron step with the counter-based background input; then the state.
  input    the same with the caller's background input, uploaded for every step.
  commit   the allocation-free conflict resolution on device buffers.

Networks have one neuron per 10^6 cubic micrometres (1,000 in a 1,000 um cube, 10^6 in 10,000 um,
16 x 10^6 in 25,000 um), 80/20 excitatory/inhibitory, Poisson(2) vacant axons and Poisson(1.5) vacant
dendrites of each type, theta 0.3, sigma 750 um.
"""
import ctypes as C
import math

import numpy as np
import torch

import relearn_amd
from relearn_amd import RL_PREC_FP32_MIXED, RL_PREC_FP64, BarnesHutHIP, StepParams

THETA, SIGMA, SEED = 0.3, 750.0, 7
PRECISION = {"fp64": RL_PREC_FP64, "mixed": RL_PREC_FP32_MIXED}
COMMIT_NEURONS, COMMIT_REQUESTS = 262144, 1048576   # limits of rl_bh_commit_requests_noalloc
IN_EDGES = 8                                        # synapses per neuron of a grown network


def listed():
    return [
        # a desktop-sized network, the size of the reference's CPU configuration: launches and waits count
        {"name": "update_1k", "kind": "update", "neurons": 1000, "networks": 1, "precision": "fp64",
         "vacancies": "host", "layout": "uniform"},
        # a reconstructed cortex patch (51,842 neurons, unevenly dense), driven from a host simulator
        {"name": "update_52k_clustered", "kind": "update", "neurons": 51842, "networks": 1, "precision": "mixed",
         "vacancies": "host", "layout": "clustered"},
        # one million neurons in either precision, synaptic elements kept on the device
        {"name": "update_1m", "kind": "update", "neurons": 1000000, "networks": 1, "precision": "mixed",
         "vacancies": "device", "layout": "uniform"},
        {"name": "update_1m_fp64", "kind": "update", "neurons": 1000000, "networks": 1, "precision": "fp64",
         "vacancies": "device", "layout": "uniform"},
        # the largest network that the benchmark names
        {"name": "update_16m", "kind": "update", "neurons": 16000000, "networks": 1, "precision": "mixed",
         "vacancies": "device", "layout": "uniform"},
        # a parameter sweep: 40 independent networks of 2,000 to 200,000 neurons in one context
        {"name": "update_sweep", "kind": "update", "neurons": 1700000, "networks": 40, "precision": "mixed",
         "vacancies": "device", "layout": "uniform"},
        # the simulation loop, 100 neuron steps per plasticity update, on a small network ...
        {"name": "period_1k", "kind": "period", "neurons": 1000, "networks": 1, "precision": "fp64",
         "steps": 100, "synaptic": True},
        # ... on a sweep of mid-sized networks with odd sizes ...
        {"name": "period_sweep", "kind": "period", "neurons": 300001, "networks": 9, "precision": "mixed",
         "steps": 100, "synaptic": True},
        # ... and on a large one
        {"name": "period_2m", "kind": "period", "neurons": 2000000, "networks": 1, "precision": "mixed",
         "steps": 100, "synaptic": True},
        # neuron steps called one by one between updates (a simulator with its own step loop)
        {"name": "steps_1m", "kind": "steps", "neurons": 1000000, "steps": 100},
        # the same with the simulator's own background input
        {"name": "steps_input", "kind": "input", "neurons": 100003, "steps": 10},
        # conflict resolution for a caller with its own search and device buffers
        {"name": "commit_262k", "kind": "commit", "neurons": 262144},
    ]


def _log_uniform(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))


def draw(rng):
    kind = rng.choice(["update", "update", "update", "period", "period", "steps", "input", "commit"])
    if kind == "update":
        precision = rng.choice(["fp64", "mixed"])
        n = _log_uniform(rng, 1000, 2000000 if precision == "fp64" else 8000000)
        networks = 1 if n < 20000 or rng.random() < 0.6 else rng.randint(2, min(64, n // 5000))
        return {"kind": kind, "neurons": n, "networks": networks, "precision": precision,
                "vacancies": rng.choice(["host", "device"]), "layout": rng.choice(["uniform", "clustered"])}
    if kind == "period":
        n = _log_uniform(rng, 1000, 2000000)
        networks = 1 if n < 20000 or rng.random() < 0.6 else rng.randint(2, min(64, n // 5000))
        return {"kind": kind, "neurons": n, "networks": networks, "precision": rng.choice(["fp64", "mixed"]),
                "steps": rng.choice([50, 100, 101]), "synaptic": rng.random() < 0.75}
    if kind == "steps":
        return {"kind": kind, "neurons": _log_uniform(rng, 1000, 4000000), "steps": rng.choice([50, 100])}
    if kind == "input":
        return {"kind": kind, "neurons": _log_uniform(rng, 1000, 1000000), "steps": rng.randint(5, 20)}
    return {"kind": kind, "neurons": _log_uniform(rng, 5000, COMMIT_NEURONS)}


# ------------------------------------------------------------------------------------ inputs


class State:
    pass


def _generator(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + case["neurons"])
    return g


def _sizes(case):
    """Neurons of each network: log-uniform over two decades, `neurons` in all."""
    n, k = case["neurons"], case.get("networks", 1)
    if k == 1:
        return [n]
    weights = [10.0 ** (2.0 * ((i * 0.6180339887498949) % 1.0)) for i in range(k)]
    sizes = [max(2, int(n * w / sum(weights))) for w in weights]
    sizes[-1] += n - sum(sizes)
    return sizes


def _network(case, g):
    """Positions, signal types, first neuron and box of each network (host arrays)."""
    n, sizes = case["neurons"], _sizes(case)
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    sides = [1000.0 * (k / 1000.0) ** (1.0 / 3.0) for k in sizes]
    boxes = np.array([[0.0, 0.0, 0.0, a, a, a] for a in sides])
    side = torch.repeat_interleave(torch.tensor(sides, dtype=torch.float64, device="cuda"),
                                   torch.tensor(sizes, device="cuda"))
    unit = torch.rand((n, 3), dtype=torch.float64, device="cuda", generator=g)
    if case.get("layout") == "clustered":
        # half of the neurons in 24 round clumps whose deviation is a fortieth of the side
        centre = torch.rand((24, 3), dtype=torch.float64, device="cuda", generator=g)
        of = torch.randint(0, 24, (n,), device="cuda", generator=g)
        clump = centre[of] + torch.randn((n, 3), dtype=torch.float64, device="cuda", generator=g) / 40.0
        inside = torch.rand(n, device="cuda", generator=g) < 0.5
        unit = torch.where(inside[:, None], torch.remainder(clump, 1.0), unit)
    xyz = (unit * side[:, None]).cpu().numpy()
    signal = (torch.rand(n, device="cuda", generator=g) >= 0.8).to(torch.uint8).cpu().numpy()
    return xyz, signal, offsets, boxes


def _poisson(n, mean, g):
    rate = torch.full((n,), mean, device="cuda")
    return torch.poisson(rate, generator=g).to(torch.int32)


def _slots(n):
    """Requests that a caller's buffers hold: the sum of n Poisson(2) counts stays below by 8 deviations."""
    return int(2 * n + 8 * math.sqrt(2 * n)) + 64


def _pinned(n, dtype):
    return torch.zeros(max(int(n), 1), dtype=dtype, pin_memory=True)


def _context(case, xyz, signal, offsets, boxes):
    lo, hi = boxes[:, :3].min(0), boxes[:, 3:].max(0)
    g = BarnesHutHIP(lo, hi, theta=THETA, sigma=SIGMA, seed=SEED, precision=PRECISION[case.get("precision", "fp64")])
    if len(offsets) > 2:
        g.init_networks(offsets, boxes, xyz, signal)
    else:
        g.init(xyz, signal)
    return g


def _ptr(t, kind):
    return C.cast(t.data_ptr(), C.POINTER(kind))


def _check(s, status):
    if status != 0:
        raise RuntimeError(s.lib.rl_bh_last_error(s.ctx.h).decode())


def _neuron_buffers(s, n):
    """Host arrays for rl_neurons_get."""
    s.x, s.u, s.ca = (_pinned(n, torch.float64) for _ in range(3))
    s.fired = _pinned(n, torch.uint8)
    s.delta, s.grown = (_pinned(3 * n, torch.float64) for _ in range(2))
    s.connected = _pinned(3 * n, torch.int32)


def _neuron_state(case, gen):
    """Membrane, recovery and calcium values as they are in a running simulation."""
    n = case["neurons"]
    u01 = lambda: torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)  # noqa: E731
    x, u = -70.0 + 20.0 * u01(), -15.0 + 5.0 * u01()
    ca = 0.1 + 0.034 * u01()
    # target calcium on either side of what the background input sustains, so that some neurons grow
    # elements and others lose them
    target = 0.06 + 0.12 * u01()
    return [t.cpu().numpy() for t in (x, u, ca, target)]


def _params(case, mode):
    p = StepParams.izhikevich(input_mode=mode, nu=1e-4)
    # thresholds below the sustained calcium, so that elements grow (the reference's 0.4 never would)
    p.eta[0], p.eta[1], p.eta[2] = 0.02, 0.01, 0.0
    if case.get("synaptic"):
        p.synaptic_input = 1
        p.synapse_conductance = 0.03
    return p


def _edges(case, offsets, signal, gen):
    """A grown network: 4 to 12 synapses per axon to random partners of the neuron's own network, as
    in-edges by target, with the element counts that match."""
    n = case["neurons"]
    dev = "cuda"
    sizes = torch.tensor(np.diff(offsets.astype(np.int64)), device=dev)
    first = torch.repeat_interleave(torch.tensor(offsets[:-1].astype(np.int64), device=dev), sizes)
    size = torch.repeat_interleave(sizes, sizes)
    out_degree = torch.randint(IN_EDGES - 4, IN_EDGES + 5, (n,), device=dev, generator=gen)
    src = torch.repeat_interleave(torch.arange(n, device=dev), out_degree)
    hop = 1 + (torch.rand(src.numel(), dtype=torch.float64, device=dev, generator=gen) * (size[src] - 1)).long()
    tgt = first[src] + (src - first[src] + hop) % size[src]
    key = torch.sort(tgt * n + src).values
    tgt, src = key // n, key % n
    sig = torch.from_numpy(signal).to(dev)[src].long()
    off = torch.zeros(n + 1, dtype=torch.int64, device=dev)
    off[1:] = torch.cumsum(torch.bincount(tgt, minlength=n), 0)
    by_type = torch.bincount(tgt + n * sig, minlength=2 * n)
    connected = torch.cat([out_degree, by_type])
    grown = connected.double() + torch.rand(3 * n, dtype=torch.float64, device=dev, generator=gen)
    return (off.cpu().numpy().astype(np.uint64), src.cpu().numpy().astype(np.uint32),
            (1 - 2 * sig).cpu().numpy().astype(np.int32), connected.cpu().numpy().astype(np.uint32),
            grown.cpu().numpy())


def prepare(case, seed):
    s = State()
    s.case, s.lib, s.step = case, relearn_amd.load(), 0
    gen = _generator(case, seed)
    n, kind = case["neurons"], case["kind"]
    if kind == "commit":
        _prepare_commit(s, n, seed, gen)
    else:
        xyz, signal, offsets, boxes = _network(case, gen)
        s.ctx = _context(case, xyz, signal, offsets, boxes)
        if kind == "update":
            vac = [_poisson(n, m, gen) for m in (2.0, 1.5, 1.5)]
            s.slots = _slots(n)
            s.vac = vac if case["vacancies"] == "device" else [_pinned(n, torch.int32).copy_(v) for v in vac]
            s.left = [_pinned(n, torch.int32) for _ in range(3)]
            s.target, s.source, s.ordinal = (_pinned(s.slots, torch.int32) for _ in range(3))
            s.signal, s.ok = (_pinned(s.slots, torch.uint8) for _ in range(2))
        else:
            _neuron_buffers(s, n)
            x, u, ca, target = _neuron_state(case, gen)
            if kind == "period":
                zero = np.zeros(n, np.uint32)
                s.ctx.prepare_update_connectivity(zero, zero, zero)
                off, src, weight, connected, grown = _edges(case, offsets, signal, gen)
                s.ctx.net_init(3 * IN_EDGES * n, off, src, weight)
                s.ctx.neurons_init(_params(case, 1), target, x=x, u=u, ca=ca, grown=grown, connected=connected)
                s.ctx.graph_create(case["steps"], 4 * n)
                s.left = [_pinned(n, torch.int32) for _ in range(3)]
            elif kind == "steps":
                s.ctx.neurons_init(_params(case, 1), target, x=x, u=u, ca=ca)
            else:
                s.ctx.neurons_init(_params(case, 0), target, x=x, u=u, ca=ca)
                s.inputs = [t.cpu().pin_memory() for t in _background(case, gen)]
    torch.cuda.synchronize()
    return s


def _background(case, gen):
    for _ in range(case["steps"]):
        yield 5.0 + 2.0 * torch.randn(case["neurons"], dtype=torch.float64, device="cuda", generator=gen)


def _prepare_commit(s, n, seed, gen):
    """Requests in (source, axon) order of a search over n neurons; targets as a search spreads them."""
    axons = _poisson(n, 2.0, gen)
    source = torch.repeat_interleave(torch.arange(n, device="cuda"), axons.long())[:COMMIT_REQUESTS]
    m = source.numel()
    starts = torch.cumsum(axons.long(), 0) - axons.long()
    s.n, s.m, s.seed = n, m, int(seed)
    s.source = source.to(torch.int32)
    s.ordinal = (torch.arange(m, device="cuda") - starts[source]).to(torch.int32)
    s.target = torch.randint(0, n, (m,), device="cuda", generator=gen, dtype=torch.int32)
    s.signal = (torch.rand(n, device="cuda", generator=gen) >= 0.8).to(torch.uint8)[source]
    s.vac = [axons] + [_poisson(n, 1.5, gen) for _ in range(2)]
    s.left = [v.clone() for v in s.vac]
    s.taken = [torch.zeros_like(v) for v in s.vac]
    s.ok = torch.zeros(_slots(n), dtype=torch.uint8, device="cuda")


# ------------------------------------------------------------------------------------ passes


def run(state):
    return {"update": _run_update, "period": _run_period, "steps": _run_steps, "input": _run_steps,
            "commit": _run_commit}[state.case["kind"]](state)


def _run_update(s):
    lib, h, step = s.lib, s.ctx.h, s.step
    s.step += 1
    if s.case["vacancies"] == "device":
        _check(s, lib.rl_bh_prepare_update_connectivity_device(h, *[v.data_ptr() for v in s.vac]))
    else:
        _check(s, lib.rl_bh_prepare_update_connectivity(h, *[_ptr(v, C.c_uint32) for v in s.vac]))
    requests, created = C.c_uint64(), C.c_uint64()
    _check(s, lib.rl_bh_find_target_neurons(h, step, C.byref(requests)))
    _check(s, lib.rl_bh_commit(h, step, None, C.byref(created)))
    _check(s, lib.rl_bh_get_requests(h, s.slots, _ptr(s.target, C.c_uint32), _ptr(s.source, C.c_uint32),
                                     _ptr(s.signal, C.c_uint8), _ptr(s.ordinal, C.c_uint32)))
    _check(s, lib.rl_bh_get_commit_result(h, s.slots, _ptr(s.ok, C.c_uint8)))
    _check(s, lib.rl_bh_get_vacancies(h, *[_ptr(v, C.c_uint32) for v in s.left]))
    return {"requests": requests.value, "created": created.value, "target": s.target, "source": s.source,
            "signal": s.signal, "ordinal": s.ordinal, "ok": s.ok, "vacant": list(s.left)}


def _run_period(s):
    steps = s.case["steps"]
    st = s.ctx.graph_launch(s.step * steps, s.step)
    s.step += 1
    _check(s, s.lib.rl_bh_get_vacancies(s.ctx.h, *[_ptr(v, C.c_uint32) for v in s.left]))
    return dict(_get_neurons(s, True), vacant=list(s.left), requests=st["requests"], created=st["created"],
                deleted=st["deleted"])


def _run_steps(s):
    lib, h, steps = s.lib, s.ctx.h, s.case["steps"]
    for k in range(steps):
        given = _ptr(s.inputs[k], C.c_double) if s.case["kind"] == "input" else None
        _check(s, lib.rl_neurons_step(h, s.step * steps + k, given))
    s.step += 1
    return _get_neurons(s, False)


def _get_neurons(s, elements):
    """The neuron state; with `elements` also the grown and connected elements."""
    grown = _ptr(s.grown, C.c_double) if elements else None
    connected = _ptr(s.connected, C.c_uint32) if elements else None
    _check(s, s.lib.rl_neurons_get(s.ctx.h, *[_ptr(t, C.c_double) for t in (s.x, s.u, s.ca)],
                                   _ptr(s.fired, C.c_uint8), _ptr(s.delta, C.c_double), grown, connected))
    out = {"x": s.x, "u": s.u, "ca": s.ca, "fired": s.fired, "delta": s.delta}
    if elements:
        out["grown"], out["connected"] = s.grown, s.connected
    return out


def _run_commit(s):
    for left, taken, v in zip(s.left, s.taken, s.vac):
        left.copy_(v)
        taken.zero_()
    status = s.lib.rl_bh_commit_requests_noalloc(
        s.n, s.m, s.target.data_ptr(), s.source.data_ptr(), s.signal.data_ptr(), s.ordinal.data_ptr(), s.seed, s.step,
        *[t.data_ptr() for t in s.left], *[t.data_ptr() for t in s.taken], s.ok.data_ptr(),
        torch.cuda.current_stream().cuda_stream or None, None)
    s.step += 1
    if status != 0:
        raise RuntimeError(s.lib.rl_bh_last_error(None).decode())
    return {"ok": s.ok, "vacant": s.left, "connected": s.taken}


# ------------------------------------------------------------------------------------ work and exact values


def _tests_per_search(n):
    """Acceptance tests of one search in a uniform network at theta 0.3 (540 at 10^3 neurons, 2,120 at
    52,000, 3,700 at 10^6, 5,280 at 16 x 10^6)."""
    return 540.0 + 490.0 * max(0.0, math.log(n / 1000.0))


def work(case):
    n = case["neurons"]
    requests = 2.0 * n
    state = n * (3 * 8 + 1 + 3 * 8)        # x, u, calcium, fired status, element deltas
    step_flops = 10 * 17 + 10 * 4 + 3 * 30 + 60   # substeps, calcium, growth curves, background input
    if case["kind"] == "update":
        node = 40 if case["precision"] == "fp64" else 24
        tree = 1.47 * n * 2 * node
        # one list per source with a vacant axon (0.86 n), a distance, a comparison and a Gaussian per test
        flops = sum(0.86 * k * _tests_per_search(k) for k in _sizes(case)) * 20.0
        return {"bytes": 24.0 * n + tree + requests * 14, "flops": flops}
    if case["kind"] == "period":
        elements = n * (3 * 8 + 3 * 4 + 3 * 4)
        edges = n * IN_EDGES * 8 if case["synaptic"] else 0
        return {"bytes": float(2 * state + 2 * elements + edges), "flops": float(n * case["steps"] * step_flops)}
    if case["kind"] in ("steps", "input"):
        # every call reads and writes the state; the caller's input is read as well
        more = 8 * n if case["kind"] == "input" else 0
        return {"bytes": float(case["steps"] * (2 * state + more)),
                "flops": float(n * case["steps"] * step_flops)}
    return {"bytes": requests * 14 + n * 6 * 8.0, "flops": requests * 40}


def exact(case, seed):
    """The neuron steps with the caller's input in plain numpy (IEEE binary64)."""
    if case["kind"] != "input":
        return None
    gen = _generator(case, seed)
    _network(case, gen)
    x, u, ca, target = _neuron_state(case, gen)
    p = _params(case, 0)
    n, h = case["neurons"], p.h
    delta = np.zeros((3, n))
    fired = np.zeros(n, bool)
    for given in _background(case, gen):
        given = given.cpu().numpy()
        fired = np.zeros(n, bool)
        for _ in range(h):
            dx = p.k1 * x * x + p.k2 * x + p.k3 - u + given
            du = p.a * p.b * x - p.a * u
            x = np.where(fired, x, x + dx * (1.0 / h))
            u = np.where(fired, u, u + du * (1.0 / h))
            now = ~fired & (x >= p.v_spike)
            x, u = np.where(now, p.c, x), np.where(now, u + p.d, u)
            fired |= now
        for _ in range(h):
            ca = ca + (1.0 / h) * (ca * (-1.0 / p.tau_ca) + p.beta_ca * fired)
        for t in range(3):
            eta = p.eta[t]
            eps = np.maximum(target, eta)
            width = (eta - eps) / (2.0 * math.sqrt(math.log(2.0)))
            grow = 2.0 * np.exp(-((ca - (eta + eps) * 0.5) / width) ** 2) - 1.0
            delta[t] += p.nu[t] * grow
    return {"x": x, "u": u, "ca": ca, "fired": fired.astype(np.uint8), "delta": delta.ravel()}
