"""The timestep as users of this framework run it, case by case.

A pass advances simulations that are resident on the GPU by a number of steps
and reads their particles back, through the package's public entry points:

  single     Engine with one replica: step(n), then smd_engine_get
  ensemble   Engine with many replicas stepped together, then smd_engine_get
             of each
  serve      Server.run over a batch of jobs
  ps         the reference's ParticleSystem: update() per step, then the
             positions and types

Passes on one state continue its simulation.  The networks are those of
gpusmoldyn_amd.configs and gpusmoldyn_amd.serving: irreversible A + B -> C in
a reflective cube, reversible with decay in a periodic cube, clustered with a
reflective sphere and an absorbing plane, Michaelis-Menten in the reference's
world, and the random networks of the job stream.
"""
import ctypes
import math
import os

import numpy as np
import torch

import gpusmoldyn_amd as smd
from gpusmoldyn_amd import configs, serving

DENSITY = 2.048  # particles per um^3 of the A + B -> C workload
KF = 1e-3


def listed():
    return [
        # a driver that shows or stores a frame every ten steps of a small system
        dict(name="frames_2k", kind="single", network="bind", n=2048, steps=10),
        # the reference's host loop: update() and the particle count each step
        dict(name="particle_system_11k", kind="ps", n=11000, steps=50),
        # the plain workload of the benchmark: 8192 A + 8192 B, 1000 steps
        dict(name="plain_16k", kind="single", network="bind", n=16384, steps=1000),
        # an ordinary system of no round size
        dict(name="plain_100k", kind="single", network="bind", n=100003, steps=500),
        # 1M particles, periodic, splits with unbinding offsets, decay
        dict(name="periodic_1m", kind="single", network="reversible", n=1 << 20, steps=500),
        # 4M particles in blobs, sphere and absorbing plane
        dict(name="clustered_4m", kind="single", network="clustered", n=1 << 22, steps=200),
        # replicas of one small system for the statistics of its trajectories
        dict(name="replicas_256x2k", kind="ensemble", network="bind", replicas=256, nmin=2048, nmax=2048, steps=400),
        # a small sweep of a reversible network in periodic boxes
        dict(name="sweep_48_reversible", kind="ensemble", network="reversible", replicas=48, nmin=4096, nmax=131072,
             steps=300),
        # the batched ensemble of the benchmark: 512 replicas of 2k to 64k
        dict(name="ensemble_512", kind="ensemble", network="bind", replicas=512, nmin=2048, nmax=65536, steps=1000),
        # a batch of jobs of the serving stream's sizes and networks
        dict(name="serve_16_jobs", kind="serve", jobs=16, nmin=1000, nmax=262144, smin=100, smax=1000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["single", "single", "single", "ensemble", "ensemble", "serve", "ps"])
    if kind == "single":
        network = rng.choice(["bind", "bind", "reversible", "clustered"])
        lo, hi = {"bind": (2000, 1 << 20), "reversible": (30000, 1 << 21), "clustered": (200000, 1 << 22)}[network]
        n = _log_int(rng, lo, hi)
        top = {"bind": 1000, "reversible": 500, "clustered": 200}[network]
        return dict(kind=kind, network=network, n=n, steps=_log_int(rng, 10, min(top, 400000000 // n)))
    if kind == "ensemble":
        replicas = _log_int(rng, 16, 512)
        nmin = _log_int(rng, 1000, 4000)
        nmax = max(nmin, min(_log_int(rng, 2000, 131072), 8000000 // replicas))
        network = rng.choice(["bind", "bind", "reversible"])
        return dict(kind=kind, network=network, replicas=replicas, nmin=nmin, nmax=nmax,
                    steps=_log_int(rng, 100, min(1000, 2000000000 // (replicas * nmax))))
    if kind == "serve":
        return dict(kind=kind, jobs=rng.randint(4, 24), nmin=1000, nmax=_log_int(rng, 16384, 262144), smin=100,
                    smax=_log_int(rng, 200, 1000))
    return dict(kind=kind, n=_log_int(rng, 2000, 60000), steps=_log_int(rng, 20, 200))


def _sizes(case):
    """Replica (or job) sizes: log-uniform quantiles in a scattered order."""
    k = case["replicas"] if case["kind"] == "ensemble" else case["jobs"]
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    return [int(math.exp(lo + (hi - lo) * ((0.5 + i * 0.6180339887498949) % 1.0))) for i in range(k)]


def _job_steps(case):
    lo, hi = math.log(case["smin"]), math.log(case["smax"])
    return [int(math.exp(lo + (hi - lo) * ((0.5 + i * 0.7548776662466927) % 1.0))) for i in range(case["jobs"])]


def _streams(network, n):
    """Random streams per system, as the configurations choose them."""
    if network == "clustered":
        return max(64, n // 16)
    return configs.streams_for(n) if n > 32768 else 32768


def _box(rng, n, lo, hi):
    p = rng.random((n, 4), dtype=np.float32)
    p[:, :3] *= np.float32(hi - lo)
    p[:, :3] += np.float32(lo)
    p[:, 3] = 1.0
    return p


def _single(network, n, seed):
    """(spec, positions, types) of one system of about the configurations'
    densities; n particles, inputs from the seed."""
    rng = np.random.default_rng(seed)
    half = n // 2
    types = np.where(np.arange(n) < half, configs.A, configs.B).astype(np.int32)
    if network == "bind":
        if n <= 65536:
            spec = configs.c1_spec(KF, _streams(network, n), seed, configs.grid_bits_for(n) if n != 16384 else (6, 6, 6))
        else:
            L = (n / DENSITY) ** (1.0 / 3.0)
            spec = configs.make_spec(
                D=[0.0, 1.0, 1.0, 0.5], dt=1e-3,
                reactions=[dict(order=2, reactants=[configs.A, configs.B], products=[configs.C], rate=KF)],
                box_lo=[0.0] * 3, box_hi=[L] * 3, faces=[smd.BC_REFLECT] * 6, grid_bits=configs.grid_bits_for(n),
                num_streams=_streams(network, n), seed=seed)
        pos = _box(rng, n, 0.0, spec.box_hi[0])
    elif network == "reversible":
        L = float(n) ** (1.0 / 3.0) * (100.0 / 101.59366732596476)
        spec = configs.c2_spec(_streams(network, n), configs.grid_bits_for(2 * n), L, 1e-3, seed)
        pos = _box(rng, n, 0.0, L)
        pos, types = configs.cell_order(spec, pos, types)
    else:
        L = 200.0
        spec = configs.c3_spec(_streams(network, n), (8, 8, 7), 0.1, L, seed)
        centres = rng.uniform(0.0, L, size=(64, 3)).astype(np.float32)
        pos = np.empty((n, 4), np.float32)
        pos[:, :3] = centres[rng.integers(0, 64, size=n)] + 2.0 * rng.standard_normal((n, 3), dtype=np.float32)
        p = pos[:, :3]
        p[:] = np.clip(np.where(p < 0.0, -p, np.where(p > L, 2 * L - p, p)), 1e-4, L - 1e-4)
        pos[:, 3] = 1.0
        types = (np.arange(n) % 3 + 1).astype(np.int32)
        pos, types = configs.cell_order(spec, pos, types)
    return spec, pos, types


def _replicas(case, seed):
    """The ensemble's systems: forward rates log-uniform over the sweep, a
    stream per eight particles, particles in cell order."""
    out = []
    for i, n in enumerate(_sizes(case)):
        rng = np.random.default_rng([seed, i])
        s = (seed * 1009 + i) & 0x7FFFFFFF
        if case["network"] == "bind":
            kf = 1e-4 * 100.0 ** ((i * 0.5698402909980532) % 1.0)
            spec = configs.c1_spec(kf, configs.streams_for(n), s, configs.grid_bits_for(n))
        else:
            L = float(n) ** (1.0 / 3.0) * (100.0 / 101.59366732596476)
            spec = configs.c2_spec(configs.streams_for(n), configs.grid_bits_for(n), L, 1e-3, s)
        pos = _box(rng, n, 0.0, spec.box_hi[0])
        types = np.where(np.arange(n) < n // 2, configs.A, configs.B).astype(np.int32)
        pos, types = configs.cell_order(spec, pos, types)
        out.append((spec, pos, types))
    return out


def _ps_lib():
    L = smd.lib()
    vp = ctypes.c_void_p
    L.smd_ps_create.restype = vp
    L.smd_ps_create.argtypes = [ctypes.POINTER(smd.SimSpec), vp, vp, ctypes.c_uint, ctypes.c_int]
    for f in ("smd_ps_update", "smd_ps_num_particles", "smd_ps_destroy"):
        getattr(L, f).argtypes = [vp]
    L.smd_ps_get_positions.argtypes = [vp, vp, ctypes.c_uint]
    L.smd_ps_get_types.argtypes = [vp, vp, ctypes.c_uint]
    return L


class _ParticleSystem:
    """The C++ ParticleSystem through its C wrappers."""

    def __init__(self, spec, pos, types):
        self.lib = _ps_lib()
        self.h = self.lib.smd_ps_create(ctypes.byref(spec), pos.ctypes.data, types.ctypes.data, len(types), 0)
        if not self.h:
            raise smd.SmdError(smd.last_error())

    def __del__(self):
        if getattr(self, "h", None):
            self.lib.smd_ps_destroy(self.h)
            self.h = None

    def update(self):
        return self.lib.smd_ps_update(self.h)

    def read(self, pos, types):
        self.lib.smd_ps_get_positions(self.h, pos.ctypes.data, len(types))
        self.lib.smd_ps_get_types(self.h, types.ctypes.data, len(types))
        return self.lib.smd_ps_num_particles(self.h)


def prepare(case, seed):
    kind = case["kind"]
    seed = int(seed)
    if kind == "ps":
        spec, pos, types = configs.ref_test2(case["n"], rng_seed=seed)
        spec.seed = seed & 0x7FFFFFFF
        return dict(case=case, ps=_ParticleSystem(spec, pos, types), **_result(case["n"]))
    if kind == "serve":
        jobs = [serving.make_job(k, 0.0, n, s, 2 + k % 3, (seed * 1009 + k) & 0x7FFFFFFF, per_stream=2)
                for k, (n, s) in enumerate(zip(_sizes(case), _job_steps(case)))]
        return dict(case=case, jobs=jobs, server=serving.Server(), **_result(sum(_sizes(case))))
    reps = [_single(case["network"], case["n"], seed & 0x7FFFFFFF)] if kind == "single" else _replicas(case, seed)
    e = smd.Engine(0)
    for spec, pos, types in reps:
        e.add_replica(spec, pos, types)
    e.finalize()
    # a third of the clustered system's particles may split in two
    total = sum(len(r[2]) for r in reps)
    room = total + total // 3 + 64 if kind == "single" and case["network"] == "clustered" else total
    return dict(case=case, engine=e, **_result(room))


def _result(room):
    """The caller's arrays that a pass reads its particles into, one system
    after the other; what lies behind the last particle is zero."""
    return dict(pos=np.zeros((room, 4), np.float32), types=np.zeros(room, np.int32), used=0)


def _end_result(state, used, counts):
    if used < state["used"]:
        state["pos"][used:state["used"]] = 0
        state["types"][used:state["used"]] = 0
    state["used"] = used
    return dict(pos=state["pos"], types=state["types"], counts=np.array(counts, np.int64))


def run(state):
    case = state["case"]
    pos, types = state["pos"], state["types"]
    if case["kind"] == "ps":
        ps = state["ps"]
        for _ in range(case["steps"]):
            if ps.update() <= 0:
                raise smd.SmdError("update: " + smd.last_error())
        n = ps.read(pos, types)
        return _end_result(state, n, [n])
    at, counts = 0, []
    if case["kind"] == "serve":
        results, _ = state["server"].run(state["jobs"], realtime=False)
        for r in sorted(results, key=lambda r: r.jid):
            n = len(r.types)
            pos[at:at + n] = r.pos
            types[at:at + n] = r.types
            at += n
            counts.append(n)
        return _end_result(state, at, counts)
    e = state["engine"]
    e.step(case["steps"])
    L, n = smd.lib(), ctypes.c_uint(0)
    for r in range(len(e.specs)):
        # smd_engine_get of the C interface, straight into the caller's arrays
        rc = L.smd_engine_get(e._h, r, pos[at:].ctypes.data, types[at:].ctypes.data, len(types) - at, ctypes.byref(n))
        if rc != 0 or n.value > len(types) - at:
            raise smd.SmdError("smd_engine_get: " + smd.last_error())
        at += n.value
        counts.append(n.value)
    return _end_result(state, at, counts)


def work(case):
    """Per step: every particle's position, fourth component and type in and
    out (40 bytes), and the state of each stream in use in and out (80 bytes
    each way); the particles once more for the result.  About 60 floating
    operations per particle and step: the move, the walls, the cell, the
    distances to the neighbours."""
    kind = case["kind"]
    if kind == "serve":
        sizes, steps = _sizes(case), _job_steps(case)
        streams = [min(configs.streams_for(n, 2), 32768) for n in sizes]
    elif kind == "ensemble":
        sizes = _sizes(case)
        steps = [case["steps"]] * len(sizes)
        streams = [configs.streams_for(n) for n in sizes]
    elif kind == "ps":
        sizes, steps, streams = [case["n"]], [case["steps"]], [32768]
    else:
        sizes, steps, streams = [case["n"]], [case["steps"]], [_streams(case["network"], case["n"])]
    b = f = 0
    for n, k, s in zip(sizes, steps, streams):
        b += k * (40 * n + 160 * min(s, n)) + 20 * n
        f += k * 60 * n
    return dict(bytes=b, flops=f)


def _mt_states(words, seeds):
    s = np.zeros((19, len(seeds)), np.uint64)
    s[0] = seeds
    for i in range(1, 19):
        s[i] = (np.uint64(1812433253) * (s[i - 1] ^ (s[i - 1] >> np.uint64(30))) + np.uint64(i)) & np.uint64(0xFFFFFFFF)
    return dict(s=s, i=0, a=words[0], mb=words[1], mc=words[2])


def _mt_next(m):
    """One 32-bit draw of every stream (dcmt, 19 words, middle word 9)."""
    s, i = m["s"], m["i"]
    one = np.uint64(1)
    x = (s[i] & np.uint64(0xFFFFFFFE)) | (s[(i + 1) % 19] & one)
    y = s[(i + 9) % 19] ^ (x >> one) ^ np.where(x & one, m["a"], np.uint64(0))
    s[i] = y
    m["i"] = (i + 1) % 19
    y = y ^ (y >> np.uint64(12))
    y = y ^ ((y << np.uint64(7)) & m["mb"])
    y = y ^ ((y << np.uint64(15)) & m["mc"])
    return y ^ (y >> np.uint64(18))


def exact(case, seed):
    """Free diffusion between reflecting walls in 64 bits, for short runs of
    the irreversible network in which no A comes near a B (nothing reacts, so
    order and types stay); None where something may react: which pairs react,
    and so every later draw and place, is decided by the 32-bit positions."""
    if case["kind"] != "single" or case["network"] != "bind" or case["steps"] > 16 or case["n"] > 20000:
        return None
    n = case["n"]
    seed = int(seed) & 0x7FFFFFFF
    spec, pos, types = _single("bind", n, seed)
    dat = np.fromfile(os.path.join(os.path.dirname(smd.__file__), "data", "MersenneTwister.dat"), dtype="<u4")
    dat = dat.reshape(-1, 4).astype(np.uint64)
    streams = int(spec.num_streams)
    if n > streams:
        return None  # a stream that serves several particles in turn
    first = _mt_states(dat[:1, :3].T, np.array([spec.seed], np.uint64))
    seeds = np.array([int(_mt_next(first)[0]) for _ in range(n)], np.uint64)
    m = _mt_states(dat[np.arange(n) % len(dat), :3].T.copy(), seeds)
    q = torch.special.ndtri((torch.arange(4096, dtype=torch.float64) + 0.5) / 4096).numpy()
    gauss = np.roll(q, 1)
    rate = np.sqrt(2.0 * np.array([spec.D[t] for t in range(4)], np.float64) * float(np.float32(1e-3)))[types]
    lo, hi = float(spec.box_lo[0]), float(spec.box_hi[0])
    x = pos[:, :3].astype(np.float64)
    a, b = types == configs.A, types == configs.B
    for _ in range(case["steps"]):
        for d in range(3):
            x[:, d] += rate * gauss[(_mt_next(m) & np.uint64(4095)).astype(np.int64)]
        x = np.where(x > hi, 2 * hi - x, x)
        x = np.where(x < lo, 2 * lo - x, x)
        xa, xb = torch.from_numpy(x[a]), torch.from_numpy(x[b])
        if min(float(torch.cdist(c, xb).min()) for c in xa.split(1024)) < 0.007:  # the binding radius is 0.0062
            return None
    out = np.concatenate([x, pos[:, 3:].astype(np.float64)], axis=1)
    return dict(pos=out, types=types, counts=np.array([n], np.int64))
