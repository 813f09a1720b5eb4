"""Performance cases of the FMM library: what its users have it do.

`listed()` are fixed cases, `draw(rng)` gives another one of the same kinds and
ranges.  `prepare(case, seed)` makes the inputs a program has in hand,
`run(state)` is one pass through the public Python entry points, `work(case)`
the bytes and flops a pass cannot do without, and `exact(case, seed)` the
all-pairs sums in FP64 by plain torch, where they finish in a few seconds.

Every solve rebuilds its tree (particles move between calls); only the
operator tables of the process-wide default context stay between passes.
"""
import importlib
import math

import numpy as np
import torch

lfmm = importlib.import_module("laplace-fmm_amd")

DEVICE = "cuda:0"
MOST_PAIRS = 6e10  # all-pairs sums beyond this take too long for exact()


def listed():
    return [
        # the smallest calls: the drop-in class on host arrays, a few thousand
        # particles, one call per time step of a small simulation
        {"name": "host_3k_p8", "kind": "host", "n": 3000, "terms": 9, "leaf_max": 64},
        # the reference's plain configuration: 65,536 particles, p = 8, at
        # most 64 particles per leaf, all FP64
        {"name": "uniform_65k_p8", "kind": "uniform", "n": 65536, "terms": 9, "leaf_max": 64, "mixed": False},
        # a call with nothing but particles: eps = 1e-8 gives 18 terms and the
        # automatic depth leaves of a few hundred particles
        {"name": "uniform_1m_default", "kind": "default", "n": 1000003},
        # 4M particles, p = 10, FP64 operators throughout
        {"name": "uniform_4m_p10", "kind": "uniform", "n": 4194304, "terms": 11, "leaf_max": 64, "mixed": False},
        # the benchmark's headline: 4M particles at 1e-6, matrix-core M2L
        {"name": "uniform_4m_p12_mixed", "kind": "uniform", "n": 4194304, "terms": 13, "leaf_max": 64, "mixed": True},
        # clustered particles (a Plummer sphere) on the adaptive octree, FP64
        {"name": "plummer_1m_p12", "kind": "plummer", "n": 1048576, "terms": 13, "leaf_max": 64, "mixed": False},
        # the same at full size with the matrix-core M2L
        {"name": "plummer_4m_p12_mixed", "kind": "plummer", "n": 4194304, "terms": 13, "leaf_max": 64, "mixed": True},
        # separate sources and targets (a boundary integral's two meshes)
        {"name": "targets_262k_100k_p12", "kind": "targets", "n": 262144, "m": 100003, "terms": 13, "leaf_max": 64},
        # vector charges (Biot-Savart): the cross-product force
        {"name": "vector_100k_p10", "kind": "vector", "n": 100003, "terms": 11, "leaf_max": 64},
        # 512 independent systems of uneven size in one call
        {"name": "batch_512_p8", "kind": "batch", "systems": 512, "terms": 9, "leaf_max": 32, "mixed": False},
        # 2D complex series: 1M points, p = 20, at most 64 per leaf
        {"name": "plane_1m_p20", "kind": "plane", "n": 1048576, "terms": 21, "leaf_max": 64, "mixed": False},
        # a sampled accuracy check: FP64 direct sums on a few thousand targets
        {"name": "direct_4k_1m", "kind": "direct", "n": 1048576, "m": 4096},
    ]


def _between(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]; most of them odd or ragged."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "uniform", "uniform", "default", "plummer", "plummer", "targets", "vector", "batch",
                       "plane", "direct"])
    if kind == "host":
        return {"kind": kind, "n": _between(rng, 500, 20000), "terms": rng.randint(6, 12), "leaf_max": 64}
    if kind == "uniform":
        mixed = rng.random() < 0.5
        return {"kind": kind, "n": _between(rng, 20000, 4194304), "terms": rng.randint(7, 13 if mixed else 11),
                "leaf_max": rng.choice([48, 64, 96]), "mixed": mixed}
    if kind == "default":
        return {"kind": kind, "n": _between(rng, 20000, 2000000)}
    if kind == "plummer":
        mixed = rng.random() < 0.5
        return {"kind": kind, "n": _between(rng, 20000, 4194304 if mixed else 2000000),
                "terms": rng.randint(8, 13 if mixed else 12), "leaf_max": rng.choice([48, 64, 96]), "mixed": mixed}
    if kind == "targets":
        return {"kind": kind, "n": _between(rng, 20000, 400000), "m": _between(rng, 1000, 200000),
                "terms": rng.randint(8, 13), "leaf_max": 64}
    if kind == "vector":
        return {"kind": kind, "n": _between(rng, 20000, 200000), "terms": rng.randint(8, 12), "leaf_max": 64}
    if kind == "batch":
        return {"kind": kind, "systems": _between(rng, 8, 400), "terms": rng.randint(7, 9), "leaf_max": 32,
                "mixed": rng.random() < 0.5}
    if kind == "plane":
        return {"kind": kind, "n": _between(rng, 20000, 1048576), "terms": rng.randint(12, 25),
                "leaf_max": rng.choice([32, 64]), "mixed": rng.random() < 0.3}
    return {"kind": "direct", "n": _between(rng, 50000, 1000000), "m": _between(rng, 200, 4096)}


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, dtype=torch.float64, device=DEVICE, generator=g)


def _charges(g, *shape):
    return 2.0 * _rand(g, *shape) - 1.0


def _plummer(g, n, a=0.05, rmax=1.0):
    """A Plummer sphere of scale radius a truncated at rmax, centred in the unit cube."""
    u = _rand(g, n) * (1.0 + (a / rmax) ** 2) ** -1.5
    r = a / torch.sqrt(u.clamp_min(1e-12) ** (-2.0 / 3.0) - 1.0)
    d = torch.randn(n, 3, dtype=torch.float64, device=DEVICE, generator=g)
    return 0.5 + r[:, None] * d / d.norm(dim=1, keepdim=True)


def _batch_sizes(k):
    """k sizes, log-uniform in [1024, 65536], the same for every seed."""
    return np.rint(np.exp(np.random.default_rng(k).uniform(math.log(1024), math.log(65536), k))).astype(np.int64)


def _batch(case, seed):
    """Independent systems packed one after another; even ones uniform in the
    unit cube, odd ones four Gaussian blobs (sigma 0.05)."""
    k = case["systems"]
    sizes = _batch_sizes(k)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    total = int(off[-1])
    g = _generator(seed)
    system = torch.repeat_interleave(torch.arange(k, device=DEVICE), torch.from_numpy(sizes).to(DEVICE))
    centres = 0.2 + 0.6 * _rand(g, k, 4, 3)
    pick = torch.randint(0, 4, (total,), device=DEVICE, generator=g)
    blob = centres[system, pick] + 0.05 * torch.randn(total, 3, dtype=torch.float64, device=DEVICE, generator=g)
    xyz = torch.where((system % 2 == 1)[:, None], blob, _rand(g, total, 3))
    return xyz.contiguous(), _charges(g, total), off


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "host":  # rows (x, y, z, q), as the class takes them
        rng = np.random.default_rng(seed)
        s["particles"] = np.concatenate([rng.random((case["n"], 3)), rng.uniform(-1.0, 1.0, (case["n"], 1))], axis=1)
        return s
    if kind == "batch":
        s["xyz"], s["q"], s["offsets"] = _batch(case, seed)
        return s
    g = _generator(seed)
    if kind == "plummer":
        s["xyz"] = _plummer(g, case["n"])
    else:
        s["xyz"] = _rand(g, case["n"], 2 if kind == "plane" else 3)
    s["q"] = _charges(g, case["n"], 3) if kind == "vector" else _charges(g, case["n"])
    if kind in ("targets", "direct"):
        s["targets"] = _rand(g, case["m"], 3)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "host":
        f = lfmm.FastMultipole3d(s["particles"], N=case["terms"], leaf_max=case["leaf_max"])
        return f.potentials, f.forces
    if kind == "uniform":
        return lfmm.fmm3d(s["xyz"], s["q"], terms=case["terms"], leaf_max=case["leaf_max"], mixed=case["mixed"])[:2]
    if kind == "default":
        return lfmm.fmm3d(s["xyz"], s["q"])[:2]
    if kind == "plummer":
        return lfmm.fmm3d(s["xyz"], s["q"], terms=case["terms"], leaf_max=case["leaf_max"], mixed=case["mixed"],
                          adaptive=True, exclude_self=True)[:2]
    if kind == "targets":
        return lfmm.fmm3d(s["xyz"], s["q"], terms=case["terms"], leaf_max=case["leaf_max"], targets=s["targets"])[:2]
    if kind == "vector":
        return lfmm.fmm3d_vec(s["xyz"], s["q"], terms=case["terms"], leaf_max=case["leaf_max"])[0]
    if kind == "batch":
        return lfmm.fmm3d_batch(s["xyz"], s["q"], s["offsets"], terms=case["terms"], leaf_max=case["leaf_max"],
                                mixed=case["mixed"], adaptive=True)
    if kind == "plane":
        return lfmm.fmm2d(s["xyz"], s["q"], terms=case["terms"], leaf_max=case["leaf_max"], mixed=case["mixed"])[:2]
    return lfmm.direct3d(s["xyz"], s["q"], targets=s["targets"])


def _m2l_flops(terms):
    """Rotate, translate along the axis, rotate back: flops of one 3D M2L."""
    rotate = sum((n + 1) * (4 * n + 2) for n in range(terms))
    return 2 * (3 * terms * (terms + 1) + rotate) + 4 * sum(t * t for t in range(1, terms + 1))


def work(case):
    """Particles read once and results written once; the pair sums of the near
    field (20 flops each) and the M2L of the far field, on leaves of typical
    filling (other passes are small beside them)."""
    kind = case["kind"]
    if kind == "direct":
        return {"bytes": 32.0 * case["n"] + 56.0 * case["m"], "flops": 20.0 * case["n"] * case["m"]}
    n = float(_batch_sizes(case["systems"]).sum()) if kind == "batch" else float(case["n"])
    m = float(case.get("m", n))
    dim = 2 if kind == "plane" else 3
    most = case.get("leaf_max")
    level = 0
    if most is None:
        level = max(1, int(1 + math.log(n / 100.0) / math.log(8.0)) - 1)
    elif kind in ("plummer", "batch"):
        level = math.log(n / (0.3 * most)) / math.log(8.0)
    else:
        while n / 2.0 ** (dim * level) > 0.6 * most:
            level += 1
    leaves = max(1.0, 2.0 ** (dim * level))
    pairs = m * 3.0 ** dim * n / leaves
    far = level >= 2
    if dim == 2:
        flops = 14.0 * pairs + (leaves * 4 / 3 * 27 * 4.5 * case["terms"] ** 2 if far else 0.0)
        return {"bytes": 24.0 * n + 24.0 * m, "flops": flops}
    reach = min(189.0, 0.8 * 189.0 * (1 - 2.0 ** (1 - level)) / 0.75) if far else 0.0
    m2l = leaves * 8 / 7 * reach * _m2l_flops(case.get("terms", 18))
    if kind == "vector":
        return {"bytes": 72.0 * n, "flops": 3.0 * (20.0 * pairs + m2l)}
    return {"bytes": 32.0 * n + (24.0 if m != n else 0.0) * m + 32.0 * m, "flops": 20.0 * pairs + m2l}


def _sums3d(targets, xyz, q, exclude_self=False):
    """All-pairs potential and field (r clamped at 1e-4, as the library's)."""
    m, n = targets.shape[0], xyz.shape[0]
    pot = torch.empty(m, dtype=torch.float64, device=targets.device)
    field = torch.empty(m, 3, dtype=torch.float64, device=targets.device)
    step = max(1, (1 << 26) // n)
    for b in range(0, m, step):
        d = [targets[b:b + step, k, None] - xyz[None, :, k] for k in range(3)]
        inv = (d[0] * d[0] + d[1] * d[1] + d[2] * d[2]).clamp_min_(1e-8).rsqrt_()
        if exclude_self:
            rows = torch.arange(inv.shape[0], device=inv.device)
            inv[rows, rows + b] = 0.0
        pot[b:b + step] = inv @ q
        inv3 = inv.pow_(3)
        for k in range(3):
            field[b:b + step, k] = d[k].mul_(inv3) @ q
    return pot, field


def _sums2d(xy, q):
    n = xy.shape[0]
    pot = torch.empty(n, dtype=torch.float64, device=xy.device)
    force = torch.empty(n, 2, dtype=torch.float64, device=xy.device)
    step = max(1, (1 << 26) // n)
    for b in range(0, n, step):
        dx = xy[b:b + step, 0, None] - xy[None, :, 0]
        dy = xy[b:b + step, 1, None] - xy[None, :, 1]
        r2 = (dx * dx + dy * dy).clamp_min_(1e-8)
        force[b:b + step, 0] = (dx / r2) @ q
        force[b:b + step, 1] = -((dy / r2) @ q)
        pot[b:b + step] = r2.log_().mul_(0.5) @ q
    return pot, force


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        pairs = float((_batch_sizes(case["systems"]).astype(np.float64) ** 2).sum())
    else:
        pairs = float(case["n"]) * case.get("m", case["n"]) * (3 if kind == "vector" else 1)
    if pairs > MOST_PAIRS:
        return None
    s = prepare(case, seed)
    if kind == "host":
        p = torch.from_numpy(s["particles"])
        pot, field = _sums3d(p[:, :3], p[:, :3], p[:, 3])
        return pot.numpy(), field.numpy()
    xyz, q = s["xyz"], s["q"]
    if kind == "plane":
        return _sums2d(xyz, q)
    if kind == "vector":  # sum q_j x r / |r|^3 from the fields of the components
        e = [_sums3d(xyz, xyz, q[:, k].contiguous())[1] for k in range(3)]
        return torch.stack([e[1][:, 2] - e[2][:, 1], e[2][:, 0] - e[0][:, 2], e[0][:, 1] - e[1][:, 0]], dim=1)
    if kind == "batch":
        off = s["offsets"]
        parts = [_sums3d(xyz[a:b], xyz[a:b], q[a:b]) for a, b in zip(off[:-1], off[1:])]
        return torch.cat([p for p, _ in parts]), torch.cat([f for _, f in parts])
    return _sums3d(s.get("targets", xyz), xyz, q, exclude_self=kind == "plummer")
