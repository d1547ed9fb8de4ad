"""The workloads a user of this framework runs, as timed cases.

Every case goes through the public entry points: ``trimem_amd.core`` and
``trimem_amd.mc`` as trimem's own samplers call them, or the C ABI
(``trimem_amd.capi``) with torch tensors on the library's stream.  Meshes are
geodesic spheres of frequency ``nu`` (10 nu^2 + 2 vertices; nu = 2^L has the
sizes of the icosphere of level L), jittered by 1% of the mean edge, with the
parameters of ``trimem_amd.workloads.base_params``, or open tubes.

  dropin     energy() and gradient() of a host array of positions: one force
             evaluation of a host sampler or minimiser
  device     the same in device memory: positions written from a torch tensor,
             the gradient read back into one in the caller's vertex order
  mc         the plain configuration's step: a device HMC trajectory, a serial
             flip sweep, the neighbour list rebuilt
  hmc        device HMC trajectories with the list rebuilt after each
  flip       serial flip sweeps (trimem's bit-exact chain)
  pflip      parallel flip sweeps
  tempering  a replica group: grouped HMC steps and kappa_b exchanges
  combined   a replica group: grouped HMC step, parallel flip sweep of every
             mesh, exchange, lists rebuilt
  surrogate  loss and parameter gradient of the force network (forward and
             backward) against the exact gradient

``draw`` gives cases of the same kinds over the same ranges: mesh sizes from
642 vertices to the largest listed ones, log-uniform in the frequency, odd
frequencies included, both precisions, both list kinds, exclusion levels 0 to
2, both bond types, closed and open meshes.
"""
import contextlib
import ctypes
import functools
import io
import math

import numpy as np
import torch


def listed():
    return [
        # one force evaluation on the smallest mesh: launches and copies
        {"name": "dropin_small", "kind": "dropin", "shape": "sphere", "nu": 8, "precision": "fp64"},
        # an open tube with a Verlet list and the area bond
        {"name": "dropin_tube", "kind": "dropin", "shape": "tube", "segments": 75, "precision": "fp64", "nlist": 1,
         "exclusion": 1, "bond": 1},
        # a biconcave vesicle whose two membranes repel each other
        {"name": "dropin_disc", "kind": "dropin", "shape": "disc", "nu": 64, "precision": "mixed"},
        # the largest single mesh from host positions, default precision
        {"name": "dropin_large", "kind": "dropin", "shape": "sphere", "nu": 128, "precision": "fp64"},
        # the largest single mesh resident on the GPU (the benchmark's mesh)
        {"name": "device_large", "kind": "device", "shape": "sphere", "nu": 128, "precision": "mixed"},
        # the plain configuration: level 4, FP64, flips of 10% of the edges
        {"name": "mc_plain", "kind": "mc", "nu": 16, "precision": "fp64", "ratio": 0.1, "steps": 2},
        # the single-mesh configuration: trajectories with a rebuild per step
        {"name": "hmc_large", "kind": "hmc", "nu": 128, "precision": "mixed", "steps": 4},
        # flip sweeps over 10% of the edges of the same mesh
        {"name": "flip_large", "kind": "flip", "nu": 128, "precision": "mixed", "ratio": 0.1, "sweeps": 2},
        {"name": "pflip_large", "kind": "pflip", "nu": 128, "precision": "mixed", "ratio": 0.1, "sweeps": 4},
        # 64 meshes of uneven sizes, exchange every 10 steps
        {"name": "tempering_64", "kind": "tempering", "replicas": 64, "precision": "mixed", "nu_lo": 8, "nu_hi": 64,
         "steps": 10},
        # 8 large meshes, flips of 20% of the edges of each per step
        {"name": "combined_8", "kind": "combined", "replicas": 8, "precision": "mixed", "nu": 128, "ratio": 0.2},
        # training the surrogate at level 6
        {"name": "surrogate", "kind": "surrogate", "nu": 64, "precision": "mixed"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "dropin", "dropin", "device", "mc", "hmc", "flip", "pflip", "tempering", "combined",
                       "surrogate"])
    case = {"kind": kind, "precision": rng.choice(["fp64", "mixed"])}
    options = {"nlist": rng.choice([0, 0, 1]), "exclusion": rng.choice([0, 1, 2, 2, 2])}
    if kind in ("dropin", "device"):
        case["shape"] = rng.choice(["sphere", "disc", "tube"] if kind == "dropin" else ["sphere", "disc"])
        case.update(options, bond=rng.choice([0, 0, 1]))
        if case["shape"] == "tube":
            case["segments"] = _log_int(rng, 20, 200)
        else:
            case["nu"] = _log_int(rng, 8, 128)
    elif kind == "mc":
        case.update(nu=_log_int(rng, 8, 48), ratio=0.1, steps=2)
    elif kind == "hmc":
        options["exclusion"] = max(options["exclusion"], 1)    # bonded neighbours do not repel in a trajectory
        case.update(options, nu=_log_int(rng, 8, 128), steps=rng.randint(1, 4))
    elif kind == "flip":
        options["exclusion"] = rng.choice([0, 2, 2])    # at level 1 no flip of a repelling mesh is ever accepted
        case.update(options, nu=_log_int(rng, 16, 128), ratio=0.1, sweeps=rng.randint(1, 2))
    elif kind == "pflip":
        options["exclusion"] = rng.choice([0, 2, 2])
        case.update(options, nu=_log_int(rng, 16, 128), ratio=rng.choice([0.1, 0.2]), sweeps=rng.randint(1, 2))
    elif kind == "tempering":
        lo = _log_int(rng, 8, 24)
        case.update(replicas=rng.randint(3, 64), nu_lo=lo, nu_hi=_log_int(rng, lo, 64), steps=rng.randint(2, 10))
    elif kind == "combined":
        case.update(replicas=rng.randint(2, 8), nu=_log_int(rng, 12, 128), ratio=0.2)
    else:
        case.update(nu=_log_int(rng, 8, 64))
    return case


# ------------------------------------------------------------------ inputs --
@functools.lru_cache(maxsize=4)
def _sphere(nu):
    """Icosahedron faces cut into nu^2 triangles each, projected onto the unit
    sphere (trimem's icospheres are those of nu = 2^L)."""
    from trimem_amd import meshes
    v, f = meshes.icosahedron()
    i, j = (a.ravel() for a in np.meshgrid(np.arange(nu + 1), np.arange(nu + 1), indexing="ij"))
    keep = i + j <= nu
    i, j = i[keep], j[keep]
    local = np.full((nu + 1, nu + 1), -1)
    local[i, j] = np.arange(len(i))
    w = np.stack([nu - i - j, i, j], axis=1) / nu
    pts = np.einsum("pk,fkd->fpd", w, v[f])
    key = np.round(pts.reshape(-1, 3) * 1e6).astype(np.int64)
    _, first, inverse = np.unique(key, axis=0, return_index=True, return_inverse=True)
    order = np.argsort(first)
    rank = np.empty_like(order)
    rank[order] = np.arange(len(order))
    ids = rank[inverse.ravel()].reshape(len(f), -1)
    p = pts.reshape(-1, 3)[first[order]]
    p = p / np.linalg.norm(p, axis=1, keepdims=True)
    up = i + j < nu
    down = i + j < nu - 1
    t = np.concatenate([np.stack([local[i[up], j[up]], local[i[up] + 1, j[up]], local[i[up], j[up] + 1]], 1),
                        np.stack([local[i[down] + 1, j[down]], local[i[down] + 1, j[down] + 1],
                                  local[i[down], j[down] + 1]], 1)])
    return p, np.ascontiguousarray(ids[:, t].reshape(-1, 3).astype(np.int32))


@functools.lru_cache(maxsize=4)
def _shape(shape, size):
    """(points, faces, mean edge length) without jitter."""
    from trimem_amd import meshes
    if shape == "tube":
        v, f = meshes.tube(length=3.0, radius=1.0, segments=size)
        f = np.ascontiguousarray(f.astype(np.int32))
        return v, f, meshes.mean_edge_length(v, f)
    v, f = _sphere(size)
    lbar = meshes.mean_edge_length(v, f)
    if shape == "disc":    # thickness 1.2 mean edges at the centre
        r2 = v[:, 0] ** 2 + v[:, 1] ** 2
        c = 0.6 * lbar
        v = v * np.stack([np.ones_like(r2), np.ones_like(r2), c + (1.0 - c) * r2], axis=1)
    return v, f, lbar


def _inputs(case, seed, nu=None):
    """(created positions, evaluated positions, faces, parameter dict)."""
    from trimem_amd import workloads
    shape = case.get("shape", "sphere")
    v, f, lbar = _shape(shape, case["segments"] if shape == "tube" else nu or case["nu"])
    rng = np.random.default_rng(seed)
    x0 = np.ascontiguousarray(v + rng.normal(0.0, 0.01 * lbar, v.shape))
    x1 = np.ascontiguousarray(x0 + rng.normal(0.0, 0.005 * lbar, v.shape))
    p = dict(workloads.base_params(lbar), rep_nlist=case.get("nlist", 0), rep_exclusion=case.get("exclusion", 2),
             bond_type=case.get("bond", 0), bond_a0=math.sqrt(3.0) / 4.0 * lbar * lbar)
    if case["kind"] in ("flip", "pflip"):
        # the tether's cost of a flip at nu = 128 whatever the mesh, so that
        # sweeps of every size accept some (about 1.4% of the proposals)
        p["kappa_t"] *= (case["nu"] / 128.0) ** 2
    return x0, x1, f, p


def _system(x, f, p, precision):
    from trimem_amd import core, workloads
    mesh = core.TriMesh(x, f)
    est = core.EnergyManager(mesh, workloads.core_params(core, p))
    est.precision = precision
    return mesh, est


class _DeviceArray:
    """A device buffer of the library as torch.as_tensor takes it; the tensor
    keeps the buffer's owner alive."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        addr = ctypes.cast(ptr, ctypes.c_void_p).value
        self.__cuda_array_interface__ = {"data": (addr, False), "shape": shape, "typestr": "<f8", "version": 2}


def _rows_of(a, b):
    """perm with b == a[perm] for two orders of the same (distinct) rows."""
    perm = np.empty(len(a), dtype=np.int64)
    perm[np.lexsort(b.T)] = np.lexsort(a.T)
    return perm


def _time_step(nu):
    return 1e-4 * (16.0 / nu) ** 1.5


def _sampler(x, f, p, precision, seed):
    from trimem_amd import core, workloads
    from trimem_amd.mc import hmc
    from trimem_amd.mc.mesh import Mesh
    mesh = Mesh(x, f)
    est = core.EnergyManager(mesh.trimesh, workloads.core_params(core, p))
    est.precision = precision
    nu = math.sqrt((len(x) - 2) / 10.0)
    opts = {"time_step": _time_step(nu), "num_integration_steps": 10, "info_step": 0}
    with contextlib.redirect_stdout(io.StringIO()):    # the options table
        chain = hmc.DeviceMeshHMC(mesh, est, counter=hmc.get_step_counters(), options=opts, rng="device", seed=seed)
    return mesh, est, chain


def prepare(case, seed):
    from trimem_amd import capi, core
    kind, precision = case["kind"], case["precision"]
    s = {"case": case, "seed": seed, "n": 0}
    if kind in ("tempering", "combined"):
        rng = np.random.default_rng(seed + 1000)
        pick = np.random.default_rng(1000)    # the sizes belong to the case
        R = case["replicas"]
        lo, hi = (case["nu_lo"], case["nu_hi"]) if kind == "tempering" else (case["nu"], case["nu"])
        if kind == "tempering":    # levels as in the 64-replica set: sizes lo, 2 lo, 4 lo ... up to hi
            sizes = [lo << k for k in range(int(math.log2(hi / lo)) + 1)]
            nus = [sizes[k] for k in pick.integers(0, len(sizes), R)]
            ladder = np.sort(np.exp(rng.uniform(np.log(10.0), np.log(100.0), R)))
            vfrac = rng.uniform(0.6, 0.95, R)
        else:
            nus = [lo] * R
            ladder = np.sort(np.exp(rng.uniform(np.log(20.0), np.log(80.0), R)))
            vfrac = rng.uniform(0.55, 0.9, R)
        s["meshes"], s["ests"] = [], []
        for r in range(R):
            x0, _, f, p = _inputs(case, seed + 7 * r + 1, nus[r])
            mesh, est = _system(x0, f, dict(p, kappa_b=float(ladder[r]), volume_frac=float(vfrac[r])), precision)
            s["meshes"].append(mesh)
            s["ests"].append(est)
        s["group"] = core.Replicas(s["meshes"], s["ests"])
        s["group"].hmc_setup(mass=1.0, time_step=_time_step(hi), temperature=1.0,
                             seeds=[seed + r for r in range(R)], num_integration_steps=10)
        s["group"].set_ladder(list(ladder), seed=seed)
        return s
    x0, x1, f, p = _inputs(case, seed)
    if kind in ("mc", "hmc"):
        s["mesh"], s["est"], s["chain"] = _sampler(x0, f, p, precision, seed)
        return s
    s["mesh"], s["est"] = _system(x0, f, p, precision)
    s["x"] = x1
    if kind == "surrogate":
        s["mesh"].points()[:] = x1
        s["net"] = core.Surrogate(s["mesh"], s["est"], seed=seed)
    if kind == "device":
        L, n = capi.lib(), len(x0)
        s["lib"] = L
        s["handles"] = ctypes.c_void_p(s["est"]._handle()), ctypes.c_void_p(s["mesh"]._handle())
        stream = ctypes.c_void_p()
        capi.check(L.tm_stream(ctypes.byref(stream)))
        s["stream"] = torch.cuda.ExternalStream(stream.value)
        capi.check(L.tm_mesh_upload_points(s["handles"][1]))
        capi.check(L.tm_energy_eval_device(*s["handles"], capi.TM_EVAL_PROPS | capi.TM_EVAL_GRAD))
        capi.check(L.tm_sync())
        for name, ptr, shape in (("points", L.tm_mesh_device_points(s["handles"][1]), (n, 3)),
                                 ("grad", L.tm_energy_device_gradient(s["handles"][0]), (n, 3)),
                                 ("globals", L.tm_energy_device_globals(s["handles"][0]), (7,))):
            s[name] = torch.as_tensor(_DeviceArray(ptr, shape, (s["mesh"], s["est"])), device="cuda")
        order = _rows_of(x0, s["points"].cpu().numpy())    # the library's vertex order
        s["to_library"] = torch.from_numpy(order).cuda()
        s["to_caller"] = torch.from_numpy(np.argsort(order)).cuda()
        s["x"] = torch.from_numpy(x1).cuda()
        torch.cuda.synchronize()
    return s


def run(s):
    from trimem_amd import capi, core
    case = s["case"]
    kind = case["kind"]
    if kind == "dropin":
        s["mesh"].points()[:] = s["x"]
        return {"energy": s["est"].energy(s["mesh"]), "gradient": s["est"].gradient(s["mesh"])}
    if kind == "device":
        with torch.cuda.stream(s["stream"]):
            torch.index_select(s["x"], 0, s["to_library"], out=s["points"])
            capi.check(s["lib"].tm_energy_eval_device(*s["handles"], capi.TM_EVAL_PROPS | capi.TM_EVAL_GRAD))
            return {"globals": s["globals"], "gradient": torch.index_select(s["grad"], 0, s["to_caller"])}
    if kind in ("mc", "hmc"):
        for _ in range(case["steps"]):
            s["chain"].step()
            if kind == "mc":
                core.flip(s["mesh"].trimesh, s["est"], case["ratio"], seed=s["seed"] + s["n"])
            s["est"].update_repulsion(s["mesh"].trimesh)
            s["n"] += 1
        out = s["chain"].result()
        out = {"energy": out["energy0"], "kinetic": out["kinetic0"], "accepted": out["n_accepted"],
               "points": s["mesh"].trimesh.points()}
        if kind == "mc":
            out["faces"] = s["mesh"].trimesh.fv_indices()
        return out
    if kind in ("flip", "pflip"):
        sweep = core.flip if kind == "flip" else core.pflip
        accepted = 0
        for _ in range(case["sweeps"]):
            accepted += sweep(s["mesh"], s["est"], case["ratio"], seed=s["seed"] + s["n"])
            s["n"] += 1
        return {"accepted": accepted, "faces": s["mesh"].fv_indices()}
    if kind == "tempering":
        s["group"].hmc_run(case["steps"], swap_every=10)
        s["group"].update_repulsion()
    if kind == "combined":
        s["group"].hmc_run(1)
        flips = s["group"].pflip(case["ratio"], [s["seed"] + 100 * s["n"] + r for r in range(case["replicas"])])
        s["group"].swap()
        s["group"].update_repulsion()
        s["n"] += 1
    if kind in ("tempering", "combined"):
        stats = s["group"].stats()
        out = {"accepted": stats["accepted"], "slots": stats["slot_of"], "properties": stats["props"],
               "points": np.concatenate([m.points() for m in s["meshes"]])}
        if kind == "combined":
            out["flips"] = np.array(flips)
            out["faces"] = np.concatenate([m.fv_indices() for m in s["meshes"]])
        return out
    loss, grad = s["net"].loss_grad()
    return {"loss": np.float32(loss), "gradient": grad}    # both are FP32 sums


# ------------------------------------------------------------------- work --
def work(case):
    """Bytes: positions (24 per vertex) and faces (12 per face) in, the
    gradient (24 per vertex) out, per force evaluation; FLOPs: about 1500 per
    vertex of a closed mesh for both passes.  A leapfrog step also reads and
    writes positions, momenta and forces; a flip proposal reads four one-rings
    (about 18 vertices and 40 halfedges) and writes a few ids."""
    kind = case["kind"]
    if case.get("shape") == "tube":
        n = case["segments"] * (int(3.0 / (2.0 * math.pi / case["segments"])) + 1)
    elif kind == "tempering":
        sizes = [case["nu_lo"] << k for k in range(int(math.log2(case["nu_hi"] / case["nu_lo"])) + 1)]
        n = case["replicas"] * sum(10 * u * u + 2 for u in sizes) // len(sizes)
    else:
        n = case.get("replicas", 1) * (10 * case["nu"] ** 2 + 2)
    force_b, force_f = 24.0 * n + 24.0 * n + 24.0 * n, 1500.0 * n
    step_b, step_f = 11 * (force_b + 5 * 24.0 * n), 11 * force_f
    list_b = 24.0 * n + 8.0 * n
    flip_b, flip_f = 18 * 24.0 + 40 * 16.0, 8 * 6 * 150.0
    if kind in ("dropin", "device"):
        return {"bytes": force_b, "flops": force_f}
    if kind == "mc":
        nflip = case["ratio"] * 3 * n
        return {"bytes": case["steps"] * (step_b + list_b + nflip * flip_b),
                "flops": case["steps"] * (step_f + nflip * flip_f)}
    if kind in ("hmc", "tempering"):
        return {"bytes": case["steps"] * (step_b + (list_b if kind == "hmc" else 0)), "flops": case["steps"] * step_f}
    if kind in ("flip", "pflip"):
        nflip = case["sweeps"] * case["ratio"] * 3 * n
        return {"bytes": nflip * flip_b, "flops": nflip * flip_f}
    if kind == "combined":
        nflip = case["ratio"] * 3 * n
        return {"bytes": step_b + list_b + nflip * flip_b, "flops": step_f + nflip * flip_f}
    dense = 16 * 64 + 3 * (64 * 64 + 128 * 64)
    return {"bytes": force_b + 4.0 * 64 * n * 2 * 10, "flops": force_f + 6.0 * n * dense}


# ------------------------------------------------------------ 64-bit values --
def _edges(f, n):
    """Undirected edges (i, j), the vertex opposite in the face of i -> j and
    in that of j -> i (-1 on a boundary)."""
    a, b, c = (np.concatenate([f[:, k % 3], f[:, (k + 1) % 3], f[:, (k + 2) % 3]]).astype(np.int64) for k in range(3))
    key, twin = a * n + b, b * n + a
    order = np.argsort(key)
    at = np.searchsorted(key[order], twin)
    at = np.minimum(at, len(key) - 1)
    has = key[order][at] == twin
    other = np.where(has, c[order][at], -1)
    keep = (a < b) | ~has
    return a[keep], b[keep], c[keep], other[keep]


def _pairs(x, f, n, cutoff, level):
    """Unordered pairs within the cutoff outside the exclusion neighbourhood."""
    cell = np.floor((x - x.min(0)) / cutoff).astype(np.int64) + 1
    dim = cell.max(0) + 2
    flat = (cell[:, 2] * dim[1] + cell[:, 1]) * dim[0] + cell[:, 0]
    order = np.argsort(flat, kind="stable")
    ids = flat[order]
    out = []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            t = flat + (dz * dim[1] + dy) * dim[0]
            lo, hi = np.searchsorted(ids, t - 1, "left"), np.searchsorted(ids, t + 1, "right")
            cnt = hi - lo
            i = np.repeat(np.arange(n), cnt)
            j = order[np.arange(cnt.sum()) - np.repeat(np.cumsum(cnt) - cnt, cnt) + np.repeat(lo, cnt)]
            near = (i < j) & (((x[i] - x[j]) ** 2).sum(1) < cutoff * cutoff)
            out.append(np.stack([i[near], j[near]], 1))
    p = np.concatenate(out)
    if level >= 1:
        a, b, _, _ = _edges(f, n)
        s, d = np.concatenate([a, b]), np.concatenate([b, a])
        o = np.argsort(s, kind="stable")
        s, d = s[o], d[o]
        bad = np.minimum(s, d) * n + np.maximum(s, d)
        if level >= 2:
            start = np.searchsorted(s, np.arange(n + 1))
            cnt = (start[1:] - start[:-1])[s]
            first = np.repeat(d, cnt)
            second = d[np.arange(cnt.sum()) - np.repeat(np.cumsum(cnt) - cnt, cnt) + np.repeat(start[s], cnt)]
            bad = np.concatenate([bad, np.minimum(first, second) * n + np.maximum(first, second)])
        p = p[~np.isin(p[:, 0] * n + p[:, 1], np.unique(bad))]
    return p


def _properties(x, f, edges, p, pairs):
    """Area, volume, curvature, bending, tethering, repulsion (FP64 torch)."""
    n = len(x)
    ft = torch.from_numpy(f.astype(np.int64))
    a, b, c = x[ft[:, 0]], x[ft[:, 1]], x[ft[:, 2]]
    af = torch.linalg.norm(torch.linalg.cross(b - a, c - a), dim=1) / 2
    vol = (a * torch.linalg.cross(b, c)).sum() / 6
    i, j, k, l = (torch.from_numpy(e) for e in edges)
    inner = l >= 0
    le = torch.linalg.norm(x[j] - x[i], dim=1)
    xi, xj, xk, xl = (x[t[inner]] for t in (i, j, k, l))
    n0, n1 = torch.linalg.cross(xk - xj, xi - xj), torch.linalg.cross(xl - xi, xj - xi)
    e = xj - xi
    th = torch.atan2((torch.linalg.cross(n0, n1) * e).sum(1) / le[inner], (n0 * n1).sum(1))
    lt = le[inner] * th / 4
    zero = torch.zeros(n, dtype=x.dtype)
    av = zero.index_add(0, ft.reshape(-1), af.repeat_interleave(3) / 3)
    cv = zero.index_add(0, i[inner], lt).index_add(0, j[inner], lt)
    if p["bond_type"] == 0:
        lc0, lc1, r = p["bond_lc0"], p["bond_lc1"], p["bond_r"]
        high, low = le > lc0, le < lc1
        short = le[low]
        w = torch.where(inner, 1.0, 0.5)    # a boundary edge is seen from one side only
        teth = (r ** (r + 1) * (le[high] - lc0) ** r * w[high]).sum() + \
            (torch.exp(short / (short - lc1)) / short ** r * w[low]).sum()
    else:
        teth = ((af / p["bond_a0"] - 1.0) ** 2).sum()
    d = torch.linalg.norm(x[pairs[:, 0]] - x[pairs[:, 1]], dim=1)
    rep = 2.0 * (torch.exp(d / (d - p["rep_lc1"])) / d ** p["rep_r"]).sum()
    return af.sum(), vol, 2.0 * lt.sum(), (2.0 * cv * cv / av).sum(), teth, rep


def exact(case, seed):
    """Energy and gradient in 64 bits: torch autograd over faces and edges.
    Chains and sweeps have no such value (each is a sequence of accept or
    reject decisions on the library's own random draws), nor has the network
    (its operands are bf16 by definition); on open meshes trimem's gradient
    is not the derivative at the rim."""
    if case["kind"] not in ("dropin", "device"):
        return None
    x0, x1, f, p = _inputs(case, seed)
    n = len(x0)
    edges = _edges(f, n)
    none = np.zeros((0, 2), dtype=np.int64)
    ref = _properties(torch.from_numpy(x0), f, edges, p, none)
    x = torch.from_numpy(x1).requires_grad_(True)
    pairs = _pairs(x1, f, n, p["rep_lc1"], p["rep_exclusion"])
    props = _properties(x, f, edges, p, pairs)
    energy = p["kappa_a"] * (props[0] / (p["area_frac"] * ref[0]) - 1.0) ** 2 + \
        p["kappa_v"] * (props[1] / (p["volume_frac"] * ref[1]) - 1.0) ** 2 + \
        p["kappa_c"] * (props[2] / (p["curvature_frac"] * ref[2]) - 1.0) ** 2 + \
        p["kappa_b"] * props[3] + p["kappa_t"] * props[4] + p["kappa_r"] * props[5]
    energy.backward()
    gradient = None if case["shape"] == "tube" else x.grad
    if case["kind"] == "dropin":
        return {"energy": float(energy.detach()), "gradient": gradient}
    return {"globals": torch.stack(props + (energy,)).detach(), "gradient": gradient}
