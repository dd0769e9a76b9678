"""The work that programs built on this framework have it do, as cases that can
be timed: hydro cycles of one mesh in every form of the cycle, whole decks,
ensembles, a mesh in pieces, the task entry points on a caller's own fields,
and training of the learned closure.

Kinds of a case:
  run     a mesh that a program holds mid-run advances by `cycles` cycles
          (Problem.run), and the program reads its state on the device
  deck    a deck from its text to its results: Problem, drive, get
  batch   `count` problems of uneven sizes advance together (Batch)
  pieces  one mesh as `numpcs` pieces (Pieces)
  abi     one cycle's task entry points in doCycle's order, on interleaved
          double2 fields that the caller allocated, on the caller's stream
  train   Adam steps of the closure network on captured-like tuples (Mlp)

Meshes mid-run: a state as a restart would load it, drawn from the seed (a
blast wave or a shock in a tube: hot gas behind a front, the gas ahead at
rest), with the steps held short by the deck's dtmax, so that every pass
works on a state of the same kind however often it is repeated.
"""
from __future__ import annotations

import ctypes
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "pennant-legion_amd"))

import pennant_amd as pa  # noqa: E402
from pennant_amd import decks  # noqa: E402
from pennant_amd.closure import NFEAT, Mlp  # noqa: E402
from pennant_amd.device import DeviceBuffer  # noqa: E402
from pennant_amd.train_closure import DEFAULT_OUT  # noqa: E402

MODES = {"tasks": pa.MODE_TASKS, "fused": pa.MODE_FUSED, "mixed": pa.MODE_MIXED, "learned": pa.MODE_LEARNED}
HELD_DT = 1.0e-7      # dtmax of the meshes held mid-run


def listed():
    return [
        # the smallest work: a deck of the reference's test size, from text to results
        dict(name="deck_sedov45", kind="deck", mesh="blast", nx=45, ny=45, mode="fused", cycles=100),
        # the drop-in path (one launch per task ID) on a small odd mesh: launches count
        dict(name="tasks_97x61", kind="run", mesh="blast", nx=97, ny=61, mode="tasks", cycles=20),
        # the drop-in path at the benchmark's size
        dict(name="tasks_sedov1440", kind="run", mesh="blast", nx=1440, ny=1440, mode="tasks", cycles=20),
        # a Legion wrapper's calls: the task entry points on its own double2 fields
        dict(name="abi_701x413", kind="abi", mesh="blast", nx=701, ny=413),
        # one mesh in pieces, triangles at the centre
        dict(name="pieces_noh640x480", kind="pieces", mesh="noh", nx=640, ny=480, mode="fused", numpcs=6, cycles=100),
        # the plain FP64 form at the benchmark's sizes, rect and pie
        dict(name="fused_sedov1440", kind="run", mesh="blast", nx=1440, ny=1440, mode="fused", cycles=20),
        dict(name="fused_noh1024", kind="run", mesh="noh", nx=1024, ny=1024, mode="fused", cycles=20),
        # an ordinary mesh of odd sizes in mixed precision, untuned
        dict(name="mixed_333x217", kind="run", mesh="blast", nx=333, ny=217, mode="mixed", cycles=50),
        # a long shock tube in mixed precision, autotuned as the benchmark does
        dict(name="mixed_leblanc", kind="run", mesh="tube", nx=4096, ny=256, mode="mixed", cycles=20, tuned=True),
        # the headline: learned closure and mixed precision, autotuned
        dict(name="learned_sedov1440", kind="run", mesh="blast", nx=1440, ny=1440, mode="learned", cycles=20,
             tuned=True),
        # an ensemble of uneven problems
        dict(name="batch_32", kind="batch", count=32, pick=20261202, mode="mixed", cycles=100),
        # training of the closure at the trainer's own batch size
        dict(name="train_8192", kind="train", tuples=200_000, batch=8192, steps=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """One more case: sizes over their logarithm, from the smallest listed to
    the largest."""
    kind = rng.choice(("deck", "run", "run", "run", "run", "abi", "pieces", "batch", "train"))
    if kind == "deck":
        n = _log_int(rng, 24, 180)
        return dict(kind=kind, mesh="blast", nx=n, ny=n, mode=rng.choice(("fused", "mixed")), cycles=100)
    if kind == "run":
        mesh = rng.choice(("blast", "noh", "tube"))
        zones = math.exp(rng.uniform(math.log(6.0e3), math.log(1.8e6)))
        aspect = math.exp(rng.uniform(math.log(0.25), math.log(4.0))) * (4.0 if mesh == "tube" else 1.0)
        nx = max(8, int(math.sqrt(zones * aspect)))
        ny = max(8, int(zones / nx))
        mode = rng.choice(("tasks", "fused", "fused", "mixed", "learned"))
        cycles = rng.choice((10, 20, 21, 32))
        return dict(kind=kind, mesh=mesh, nx=nx, ny=ny, mode=mode, cycles=cycles if zones * cycles < 4.0e7 else 20,
                    tuned=mode != "tasks" and rng.random() < 0.5)
    if kind == "abi":
        return dict(kind=kind, mesh="blast", nx=_log_int(rng, 100, 1400), ny=_log_int(rng, 100, 1400))
    if kind == "pieces":
        return dict(kind=kind, mesh="noh", nx=_log_int(rng, 100, 700), ny=_log_int(rng, 100, 700),
                    mode=rng.choice(("fused", "mixed")), numpcs=rng.randrange(2, 9), cycles=50)
    if kind == "batch":
        return dict(kind=kind, count=rng.randrange(8, 33), pick=rng.randrange(1 << 30),
                    mode=rng.choice(("fused", "mixed")), cycles=rng.choice((48, 64, 75, 100)))
    return dict(kind=kind, tuples=_log_int(rng, 20_000, 400_000), batch=_log_int(rng, 500, 16_384),
                steps=rng.choice((8, 15, 20)))


# -- decks and states ---------------------------------------------------------

def _lengths(case):
    if case["mesh"] == "tube":
        return 9.0, 0.5625
    if case["mesh"] == "noh":
        return 90.0, 1.0
    return 1.125, 1.125 * case["ny"] / case["nx"]


def _deck(case, seed):
    """The deck's text.  A deck run from its start draws its energy from the
    seed; a held mesh takes its state from _state."""
    rng = random.Random(seed)
    nx, ny = case["nx"], case["ny"]
    if case["mesh"] == "noh":
        text = decks.noh_pie(ny, nx, speed=rng.uniform(0.5, 2.0))
    elif case["mesh"] == "tube":
        text = decks.leblanc_rect(nx, ny)
    else:
        text = decks.sedov_rect(nx, energy=rng.uniform(0.1, 1.0),
                                cstop=case["cycles"] if case["kind"] == "deck" else None)
        lx, ly = _lengths(case)
        text = text.replace(f"meshparams {nx} {nx} {lx!r} {lx!r}", f"meshparams {nx} {ny} {lx!r} {ly!r}")
    return text if case["kind"] == "deck" else text + f"dtmax {HELD_DT!r}\n"


def _state(case, seed, px, zx):
    """Point velocities and zone energies of a mesh mid-run: a front (circular
    with a ripple for a blast, plane with one for a tube), behind it hot gas
    with a velocity rising to the front and falling to zero across a narrow
    band, ahead of it cold gas at rest."""
    rng = random.Random(seed)
    lx, ly = _lengths(case)
    speed, hot = rng.uniform(0.5, 1.5), rng.uniform(0.5, 2.0)
    wave, phase, ripple = rng.randrange(3, 9), rng.uniform(0, 6.28), 0.03
    front = rng.uniform(0.45, 0.65)

    def along(x):
        if case["mesh"] == "tube":
            return x[:, 0] / (lx * front * (1 + ripple * np.cos(wave * 6.28 * x[:, 1] / ly + phase)))
        r = np.hypot(x[:, 0], x[:, 1])
        theta = np.arctan2(x[:, 1], x[:, 0])
        return r / (min(lx, ly) * front * (1 + ripple * np.cos(2 * wave * theta + phase)))

    s = along(px)
    u = np.where(s < 1, s, np.clip((1.03 - s) / 0.03, 0, 1)) * speed
    if case["mesh"] == "tube":
        pu = np.stack([u, np.zeros_like(u)], axis=1)
    else:
        pu = px * (u / np.maximum(np.hypot(px[:, 0], px[:, 1]), 1e-30))[:, None]
    s = along(zx)
    ze = hot * np.where(s < 1, 1.6 - s * s, 0.6 * np.clip((1.02 - s) / 0.02, 0, 1)) + 1e-6
    return pu, ze


class _Buffer:
    """A device array of a problem as torch sees it; it keeps the problem,
    whose memory it is."""

    def __init__(self, problem, name, comp):
        n, _ = problem.field_info(name)
        self.problem = problem
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", version=2,
                                             data=(problem.device_ptr(name, comp), False))

    def tensor(self):
        t = torch.as_tensor(self, device="cuda")
        t.buffer = self
        return t


def _closure():
    return Mlp.load(DEFAULT_OUT)


def _ensemble(case, seed):
    """The decks of an ensemble: sizes from the case, energies and inflow
    speeds from the seed."""
    pick, rng = random.Random(case["pick"]), random.Random(seed)
    out = []
    for k in range(case["count"]):
        n = _log_int(pick, 32, 512)
        if k % 2 == 0:
            mesh, text = "blast", decks.sedov_rect(n, energy=rng.uniform(0.1, 1.0))
        else:
            mesh, text = "noh", decks.noh_pie(n, n, speed=rng.uniform(0.5, 2.0))
        out.append((dict(kind="batch", mesh=mesh, nx=n, ny=n), text + f"dtmax {HELD_DT!r}\n"))
    return out


# -- task entry points on a caller's fields -------------------------------------

POINT_VECS = ("px0", "pu0", "pxp", "pf", "pap", "pu", "px")
ZONE_VECS = ("zxp", "zuc")
SIDE_VECS = ("exp", "ssurfp", "sfp", "sfq", "sft", "cqe1", "cqe2")
ZONES = ("zareap", "zvolp", "zvol0", "zdl", "zm", "zr", "zrp", "ze", "zetot", "zw", "zwrate", "zp", "zss", "zdu",
         "ztmp")
SIDES = ("sareap", "svolp", "elen", "smf", "carea", "cevol", "cdu", "cdiv", "ccos", "crmu", "cw")


def _abi_prepare(case, seed):
    m, f = _initial(case, seed, torch.device("cuda"))
    dev = torch.device("cuda")
    maps = {k: m[k].to(torch.int32) for k in ("mapsp1", "mapsp2", "mapsz", "mapss3", "mapss4", "znump", "zsbeg",
                                              "pcbeg", "pcside")}
    mesh = pa.Mesh()
    mesh.nump, mesh.numz, mesh.nums, mesh.maxznump = m["nump"], m["numz"], m["nums"], 4
    for k, v in maps.items():
        setattr(mesh, k, v.data_ptr())
    d = {}
    for names, n, shape in ((POINT_VECS, m["nump"], (2,)), (ZONE_VECS, m["numz"], (2,)), (SIDE_VECS, m["nums"], (2,)),
                            (ZONES, m["numz"], ()), (SIDES, m["nums"], ()), (("pmaswt",), m["nump"], ())):
        for k in names:
            d[k] = torch.zeros((n,) + shape, dtype=torch.float64, device=dev)
    d["px0"].copy_(f["px"])
    d["pu0"].copy_(f["pu"])
    for k, v in (("zvol0", "zvol"), ("zm", "zm"), ("zr", "zr"), ("ze", "ze"), ("zetot", "zetot"), ("smf", "smf")):
        d[k].copy_(f[v])
    d["dt"] = torch.full((1,), HELD_DT, dtype=torch.float64, device=dev)
    d["dtnew"] = torch.zeros(1, dtype=torch.float64, device=dev)
    bad = torch.zeros(1, dtype=torch.int32, device=dev)
    ws = torch.zeros(int(pa.lib().pennant_hip_reduce_workspace_bytes()) // 8 + 1, dtype=torch.float64, device=dev)
    bcs = [(torch.nonzero(m["bits"] & (1 << i)).reshape(-1).to(torch.int32), v) for i, v in enumerate(m["planes"])]
    return dict(case=case, mesh=mesh, maps=maps, d=d, bad=bad, ws=ws, bcs=bcs, par=_params(case))


def _abi_run(st):
    """One cycle's tasks, src/Hydro.cc:342-983, as a wrapper calls them."""
    L, M, d, q = pa.lib(), ctypes.byref(st["mesh"]), st["d"], st["par"]
    s = torch.cuda.current_stream().cuda_stream
    p = {k: (pa.vec_interleaved(t.data_ptr()) if t.dim() == 2 else t.data_ptr()) for k, t in d.items()}

    def call(name, *args):
        rc = getattr(L, "pennant_hip_" + name)(*args, s)
        if rc:
            raise RuntimeError(f"{name}: {rc}")

    d["pmaswt"].zero_()
    d["pf"].zero_()
    call("adv_pos_half", M, p["px0"], p["pu0"], p["pxp"], p["dt"])
    call("calc_ctrs", M, p["pxp"], p["exp"], p["zxp"])
    call("calc_vols", M, p["pxp"], p["zxp"], p["sareap"], p["svolp"], p["zareap"], p["zvolp"], st["bad"].data_ptr(),
         st["ws"].data_ptr())
    call("calc_surf_vecs", M, p["exp"], p["zxp"], p["ssurfp"])
    call("calc_edge_len", M, p["pxp"], p["elen"])
    call("calc_char_len", M, p["sareap"], p["elen"], p["zdl"])
    call("calc_rho", M, p["zm"], p["zvolp"], p["zrp"])
    call("calc_crnr_mass", M, p["smf"], p["zrp"], p["zareap"], p["pmaswt"])
    call("calc_state_half", M, p["zr"], p["zvolp"], p["zvol0"], p["ze"], p["zwrate"], p["zm"], p["zp"], p["zss"],
         q["gamma"], q["ssmin"], p["dt"])
    call("calc_force_pgas", M, p["ssurfp"], p["zp"], p["sfp"])
    call("calc_force_tts", M, p["sareap"], p["smf"], p["ssurfp"], p["zareap"], p["zrp"], p["zss"], p["sft"],
         q["alfa"], q["ssmin"])
    call("set_corner_div", M, p["exp"], p["elen"], p["zxp"], p["pxp"], p["pu0"], p["zuc"], p["carea"], p["ccos"],
         p["cdiv"], p["cevol"], p["cdu"])
    call("set_qcn_force", M, p["elen"], p["cdiv"], p["cdu"], p["cevol"], p["zrp"], p["zss"], p["pu0"], p["crmu"],
         p["cqe1"], p["cqe2"], q["qgamma"], q["q1"], q["q2"])
    call("set_force_qcs", M, p["carea"], p["cqe1"], p["cqe2"], p["elen"], p["ccos"], p["cw"], p["sfq"])
    call("set_vel_diff", M, p["elen"], p["zss"], p["pxp"], p["pu0"], p["ztmp"], p["zdu"], q["q1"], q["q2"])
    call("sum_crnr_force", M, p["sfp"], p["sfq"], p["sft"], p["pf"])
    for pts, (vx, vy) in st["bcs"]:
        call("apply_fixed_bc", pts.data_ptr(), pts.numel(), vx, vy, p["pf"], p["pu0"])
    call("calc_accel", M, p["pf"], p["pmaswt"], p["pap"])
    call("adv_pos_full", M, p["px0"], p["pu0"], p["pap"], p["px"], p["pu"], p["dt"])
    call("calc_work", M, p["sfp"], p["sfq"], p["pu"], p["pu0"], p["pxp"], p["zw"], p["zetot"], p["dt"])
    call("calc_dt_new", M, p["zdl"], p["zdu"], p["zss"], q["cfl"], p["dtnew"], st["ws"].data_ptr())
    return {k: d[k] for k in ABI_OUT}


ABI_OUT = ("px", "pu", "pf", "pmaswt", "zdl", "zp", "zdu", "zw", "zetot", "sfq", "sft", "crmu", "dtnew")


# -- the four functions ---------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "deck":
        return dict(case=case, text=_deck(case, seed))
    if kind == "abi":
        return _abi_prepare(case, seed)
    if kind == "batch":
        return dict(case=case, batch=pa.Batch([t for _, t in _ensemble(case, seed)]))
    if kind == "pieces":
        return dict(case=case, pieces=pa.Pieces(_deck(case, seed), case["numpcs"]))
    if kind == "train":
        # feature distribution of captured tuples: slog of velocity ratios within
        # a few units, two ratios in (0, 1], the compression ratio near 1
        g = torch.Generator(device="cuda").manual_seed(seed)
        n = case["tuples"]
        t = torch.randn((n, NFEAT + 2), generator=g, device="cuda")
        t[:, 5:8] = 1.0 - 0.4 * torch.rand((n, 3), generator=g, device="cuda")
        t[:, 9] = torch.rand(n, generator=g, device="cuda").clamp_min(1e-3)
        f9 = t[:, 9].double()
        size = torch.sqrt((1 - f9) ** 2 + f9 ** 2)
        t[:, 10] = ((1 - f9) / size).float()
        t[:, 11] = (1 + f9 / size).float()
        return dict(case=case, mlp=Mlp(seed % 1000), tuples=DeviceBuffer.from_host(t.cpu().numpy()))
    pb = pa.Problem(_deck(case, seed))
    if case["mesh"] != "noh":
        zm = pb.get("zm")
        pu, ze = _state(case, seed, pb.get("px"), _zone_centres(case))
        pb.set("pu", pu)
        pb.set("ze", ze)
        pb.set("zetot", ze * zm)
    state = dict(case=case, problem=pb)
    if case["mode"] == "learned":
        state["closure"] = _closure()
        pb.set_closure(state["closure"])
    if case.get("tuned"):
        pb.autotune(MODES[case["mode"]])
    out = {}
    for name in ("px", "pu", "zetot", "zwrate", "zvol", "zp"):
        comps = pb.field_info(name)[1]
        for c in range(comps):
            out[name + ("xy"[c] if comps == 2 else "")] = _Buffer(pb, name, c).tensor()
    state["out"] = out
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "deck":
        with pa.Problem(state["text"]) as pb:
            pb.drive(MODES[case["mode"]])
            out = {k: pb.get(k) for k in ("px", "pu", "zr", "ze", "zp")}
            out["time"] = np.array([pb.scalars()["time"]])
        return out
    if kind == "abi":
        return _abi_run(state)
    if kind == "batch":
        b = state["batch"]
        b.run(case["cycles"], MODES[case["mode"]])
        return [[b.get(i, k) for k in ("zetot", "zp")] for i in range(b.count)]
    if kind == "pieces":
        pp = state["pieces"]
        pp.run(case["cycles"], MODES[case["mode"]])
        return {k: pp.get(k) for k in ("pu", "zetot", "zp")}
    if kind == "train":
        m = state["mlp"]
        losses = m.train(state["tuples"], case["steps"], batch=case["batch"], lr=2e-3, seed=1)
        return {"losses": losses, "params": m.get_params()}
    state["problem"].run(case["cycles"], MODES[case["mode"]])
    return state["out"]


def _counts(case):
    nx, ny = case["nx"], case["ny"]
    if case["mesh"] == "noh":
        return nx * ny, (nx + 1) * ny + 1, 3 * nx + 4 * nx * (ny - 1)
    return nx * ny, (nx + 1) * (ny + 1), 4 * nx * ny


def work(case):
    """Bytes and flops of a pass.  A fused cycle reads a mesh's state (px, pu;
    zm, zr, ze, zetot, zwrate, zvol; the side fractions) and writes it (px,
    pu; zr, ze, zetot, zwrate, zvol, zp) once; the mixed forms derive zr and
    ze and hold the side fractions in FP32.  The task form moves every task's
    own fields (688 bytes a side, 536 a zone, 512 a point, a cycle).  Flops
    of a cycle: about 280 a side.  Training: the network's three products,
    forward and twice over backward, on every row of every minibatch."""
    kind = case["kind"]
    if kind == "train":
        rows = case["steps"] * case["batch"]
        return {"bytes": 48 * rows, "flops": 6 * rows * (16 * 64 + 64 * 64 + 64 * 2)}
    meshes = [c for c, _ in _ensemble(case, 0)] if kind == "batch" else [case]
    cycles = case.get("cycles", 1)
    total, flops = 0, 0
    for c in meshes:
        z, p, s = _counts(c)
        if kind == "abi" or case["mode"] == "tasks":
            total += 688 * s + 536 * z + 512 * p
        elif case["mode"] == "fused":
            total += 64 * p + 96 * z + 8 * s
        else:
            total += 64 * p + 64 * z + 4 * s
        flops += 280 * s
    return {"bytes": total * cycles, "flops": flops * cycles}


# -- the same results in 64 bits, from plain torch --------------------------------

def _params(case):
    blast = dict(gamma=5 / 3, qgamma=5 / 3, ssmin=0.1, alfa=0.5, q1=0.1, q2=1.0, cfl=0.6, cflv=0.1, dtfac=1.2)
    if case["mesh"] == "noh":
        return dict(blast, q1=1.0)
    return dict(blast, q1=0.3, q2=2.0) if case["mesh"] == "tube" else blast


def _zone_points(case):
    """Corner points of every zone as the generator numbers them, counter-
    clockwise, -1 where a triangle has no fourth."""
    nx, ny, npx = case["nx"], case["ny"], case["nx"] + 1
    i, j = np.meshgrid(np.arange(nx), np.arange(ny))
    if case["mesh"] != "noh":
        p0 = j * npx + i
        return np.stack([p0, p0 + 1, p0 + 1 + npx, p0 + npx], axis=2).reshape(-1, 4)
    p0 = (j - 1) * npx + i + 1
    c = np.stack([p0, p0 + 1, p0 + 1 + npx, p0 + npx], axis=2)
    k = np.arange(nx) + 1
    c[0] = np.stack([np.zeros(nx, dtype=c.dtype), k + 1, k, np.full(nx, -1)], axis=1)
    return c.reshape(-1, 4)


def _points(case):
    nx, ny = case["nx"], case["ny"]
    lx, ly = _lengths(case)
    if case["mesh"] != "noh":
        x, y = np.meshgrid(lx / nx * np.arange(nx + 1), ly / ny * np.arange(ny + 1))
        return np.stack([x, y], axis=2).reshape(-1, 2)
    dth = math.radians(lx) / nx
    th, r = np.meshgrid(dth * (nx - np.arange(nx + 1)), ly / ny * np.arange(1, ny + 1))
    p = np.stack([r * np.cos(th), r * np.sin(th)], axis=2).reshape(-1, 2)
    return np.concatenate([np.zeros((1, 2)), p])


def _zone_centres(case):
    c, px = _zone_points(case), _points(case)
    have = c >= 0
    x = np.where(have[:, :, None], px[np.maximum(c, 0)], 0.0)
    return x.sum(axis=1) / have.sum(axis=1)[:, None]


def _initial(case, seed, dev):
    """Maps and initial fields of a case's mesh."""
    c = _zone_points(case)
    have = c >= 0
    znump = have.sum(axis=1)
    p1 = c[have]
    beg = np.concatenate([[0], np.cumsum(znump)])
    numz, nums = len(znump), len(p1)
    mapsz = np.repeat(np.arange(numz), znump)
    k = np.arange(nums) - beg[mapsz]
    s3 = np.where(k == 0, beg[mapsz + 1] - 1, np.arange(nums) - 1)
    s4 = np.where(k + 1 == znump[mapsz], beg[mapsz], np.arange(nums) + 1)
    px = _points(case)
    order = np.argsort(p1, kind="stable")
    pcbeg = np.concatenate([[0], np.cumsum(np.bincount(p1, minlength=len(px)))])
    lx, ly = _lengths(case)
    planes = [(0, 0.0)] if case["mesh"] != "tube" else [(0, 0.0), (0, lx)]
    planes += [(1, 0.0)] if case["mesh"] != "tube" else [(1, 0.0), (1, ly)]
    bits = np.zeros(len(px), dtype=np.int32)
    for i, (axis, at) in enumerate(planes):
        bits |= (np.abs(px[:, axis] - at) < 1e-12).astype(np.int32) << i
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    m = dict(nump=len(px), numz=numz, nums=nums, mapsp1=t(p1), mapsp2=t(p1[s4]), mapsz=t(mapsz), mapss3=t(s3),
             mapss4=t(s4), znump=t(znump), zsbeg=t(beg), pcbeg=t(pcbeg), pcside=t(order), bits=t(bits),
             planes=[(1.0, 0.0) if axis == 0 else (0.0, 1.0) for axis, _ in planes])
    f = dict(px=t(px))
    ex, zx = _centres(m, f["px"])
    sarea, svol, zarea, zvol = _volumes(m, f["px"], zx)
    f["smf"] = sarea / zarea[m["mapsz"]]
    f["zvol"] = zvol
    zr = np.ones(numz)
    text = {ln.split()[0]: ln.split()[1:] for ln in _deck(case, seed).splitlines() if ln.split()} \
        if case["kind"] != "batch" else {ln.split()[0]: ln.split()[1:] for ln in case["text"].splitlines()
                                         if ln.split()}
    ze = np.full(numz, float(text["einit"][0]))
    if "subregion" in text:
        b, zc, eps = [float(v) for v in text["subregion"]], zx.cpu().numpy(), 1e-12
        inside = ((zc[:, 0] > b[0] - eps) & (zc[:, 0] < b[1] + eps) & (zc[:, 1] > b[2] - eps)
                  & (zc[:, 1] < b[3] + eps))
        zr[inside], ze[inside] = float(text["rinitsub"][0]), float(text["einitsub"][0])
    pu = np.zeros_like(px)
    if "uinitradial" in text:
        r = np.hypot(px[:, 0], px[:, 1])
        pu = np.where((r > 1e-12)[:, None], float(text["uinitradial"][0]) * px / np.maximum(r, 1e-30)[:, None], 0.0)
    if case["kind"] in ("run", "abi") and case["mesh"] != "noh":
        pu, ze = _state(case, seed, px, _zone_centres(case))
    f["zr"], f["ze"], f["pu"] = t(zr), t(ze), t(pu)
    f["zm"] = f["zr"] * zvol
    f["zetot"] = f["ze"] * f["zm"]
    f["zwrate"] = torch.zeros_like(zvol)
    f["dtinit"] = float(text.get("dtinit", [1e99])[0])
    f["dtmax"] = float(text.get("dtmax", [1e99])[0])
    return m, f


def _cross(a, b):
    return a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]


def _dot(a, b):
    return (a * b).sum(dim=1)


def _zone_sum(m, v):
    out = torch.zeros((m["numz"],) + v.shape[1:], dtype=v.dtype, device=v.device)
    return out.index_add_(0, m["mapsz"], v)


def _zone_fold(m, v, start, how):
    out = torch.full((m["numz"],), start, dtype=v.dtype, device=v.device)
    return out.scatter_reduce_(0, m["mapsz"], v, how)


def _point_sum(m, v):
    out = torch.zeros((m["nump"],) + v.shape[1:], dtype=v.dtype, device=v.device)
    return out.index_add_(0, m["mapsp1"], v)


def _centres(m, px):
    p1 = px[m["mapsp1"]]
    return 0.5 * (p1 + px[m["mapsp2"]]), _zone_sum(m, p1) / m["znump"][:, None]


def _volumes(m, px, zx):
    p1, p2, c = px[m["mapsp1"]], px[m["mapsp2"]], zx[m["mapsz"]]
    sarea = 0.5 * _cross(p2 - p1, c - p1)
    svol = sarea * (p1[:, 0] + p2[:, 0] + c[:, 0]) / 3
    return sarea, svol, _zone_sum(m, sarea), _zone_sum(m, svol)


def _cycle(m, f, q, dt):
    """One cycle of the staggered-grid scheme (src/Hydro.cc:342-983) on the
    fields f, in 64 bits; returns every value that a case hands out."""
    z, p1, p2, s3, s4 = (m[k] for k in ("mapsz", "mapsp1", "mapsp2", "mapss3", "mapss4"))
    pu0 = f["pu"]
    pxp = f["px"] + 0.5 * dt * pu0
    ex, zx = _centres(m, pxp)
    sarea, svol, zarea, zvolp = _volumes(m, pxp, zx)
    c = zx[z]
    ss = ex - c
    ss = torch.stack([-ss[:, 1], ss[:, 0]], dim=1)
    edge = pxp[p2] - pxp[p1]
    elen = torch.sqrt(_dot(edge, edge))
    fac = torch.where(m["znump"] == 3, 3.0, 4.0)[z]
    zdl = _zone_fold(m, fac * sarea / elen, 1e99, "amin")
    zrp = f["zm"] / zvolp
    mass = (zrp * zarea)[z] * 0.5 * (f["smf"] + f["smf"][s3])
    pmaswt = _point_sum(m, mass)
    # the gas at the half step
    gm1, r, e = q["gamma"] - 1, f["zr"], f["ze"].clamp_min(0)
    csq = (gm1 * e + gm1 * gm1 * e).clamp_min(max(q["ssmin"] ** 2, 1e-99))
    zss = torch.sqrt(csq)
    dv = (zvolp - f["zvol"]) / f["zm"]
    zp = gm1 * r * e + (gm1 * r * f["zwrate"] * 0.5 * dt / f["zm"] - r * r * csq * dv) / (1 + 0.5 * gm1 * r * dv)
    sfp = -zp[z][:, None] * ss
    stiff = q["alfa"] * zss.clamp_min(q["ssmin"]) ** 2
    sft = -(stiff[z] * (zrp[z] * f["smf"] * zarea[z] / sarea - zrp[z]))[:, None] * ss
    # the tensor viscosity
    zuc = _zone_sum(m, pu0[p1]) / m["znump"][:, None]
    u0, x0, x1, x3 = pu0[p1], pxp[p1], ex, ex[s3]
    u1, u2, u3 = 0.5 * (u0 + pu0[p2]), zuc[z], 0.5 * (pu0[p1[s3]] + u0)
    carea = 0.5 * _cross(c - x0, x3 - x1)
    de1, de2 = elen[s3], elen
    low = torch.minimum(de1, de2)
    ccos = torch.where(low < 1e-12, 0.0, 4 * _dot(x3 - x0, x1 - x0) / (de1 * de2))
    cdiv = (_cross(u2 - u0, x3 - x1) - _cross(u3 - u1, c - x0)) / (2 * carea)
    a1, a2 = 0.5 * (x1 + c - x0 - x3), 0.5 * (c + x3 - x0 - x1)
    d1, d2 = torch.sqrt(_dot(a1, a1)), torch.sqrt(_dot(a2, a2))
    mean = 0.25 * (u0 + u1 + u2 + u3)
    first = (_dot(a1, mean) * d2).abs() > (_dot(a2, mean) * d1).abs()
    ratio = torch.where(first, d1 / d2, d2 / d1)
    squeezed = cdiv < 0
    cevol = torch.where(squeezed, torch.minimum(torch.sqrt((4 * carea * ratio).clamp_min(0)), 2 * low), 0.0)
    v1, v2 = u1 + u2 - u0 - u3, u2 + u3 - u0 - u1
    cdu = torch.where(squeezed, torch.sqrt(torch.maximum(_dot(v1, v1), _dot(v2, v2))), 0.0)
    t2, t1 = q["q2"] * 0.25 * (q["qgamma"] + 1) * cdu, q["q1"] * zss[z]
    crmu = torch.where(cdiv > 0, 0.0, (t2 + torch.sqrt(t2 * t2 + t1 * t1)) * zrp[z] * cevol)
    cqe1 = (crmu / de1)[:, None] * (u0 - pu0[p1[s3]])
    cqe2 = (crmu / de2)[:, None] * (pu0[p2] - u0)
    sin2 = 1 - ccos * ccos
    flat = sin2 < 1e-4
    cw, ccos = torch.where(flat, 0.0, carea / sin2)[:, None], torch.where(flat, 0.0, ccos)[:, None]
    sfq = (cw * (cqe2 + ccos * cqe1) + cw[s4] * (cqe1[s4] + ccos[s4] * cqe2[s4])) / elen[:, None]
    jump = torch.where(elen > 0, _dot(pu0[p2] - pu0[p1], edge).abs() / elen, 0.0)
    zdu = q["q1"] * zss + 2 * q["q2"] * _zone_fold(m, jump, 0.0, "amax")
    # points
    tot = sfp + sfq + sft
    pf = _point_sum(m, tot - tot[s3])
    pu0 = pu0.clone()
    for i, (vx, vy) in enumerate(m["planes"]):
        on = ((m["bits"] >> i) & 1).to(pf.dtype)[:, None]
        v = torch.tensor([vx, vy], dtype=pf.dtype, device=pf.device)
        pf = pf - on * _dot(pf, v.expand_as(pf))[:, None] * v
        pu0 = pu0 - on * _dot(pu0, v.expand_as(pu0))[:, None] * v
    pu = pu0 + dt * pf / pmaswt.clamp_min(1e-99)[:, None]
    px = f["px"] + 0.5 * dt * (pu0 + pu)
    # corrector
    _, zxn = _centres(m, px)
    _, _, _, zvol = _volumes(m, px, zxn)
    vs, w = pu0 + pu, pxp[:, 0]
    dwork = -0.5 * dt * (_dot(sfp + sfq, vs[p1]) * w[p1] - _dot(sfp + sfq, vs[p2]) * w[p2])
    zw = _zone_sum(m, dwork)
    zetot = f["zetot"] + zw
    new = dict(f, px=px, pu=pu, zvol=zvol, zetot=zetot, zp=zp, zwrate=(zw + zp * (zvol - f["zvol"])) / dt,
               ze=zetot / (f["zm"] + 1e-99), zr=f["zm"] / zvol)
    dtnew = float((zdl * q["cfl"] / torch.maximum(zdu, zss.clamp_min(1e-99))).min().clamp_max(1e99))
    grown = max(1e-99, float(((zvol - f["zvol"]) / f["zvol"]).abs().max()))
    extra = dict(pf=pf, pmaswt=pmaswt, zdl=zdl, zdu=zdu, zw=zw, sfq=sfq, sft=sft, crmu=crmu,
                 dtnew=torch.tensor([dtnew], dtype=torch.float64))
    return new, min(dtnew, dt * q["cflv"] / grown), extra


def _march(case, seed, cycles, tstop):
    m, f = _initial(case, seed, torch.device("cuda" if torch.cuda.is_available() else "cpu"))
    q, time, dt, limit = _params(case), 0.0, 0.0, 1e99
    for k in range(cycles):
        dt = min(f["dtmax"], f["dtinit"] if k == 0 else q["dtfac"] * dt, tstop - time, limit)
        f, limit, _ = _cycle(m, f, q, dt)
        time += dt
        if time >= tstop:
            break
    return f, time


def exact(case, seed):
    kind = case["kind"]
    if kind == "train" or case.get("mode") == "learned":
        return None           # a network in BF16 has no 64-bit value of its own
    if kind == "abi":
        m, f = _initial(case, seed, torch.device("cuda" if torch.cuda.is_available() else "cpu"))
        new, _, extra = _cycle(m, f, _params(case), HELD_DT)
        return {k: extra.get(k, new.get(k)) for k in ABI_OUT}
    if kind == "batch":
        out = []
        for c, text in _ensemble(case, seed):
            f, _ = _march(dict(c, text=text), seed, case["cycles"], 1.0 if c["mesh"] == "blast" else 0.6)
            out.append([f["zetot"], f["zp"]])
        return out
    f, time = _march(case, seed, case["cycles"], {"noh": 0.6, "tube": 6.0}.get(case["mesh"], 1.0))
    if kind == "deck":
        return dict({k: f[k] for k in ("px", "pu", "zr", "ze", "zp")}, time=np.array([time]))
    if kind == "pieces":
        return {k: f[k] for k in ("pu", "zetot", "zp")}
    out = {}
    for k in ("px", "pu"):
        out[k + "x"], out[k + "y"] = f[k][:, 0].contiguous(), f[k][:, 1].contiguous()
    return dict(out, **{k: f[k] for k in ("zetot", "zwrate", "zvol", "zp")})
