"""Performance cases of the framework: what its users have it compute, through its public entry
points, over the range of sizes, types and options that they use.

A case is a dict of plain values; ``kind`` says which stage it runs:

  refine   one refine step of the host loop: the system's Cmm and Ctm (matcov), then R
  matcov   the generator alone: a whole Cmm and Ctm
  tile     the generator on one tile of Cmm at any offset (tile-by-tile callers)
  solve    the reconstructor R = Ctm Cmm^-1 on matrices in hand, FP64 or FP32 storage
  mixed    the refined reconstructor (low-precision factorization, FP64 residuals)
  cee      Cee / Cvv of 1 .. 8 targets of an observation step
  psf      the intersample PSF of 1 .. 8 directions, FP32 or FP64 transforms

``prepare`` puts on the GPU what a caller has before the call, ``run`` makes one pass on a stream
of its own (in-place stages start from a device-to-device copy of their inputs, as a loop over
profiles does), ``exact`` computes the same outputs with plain torch and numpy in 64 bits.
Matrices are column-major: a torch buffer of shape (columns, ld) holds element (r, c) at [c, r].
"""
from __future__ import annotations

import ctypes
import functools
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from moao_amd import matcov as gm
from moao_amd import psf_inputs as pi
from moao_amd import systems
from moao_amd.lib import MOAO_MIXED_BF16, MOAO_MIXED_FP32, check, lib
from moao_amd.reconstructor import reconstructor_dev, reconstructor_mixed_dev
from moao_amd.tomo import Tomo

F64 = torch.float64
F32 = torch.float32
VP = ctypes.c_void_p


# ------------------------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest system of the tests and the check harness: launches and the serial
        # leaves are most of it (n = 456, m = 152)
        {"name": "refine_n456", "kind": "refine", "nlgs": 3, "nngs": 0, "nssp": 10, "nlayer": 2,
         "diam": 8.0, "ring": 60.0},
        # an ordinary request of the serving stream: 4 LGS + 2 NGS, 10 layers (n = 5,952)
        {"name": "refine_n6k", "kind": "refine", "nlgs": 4, "nngs": 2, "nssp": 26, "nlayer": 10,
         "diam": 39.0, "ring": 450.0},
        # a small solve of odd size on padded leading dimensions
        {"name": "solve_n2037", "kind": "solve", "n": 2037, "m": 385, "pad": 11, "fp32": False},
        # an ordinary solve (a size of the reconstructor's tests)
        {"name": "solve_n9000", "kind": "solve", "n": 9000, "m": 1500, "pad": 0, "fp32": False},
        # the headline configuration: 74 x 74 subapertures, 3 LGS + 2 NGS
        {"name": "solve_n39720", "kind": "solve", "n": 39720, "m": 7944, "pad": 0, "fp32": False},
        # FP32 storage, the precision of the asynchronous tiled driver
        {"name": "solve32_n18688", "kind": "solve", "n": 18688, "m": 2336, "pad": 0, "fp32": True},
        # the refined solve with split-BF16 updates (n = 9,632)
        {"name": "mixed_bf16_n10k", "kind": "mixed", "nlgs": 5, "nngs": 2, "nssp": 31,
         "bf16": True},
        # generator: 40 x 40 subapertures, 6 LGS + 2 NGS, 10 layers (n = 18,688, m = 2,336)
        {"name": "matcov_n18688", "kind": "matcov", "nlgs": 6, "nngs": 2, "nssp": 40,
         "nlayer": 10, "diam": 39.0, "ring": 450.0},
        # one tile of that system, as a tile-by-tile caller asks for it
        {"name": "tile_1000", "kind": "tile", "nlgs": 6, "nngs": 2, "nssp": 40, "nlayer": 10,
         "diam": 39.0, "ring": 450.0, "rows": 1000, "cols": 1000, "at": 0.71, "left": 0.13,
         "pad": 24},
        # an observation step's error covariances: 8 targets, an 80 x 80-actuator DM
        {"name": "cee_8x18688", "kind": "cee", "n": 18688, "m": 2336, "nact": 4724, "ngal": 8},
        # the observation step's PSFs: 8 directions, 2048 grid, FP32 transforms
        {"name": "psf_8x2048", "kind": "psf", "nssp": 79, "N": 2048, "batch": 8, "fp64": False,
         "diam": 39.0},
        # the reference's own PSF arithmetic on the smallest system: one direction, FP64
        {"name": "psf64_1x512", "kind": "psf", "nssp": 10, "N": 512, "batch": 1, "fp64": True,
         "diam": 8.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["refine", "solve", "solve32", "mixed", "matcov", "tile", "cee", "psf"])
    if kind == "refine":
        small = rng.random() < 0.4
        return {"kind": kind, "nlgs": rng.randint(1, 4), "nngs": rng.randint(0, 2),
                "nssp": _log(rng, 8, 24), "nlayer": rng.randint(1, 10),
                "diam": 8.0 if small else 39.0, "ring": 60.0 if small else 450.0}
    if kind in ("solve", "solve32"):
        n = _log(rng, 400, 16000)
        return {"kind": "solve", "n": n, "m": max(1, int(n * rng.uniform(0.08, 0.35))),
                "pad": rng.choice([0, 0, 3, 8, 17]), "fp32": kind == "solve32"}
    if kind == "mixed":
        return {"kind": kind, "nlgs": rng.randint(2, 5), "nngs": rng.randint(1, 3),
                "nssp": _log(rng, 15, 30), "bf16": rng.random() < 0.5}
    if kind in ("matcov", "tile"):
        c = {"kind": kind, "nlgs": rng.randint(1, 6), "nngs": rng.randint(0, 3),
             "nssp": _log(rng, 10, 40), "nlayer": rng.randint(1, 10), "diam": 39.0,
             "ring": 450.0}
        if kind == "tile":
            c.update(rows=_log(rng, 50, 2000), cols=_log(rng, 50, 2000), at=rng.random(),
                     left=rng.random(), pad=rng.choice([0, 1, 24]))
        return c
    if kind == "cee":
        n = _log(rng, 456, 12000)
        return {"kind": kind, "n": n, "m": max(1, int(n * rng.uniform(0.1, 0.33))),
                "nact": _log(rng, 100, 2500), "ngal": rng.randint(1, 8)}
    return {"kind": "psf", "nssp": _log(rng, 8, 79), "N": rng.choice([512, 1024, 2048]),
            "batch": rng.randint(1, 8), "fp64": rng.random() < 0.4, "diam": 39.0}


# ------------------------------------------------------------------- inputs: systems on disk

def _tomo(case, seed):
    """The seeded system of a case, written and read as users hold it (parameter files)."""
    spec = systems.SystemSpec(diam=case.get("diam", 39.0), nssp=case["nssp"], nlgs=case["nlgs"],
                              nngs=case["nngs"], nlayer=case.get("nlayer", 10),
                              lgs_ring_diam_as=case.get("ring", 450.0), seed=seed)
    d = tempfile.mkdtemp(prefix="moao_perf_")
    try:
        s, atms = systems.make_system(d, spec)
        t = Tomo(s, atms[0])
    finally:
        shutil.rmtree(d, ignore_errors=True)
    t.set_target(0)
    return t


# ---------------------------------------------------- inputs: covariance matrices in hand

def _measurements(nsub, seed, shift):
    """Slopes of sensors of nsub[w] subapertures on an annulus: positions (k, 2), axis (k,) and
    sensor (k,) of every measurement, x slopes of a sensor before its y slopes."""
    g = torch.Generator().manual_seed(seed)
    pos, axis, sensor = [], [], []
    for w, k in enumerate(nsub):
        r = 19.5 * torch.sqrt(0.0784 + 0.9216 * torch.rand(k, generator=g, dtype=F64))
        a = 2 * math.pi * torch.rand(k, generator=g, dtype=F64)
        p = torch.stack([r * torch.cos(a), r * torch.sin(a)], 1)
        p += shift * torch.rand(2, generator=g, dtype=F64)
        pos += [p, p]
        axis += [torch.zeros(k, dtype=torch.long), torch.ones(k, dtype=torch.long)]
        sensor += [torch.full((2 * k,), w)]
    return [torch.cat(v).cuda() for v in (pos, axis, sensor)]


def _slope_cov(out, a, b):
    """out[c, r] = covariance of slope r of ``a`` with slope c of ``b`` for a phase of covariance
    sum_k w_k exp(-d^2 / 2 l_k^2): large and small scales, as turbulence has."""
    (pa, ia, _), (pb, ib, _) = a, b
    rows = pa.shape[0]
    step = max(1, (1 << 26) // max(1, rows))
    for c0 in range(0, pb.shape[0], step):
        c1 = min(pb.shape[0], c0 + step)
        dx = pa[None, :, 0] - pb[c0:c1, None, 0]
        dy = pa[None, :, 1] - pb[c0:c1, None, 1]
        da = torch.where(ia[None, :] == 0, dx, dy)
        da *= torch.where(ib[c0:c1, None] == 0, dx, dy)
        r2 = dx.square_().add_(dy.square_())
        same = (ia[None, :] == ib[c0:c1, None]).to(F64)
        acc = torch.zeros_like(r2)
        for w, l in ((8.0, 6.0), (0.7, 1.6), (0.05, 0.5)):
            acc += (same - da / (l * l)) * torch.exp(r2 * (-0.5 / (l * l))) * (w / (l * l))
        out[c0:c1, :rows] = acc


def _covariances(n, m, nsub, nts, nlgs, seed, noise, ngal=1, cst=1.0):
    """Cmm (n x n, both triangles) and ngal Ctm (m x n) of such sensors: SPD, noise on the
    diagonal, the constant that LGS x and y slopes share on the first nlgs sensors."""
    meas = [v[:n] for v in _measurements(nsub, seed, 2.0)]
    C = torch.empty((n, n), dtype=F64, device="cuda")
    _slope_cov(C, meas, meas)
    if cst:
        tag = torch.where(meas[2] < nlgs, 2 * meas[2] + meas[1], -1 - torch.arange(n, device="cuda"))
        for c0 in range(0, n, 4096):
            C[c0:c0 + 4096] += cst * (tag[c0:c0 + 4096, None] == tag[None, :])
    C.diagonal().add_(noise)
    B = []
    for g in range(ngal):
        truth = [v[:m] for v in _measurements([nts], seed + 7919 * (g + 1), 2.0)]
        b = torch.empty((n, m), dtype=F64, device="cuda")
        _slope_cov(b, truth, meas)
        B.append(b)
    return C, B


def _even_sensors(n, m):
    """Subapertures per sensor for n measurements of 5 sensors (the last ones cut off at n)."""
    return [-(-n // 10)] * 5, -(-m // 2), 3


# ------------------------------------------------------------------------------- prepare

def _prepare_generator(case, seed, with_tile):
    t = _tomo(case, seed)
    n, m = t.nmeas(), t.nmeasts()
    st = {"tomo": t, "n": n, "m": m}
    if with_tile:
        rows, cols = min(case["rows"], n), min(case["cols"], n)
        st.update(rows=rows, cols=cols, x0=int(case["at"] * (n - rows)),
                  y0=int(case["left"] * (n - cols)))
        st["T"] = torch.zeros((cols, rows + case["pad"]), dtype=F64, device="cuda")
    else:
        st["Cmm"] = torch.zeros((n, n), dtype=F64, device="cuda")
        st["Ctm"] = torch.zeros((n, m), dtype=F64, device="cuda")
    return st


def _prepare_solve(case, seed):
    n, m, pad = case["n"], case["m"], case["pad"]
    nsub, nts, nlgs = _even_sensors(n, m)
    # FP32 storage holds definiteness only on well-conditioned matrices: faint sensors
    fp32 = case["fp32"]
    C, (B,) = _covariances(n, m, nsub, nts, nlgs, seed, 40.0 if fp32 else 0.02,
                           cst=0.0 if fp32 else 1.0)
    dt = F32 if fp32 else F64
    if pad:
        C = torch.nn.functional.pad(C, (0, pad))
        B = torch.nn.functional.pad(B, (0, pad))
    C, B = C.to(dt), B.to(dt)
    return {"Cmm0": C, "Ctm0": B, "Cmm": torch.empty_like(C), "Ctm": torch.empty_like(B)}


def _prepare_mixed(case, seed):
    t = _tomo(case, seed)
    n, m = t.nmeas(), t.nmeasts()
    nsub = [int(k) for k in t.field("Nsubap")]
    C, (B,) = _covariances(n, m, nsub[:-1], nsub[-1], case["nlgs"], seed, 0.1)
    return {"tomo": t, "n": n, "m": m, "Cmm": C, "Ctm0": B, "Ctm": torch.empty_like(B)}


def _prepare_cee(case, seed):
    n, m, nact, G = case["n"], case["m"], case["nact"], case["ngal"]
    nsub, nts, nlgs = _even_sensors(n, m)
    C, Bs = _covariances(n, m, nsub, nts, nlgs, seed, 0.05, ngal=G)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    Ctt = torch.empty((m, m), dtype=F64, device="cuda")
    truth = [v[:m] for v in _measurements([nts], seed + 7919, 2.0)]
    _slope_cov(Ctt, truth, truth)
    st = {"Cmm": C, "Cpp0": torch.stack([Ctt] * G), "Cpm0": torch.stack(Bs)}
    # a reconstructor in hand: each row averages the slopes measured near its subaperture
    meas = [v[:n] for v in _measurements(nsub, seed, 2.0)]
    R = []
    for g in range(G):
        truth = [v[:m] for v in _measurements([nts], seed + 7919 * (g + 1), 2.0)]
        d = torch.cdist(meas[0], truth[0])
        w = torch.exp(-0.5 * d * d) * (meas[1][:, None] == truth[1][None, :]) + 1e-4
        R.append(w / w.sum(0))
    st["R"] = torch.stack(R)
    st["Dx"] = torch.randn((m, nact), generator=gen, dtype=F64, device="cuda") / math.sqrt(n)
    for name, shape in (("Cpp", (G, m, m)), ("Cpm", (G, n, m)), ("Cee", (G, m, m)),
                        ("Cvv", (G, nact, nact)), ("Tmp", (G, m, nact))):
        st[name] = torch.empty(shape, dtype=F64, device="cuda")
    return st


@functools.lru_cache(maxsize=4)
def _optics(nssp, N, diam):
    dm = pi.make_dm(nssp)
    return dm, pi.make_idx(dm), pi.make_abs2fi(N, diam, dm), pi.make_otf_tel(N, diam, 0.28)


class _Stage:
    """The PSF stage a program keeps."""

    def __init__(self, idx, np_, N, a2f, otf, fp64):
        lp, dp = ctypes.POINTER(ctypes.c_long), ctypes.POINTER(ctypes.c_double)
        self.h = VP()
        check(lib().moao_hip_intersample_create(
            idx.size, np_, N, idx.ctypes.data_as(lp), a2f.ctypes.data_as(dp),
            otf.ctypes.data_as(dp), int(fp64), ctypes.byref(self.h)), "intersample_create")

    def __del__(self):
        if self.h:
            lib().moao_hip_intersample_destroy(self.h)


def _prepare_psf(case, seed):
    N, G = case["N"], case["batch"]
    dm, idx, a2f, otf = _optics(case["nssp"], N, case["diam"])
    # voltage covariances: correlated over a few actuators plus a random part, scaled to
    # residuals of about a radian
    dact = N // (3 * (dm.ndiam - 1)) + 1
    unit = 2 * (2 * 3.14159 / 1.65e-6) ** 2 / (float(N) * N * dact * dact) * float(a2f.sum())
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.from_numpy(dm.csI % dm.ndiam).cuda().to(F64)
    y = torch.from_numpy(dm.csI // dm.ndiam).cuda().to(F64)
    near = torch.exp(-((x[:, None] - x[None, :]) ** 2 + 0.3 * (y[:, None] - y[None, :]) ** 2) / 20)
    cvv = torch.empty((G, dm.nact, dm.nact), dtype=F64, device="cuda")
    for g in range(G):
        a = torch.randn((dm.nact, max(4, dm.nact // 4)), generator=gen, dtype=F64, device="cuda")
        cvv[g] = (0.4 + 0.1 * g) / unit * (a @ a.T) / a.shape[1] + 0.01 * (1 + g % 3) / unit * near
    return {"stage": _Stage(idx, dm.ndiam, N, a2f, otf, case["fp64"]), "cvv": cvv,
            "psf": torch.empty((G, N, N), dtype=F64, device="cuda")}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("refine", "matcov", "tile"):
        st = _prepare_generator(case, seed, kind == "tile")
    elif kind == "solve":
        st = _prepare_solve(case, seed)
    elif kind == "mixed":
        st = _prepare_mixed(case, seed)
    elif kind == "cee":
        st = _prepare_cee(case, seed)
    else:
        st = _prepare_psf(case, seed)
    st["case"] = case
    st["stream"] = torch.cuda.Stream()
    torch.cuda.synchronize()
    return st


# ----------------------------------------------------------------------------------- run

def _generate(st, h):
    t, n, m = st["tomo"], st["n"], st["m"]
    gm.matcov_tile_dev(st["Cmm"].data_ptr(), n, n, 0, 0, n, t, gm.CMM, h)
    gm.matcov_tile_dev(st["Ctm"].data_ptr(), m, n, 0, 0, m, t, gm.CTM, h)


def run(state):
    st, case, kind = state, state["case"], state["case"]["kind"]
    h = st["stream"].cuda_stream
    if kind == "refine":
        st["tomo"].set_target(0)
        _generate(st, h)
        info = reconstructor_dev(st["n"], st["m"], st["Cmm"].data_ptr(), st["n"],
                                 st["Ctm"].data_ptr(), st["m"], 1, h)
        return {"info": info, "L": st["Cmm"], "R": st["Ctm"]}
    if kind == "matcov":
        st["tomo"].set_target(0)
        _generate(st, h)
        return {"Cmm": st["Cmm"], "Ctm": st["Ctm"]}
    if kind == "tile":
        T = st["T"]
        gm.matcov_tile_dev(T.data_ptr(), st["rows"], st["cols"], st["x0"], st["y0"], T.shape[1],
                           st["tomo"], gm.CMM, h)
        return T
    if kind == "solve":
        C, B, n, m = st["Cmm"], st["Ctm"], case["n"], case["m"]
        with torch.cuda.stream(st["stream"]):
            C.copy_(st["Cmm0"])
            B.copy_(st["Ctm0"])
        if case["fp32"]:
            info = check(lib().moao_hip_sreconstructor_dev(
                n, m, VP(C.data_ptr()), C.shape[1], VP(B.data_ptr()), B.shape[1], 1, VP(h)),
                "moao_hip_sreconstructor_dev")
        else:
            info = reconstructor_dev(n, m, C.data_ptr(), C.shape[1], B.data_ptr(), B.shape[1], 1, h)
        return {"info": info, "L": C, "R": B}
    if kind == "mixed":
        with torch.cuda.stream(st["stream"]):
            st["Ctm"].copy_(st["Ctm0"])
        reconstructor_mixed_dev(st["n"], st["m"], st["Cmm"].data_ptr(), st["n"],
                                st["Ctm"].data_ptr(), st["m"], st["tomo"], 1e-12, 8, h,
                                mode=MOAO_MIXED_BF16 if case["bf16"] else MOAO_MIXED_FP32)
        return st["Ctm"]
    if kind == "cee":
        n, m, nact = case["n"], case["m"], case["nact"]
        with torch.cuda.stream(st["stream"]):
            st["Cpp"].copy_(st["Cpp0"])
            st["Cpm"].copy_(st["Cpm0"])
        p = {k: VP(st[k].data_ptr()) for k in ("Cmm", "Cpp", "Cpm", "R", "Dx", "Cee", "Cvv", "Tmp")}
        check(lib().moao_hip_cee_cvv_batched_dev(
            n, m, nact, case["ngal"], p["Cmm"], n, p["Cpp"], m, p["Cpm"], m, p["R"], m, p["Dx"],
            nact, p["Cee"], m, p["Cvv"], nact, p["Tmp"], nact, VP(h)),
            "moao_hip_cee_cvv_batched_dev")
        return {k: st[k] for k in ("Cpp", "Cpm", "Cee", "Cvv", "Tmp")}
    check(lib().moao_hip_intersample_process_dev(
        st["stage"].h, VP(st["cvv"].data_ptr()), case["batch"], VP(st["psf"].data_ptr()), VP(h)),
        "moao_hip_intersample_process_dev")
    if case["fp64"]:
        return st["psf"]
    with torch.cuda.stream(st["stream"]):  # FP32 transforms: the images are kept in FP32
        return st["psf"].to(F32)


# ---------------------------------------------------------------------------------- work

def _sizes(case):
    nv = systems.valid_subaps(case["nssp"], 0.28, case.get("diam", 39.0))
    return 2 * (case["nlgs"] + case["nngs"]) * nv, 2 * nv


def work(case):
    kind = case["kind"]
    if kind in ("refine", "matcov", "mixed"):
        n, m = _sizes(case)
    elif kind != "psf" and kind != "tile":
        n, m = case["n"], case["m"]
    if kind in ("refine", "solve", "mixed"):
        # Cholesky and two triangular solves (LAWN 41); the factor and R written, inputs read
        # (generated in place by a refine step)
        flops = n ** 3 / 3 + n * n / 2 + n / 6 + 2.0 * m * n * (n + 1)
        item = 4 if case.get("fp32") else 8
        cells = n * (n + 1) / 2 + m * n
        return {"bytes": item * cells * (1 if kind == "refine" else 2), "flops": flops}
    if kind == "matcov":
        return {"bytes": 8 * (n * (n + 1) / 2 + m * n), "flops": 0}
    if kind == "tile":
        n, _ = _sizes(case)
        rows, cols = min(case["rows"], n), min(case["cols"], n)
        x0, y0 = int(case["at"] * (n - rows)), int(case["left"] * (n - cols))
        cells = sum(max(0, min(rows, x0 + rows - (y0 + c))) for c in range(cols))
        return {"bytes": 8.0 * max(cells, 1), "flops": 0}
    if kind == "cee":
        a, G = case["nact"], case["ngal"]
        # dsyr2k and Cvv, Cee as symmetric results; R Cmm and Dx Cee in full
        flops = G * (2.0 * m * n * n + 3.0 * m * m * n + 2.0 * a * m * m + 1.0 * a * a * m)
        cells = n * n / 2 + a * m + G * (m * m * 1.5 + 2 * m * n + m * n + m * m + a * a + a * m)
        return {"bytes": 8.0 * cells, "flops": flops}
    N, G = case["N"], case["batch"]
    nact = pi.make_dm(case["nssp"]).nact
    item = 8 if case["fp64"] else 4
    # the covariance, its index list, the two filters and the images; three real transforms
    return {"bytes": G * (8.0 * nact * nact + 8.0 * N * N) + 4.0 * nact * nact + 2.0 * item * N * N,
            "flops": G * 3 * 2.5 * N * N * math.log2(N * N)}


# --------------------------------------------------------------------------------- exact

def _von_karman(x, y, L0):
    """Phase structure function of the reference's two-branch form, per layer scale L0."""
    ga = [0, 12.067619015983075, 5.17183672113560444, 0.795667187867016068, 0.0628158306210802181,
          0.00301515986981185091, 9.72632216068338833e-05, 2.25320204494595251e-06,
          3.93000356676612095e-08, 5.34694362825451923e-10, 5.83302941264329804e-12]
    gma = [-3.74878707653729304, -2.04479295083852408, -0.360845814853857083, -0.0313778969438136685,
           -0.001622994669507603, -5.56455315259749673e-05, -1.35720808599938951e-06,
           -2.47515152461894642e-08, -3.50257291219662472e-10, -3.95770950530691961e-12,
           -3.65327031259100284e-14]
    pi_ = 3.1415926535897932384626433
    q = (2 * pi_ / L0) * torch.sqrt(x * x + y * y)
    t, q53 = q * q / 4, q.pow(5 / 3)
    near, tn = torch.zeros_like(q), torch.full_like(q, 0.5)
    for k in range(11):
        near += (gma[k] * q53 + ga[k]) * tn
        tn = tn * t
    iq = 1 / q.clamp_min(1e-300)
    far = 1.00563491799858928388289314170833 - 1.25331413731550012081 * torch.exp(-q) * q.pow(1 / 3) \
        * (1 + iq * (0.22222222222222222222 + iq * (-0.08641975308641974829 + iq * 0.08001828989483310284)))
    return 0.1716613621245709486 * L0 ** (5 / 3) * torch.where(q > 0.75 * 2 * pi_, far, -near)


def _generator_exact(t, case, rows, cols, lower, truth_rows):
    """Covariances of measurements ``rows`` (of the truth sensor with truth_rows) with ``cols``,
    as a (cols, rows) tensor; zero above the diagonal with ``lower``."""
    f = {k: torch.from_numpy(t.field(k)).cuda()
         for k in ("u", "v", "sspSizeL", "L0", "cn2", "noiseNGS", "noiseLGSxx", "noiseLGSyy",
                   "noiseLGSxy")}
    nsub = [int(k) for k in t.field("Nsubap")]
    Nw, L, nlgs = len(nsub), int(f["L0"].numel()), case["nlgs"]
    Nx = sum(nsub)
    first = np.concatenate([[0], np.cumsum(nsub)])
    sens, axis, point = [], [], []
    for w in range(Nw):
        for a in (0, 1):
            sens.append(np.full(nsub[w], w))
            axis.append(np.full(nsub[w], a))
            point.append(first[w] + np.arange(nsub[w]))
    sens, axis, point = (torch.from_numpy(np.concatenate(v)).cuda() for v in (sens, axis, point))
    base = 2 * int(first[-2]) if truth_rows else 0
    ri = base + rows
    out = torch.zeros((cols.numel(), rows.numel()), dtype=F64, device="cuda")
    u, v = f["u"].reshape(L, Nx), f["v"].reshape(L, Nx)
    size = f["sspSizeL"].reshape(Nw, L)
    pitch = case.get("diam", 39.0) / case["nssp"]
    ax = axis[ri][None, :]
    ex, ey = (ax == 0).to(F64), (ax == 1).to(F64)
    step = max(1, (1 << 24) // max(1, rows.numel()))
    for c0 in range(0, cols.numel(), step):
        ci = cols[c0:c0 + step]
        bx = axis[ci][:, None]
        fx, fy = (bx == 0).to(F64), (bx == 1).to(F64)
        acc = torch.zeros((ci.numel(), rows.numel()), dtype=F64, device="cuda")
        for l in range(L):
            du = u[l, point[ri]][None, :] - u[l, point[ci]][:, None]
            dv = v[l, point[ri]][None, :] - v[l, point[ci]][:, None]
            s1 = 0.5 * size[sens[ri], l][None, :]
            s2 = 0.5 * size[sens[ci], l][:, None]
            L0 = float(f["L0"][l])
            # slopes are differences across a subaperture along its axis: four corners
            d = 0
            for p in (1, -1):
                for q in (1, -1):
                    d = d - p * q * _von_karman(du + p * s1 * ex - q * s2 * fx,
                                                dv + p * s1 * ey - q * s2 * fy, L0)
            acc += 0.5 * d * float(f["cn2"][l]) * ((s1 > 0) & (s2 > 0))
        acc *= 0.00026942094446267851 / (pitch * pitch)
        both = sens[ri][None, :] == sens[ci][:, None]
        here = both & (point[ri][None, :] == point[ci][:, None])
        same = ax == bx
        lgs = sens[ri][None, :] < nlgs
        pr = point[ri]
        noise = torch.where(ax == 0, f["noiseLGSxx"][pr][None, :], f["noiseLGSyy"][pr][None, :])
        acc += torch.where(here & lgs, torch.where(same, noise, f["noiseLGSxy"][pr][None, :]), 0.0)
        acc += (both & lgs & same) * 1.0
        ngs = f["noiseNGS"][(sens[ri] - nlgs).clamp_min(0)][None, :]
        acc += torch.where(here & ~lgs & same, ngs, 0.0)
        if lower:
            acc *= rows[None, :] >= ci[:, None]
        out[c0:c0 + step] = acc
    return out


def _solve_exact(C, B, n, m):
    """(factor over the lower part, R) on the host in 64 bits; C, B: (n, >= n), (n, >= m)."""
    S = C[:, :n].to(F64).cpu()
    S = torch.triu(S) + torch.triu(S, 1).T  # buffers are transposed: the lower part is triu here
    Lf = torch.linalg.cholesky(S)
    X = torch.cholesky_solve(B[:, :m].to(F64).cpu(), Lf)
    Lb, Rb = C.to(F64).cpu().clone(), B.to(F64).cpu().clone()
    low = torch.triu(torch.ones((n, n), dtype=torch.bool))
    Lb[:, :n] = torch.where(low, Lf.T, Lb[:, :n])
    Rb[:, :m] = X
    return Lb, Rb


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve" and case["n"] > 20000:
        return None
    if kind in ("refine", "matcov", "tile"):
        st = _prepare_generator(case, seed, kind == "tile")
        t, n, m = st["tomo"], st["n"], st["m"]
        every = torch.arange(n, device="cuda")
        if kind == "tile":
            T = st["T"]
            T[:, :st["rows"]] = _generator_exact(t, case, st["x0"] + every[:st["rows"]],
                                                 st["y0"] + every[:st["cols"]], True, False)
            return T
        C = _generator_exact(t, case, every, every, True, False)
        B = _generator_exact(t, case, every[:m], every, False, True)
        if kind == "matcov":
            return {"Cmm": C, "Ctm": B}
        Lb, Rb = _solve_exact(C, B, n, m)
        return {"info": None, "L": Lb, "R": Rb}
    if kind == "solve":
        st = _prepare_solve(case, seed)
        Lb, Rb = _solve_exact(st["Cmm0"], st["Ctm0"], case["n"], case["m"])
        return {"info": None, "L": Lb, "R": Rb}
    if kind == "mixed":
        st = _prepare_mixed(case, seed)
        return _solve_exact(st["Cmm"], st["Ctm0"], st["n"], st["m"])[1]
    if kind == "cee":
        st = _prepare_cee(case, seed)
        out = {k: [] for k in ("Cpp", "Cpm", "Cee", "Cvv", "Tmp")}
        D = st["Dx"].T  # nact x m
        for Cpp, B, R in zip(st["Cpp0"], st["Cpm0"], st["R"]):
            X = R.T @ B  # (m x m) buffer of Ctm R^T: [c, r]
            low = Cpp - X - X.T
            Cpm = st["Cmm"] @ R
            sym = torch.triu(low) + torch.triu(low, 1).T
            Cee = sym + R.T @ Cpm
            sym = torch.triu(Cee) + torch.triu(Cee, 1).T
            Tmp = sym @ D.T
            out["Cpp"].append(torch.where(torch.ones_like(low).triu() > 0, low, Cpp))
            out["Cpm"].append(Cpm)
            out["Cee"].append(Cee)
            out["Tmp"].append(Tmp)
            out["Cvv"].append(D @ Tmp)
        return {k: torch.stack(v) for k, v in out.items()}
    st = _prepare_psf(case, seed)
    N = case["N"]
    dm, idx, a2f, otf = _optics(case["nssp"], N, case["diam"])
    np_, h = dm.ndiam, N // 2 + 1
    dact, ncov = N // (3 * (np_ - 1)) + 1, 2 * np_ - 1
    at = torch.arange(ncov, device="cuda") * dact + N // 2 - (np_ - 1) * dact
    hits = torch.from_numpy(np.bincount(idx - 1, minlength=ncov * ncov)).cuda().clamp_min(1)
    bins = torch.from_numpy(idx - 1).cuda()
    w = torch.from_numpy(a2f).cuda().reshape(N, N).T[:, :h]
    tel = torch.from_numpy(otf).cuda().reshape(N, N)
    scale = 2 * (2 * 3.14159 / 1.65e-6) ** 2 / (float(N) * N * dact * dact)
    images = []
    for c in st["cvv"]:
        total = torch.zeros(ncov * ncov, dtype=F64, device="cuda").index_add_(0, bins, c.reshape(-1))
        grid = torch.zeros((N, N), dtype=F64, device="cuda")
        grid[at[:, None], at[None, :]] = (total / hits).reshape(ncov, ncov)
        d = torch.fft.irfft2(torch.fft.rfft2(grid).real * w + 0j, s=(N, N)) * (N * N) * scale
        d = torch.fft.fftshift(torch.exp(-0.5 * (d[N // 2, N // 2] - d)))
        s = (tel * d).T[:, :h]
        images.append(torch.fft.fftshift(torch.fft.irfft2(s + 0j, s=(N, N)) * (N * N)))
    return torch.stack(images)
