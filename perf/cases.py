"""Workloads of the framework through its public entry points.

Each case is one call that a search program makes: a period / acceleration / jerk search on
resident series, a fold returned to the caller, a Fourier-domain search, a batch of uneven
series, a one-shot host call, the candidate refinement's forward and backward pass, and the
pruning seeds.  The listed sizes are those of the benchmark's workloads and of the tests, plus
smaller and ragged ones; ``draw`` spreads over the same ranges.

``exact`` restates the whole path in 64 bits with plain torch: the cell-centred grids and shift
tables, the phase-binned or DFT level 0, the tree merges and the boxcar S/N.
"""

from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

import loki_amd
from loki_amd import libculoki, libloki, refine

TSAMP = 64e-6
C_LIGHT = 299792458.0
INV_C = 3.3356409519815204e-09
BOXCARS = (1, 2, 3, 4, 6, 8, 12, 16, 24, 32)
DEVICE = "cuda:0"
# Fourier searches with more bins than this start from a binned level 0 (the default config's)
LOSSY_ABOVE = 64

# largest number of final trials, and of stored or level-0 values, a drawn case may have
MAX_TRIALS = 60_000_000
MAX_VALUES = 1_500_000_000


def listed() -> list[dict]:
    return [
        # The smallest search: a slow-pulsar period search of 8 s of data, a few launches.
        dict(name="period_short", kind="search", domain="time", nsamps=2**17, nbins=32,
             f_lo=2.0, f_hi=10.0, accel=0.0, jerk=0.0, storage="f32", best=False),
        # An ordinary period search (0.5-2 s periods, 67 s of data): long level-0 segments.
        dict(name="period_long_segments", kind="search", domain="time", nsamps=2**20, nbins=64,
             f_lo=0.5, f_hi=2.0, accel=0.0, jerk=0.0, storage="f32", best=False),
        # A moderate acceleration search with fine bins that keeps each trial's best width.
        dict(name="accel_fine_bins", kind="search", domain="time", nsamps=2**20, nbins=64,
             f_lo=40.0, f_hi=120.0, accel=30.0, jerk=0.0, storage="f32", best=True),
        # The headline acceleration search: 9 minutes of data, 100-400 Hz, every width's S/N.
        dict(name="accel_headline", kind="search", domain="time", nsamps=2**23, nbins=32,
             f_lo=100.0, f_hi=400.0, accel=50.0, jerk=0.0, storage="f32", best=False),
        # The jerk search with block floating-point fold storage.
        dict(name="jerk_bfp16", kind="search", domain="time", nsamps=2**22, nbins=32,
             f_lo=50.0, f_hi=300.0, accel=30.0, jerk=2.0, storage="bfp16", best=False),
        # A ragged number of bins, the final folds returned (a caller that prunes or plots).
        dict(name="accel_fold_ragged", kind="fold", domain="time", nsamps=2**19, nbins=50,
             f_lo=60.0, f_hi=130.0, accel=40.0, jerk=0.0, storage="f32"),
        # The Fourier-domain search over (fddot, fdot, f), the benchmark's grid.
        dict(name="fourier_search", kind="search", domain="fourier", nsamps=2**22, nbins=64,
             f_lo=50.0, f_hi=500.0, accel=C_LIGHT * 1e-8 / 50.0, jerk=C_LIGHT * 1e-14 / 50.0,
             storage="f32", best=False),
        # Fourier folds returned as harmonics, a ragged number of bins, an acceleration range.
        dict(name="fourier_fold_ragged", kind="fold", domain="fourier", nsamps=2**19, nbins=50,
             f_lo=30.0, f_hi=90.0, accel=25.0, jerk=0.0, storage="f32"),
        # Many independent period searches of uneven length in one batch.
        dict(name="batch_uneven", kind="batch", nseries=24, grid_seed=7000, lo=18, hi=21),
        # The one-shot host call of a search script: host series in, host scores out, the
        # Fourier domain (the default), plan and buffers made by the call.
        dict(name="search_call", kind="call", domain="fourier", nsamps=2**18, nbins=64,
             f_lo=20.0, f_hi=60.0, accel=20.0, jerk=0.0),
        # Candidate refinement: S/N and its gradient in (f, fdot, fddot).
        dict(name="refine_candidates", kind="refine", nsamps=2**20, ncand=384, nbins=64,
             width=4, f_lo=50.0, f_hi=500.0),
        # Pruning seeds over the rows of a final level, time and Fourier domain.
        dict(name="pruning_seeds", kind="seeds", nbins=64, nleaves=2**19, segments=8,
             rows=2**15),
    ]


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    kind = rng.choice(["period", "accel", "accel", "jerk", "fourier", "fold", "fourier_fold",
                       "batch", "call", "refine", "seeds"])
    if kind == "batch":
        return dict(kind="batch", nseries=rng.randint(3, 24), grid_seed=rng.randint(0, 10**6),
                    lo=17, hi=rng.randint(18, 21))
    if kind == "refine":
        nsamps = int(_log(rng, 2**15, 2**20))
        return dict(kind="refine", nsamps=nsamps, ncand=int(_log(rng, 8, 384)),
                    nbins=rng.choice([16, 32, 64, 128]) if nsamps < 2**19 else 32,
                    width=rng.randint(1, 8), f_lo=50.0, f_hi=500.0)
    if kind == "seeds":
        return dict(kind="seeds", nbins=rng.choice([32, 50, 63, 64, 128]),
                    nleaves=int(_log(rng, 2**10, 2**18)), segments=rng.randint(1, 8),
                    rows=int(_log(rng, 2**8, 2**14)))
    for _ in range(1000):
        case = _draw_search(rng, kind)
        if _drawable(case):
            return case
    raise RuntimeError("no drawable case")


def _draw_search(rng, kind: str) -> dict:
    domain = "fourier" if kind in ("fourier", "fourier_fold", "call") else "time"
    accel = jerk = 0.0
    if kind == "period":
        nsamps = 2 ** rng.randint(16, 21)
        lo = _log(rng, 0.5, 20.0)
        hi = lo * rng.uniform(1.5, 6.0)
    else:
        nsamps = 2 ** rng.randint(17, 22)
        lo = _log(rng, 20.0, 200.0)
        hi = lo * rng.uniform(1.1, 4.0)
        accel = _log(rng, 0.5, 60.0)
        jerk = _log(rng, 0.01, 3.0) if kind == "jerk" else 0.0
    base = dict(domain=domain, nsamps=nsamps, f_lo=lo, f_hi=hi, accel=accel, jerk=jerk)
    if kind == "call":
        return dict(base, kind="call", nsamps=min(nsamps, 2**19), nbins=rng.choice([32, 64]))
    if kind in ("fold", "fourier_fold"):
        return dict(base, kind="fold", storage="f32", nbins=rng.choice([30, 32, 50, 63, 64]))
    if kind == "fourier":
        return dict(base, kind="search", storage="f32", best=rng.random() < 0.5,
                    nbins=rng.choice([16, 32, 50, 64, 128]))
    return dict(base, kind="search", best=rng.random() < 0.5,
                nbins=rng.choice([16, 32, 32, 64, 128]),
                storage=rng.choice(["f32", "f32", "f32", "f16", "bf16", "bfp16"]))


def _drawable(case: dict) -> bool:
    """Whether the search's plan exists and is no larger than the listed ones."""
    try:
        cfg = _config(case)
        plan = _plan(case, cfg)
    except RuntimeError:
        return False
    scale = 4 if case["kind"] != "search" or case["domain"] == "fourier" else 1
    levels = [math.prod(int(x) for x in s) for s in plan.fold_shapes]
    pairs = case["nsamps"] * int(plan.ncoords[0])
    return (int(plan.n_levels) >= 3 and int(plan.ncoords[-1]) <= MAX_TRIALS // scale
            and max(levels[:-1]) <= MAX_VALUES // scale and pairs <= 2 * 10**10
            and (case["kind"] == "search" or levels[-1] <= MAX_VALUES // 8))


def _limits(case: dict) -> list[tuple[float, float]]:
    lims = [(case["f_lo"], case["f_hi"])]
    if case["accel"] > 0.0:
        lims.insert(0, (-case["accel"], case["accel"]))
        if case["jerk"] > 0.0:
            lims.insert(0, (-case["jerk"], case["jerk"]))
    return lims


def _config(case: dict):
    return libloki.configs.PulsarSearchConfig(
        nsamps=case["nsamps"], tsamp=TSAMP, nbins=case["nbins"], eta=1.0,
        param_limits=np.array(_limits(case)), use_fourier=case["domain"] == "fourier")


def _plan(case: dict, cfg):
    fourier = case["domain"] == "fourier"
    return libloki.plans.FFAPlanFourier(cfg) if fourier else libloki.plans.FFAPlanTime(cfg)


def _widths(nbins: int) -> np.ndarray:
    return np.array([w for w in BOXCARS if w < nbins], np.uint64)


def _series(nsamps: int, seed: int, period: float) -> tuple[torch.Tensor, torch.Tensor]:
    """N(0, 1) noise with a weak pulse train, and variances that wander by a few per cent as a
    real receiver's do."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    e = torch.randn(nsamps, device=DEVICE, generator=g)
    t = torch.arange(nsamps, device=DEVICE, dtype=torch.float64) * TSAMP
    ph = t / period
    ph = ph - torch.floor(ph) - 0.5
    e += (6.0 / math.sqrt(nsamps * 0.05) * torch.exp(-0.5 * (ph / 0.02) ** 2)).float()
    drift = torch.randn(64, device=DEVICE, generator=g).repeat_interleave(-(-nsamps // 64))
    v = 1.0 + 0.02 * drift[:nsamps]
    return e, v


def _batch_specs(case: dict) -> list[dict]:
    rng = np.random.default_rng(case["grid_seed"])
    specs = []
    for i in range(case["nseries"]):
        nsamps = 2 ** int(rng.integers(case["lo"], case["hi"] + 1))
        period = float(np.exp(rng.uniform(np.log(0.1), np.log(1.0))))
        specs.append(dict(nsamps=nsamps, nbins=(32, 64, 128)[i % 3], domain="time", accel=0.0,
                          jerk=0.0, f_lo=0.5 / period, f_hi=2.0 / period))
    return specs


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    st: dict = {"case": case}
    if kind == "batch":
        specs = _batch_specs(case)
        batch = libculoki.ffa.FFABatchCUDA([_config(s) for s in specs],
                                           widths=np.array(BOXCARS, np.uint64))
        for i, s in enumerate(specs):
            e, v = _series(s["nsamps"], seed * 1009 + i, 1.0 / s["f_lo"])
            batch.set_input(i, e.cpu().numpy(), v.cpu().numpy())
        views = []
        for i in range(len(specs)):
            views.append(_view(batch, *batch.scores_ptr(i)))
        st.update(batch=batch, views=views)
        return st
    if kind == "refine":
        e, v = _series(case["nsamps"], seed, 2.0 / (case["f_lo"] + case["f_hi"]))
        st.update(e=e, v=v, theta=_thetas(case, seed), t_ref=0.5 * case["nsamps"] * TSAMP)
        return st
    if kind == "seeds":
        st.update(_seed_inputs(case, seed))
        return st
    e, v = _series(case["nsamps"], seed, 2.0 / (case["f_lo"] + case["f_hi"]))
    cfg = _config(case)
    if kind == "call":
        st.update(e=e.cpu().numpy(), v=v.cpu().numpy(), cfg=cfg)
        return st
    fourier = case["domain"] == "fourier"
    ffa = (libculoki.ffa.FFACOMPLEXCUDA if fourier else libculoki.ffa.FFACUDA)(cfg, device_id=0)
    if case["storage"] != "f32":
        ffa.set_fold_storage(case["storage"])
    plan = ffa.plan
    st.update(e=e, v=v, ffa=ffa)
    if kind == "fold":
        st["fold"] = torch.empty(int(plan.buffer_size), device=DEVICE,
                                 dtype=torch.complex64 if fourier else torch.float32)
        st["fold_len"] = math.prod(int(x) for x in plan.fold_shapes[-1])
        st["fold_shape"] = [int(x) for x in plan.fold_shapes[-1]]
    else:
        w = _widths(case["nbins"])
        n = int(plan.ncoords[-1]) * (1 if case["best"] else w.size)
        st.update(widths=w, scores=torch.empty(n, device=DEVICE))
    return st


class _DeviceArray:
    """A device buffer of `owner`, which it keeps alive, for torch.as_tensor."""

    def __init__(self, owner, ptr: int, n: int) -> None:
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (ptr, False),
                                         "version": 3, "strides": None}


def _view(owner, ptr: int, n: int) -> torch.Tensor:
    return torch.as_tensor(_DeviceArray(owner, ptr, n), device=DEVICE)


def _thetas(case: dict, seed: int) -> torch.Tensor:
    """Candidate ephemerides: grid frequencies with the small drifts of a binary."""
    rng = np.random.default_rng(seed + 17)
    span = case["nsamps"] * TSAMP
    th = np.empty((case["ncand"], 3))
    th[:, 0] = rng.uniform(case["f_lo"], case["f_hi"], case["ncand"])
    th[:, 1] = rng.uniform(-8.0, 8.0, case["ncand"]) / span**2
    th[:, 2] = rng.uniform(-16.0, 16.0, case["ncand"]) / span**3
    return torch.from_numpy(th).to(DEVICE)


def _seed_inputs(case: dict, seed: int) -> dict:
    nb, n, segs, rows = case["nbins"], case["nleaves"], case["segments"], case["rows"]
    nbf = nb // 2 + 1
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    kw = dict(device=DEVICE, generator=g)

    def ints(high, shape):
        return torch.randint(0, high, shape, dtype=torch.int32, **kw)

    return dict(
        tree=torch.randn(n, 2, nb, **kw), ffa=torch.randn(segs, rows, 2, nb, **kw),
        tree_c=torch.randn(n, 2, nbf, dtype=torch.complex64, **kw),
        ffa_c=torch.randn(segs * rows, 2, nbf, dtype=torch.complex64, **kw),
        itree=torch.randperm(n, **kw).to(torch.int32), iffa=ints(segs * rows, (n,)),
        iffa_a=ints(rows, (segs, n)), iseg=torch.arange(segs, device=DEVICE, dtype=torch.int32),
        shift=torch.rand(n, **kw) * nb, shift_a=torch.rand(segs, n, **kw) * nb,
        mask=torch.ones(n, device=DEVICE, dtype=torch.uint8),
        out=torch.empty(n, 2, nb, device=DEVICE), out_a=torch.empty(n, 2, nb, device=DEVICE),
        out_c=torch.empty(n, 2, nbf, device=DEVICE, dtype=torch.complex64))


@functools.lru_cache(maxsize=1)
def _library():
    lib = ctypes.CDLL(str(loki_amd.LIBRARY_PATH))
    vp, sz, u32 = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_uint32
    lib.loki_shift_add_linear_batch_device.argtypes = [vp] * 7 + [sz, sz, u32, u32, sz, vp]
    lib.loki_shift_add_ascend_linear_batch_device.argtypes = [vp] * 5 + [sz] * 5 + [vp]
    lib.loki_shift_add_linear_complex_batch_device.argtypes = [vp] * 7 + [sz, sz, sz, u32, u32,
                                                                         sz, vp]
    lib.loki_last_error.restype = ctypes.c_char_p
    return lib


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "batch":
        state["batch"].execute(stream)
        return state["views"]
    if kind == "refine":
        theta = state["theta"].detach().requires_grad_()
        s = refine.fourier_score(theta, state["e"], state["v"], TSAMP, state["t_ref"],
                                 case["nbins"], case["width"])
        s.sum().backward()
        g = theta.grad
        return {"scores": s.detach(), "d_f": g[:, 0], "d_fdot": g[:, 1], "d_fddot": g[:, 2]}
    if kind == "seeds":
        return _run_seeds(state, stream)
    if kind == "call":
        scores, _plan_used = libculoki.ffa.compute_ffa_scores_cuda(state["e"], state["v"],
                                                                   state["cfg"], device_id=0,
                                                                   quiet=True)
        return scores
    ffa, e, v = state["ffa"], state["e"], state["v"]
    if kind == "fold":
        ffa.execute_device(e.data_ptr(), v.data_ptr(), state["fold"].data_ptr(),
                           state["fold"].numel(), stream)
        return state["fold"][: state["fold_len"]].view(state["fold_shape"])
    out = state["scores"]
    ffa.scores_device(e.data_ptr(), v.data_ptr(), state["widths"], out.data_ptr(), out.numel(),
                      case["best"], stream)
    return out


def _run_seeds(st: dict, stream: int) -> dict:
    case, lib = st["case"], _library()
    nb, n, segs, rows = case["nbins"], case["nleaves"], case["segments"], case["rows"]

    def p(name):
        return st[name].data_ptr()

    rc = lib.loki_shift_add_linear_batch_device(p("tree"), p("itree"), p("mask"), p("ffa"),
                                                p("iffa"), p("shift"), p("out"), nb, n, 0, n,
                                                segs * rows, stream)
    rc = rc or lib.loki_shift_add_ascend_linear_batch_device(p("ffa"), p("iseg"), p("iffa_a"),
                                                             p("shift_a"), p("out_a"), nb, rows,
                                                             n, segs, segs, stream)
    rc = rc or lib.loki_shift_add_linear_complex_batch_device(
        p("tree_c"), p("itree"), p("mask"), p("ffa_c"), p("iffa"), p("shift"), p("out_c"),
        nb // 2 + 1, nb, n, 0, n, segs * rows, stream)
    if rc:
        raise RuntimeError(lib.loki_last_error().decode())
    return {"linear": st["out"], "ascend": st["out_a"], "complex": st["out_c"]}


# --------------------------------------------------------------------------------------------
# Work: inputs read once, outputs written once; the adds, rotations and scores of the tree
# --------------------------------------------------------------------------------------------
def _search_work(case: dict, out_bytes_per_trial: int, scored: bool) -> dict:
    g = _Grid(case)
    nb = case["nbins"]
    fourier = case["domain"] == "fourier"
    nc = g.ncoords(g.levels - 1)
    rows = [g.nseg(lv) * g.ncoords(lv) for lv in range(1, g.levels)]
    if fourier:
        # level 0: at least an inner product of a few terms per harmonic; merges: two rotations
        flops = 2 * (nb // 2 + 1) * (16 * g.nseg(0) * g.ncoords(0) + sum(14 * r for r in rows))
    else:
        flops = 2 * case["nsamps"] * g.ncoords(0) + 2 * nb * sum(rows)
    if scored:
        # normalisation (3), prefix sum, a difference and a maximum per width
        flops += nc * nb * (4 + 2 * _widths(nb).size)
    return {"bytes": 8 * case["nsamps"] + nc * out_bytes_per_trial, "flops": flops}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "batch":
        parts = [_search_work(s, 4 * _widths(s["nbins"]).size, True) for s in _batch_specs(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "refine":
        nh = case["nbins"] // 2 + 1
        # per (sample, candidate): a phase; per harmonic: the fold's two and the adjoint's two
        # real products of both series
        return {"bytes": 8 * case["nsamps"] + case["ncand"] * (24 + 4 + 24),
                "flops": case["nsamps"] * case["ncand"] * (8 + 2 * 8 * nh)}
    if kind == "seeds":
        nb, n, segs = case["nbins"], case["nleaves"], case["segments"]
        nbf = nb // 2 + 1
        ffa = min(segs * case["rows"], n * segs) * 8 * nb
        return {"bytes": n * (16 * nb + 13) + 2 * ffa + n * (8 * nb + 8 * segs)
                + n * (32 * nbf + 13),
                "flops": n * (2 * nb * (1 + segs) + 2 * nbf * 8)}
    if kind == "fold":
        per = 16 * (case["nbins"] // 2 + 1) if case["domain"] == "fourier" else 8 * case["nbins"]
        return _search_work(case, per, False)
    if kind == "call":
        return _search_work(case, 4 * int(_config(case).score_widths.size), True)
    nw = 1 if case["best"] else _widths(case["nbins"]).size
    return _search_work(case, 4 * nw, True)


def tolerance(case: dict) -> dict:
    """About four times the distance to ``exact`` that the path shows at these precisions."""
    kind = case["kind"]
    if kind == "refine":
        return {"rel": 1e-5}
    if kind == "seeds":
        return {"rel": 2.5e-7}
    if kind == "fold":
        return {"rel": 1e-6}
    if case.get("domain") == "fourier":
        return {"rel": 2e-6}
    # time-domain scores: running sums over whole level-0 segments in 32 bits (1.4e-6 at
    # segments of 65536 samples); reduced-precision folds, one rounding of the stored type a level
    storage = case.get("storage", "f32")
    return {"rel": {"f32": 6e-6, "f16": 1.5e-3, "bf16": 1.2e-2, "bfp16": 2e-4}[storage]}


# --------------------------------------------------------------------------------------------
# The path in 64 bits
# --------------------------------------------------------------------------------------------
class _Grid:
    """Level geometry and shift tables: cell-centred grids whose Taylor steps halve the phase
    error tolerance of one bin, parents by the nearest lower cell."""

    def __init__(self, case: dict) -> None:
        self.nbins = case["nbins"]
        self.nsamps = case["nsamps"]
        self.lims = _limits(case)
        self.np = len(self.lims)
        f_min = self.lims[-1][0]
        levels = int(math.log2(float(self.nsamps) * TSAMP * f_min))
        self.seglen = self.nsamps // (1 << (levels - (1 if self.np == 1 else 2)))
        self.levels = int(math.log2(self.nsamps / self.seglen)) + 1

    def nseg(self, lv: int) -> int:
        return self.nsamps // (self.seglen << lv)

    def steps(self, lv: int) -> list[float]:
        tseg = float(self.seglen << lv) * TSAMP
        dt = tseg - (0.0 if self.np == 1 else tseg / 2.0)
        dphi = 1.0 / float(self.nbins)
        out = []
        for i in reversed(range(self.np)):
            d = dphi * 2.0**i * math.gamma(i + 2.0) / math.pow(dt, i + 1)
            out.append(d if i == 0 else d * C_LIGHT / self.lims[-1][1])
        return out

    def counts(self, lv: int) -> tuple[int, ...]:
        return tuple(1 if d >= hi - lo else int(math.ceil((hi - lo) / d))
                     for (lo, hi), d in zip(self.lims, self.steps(lv)))

    def ncoords(self, lv: int) -> int:
        return math.prod(self.counts(lv))

    def level0_freqs(self) -> torch.Tensor:
        lo, hi = self.lims[-1]
        n = self.counts(0)[-1]
        if n == 1:
            return torch.tensor([(hi + lo) / 2.0], dtype=torch.float64, device=DEVICE)
        dv = (hi - lo) / float(n)
        return (lo + 0.5 * dv) + dv * torch.arange(n, dtype=torch.float64, device=DEVICE)

    def cells(self, p: int, lv: int) -> torch.Tensor:
        lo, hi = self.lims[p]
        n = self.counts(lv)[p]
        if n == 1:
            return torch.tensor([(hi + lo) / 2.0], dtype=torch.float64, device=DEVICE)
        dv = (hi - lo) / float(n)
        return lo + dv * (torch.arange(n, dtype=torch.float64, device=DEVICE) + 0.5)

    def nearest(self, val: torch.Tensor, p: int, lv: int) -> torch.Tensor:
        lo, hi = self.lims[p]
        n = self.counts(lv)[p]
        if n == 1:
            return torch.zeros_like(val, dtype=torch.int64)
        raw = (float(n) * (val - lo)) / (hi - lo)
        return torch.trunc(raw + 1e-6).clamp(0, n - 1).to(torch.int64)

    def side(self, lv: int, head: int) -> tuple[torch.Tensor, torch.Tensor]:
        """(parent coordinate, phase shift in bins) of every coordinate of level lv."""
        tseg = math.ldexp(self.seglen * TSAMP, lv - 1)
        f = self.cells(self.np - 1, lv)
        if self.np == 1:
            idx = self.nearest(f, 0, lv - 1)
            shift = _phase_bins(tseg * f, self.nbins) if head else torch.zeros_like(f).float()
            return idx, shift
        dt = (head - 0.5) * tseg
        n_prev = self.counts(lv - 1)
        a = self.cells(self.np - 2, lv)
        if self.np == 2:
            v, d, base = a * dt, a * (0.5 * dt * dt), self.nearest(a, 0, lv - 1) * n_prev[1]
        else:
            j = self.cells(0, lv)[:, None]
            v = (a * dt) + 0.5 * j * (dt * dt)
            d = (a * (0.5 * (dt * dt))) + j * (dt * dt * dt / 6.0)
            base = (self.nearest(j, 0, lv - 1) * n_prev[1] * n_prev[2]
                    + self.nearest(a + j * dt, 1, lv - 1) * n_prev[2])
        v, d, base = v.reshape(-1, 1), d.reshape(-1, 1), base.reshape(-1, 1)
        f_new = f * (1.0 - v * INV_C)
        shift = _phase_bins((dt - d * INV_C) * f, self.nbins)
        idx = base + self.nearest(f_new, self.np - 1, lv - 1)
        return idx.reshape(-1), shift.reshape(-1)


def _phase_bins(turns: torch.Tensor, nbins: int) -> torch.Tensor:
    ph = (turns - torch.floor(turns)) * float(nbins)
    return torch.where(ph >= float(nbins), torch.zeros_like(ph), ph).float()


def _bin_index(shift: torch.Tensor, nbins: int) -> torch.Tensor:
    b = (shift + 0.5).to(torch.int64)
    return torch.where(b == nbins, torch.zeros_like(b), b)


def _phases0(g: _Grid, f: torch.Tensor) -> torch.Tensor:
    """Turns of every sample of a segment at the level-0 frequencies f: [len(f), seglen]."""
    t = torch.arange(g.seglen, dtype=torch.float64, device=DEVICE) * TSAMP
    t_ref = 0.0 if g.np == 1 else float(g.seglen) * TSAMP / 2.0
    return (t - t_ref)[None, :] * f[:, None]


def _level0_time(g: _Grid, x: torch.Tensor) -> torch.Tensor:
    """x [2 nseg, seglen] -> [nseg, nfreq, 2, nbins]: sums over the runs of equal bins from
    the running sums of the samples."""
    freqs = g.level0_freqs()
    nb, nrow = g.nbins, x.shape[0]
    run = torch.zeros(g.seglen + 1, nrow, dtype=torch.float64, device=DEVICE)
    run[1:] = torch.cumsum(x.t(), dim=0)
    out = torch.empty(nrow, freqs.numel(), nb, dtype=torch.float64, device=DEVICE)
    step = max(1, min(2**24 // g.seglen, 2**29 // (nrow * min(g.seglen, 4096))))
    for i in range(0, freqs.numel(), step):
        f = freqs[i:i + step]
        b = _bin_index(_phase_bins(_phases0(g, f), nb), nb)
        start = torch.ones_like(b, dtype=torch.bool)
        start[:, 1:] = b[:, 1:] != b[:, :-1]
        fi, k = torch.nonzero(start, as_tuple=True)
        end = torch.full_like(k, g.seglen)
        same = fi[1:] == fi[:-1]
        end[:-1] = torch.where(same, k[1:], end[:-1])
        acc = torch.zeros(f.numel() * nb, nrow, dtype=torch.float64, device=DEVICE)
        acc.index_add_(0, fi * nb + b[fi, k], run[end] - run[k])
        out[:, i:i + step] = acc.t().reshape(nrow, f.numel(), nb)
    return out.view(-1, 2, freqs.numel(), nb).transpose(1, 2).contiguous()


def _level0_fourier(g: _Grid, x: torch.Tensor) -> torch.Tensor:
    """x [2 nseg, seglen] -> [nseg, nfreq, 2, nbins/2+1]: a plain DFT per frequency."""
    freqs = g.level0_freqs()
    nbf = g.nbins // 2 + 1
    m = torch.arange(nbf, dtype=torch.float64, device=DEVICE)
    out = torch.empty(x.shape[0], freqs.numel(), nbf, dtype=torch.complex128, device=DEVICE)
    for i in range(freqs.numel()):
        ph = _phases0(g, freqs[i:i + 1])[0]
        ang = (2.0 * math.pi) * torch.frac((ph - torch.floor(ph))[:, None] * m)
        out[:, i] = torch.complex(x @ torch.cos(ang), -(x @ torch.sin(ang)))
    return out.view(-1, 2, freqs.numel(), nbf).transpose(1, 2).contiguous()


def _merge(g: _Grid, fold: torch.Tensor, lv: int, fourier: bool) -> torch.Tensor:
    nb = g.nbins
    w = fold.shape[-1]
    nc = g.ncoords(lv)
    sides = [g.side(lv, h) for h in (0, 1)]
    out = torch.empty(g.nseg(lv), nc, 2, w, dtype=fold.dtype, device=DEVICE)
    k = torch.arange(w, dtype=torch.float64, device=DEVICE)
    step = max(1, 2**26 // (w * 2 * max(1, g.nseg(lv))))
    for c in range(0, nc, step):
        acc = None
        for h, (idx, shift) in enumerate(sides):
            rows = fold[h::2][:, idx[c:c + step]]
            sh = shift[c:c + step]
            if fourier:
                ang = (-2.0 * math.pi) * torch.frac(sh.double()[:, None] * k / nb)
                rows = rows * torch.polar(torch.ones_like(ang), ang)[None, :, None, :]
            else:
                src = (torch.arange(nb, device=DEVICE) - _bin_index(sh, nb)[:, None]) % nb
                rows = torch.gather(rows, 3, src[None, :, None, :].expand(rows.shape))
            acc = rows if acc is None else acc + rows
        out[:, c:c + step] = acc
    return out


def _exact_fold(case: dict, e: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    g = _Grid(case)
    fourier = case["domain"] == "fourier"
    x = torch.stack([e.double().view(-1, g.seglen), v.double().view(-1, g.seglen)], dim=1)
    x = x.reshape(-1, g.seglen)
    if fourier and case["nbins"] <= LOSSY_ABOVE:
        fold = _level0_fourier(g, x)
    else:
        fold = _level0_time(g, x)
        if fourier:
            fold = torch.fft.rfft(fold, dim=-1)
    for lv in range(1, g.levels):
        fold = _merge(g, fold, lv, fourier)
    return fold


def _exact_scores(case: dict, e, v, widths, best: bool) -> torch.Tensor:
    fold = _exact_fold(case, e, v)[0]
    n = case["nbins"]
    out = torch.empty(fold.shape[0], len(widths), dtype=torch.float64, device=DEVICE)
    for c in range(0, fold.shape[0], 2**19):
        part = fold[c:c + 2**19]
        if part.is_complex():
            part = torch.fft.irfft(part, n=n)
        p = part[:, 0] / torch.sqrt(part[:, 1])
        ps = torch.cumsum(torch.nn.functional.pad(torch.cat([p, p], dim=1), (1, 0)), dim=1)
        total = ps[:, n]
        for i, w in enumerate(int(w) for w in widths):
            h = math.sqrt((n - w) / (n * w))
            b = w * h / (n - w)
            d = (ps[:, w:w + n] - ps[:, :n]).amax(dim=1)
            out[c:c + 2**19, i] = (h + b) * d - b * total
    return out.amax(dim=1) if best else out.reshape(-1)


def _exact_refine(case: dict, seed: int) -> dict:
    e, v = _series(case["nsamps"], seed, 2.0 / (case["f_lo"] + case["f_hi"]))
    e, v = e.double(), v.double()
    theta = _thetas(case, seed)
    n, w = case["nbins"], case["width"]
    tau = torch.arange(case["nsamps"], dtype=torch.float64, device=DEVICE) * TSAMP
    tau = tau - 0.5 * case["nsamps"] * TSAMP
    basis = torch.stack([tau, tau**2 / 2.0, tau**3 / 6.0])
    m = torch.arange(n // 2 + 1, dtype=torch.float64, device=DEVICE)
    h = math.sqrt((n - w) / (n * w))
    b = w * h / (n - w)
    win = torch.arange(w, device=DEVICE)
    scores, grads = [], []
    for th in theta:
        ph = th @ basis
        ang = (-2.0 * math.pi) * torch.frac((ph - torch.floor(ph)) * m[:, None])
        cs, sn = torch.cos(ang), torch.sin(ang)
        fold = torch.stack([torch.complex(cs @ s, sn @ s) for s in (e, v)])
        fold.requires_grad_()
        x = torch.fft.irfft(fold, n=n)
        p = x[0] / torch.sqrt(x[1])
        wins = p[(torch.arange(n, device=DEVICE)[:, None] + win) % n].sum(dim=1)
        s = (h + b) * wins.max() - b * p.sum()
        (gr,) = torch.autograd.grad(s, fold)
        # dE_m / dphi_k = -2 pi i m x_k w_mk
        scores.append(s.detach())
        dphi = torch.zeros_like(tau)
        for q, series in enumerate((e, v)):
            re, im = gr[q].real * m, gr[q].imag * m
            dphi += 2.0 * math.pi * series * (re @ sn - im @ cs)
        grads.append(basis @ dphi)
    gr = torch.stack(grads)
    return {"scores": torch.stack(scores), "d_f": gr[:, 0], "d_fdot": gr[:, 1],
            "d_fddot": gr[:, 2]}


def _exact_seeds(case: dict, seed: int) -> dict:
    st = _seed_inputs(case, seed)
    nb, n, segs, rows = case["nbins"], case["nleaves"], case["segments"], case["rows"]
    j = torch.arange(nb, device=DEVICE)
    ffa = st["ffa"].double().view(-1, 2, nb)

    def rotated(index, shift):
        src = (j - _bin_index(shift, nb)[:, None]) % nb
        return torch.gather(ffa[index.long()], 2, src[:, None, :].expand(n, 2, nb))

    linear = st["tree"].double()[st["itree"].long()] + rotated(st["iffa"], st["shift"])
    ascend = sum(rotated(st["iffa_a"][s] + s * rows, st["shift_a"][s]) for s in range(segs))
    k = torch.arange(nb // 2 + 1, dtype=torch.float64, device=DEVICE)
    ang = (-2.0 * math.pi) * torch.frac(st["shift"].double()[:, None] * k / nb)
    cplx = (st["tree_c"].to(torch.complex128)[st["itree"].long()]
            + st["ffa_c"].to(torch.complex128)[st["iffa"].long()]
            * torch.polar(torch.ones_like(ang), ang)[:, None, :])
    return {"linear": linear, "ascend": ascend, "complex": cplx}


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "refine":
        return _exact_refine(case, seed)
    if kind == "seeds":
        return _exact_seeds(case, seed)
    if kind == "batch":
        out = []
        for i, s in enumerate(_batch_specs(case)):
            e, v = _series(s["nsamps"], seed * 1009 + i, 1.0 / s["f_lo"])
            out.append(_exact_scores(s, e, v, _widths(s["nbins"]), False))
        return out
    if _Grid(case).ncoords(_Grid(case).levels - 1) > 20_000_000:
        return None  # tens of gigabytes of 64-bit folds
    e, v = _series(case["nsamps"], seed, 2.0 / (case["f_lo"] + case["f_hi"]))
    if kind == "fold":
        return _exact_fold(case, e, v)
    if kind == "call":
        widths = [int(w) for w in _config(case).score_widths]
        return _exact_scores(case, e, v, widths, False).cpu().numpy()
    return _exact_scores(case, e, v, _widths(case["nbins"]), case["best"])
