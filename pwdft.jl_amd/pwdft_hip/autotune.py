"""Autotuner for the launch parameters of op_H on one Hamiltonian's shape.

Every candidate is timed on the device with the library's own per-kernel events
(pw_profile_*) on the Hamiltonian's largest k-point and its band count, in four stages, each
keeping the best setting of the previous ones:

1. FFT plans: the radix mode of the line FFTs (PW_TUNE_FFT_ORDER: 0, the plane and column
   kernels' two-pass plans with the largest radices first elsewhere; the general column
   kernels with the same radices reversed, or with radices 5/4/3/2 only) x the z-plane kernel
   (as sizes choose it, or the general compressed plane of the active x lines) x the z-columns
   per workgroup of the general column kernels (0: as sizes choose), scored by the three FFT
   kernels' time;
2. the band split: bands per FFT launch (PW_TUNE_BAND_BATCH), same score;
3. the projector GEMMs: tile shape (a tile per wavefront, or one that four or eight
   wavefronts share along K) and split-K workgroup target of beta^H psi and of beta (D B),
   each scored by its own kernel time;
4. whole-op_H choices scored by wall time: beta^H psi on a second stream where the sizes
   make that pay or not, and (mixed precision) the BF16-split MFMA GEMM off or on, each with
   the tiles of stage 3 timed under it.

Stages 1-3 score kernels run one at a time (no second stream), so that no kernel's time
includes a neighbour's; the result is kept only if the whole op_H beats the settings the
context ran on entry (timed alternately with them, at least 1 % faster).

The chosen settings are applied with pw_tune_set and cached in a JSON file keyed by the
shape (grid, plane waves, projectors, bands, precision), with the generation of the kernels they
were timed on, so a later Hamiltonian of the same shape applies them without timing (Hamiltonian(..., autotune=True)).  Settings change the
order of floating-point operations only; the tests check that a tuned op_H equals the
default one to rounding."""
import json
import os
import time

import numpy as np

from ._lib import DeviceMatrix, PW_MIXED, PW_TERM_ALL

(TUNE_GEMM_CN_SHAPE, TUNE_GEMM_NN_SHAPE, TUNE_GEMM_CN_WG, TUNE_GEMM_NN_WG, TUNE_BAND_BATCH,
 TUNE_PLANE_COMPRESSED, TUNE_OVERLAP, TUNE_COL_CHUNK, TUNE_GEMM_SPLIT_BF16) = range(9)
TUNE_FFT_ORDER = 15
SHAPES = {-1: "auto", 0: "64x64", 1: "128x64", 2: "64x128", 3: "128x128", 4: "128x32", 5: "64x32",
          6: "16x16 by eight", 7: "32x32 by four"}

# Generation of the kernels that the settings name: raised whenever a code means another kernel than
# before (2: the plane and column kernels, which a column chunk, a radix mode or a plane mode of the
# general kernels switches off, and GEMM tiles without LDS).  An entry of another generation is timed anew.
KERNELS = 2

# the library's defaults (what a fresh context runs)
DEFAULTS = {"fft_order": 0, "plane_compressed": 0, "col_chunk": 0, "band_batch": 64,
            "gemm_cn_shape": -1, "gemm_cn_wg": 0, "gemm_nn_shape": -1, "gemm_nn_wg": 0,
            "overlap": 1, "gemm_split_bf16": -1}
_KEYS = {"fft_order": TUNE_FFT_ORDER, "plane_compressed": TUNE_PLANE_COMPRESSED, "col_chunk": TUNE_COL_CHUNK,
         "band_batch": TUNE_BAND_BATCH, "gemm_cn_shape": TUNE_GEMM_CN_SHAPE, "gemm_cn_wg": TUNE_GEMM_CN_WG,
         "gemm_nn_shape": TUNE_GEMM_NN_SHAPE, "gemm_nn_wg": TUNE_GEMM_NN_WG, "overlap": TUNE_OVERLAP,
         "gemm_split_bf16": TUNE_GEMM_SPLIT_BF16}
# applied in this order: the FFT radix mode re-plans the grid before anything sized by it
_ORDER = ["fft_order", "plane_compressed", "col_chunk", "band_batch", "gemm_cn_shape", "gemm_cn_wg",
          "gemm_nn_shape", "gemm_nn_wg", "overlap", "gemm_split_bf16"]


def cache_path():
    """The tuning cache: $PWDFT_HIP_TUNE_CACHE, else ~/.cache/pwdft_hip/tune.json."""
    p = os.environ.get("PWDFT_HIP_TUNE_CACHE")
    if p:
        return p
    return os.path.join(os.path.expanduser("~"), ".cache", "pwdft_hip", "tune.json")


def shape_key(Ns, ngw, nbeta, nbands, mixed):
    """Cache key of one op_H shape: grid, plane waves of the tuned k-point, projectors,
    bands, precision."""
    n1, n2, n3 = (int(x) for x in Ns)
    return f"{n1}x{n2}x{n3}/ngw{int(ngw)}/nbeta{int(nbeta)}/nb{int(nbands)}/{'mixed' if mixed else 'fp64'}"


def load_cache(path=None):
    path = path or cache_path()
    try:
        with open(path) as f:
            d = json.load(f)
        return d if isinstance(d, dict) else {}
    except (OSError, ValueError):
        return {}


def save_cache(entries, path=None):
    """Merge entries into the cache file (written atomically)."""
    path = path or cache_path()
    d = load_cache(path)
    d.update(entries)
    os.makedirs(os.path.dirname(os.path.abspath(path)), exist_ok=True)
    tmp = f"{path}.{os.getpid()}.tmp"
    with open(tmp, "w") as f:
        json.dump(d, f, indent=1, sort_keys=True)
    os.replace(tmp, path)


def apply_settings(ctx, settings):
    """pw_tune_set for every known key of settings (unknown keys are ignored)."""
    for k in _ORDER:
        if k in settings:
            ctx.call("pw_tune_set", _KEYS[k], int(settings[k]))


def _profiled(H, X, Y, flags, steps):
    """Per-kernel ms per step from the library's events (kernels run one at a time: the
    nonlocal products are kept off the second stream while kernels are scored)."""
    c = H.ctx
    c.call("pw_op_H_dev", H.ik, H.ispin, X.cols, X.p, X.rows, Y.p, Y.rows, flags)   # warm
    c.call("pw_synchronize")
    c.profile(True)
    for _ in range(steps):
        c.call("pw_op_H_dev", H.ik, H.ispin, X.cols, X.p, X.rows, Y.p, Y.rows, flags)
    c.call("pw_synchronize")
    prof = c.profile_read()
    c.profile(False)
    return {k: v[0] / steps for k, v in prof.items()}


def _wall(H, X, Y, flags, steps):
    """Device time per op_H between two events on the library's stream (no per-kernel
    events recorded), the best of three runs of `steps` calls."""
    import ctypes
    c = H.ctx
    c.call("pw_op_H_dev", H.ik, H.ispin, X.cols, X.p, X.rows, Y.p, Y.rows, flags)   # warm
    c.call("pw_synchronize")
    best = float("inf")
    ms = ctypes.c_float()
    for _ in range(3):
        c.call("pw_event_record", 0)
        for _ in range(steps):
            c.call("pw_op_H_dev", H.ik, H.ispin, X.cols, X.p, X.rows, Y.p, Y.rows, flags)
        c.call("pw_event_record", 1)
        c.call("pw_synchronize")
        c.call("pw_event_elapsed_ms", 0, 1, ctypes.byref(ms))
        best = min(best, ms.value / steps)
    return best


def _fft_ms(t):
    return t["col_ifft"] + t["plane_vloc"] + t["col_fft"]


def tune_op_H(H, nbands=None, mixed=None, steps=3, quick=False):
    """Time the candidates on H (see the module docstring), apply the best settings and
    return (settings, table) where table lists every timed candidate.  The settings the
    context runs on entry are timed first; the tuned ones are kept only if their op_H is
    faster."""
    mixed = H.mixed if mixed is None else mixed
    flags = PW_TERM_ALL | (PW_MIXED if mixed else 0)
    c = H.ctx
    ik = int(np.argmax(H.pw.Ngw))
    ik_save = H.ik
    H.ik = ik
    nb = int(nbands or H.electrons.Nstates)
    ngw = int(H.pw.Ngw[ik])
    rng = np.random.default_rng(12345)
    X = DeviceMatrix.from_host(c, rng.standard_normal((ngw, nb)) + 1j * rng.standard_normal((ngw, nb)))
    Y = DeviceMatrix(c, ngw, nb)
    entry = dict(DEFAULTS)
    entry["band_batch"] = int(getattr(H, "band_batch", DEFAULTS["band_batch"]))
    apply_settings(c, entry)
    table = [dict(entry, op_H_ms=_wall(H, X, Y, flags, 3 * steps), stage="entry")]
    best = dict(entry)
    try:
        apply_settings(c, {"overlap": 0})
        # 1. FFT plans
        score = None
        for order in (0, 1, 2):
            for plane in (0, 1):
                for chunk in ((0,) if quick else (0, 16, 32)):
                    cand = {"fft_order": order, "plane_compressed": plane, "col_chunk": chunk}
                    try:
                        apply_settings(c, cand)
                    except Exception:   # a radix mode with no plan for this grid
                        continue
                    ms = _fft_ms(_profiled(H, X, Y, flags, steps))
                    table.append(dict(cand, fft_ms=ms))
                    if score is None or ms < score:
                        score = ms
                        best.update(cand)
        apply_settings(c, best)
        apply_settings(c, {"overlap": 0})
        # 2. band split
        for bb in sorted({b for b in (16, 32, 64, 96, 128, 160, 256, nb) if b <= nb}):
            apply_settings(c, {"band_batch": bb})
            ms = _fft_ms(_profiled(H, X, Y, flags, steps))
            table.append({"band_batch": bb, "fft_ms": ms})
            if ms < score:
                score = ms
                best["band_batch"] = bb
        apply_settings(c, {"band_batch": best["band_batch"]})
        # 3. projector GEMMs (both products timed in one run per candidate)
        def products(split):
            """The best tiles and targets of both products under one split-BF16 setting.  Codes 6 and 7 run
            FP32 MFMA under any, so with it on either product can still go without."""
            shapes = (-1, 0, 5, 6, 7) if quick else (-1, 0, 1, 2, 4, 5, 6, 7)
            targets = (0, 512) if quick else (0, 256, 512, 1024, 2048)
            bcn = bnn = None
            apply_settings(c, {"gemm_split_bf16": split, "overlap": 0})
            for shape in shapes:
                for wg in targets:
                    apply_settings(c, {"gemm_cn_shape": shape, "gemm_nn_shape": shape, "gemm_cn_wg": wg,
                                       "gemm_nn_wg": wg})
                    t = _profiled(H, X, Y, flags, steps)
                    table.append({"gemm_shape": SHAPES[shape], "gemm_wg": wg, "gemm_split_bf16": split,
                                  "gemm_cn_ms": t["gemm_cn"], "gemm_nn_ms": t["gemm_nn"]})
                    # the solvers' own products run under these settings too: a tile other than the
                    # rules' (-1, 7) must be a tenth faster, or a smaller product loses what op_H gains
                    # (mixed LOBPCG at Si64, A^H B in 64 x 64 tiles: 7.7 against 7.4 ms an iteration)
                    f = 1.0 if shape in (-1, 7) else 1.1
                    if bcn is None or f * t["gemm_cn"] < bcn[0]:
                        bcn = (f * t["gemm_cn"], shape, wg)
                    if bnn is None or f * t["gemm_nn"] < bnn[0]:
                        bnn = (f * t["gemm_nn"], shape, wg)
            return {"gemm_cn_shape": bcn[1], "gemm_cn_wg": bcn[2], "gemm_nn_shape": bnn[1], "gemm_nn_wg": bnn[2],
                    "gemm_split_bf16": split}
        nonlocal_term = H.pspotNL.NbetaNL > 0
        if nonlocal_term:
            best.update(products(best["gemm_split_bf16"]))
        apply_settings(c, best)
        # 4. whole op_H: second stream, BF16-split GEMMs (mixed only), by wall time
        wall = _wall(H, X, Y, flags, 3 * steps)
        cands = [lambda: {"overlap": 1 - best["overlap"]}]
        if mixed and nonlocal_term:
            cands += [lambda: products(0), lambda: products(1)]
        for cand in cands:
            new = cand()
            apply_settings(c, dict(best, **new))
            w = _wall(H, X, Y, flags, 3 * steps)
            table.append(dict(new, op_H_ms=w))
            if w < wall:
                wall = w
                best.update(new)
        apply_settings(c, best)
        # final check, entry and tuned settings timed alternately (drift and noise hit both):
        # the tuned ones are kept only if at least 1 % faster
        t_entry, t_best = float("inf"), float("inf")
        for _ in range(3):
            apply_settings(c, entry)
            t_entry = min(t_entry, _wall(H, X, Y, flags, 5 * steps))
            apply_settings(c, best)
            t_best = min(t_best, _wall(H, X, Y, flags, 5 * steps))
        table.append({"final_entry_ms": t_entry, "final_tuned_ms": t_best})
        if t_best > 0.99 * t_entry:
            best, t_best = dict(entry), t_entry
        apply_settings(c, best)
        best["op_H_ms"] = t_best
    finally:
        H.ik = ik_save
        X.free()
        Y.free()
    return best, table


def autotune(H, nbands=None, mixed=None, cache=True, path=None, **kw):
    """Settings for H's op_H shape: from the cache when present, else timed by tune_op_H
    and stored.  Applies them to H's context and returns (settings, source) with source
    "cache" or "tuned"."""
    mixed = H.mixed if mixed is None else mixed
    ik = int(np.argmax(H.pw.Ngw))
    nb = int(nbands or H.electrons.Nstates)
    key = shape_key(H.pw.Ns, H.pw.Ngw[ik], H.pspotNL.NbetaNL, nb, mixed)
    if cache:
        hit = load_cache(path).get(key)
        if isinstance(hit, dict) and hit.get("kernels") == KERNELS:
            apply_settings(H.ctx, hit)
            return hit, "cache"
    settings, _ = tune_op_H(H, nbands=nb, mixed=mixed, **kw)
    if cache:
        save_cache({key: dict(settings, kernels=KERNELS)}, path)
    return settings, "tuned"
