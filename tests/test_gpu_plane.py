"""The plane and column kernels (csrc/pw_plane.h, pw_col.h) through the C ABI against numpy's FFT: every line
length with a two-pass plan, lengths without one, unequal lengths, index sets inside and
outside the half-sphere window, and density groups of several bands.  Tolerances are those
of the operator tests: 1e-12 (FP64) and 2e-5 (mixed) of the largest value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PLANS = [12, 15, 16, 18, 20, 24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108,
         120, 128, 135, 144, 150, 160, 180, 192]


def index_set(ns, radius, shift=0.3):
    """Grid points of an ellipsoid of the given half axes, off centre by `shift` points."""
    m = [np.where(np.arange(n) > n // 2, np.arange(n) - n, np.arange(n)) for n in ns]
    r2 = sum((((a - shift) / max(r, 0.5)) ** 2).reshape([-1 if d == i else 1 for i in range(3)])
             for d, (a, r) in enumerate(zip(m, radius)))
    x, y, z = np.nonzero(r2 <= 1.0)
    idx = np.sort(x + ns[0] * (y + ns[1] * z))
    return np.random.default_rng(5).permutation(idx).astype(np.int64)


def context(ns, idx, omega=3.7):
    import pwdft_hip as ph
    from pwdft_hip._lib import ptr
    c = ph.Context()
    c.call("pw_set_grid", *ns, omega)
    c.call("pw_set_band_batch", 64)
    gk = np.random.default_rng(6).standard_normal((idx.size, 3))
    c.call("pw_set_kpoint", 0, idx.size, ptr(idx), 0, ptr(gk))
    return c


def apply_v(c, ns, idx, V, psi, mixed):
    from pwdft_hip._lib import PW_MIXED, PW_TERM_VLOC, ptr
    c.call("pw_set_vloc", 0, ptr(V))
    out = np.zeros_like(psi)
    c.call("pw_op_H", 0, 0, psi.shape[1], ptr(psi), psi.shape[0], ptr(out), out.shape[0],
           PW_TERM_VLOC | (PW_MIXED if mixed else 0))
    f = np.zeros((psi.shape[1], ns[2], ns[1], ns[0]), dtype=complex)
    f.reshape(psi.shape[1], -1)[:, idx] = psi.T
    f = np.fft.fftn(np.fft.ifftn(f, axes=(1, 2, 3)) * V.reshape(ns[2], ns[1], ns[0]), axes=(1, 2, 3))
    return out, f.reshape(psi.shape[1], -1)[:, idx].T


def rand(rng, n, nb):
    return np.asfortranarray(rng.standard_normal((n, nb)) + 1j * rng.standard_normal((n, nb)))


VLOC = [((n, n, 12), "half", m) for n in PLANS for m in (False, True)]
VLOC += [((n, n, 12), "full", False) for n in (12, 20, 27, 45, 72, 75, 96)]
VLOC += [((n, n, 12), "full", True) for n in (27, 72)]
VLOC += [((40, 75, 12), "half", m) for m in (False, True)] + [((75, 40, 12), "half", m) for m in (False, True)]
VLOC += [((108, 64, 16), "half", False), ((27, 160, 12), "half", True), ((45, 36, 12), "full", False)]
VLOC += [((16, 15, n), "half", m) for n in PLANS for m in (False, True)]
VLOC += [((16, 15, n), "full", False) for n in PLANS] + [((16, 15, n), "full", True) for n in (27, 72, 125)]
VLOC += [((n, n, 12), "full", True) for n in PLANS if n <= 135 and n not in (27, 72)]
VLOC += [((16, 15, n), "full", True) for n in PLANS if n not in (27, 72)]
VLOC += [((125, 8, 12), "half", False), ((10, 125, 12), "half", True), ((5, 6, 4), "full", False)]


@pytest.mark.parametrize("ns,extent,mixed", VLOC)
def test_vloc_plane(ns, extent, mixed):
    idx = index_set(ns, [((n - 1) // 4) if extent == "half" else n // 2 - 0.6 for n in ns])
    c = context(ns, idx)
    rng = np.random.default_rng(1)
    V = rng.standard_normal(int(np.prod(ns)))
    print(f"case {ns} {extent} mixed={mixed}", flush=True)
    got, ref = apply_v(c, ns, idx, V, rand(rng, idx.size, 3), mixed)
    assert np.abs(got - ref).max() <= (2e-5 if mixed else 1e-12) * np.abs(ref).max()
    c.close()


RHO = [((n, n, 120), m) for n in (15, 24, 27, 45, 72, 75) for m in (False, True)]
RHO += [((108, 108, 120), False), ((135, 135, 150), True), ((40, 75, 120), True), ((75, 27, 120), False)]


def check_rho(ns, idx, nb, mixed):
    from pwdft_hip._lib import PW_MIXED, ptr
    c = context(ns, idx)
    rng = np.random.default_rng(2)
    psi = rand(rng, idx.size, nb)
    w = rng.random(nb)
    N = int(np.prod(ns))
    print(f"case rho {ns} ngw={idx.size} mixed={mixed}", flush=True)
    c.call("pw_rhoe_zero")
    c.call("pw_rhoe_accum", 0, nb, ptr(psi), idx.size, ptr(w), PW_MIXED if mixed else 0)
    got = np.empty(N)
    c.call("pw_rhoe_get", ptr(got))
    ref = np.zeros(N)
    for b in range(nb):
        f = np.zeros(N, dtype=complex)
        f[idx] = psi[:, b]
        ref += w[b] * np.abs(np.fft.ifftn(f.reshape(ns[2], ns[1], ns[0])).reshape(-1)) ** 2
    ref *= float(N) ** 2 / 3.7
    assert np.abs(got - ref).max() <= (2e-5 if mixed else 1e-12) * np.abs(ref).max()
    c.close()


@pytest.mark.parametrize("ns,mixed", RHO)
def test_rho_groups(ns, mixed):
    """More bands than groups, so a workgroup carries its plane state over several bands."""
    check_rho(ns, index_set(ns, [(n - 1) // 4 for n in ns]), 16, mixed)


# planes long in x (whose compressed form leaves no room for row buffers), lengths without a plan, and
# spheres beyond the half-sphere window
RHO_GENERAL = [((375, 20, 12), "half", False), ((320, 30, 12), "half", False), ((125, 50, 12), "half", True),
               ((10, 10, 12), "half", False), ((125, 80, 12), "full", False), ((16, 15, 12), "full", True),
               ((36, 72, 12), "wide", False), ((72, 36, 12), "wide", True)]
# (a plane whose active lines LDS cannot hold has no density kernel: 135 in FP64, 192 in FP32)
RHO_GENERAL += [((n, n, 12), "wide", m) for n in PLANS for m in (False, True) if n <= (180 if m else 128)]
RHO_GENERAL += [((n, n, 12), "full", False) for n in (12, 27, 45, 96)] + [((n, n, 12), "full", True) for n in (45, 128)]


@pytest.mark.parametrize("ns,extent,mixed", RHO_GENERAL)
def test_rho_general(ns, extent, mixed):
    radius = {"half": [(n - 1) // 4 for n in ns], "wide": [0.28 * n for n in ns],
              "full": [n // 2 - 0.6 for n in ns]}[extent]
    check_rho(ns, index_set(ns, radius), 3, mixed)


# the plane passes of the batched op_H: plane kernels (also where LDS holds no padded plane), padded planes
# (one length without a plan, planes long in x), compressed planes k-point after k-point
@pytest.mark.parametrize("ns,extent,mixed", [
    ((24, 36, 20), "half", False), ((24, 36, 20), "half", True), ((125, 12, 12), "half", False),
    ((12, 125, 12), "half", True), ((375, 20, 12), "half", False),
    ((108, 108, 12), "half", False), ((125, 100, 12), "half", False),
    ((45, 45, 12), "wide", True), ((45, 45, 12), "wide", False), ((96, 96, 12), "full", False)])
@pytest.mark.parametrize("acc", [False, True])
def test_op_H_batch(ns, extent, mixed, acc):
    """Local potential and kinetic term over k-points of different spheres, against numpy."""
    from pwdft_hip._lib import (PW_ACCUMULATE, PW_MIXED, PW_TERM_K, PW_TERM_VLOC, PW_TUNE_FUSED_BATCH, DeviceMatrix,
                                ptr)
    rng = np.random.default_rng(4)
    nk, nb = 3, 2
    # the first sphere is the widest, and one k-point alone goes beyond the window
    scale = {"half": [(n - 1) // 4 for n in ns], "wide": [0.3 * n for n in ns],
             "full": [n // 2 - 0.6 for n in ns]}[extent]
    sets = [index_set(ns, [r - ik * (0.5 if extent == "half" else 0.1 * r) for r in scale], shift=0.2 * ik / nk)
            for ik in range(nk)]
    c = context(ns, sets[0])
    c.call("pw_tune_set", PW_TUNE_FUSED_BATCH, 0)   # the three-stage launches also where a box fits LDS
    gk = [rng.standard_normal((s.size, 3)) for s in sets]
    for ik in range(nk):
        c.call("pw_set_kpoint", ik, sets[ik].size, ptr(sets[ik]), 0, ptr(gk[ik]))
    V = rng.standard_normal(int(np.prod(ns)))
    c.call("pw_set_vloc", 0, ptr(V))
    psi = [rand(rng, s.size, nb) for s in sets]
    # what is there before is added to, or (NaN) never read
    old = [rand(rng, s.size, nb) if acc else np.full((s.size, nb), np.nan + 0j) for s in sets]
    dev = [DeviceMatrix.from_host(c, p) for p in psi]
    out = [DeviceMatrix.from_host(c, o) for o in old]
    iks = np.arange(nk, dtype=np.int32)
    ld = np.array([s.size for s in sets], dtype=np.int64)
    pp = np.array([d.p.value for d in dev], dtype=np.uint64)
    hp = np.array([d.p.value for d in out], dtype=np.uint64)
    print(f"case op_H batch {ns} {extent} mixed={mixed} acc={acc}", flush=True)
    c.call("pw_op_H_batch_dev", nk, ptr(iks), 0, nb, ptr(pp), ptr(ld), ptr(hp), ptr(ld),
           PW_TERM_VLOC | PW_TERM_K | (PW_MIXED if mixed else 0) | (PW_ACCUMULATE if acc else 0))
    c.call("pw_synchronize")
    for ik in range(nk):
        f = np.zeros((nb, ns[2], ns[1], ns[0]), dtype=complex)
        f.reshape(nb, -1)[:, sets[ik]] = psi[ik].T
        f = np.fft.fftn(np.fft.ifftn(f, axes=(1, 2, 3)) * V.reshape(ns[2], ns[1], ns[0]), axes=(1, 2, 3))
        ref = f.reshape(nb, -1)[:, sets[ik]].T + 0.5 * (gk[ik] ** 2).sum(1)[:, None] * psi[ik]
        if acc:
            ref = ref + old[ik]
        got = out[ik].download()
        assert np.abs(got - ref).max() <= (2e-5 if mixed else 1e-12) * np.abs(ref).max(), ik
    for d in dev + out:
        d.free()
    c.close()

def check_rho_batch(ns, sets, nb, mixed):
    from pwdft_hip._lib import PW_MIXED, DeviceMatrix, ptr
    rng = np.random.default_rng(3)
    nk = len(sets)
    c = context(ns, sets[0])
    for ik in range(1, nk):
        gk = rng.standard_normal((sets[ik].size, 3))
        c.call("pw_set_kpoint", ik, sets[ik].size, ptr(sets[ik]), 0, ptr(gk))
    psi = [rand(rng, s.size, nb) for s in sets]
    dev = [DeviceMatrix.from_host(c, p) for p in psi]
    w = np.ascontiguousarray(rng.random((nk, nb)))
    ld = np.array([p.shape[0] for p in psi], dtype=np.int64)
    pp = np.array([d.p.value for d in dev], dtype=np.uint64)
    iks = np.arange(nk, dtype=np.int32)
    N = int(np.prod(ns))
    got = np.empty(N)
    print(f"case rho batch {ns} nk={nk} nb={nb} mixed={mixed}", flush=True)
    c.call("pw_rhoe_zero")
    c.call("pw_rhoe_accum_batch_dev", nk, ptr(iks), nb, ptr(pp), ptr(ld), ptr(w),
           PW_MIXED if mixed else 0)
    c.call("pw_rhoe_get", ptr(got))
    ref = np.zeros(N)
    for ik in range(nk):
        f = np.zeros((nb, N), dtype=complex)
        f[:, sets[ik]] = psi[ik].T
        g = np.fft.ifftn(f.reshape(nb, ns[2], ns[1], ns[0]), axes=(1, 2, 3)).reshape(nb, N)
        ref += (w[ik][:, None] * np.abs(g) ** 2).sum(0)
    ref *= float(N) ** 2 / 3.7
    assert np.abs(got - ref).max() <= (2e-5 if mixed else 1e-12) * np.abs(ref).max()
    for d in dev:
        d.free()
    c.close()


@pytest.mark.parametrize("ns,nk,nb,mixed", [((20, 20, 20), 9, 3, False), ((27, 27, 27), 5, 7, True),
                                            ((36, 24, 45), 3, 5, False), ((24, 36, 20), 4, 40, True),
                                            ((125, 12, 12), 2, 2, False)])
def test_rho_batch(ns, nk, nb, mixed):
    """k-points with different index sets in the same launches (and, without a plan, one by one)."""
    check_rho_batch(ns, [index_set(ns, [(n - 1) // 4 - (ik % 2) for n in ns], shift=0.2 * ik / nk) for ik in range(nk)],
                    nb, mixed)


@pytest.mark.parametrize("mixed", [False, True])
def test_rho_batch_wide(mixed):
    """One k-point beyond the half-sphere window among others within it."""
    ns = (45, 36, 24)
    check_rho_batch(ns, [index_set(ns, [(0.3 if ik == 1 else 0.22) * n for n in ns]) for ik in range(3)], 4, mixed)


def test_rho_batch_workspace():
    """Fewer bands per launch than the default bound the batched density's work array: eight k-points of
    eight bands on 72^3 hold 8 x 8 MiB of transforms, one k-point's 8 MiB where the caller set 8 bands."""
    import ctypes
    from pwdft_hip._lib import DeviceMatrix, ptr
    hip = ctypes.CDLL("libamdhip64.so")
    ns, nk, nb = (72, 72, 72), 8, 8
    idx = index_set(ns, [17] * 3)
    w = np.ones((nk, nb))
    gk = np.ones((idx.size, 3))
    iks = np.arange(nk, dtype=np.int32)
    ld = np.full(nk, idx.size, dtype=np.int64)

    def free_bytes():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    grown, rho = {}, {}
    for bands in (64, nb):
        c = context(ns, idx)
        for ik in range(1, nk):
            c.call("pw_set_kpoint", ik, idx.size, ptr(idx), 0, ptr(gk))
        c.call("pw_set_band_batch", bands)
        dev = DeviceMatrix.from_host(c, rand(np.random.default_rng(9), idx.size, nb))
        pp = np.full(nk, dev.p.value, dtype=np.uint64)
        print(f"case rho batch workspace, {bands} bands a launch", flush=True)
        before = free_bytes()
        c.call("pw_rhoe_accum_batch_dev", nk, ptr(iks), nb, ptr(pp), ptr(ld), ptr(w), 0)
        grown[bands] = before - free_bytes()
        rho[bands] = np.empty(int(np.prod(ns)))
        c.call("pw_rhoe_get", ptr(rho[bands]))
        dev.free()
        c.close()
    assert np.abs(rho[64] - rho[nb]).max() <= 1e-12 * rho[nb].max()
    assert grown[nb] <= grown[64] - (40 << 20), grown
