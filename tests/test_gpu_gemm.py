"""pw_zgemm_dev against numpy at the edges of its tiles, of its k-steps and of the size rule
that picks a kernel.  The operands sit in larger arrays whose other entries are NaN, so a read
past a matrix that reaches a result shows.  Tolerances are those of the operator tests: 1e-14
(FP64) and 1e-5 (mixed) of max|A| max|B| sqrt(K)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16, 4), (15, 17, 3), (17, 1, 5), (1, 33, 127), (10, 8, 411), (40, 20, 4573), (31, 33, 2049),
          (65, 63, 515), (257, 160, 1633), (300, 243, 1000), (160, 160, 2625), (4000, 17, 31), (33000, 33, 64),
          (240, 240, 240), (409, 405, 411), (8, 8, 411), (9, 8, 2100), (8, 7, 3), (24, 24, 513), (1, 1, 1)]


def padded(rng, rows, cols, ld):
    a = np.full((ld, cols + 1), np.nan + 1j * np.nan, dtype=complex, order="F")
    a[:rows, :cols] = rng.standard_normal((rows, cols)) + 1j * rng.standard_normal((rows, cols))
    return a


@pytest.fixture(scope="module")
def ctx():
    import pwdft_hip as ph
    c = ph.Context()
    yield c
    c.close()


@pytest.mark.parametrize("tile", [-1, 6, 7])
@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_zgemm_edges(ctx, shape, transa, tile):
    from pwdft_hip._lib import DeviceMatrix, PW_MIXED, ptr
    M, N, K = shape
    if tile >= 0 and M > 1000:
        pytest.skip("large products: the default rule only")
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    ar, ac = (K, M) if transa else (M, K)
    A, B = padded(rng, ar, ac, ar + 3), padded(rng, K, N, K + 2)
    a, b = A[:ar, :ac], B[:K, :N]
    opA = a.conj().T if transa else a
    ref = (0.7 - 0.2j) * (opA @ b)
    alpha, zero = np.array([0.7, -0.2]), np.zeros(2)
    scale = np.abs(a).max() * np.abs(b).max() * np.sqrt(K)
    try:
        for key in (0, 1):
            ctx.call("pw_tune_set", key, tile)
        for mixed in (False, True):
            dA, dB = DeviceMatrix.from_host(ctx, A), DeviceMatrix.from_host(ctx, B)
            dC = DeviceMatrix.from_host(ctx, np.full((M + 1, N), np.nan, dtype=complex))
            print(f"case zgemm {shape} transa={transa} tile={tile} mixed={mixed}", flush=True)
            # beta = 0: what C held does not matter
            ctx.call("pw_zgemm_dev", transa, M, N, K, ptr(alpha), dA.p, dA.rows, dB.p, dB.rows,
                     ptr(zero), dC.p, M + 1, PW_MIXED if mixed else 0)
            got = dC.download()
            assert np.abs(got[:M] - ref).max() <= (1e-5 if mixed else 1e-14) * scale
            assert np.all(np.isnan(got[M])), "a row past C was written"
    finally:
        for key in (0, 1):
            ctx.call("pw_tune_set", key, -1)


# (tile code, split-BF16 switch, transa, (M, N, K)): the kernels of the mixed path over long and short K
F32_SUMS = [(-1, -1, 1, (500, 300, 9000)), (0, 0, 1, (700, 400, 12000)), (4, 0, 1, (300, 100, 9001)),
            (5, 1, 1, (700, 400, 12000)), (1, 1, 1, (500, 300, 9000)), (6, 0, 1, (40, 20, 30000)),
            (-1, -1, 0, (9000, 300, 500)), (0, 0, 0, (9000, 300, 500)), (0, 1, 0, (9000, 300, 500))]


@pytest.mark.parametrize("tile,split,transa,shape", F32_SUMS)
def test_f32_product_error(ctx, tile, split, transa, shape):
    """The 2-norm error of FP32 products against FP64: operands rounded to FP32 (u / sqrt(3) each, u =
    2^-24), sums in chains of at most 48 additions and second sums of at most 512: random roundings of
    the running sum, sqrt(48 / 6) u and sqrt(512 / 6) u at worst, are 10 u in quadrature; 8 u is asked,
    as no case here has more than 200 second additions (6 u)."""
    from pwdft_hip._lib import DeviceMatrix, PW_MIXED, ptr
    M, N, K = shape
    rng = np.random.default_rng(K)
    a = rng.standard_normal((K, M) if transa else (M, K)) + 1j * rng.standard_normal((K, M) if transa else (M, K))
    b = rng.standard_normal((K, N)) + 1j * rng.standard_normal((K, N))
    ref = (a.conj().T if transa else a) @ b
    one, zero = np.array([1.0, 0.0]), np.zeros(2)
    dA, dB, dC = DeviceMatrix.from_host(ctx, a), DeviceMatrix.from_host(ctx, b), DeviceMatrix(ctx, M, N)
    try:
        for key, value in ((0, tile), (1, tile), (8, split)):
            ctx.call("pw_tune_set", key, value)
        print(f"case zgemm FP32 sums {shape} transa={transa} tile={tile} split={split}", flush=True)
        ctx.call("pw_zgemm_dev", transa, M, N, K, ptr(one), dA.p, dA.rows, dB.p, dB.rows, ptr(zero), dC.p, M, PW_MIXED)
        got = dC.download()
    finally:
        for key in (0, 1, 8):
            ctx.call("pw_tune_set", key, -1)
    assert np.linalg.norm(got - ref) <= 8 * 2.0 ** -24 * np.linalg.norm(ref)
    for d in (dA, dB, dC):
        d.free()
