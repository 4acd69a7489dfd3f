"""The G(r) -> S(Q) transform entry and the reciprocal_space drop-in:
oracle pins on the CPU (closed forms, identities, float64 round trips) and
GPU parity of the HIP kernels against the oracle and NumPy."""
import numpy as np
import pytest

from fullrmc_amd.Core import reciprocal_space as grs
from oracle import chain
from oracle import reciprocal as orc

F32 = np.float32


def _ulps(a, b):
    a = np.asarray(a, F32).view(np.int32).astype(np.int64)
    b = np.asarray(b, F32).view(np.int32).astype(np.int64)
    a = np.where(a < 0, -(a & 0x7FFFFFFF), a)
    b = np.where(b < 0, -(b & 0x7FFFFFFF), b)
    return np.abs(a - b)


# ------------------------------------------------------------ oracle pins

def test_oracle_Gr_to_sq_single_shell_closed_form():
    """One non-zero G(r) bin at r0: S(q) = 1 + dr*sin(q*r0)/q*G0."""
    r = (0.05 + 0.1 * np.arange(60)).astype(F32)
    G = np.zeros(60, F32)
    G[23] = F32(2.5)
    q = np.linspace(0.3, 20, 40).astype(F32)
    S = orc.Gr_to_sq(r, G, q)
    q64 = q.astype(np.float64)
    ref = 1 + 0.1 * np.sin(q64 * float(r[23])) / q64 * 2.5
    assert np.max(np.abs(S - ref)) < 1e-6


def test_oracle_Gr_to_sq_matches_the_constraint_transform():
    """Gr_to_sq and the S(Q) constraints' matrix transform are the same sum
    up to float32 rounding (each pinned against float64)."""
    rng = np.random.default_rng(3)
    r = (0.01 + 0.02 * np.arange(250)).astype(F32)
    G = (rng.standard_normal(250) * np.exp(-r / 3)).astype(F32)
    q = np.linspace(0.5, 25, 60).astype(F32)
    S = orc.Gr_to_sq(r, G, q)
    S_m = np.sum(G.reshape((-1, 1)) * chain.sq_matrix(r, q), axis=0) + 1
    q64, r64 = q.astype(np.float64), r.astype(np.float64)
    S64 = 1 + (G.astype(np.float64)[:, None] * 0.02 * np.sin(np.outer(r64, q64)) / q64).sum(0)
    assert np.max(np.abs(S - S64)) < 2e-6 * (1 + np.max(np.abs(S64)))
    assert np.max(np.abs(S - S_m)) < 4e-6 * (1 + np.max(np.abs(S64)))


def test_oracle_gr_to_sq_is_Gr_to_sq_of_the_matching_G():
    """g(r) = 1 + G(r)/(4*PI*rho*r) gives the same S(q) through gr_to_sq as
    G(r) through Gr_to_sq (pins 4*PI*rho, the factor r and the -1)."""
    rng = np.random.default_rng(4)
    r = (0.05 + 0.1 * np.arange(120)).astype(F32)
    G = (rng.standard_normal(120) * 0.5).astype(F32)
    rho = F32(0.07)
    g = (1 + G.astype(np.float64) / (4 * np.pi * 0.07 * r.astype(np.float64))).astype(F32)
    q = np.linspace(0.4, 18, 50).astype(F32)
    a = orc.gr_to_sq(r, g, q, rho)
    b = orc.Gr_to_sq(r, G, q)
    assert np.max(np.abs(a - b)) < 2e-5 * (1 + np.max(np.abs(b)))


def test_oracle_sq_to_Gr_inverts_the_forward_transform():
    """A smooth G(r) through the forward sine transform (float64) and back
    through sq_to_Gr: G(r) = (2/PI) int Q (S-1) sin(Qr) dQ."""
    r = np.arange(0.0, 12.0, 0.01)
    G = np.exp(-((r - 3.0) ** 2) / (2 * 0.25 ** 2)) - 0.5 * np.exp(-((r - 5.0) ** 2) / (2 * 0.4 ** 2))
    q = np.arange(0.005, 40.0, 0.01)
    S = 1 + (G[:, None] * 0.01 * np.sin(np.outer(r, q)) / q).sum(0)
    rv = np.linspace(1.0, 8.0, 71).astype(F32)
    back = orc.sq_to_Gr(q.astype(F32), rv, S.astype(F32))
    ref = np.exp(-((rv - 3.0) ** 2) / (2 * 0.25 ** 2)) - 0.5 * np.exp(-((rv - 5.0) ** 2) / (2 * 0.4 ** 2))
    assert np.max(np.abs(back - ref)) < 2e-3


def test_argument_errors_match_reference_types():
    r = np.arange(5, dtype=F32)
    with pytest.raises(ValueError, match="Buffer dtype mismatch"):
        grs.Gr_to_sq(r.astype(np.float64), r, r)
    with pytest.raises(TypeError):
        grs.gr_to_sq(None, r, r, 1.0)
    with pytest.raises(ValueError, match="wrong number of dimensions"):
        grs.sq_to_Gr(r, r.reshape(5, 1), r)
    with pytest.raises(ValueError):
        grs.sq_transform(r, np.zeros((4, 3), F32))


# ------------------------------------------------------------- GPU parity

@pytest.mark.gpu
@pytest.mark.parametrize("k,H,nQ", [(1, 300, 7), (5, 1000, 500), (3, 4500, 300), (130, 700, 65)])
@pytest.mark.parametrize("addOne", [True, False])
def test_sq_transform_exact_is_numpy_axis0_sum(k, H, nQ, addOne):
    rng = np.random.default_rng(k * 7 + H)
    G = rng.standard_normal((k, H)).astype(F32)
    M = (rng.standard_normal((H, nQ)) * 0.02).astype(F32)
    S = grs.sq_transform(G, M, addOne=addOne)
    for p in range(k):
        ref = np.sum(G[p].reshape((-1, 1)) * M, axis=0)
        if addOne:
            ref = ref + 1
        assert S[p].tobytes() == ref.astype(F32).tobytes(), "curve %d" % p


@pytest.mark.gpu
def test_sq_transform_exact_zero_sign_and_the_constraint_S():
    # NumPy's reduction starts from +0: a sum of -0 products is +0
    H, nQ = 50, 9
    M = np.abs(np.random.default_rng(1).standard_normal((H, nQ))).astype(F32)
    G = np.full(H, -0.0, F32)
    S = grs.sq_transform(G, M, addOne=False)
    assert S.tobytes() == np.sum(G.reshape((-1, 1)) * M, axis=0).tobytes()
    assert not np.any(np.signbit(S))
    # the S(Q) constraint's own matrix and G(r)
    centers = (0.01 + 0.02 * np.arange(1000)).astype(F32)
    q = np.linspace(0.5, 25, 500).astype(F32)
    Mc = chain.sq_matrix(centers, q)
    Gc = (np.sin(centers) * np.exp(-centers / 5)).astype(F32)
    ref = np.sum(Gc.reshape((-1, 1)) * Mc, axis=0) + 1
    assert grs.sq_transform(Gc, Mc).tobytes() == ref.tobytes()


@pytest.mark.gpu
@pytest.mark.parametrize("k,H,nQ", [(1, 5, 3), (16, 64, 16), (37, 1003, 501), (128, 2000, 1000)])
def test_sq_transform_mfma_vs_float64(k, H, nQ):
    """Matrix-core contraction: within float32 accumulation error of the
    float64 product (bound: 1e-6 of the sum of |terms| per Q)."""
    rng = np.random.default_rng(H + nQ)
    G = rng.standard_normal((k, H)).astype(F32)
    M = (rng.standard_normal((H, nQ)) * 0.02).astype(F32)
    S = grs.sq_transform(G, M, addOne=True, mode="mfma")
    S64 = G.astype(np.float64) @ M.astype(np.float64) + 1
    scale = np.abs(G.astype(np.float64)) @ np.abs(M.astype(np.float64)) + 1
    assert np.max(np.abs(S - S64) / scale) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(2, 1), (120, 40), (2300, 37)])
def test_Gr_to_sq_and_gr_to_sq_vs_oracle(n, m):
    """Terms in double, float32 accumulator: the device and host double sin
    may differ in the last bit, which reaches the float32 result only at a
    rounding boundary; every value within 1 ulp, nearly all identical."""
    rng = np.random.default_rng(n + m)
    r = (0.05 + 0.1 * np.arange(n)).astype(F32)
    G = rng.standard_normal(n).astype(F32)
    q = np.linspace(0.3, 20, m).astype(F32)
    for got, ref in [(grs.Gr_to_sq(r, G, q), orc.Gr_to_sq(r, G, q)),
                     (grs.gr_to_sq(r, 1 + G, q, 0.05), orc.gr_to_sq(r, 1 + G, q, F32(0.05)))]:
        u = _ulps(got, ref)
        assert u.max() <= 1
        assert np.mean(u == 0) >= 0.99


@pytest.mark.gpu
def test_sq_to_Gr_vs_oracle():
    q = np.arange(0.01, 30.0, 0.02).astype(F32)
    S = (1 + np.sin(q) / q).astype(F32)
    rv = np.linspace(0.5, 10, 200).astype(F32)
    got = grs.sq_to_Gr(q, rv, S)
    ref = orc.sq_to_Gr(q, rv, S)
    assert _ulps(got, ref).max() <= 1 or np.max(np.abs(got - ref)) < 1e-6 * np.max(np.abs(ref))


@pytest.mark.gpu
@pytest.mark.parametrize("H", [1, 15, 63, 64, 65, 130, 200])
@pytest.mark.parametrize("k,nQ", [(1, 1), (3, 64), (5, 65), (33, 17), (2100, 3), (4101, 2)])
def test_sq_transform_edges_of_tiles(k, H, nQ):
    """Partly filled chunks of rows, tiles of Q and groups of curves (one, two and
    four per wave): the exact mode is the sequential sum bit for bit, the matrix cores
    stay within float32 rounding of the terms' magnitudes."""
    rng = np.random.default_rng(k + H + nQ)
    G = rng.standard_normal((k, H)).astype(F32)
    M = rng.standard_normal((H, nQ)).astype(F32)
    S = grs.sq_transform(G, M, addOne=False)
    ref = np.zeros((k, nQ), F32)
    for r in range(H):  # NumPy's axis-0 order (its sum of a single column would be pairwise)
        ref += G[:, r:r + 1] * M[r]
    assert S.tobytes() == ref.tobytes()
    T = grs.sq_transform(G, M, addOne=False, mode="mfma").astype(np.float64)
    exact, terms = G.astype(np.float64) @ M.astype(np.float64), np.abs(G).astype(np.float64) @ np.abs(M)
    # at most H roundings of 2^-24 relative to the sum of magnitudes, plus the products'
    assert np.all(np.abs(T - exact) <= (H + 1) * 2.0 ** -24 * terms)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [2097120, 2097153, 4194240])
def test_mfma_curves_past_the_rows_of_a_grid(k):
    """More curves than the tiles of one launch hold, up to the most that a call
    takes: each curve within float32 rounding, the ones after the first launch too;
    one more is refused."""
    from fullrmc_amd import _device as D, _lib
    rng = np.random.default_rng(k % 97)
    H, nQ = 5, 3
    G = rng.standard_normal((k, H)).astype(F32)
    M = rng.standard_normal((H, nQ)).astype(F32)
    S = grs.sq_transform(G, M, addOne=True, mode="mfma").astype(np.float64)
    exact, terms = G.astype(np.float64) @ M.astype(np.float64) + 1.0, np.abs(G).astype(np.float64) @ np.abs(M) + 1.0
    assert np.all(np.abs(S - exact) <= (H + 2) * 2.0 ** -24 * terms)
    if k == 4194240:
        d = D.empty((1,), F32)  # refused before anything is read
        for f in (_lib.lib().frmc_sq_transform, _lib.lib().frmc_sq_transform_noalloc):
            assert f(d.data_ptr(), k + 1, H, d.data_ptr(), nQ, 1, 1, d.data_ptr(), D.stream()) == 1


def _best_time(k, H, nQ, mode):
    import time

    import torch

    from fullrmc_amd import _lib
    G, M, S = (torch.ones(s, device="cuda") for s in ((k, H), (H, nQ), (k, nQ)))
    times = []
    for _ in range(5):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(10):
            _lib.check(_lib.lib().frmc_sq_transform(G.data_ptr(), k, H, M.data_ptr(), nQ, 1, mode, S.data_ptr(),
                                                    torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        times.append((time.perf_counter() - t0) / 10)
    return min(times)


@pytest.mark.gpu
@pytest.mark.parametrize("k,H,nQ", [(40, 64, 70), (40, 65, 70), (65, 5000, 33), (65, 5001, 33), (700, 130, 500),
                                    (701, 130, 511), (737, 130, 513), (257, 2500, 700), (70000, 100, 16),
                                    (70000, 100, 17), (3, 20001, 5), (2000, 8, 1000)])
def test_mfma_on_both_sides_of_the_tiles_lines(k, H, nQ):
    """Shapes around the lines between the two matrix-core kernels (one chunk of r,
    long r, many tiles, few Q): within float32 rounding, and the no-allocation entry
    gives the same bits where it takes the shape."""
    import torch

    from fullrmc_amd import _lib
    rng = np.random.default_rng(k + H + nQ)
    G = rng.standard_normal((k, H)).astype(F32)
    M = rng.standard_normal((H, nQ)).astype(F32)
    S = grs.sq_transform(G, M, addOne=False, mode="mfma")
    exact, terms = G.astype(np.float64) @ M.astype(np.float64), np.abs(G).astype(np.float64) @ np.abs(M)
    assert np.all(np.abs(S - exact) <= (H + 1) * 2.0 ** -24 * terms)
    dG, dM = torch.from_numpy(G).cuda(), torch.from_numpy(M).cuda()
    dS = torch.zeros((k, nQ), device="cuda")
    rc = _lib.lib().frmc_sq_transform_noalloc(dG.data_ptr(), k, H, dM.data_ptr(), nQ, 0, 1, dS.data_ptr(),
                                              torch.cuda.current_stream().cuda_stream)
    tiles = -(-k // 64) * -(-nQ // 64)
    parts = min(-(-1024 // tiles), -(-H // 64))
    per = -(-(-(-H // 64)) // parts) * 64
    parts = -(-H // per)
    assert rc == (0 if parts == 1 or parts * k * nQ <= 2 ** 22 else 1)
    if rc == 0:
        torch.cuda.synchronize()
        assert dS.cpu().numpy().tobytes() == S.tobytes()


@pytest.mark.gpu
def test_mfma_of_many_curves_or_long_ranges_uses_the_chip():
    """Short r ranges of many curves cost their stores (2,000 curves x 8 r x 1,000 Q
    took 76 us in small tiles, 10 in large ones), and one curve's long range is spread
    over the chip (60,000 r 241 us in one workgroup per tile, 49 over all)."""
    assert _best_time(2000, 8, 1000, 1) < 3 * _best_time(2000, 8, 16, 1)
    assert _best_time(1, 60000, 100, 1) < 5 * _best_time(1, 5000, 100, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("H", [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 79])
@pytest.mark.parametrize("k,nQ", [(1, 129), (5, 128), (40, 700), (65535, 130), (3000, 257)])
def test_exact_sums_of_few_rows(H, k, nQ):
    """Few rows, on both sides of the line to the staged form and of its sixteens:
    the sequential sum bit for bit."""
    rng = np.random.default_rng(H + k + nQ)
    G = rng.standard_normal((k, H)).astype(F32)
    M = rng.standard_normal((H, nQ)).astype(F32)
    ref = np.zeros((k, nQ), F32)
    for r in range(H):
        ref += G[:, r:r + 1] * M[r]
    assert grs.sq_transform(G, M, addOne=False).tobytes() == ref.tobytes()


@pytest.mark.gpu
def test_exact_sums_of_few_rows_cost_their_stores():
    """1,000 curves x 4,000 Q: 8 rows 15 us and 64 rows 28; both 28 when the staged form
    added 64 rows for 8."""
    assert _best_time(1000, 8, 4000, 0) < 0.8 * _best_time(1000, 64, 4000, 0)
