"""QRCP interpolation points on the GPU (thc_qrcp_points) against the oracle's
column-pivoted QR of the explicit orbital-product matrix
(src/qrcp.cpp:100-173)."""
import numpy as np
import pytest

from oracle import qrcp_oracle as QO
from thcpp_amd import _lib as L

pytestmark = pytest.mark.gpu


def _orbitals(n, m, seed):
    q, _ = np.linalg.qr(np.random.default_rng(seed).standard_normal((n, m)))
    return q


@pytest.mark.parametrize("n,m,k,seed", [(4096, 8, 24, 0), (3375, 10, 40, 1), (20000, 16, 100, 2)])
def test_qrcp_vs_oracle(ctx, n, m, k, seed):
    print("qrcp n=%d m=%d k=%d" % (n, m, k), flush=True)
    a = _orbitals(n, m, seed)
    st, idx, rd = ctx.qrcp_points(a, k)
    assert st == L.THC_OK
    ref_idx, ref_rd, _ = QO.qrcp_points(a, k)
    np.testing.assert_array_equal(idx.cpu().numpy(), ref_idx)
    # the Gram downdate carries the late residuals to about half the digits
    np.testing.assert_allclose(rd, ref_rd, rtol=1e-7)


def test_qrcp_half_rotated(ctx):
    a = _orbitals(5000, 12, 5)
    occ = np.ascontiguousarray(a[:, :5])
    st, idx, rd = ctx.qrcp_points(a, 30, occ)
    assert st == L.THC_OK
    ref_idx, ref_rd, _ = QO.qrcp_points(a, 30, occ)
    np.testing.assert_array_equal(idx.cpu().numpy(), ref_idx)
    np.testing.assert_allclose(rd, ref_rd, rtol=1e-7)


def test_qrcp_cfg0(ctx, cfg0):
    s = cfg0
    k = 4 * s.M
    st, idx, rd = ctx.qrcp_points(s.aoR, k)
    assert st == L.THC_OK
    ref_idx, ref_rd, _ = QO.qrcp_points(s.aoR, k)
    print("cfg0 qrcp |R_kk|/|R_00| = %.3e" % (rd[-1] / rd[0]))
    np.testing.assert_array_equal(idx.cpu().numpy(), ref_idx)


def test_qrcp_rank_exhausted(ctx):
    """M = 3 real orbitals span at most M (M + 1) / 2 = 6 product columns."""
    a = _orbitals(2000, 3, 7)
    st, _, _ = ctx.qrcp_points(a, 8)
    assert st == L.THC_ERR_NOT_POSDEF


def _complex_orbitals(n, m, seed):
    rng = np.random.default_rng(seed)
    q, _ = np.linalg.qr(rng.standard_normal((n, m)) + 1j * rng.standard_normal((n, m)))
    return q


@pytest.mark.parametrize("n,m,mo,k", [(4096, 8, 0, 30), (3375, 10, 4, 36), (20000, 12, 5, 60)])
def test_qrcp_complex_vs_oracle(ctx, n, m, mo, k):
    """Complex orbitals: |P|^2 pivots (mo = 0) and the complex Hermitian
    half-rotated Gram (mo occupied orbitals) against zgeqp3 of the explicit ZT."""
    print("complex qrcp n=%d m=%d m_occ=%d k=%d" % (n, m, mo, k), flush=True)
    a = _complex_orbitals(n, m, n + m)
    occ = np.ascontiguousarray(a[:, :mo]) if mo else None
    st, idx, rd = ctx.qrcp_points_complex(a, k, occ)
    assert st == L.THC_OK
    ref_idx, ref_rd, _ = QO.qrcp_points(a, k, occ)
    np.testing.assert_array_equal(idx.cpu().numpy(), ref_idx)
    np.testing.assert_allclose(rd, ref_rd, rtol=1e-7)


def test_qrcp_complex_real_orbitals_match_real_path(ctx):
    a = _orbitals(5000, 9, 6)
    occ = np.ascontiguousarray(a[:, :4])
    for o in (None, occ):
        st_r, idx_r, rd_r = ctx.qrcp_points(a, 25, o)
        st_c, idx_c, rd_c = ctx.qrcp_points_complex(a.astype(np.complex128), 25,
                                                    o.astype(np.complex128) if o is not None else None)
        assert st_r == L.THC_OK and st_c == L.THC_OK
        np.testing.assert_array_equal(idx_c.cpu().numpy(), idx_r.cpu().numpy())
        np.testing.assert_allclose(rd_c, rd_r, rtol=1e-12)


@pytest.mark.parametrize("n,m,mo,k", [(40, 6, 0, 21), (255, 9, 0, 40), (257, 5, 3, 12), (1030, 11, 0, 66),
                                      (5000, 30, 0, 300), (9001, 13, 7, 70)])
def test_qrcp_rounds_edges(ctx, n, m, mo, k):
    """Rounds of shared pivots at the edges: fewer points than candidates, k up to the rank M (M + 1) / 2, point
    counts either side of a workgroup's 256, orbital counts that are no multiple of 4, runs beyond one 16-pivot
    tile.  Residuals as separated as those of test_qrcp_vs_oracle, hence its tolerance."""
    print("qrcp rounds n=%d m=%d m_occ=%d k=%d" % (n, m, mo, k), flush=True)
    rng = np.random.default_rng(n + k)
    a = _orbitals(n, m, n + k) * rng.uniform(0.2, 1.0, (n, 1))
    occ = np.ascontiguousarray(a[:, :mo]) if mo else None
    st, idx, rd = ctx.qrcp_points(a, k, occ)
    assert st == L.THC_OK
    ref_idx, ref_rd, _ = QO.qrcp_points(a, k, occ)
    np.testing.assert_array_equal(idx.cpu().numpy(), ref_idx)
    np.testing.assert_allclose(rd, ref_rd, rtol=1e-7)


@pytest.mark.parametrize("repeat", [2, 300])
def test_qrcp_equal_points(ctx, repeat):
    """Points with the same orbital values have bit-equal residuals: the first one is the pivot (more of them than
    candidates fit in a round, with 300), and its copies never are."""
    a = _orbitals(40, 10, 11) * np.random.default_rng(4).uniform(0.3, 1.0, (40, 1))
    ref_idx, ref_rd, _ = QO.qrcp_points(a, 30)
    st, idx, rd = ctx.qrcp_points(np.repeat(a, repeat, axis=0), 30)
    assert st == L.THC_OK
    np.testing.assert_array_equal(idx.cpu().numpy(), repeat * ref_idx)
    np.testing.assert_allclose(rd, ref_rd, rtol=1e-7)


def test_qrcp_no_finite_residual(ctx):
    """All-zero and NaN orbitals have no pivot."""
    for fill in (0.0, np.nan):
        st, _, _ = ctx.qrcp_points(np.full((700, 4), fill), 3)
        assert st == L.THC_ERR_NOT_POSDEF


@pytest.mark.parametrize("m,copies,alone,k,half,cplx", [(10, 1100, 0, 40, False, False), (14, 400, 45, 64, False, False),
                                                        (14, 300, 70, 72, False, False), (12, 350, 60, 64, True, False),
                                                        (9, 300, 40, 64, False, True)])
def test_qrcp_equal_points_in_rounds(ctx, m, copies, alone, k, half, cplx):
    """More equal points than a round takes candidates, as symmetry gives, in runs long enough for rounds: the first
    copy of a point is the pivot; with points of their own between them the run changes between rounds and steps."""
    rng = np.random.default_rng(k + copies)
    base = 90 if alone else 45
    a = _orbitals(base, m, k) * rng.uniform(0.3, 1.0, (base, 1))
    if cplx:
        a = a * np.exp(2j * np.pi * rng.random(a.shape))
    reps = np.where(np.arange(base) % 90 < alone, 1, copies)[rng.permutation(base)]
    occ = np.ascontiguousarray(a[:, : m - 2]) if half else None
    big, bocc = np.repeat(a, reps, axis=0), None if occ is None else np.repeat(occ, reps, axis=0)
    assert k >= 64 or len(big) > 40000
    first = np.concatenate([[0], np.cumsum(reps)[:-1]])
    print("qrcp equal points: m=%d n=%d k=%d" % (m, len(big), k), flush=True)
    ref_idx, ref_rd, _ = QO.qrcp_points(a, k, occ)
    st, idx, rd = ctx.qrcp_points_complex(big, k) if cplx else ctx.qrcp_points(big, k, bocc)
    assert st == L.THC_OK
    np.testing.assert_array_equal(idx.cpu().numpy(), first[ref_idx])
    np.testing.assert_allclose(rd, ref_rd, rtol=1e-7)


@pytest.mark.parametrize("n,m,k,cplx", [(40001, 4, 4, False), (40001, 4, 5, False), (120001, 4, 1, False),
                                        (120001, 4, 2, False), (3000, 5, 8, True), (3000, 5, 9, True), (41000, 3, 4, True)])
def test_qrcp_few_pivots(ctx, n, m, k, cplx):
    """Either side of the point and pivot counts up to which a run goes one pivot a step."""
    print("qrcp few pivots n=%d m=%d k=%d" % (n, m, k), flush=True)
    a = (_complex_orbitals if cplx else _orbitals)(n, m, n + k)
    st, idx, rd = (ctx.qrcp_points_complex if cplx else ctx.qrcp_points)(a, k)
    assert st == L.THC_OK
    ref_idx, ref_rd, _ = QO.qrcp_points(a, k)
    np.testing.assert_array_equal(idx.cpu().numpy(), ref_idx)
    np.testing.assert_allclose(rd, ref_rd, rtol=1e-7)
