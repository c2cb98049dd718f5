"""fp32 contractions formed on the bf16 matrix cores (three bf16 pieces per
value, eight of nine piece products): the row layouts' wide tiles; the narrow
tiles and the weight gradients on fp32 MFMA beside them.

Bars: one product an output comes out within 0.51 of its last place (half from
the one rounding, 2^-7 at most from the smaller products' sum), whatever its
operands' magnitudes, so a piece product left out shows at every K; sums within
2^-24 (1 + sqrt(K) / 4) of float64 in norm (the leading products round once per
16 reduction elements, each time by half a last place at most) and within the
fp32 summation bound K 2^-24 sum |a b| element by element; the split tiles the
same bits, and the others; infinities and NaN where a float64 product of the
same operands has them (sums that are not finite are formed again in fp32)."""
import numpy as np
import pytest
import torch

from boonta_amd import _lib

pytestmark = pytest.mark.gpu


def gemm(al, bl, A, B, rows=None, splits=1, tile=-1):
    K = B.shape[0] if bl == 0 else B.shape[1]
    N = B.shape[1] if bl == 0 else B.shape[0]
    M = (A.shape[0] if rows is None else len(rows)) if al == 0 else A.shape[1]
    C = torch.empty(splits, M, N, device="cuda")
    _lib.call("ppo_gemm_f32", torch.cuda.current_stream().cuda_stream, al, bl, A.data_ptr(), A.stride(0),
              None if rows is None else rows.data_ptr(), B.data_ptr(), B.stride(0), C.data_ptr(), N, M, N, K, splits,
              M * N, 0, None, 0, None, None, 0, None, tile)
    return C.double().sum(0)


def operands(al, bl, M, N, K, seed, gather):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    n_rows = (M if al == 0 else K) + gather
    A = r(n_rows, K if al == 0 else M) * torch.exp(2 * r(n_rows, 1))
    B = (r(K, N) if bl == 0 else r(N, K)) * 0.06
    rows = torch.randperm(n_rows, device="cuda", generator=g)[:n_rows - gather].to(torch.int32) if gather else None
    return A, B, rows


def check(al, bl, A, B, rows, got):
    X = (A if rows is None else A[rows.long()]).double()
    X = X if al == 0 else X.t()
    Y = B.double() if bl == 0 else B.double().t()
    bound = X.shape[1] * 2.0 ** -24 * (X.abs() @ Y.abs())
    assert bool(((got - X @ Y).abs() <= bound + 1e-30).all())


SPLIT_TILES, FP32_TILES = (2, 8, 9), (0, 1, 3, -1)


@pytest.mark.parametrize("al, bl, M, N, K, splits, gather", [
    (0, 0, 8192, 256, 36, 1, 7), (0, 0, 8191, 256, 64, 1, 0), (0, 0, 1000, 96, 16, 1, 0),
    (0, 0, 16389, 132, 68, 1, 3), (0, 1, 8200, 260, 100, 1, 0), (0, 1, 300, 68, 4096, 1, 0),  # ragged rows, columns, stages
    (1, 0, 68, 260, 1000, 3, 5), (1, 0, 4, 4, 16, 1, 0), (1, 0, 400, 256, 4096, 8, 0), (1, 1, 36, 68, 200, 1, 0)])
def test_sums_stay_within_their_bound_of_float64_on_every_tile(al, bl, M, N, K, splits, gather):
    A, B, rows = operands(al, bl, M, N, K, M + K, gather)
    ref = gemm(al, bl, A, B, rows, splits, 3)
    check(al, bl, A, B, rows, ref)
    for t in FP32_TILES + (SPLIT_TILES if al == 1 else ()):
        assert torch.equal(gemm(al, bl, A, B, rows, splits, t), ref), t
    if al == 0:
        got = gemm(al, bl, A, B, rows, splits, 9)
        check(al, bl, A, B, rows, got)
        X, Y = (A if rows is None else A[rows.long()]).double(), B.double() if bl == 0 else B.double().t()
        want = X @ Y
        # (a row's own norm: the rows' scales differ)
        assert bool(((got - want).norm(dim=1) <= 2.0 ** -24 * (1 + K ** 0.5 / 4) * want.norm(dim=1)).all())
        for t in SPLIT_TILES:
            assert torch.equal(gemm(al, bl, A, B, rows, splits, t), got), t


def values(g, n, lo, hi):
    """Random mantissas and signs at exponents lo .. hi - 1 (exact float32, subnormals rounded)."""
    m = 1 + torch.randint(0, 1 << 23, n, device="cuda", generator=g).double() / (1 << 23)
    e = torch.randint(lo, hi, n, device="cuda", generator=g).double()
    return (m * torch.exp2(e) * (1 - 2 * torch.randint(0, 2, n, device="cuda", generator=g).double())).float()


@pytest.mark.parametrize("al, bl, tile", [(0, 0, 2), (0, 0, 9), (0, 1, 2), (0, 1, 8), (0, 0, 3), (1, 0, 2), (1, 0, 3)])
@pytest.mark.parametrize("K", [8, 64, 1000])
@pytest.mark.parametrize("ea, eb", [((0, 1), (0, 1)), ((-149, -110), (30, 60)), ((-126, -100), (20, 50)),
                                    ((60, 100), (-100, -60))])
def test_one_product_an_output_is_rounded_once(al, bl, tile, K, ea, eb):
    g = torch.Generator(device="cuda").manual_seed(K)
    M, N = 260, 132
    k = torch.arange(M, device="cuda") % K
    v, B = values(g, (M,), *ea), values(g, (K, N), *eb)
    if ea == (0, 1):  # the pieces past the first at their largest
        v[:K] = B[:, 0] = 1 + 2.0 ** -8 - 2.0 ** -17
    A = torch.zeros(M, K, device="cuda")
    A[torch.arange(M, device="cuda"), k] = v
    want = v.double()[:, None] * B.double()[k]
    got = gemm(al, bl, A if al == 0 else A.t().contiguous(), B if bl == 0 else B.t().contiguous(), tile=tile)
    ulp = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(2.0 ** -126))) - 23)
    assert float(((got - want).abs() / ulp).max()) <= 0.51


@pytest.mark.parametrize("al, bl, M, N, K, tile", [(0, 0, 8192, 256, 64, 9), (0, 1, 8192, 256, 64, 2),
                                                   (1, 0, 128, 64, 96, -1)])
def test_infinities_and_nans_come_out_where_float64_has_them(al, bl, M, N, K, tile):
    A, B, _ = operands(al, bl, M, N, K, 3, 0)
    at = (lambda m, k: (m, k)) if al == 0 else (lambda m, k: (k, m))
    A[at(5, 3)], A[at(40, 9)], A[at(41, 0)], A[at(100, K - 1)] = np.inf, -np.inf, np.nan, 3.4e38
    A[at(101, 2)], A[at(102, 5)], A[at(103, 1)] = 1e-42, 2.0 ** 90, -2.0 ** 110   # a subnormal; past the split's range
    B[(7, 33) if bl == 0 else (33, 7)] = np.inf
    B[(3, 34) if bl == 0 else (34, 3)] = 0.0   # inf * 0
    X, Y = (A if al == 0 else A.t()).double(), (B if bl == 0 else B.t()).double()
    want = (X.cpu().numpy() @ Y.cpu().numpy()).astype(np.float32)
    got = gemm(al, bl, A, B, tile=tile).float().cpu().numpy()
    fin = np.isfinite(want)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    bound = K * 2.0 ** -24 * (np.abs(X.cpu().numpy()) @ np.abs(Y.cpu().numpy()))
    assert (np.abs(got[fin].astype(np.float64) - want[fin]) <= bound[fin] + np.abs(want[fin]) * 2.0 ** -23).all()
