"""fp32 contractions formed on the bf16 matrix cores (three bf16 pieces per
value, six piece products): row-layout problems from 2^21 outputs on and every
weight gradient.

Bar: within the fp32 summation bound K 2^-24 sum |a b| of float64, element by
element; every tile of one problem the same bits; infinities and NaN where a
float64 product of the same operands has them (a split infinity has no finite
pieces, so such sums are formed again in fp32)."""
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


@pytest.mark.parametrize("al, bl, M, N, K, splits, gather", [
    (0, 0, 8192, 256, 36, 1, 7), (0, 0, 8191, 256, 64, 1, 0),   # either side of 2^21 outputs
    (0, 0, 16389, 132, 68, 1, 3), (0, 1, 8200, 260, 100, 1, 0),  # ragged rows, columns and stages
    (1, 0, 68, 260, 1000, 3, 5), (1, 0, 4, 4, 16, 1, 0), (1, 0, 400, 256, 4096, 8, 0), (1, 1, 36, 68, 200, 1, 0)])
def test_split_products_stay_within_the_fp32_bound_on_every_tile(al, bl, M, N, K, splits, gather):
    A, B, rows = operands(al, bl, M, N, K, M + K, gather)
    ref = gemm(al, bl, A, B, rows, splits, 3)
    check(al, bl, A, B, rows, ref)
    tiles = (0, 1, 2, 8, 9, -1) if al == 1 or M * N >= 1 << 21 else (0, -1)
    for t in tiles:
        assert torch.equal(gemm(al, bl, A, B, rows, splits, t), ref), t


@pytest.mark.parametrize("al, bl, M, N, K", [(0, 0, 8192, 256, 64), (0, 1, 8192, 256, 64), (1, 0, 128, 64, 96)])
def test_infinities_and_nans_come_out_where_float64_has_them(al, bl, M, N, K):
    A, B, _ = operands(al, bl, M, N, K, 3, 0)
    at = (lambda m, k: (m, k)) if al == 0 else (lambda m, k: (k, m))
    A[at(5, 3)], A[at(40, 9)], A[at(41, 0)], A[at(100, K - 1)] = np.inf, -np.inf, np.nan, 3.4e38
    A[at(101, 2)] = 1e-42   # a subnormal
    B[(7, 33) if bl == 0 else (33, 7)] = np.inf
    B[(3, 34) if bl == 0 else (34, 3)] = 0.0   # inf * 0
    X, Y = (A if al == 0 else A.t()).double(), (B if bl == 0 else B.t()).double()
    want = (X.cpu().numpy() @ Y.cpu().numpy()).astype(np.float32)
    got = gemm(al, bl, A, B).float().cpu().numpy()
    fin = np.isfinite(want)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    bound = K * 2.0 ** -24 * (np.abs(X.cpu().numpy()) @ np.abs(Y.cpu().numpy()))
    assert (np.abs(got[fin].astype(np.float64) - want[fin]) <= bound[fin] + np.abs(want[fin]) * 2.0 ** -23).all()
