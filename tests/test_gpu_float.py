"""GPU parity of the floating-point compute path (bfloat16 / float32 Dense, MatMul, Add) through the C ABI.

The oracle accumulates exactly and rounds once; the kernels accumulate in float32 in matrix-core order. Two
bars, both written out below: the tolerances of the reference's own float test (tests/test_float_sim.py:81-87:
rtol 1e-2 / atol 5e-2 for bfloat16, rtol 1e-3 / atol 1e-3 for float32), and the tighter forward error bound
of a float32 dot product plus one rounding to the output format.
"""

import numpy as np
import pytest

torch = pytest.importorskip('torch')

pytestmark = pytest.mark.gpu

# fp8: the reference has no fp8 test; the bar is one unit in the last place (relative 2^-3) of the output format
REF_TOL = {'bfloat16': (1e-2, 5e-2), 'float32': (1e-3, 1e-3), 'fp8_e4m3': (2.0 ** -3, 2.0 ** -9)}
TORCH_DT = {'bfloat16': torch.bfloat16, 'float32': torch.float32, 'fp8_e4m3': torch.float8_e4m3fn}
HALF_ULP = {'bfloat16': 2.0 ** -8, 'float32': 2.0 ** -24, 'fp8_e4m3': 2.0 ** -4}
FORMATS = ['bfloat16', 'float32', 'fp8_e4m3']


@pytest.fixture(scope='module')
def ops():
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from aie4ml_amd import ops as _ops

    return _ops


def operand(r, shape, fmt, oracle, scale=1.0):
    x = (r.normal(0, scale, shape)).astype(np.float32)
    if fmt == 'fp8_e4m3':
        return oracle.fp8_quantize(x)
    return oracle.bf16_truncate(x) if fmt == 'bfloat16' else x


def dev(a, fmt):
    if fmt == 'fp8_e4m3':  # by code: the values are exact in the format, the codes are the oracle's
        from oracle import oracle as o
        return torch.from_numpy(o.fp8_encode(np.ascontiguousarray(a, dtype=np.float32))).cuda().view(torch.float8_e4m3fn)
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(TORCH_DT[fmt])


def host(t):
    torch.cuda.synchronize()
    return t.float().cpu().numpy()


def check(got, exp, fmt, k, abs_products):
    rtol, atol = REF_TOL[fmt]
    np.testing.assert_allclose(got, exp, rtol=rtol, atol=atol)
    # float32 accumulation of k terms, any order: |err| <= k * 2^-24 * sum|a||w|; then one rounding of the
    # result (half an ulp), which can land on the neighbouring value when the two sums straddle a tie
    bound = 2.0 * HALF_ULP[fmt] * np.abs(exp) + (k + 2) * 2.0 ** -24 * abs_products + 1e-30
    if fmt == 'fp8_e4m3':
        bound = bound + 2.0 ** -9  # one step of the subnormal range
    assert np.all(np.abs(got.astype(np.float64) - exp.astype(np.float64)) <= bound)


@pytest.mark.parametrize('fmt', FORMATS)
@pytest.mark.parametrize('shape', [(4, 32, 32), (4, 32, 16), (7, 19, 5), (130, 96, 70), (256, 256, 256), (300, 128, 260),
                                   (512, 1024, 384), (1024, 64, 64)])
def test_dense_float(ops, oracle, fmt, shape):
    M, K, N = shape
    r = np.random.default_rng(M + K + N)
    A = operand(r, (M, K), fmt, oracle, 2.0)
    W = operand(r, (K, N), fmt, oracle, 0.1)
    b = r.normal(0, 0.05, N).astype(np.float32)
    absprod = np.abs(A).astype(np.float64) @ np.abs(W).astype(np.float64) + np.abs(b)
    p = ops.pack_dense_float(dev(W, fmt), torch.from_numpy(b).cuda())
    for relu in (False, True):
        got = host(ops.dense_float(dev(A, fmt), p, relu=relu))
        check(got, oracle.dense_float(A, W, b, relu=relu, fmt=fmt), fmt, K, absprod)
    p0 = ops.pack_dense_float(dev(W, fmt), None)
    check(host(ops.dense_float(dev(A, fmt), p0)), oracle.dense_float(A, W, None, fmt=fmt), fmt, K, absprod)


@pytest.mark.parametrize('fmt', FORMATS)
def test_dense_float_exact_cases(ops, oracle, fmt):
    # small integers: every product and partial sum is exact in float32, so any order gives the same bits
    r = np.random.default_rng(5)
    amax, wmax = (2, 1) if fmt == 'fp8_e4m3' else (8, 4)  # fp8: keep every sum below the largest value, 448
    A = r.integers(-amax, amax + 1, (200, 128)).astype(np.float32)
    W = r.integers(-wmax, wmax + 1, (128, 192)).astype(np.float32)
    b = r.integers(-16, 17, 192).astype(np.float32)
    p = ops.pack_dense_float(dev(W, fmt), torch.from_numpy(b).cuda())
    got = host(ops.dense_float(dev(A, fmt), p, relu=True))
    assert np.array_equal(got, oracle.dense_float(A, W, b, relu=True, fmt=fmt))
    # identity weights return the input; empty batch
    eye = np.eye(64, dtype=np.float32)
    X = operand(r, (33, 64), fmt, oracle)
    pe = ops.pack_dense_float(dev(eye, fmt), None)
    assert np.array_equal(host(ops.dense_float(dev(X, fmt), pe)), X)
    empty = ops.dense_float(torch.empty((0, 64), dtype=TORCH_DT[fmt], device='cuda'), pe)
    assert tuple(empty.shape) == (0, 64)


@pytest.mark.parametrize('fmt', FORMATS)
@pytest.mark.parametrize('trans_b', [True, False])
@pytest.mark.parametrize('shape', [((2, 3), 64, 64, 64), ((4,), 128, 96, 32), ((), 130, 70, 48), ((2,), 50, 17, 24),
                                   ((3,), 256, 128, 256)])
def test_matmul_float(ops, oracle, fmt, trans_b, shape):
    lead, M, K, N = shape
    r = np.random.default_rng(M * 3 + K + N)
    A = operand(r, lead + (M, K), fmt, oracle)
    B = operand(r, lead + ((N, K) if trans_b else (K, N)), fmt, oracle)
    got = host(ops.matmul_float(dev(A, fmt), dev(B, fmt), trans_b=trans_b))
    Bm = np.swapaxes(B, -1, -2) if trans_b else B
    absprod = np.abs(A).astype(np.float64) @ np.abs(Bm).astype(np.float64)
    check(got, oracle.matmul_float(A, B, trans_b=trans_b, fmt=fmt), fmt, K, absprod)


@pytest.mark.parametrize('fmt', FORMATS)
@pytest.mark.parametrize('shape', [((), 64, 64, 64), ((3,), 130, 70, 48), ((2,), 50, 17, 24), ((), 300, 256, 128)])
def test_transposed_lhs_in_kernel_float(ops, oracle, fmt, shape):
    """Float Dense and MatMul read a left operand stored as [..., K, M] themselves (TRANSPOSE_A, matmul.cpp:60-66,
    dense_bias_relu.cpp:95-101); same tolerances as the untransposed operand, against the oracle on the materialised
    transpose."""
    lead, M, K, N = shape
    r = np.random.default_rng(M * 5 + K + N)
    At = operand(r, lead + (K, M), fmt, oracle)
    A = np.ascontiguousarray(np.swapaxes(At, -1, -2))
    W = operand(r, (K, N), fmt, oracle, 0.1)
    b = r.normal(0, 0.05, N).astype(np.float32)
    p = ops.pack_dense_float(dev(W, fmt), torch.from_numpy(b).cuda())
    got = host(ops.dense_float(dev(At, fmt), p, relu=True, trans_a=True))
    absprod = np.abs(A).astype(np.float64) @ np.abs(W).astype(np.float64) + np.abs(b)
    want = oracle.dense_float(A.reshape(-1, K), W, b, relu=True, fmt=fmt).reshape(lead + (M, N))
    check(got, want, fmt, K, absprod)
    for trans_b in (True, False):
        B = operand(r, lead + ((N, K) if trans_b else (K, N)), fmt, oracle)
        got = host(ops.matmul_float(dev(At, fmt), dev(B, fmt), trans_b=trans_b, trans_a=True))
        Bm = np.swapaxes(B, -1, -2) if trans_b else B
        absprod = np.abs(A).astype(np.float64) @ np.abs(Bm).astype(np.float64)
        check(got, oracle.matmul_float(A, B, trans_b=trans_b, fmt=fmt), fmt, K, absprod)


@pytest.mark.parametrize('fmt', FORMATS)
def test_add_float(ops, oracle, fmt):
    r = np.random.default_rng(9)
    a = operand(r, (5, 1001), fmt, oracle, 3.0)
    b = operand(r, (5, 1001), fmt, oracle, 3.0)
    got = host(ops.add_float(dev(a, fmt), dev(b, fmt)))
    assert np.array_equal(got, oracle.add_float(a, b, fmt))  # one exact sum, one rounding: bit-exact


def test_float_argument_errors(ops):
    w = torch.zeros((8, 8), dtype=torch.float16, device='cuda')
    with pytest.raises(NotImplementedError):
        ops.pack_dense_float(w, None)
    p = ops.pack_dense_float(torch.zeros((8, 8), dtype=torch.bfloat16, device='cuda'), None)
    with pytest.raises(ValueError, match='share float precision'):
        ops.dense_float(torch.zeros((2, 8), dtype=torch.float32, device='cuda'), p)
    with pytest.raises(ValueError, match='features'):
        ops.dense_float(torch.zeros((2, 9), dtype=torch.bfloat16, device='cuda'), p)


@pytest.mark.parametrize('fmt', ['bfloat16', 'fp8_e4m3', 'float32'])
@pytest.mark.parametrize('K', [3, 7, 8, 9, 17, 33, 131, 300])
def test_dense_float_rows_at_any_address(ops, oracle, fmt, K):
    """A column window of a wider matrix whose other columns hold NaN: rows at any address, K around 16 bytes of operand and
    a K tile. Small integers, so every order of summation gives the same bits."""
    r = np.random.default_rng(K)
    A, W = (r.integers(-2, 3, sh).astype(np.float32) for sh in ((70, K), (K, 37)))
    t = {'bfloat16': torch.bfloat16, 'fp8_e4m3': torch.float8_e4m3fn, 'float32': torch.float32}[fmt]
    wide = torch.full((70, K + 3), float('nan')).to(t)
    wide[:, 1:K + 1] = torch.from_numpy(A).to(t)
    p = ops.pack_dense_float(torch.from_numpy(W).to(t).cuda(), None)
    got = ops.dense_float(wide.cuda()[:, 1:K + 1], p).float().cpu()
    want = torch.from_numpy(A @ W)  # exact; fp8 results up to 16 are, larger ones round to even or away from zero at ties
    if fmt == 'fp8_e4m3':
        exact = want.abs() <= 16
        got, want = got[exact], want[exact]
    assert torch.equal(got, want if fmt == 'float32' else want.to(t).float())


@pytest.mark.parametrize('fmt', FORMATS)
@pytest.mark.parametrize('M,K,N', [(1, 32, 8), (16, 1000, 40), (17, 129, 129), (64, 2048, 1024), (130, 96, 770), (512, 1536, 1024)])
def test_dense_float_with_few_output_tiles(ops, oracle, fmt, M, K, N):
    """The kernel for small outputs in the floating-point formats: every tile form, K on and off its tiles, bias and ReLU,
    against the oracle's exact sums within the bound on a float32 dot product in any order plus one rounding."""
    r = np.random.default_rng(M + K + N)
    A, W = operand(r, (M, K), fmt, oracle), operand(r, (K, N), fmt, oracle, 1.0 / np.sqrt(K))
    b = r.normal(0, 1, N).astype(np.float32)
    p = ops.pack_dense_float(dev(W, fmt), torch.from_numpy(b).cuda())
    for relu in (False, True):
        got = host(ops.dense_float(dev(A, fmt), p, relu=relu))
        check(got, oracle.dense_float(A, W, b, relu=relu, fmt=fmt), fmt, K, np.abs(A).astype(np.float64) @ np.abs(W) + np.abs(b))


@pytest.mark.parametrize('fmt', ['bfloat16', 'float32'])
@pytest.mark.parametrize('K', [32, 64, 96, 129, 200, 257, 320])
def test_dense_float_with_two_k_tiles_ahead(ops, oracle, fmt, K):
    """Enough output tiles for the tiled kernel, reductions of one to ten K tiles of 128 bytes, odd and even, whole and not,
    rows aligned and at odd elements with NaN around them. Small integers: every order of summation gives the same bits."""
    r = np.random.default_rng(K)
    M, N = 8200, 330
    A, W = (r.integers(-2, 3, sh).astype(np.float32) for sh in ((M, K), (K, N)))
    t = {'bfloat16': torch.bfloat16, 'float32': torch.float32}[fmt]
    wide = torch.full((M, K + 8), float('nan')).to(t)
    wide[:, 1:K + 1] = torch.from_numpy(A).to(t)
    p = ops.pack_dense_float(torch.from_numpy(W).to(t).cuda(), None)
    want = torch.from_numpy(A @ W).to(t)
    for x in (torch.from_numpy(A).to(t).cuda(), wide.cuda()[:, 1:K + 1]):
        assert torch.equal(ops.dense_float(x, p).cpu(), want), tuple(x.stride())


@pytest.mark.parametrize('fmt', FORMATS)
@pytest.mark.parametrize('K', [9, 33, 131, 300])
def test_matmul_float_in_place_operand_with_nan_behind_its_rows(ops, fmt, K):
    """A transposed right operand on 16-byte aligned rows whose pitch holds NaN past K: few output tiles, so the kernel
    whose waves share K reads it where it lies. Small integers: every order of summation gives the same bits."""
    from aie4ml_amd import _lib

    r = np.random.default_rng(K)
    M, N, t = 20, 37, TORCH_DT[fmt]
    A, B = (r.integers(-1, 2, sh).astype(np.float32) for sh in ((M, K), (N, K)))
    A[:, 16:] = 0  # sums up to 16: exact in every format
    ld = -(-K // 16) * 16
    wide = torch.full((N, ld), float('nan')).to(t)
    wide[:, :K] = torch.from_numpy(B).to(t)
    a, b = torch.from_numpy(A).to(t).cuda(), wide.cuda()
    out = torch.empty((M, N), dtype=t, device='cuda')
    _lib.check(_lib.load().a4g_matmul_f(ops._ptr(a), ops._float_format(a, 'a'), 0, K, M * K, ops._ptr(b), ld, N * ld, 1, ops._ptr(out), N,
                                        M * N, 1, M, N, K, None, 0, ops._stream()))
    assert torch.equal(out.float().cpu(), torch.from_numpy(A @ B.T))


@pytest.mark.parametrize('fmt', FORMATS)
@pytest.mark.parametrize('M,K,N', [(130, 96, 770), (90, 2000, 1300), (512, 1536, 1024), (300, 1100, 4200), (700, 2000, 2000), (300, 200, 3000)])
def test_dense_float_small_outputs_on_wider_tiles(ops, fmt, M, K, N):
    """The kernel for small outputs on its tiles of 32 x 16 (the first two sizes), 32 x 32 and 64 x 64 (the last three; float32 the
    last one): K and the output off them. Products of -1, 0 and 1 with at most sixteen that count per row: exact in every format."""
    r = np.random.default_rng(M + K)
    t = TORCH_DT[fmt]
    A, W = np.zeros((M, K), np.float32), r.integers(-1, 2, (K, N)).astype(np.float32)
    at = r.integers(0, K, (M, 16))
    A[np.arange(M)[:, None], at] = r.integers(-1, 2, (M, 16))
    p = ops.pack_dense_float(torch.from_numpy(W).to(t).cuda(), None)
    got = ops.dense_float(torch.from_numpy(A).to(t).cuda(), p)
    assert torch.equal(got.float().cpu(), torch.from_numpy(A @ W))


@pytest.mark.parametrize('M,N,K', [(8200, 330, 32), (8200, 330, 64), (8200, 330, 129), (8200, 330, 200), (8200, 330, 257), (8200, 330, 512), (8200, 330, 1025),
                                   (4096, 4096, 512), (4100, 4000, 640)])
def test_dense_fp8_on_many_tiles(ops, M, N, K):
    """fp8 with more outputs than the kernel for small ones takes: the tiled kernels of 128 x 128 and (the last two sizes) 256 x 256, K in
    whole tiles, in whole chunks and off them, rows aligned and at odd bytes between NaN. Exact products as above."""
    r = np.random.default_rng(M + K)
    t = torch.float8_e4m3fn
    A, W = np.zeros((M, K), np.float32), r.integers(-1, 2, (K, N)).astype(np.float32)
    at = r.integers(0, K, (M, 16))
    A[np.arange(M)[:, None], at] = r.integers(-1, 2, (M, 16))
    wide = torch.full((M, K + 3), float('nan')).to(t)
    wide[:, 1:K + 1] = torch.from_numpy(A).to(t)
    p = ops.pack_dense_float(torch.from_numpy(W).to(t).cuda(), None)
    want = torch.from_numpy(A @ W)
    for x in (torch.from_numpy(A).to(t).cuda(), wide.cuda()[:, 1:K + 1]):
        assert torch.equal(ops.dense_float(x, p).float().cpu(), want), tuple(x.stride())
