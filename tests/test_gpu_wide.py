"""GPU parity of the wide-tile prefill kernel (WideKernel, 256 x 256 tiles).

It multiplies PrefillKernel's fp16 operands with fp32 accumulation over the
whole of K, so it is held to the GEMM's bound, ||y - y64||_2 / ||y64||_2 <=
2e-3 against the fp64 oracle, and to PrefillKernel's own result within 1e-4
(the order of the fp32 sums).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,bs,zp,M", [
    (2048, 24580, 32, True, 500),    # smallest K; 4 columns and 244 rows in the last tiles; 32-k blocks
    (2112, 12292, 64, False, 1030),  # odd tiles of K; 6 rows in the last row tile
    (2304, 28672, 256, True, 449),   # a scale per four k-tiles; 224 tiles: a contiguous run per XCD
    (4096, 4100, 128, False, 3700),  # 255 tiles, 4 columns in the last: no contiguous run per XCD
])
def test_wide_kernel(pkg, orc, cuda, K, N, bs, zp, M):
    """Edges of the 256-row and 256-column tiles, with the plain input, a bias
    and the RMSNorm input; rows of very different magnitude and a zero row."""
    import torch
    B, S, Z = pkg.workloads.make_weights(pkg.workloads.Projection("wide", K, N, bs, zp), K + N)
    op = pkg.MatMulNBits(K, N, 4, bs).prepare(B, S, Z)
    A = pkg.workloads.make_activations(M, K, 1.0, M)
    A[1] *= 1e20
    A[2] *= 1e-20
    A[3] = 0.0
    dA = torch.from_numpy(A).to(cuda)
    rng = np.random.default_rng(N)
    cols = np.unique(np.concatenate([rng.integers(0, N, 60), [0, 255, 256, N - 5, N - 1]]))
    rows = np.unique(np.concatenate([rng.integers(0, M, 40), [0, 1, 2, 255, 256, M - 1]]))
    print(f"case wide K={K} N={N} bs={bs} M={M} kernel={op.kernel_name(M)}", flush=True)
    assert op.kernel_name(M) == "WideKernel"
    ref = lambda X: orc.matmul_nbits_f64(X[rows], B[cols], S[cols], None if Z is None else Z[cols],
                                         K, len(cols), bs)

    def check(Y, want):
        for i, m in enumerate(rows):  # row by row: their magnitudes differ by 40 decades
            assert orc.l2_rel_error(Y[m:m + 1, cols], want[i:i + 1]) <= 2e-3, m

    Y = op(dA).cpu().numpy()
    check(Y, ref(A))
    assert not Y[3].any()
    Yp = op.run_kernel(dA, pkg.KERNEL_PREFILL).cpu().numpy()
    for m in (0, 1, 2, M // 2, M - 1):
        assert orc.l2_rel_error(Y[m:m + 1], Yp[m:m + 1]) <= 1e-4, m
    bias = rng.standard_normal(N).astype(np.float32)
    Yb = op(dA, bias=torch.from_numpy(bias).to(cuda)).cpu().numpy()
    np.testing.assert_array_equal(Yb, Y + bias[None, :])
    A[1] *= 1e-20  # squares in fp32's range
    A[2] *= 1e20
    gamma = rng.uniform(0.5, 1.5, K).astype(np.float32)
    Yn = op.run_rmsnorm(torch.from_numpy(A).to(cuda), torch.from_numpy(gamma).to(cuda), 1e-5)
    check(Yn.cpu().numpy(), ref(orc.rmsnorm_f64(A.astype(np.float64), gamma.astype(np.float64),
                                                1e-5).astype(np.float32)))
    op.release()


def test_wide_kernel_gate_up(pkg, cuda):
    """The gate/up activation in the stores: against the two projections run
    apart (each by its own kernel) and multiplied in fp64."""
    import torch
    K, N, bs, M = 2048, 12296, 64, 501
    mk = lambda seed: pkg.workloads.make_weights(pkg.workloads.Projection("gu", K, N, bs, True), seed)
    g, u = mk(1), mk(2)
    dA = torch.from_numpy(pkg.workloads.make_activations(M, K, 1.0, 3)).to(cuda)
    fused = pkg.GateUpSiLU(K, N, 4, bs).prepare(*g, *u)
    print(f"case wide gate/up K={K} N={N} M={M} kernel={fused.kernel_name(M)}", flush=True)
    assert fused.kernel_name(M) == "WideKernel"
    H = fused(dA).double()
    fused.release()
    y = []
    for w in (g, u):
        op = pkg.MatMulNBits(K, N, 4, bs).prepare(*w)
        y.append(op(dA).double())
        op.release()
    want = torch.nn.functional.silu(y[0]) * y[1]
    err = ((H - want).norm() / want.norm()).item()
    # both sides round the same operands to fp16; the sums' order and SiLU's fp32 differ
    assert err <= 1e-5, err
