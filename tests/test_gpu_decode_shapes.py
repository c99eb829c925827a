"""GPU: DecodeFragKernel with two column groups per workgroup and with the
activations split inside the kernel, at the edges of both: an odd group count,
a last unit that K does not fill, one to four units per wavefront, rows 2 to
16. Against the fp64 oracle at the decode bound 1e-5, and bit for bit against
the exact GEMM's rows (accuracy_level 1), which are split by a kernel of their
own and multiplied group by group.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("K,N,bs,zp", [
    (4096, 28676, 32, True),     # pairs, 449 groups: the last workgroup's second group is padding
    (14336, 16260, 128, False),  # pairs, 255 groups, two runs of seven wavefronts of four units
    (2048, 65540, 64, True),     # single groups (four wavefronts), more than a round
    (4096, 4096, 128, True),     # split in the kernel, four runs
    (1088, 132, 64, False),      # split in the kernel, the last unit of one 64-k tile
    (512, 64, 32, True),         # split in the kernel, one group
])
def test_decode_shapes(pkg, orc, cuda, K, N, bs, zp):
    import torch
    p = pkg.workloads.Projection("decode", K, N, bs, zp)
    B, S, Z = pkg.workloads.make_weights(p, K + N)
    op = pkg.MatMulNBits(K, N, 4, bs, accuracy_level=1).prepare(B, S, Z)
    A = pkg.workloads.make_activations(32, K, 1.0, N)
    A[1] *= 1e-20
    A[2] = 0.0
    A[4, :min(256, K // 2)] *= 1e-6
    dA = torch.from_numpy(A).to(cuda)
    rng = np.random.default_rng(N)
    cols = np.unique(np.concatenate([rng.integers(0, N, 80), [0, 63, N - 1]]))
    bias = torch.from_numpy(rng.standard_normal(N).astype(np.float32)).to(cuda)
    gamma = rng.uniform(0.5, 1.5, K).astype(np.float32)
    ref = lambda X: orc.matmul_nbits_f64(X, B[cols], S[cols], None if Z is None else Z[cols],
                                         K, len(cols), bs)
    y64 = ref(A)
    print(f"case decode shapes K={K} N={N} bs={bs}: {op.kernel_name(16)}, {op.kernel_name(32)}",
          flush=True)
    exact = op(dA)
    for M in (2, 5, 8, 9, 16):
        buf = torch.full((M * N + 8,), float("nan"), device=cuda)
        Y = op(dA[:M].contiguous(), out=buf[4:4 + M * N].view(M, N), path=pkg.PATH_GEMV)
        assert torch.isnan(buf[:4]).all() and torch.isnan(buf[4 + M * N:]).all()
        y = Y.cpu().numpy()
        for m in range(M):
            if y64[m].any():
                assert orc.normwise_max_error(y[m:m + 1, cols], y64[m:m + 1]) <= TOL, (M, m)
            else:
                assert not y[m].any()
        Yb = op(dA[:M].contiguous(), path=pkg.PATH_GEMV, bias=bias)
        assert torch.equal(Yb, Y + bias), M
    if op.kernel_name(32) == "ExactKernel":
        for m0 in (0, 16):
            assert torch.equal(op(dA[m0:m0 + 16].contiguous(), path=pkg.PATH_GEMV),
                               exact[m0:m0 + 16])
    keep = [m for m in range(17) if m != 1]  # squares in fp32's range
    Yn = op.run_rmsnorm(dA[keep].contiguous(), torch.from_numpy(gamma).to(cuda), 1e-5).cpu().numpy()
    n64 = ref(orc.rmsnorm_f64(A[keep].astype(np.float64), gamma.astype(np.float64), 1e-5)
              .astype(np.float32))
    for i, m in enumerate(keep):
        if n64[i].any():
            assert orc.normwise_max_error(Yn[i:i + 1, cols], n64[i:i + 1]) <= TOL, m
    op.release()
