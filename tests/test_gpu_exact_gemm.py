"""GPU: the exact-activation GEMM (mnb_exact.hip) at the sizes where it can go
wrong: row tiles of 16 and 32 and their remainders, column tiles of 256, K
that ends inside a block, a word, a 64-k tile or a 256-k unit, one and several
K runs, launches of fewer rows than the call (a small workspace).

K not a multiple of 64 (three activation terms, every bit of A) against the
fp64 oracle at the decode bound 1e-5; accuracy_level 1 (two terms) bit for bit
against the decode kernels' groups of 16 rows. Every case prints its shape and
kernel before touching the GPU.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _plan(pkg, K, N, bs, zp, seed, level=0):
    p = pkg.workloads.Projection("exact", K, N, bs, zp)
    B, S, Z = pkg.workloads.make_weights(p, seed)
    return pkg.MatMulNBits(K, N, 4, bs, accuracy_level=level).prepare(B, S, Z), B, S, Z


@pytest.mark.parametrize("K,N,bs,zp,M", [
    (2817, 1, 32, True, 1),        # one column; K one past a step
    (65, 257, 32, False, 44),      # second 64-k tile of one value; one column past the tile
    (255, 255, 64, True, 16),      # a unit less one value; a full row tile of 16
    (257, 256, 128, True, 17),     # a second unit of one value; one row past the tile
    (1000, 300, 256, False, 31),   # blocks of a whole unit
    (1000, 300, 512, True, 33),    # blocks longer than a unit
    (5000, 70, 32, False, 64),     # many runs on one column tile
    (3100, 9000, 64, True, 300),   # every run in one workgroup
    (4128, 130, 128, True, 50),    # K an odd multiple of 32 (path 4)
])
@pytest.mark.parametrize("bias", [False, True])
def test_ragged_k(pkg, orc, cuda, K, N, bs, zp, M, bias):
    import torch
    op, B, S, Z = _plan(pkg, K, N, bs, zp, K + N + M)
    A = pkg.workloads.make_activations(M, K, 1.0, M + 1)
    b = np.random.default_rng(N).standard_normal(N).astype(np.float32)
    print(f"case exact ragged K={K} N={N} bs={bs} zp={zp} M={M} kernel={op.kernel_name(M)}",
          flush=True)
    assert op.kernel_name(M) == "ExactKernel"
    buf = torch.full((M * N + 8,), float("nan"), device=cuda)
    out = buf[4:4 + M * N].view(M, N)
    op(torch.from_numpy(A).to(cuda), out=out, bias=torch.from_numpy(b).to(cuda) if bias else None)
    Y = out.cpu().numpy()
    assert torch.isnan(buf[:4]).all() and torch.isnan(buf[4 + M * N:]).all()
    op.release()
    y64 = orc.matmul_nbits_f64(A, B, S, Z, K, N, bs) + (b.astype(np.float64) if bias else 0.0)
    assert orc.normwise_max_error(Y, y64) <= TOL


@pytest.mark.parametrize("K,N,bs,zp,M", [
    (512, 64, 32, True, 32),       # one row tile, one unit per wavefront and run
    (1088, 260, 64, False, 48),    # a last unit of one tile; 1.5 row tiles
    (4096, 6144, 32, True, 80),    # four runs, partial sums
    (4096, 14336, 256, True, 96),  # one run of eight ranges
    (14336, 4096, 128, True, 512),  # four runs in one workgroup
    (1024, 128, 128, True, 2064),  # two launches (2048 + 16 rows)
])
def test_level_1_groups_are_the_decode_kernels(pkg, cuda, K, N, bs, zp, M):
    import torch
    op, *_ = _plan(pkg, K, N, bs, zp, K + M, level=1)
    A = torch.from_numpy(pkg.workloads.make_activations(M, K, 1.0, M + 2)).to(cuda)
    print(f"case exact level 1 K={K} N={N} bs={bs} M={M} kernel={op.kernel_name(M)}", flush=True)
    assert op.kernel_name(M) == "ExactKernel"
    Y = op(A)
    for m0 in sorted({0, 16, M // 32 * 16, M - 16}):
        ref = op(A[m0:m0 + 16].contiguous(), path=pkg.PATH_GEMV)
        assert torch.equal(Y[m0:m0 + 16], ref), m0
    op.release()


def test_non_finite_rows(pkg, orc, cuda):
    """+inf, -inf and NaN keep the reference's kinds and stay in their row,
    also next to the values past K that a tile holds."""
    import torch
    K, N, bs, M = 1003, 70, 32, 20
    op, B, S, Z = _plan(pkg, K, N, bs, True, 5)
    A = pkg.workloads.make_activations(M, K, 1.0, 6)
    clean = op(torch.from_numpy(A).to(cuda)).cpu().numpy()
    bad = A.copy()
    bad[3, 37], bad[7, K - 1], bad[17, 5] = np.inf, -np.inf, np.nan
    print(f"case exact non-finite K={K} kernel={op.kernel_name(M)}", flush=True)
    Y = op(torch.from_numpy(bad).to(cuda)).cpu().numpy()
    op.release()
    rows = [3, 7, 17]
    keep = [m for m in range(M) if m not in rows]
    np.testing.assert_array_equal(Y[keep], clean[keep])
    ref = orc.matmul_nbits_ref_f32(bad[rows], B, S, Z, K, N, bs)
    for kind in (np.isposinf, np.isneginf, np.isnan):
        np.testing.assert_array_equal(kind(Y[rows]), kind(ref))


@pytest.mark.parametrize("K,level", [(1000, 0), (1024, 1)])
def test_small_workspaces(pkg, orc, cuda, K, level):
    """Less workspace than asked for: launches of fewer rows (every row the
    same bits), then the kernels without the image."""
    import torch
    N, bs, M = 192, 64, 200
    op, B, S, Z = _plan(pkg, K, N, bs, False, 9, level=level)
    A = pkg.workloads.make_activations(M, K, 1.0, 10)
    dA = torch.from_numpy(A).to(cuda)
    y64 = orc.matmul_nbits_f64(A, B, S, Z, K, N, bs)
    L = pkg.library()
    need = op.workspace_bytes(M)
    work = torch.empty(need, dtype=torch.uint8, device=cuda)
    for nbytes in (need, need // 2, need // 5, 0):
        Y = torch.full((M, N), float("nan"), device=cuda)
        print(f"case exact workspace K={K} {nbytes} of {need}: {op.kernel_name(M, nbytes)}", flush=True)
        st = L.mnb_run(op._plan, M, ctypes.c_void_p(dA.data_ptr()), ctypes.c_void_p(Y.data_ptr()),
                       ctypes.c_void_p(work.data_ptr()) if nbytes else None, nbytes,
                       ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert st == 0
        assert orc.normwise_max_error(Y.cpu().numpy(), y64) <= TOL
    op.release()


def test_gate_up_and_graph(pkg, orc, cuda):
    """The gate/up activation in the pass that adds the partial sums of two runs,
    and a captured call replayed on changed activations."""
    import torch
    K, I, bs, M = 1000, 100, 32, 40
    p = pkg.workloads.Projection("gu", K, I, bs, True)
    W = [pkg.workloads.make_weights(p, s) for s in (61, 62)]
    gu = pkg.GateUpSiLU(K, I, 4, bs).prepare(*W[0], *W[1])
    A = pkg.workloads.make_activations(M, K, 1.0, 63)
    dA = torch.from_numpy(A).to(cuda)
    out = torch.empty(M, I, device=cuda)
    print(f"case exact gate/up K={K} I={I} kernel={gu.kernel_name(M)}", flush=True)
    gu(dA, out=out)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        gu(dA, out=out)
    for seed in (63, 64, 65):
        A = pkg.workloads.make_activations(M, K, 1.0, seed)
        dA.copy_(torch.from_numpy(A))
        out.fill_(float("nan"))
        g.replay()
        h64 = orc.gate_up_silu_f64(A, *W[0], *W[1], K, I, bs)
        assert orc.normwise_max_error(out.cpu().numpy(), h64) <= 4 * TOL
    gu.release()


@pytest.mark.parametrize("K,I,bs,level,M", [
    (200, 300, 64, 0, 37),     # one unit; 88 columns in the third tile, 5 rows in the second
    (160, 33, 32, 0, 50),      # K an odd multiple of 32 (path 4), 66 columns
    (1000, 1555, 128, 0, 1000),  # 416 tiles: one run of four units
    (1024, 770, 64, 1, 2050),  # 448 tiles: every run in one workgroup; two rows by the decode kernels
])
def test_gate_up_in_the_epilogue(pkg, orc, cuda, K, I, bs, level, M):
    """The gate/up activation in ExactKernel's own stores, where one workgroup
    has all of K: half the columns, nothing written outside H."""
    import torch
    p = pkg.workloads.Projection("gu", K, I, bs, True)
    W = [pkg.workloads.make_weights(p, s) for s in (71, 72)]
    gu = pkg.GateUpSiLU(K, I, 4, bs, level).prepare(*W[0], *W[1])
    print(f"case exact gate/up epilogue K={K} I={I} M={M} kernel={gu.kernel_name(M)}", flush=True)
    assert gu.kernel_name(M) == "ExactKernel"
    A = pkg.workloads.make_activations(M, K, 1.0, 73)
    buf = torch.full((M * I + 8,), float("nan"), device=cuda)
    out = buf[4:4 + M * I].view(M, I)
    gu(torch.from_numpy(A).to(cuda), out=out)
    H = out.cpu().numpy()
    assert torch.isnan(buf[:4]).all() and torch.isnan(buf[4 + M * I:]).all()
    gu.release()
    assert np.isfinite(H).all()
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 48)), [M - 2, M - 1]]))
    h64 = orc.gate_up_silu_f64(A[rows], *W[0], *W[1], K, I, bs)
    assert orc.normwise_max_error(H[rows], h64) <= 4 * TOL


@pytest.mark.parametrize("top,route", [
    (1e32, "ExactKernel"),    # scales below 2^101: times the 2^27 of a unit's products finite
    (1e36, "GenericKernel"),  # above: a unit's sum before its exponent is undone would overflow
    (np.inf, "GenericKernel"),
])
def test_ragged_scales_at_the_end_of_the_range(pkg, orc, cuda, top, route):
    """Weight scales near fp32's largest with activations near its smallest:
    finite outputs stay finite, and an infinite scale gives its weight row the
    reference's kinds (it meets no value past K)."""
    import torch
    K, N, bs, M = 1060, 70, 32, 20
    p = pkg.workloads.Projection("scales", K, N, bs, True)
    B, S, Z = pkg.workloads.make_weights(p, 21)
    A = pkg.workloads.make_activations(M, K, 1.0, 22)
    if np.isinf(top):
        S[9, -1] = np.inf
        B[9, -1], Z[9, -1] = 0x99, 0x33  # q - zp = 6 in the last block: A's sign decides
        A[:, K // bs * bs:] = np.abs(A[:, K // bs * bs:]) + 0.5
    else:
        S[9] *= np.float32(top)
        A *= np.float32(1e-30)
    op = pkg.MatMulNBits(K, N, 4, bs).prepare(B, S, Z)
    name = op.kernel_name(M)
    print(f"case exact scales {top} kernel={name}", flush=True)
    Y = op(torch.from_numpy(A).to(cuda)).cpu().numpy()
    op.release()
    ref = orc.matmul_nbits_ref_f32(A, B, S, Z, K, N, bs)
    if np.isinf(top):
        assert np.isposinf(ref[:, 9]).all()
        np.testing.assert_array_equal(np.isposinf(Y), np.isposinf(ref))
        assert np.isfinite(np.delete(Y, 9, axis=1)).all()
    else:
        assert np.isfinite(ref).all() and np.isfinite(Y).all()
        y64 = orc.matmul_nbits_f64(A, B, S, Z, K, N, bs)
        for n in (9, 10):
            assert orc.normwise_max_error(Y[:, n:n + 1], y64[:, n:n + 1]) <= TOL
    assert name == route


def _graph_us(torch, call):
    """GPU time of a call in us: the least of 10 replays of a graph of 20."""
    call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(20):
            call()
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    best = float("inf")
    for _ in range(10):
        start.record()
        g.replay()
        end.record()
        end.synchronize()
        best = min(best, start.elapsed_time(end) * 50)
    return best


@pytest.mark.parametrize("K,N,bs,M", [
    (14336, 4096, 32, 32),  # the exact GEMM took 50% longer than two groups
    (14336, 4096, 32, 47),
    (4096, 28672, 128, 32),
    (2048, 2048, 128, 32),  # the exact GEMM's
])
def test_level_1_few_rows_take_the_faster_route(pkg, cuda, K, N, bs, M):
    """accuracy_level 1 at two or three groups of 16 rows: at most 15% more time
    than the decode kernel's groups one after the other."""
    import torch
    op, *_ = _plan(pkg, K, N, bs, True, K + N, level=1)
    A = torch.from_numpy(pkg.workloads.make_activations(M, K, 1.0, M)).to(cuda)
    out = torch.empty(M, N, device=cuda)
    print(f"case exact few rows K={K} N={N} M={M}: {op.kernel_name(M)}", flush=True)

    def groups():
        for m0 in range(0, M, 16):
            op(A[m0:m0 + 16], out=out[m0:m0 + 16], path=pkg.PATH_GEMV)

    auto = _graph_us(torch, lambda: op(A, out=out))
    ref = _graph_us(torch, groups)
    op.release()
    print(f"  automatic {auto:.1f} us, groups {ref:.1f} us")
    assert auto <= 1.15 * ref


@pytest.mark.parametrize("K,N,bs,zp", [
    (4096, 28676, 32, True),     # two column groups per decode workgroup, the last half empty
    (14336, 16260, 128, False),
    (2048, 65540, 64, True),
    (4096, 4096, 128, True),     # activations split in the decode kernel
])
def test_level_1_rows_are_the_decode_kernels_on_wide_weights(pkg, cuda, K, N, bs, zp):
    import torch
    M = 64
    op, *_ = _plan(pkg, K, N, bs, zp, K + M, level=1)
    A = torch.from_numpy(pkg.workloads.make_activations(M, K, 1.0, M + 2)).to(cuda)
    print(f"case exact wide K={K} N={N} bs={bs} kernel={op.kernel_name(M)}", flush=True)
    assert op.kernel_name(M) == "ExactKernel"
    Y = op(A)
    for m0 in range(0, M, 16):
        assert torch.equal(Y[m0:m0 + 16], op(A[m0:m0 + 16].contiguous(), path=pkg.PATH_GEMV)), m0
    op.release()


@pytest.mark.parametrize("K,N,M", [
    (2500, 500, 33),   # several K runs; two row tiles, the second of one row
    (2500, 5000, 20),
    (1004, 300, 17),   # the last unit and block filled in part
])
def test_rmsnorm_takes_the_exact_gemm(pkg, orc, cuda, K, N, M):
    """mnb_run_rmsnorm on K % 64 != 0: the automatic route of the plain call,
    which its workspace is sized for, on the normalized input."""
    import torch
    op, B, S, Z = _plan(pkg, K, N, 64, True, K + N + 5)
    X = torch.from_numpy(pkg.workloads.make_activations(M, K, 3.0, M)).to(cuda)
    gamma = np.random.default_rng(K).uniform(0.5, 1.5, K).astype(np.float32)
    print(f"case exact rmsnorm K={K} N={N} M={M} kernel={op.kernel_name(M)}", flush=True)
    assert op.kernel_name(M) == "ExactKernel"
    Y = op.run_rmsnorm(X, torch.from_numpy(gamma).to(cuda), 1e-5)
    # the normalized input as the call forms it, at the front of its workspace
    Xn = op._work[:M * K * 4].view(torch.float32).view(M, K).clone()
    plain = op(Xn)
    op.release()
    An = orc.rmsnorm_f64(X.cpu().numpy(), gamma, 1e-5)
    assert orc.normwise_max_error(Xn.cpu().numpy(), An) <= 1e-6
    assert torch.equal(Y, plain)
    y64 = orc.matmul_nbits_f64(An.astype(np.float32), B, S, Z, K, N, 64)
    assert orc.normwise_max_error(Y.cpu().numpy(), y64) <= 2 * TOL


@pytest.mark.parametrize("explicit", [False, True])
def test_ragged_calls_on_two_streams(pkg, cuda, explicit):
    """One object's calls of a K that 64 does not divide may overlap on several
    streams (the generic kernel needs no workspace; the exact GEMM's must not be
    shared): each stream has a workspace of its own, at most 8 are kept."""
    import torch
    K, N, M = 2500, 1501, 64
    p = pkg.workloads.Projection("two streams", K, N, 32, True)
    op = pkg.MatMulNBits(K, N, 4, 32).prepare(*pkg.workloads.make_weights(p, 7))
    print(f"case ragged two streams K={K} N={N} M={M} {op.kernel_name(M)}", flush=True)
    assert op.kernel_name(M) == "ExactKernel"
    As = [torch.from_numpy(pkg.workloads.make_activations(M, K, 1.0, s)).to(cuda) for s in (1, 2)]
    want = [op(A).cpu() for A in As]
    streams = [torch.cuda.Stream(device=cuda) for _ in range(9)]
    works = []
    for s in streams:
        with torch.cuda.stream(s):
            works.append(op.workspace(M, cuda))
    assert len({w.data_ptr() for w in works}) == 9 and len(op._works) == 8
    del works
    names = [op.workspace(M, d) for d in (cuda, "cuda:0", "cuda", torch.device("cuda"))]
    assert len({w.data_ptr() for w in names}) == 1  # one stream, one workspace
    outs = [[torch.empty(M, N, device=cuda) for _ in range(16)] for _ in As]
    torch.cuda.synchronize()
    for i in range(16):
        for A, s, out in zip(As, streams, outs):
            if explicit:
                op(A, out=out[i], stream=s)
            else:
                with torch.cuda.stream(s):
                    op(A, out=out[i])
    torch.cuda.synchronize()
    op.release()
    for w, out in zip(want, outs):
        assert all(torch.equal(o.cpu(), w) for o in out)


def test_gate_up_generic_path(pkg, orc, cuda):
    """The generic path chosen by the caller on a gate/up plan: its scratch sum is
    the one workspace that it needs."""
    import torch
    K, I, bs, M = 1000, 100, 32, 20
    p = pkg.workloads.Projection("gu", K, I, bs, True)
    W = [pkg.workloads.make_weights(p, s) for s in (81, 82)]
    gu = pkg.GateUpSiLU(K, I, 4, bs).prepare(*W[0], *W[1])
    A = pkg.workloads.make_activations(M, K, 1.0, 83)
    dA = torch.from_numpy(A).to(cuda)
    print(f"case gate/up generic K={K} I={I} M={M}", flush=True)
    H = gu(dA, path=pkg.PATH_GENERIC, stream=torch.cuda.current_stream()).cpu().numpy()
    gu.release()
    h64 = orc.gate_up_silu_f64(A, *W[0], *W[1], K, I, bs)
    assert orc.normwise_max_error(H, h64) <= 4 * TOL


def test_ragged_weights_of_18_gb(pkg, orc, cuda):
    """18 GB of weights: their re-laid copy has more than 2^32 words, and one
    launch has fewer threads than that. Columns from its start, its end and both
    sides of the word where the launch's threads would end."""
    import torch
    K, N, bs, M = 131073, 270000, 256, 2
    nb = -(-K // bs)
    if torch.cuda.mem_get_info(cuda)[0] < 40 << 30:
        pytest.skip("less than 40 GiB of device memory free")
    gen = torch.Generator(device=cuda).manual_seed(5)
    B = torch.randint(0, 256, (N, nb, bs // 2), dtype=torch.uint8, device=cuda, generator=gen)
    S = torch.rand((N, nb), device=cuda, generator=gen) * 0.015 + 0.005
    A = pkg.workloads.make_activations(M, K, 1.0, 6)
    print(f"case ragged 18 GB K={K} N={N} bs={bs} {B.numel()} bytes", flush=True)
    op = pkg.MatMulNBits(K, N, 4, bs).prepare_device(B, S)
    assert op.kernel_name(M) == "ExactKernel"
    Y = op(torch.from_numpy(A).to(cuda)).cpu().numpy()
    op.release()
    group = -(-K // 64) * 2 * 256  # words of 64 columns, which follow each other in the copy
    last = (-(-N // 256) * 4 * group - 2**32) // group * 64
    cols = [0, 1, last - 1, last, last + 64, last + 128, 131071, N - 1]
    y64 = orc.matmul_nbits_f64(A, B[cols].cpu().numpy(), S[cols].cpu().numpy(), None, K, len(cols), bs)
    del B, S
    torch.cuda.empty_cache()
    assert orc.normwise_max_error(Y[:, cols], y64) <= TOL


def test_ragged_weights_that_fit_once(pkg, orc, cuda):
    """Weights of 55% of the free device memory: no room for the exact GEMM's
    copy. The plan is created all the same and the generic kernel serves it."""
    import torch
    torch.cuda.empty_cache()
    K, bs = 131073, 256
    nb = -(-K // bs)
    N = int(torch.cuda.mem_get_info(cuda)[0] * 0.55) // (nb * bs // 2)
    if N >= 1 << 22:
        pytest.skip("more device memory than this width fills")
    B = torch.empty((N, nb, bs // 2), dtype=torch.uint8, device=cuda)
    S = torch.full((N, nb), 0.01, device=cuda)
    print(f"case ragged fits once K={K} N={N} bs={bs} {B.numel()} bytes", flush=True)
    op = pkg.MatMulNBits(K, N, 4, bs).prepare_device(B, S)
    assert op.kernel_name(1) == "GenericKernel"
    A = pkg.workloads.make_activations(1, K, 1.0, 8)
    Y = op(torch.from_numpy(A).to(cuda)).cpu().numpy()
    op.release()
    cols = [0, N // 2, N - 1]
    y64 = orc.matmul_nbits_f64(A, B[cols].cpu().numpy(), S[cols].cpu().numpy(), None, K, len(cols), bs)
    del B, S
    torch.cuda.empty_cache()
    assert np.abs(Y[:, cols] - y64).max() <= TOL * 8 * 0.01 * np.abs(A).sum()
