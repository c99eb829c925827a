// Prefill GEMM for MatMulNBits on CDNA4 fp16 MFMA (the roadmap's `int4_gemm`,
// docs/next_steps/2026/2026_08_qwen3_inference.rst:223-225).
//
// Y[M, N] = A[M, K] * W[N, K]^T with W dequantized from 4-bit blocks; fp16
// operands, fp32 accumulation. Two kernels per call:
//
// 1. ConvertAKernel rounds A to fp16 once (round to nearest even, as
//    onnx_light_cpu/impl/math/half_conversion.h:42-78) into the caller's
//    workspace, already laid out as the LDS image of each 128 x 64 A tile
//    (tile-major, rows swizzled as below, rows past M zero). Rounding A once
//    instead of once per N tile removes that work from the GEMM and halves the
//    A bytes it streams.
//
// 2. GemmKernel: one workgroup (256 threads, 4 wavefronts as 2 x 2) owns a
//    BM x 128 output tile (BM = 128, 64 or 32, by M); each wavefront a
//    BM/2 x 64 sub-tile of v_mfma_f32_16x16x32_f16 tiles. K advances in
//    k-tiles of 64, optionally split over several workgroups (split-K; the
//    partial sums are added in split order by SplitReduceKernel). 80 KiB of
//    LDS per workgroup (BM = 128) lets two workgroups share a CU, so one
//    hides the other's barrier and dequantization stalls.
//    - A tiles go global -> LDS directly (global_load_lds_dwordx4 through
//      inline asm, no registers) into a 3-stage ring, two k-tiles ahead.
//    - B tiles: each thread loads 32 nibbles of one weight row into
//      registers four k-tiles ahead, dequantizes them one k-tile ahead into a
//      double-buffered LDS tile (DequantWord: masks and fp16 exponent
//      constants give 1024 + q and 64 + q exactly, a packed add of the
//      matching -(1024 + zp) or -(64 + zp) makes q - zp exact, one packed
//      multiply by the block's fp16 scale rounds the weight once).
//    - One barrier per k-tile; the loop is written so that the compiler's
//      own waits never drain the prefetch (see the pipeline comment below).
//    Inside every group of 8 k the LDS order is [0,4,1,5,2,6,3,7] for both A
//    and B (the order the masked words produce); the contraction is unchanged.
//    LDS rows are 64 fp16 = 8 units of 16 B; unit u of row r is stored at
//    r * 8 + (u ^ ((r >> 1) & 7)), so the 16 lanes of an MFMA fragment read
//    (16 consecutive rows, one unit) hit 16 distinct 16-byte bank groups.
//    Tile order is XCD-aware: workgroup b runs on XCD b % 8; when the M tiles
//    split evenly over the 8 XCDs, XCD x gets a contiguous band of M tiles with
//    all their N tiles, so each XCD's L2 holds one slab of A.
#include "mnb_gemm_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace mnb {
namespace {

using namespace gemm;

constexpr int kMaxBM = 128;  // largest tile height; the workspace pads M to it
constexpr int kBN = 128;
constexpr int kBUnits = kBN * kUnits;       // units per B tile (16 KiB)
constexpr int kAStages = 3;
// Output tiles are BM x 128 with BM in {32, 64, 128}; A tiles BM x 64 fp16.
template <int BM>
constexpr int AUnits() { return BM * kUnits; }  // units per A tile
template <int BM>
constexpr size_t LdsBytes() { return (kAStages * AUnits<BM>() + 2 * kBUnits) * 16; }  // <= 80 KiB

// Largest value over the 256 threads of a workgroup (4 wavefronts); every
// thread gets it. `red` holds 4 floats of LDS.
__device__ __forceinline__ float BlockMax256(float v, float *red) {
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  __syncthreads();  // red may still be read by an earlier reduction
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__device__ __forceinline__ float BlockSum256(float v, float *red) {
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// One workgroup per row of A (rows past M, up to the tile padding, are written
// as zeros). The row is scaled by 2^f, f = RangeExponent(max_k |A[m][k]|, 14),
// and rounded to fp16 (round to nearest even, as FloatToFloat16Bits,
// onnx_light_cpu/impl/math/half_conversion.h:42-78): no finite input becomes
// inf, and only values below 2^-24 of the row's largest magnitude flush to
// zero. f goes to row_exp[m]; the GEMM's epilogue multiplies by 2^-f. Each
// 16-byte unit holds 8 consecutive k in [0,4,1,5,2,6,3,7] order and lands
// where GemmKernel's direct copy expects it.
// With gamma (RMSNorm folded in), the row is x * gamma * inv_rms with
// inv_rms = 1 / sqrt(mean_k x^2 + eps) reduced here as well.
// NV > 0: each thread keeps its NV units of the row in registers between the
// reduction and the conversion (K <= 2048 NV); NV = 0 reads the row twice.
template <int BM, int NV, bool RMS>
__global__ __launch_bounds__(256) void ConvertAKernel(const float *__restrict__ A,
                                                      uint4 *__restrict__ Ah,
                                                      int *__restrict__ row_exp, int M, int K,
                                                      const float *__restrict__ gamma,
                                                      float eps) {
  __shared__ float red[4];
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const int units = K / 8;
  const int ktiles = K / kBK;
  const int mt = row / BM;
  const int r = row - mt * BM;
  uint4 *base = Ah + static_cast<size_t>(mt) * ktiles * AUnits<BM>();
  auto dst = [&](int u) -> uint4 & { return base[(u / kUnits) * AUnits<BM>() + Swz(r, u % kUnits)]; };
  if (row >= M) {
    for (int u = tid; u < units; u += 256) dst(u) = make_uint4(0u, 0u, 0u, 0u);
    if (tid == 0) row_exp[row] = 0;
    return;
  }
  const float *src = A + static_cast<size_t>(row) * K;
  auto load = [&](int u, float4 &x, float4 &y, float &amax, float &ss) {
    x = reinterpret_cast<const float4 *>(src + 8 * u)[0];
    y = reinterpret_cast<const float4 *>(src + 8 * u)[1];
    if constexpr (RMS) {
      ss += ((x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w)) +
            ((y.x * y.x + y.y * y.y) + (y.z * y.z + y.w * y.w));
      const float4 g0 = reinterpret_cast<const float4 *>(gamma + 8 * u)[0];
      const float4 g1 = reinterpret_cast<const float4 *>(gamma + 8 * u)[1];
      x = make_float4(x.x * g0.x, x.y * g0.y, x.z * g0.z, x.w * g0.w);
      y = make_float4(y.x * g1.x, y.y * g1.y, y.z * g1.z, y.w * g1.w);
    }
    amax = fmaxf(amax, fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
    amax = fmaxf(amax, fmaxf(fmaxf(fabsf(y.x), fabsf(y.y)), fmaxf(fabsf(y.z), fabsf(y.w))));
  };
  // x * mul, then * 2^f (exact): the value FloatToFloat16Bits rounds
  auto store = [&](int u, float4 x, float4 y, float mul, int f) {
    if constexpr (RMS) {
      x = make_float4(x.x * mul, x.y * mul, x.z * mul, x.w * mul);
      y = make_float4(y.x * mul, y.y * mul, y.z * mul, y.w * mul);
    }
    auto sc = [f](float v) { return __builtin_amdgcn_ldexpf(v, f); };
    dst(u) = make_uint4(PackHalf2(sc(x.x), sc(y.x)), PackHalf2(sc(x.y), sc(y.y)),
                        PackHalf2(sc(x.z), sc(y.z)), PackHalf2(sc(x.w), sc(y.w)));
  };
  float amax = 0.0f, ss = 0.0f;
  float4 kx[NV > 0 ? NV : 1], ky[NV > 0 ? NV : 1];
  if constexpr (NV > 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int u = tid + 256 * i;
      if (u < units) load(u, kx[i], ky[i], amax, ss);
    }
  } else {
    for (int u = tid; u < units; u += 256) load(u, kx[0], ky[0], amax, ss);
  }
  amax = BlockMax256(amax, red);
  float mul = 1.0f;
  if constexpr (RMS) {
    mul = 1.0f / sqrtf(BlockSum256(ss, red) / static_cast<float>(K) + eps);
    amax *= mul;
  }
  const int f = RangeExponent(amax, kRowExpTarget);
  if (tid == 0) row_exp[row] = f;
  if constexpr (NV > 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int u = tid + 256 * i;
      if (u < units) store(u, kx[i], ky[i], mul, f);
    }
  } else {
    for (int u = tid; u < units; u += 256) {
      float dummy_a = 0.0f, dummy_s = 0.0f;
      float4 x, y;
      load(u, x, y, dummy_a, dummy_s);
      store(u, x, y, mul, f);
    }
  }
}

// StreamKernel's conversion of A: one workgroup of 4 wavefronts per (chunk of
// kChunkK k, kChunkRows rows), a thread 8 k of one row. Each row's chunk is
// scaled by 2^f, f = RangeExponent of the chunk's largest magnitude
// (StreamKernel's wavefronts stay inside one chunk and undo f in their sums),
// rounded to fp16 as ConvertAKernel does and written into 1 KiB operand records
// of 16 rows: no row-wide reduction. With gamma (RMSNorm folded in) the values
// are x * gamma and sq receives each row's sum of x^2 over the chunk, from which
// StreamKernel forms 1 / rms. A CU reads and writes kChunkRows x 3 KiB: with 16
// rows per workgroup a few CUs had four times that to do (K = 4096
// at M = 33 to 48 3.5 us, now 2.9).
constexpr int kChunkRows = 4;
constexpr int kChunkK = 512;
template <bool RMS>
__global__ __launch_bounds__(256) void ConvertChunkKernel(const float *__restrict__ A,
                                                          uint4 *__restrict__ img,
                                                          int *__restrict__ exps,
                                                          float *__restrict__ sq,
                                                          const float *__restrict__ gamma, int M,
                                                          int K, int chunks, int rows_padded) {
  __shared__ float red[4][kChunkRows], reds[RMS ? 4 : 1][kChunkRows];
  const int ch = static_cast<int>(blockIdx.x) % chunks;
  const int m0 = static_cast<int>(blockIdx.x) / chunks * kChunkRows;
  const int tid = threadIdx.x, wave = tid >> 6;
  const int r = tid % kChunkRows, unit = tid / kChunkRows;
  const int T = K / 32;
  const int s = ch * (kChunkK / 32) + unit / 4;
  const int rows = min(kChunkRows, M - m0);  // <= 0: padding rows, zeros
  const int bytes = max(rows, 0) * K * 4;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(A + static_cast<size_t>(min(m0, M - 1)) * K), 0, bytes, 0x00020000);
  // rows past M and steps past K read beyond the buffer: zeros
  const int k = 32 * s + 8 * (unit % 4);
  const int vo = r < rows && s < T ? (r * K + k) * 4 : bytes;
  floatx4 x[2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
    x[p] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ra, vo + 16 * p, 0, 0));
  if constexpr (RMS) {
    const floatx4 *gp = reinterpret_cast<const floatx4 *>(gamma + min(k, K - 8));
    const floatx4 g0 = gp[0], g1 = gp[1];
    float q = 0.0f;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int v = 0; v < 4; ++v) q += x[p][v] * x[p][v];
    x[0] *= g0;
    x[1] *= g1;
#pragma unroll
    for (int o = kChunkRows; o < 64; o *= 2) q += __shfl_xor(q, o, 64);
    if ((tid & 63) < kChunkRows) reds[wave][r] = q;
  }
  float amax = 0.0f;
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int v = 0; v < 4; ++v) amax = fmaxf(amax, fabsf(x[p][v]));
#pragma unroll
  for (int o = kChunkRows; o < 64; o *= 2) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
  if ((tid & 63) < kChunkRows) red[wave][r] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) amax = fmaxf(amax, red[w][r]);
  const int f = RangeExponent(amax, kRowExpTarget);
  if (tid < kChunkRows) {
    exps[ch * rows_padded + m0 + r] = f;
    if constexpr (RMS)
      sq[ch * rows_padded + m0 + r] = (reds[0][r] + reds[1][r]) + (reds[2][r] + reds[3][r]);
  }
  auto sc = [f](float v) { return __builtin_amdgcn_ldexpf(v, f); };
  if (s < T)
    img[(static_cast<size_t>(m0 / 16) * T + s) * 64 + 16 * (unit % 4) + m0 % 16 + r] =
        make_uint4(PackHalf2(sc(x[0][0]), sc(x[1][0])), PackHalf2(sc(x[0][1]), sc(x[1][1])),
                   PackHalf2(sc(x[0][2]), sc(x[1][2])), PackHalf2(sc(x[0][3]), sc(x[1][3])));
}

// One k-tile of B for this thread: 32 nibbles of one weight row (one
// quantization block, block_size >= 32), its scale, and the byte holding its
// zero point with the nibble's shift. The nibble is extracted only when the
// tile is dequantized: extracting it at load time would make the compiler wait
// for the load right after issuing it.
struct BRegs {
  uint4 b;
  float s;
  uint32_t z;
  uint32_t zshift;
};

template <int BM, bool HAS_ZP>
__global__ __launch_bounds__(256, 2) void GemmKernel(const uint4 *__restrict__ Ah,
                                                     const uint8_t *__restrict__ B,
                                                     const float *__restrict__ S,
                                                     const uint8_t *__restrict__ Z,
                                                     float *__restrict__ Y, int M, int K, int N,
                                                     int nb, int log2_bs, int row_bytes,
                                                     int zp_row_bytes, int kt_per_split,
                                                     float *__restrict__ partials,
                                                     float *__restrict__ H,
                                                     const int *__restrict__ row_exp,
                                                     const int *__restrict__ col_exp) {
  extern __shared__ uint4 lds[];
  constexpr int kAUnits = AUnits<BM>();
  uint4 *Astage = lds;                        // [kAStages][kAUnits]
  uint4 *Bbuf = lds + kAStages * kAUnits;     // [2][kBUnits]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1;
  const int wn = wave & 1;

  // Workgroup b computes output tile b % tiles over the k-tiles of split
  // b / tiles. XCD-aware tile order.
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = (N + kBN - 1) / kBN;
  const int split = static_cast<int>(blockIdx.x) / (tiles_m * tiles_n);
  int tm, tn;
  {
    const int b = static_cast<int>(blockIdx.x) - split * tiles_m * tiles_n;
    if (tiles_m % 8 == 0) {
      const int xcd = b & 7, local = b >> 3;
      const int band = tiles_m / 8;
      tm = xcd * band + local / tiles_n;
      tn = local % tiles_n;
    } else {
      tm = b / tiles_n;
      tn = b % tiles_n;
    }
  }
  const int m0 = tm * BM;
  const int n0 = tn * kBN;
  // This split's k-tiles: kt0 .. kt0 + ktiles - 1 (the host leaves no split empty).
  const int kt0 = split * kt_per_split;
  const int ktiles = min(kt_per_split, K / kBK - kt0);

  // B resources based at this tile's first weight row; rows past N read as
  // zero and their outputs are never stored.
  const int rows_b = min(kBN, N - n0);
  const auto rb_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t *>(B + static_cast<size_t>(n0) * row_bytes), 0, rows_b * row_bytes,
      0x00020000);
  const auto rs_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(S + static_cast<size_t>(n0) * nb), 0, rows_b * nb * 4, 0x00020000);
  const auto rz_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t *>(HAS_ZP ? Z + static_cast<size_t>(n0) * zp_row_bytes : B), 0,
      HAS_ZP ? rows_b * zp_row_bytes : 0, 0x00020000);

  // A: converted tile (tm, kt) is kAUnits contiguous units; instruction i of
  // wavefront w copies units i*256 + w*64 + lane to the same LDS offsets.
  const uint4 *a_tiles = Ah + (static_cast<size_t>(tm) * (K / kBK) + kt0) * kAUnits;
  // The copies go through CopyToLds16: with the builtin, the compiler waits
  // for every outstanding load (s_waitcnt vmcnt(0)) before the next LDS read,
  // which would stall each k-tile's MFMAs on the loads of tile kt + 2. The
  // WaitVm + barrier at the top of each iteration covers the copies.
  const uint32_t lds_a = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(Astage)) +
                         __builtin_amdgcn_readfirstlane(wave) * 64 * 16;  // uniform
  const uint4 *a_src = a_tiles + wave * 64 + lane;
  auto issue_a = [&](int kt, int stage) {
    const uint4 *src = a_src + static_cast<size_t>(kt) * kAUnits;
#pragma unroll
    for (int i = 0; i < kAUnits / 256; ++i)
      CopyToLds16(src + i * 256, lds_a + (stage * kAUnits + i * 256) * 16);
  };

  // B: thread t -> weight row t >> 1, 32 nibbles at k offset 32 * (t & 1).
  // Buffer offsets are a per-thread constant (voffset) plus the k-tile's
  // uniform part (soffset), so the loads cost no address arithmetic. The
  // block of the thread's 32 nibbles is blk_u + blk_l: blk_u = (k-tile start)
  // >> log2_bs, plus the thread's half when blocks are 32 wide (then blk_u is
  // even, so the zero-point byte is blk_u >> 1 and the nibble blk_l).
  const int b_row = tid >> 1;
  const int b_half = tid & 1;
  const int blk_l = log2_bs == 5 ? b_half : 0;
  const int vo_b = b_row * row_bytes + 16 * b_half;
  const int vo_s = (b_row * nb + blk_l) * 4;
  const int vo_z = b_row * zp_row_bytes;
  auto load_b = [&](BRegs &r, int kt) {
    const int kg = kt0 + kt;
    const int blk_u = (kg * kBK) >> log2_bs;
    r.b = __builtin_bit_cast(uint4,
                             __builtin_amdgcn_raw_buffer_load_b128(rb_rsrc, vo_b, kg * 32, 0));
    r.s = __builtin_bit_cast(float,
                             __builtin_amdgcn_raw_buffer_load_b32(rs_rsrc, vo_s, blk_u * 4, 0));
    if (HAS_ZP) {
      r.z = __builtin_amdgcn_raw_buffer_load_b8(rz_rsrc, vo_z, blk_u >> 1, 0);
      r.zshift = ((blk_u & 1) + blk_l) * 4;
    } else {
      r.z = 8u;
      r.zshift = 0;
    }
  };
  const Masks dq = MakeMasks();
  // The weight row's power-of-two exponent (plan time): its block scales times
  // 2^e_b are normal fp16 numbers and (q - zp) * scale stays below 65504.
  const int e_b = col_exp[min(n0 + b_row, N - 1)];
  auto store_b = [&](const BRegs &r, int buf) {
    const uint32_t words[4] = {r.b.x, r.b.y, r.b.z, r.b.w};
    const DequantRow dr =
        MakeDequantRow(__builtin_amdgcn_ldexpf(r.s, e_b), (r.z >> r.zshift) & 0xFu);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      Bbuf[buf * kBUnits + Swz(b_row, 4 * b_half + u)] = DequantWord(words[u], dr, dq);
  };

  constexpr int kMI = BM / 32;  // 16-row MFMA tiles per wavefront along M
  floatx4 acc[kMI][4];
#pragma unroll
  for (int i = 0; i < kMI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto mma_tile = [&](int stage, int buf) {
    const uint4 *as = Astage + stage * kAUnits;
    const uint4 *bs = Bbuf + buf * kBUnits;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int unit = 4 * ks + (lane >> 4);
      half8 bf[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bf[j] = __builtin_bit_cast(half8, bs[Swz(wn * 64 + j * 16 + (lane & 15), unit)]);
#pragma unroll
      for (int i = 0; i < kMI; ++i) {
        const half8 af =
            __builtin_bit_cast(half8, as[Swz(wm * (BM / 2) + i * 16 + (lane & 15), unit)]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf[j], acc[i][j], 0, 0, 0);
      }
    }
  };

  // Pipeline: A tile t is copied to LDS stage t % 3 two k-tiles ahead; the B
  // registers of tile t are loaded kPD k-tiles ahead (HBM latency under load
  // is several k-tiles long) and dequantized into LDS buffer t % 2 one k-tile
  // ahead. Iteration t:
  //  1. wait until A tile t (and with it B tile t+1) has landed, then a
  //     barrier: A tile t and B buffer t % 2 are complete and visible, and
  //     every read of stage (t+2) % 3 and buffer (t+1) % 2 from iteration
  //     t-1 is retired;
  //  2. dequantize B tile t+1 into buffer (t+1) % 2;
  //  3. copy A tile t+2, load the B registers of tile t+kPD into the set that
  //     held tile t;
  //  4. multiply tile t.
  // Every copy, load and store is issued unconditionally, with the k-tile
  // index clamped to the last one (the tail re-reads the last tile into
  // buffers nobody reads again): a branch around a load makes the compiler
  // wait for all outstanding loads where the paths join. So per iteration the
  // vector memory operations are exactly [kAOps A copies, kBOps B loads], and
  // after A tile t come B tile t+2, A tile t+1 and B tile t+3.
  constexpr int kPD = 4;
  constexpr int kAOps = kAUnits / 256;
  constexpr int kBOps = HAS_ZP ? 3 : 2;
  const int klast = ktiles - 1;
  BRegs rb[kPD];
  issue_a(0, 0);
  load_b(rb[0], 0);
  load_b(rb[1], min(1, klast));
  issue_a(min(1, klast), 1);
#pragma unroll
  for (int p = 2; p < kPD; ++p) load_b(rb[p], min(p, klast));
  store_b(rb[0], 0);

  // One iteration; u = t % kPD is a compile-time constant so the register
  // sets are static.
  auto step = [&](int t, auto uc) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    // Nothing crosses the wait and barrier at the top of an iteration:
    // hoisted above them, the tile's dequantization would make the compiler
    // wait for its B registers with a count that ignores the A copies (it
    // cannot see them), i.e. for the copies just issued.
    __builtin_amdgcn_sched_barrier(0);
    WaitVm<2 * kBOps + kAOps>();
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    store_b(rb[(u + 1) % kPD], (t + 1) & 1);
    issue_a(min(t + 2, klast), (t + 2) % kAStages);
    load_b(rb[u], min(t + kPD, klast));
    mma_tile(t % kAStages, t & 1);
  };
  // Whole groups of kPD iterations, then the remainder: a loop body with an
  // exit in the middle would merge different sets of outstanding loads at the
  // back edge, and the compiler would wait for all of them there.
  int kt = 0;
  for (; kt + kPD <= ktiles; kt += kPD) {
    step(kt, std::integral_constant<int, 0>{});
    step(kt + 1, std::integral_constant<int, 1>{});
    step(kt + 2, std::integral_constant<int, 2>{});
    step(kt + 3, std::integral_constant<int, 3>{});
  }
  if (kt < ktiles) step(kt, std::integral_constant<int, 0>{});
  if (kt + 1 < ktiles) step(kt + 1, std::integral_constant<int, 1>{});
  if (kt + 2 < ktiles) step(kt + 2, std::integral_constant<int, 2>{});
  // The remainder steps' B loads feed no later tile, so the compiler would
  // drop them, and from the second remainder step on the wait at a step's
  // top (which counts kBOps loads per step) would no longer cover that step's
  // A copy: a wavefront could read an A stage before the copy landed (seen as
  // one 8-row x 64-column block of an output tile off by a k-tile's share,
  // intermittently, with split K). Using the registers here keeps every load.
#pragma unroll
  for (int p = 0; p < kPD; ++p)
    __asm__ volatile("" ::"v"(rb[p].b.x), "v"(rb[p].b.y), "v"(rb[p].b.z), "v"(rb[p].b.w),
                     "v"(rb[p].s), "v"(rb[p].z));
  // No copy into this workgroup's LDS may land after it exits.
  WaitVm<0>();

  // Output: split 0 writes Y, split s > 0 of a split-K launch its partial sum
  // at partials + (s - 1) * M * N. Lane holds column (lane & 15), rows
  // 4*(lane >> 4) + v of each 16 x 16 tile. The accumulators are in units of
  // 2^(f_m + e_n) (A row m scaled by 2^f_m, weight row n by 2^e_n): one ldexp
  // per element undoes both exactly (a single rounding, only if the result is
  // an fp32 subnormal).
  {
    int ec[4], er[kMI][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) ec[j] = col_exp[min(n0 + wn * 64 + j * 16 + (lane & 15), N - 1)];
#pragma unroll
    for (int i = 0; i < kMI; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        er[i][v] = row_exp[m0 + wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + v];
#pragma unroll
    for (int i = 0; i < kMI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc[i][j][v] = __builtin_amdgcn_ldexpf(acc[i][j][v], -(er[i][v] + ec[j]));
  }
  if (H != nullptr) {
    // Gate/up epilogue of a one-split launch. Column gn + 1 (the up of gate
    // gn, N even) is held by lane ^ 1 for the same four rows v = 0..3; the
    // even lane finishes rows 0 and 1 of each fragment, the odd lane rows 2
    // and 3, each receiving the two values it lacks through one DPP swap.
    // Stores are buffer stores at byte offsets from this tile's first output
    // row: rows past M fall beyond the resource and columns past N are sent
    // there, so nothing branches (the host fuses only when M * N / 2 * 4 <
    // 2^31 and N < 2^22, so a tile's offsets stay below 2^30).
    const int half_n = N >> 1;
    const bool odd = (lane & 1) != 0;
    const auto hr = __builtin_amdgcn_make_buffer_rsrc(
        H + static_cast<size_t>(m0) * half_n, 0, min(M - m0, BM) * half_n * 4, 0x00020000);
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const floatx4 a = acc[i][j];
        const float r0 = PairSwap(odd ? a[0] : a[2]);
        const float r1 = PairSwap(odd ? a[1] : a[3]);
        const float h0 = odd ? SiluMul(r0, a[2]) : SiluMul(a[0], r0);
        const float h1 = odd ? SiluMul(r1, a[3]) : SiluMul(a[1], r1);
        const int gn = n0 + wn * 64 + j * 16 + (lane & 15);
        const int row = wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + (odd ? 2 : 0);
        const int off = gn < N ? (row * half_n + (gn >> 1)) * 4 : 0x7FFFFFF0;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, h0), hr, off, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, h1), hr,
                                              gn < N ? off + half_n * 4 : off, 0, 0);
      }
    }
    return;
  }
  if (split > 0) Y = partials + static_cast<size_t>(split - 1) * M * N;
  if (N < (1 << 22)) {
    // Buffer stores at byte offsets from this tile's first output row (below
    // 2^31 for N < 2^22): rows past M fall beyond the resource and columns
    // past N are sent there, so no store needs a branch.
    const auto yr = __builtin_amdgcn_make_buffer_rsrc(Y + static_cast<size_t>(m0) * N, 0,
                                                      min(M - m0, BM) * N * 4, 0x00020000);
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int gn = n0 + wn * 64 + j * 16 + (lane & 15);
        const int row = wm * (BM / 2) + i * 16 + 4 * (lane >> 4);
        const int off = gn < N ? (row * N + gn) * 4 : 0x7FFFFFF0;
        // (one element of the MFMA result vector at a time, through a scalar:
        // a bit cast of the vector element itself was compiled into a store of
        // element 0 for every v on ROCm 7.2)
        const floatx4 a = acc[i][j];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float val = a[v];
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(val), yr,
                                                gn < N ? off + v * N * 4 : off, 0, 0);
        }
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < kMI; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gn = n0 + wn * 64 + j * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gm = m0 + wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + v;
        if (gm < M && gn < N) Y[static_cast<size_t>(gm) * N + gn] = acc[i][j][v];
      }
    }
  }
}

// Split-K epilogue: Y += partials[0] + ... + partials[PARTS - 1], summed in
// that order for every element, so results do not depend on scheduling; then
// + bias[n] when a bias is given (Y is [mn / N, N]), after the sum, as a
// separate bias pass would add it. PARTS is a template argument so that every
// load is in flight before the first add (one HBM round trip per thread, not
// PARTS of them).
template <bool VEC, int PARTS>
__global__ __launch_bounds__(256) void SplitReduceKernel(float *__restrict__ Y,
                                                         const float *__restrict__ P,
                                                         int64_t mn, float *__restrict__ H,
                                                         const float *__restrict__ bias,
                                                         int64_t N) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * (VEC ? 4 : 1);
  if (i >= mn) return;
  if constexpr (VEC) {
    f32x4 v[PARTS];
#pragma unroll
    for (int p = 0; p < PARTS; ++p)
      v[p] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(P + p * mn + i));
    f32x4 y = *reinterpret_cast<const f32x4 *>(Y + i);
#pragma unroll
    for (int p = 0; p < PARTS; ++p) y += v[p];
    if (bias != nullptr) {  // N % 4 == 0 on this path: the 4 elements share a row
      const int64_t n = i % N;
      y += f32x4{bias[n], bias[n + 1], bias[n + 2], bias[n + 3]};
    }
    if (H != nullptr)  // gate/up pairs (N even: a pair never straddles rows)
      *reinterpret_cast<float2 *>(H + i / 2) = make_float2(SiluMul(y[0], y[1]), SiluMul(y[2], y[3]));
    else
      *reinterpret_cast<f32x4 *>(Y + i) = y;
  } else {
    float v[PARTS];
#pragma unroll
    for (int p = 0; p < PARTS; ++p) v[p] = __builtin_nontemporal_load(P + p * mn + i);
    float y = Y[i];
#pragma unroll
    for (int p = 0; p < PARTS; ++p) y += v[p];
    if (bias != nullptr) y += bias[i % N];
    if (H != nullptr) {
      // mn is even: lanes i and i ^ 1 are both in range, in the same wavefront
      const float other = PairSwap(y);
      if ((i & 1) == 0) H[i / 2] = SiluMul(y, other);
    } else {
      Y[i] = y;
    }
  }
}

template <int PARTS>
hipError_t LaunchReduce(float *Y, const float *P, int64_t mn, hipStream_t s, float *H,
                        const float *bias, int64_t N) {
  if (mn % 4 == 0 && reinterpret_cast<uintptr_t>(Y) % 16 == 0 &&
      reinterpret_cast<uintptr_t>(H) % 8 == 0 && (bias == nullptr || N % 4 == 0)) {
    hipLaunchKernelGGL((SplitReduceKernel<true, PARTS>),
                       dim3(static_cast<unsigned>((mn / 4 + 255) / 256)), dim3(256), 0, s, Y, P,
                       mn, H, bias, N);
  } else {
    hipLaunchKernelGGL((SplitReduceKernel<false, PARTS>),
                       dim3(static_cast<unsigned>((mn + 255) / 256)), dim3(256), 0, s, Y, P, mn,
                       H, bias, N);
  }
  return hipGetLastError();
}

template <int... Ps>
hipError_t DispatchReduce(int parts, float *Y, const float *P, int64_t mn, hipStream_t s,
                          float *H, std::integer_sequence<int, Ps...>, const float *bias = nullptr,
                          int64_t N = 1) {
  hipError_t e = hipErrorInvalidValue;
  (void)((parts == Ps + 1 ? (e = LaunchReduce<Ps + 1>(Y, P, mn, s, H, bias, N), true) : false) ||
         ...);
  return e;
}

constexpr int kMaxSplits = 16;

struct Shape {
  int bm;      // tile height: 32, 64 or 128
  int splits;  // K splits, each a contiguous run of kt_per_split k-tiles
  int kt_per_split;
};

// Normalises a requested split count: no split is left without k-tiles.
inline Shape MakeShape(const WeightView &w, int bm, int splits) {
  const int ktiles = static_cast<int>(w.K / kBK);
  splits = std::max(1, std::min({splits, ktiles, kMaxSplits}));
  const int per = (ktiles + splits - 1) / splits;
  return Shape{bm, (ktiles + per - 1) / per, per};
}

inline int64_t PaddedRows(int64_t M) { return (M + kMaxBM - 1) / kMaxBM * kMaxBM; }

// The workspace starts with the fp16 image of A (every tile height's padding
// is covered by kMaxBM), then the rows' power-of-two exponents (int32 per
// padded row, rounded up to 256 bytes), then the split-K partial sums.
inline size_t AImageBytes(const WeightView &w, int64_t M) {
  return static_cast<size_t>(PaddedRows(M)) * static_cast<size_t>(w.K) * 2;
}

inline size_t RowExpBytes(int64_t M) {
  return (static_cast<size_t>(PaddedRows(M)) * 4 + 255) / 256 * 256;
}
// StreamKernel (at most 64 rows): an exponent and a sum of squares per row and
// chunk of K.
inline size_t StreamExpBytes(const WeightView &w, int64_t M) {
  return RowExpBytes(M) * static_cast<size_t>((w.K + kChunkK - 1) / kChunkK);
}

inline size_t PartialBytes(const WeightView &w, int64_t M, const Shape &sh) {
  return static_cast<size_t>(sh.splits - 1) * static_cast<size_t>(M) * w.N * 4;
}

template <int BM, bool HAS_ZP>
hipError_t LaunchT(const WeightView &w, int64_t M, const uint4 *Ah, float *Y, float *partials,
                   const Shape &sh, hipStream_t s, float *H, const int *row_exp) {
  const int tiles = static_cast<int>(((M + BM - 1) / BM) * ((w.N + kBN - 1) / kBN));
  hipLaunchKernelGGL((GemmKernel<BM, HAS_ZP>), dim3(tiles * sh.splits), dim3(256), LdsBytes<BM>(),
                     s, Ah, w.B, w.scales, w.zp, Y, static_cast<int>(M), static_cast<int>(w.K),
                     static_cast<int>(w.N), static_cast<int>(w.nb), w.log2_bs,
                     static_cast<int>(w.row_bytes), static_cast<int>(w.zp_row_bytes),
                     sh.kt_per_split, partials, H, row_exp, w.col_exp);
  return hipGetLastError();
}

// ConvertAKernel over the padded rows of a BM tiling, keeping each thread's
// share of the row in registers when K allows.
template <int BM, bool RMS>
hipError_t LaunchConvertA(const WeightView &w, int64_t M, const float *A, uint4 *Ah, int *row_exp,
                          hipStream_t s, const float *gamma, float eps) {
  const dim3 grid(static_cast<unsigned>((M + BM - 1) / BM * BM)), block(256);
  const int K = static_cast<int>(w.K), m = static_cast<int>(M);
  if (K <= 2048 * 2)
    hipLaunchKernelGGL((ConvertAKernel<BM, 2, RMS>), grid, block, 0, s, A, Ah, row_exp, m, K, gamma, eps);
  else if (K <= 2048 * 4)
    hipLaunchKernelGGL((ConvertAKernel<BM, 4, RMS>), grid, block, 0, s, A, Ah, row_exp, m, K, gamma, eps);
  else if (K <= 2048 * 8)
    hipLaunchKernelGGL((ConvertAKernel<BM, 8, RMS>), grid, block, 0, s, A, Ah, row_exp, m, K, gamma, eps);
  else
    hipLaunchKernelGGL((ConvertAKernel<BM, 0, RMS>), grid, block, 0, s, A, Ah, row_exp, m, K, gamma, eps);
  return hipGetLastError();
}

template <int BM>
hipError_t LaunchBM(const WeightView &w, int64_t M, const float *A, float *Y, void *work,
                    const Shape &sh, hipStream_t s, float *H, const float *gamma, float eps) {
  uint4 *Ah = static_cast<uint4 *>(work);
  int *row_exp = reinterpret_cast<int *>(static_cast<char *>(work) + AImageBytes(w, M));
  float *partials = reinterpret_cast<float *>(static_cast<char *>(work) + AImageBytes(w, M) +
                                              RowExpBytes(M));
  hipError_t e = gamma != nullptr
                     ? LaunchConvertA<BM, true>(w, M, A, Ah, row_exp, s, gamma, eps)
                     : LaunchConvertA<BM, false>(w, M, A, Ah, row_exp, s, nullptr, 0.0f);
  if (e != hipSuccess) return e;
  // Gate/up activation: fused into the GEMM's stores with one split, into the
  // reduction (split 0 then writes the scratch Y) with several.
  float *Hk = sh.splits == 1 ? H : nullptr;
  e = w.zp != nullptr ? LaunchT<BM, true>(w, M, Ah, Y, partials, sh, s, Hk, row_exp)
                      : LaunchT<BM, false>(w, M, Ah, Y, partials, sh, s, Hk, row_exp);
  if (e != hipSuccess || sh.splits == 1) return e;
  return DispatchReduce(sh.splits - 1, Y, partials, M * w.N, s, H,
                        std::make_integer_sequence<int, kMaxSplits - 1>{});
}

// Tile height and K splits, from sweeps on MI355X of every tile height
// against 1..16 splits (c2..c5 shapes, M = 2..2048):
// - tile height: 32 for M <= 32, 64 for M <= 64, else 128 (taller tiles
//   amortise the B dequantization over more rows and won at every M >= 128,
//   once split-K supplies the workgroups);
// - splits: as many as keep the whole launch within one wave of two
//   workgroups per CU (a partial second wave costs a full k-loop), and no
//   fewer than 8 k-tiles per split (the prologue and the reduction are not
//   free).
inline Shape PickShape(const WeightView &w, int64_t M) {
  const int bm = M <= 32 ? 32 : M <= 64 ? 64 : 128;
  const int64_t tiles = (M + bm - 1) / bm * ((w.N + kBN - 1) / kBN);
  const int64_t slots = 2 * static_cast<int64_t>(w.num_cus);
  const int ktiles = static_cast<int>(w.K / kBK);
  int64_t splits = std::max<int64_t>(1, slots / tiles);
  splits = std::min<int64_t>({splits, kMaxSplits, std::max(1, ktiles / 8)});
  return MakeShape(w, bm, static_cast<int>(splits));
}

// ---------------------------------------------------------------------------
// Prefill GEMM over the plan's fragment-ordered weights (PrefillKernel).
//
// At plan creation the weights are re-laid for this kernel (RelayoutBKernel,
// RelayoutSKernel): for each group g of 64 weight rows and each 32-k step s,
// the 1 KiB record Bp[g][s][lane][j] holds in lane l's 16 bytes the packed
// word (8 nibbles, original order) of weight row 64g + 16j + (l & 15) at k =
// 32s + 8(l >> 4): exactly lane l's MFMA operand for the 16 rows of slice j.
// The 256-byte record Sp[g][b][c][j] holds, per quantization block b, the
// fp16 scale (times the row's 2^e) in the low half, the zero point in byte 2
// and 16 times it in byte 3, for row 64g + 16j + c. Rows past N are zero (scale 0). One record
// per block, not per step: every step of a block reads the same record.
//
// A workgroup of 8 wavefronts (two per SIMD, one workgroup per CU) computes a
// 128 x 256 output tile. Wavefronts w and w + 4 own columns 64(w % 4) ..
// 64(w % 4) + 63 of all 128 rows and split K: w takes the first 32-k step of
// every 64-k tile, w + 4 the second, so each dequantized weight fragment
// feeds 8 MFMAs (13 VALU per 8 nibbles: 1.6 VALU per MFMA) and each SIMD
// holds two independent instruction streams to fill the other's waits. At
// the end the two halves meet in LDS (each wavefront adds the other's sum
// for 64 of the rows, in a fixed order). The MFMA takes the weights as its A
// operand and the activations as its B operand, so each lane's result is 4
// consecutive output columns of one row: 16-byte stores, and a gate/up pair
// (columns 2n, 2n + 1) lands in one lane.
// Every operand streams global -> LDS through direct copies (no registers)
// into a ring of kPNS stages of one 64-k tile each (A 16 KiB, weights 8 KiB,
// scales 4 KiB); the copies of tile t + kPSA are issued as tile t starts.
// The copy order per k-tile is fixed (2 A copies and 1 weight copy per
// thread, plus 1 scale copy in the first four wavefronts), so each wait is an
// exact vmcnt. One barrier per k-tile, at its top, makes tile t + 1 visible:
// tile t's MFMAs then run on fragments read during the previous tile, while
// tile t + 1's fragments are read (into a second register set) and
// dequantized.
constexpr int kPTM = 128;                             // output tile rows
constexpr int kPTN = 256;                             // output tile columns
constexpr int kPThreads = 512;                        // 8 wavefronts
constexpr int kPNS = 5;                               // LDS stages (k-tiles)
constexpr int kPSA = kPNS - 1;                        // copy distance (k-tiles)
constexpr int kPAU = kPTM * kUnits;                   // A units per stage (1024)
constexpr int kPBU = 128;                             // weight units per column group per stage
constexpr int kPSU = 64;                              // scale units per column group per stage
constexpr int kPStage = kPAU + 4 * (kPBU + kPSU);     // 1792 units, 28 KiB
constexpr size_t kPLds = size_t{kPNS} * kPStage * 16; // 140 KiB
constexpr int kPOps0 = kPAU / kPThreads + 2;          // copies per k-tile, wavefronts 0-3
constexpr int kPOps1 = kPAU / kPThreads + 1;          // wavefronts 4-7 (no scale copy)
// Cache policy of the output stores: non-temporal. Y is not read again by
// this kernel; streaming it out keeps the L2 for the operand tiles (measured:
// K = 1536, N = 14336, M = 8192, 448 MiB of Y, 443 -> 410 us; c4 unchanged). With K
// split, the split reduction reads Y and the partial sums straight back, and
// plain stores serve it better (c4 and c5 o at M = 512, 4 splits: 37.1 ->
// 35.4 and 38.0 -> 36.3 us per call; qkv at M = 256 33.2 -> 32.2).
constexpr int kStoreNT = 2;

template <bool HAS_ZP, bool BS32>
__global__ __launch_bounds__(kPThreads, 1) __attribute__((amdgpu_waves_per_eu(2, 2))) void
PrefillKernel(const uint4 *__restrict__ Ah, const uint8_t *__restrict__ Bp,
              const uint8_t *__restrict__ Sp, float *__restrict__ Y, int M, int N, int K,
              int log2_bs, int kt_per_split, float *__restrict__ partials, float *__restrict__ H,
              const int *__restrict__ row_exp, const int *__restrict__ col_exp,
              const float *__restrict__ bias) {
  extern __shared__ uint4 lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cg = wave & 3;   // column group: columns 64 cg .. 64 cg + 63 of the tile

  // Workgroup b -> (split, output tile). XCD x (b % 8) takes a contiguous run
  // of the tile order, which walks groups of 4 M tiles N tile by N tile, so
  // an XCD's L2 holds about 4 A bands and a run of weight bands.
  const int tiles_m = (M + kPTM - 1) / kPTM;
  const int tiles_n = (N + kPTN - 1) / kPTN;
  const int tiles = tiles_m * tiles_n;
  const int split = static_cast<int>(blockIdx.x) / tiles;
  int tm, tn;
  {
    int L = static_cast<int>(blockIdx.x) - split * tiles;
    if (tiles % 8 == 0) L = (L & 7) * (tiles / 8) + (L >> 3);
    constexpr int kGM = 4;
    const int group = L / (kGM * tiles_n);
    const int gm = min(kGM, tiles_m - group * kGM);
    const int rem = L - group * kGM * tiles_n;
    tm = group * kGM + rem % gm;
    tn = rem / gm;
  }
  const int m0 = tm * kPTM;
  const int n0 = tn * kPTN;
  const int T = K / 32;
  const int kt0 = split * kt_per_split;
  const int ktiles = min(kt_per_split, K / kBK - kt0);
  const int klast = ktiles - 1;
  const int g = n0 / 64 + cg;

  // The body, for the 32-k step sg (0 for wavefronts 0-3, 1 for 4-7) as a
  // template argument: no branch inside the loop, every index a constant.
  auto body = [&](auto sg_c) __attribute__((always_inline)) {
  constexpr int sg = decltype(sg_c)::value;
  // Copies per k-tile: A instruction i of wavefront w takes units
  // i * 512 + 64 w + lane; wavefront w the weight record of (g, step sg);
  // wavefronts 0-3 the scale records of g for both steps (lanes 16-31 the
  // second step's, lanes 32-63 repeat lanes 0-31). 32-k blocks: one record per
  // step; larger blocks hold both steps of a 64-k tile, whose record repeats.
  // Sources as a wave-uniform base (SGPRs) plus the lane's byte offset.
  const int nb = (K + (1 << log2_bs) - 1) >> log2_bs;
  const uint4 *a_base = Ah + (static_cast<size_t>(tm) * (K / kBK) + kt0) * kPAU + wave * 64;
  const uint8_t *b_base = Bp + (static_cast<size_t>(g) * T + 2 * kt0 + sg) * 1024;
  const uint8_t *s_base = Sp + static_cast<size_t>(g) * nb * 256;
  const uint32_t a_off = static_cast<uint32_t>(lane) * 16;
  const uint32_t s_off = static_cast<uint32_t>(lane & (BS32 ? 31 : 15)) * 16;
  const int bt_shift = BS32 ? 0 : log2_bs - 6;  // 64-k tiles per block, log2
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  auto issue = [&](int kt, int st) {
    const uint32_t base = lds0 + static_cast<uint32_t>(st * kPStage * 16);
#pragma unroll
    for (int i = 0; i < kPAU / kPThreads; ++i)
      CopyToLds16S(a_base + static_cast<size_t>(kt) * kPAU + i * kPThreads, a_off,
                   base + static_cast<uint32_t>((i * kPThreads + wave * 64) * 16));
    CopyToLds16S(b_base + static_cast<size_t>(kt) * 2048, a_off,
                 base + static_cast<uint32_t>((kPAU + cg * kPBU + sg * 64) * 16));
    if constexpr (sg == 0)
      CopyToLds16S(s_base + (BS32 ? static_cast<size_t>(2 * (kt0 + kt)) * 256
                                  : static_cast<size_t>((kt0 + kt) >> bt_shift) * 256),
                   s_off, base + static_cast<uint32_t>((kPAU + 4 * kPBU + cg * kPSU) * 16));
  };
  // Tile t + 1 has landed once only the copies of tiles t + 2 .. t + kPSA - 1
  // (issued at the tops of the iterations since) are outstanding.
  constexpr int kOps = sg == 0 ? kPOps0 : kPOps1;
  auto readA = [&](const uint4 *sb, int i) {
    return __builtin_bit_cast(half8, sb[Swz(i * 16 + (lane & 15), 4 * sg + (lane >> 4))]);
  };
  auto readB = [&](const uint4 *sb) { return sb[kPAU + cg * kPBU + sg * 64 + lane]; };
  auto readS = [&](const uint4 *sb) {
    return sb[kPAU + 4 * kPBU + cg * kPSU + sg * 16 + (lane & 15)];
  };

  floatx4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const Masks dq = MakeMasks();
  // Dequantized weight fragments of one 32-k step (MFMA A operands, slices j).
  auto dequant = [&](uint4 bw, uint4 sw, half8 (&bf)[4]) __attribute__((always_inline)) {
    const uint32_t w[4] = {bw.x, bw.y, bw.z, bw.w};
    const uint32_t z[4] = {sw.x, sw.y, sw.z, sw.w};
#pragma unroll
    for (int j = 0; j < 4; ++j)
      bf[j] = __builtin_bit_cast(half8, DequantWord(w[j], RowFromSz<HAS_ZP>(z[j]), dq));
  };
  // One k-tile: tile t + 1's weight words are dequantized and its activation
  // fragments read into the second register set while tile t's 32 MFMAs run
  // on the first, so no MFMA waits for an LDS read issued in the same
  // iteration (reading the fragments after their last use, into one set,
  // left the first MFMAs of every tile waiting for the reads: c4 75.9 ->
  // 69.3 us with the second set, bit-identical). The scheduler interleaves
  // each MFMA with up to two VALU of the dequantization.
  auto iter = [&](int t, half8 (&ac)[8], half8 (&an)[8], half8 (&bc)[4], half8 (&bn)[4])
                  __attribute__((always_inline)) {
    const uint4 *sb1 = lds + ((t + 1) % kPNS) * kPStage;
    // Tile t + 1 complete and visible (only the copies of tiles t + 2 ..
    // t + kPSA - 1 are outstanding); every wavefront is past tile t - 1.
    WaitVm<kOps * (kPSA - 2)>();
    __syncthreads();
    // Tile t + kPSA into stage (t - 1) % kPNS, last read in iteration t - 2.
    issue(min(t + kPSA, klast), (t + kPSA) % kPNS);
    const uint4 bwn = readB(sb1);
    const uint4 swn = readS(sb1);
#pragma unroll
    for (int i = 0; i < 8; ++i) an[i] = readA(sb1, i);
    __builtin_amdgcn_sched_barrier(0);
    dequant(bwn, swn, bn);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bc[j], ac[i], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // VALU
    }
  };

  // Prologue: tiles 0 .. kPSA-1 into stages 0 .. kPSA-1; wait for tile 0.
#pragma unroll
  for (int p = 0; p < kPSA; ++p) issue(min(p, klast), p);
  WaitVm<kOps * (kPSA - 1)>();
  __syncthreads();
  half8 a0[8], a1[8], b0[4], b1[4];
#pragma unroll
  for (int i = 0; i < 8; ++i) a0[i] = readA(lds, i);
  dequant(readB(lds), readS(lds), b0);
  // Two iterations per trip, the register sets trading roles.
  int t = 0;
  for (; t + 1 < ktiles; t += 2) {
    iter(t, a0, a1, b0, b1);
    iter(t + 1, a1, a0, b1, b0);
  }
  if (t < ktiles) iter(t, a0, a1, b0, b1);
  // No copy into this workgroup's LDS may land after it exits, or after the
  // LDS is reused below.
  WaitVm<0>();
  __syncthreads();

  // The two K halves meet: wavefront w + 4s finishes rows 64s .. 64s + 63
  // (fragments i = 4s .. 4s + 3) of column group cg and hands the other rows
  // to its partner through LDS (16 KiB per wavefront, as 16 x 16 fragments of
  // 16 bytes per lane). Sum order: step 0's half, then step 1's. The half is
  // a template argument so every accumulator index is a constant.
  float *out = split > 0 ? partials + static_cast<size_t>(split - 1) * M * N : Y;
  const int nl = n0 + cg * 64 + 4 * (lane >> 4);
  const int rows = min(M - m0, kPTM);
  {
    constexpr int S = sg;
    uint4 *xb = lds + wave * 1024;  // this wavefront's outgoing fragments
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const floatx4 v = acc[4 * (1 - S) + q][j];
        xb[(q * 4 + j) * 64 + lane] = make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]),
                                                 __float_as_uint(v[2]), __float_as_uint(v[3]));
      }
    // The exponents and the bias, all loaded here, behind the exchange:
    // between the stores each load waited out the stores before it (M = 512,
    // K = 14336, N = 4096 79.2 -> 76.5 us, M = 200, N = 28672 67.2 -> 64.7).
    int er[4];
    int4 ec[4];
    float4 bv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) er[q] = row_exp[m0 + (4 * S + q) * 16 + (lane & 15)];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int nc = min(nl + 16 * j, N - 4);
      ec[j] = *reinterpret_cast<const int4 *>(col_exp + nc);
      bv[j] = bias != nullptr && split == 0
                  ? make_float4(bias[nc], bias[nc + 1], bias[nc + 2], bias[nc + 3])
                  : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __syncthreads();
    const uint4 *pb = lds + (wave ^ 4) * 1024;  // the partner's fragments for my rows
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 u = pb[(q * 4 + j) * 64 + lane];
        const floatx4 o = {__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z),
                           __uint_as_float(u.w)};
        acc[4 * S + q][j] = S == 0 ? acc[4 * S + q][j] + o : o + acc[4 * S + q][j];
      }

    // Epilogue over this wavefront's 64 rows. Lane l holds, for fragment i
    // (rows 16i .. 16i + 15) and slice j, row m0 + 16i + (l & 15) and the 4
    // columns n0 + 64 cg + 16j + 4(l >> 4) + v. The accumulators are in units
    // of 2^(f_m + e_n): one ldexp per element undoes both. Split 0 writes Y
    // (and adds the bias), split s > 0 its partial sum.
    if (H != nullptr) {
      const int half_n = N >> 1;
      const auto hr = __builtin_amdgcn_make_buffer_rsrc(H + static_cast<size_t>(m0) * half_n, 0,
                                                        rows * half_n * 4, 0x00020000);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = nl + 16 * j;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx4 a = acc[4 * S + q][j];
          const float x0 = a[0], x1 = a[1], x2 = a[2], x3 = a[3];
          const float h0 = SiluMul(__builtin_amdgcn_ldexpf(x0, -(er[q] + ec[j].x)),
                                   __builtin_amdgcn_ldexpf(x1, -(er[q] + ec[j].y)));
          const float h1 = SiluMul(__builtin_amdgcn_ldexpf(x2, -(er[q] + ec[j].z)),
                                   __builtin_amdgcn_ldexpf(x3, -(er[q] + ec[j].w)));
          const int row = (4 * S + q) * 16 + (lane & 15);
          const int off = n < N ? (row * half_n + (n >> 1)) * 4 : 0x7FFFFFF0;
          // H columns n / 2 and n / 2 + 1 are adjacent: one 8-byte store. (A
          // non-temporal hint on these partial-line stores made the fused
          // plan 20-30% slower than the plain product; they stay cached.)
          typedef unsigned int u32x2 __attribute__((vector_size(8)));
          const u32x2 hv = {__float_as_uint(h0), __float_as_uint(h1)};
          __builtin_amdgcn_raw_buffer_store_b64(hv, hr, off, 0, 0);
        }
      }
      return;
    }
    const auto yr = __builtin_amdgcn_make_buffer_rsrc(out + static_cast<size_t>(m0) * N, 0,
                                                      rows * N * 4, 0x00020000);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = nl + 16 * j;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 a = acc[4 * S + q][j];
        const float x0 = a[0], x1 = a[1], x2 = a[2], x3 = a[3];
        typedef unsigned int u32x4 __attribute__((vector_size(16)));
        const u32x4 v = {__float_as_uint(__builtin_amdgcn_ldexpf(x0, -(er[q] + ec[j].x)) + bv[j].x),
                         __float_as_uint(__builtin_amdgcn_ldexpf(x1, -(er[q] + ec[j].y)) + bv[j].y),
                         __float_as_uint(__builtin_amdgcn_ldexpf(x2, -(er[q] + ec[j].z)) + bv[j].z),
                         __float_as_uint(__builtin_amdgcn_ldexpf(x3, -(er[q] + ec[j].w)) + bv[j].w)};
        const int row = (4 * S + q) * 16 + (lane & 15);
        const int off = n < N ? (row * N + n) * 4 : 0x7FFFFFF0;
        if (kt_per_split < K / kBK)  // split K: read back by the reduction
          __builtin_amdgcn_raw_buffer_store_b128(v, yr, off, 0, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b128(v, yr, off, 0, kStoreNT);
      }
    }
  }
  };
  if ((wave >> 2) == 0)
    body(std::integral_constant<int, 0>{});
  else
    body(std::integral_constant<int, 1>{});
}

// ---------------------------------------------------------------------------
// Small-M prefill (17 <= M <= 64) streaming the fragment-ordered weights
// (StreamKernel). With so few rows a 128 x 256 tile holds mostly padding and
// the GEMM is bound by reading the weights once, so the grid is laid out
// like the decode kernels': one workgroup per (group g of 64 weight rows, K
// segment), WPG wavefronts each taking SPW consecutive 32-k steps of the
// segment. Per step a wavefront loads the group's 1 KiB weight record and
// 256-byte scale record (the PrefillKernel layouts), dequantizes the four
// words exactly as PrefillKernel does (DequantWord on the fp16 scale times
// 2^e_n), reads TG activation fragments of the fp16 image ConvertChunkKernel
// wrote (rows past M zero) and issues
// 4 TG v_mfma_f32_16x16x32_f16 into TG x 4 fp32 tiles. The operands are
// those of the prefill GEMM (a chunk's exponent instead of the row's), so the
// product is the same up to the order of the fp32 sums. Loads stream through a rolling window of WIN steps in
// registers (multiply the oldest, issue the one WIN further on), with no
// branch around any load. The wavefronts' tiles meet in LDS and are added
// in wavefront order; segment 0 writes Y (adding the bias or applying the
// gate/up activation when K is not split), segment s > 0 its partial sum,
// added in segment order by SplitReduceKernel.
//
// G = 2 takes two column groups per workgroup, each activation fragment loaded
// once for both: with many groups the loads of the activations (TG KiB per
// step beside 1.25 KiB of weights, from the L2) bound the kernel (K = 4096,
// N = 28672, 448 groups: M = 48 / 64 30.4 / 34.0 -> 27.3 / 29.8 us).
constexpr int kSGroupRows = 64;
// PARTS: in how many parts a group's tiles meet in LDS. All at once (4 TG KiB
// per wavefront) saves barriers and lets every wavefront of eight finish a
// fragment (K = N = 4096 at M = 17 8.6 -> 8.1 us); with more than two row tiles
// and more than four wavefronts in two parts, so that two workgroups fit a CU.
template <int TG, int G>
constexpr int StreamParts(int wpg) { return G == 1 && (TG == 2 || wpg == 4) ? 1 : 2; }

//
// CVT: the wavefront converts its own activations instead of reading the
// image (no ConvertAKernel launch; used for small fragment counts, see
// StreamConverts): it loads A's fp32 values for its SPW steps first (L2-
// resident, ahead of the weights), reduces each row's largest magnitude over
// its own k range across the four lanes that hold the row, scales by 2^f and
// rounds to fp16 as ConvertAKernel does, and undoes f (with the column's exponent)
// before the wavefronts' tiles meet. A finer exponent than the row's, so the
// operands are ConvertAKernel's except where those fall into fp16
// subnormals.
template <bool HAS_ZP, int TG, int SPW, int WIN, bool CVT, int G, int PARTS>
__global__ __launch_bounds__(512) void StreamKernel(
    const uint4 *__restrict__ Ah, const float *__restrict__ A, const uint8_t *__restrict__ Bp,
    const uint8_t *__restrict__ Sp, float *__restrict__ Y, float *__restrict__ partials,
    float *__restrict__ H, const int *__restrict__ row_exp, const int *__restrict__ col_exp,
    const float *__restrict__ bias, const float *__restrict__ sq, float eps, int M, int N, int K,
    int log2_bs, int segs, int wpg) {
  extern __shared__ floatx4 sred[];  // [wave][kJ tg + j % kJ][lane], one part of the fragments
  __shared__ float qs[CVT ? 1 : 8][TG][16], rms_inv[CVT ? 1 : 8][16 * TG];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int g = static_cast<int>(blockIdx.x) / segs * G;  // first group
  const int seg = static_cast<int>(blockIdx.x) % segs;
  const int T = K / 32;
  const int s0 = (seg * wpg + wave) * SPW;  // first step of this wavefront
  __amdgpu_buffer_rsrc_t rb[G], rs[G];
  const int nb = (K + (1 << log2_bs) - 1) >> log2_bs;
  const int sb_shift = log2_bs - 5;  // 32-k steps per block, log2
#pragma unroll
  for (int x = 0; x < G; ++x) {  // a G past the last group reads zero weights (padded records)
    rb[x] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(Bp + static_cast<size_t>(g + x) * T * 1024), 0, T * 1024, 0x00020000);
    rs[x] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(Sp + static_cast<size_t>(g + x) * nb * 256), 0, nb * 256, 0x00020000);
  }
  // Lane l's activation fragment tg of step s: 16 bytes of the 1 KiB record
  // (tg, s), contiguous over the lanes. (In the prefill kernel's swizzled rows
  // every four lanes of such a load fall into four cache lines, and the L1's
  // one line per cycle bounded the kernel: K = 4096, N = 28672 at M = 48 / 64 35.4 / 41.6 ->
  // 29.7 / 33.9 us.)
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint4 *>(Ah), 0, TG * T * 1024, 0x00020000);

  typedef uint32_t u32x4e __attribute__((ext_vector_type(4)));
  typedef float f32x4e __attribute__((ext_vector_type(4)));
  // CVT: the wavefront's fp32 activations, [step][tg] pairs of 4 k (k order
  // 0..3, 4..7 of the lane's 8), loaded before anything else.
  f32x4e alo[CVT ? SPW : 1][CVT ? TG : 1], ahi[CVT ? SPW : 1][CVT ? TG : 1];
  if constexpr (CVT) {
    const __amdgpu_buffer_rsrc_t rA =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A), 0, M * K * 4, 0x00020000);
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) {
      const int m = 16 * tg + (lane & 15);
#pragma unroll
      for (int i = 0; i < SPW; ++i) {
        // rows past M read past the end of the buffer: zeros
        const int off = m < M ? (m * K + 32 * (s0 + i) + 8 * (lane >> 4)) * 4 : M * K * 4;
        alo[i][tg] = __builtin_bit_cast(f32x4e, __builtin_amdgcn_raw_buffer_load_b128(rA, off, 0, 0));
        ahi[i][tg] = __builtin_bit_cast(f32x4e, __builtin_amdgcn_raw_buffer_load_b128(rA, off + 16, 0, 0));
      }
    }
  }
  struct Slot {
    u32x4e w[G], sz[G];
    half8 a[CVT ? 1 : TG];
  };
  Slot ring[WIN];
  auto issue = [&](int i) __attribute__((always_inline)) {
    Slot &sl = ring[i % WIN];
    const int s = s0 + i;
#pragma unroll
    for (int x = 0; x < G; ++x) {
      sl.w[x] = __builtin_bit_cast(
          u32x4e, __builtin_amdgcn_raw_buffer_load_b128(rb[x], s * 1024 + 16 * lane, 0, 2));
      sl.sz[x] = __builtin_bit_cast(u32x4e, __builtin_amdgcn_raw_buffer_load_b128(
                                                rs[x], (s >> sb_shift) * 256 + 16 * (lane & 15), 0, 0));
    }
    if constexpr (!CVT) {
#pragma unroll
      for (int tg = 0; tg < TG; ++tg)
        sl.a[tg] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(
                                                 ra, (tg * T + s) * 1024 + 16 * lane, 0, 0));
    }
  };
  // The columns' exponents come ahead of the weights and the epilogue's bias
  // behind the first of them, so that their latency hides under the main loop
  // (with two groups, whose registers they would take, in the epilogue).
  constexpr bool kPreload = G == 1;
  int4 ec[4 * G];  // [group, j]: this lane's columns of every fragment
  auto ec_load = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int y = 0; y < 4 * G; ++y)
      ec[y] = *reinterpret_cast<const int4 *>(
          col_exp + min(kSGroupRows * g + 16 * y + 4 * (lane >> 4), N - 4));
  };
  if constexpr (kPreload) ec_load();
  // RMSNorm input: this wavefront's part of each row's sum of squares, chunks
  // 4 wave + (lane >> 4), + 4 wpg, ... (64 TG bytes each, zeros past the last).
  // Loaded ahead of the weights and added while those are on their way: every
  // wavefront adding all of them after the main loop took 1 to 2 us more.
  const int sq_bytes = CVT || sq == nullptr ? 0 : (K + kChunkK - 1) / kChunkK * 64 * TG;
  const int sq_off = (4 * wave + (lane >> 4)) * 64 * TG + 4 * (lane & 15);
  const int sq_step = 4 * wpg * 64 * TG;
  const __amdgpu_buffer_rsrc_t rq =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(sq), 0, sq_bytes, 0x00020000);
  float sqv[TG];
  if constexpr (!CVT) {
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
      sqv[tg] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rq, sq_off + 64 * tg, 0, 0));
  }
#pragma unroll
  for (int i = 0; i < WIN && i < SPW; ++i) issue(i);
  // The epilogue finishes, group by group, PARTS parts of the fragments (tg, j)
  // (part j / kJ, kPart fragments), x = wave, wave + wpg, ... of each (wpg >= 4).
  constexpr int kJ = 4 / PARTS;
  constexpr int kPart = kJ * TG;
  constexpr int kPartItems = (kPart + 3) / 4;
  constexpr int kMaxItems = PARTS * G * kPartItems;
  float4 bv[kMaxItems];
  auto item_col = [&](int it) {
    const int x = min(wave + it % kPartItems * wpg, kPart - 1), ph = it / kPartItems;
    return kSGroupRows * g + 16 * (kJ * ph + x % kJ) + 4 * (lane >> 4);
  };
  auto item_bias = [&](int it) __attribute__((always_inline)) {
    const int nc = min(item_col(it), N - 4);
    bv[it] = bias != nullptr ? make_float4(bias[nc], bias[nc + 1], bias[nc + 2], bias[nc + 3])
                             : make_float4(0.f, 0.f, 0.f, 0.f);
  };
  if constexpr (kPreload) {
#pragma unroll
    for (int it = 0; it < kMaxItems; ++it) item_bias(it);
  }
  __builtin_amdgcn_sched_barrier(0);

  if (!CVT && sq != nullptr) {
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) {
      for (int o = sq_off + sq_step; o < sq_bytes; o += sq_step)
        sqv[tg] += __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rq, o + 64 * tg, 0, 0));
      float q = sqv[tg];
      q += Xor16(q);
      q += __shfl_xor(q, 32, 64);
      if (lane < 16) qs[wave][tg][lane] = q;
    }
    __syncthreads();
    // row `lane`'s 1 / rms, kept for this wavefront's epilogue
    const int rl = min(lane, 16 * TG - 1);
    float q = 0.0f;
    for (int w = 0; w < wpg; ++w) q += qs[w][rl / 16][rl % 16];
    if (lane < 16 * TG) rms_inv[wave][lane] = 1.0f / sqrtf(q / static_cast<float>(K) + eps);
  }

  // CVT: each row's exponent over this wavefront's k range (the row's values
  // sit in lanes r, r + 16, r + 32, r + 48), then the fp16 fragments.
  half8 af[CVT ? SPW : 1][CVT ? TG : 1];
  int fw[TG];
  if constexpr (!CVT) {
    // the chunk's (a wavefront past K reads the last chunk's and adds nothing)
    const int ch = min(s0 / (kChunkK / 32), (T - 1) / (kChunkK / 32));
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) fw[tg] = row_exp[ch * 16 * TG + 16 * tg + (lane & 15)];
  } else {
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) {
      float amax = 0.0f;
#pragma unroll
      for (int i = 0; i < SPW; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          amax = fmaxf(amax, fmaxf(fabsf(alo[i][tg][c]), fabsf(ahi[i][tg][c])));
      amax = fmaxf(amax, Xor16(amax));
      amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
      const int f = RangeExponent(amax, kRowExpTarget);
      fw[tg] = f;
#pragma unroll
      for (int i = 0; i < SPW; ++i) {
        auto sc = [f](float v) { return __builtin_amdgcn_ldexpf(v, f); };
        const f32x4e x = alo[i][tg], y = ahi[i][tg];
        // k order [0,4,1,5,2,6,3,7], the order DequantWord produces
        af[i][tg] = __builtin_bit_cast(
            half8, make_uint4(PackHalf2(sc(x[0]), sc(y[0])), PackHalf2(sc(x[1]), sc(y[1])),
                              PackHalf2(sc(x[2]), sc(y[2])), PackHalf2(sc(x[3]), sc(y[3]))));
      }
    }
  }

  const Masks dq = MakeMasks();
  floatx4 acc[G][TG][4];
#pragma unroll
  for (int x = 0; x < G; ++x)
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[x][tg][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < SPW; ++i) {
    Slot &sl = ring[i % WIN];
#pragma unroll
    for (int x = 0; x < G; ++x) __asm__ volatile("" : "+v"(sl.w[x]), "+v"(sl.sz[x]));
#pragma unroll
    for (int x = 0; x < G; ++x) {
      half8 bf[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bf[j] = __builtin_bit_cast(half8, DequantWord(sl.w[x][j], RowFromSz<HAS_ZP>(sl.sz[x][j]), dq));
#pragma unroll
      for (int tg = 0; tg < TG; ++tg) {
        half8 a;
        if constexpr (CVT)
          a = af[i][tg];
        else
          a = sl.a[tg];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[x][tg][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[j], a, acc[x][tg][j], 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (i + WIN < SPW) issue(i + WIN);
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (!kPreload) ec_load();
  // RMSNorm input: each row's 1 / rms as a factor in [0.5, 1) (0 and infinity
  // themselves) and a power of two that joins the exponents.
  float inv[TG];
#pragma unroll
  for (int tg = 0; tg < TG; ++tg) inv[tg] = 1.0f;
  if (!CVT && sq != nullptr) {
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) {
      const float r = rms_inv[wave][16 * tg + (lane & 15)];
      inv[tg] = __builtin_amdgcn_frexp_mantf(r);
      fw[tg] -= __builtin_amdgcn_frexp_expf(r);
    }
  }

  // The wavefronts' tiles meet in LDS, part by part; wavefront w finishes the
  // part's fragments x = kJ tg + j % kJ = w, w + wpg, ..., adding the
  // wavefronts' tiles in wavefront order. Lane l holds row 16 tg + (l & 15)
  // and the 4 columns 64 g + 16 j + 4 (l >> 4) .. + 3. A wavefront past K
  // (the end of a shorter last segment) ran on loads beyond the weights'
  // buffers (zeros) and activations past its rows: it adds nothing. The row's
  // and the column's exponent are undone together: the sums are products times
  // 2^(f + e), and undoing f alone leaves large rows beyond fp32.
  const bool past_k = s0 >= T;
  float *out = seg == 0 ? Y : partials + static_cast<size_t>(seg - 1) * M * N;
#pragma unroll
  for (int ph = 0; ph < PARTS * G; ++ph) {  // (group, part)
    if (ph > 0) __syncthreads();
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
#pragma unroll
      for (int jj = 0; jj < kJ; ++jj) {
        floatx4 t = acc[ph / PARTS][tg][kJ * (ph % PARTS) + jj];
        const int4 e4 = ec[kJ * ph + jj];
        const int ev[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
          t[q] = __builtin_amdgcn_ldexpf(t[q] * inv[tg], -(fw[tg] + ev[q]));
        sred[(wave * kPart + tg * kJ + jj) * 64 + lane] = past_k ? floatx4{0.f, 0.f, 0.f, 0.f} : t;
      }
    __syncthreads();
#pragma unroll
    for (int hi = 0; hi < kPartItems; ++hi) {
      const int x = wave + hi * wpg;
      if (x >= kPart) break;
      const int it = ph * kPartItems + hi;
      if constexpr (!kPreload) item_bias(it);
      floatx4 v = sred[x * 64 + lane];
      for (int w = 1; w < wpg; ++w) v += sred[(w * kPart + x) * 64 + lane];
      const int m = 16 * (x / kJ) + (lane & 15);
      const int n = item_col(it);
      const bool ok = m < M && n < N;
      if (H != nullptr) {
        // gate/up pairs (columns n, n + 1 and n + 2, n + 3): H columns n / 2, n / 2 + 1
        const int half_n = N >> 1;
        const auto hr = __builtin_amdgcn_make_buffer_rsrc(H, 0, M * half_n * 4, 0x00020000);
        typedef unsigned int u32x2 __attribute__((vector_size(8)));
        const u32x2 hv = {__float_as_uint(SiluMul(v[0], v[1])), __float_as_uint(SiluMul(v[2], v[3]))};
        __builtin_amdgcn_raw_buffer_store_b64(
            hv, hr, ok ? (m * half_n + (n >> 1)) * 4 : M * half_n * 4, 0, 0);
      } else {
        if (bias != nullptr) {
          v[0] += bv[it].x;
          v[1] += bv[it].y;
          v[2] += bv[it].z;
          v[3] += bv[it].w;
        }
        const auto yr = __builtin_amdgcn_make_buffer_rsrc(out, 0, M * N * 4, 0x00020000);
        typedef unsigned int u32x4 __attribute__((vector_size(16)));
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), yr,
                                               ok ? (m * N + n) * 4 : M * N * 4, 0, 0);
      }
    }
  }
}

// Steps in flight with two groups per wavefront: 16 (w, sz) + 4 TG VGPRs each
// beside 32 TG accumulators.
template <int TG>
constexpr int WinG2() { return TG == 2 ? 4 : TG == 3 ? 3 : 2; }

// Whether a launch's wavefronts convert their own activations: at most 8
// fragments per wavefront (two row tiles of 4 steps) and no more workgroups
// than CUs. It saves the conversion's launch, 1.3 us of a call at M = 17 and 0.9
// at M = 32 with four wavefronts per workgroup, 0.9 and nothing with eight (K =
// 2048, N = 512 9.7 -> 8.2 and 9.8 -> 8.9 us); slower where the fragments or the
// workgroups are more (K = N = 4096 at M = 48 / 64 +0.4 / +1.2 us, 8 steps per
// wavefront at M = 32 +4.9 us, 1.5 workgroups per CU +1.4 us).
inline bool StreamConverts(const WeightView &w, int64_t M, const StreamShape &sh) {
  const int64_t wgs = (w.N + kSGroupRows - 1) / kSGroupRows * sh.segs;
  return sh.groups == 1 && (M + 15) / 16 * sh.spw <= 8 && wgs <= w.num_cus;
}

// The launch shape: groups of 64 rows per workgroup, K segments, wavefronts
// per workgroup (4 to 8) and steps per wavefront (4, 8 or 16; 8 or 16 with two
// groups); the last segment may be shorter. The least estimated time in us, a
// fit to 5700 measured calls (51 weights, six M, every shape; the shape taken is
// 0.5% from the fastest on average, 10% at most): the busiest SIMD runs `waves`
// wavefronts, each of `spw` steps, a fill and an exchange per fragment (five to
// seven in a workgroup put two on some SIMDs; with two groups, whose registers
// allow one workgroup per CU, they cost as eight); several segments add the
// launch and the traffic of the reduction. Estimated by rounds of workgroups
// times steps the shape was 7% from the fastest, and up to 40% on small
// weights, where a step costs a memory latency. us: K = 2048, N = 512 at M =
// 17 / 33 one segment of 8 x 8 10.2 / 12.2, four of 4 x 4 8.2 / 10.4; K = N =
// 5120 at M = 48 two groups, four of 5 x 8 20.6, one group, three of 4 x 16 15.1;
// K = 12288, N = 16384 at M = 17 six of 8 x 8 46.9, six of 4 x 16 35.4; K = 4096,
// N = 28672 at M = 48 two groups, one of 8 x 16 26.3, one group 30.2.
// M counts as the largest of its class: 24, 32, 48 or 64.
inline StreamShape SearchStreamShape(const WeightView &w, int64_t M) {
  const int64_t groups = (w.N + kSGroupRows - 1) / kSGroupRows;
  const int T = static_cast<int>(w.K / 32);
  const int tg = static_cast<int>((M + 15) / 16);
  StreamShape best{0, 0, 0};
  double best_us = 0.0;
  for (int g : {1, 2})
    for (int spw : {16, 8, 4}) {
      if (T % spw != 0 || (g == 2 && spw == 4)) continue;
      for (int segs = 1; segs <= kMaxSplits; ++segs) {
        const int wpg = std::max(4, (T / spw + segs - 1) / segs);  // wavefronts cover a segment
        const int per = wpg * spw, simd = (wpg + 3) / 4;
        if (wpg > 8 || (T + per - 1) / per != segs) continue;
        const StreamShape sh{segs, wpg, spw, g};
        const int64_t wgs = (groups + g - 1) / g * segs;
        const int64_t rounds = (wgs + w.num_cus - 1) / std::max(1, w.num_cus);
        const double waves = rounds * (g == 1 ? 0.8 * simd + 0.05 * wpg : simd);
        double us = g == 1 ? waves * ((0.1 + 0.035 * tg) * spw + 0.25 * tg)
                           : waves * ((0.15 + 0.04 * tg) * spw + 0.3 * tg + 1.4) + 1.3;
        if (segs > 1) us += 1.65 + 0.05 * segs + 0.6e-6 * (segs + 1) * M * w.N;
        if (StreamConverts(w, M, sh)) us -= M <= 24 ? 1.75 - 0.4 * simd : 1.9 - simd;
        if (best.segs == 0 || us < best_us) {
          best = sh;
          best_us = us;
        }
      }
    }
  return best;
}

// The plan's shape for M rows (17 to 64), or the one asked for.
inline StreamShape PickStreamShape(const WeightView &w, int64_t M, int segs_req, int spw_req) {
  if (segs_req > 0 && spw_req > 0) {
    const int per = segs_req * spw_req, T = static_cast<int>(w.K / 32);
    return StreamShape{segs_req, T % per == 0 ? T / per : 0, spw_req};
  }
  return w.stream[M <= 24 ? 0 : M <= 32 ? 1 : M <= 48 ? 2 : 3];
}

// Whether K / 32 steps divide evenly into such segments.
inline bool StreamEven(const WeightView &w) {
  const int T = static_cast<int>(w.K / 32);
  for (int spw : {16, 8, 4})
    for (int wpg = 4; wpg <= 8; ++wpg)
      if (T % (wpg * spw) == 0 && T / (wpg * spw) <= kMaxSplits) return true;
  return false;
}

// The launch's operands: the fp16 image with its chunk exponents and (RMSNorm)
// sums of squares, or A itself for the wavefronts to convert.
struct StreamIn {
  const uint4 *Ah;
  const float *A;
  const int *exps;
  const float *sq;
  float eps;
};

template <bool HAS_ZP, int TG, int SPW, int WIN, bool CVT, int G, int PARTS>
hipError_t LaunchStreamParts(const WeightView &w, int64_t M, const StreamIn &in, float *Y, float *P,
                             float *H, const float *bias, const StreamShape &sh, hipStream_t s) {
  const int64_t groups = (w.N + kSGroupRows - 1) / kSGroupRows;
  const size_t lds = static_cast<size_t>(sh.wpg) * TG * (4 / PARTS) * 64 * 16;
  const dim3 grid(static_cast<unsigned>((groups + G - 1) / G * sh.segs)), block(64 * sh.wpg);
  hipLaunchKernelGGL((StreamKernel<HAS_ZP, TG, SPW, WIN, CVT, G, PARTS>), grid, block, lds, s, in.Ah,
                     in.A, w.Bp, w.Sp, Y, P, H, in.exps, w.col_exp, bias, in.sq, in.eps,
                     static_cast<int>(M), static_cast<int>(w.N), static_cast<int>(w.K), w.log2_bs,
                     sh.segs, sh.wpg);
  return hipGetLastError();
}

template <bool HAS_ZP, int TG, int SPW, int WIN, bool CVT, int G>
hipError_t LaunchStreamT(const WeightView &w, int64_t M, const StreamIn &in, float *Y, float *P,
                         float *H, const float *bias, const StreamShape &sh, hipStream_t s) {
  if constexpr (StreamParts<TG, G>(4) == 1) {
    if (StreamParts<TG, G>(sh.wpg) == 1)
      return LaunchStreamParts<HAS_ZP, TG, SPW, WIN, CVT, G, 1>(w, M, in, Y, P, H, bias, sh, s);
  }
  if constexpr (StreamParts<TG, G>(8) == 2)
    return LaunchStreamParts<HAS_ZP, TG, SPW, WIN, CVT, G, 2>(w, M, in, Y, P, H, bias, sh, s);
  return hipErrorInvalidValue;
}

template <bool HAS_ZP, int TG>
hipError_t LaunchStreamTG(const WeightView &w, int64_t M, const StreamIn &in, float *Y, float *P,
                          float *H, const float *bias, const StreamShape &sh, hipStream_t s) {
  if (in.A != nullptr) {  // StreamConverts: two row tiles, 4 steps
    if constexpr (TG == 2)
      return LaunchStreamT<HAS_ZP, TG, 4, 4, true, 1>(w, M, in, Y, P, H, bias, sh, s);
    return hipErrorInvalidValue;
  }
  if (sh.groups == 2) switch (sh.spw) {
    case 8: return LaunchStreamT<HAS_ZP, TG, 8, WinG2<TG>(), false, 2>(w, M, in, Y, P, H, bias, sh, s);
    case 16: return LaunchStreamT<HAS_ZP, TG, 16, WinG2<TG>(), false, 2>(w, M, in, Y, P, H, bias, sh, s);
    default: return hipErrorInvalidValue;
  }
  switch (sh.spw) {
  case 4: return LaunchStreamT<HAS_ZP, TG, 4, 4, false, 1>(w, M, in, Y, P, H, bias, sh, s);
  case 8: return LaunchStreamT<HAS_ZP, TG, 8, 4, false, 1>(w, M, in, Y, P, H, bias, sh, s);
  case 16: return LaunchStreamT<HAS_ZP, TG, 16, 4, false, 1>(w, M, in, Y, P, H, bias, sh, s);
  default: return hipErrorInvalidValue;
  }
}

template <bool HAS_ZP>
hipError_t LaunchStreamZp(const WeightView &w, int64_t M, const StreamIn &in, float *Y, float *P,
                          float *H, const float *bias, const StreamShape &sh, hipStream_t s) {
  switch ((M + 15) / 16) {
  case 2: return LaunchStreamTG<HAS_ZP, 2>(w, M, in, Y, P, H, bias, sh, s);
  case 3: return LaunchStreamTG<HAS_ZP, 3>(w, M, in, Y, P, H, bias, sh, s);
  case 4: return LaunchStreamTG<HAS_ZP, 4>(w, M, in, Y, P, H, bias, sh, s);
  default: return hipErrorInvalidValue;
  }
}

// Splits of a prefill launch: as many as keep the workgroups within one per
// CU when the tiles alone do not fill the chip (a second, partial wave costs
// a whole k-loop), at most kPrefillMaxSplits, each split at least 8 k-tiles.
// Up to 16 splits serve long rows on few tiles (against 8: K = 14336,
// N = 4096 at M = 65 / 128 38.1 / 40.4 -> 33.1 / 38.4 us; K = 14336,
// N = 2048 at M = 128 38.2 -> 31.8; K = 11008, N = 4096 at M = 65 33.0 ->
// 30.2; c4, c5 qkv and o unchanged). Whether the prefill kernel takes such
// rows at all is judged at 8 splits (UsePrefill, kPrefillCheckSplits).
constexpr int kPrefillMaxSplits = 16;
constexpr int kPrefillCheckSplits = 8;
inline int PrefillSplits(const WeightView &w, int64_t M) {
  const int64_t tiles = (M + kPTM - 1) / kPTM * ((w.N + kPTN - 1) / kPTN);
  const int ktiles = static_cast<int>(w.K / kBK);
  int64_t splits = std::max<int64_t>(1, w.num_cus / tiles);
  splits = std::min<int64_t>({splits, kPrefillMaxSplits, std::max(1, ktiles / 8)});
  const int per = static_cast<int>((ktiles + splits - 1) / splits);
  return (ktiles + per - 1) / per;
}

template <bool HAS_ZP, bool BS32>
hipError_t LaunchPrefillT(const WeightView &w, int64_t M, const uint4 *Ah, float *Y,
                          float *partials, int splits, hipStream_t s, float *H,
                          const int *row_exp, const float *bias) {
  const int ktiles = static_cast<int>(w.K / kBK);
  const int per = (ktiles + splits - 1) / splits;
  const int tiles = static_cast<int>((M + kPTM - 1) / kPTM * ((w.N + kPTN - 1) / kPTN));
  hipLaunchKernelGGL((PrefillKernel<HAS_ZP, BS32>), dim3(tiles * splits), dim3(kPThreads), kPLds, s, Ah,
                     w.Bp, w.Sp, Y, static_cast<int>(M), static_cast<int>(w.N),
                     static_cast<int>(w.K), w.log2_bs, per, partials, H, row_exp, w.col_exp, bias);
  return hipGetLastError();
}

// The plan-time re-layout (once per plan, see PrefillKernel).
__global__ __launch_bounds__(256) void RelayoutBKernel(const uint8_t *__restrict__ B,
                                                       uint32_t *__restrict__ Bp, int64_t N,
                                                       int64_t row_bytes, int64_t T,
                                                       int64_t words) {
  for (int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; idx < words;
       idx += static_cast<int64_t>(gridDim.x) * 256) {
    const int j = static_cast<int>(idx & 3);
    const int l = static_cast<int>((idx >> 2) & 63);
    const int64_t gs = idx >> 8;
    const int64_t s = gs % T, g = gs / T;
    const int64_t n = 64 * g + 16 * j + (l & 15);
    Bp[idx] = n < N ? *reinterpret_cast<const uint32_t *>(B + n * row_bytes + 16 * s + 4 * (l >> 4))
                    : 0u;
  }
}

__global__ __launch_bounds__(256) void RelayoutSKernel(const float *__restrict__ S,
                                                       const uint8_t *__restrict__ Z,
                                                       const int32_t *__restrict__ col_exp,
                                                       uint32_t *__restrict__ Sp, int64_t N,
                                                       int64_t nb, int64_t zp_row_bytes,
                                                       int64_t words) {
  for (int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; idx < words;
       idx += static_cast<int64_t>(gridDim.x) * 256) {
    const int j = static_cast<int>(idx & 3);
    const int c = static_cast<int>((idx >> 2) & 15);
    const int64_t gb = idx >> 6;
    const int64_t b = gb % nb, g = gb / nb;
    const int64_t n = 64 * g + 16 * j + c;
    uint32_t v = (8u << 16) | (8u << 28);  // rows past N: scale 0
    if (n < N) {
      const _Float16 h = static_cast<_Float16>(__builtin_amdgcn_ldexpf(S[n * nb + b], col_exp[n]));
      const uint32_t z = Z != nullptr ? (Z[n * zp_row_bytes + (b >> 1)] >> (4 * (b & 1))) & 0xFu : 8u;
      v = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, h)) | (z << 16) | (z << 28);
    }
    Sp[idx] = v;
  }
}

bool PrefillSupportsShape(const WeightView &w) {
  return w.Bp != nullptr && w.Sp != nullptr && (w.K % kBK) == 0 && w.block_size >= 32 &&
         (w.N % 4) == 0 && w.N < (int64_t{1} << 22) && w.K <= (int64_t{1} << 24);
}

bool PrefillSupportsM(const WeightView &w, int64_t M) {
  return M >= 1 && M <= (int64_t{1} << 30) && PrefillSupportsShape(w) &&
         (M + kPTM - 1) / kPTM * ((w.N + kPTN - 1) / kPTN) * kMaxSplits < (int64_t{1} << 31);
}

// Weights whose K / 32 steps, cut evenly into segments (of 4 or 8 wavefronts of
// 4, 8 or 16 steps, covering 85% of the CUs), make more than three groups x
// segments per CU.
bool StreamManyGroups(const WeightView &w, int64_t M) {
  const int64_t groups = (w.N + kSGroupRows - 1) / kSGroupRows;
  const int T = static_cast<int>(w.K / 32);
  if (M <= 32) return false;
  int best = 0;
  for (int segs = 1; segs <= kMaxSplits; ++segs) {
    const int per = T % segs == 0 ? T / segs : 0;
    if (per != 16 && per != 32 && per != 64 && per != 128) continue;
    best = segs;
    if (groups * segs * 100 >= static_cast<int64_t>(w.num_cus) * 85) break;
  }
  return (best > 1 || (best == 1 && M > 48)) &&
         groups * best > 3 * static_cast<int64_t>(w.num_cus);
}

// Those of them that the prefill kernel keeps above 32 rows: K / 32 steps that
// segments of 8 x 16 steps do not divide. Streaming them was slower than
// the prefill kernel before the activations came in operand order; now it is
// 8 to 16% faster (K = 5120, N = 13824 at M = 33 / 64 26.7 / 29.3 against
// 29.0 / 32.3 us, K = 3584, N = 18944 23.7 / 27.2 against 28.2 / 31.4), but
// their route is part of what the tests fix, so it stays.
bool StreamCrowded(const WeightView &w, int64_t M) {
  return (w.K / 32) % 128 != 0 && StreamManyGroups(w, M);
}

// The prefill kernel serves the automatic GEMM path
// - when its 128 x 256 tiles alone fill at least one wave of CUs and the
//   last wave is at least half full: no split-K, one workgroup per CU (c5
//   qkv at M = 2048, 1.5 waves: 121.4 against GemmKernel's 130.6 us in one
//   process; a last wave below half stays with GemmKernel's smaller tiles);
// - when they do not fill one wave, with K split (PrefillSplits) as long as
//   each split keeps at least 12 k-tiles (shorter splits spend most of their
//   time in the prologue and the epilogue).
// Measured on MI355X (us per call, GemmKernel's best shape against the
// prefill kernel with PrefillSplits): M = 2048 c4, c5 o, gate+up, down
// 10-17% faster; M = 1024 c5 qkv 81.5 -> 61.8, o 61.8 -> 52.8, down
// 162.7 -> 125.9, c4 60.2 -> 52.6; M = 512 qkv 55.1 -> 46.3, down 96.4 ->
// 77.2, o and c4 within 3%; M = 256 gate+up 84.8 -> 63.8, qkv 34.6 -> about
// 32, down 56.8 -> 50.0; with fewer than 12 k-tiles per split (o and c4 at
// M <= 256, qkv at M = 128) GemmKernel's smaller tiles were 1-2 us faster;
// - from 33 rows where groups x segments are many (above).
// Asked where the streaming kernel does not serve: its rows, sizes or routes, or
// too little workspace.
bool UsePrefill(const WeightView &w, int64_t M) {
  if (!PrefillSupportsM(w, M)) return false;
  // 17-64 rows the streaming kernel does not serve, on weights of 192 Mi
  // elements and more: the prefill kernel's tiles over GemmKernel's (K =
  // 29568, N = 8192 at M = 17 / 32 / 64: 66.5 / 67.2 / 74.1 against 80.2 /
  // 81.6 / 92.3 us; smaller weights stay: K = 20608, N = 2048 45 against 27).
  const bool large = M >= 17 && w.K * w.N >= (int64_t{192} << 20);
  if (M < 65 && !large && !StreamManyGroups(w, M)) return false;
  const int64_t tiles = (M + kPTM - 1) / kPTM * ((w.N + kPTN - 1) / kPTN);
  const int64_t cus = w.num_cus;
  if (tiles < cus) {
    const int64_t splits = std::min<int64_t>(cus / tiles, kPrefillCheckSplits);
    return w.K / kBK >= 12 * splits;
  }
  const int64_t last = tiles - (tiles - 1) / cus * cus;  // workgroups in the last wave
  return last * 2 >= cus;
}

// The wide kernel, by waves of one workgroup per CU: one of its tiles takes
// 1.75 times a PrefillKernel tile (about 112 and 64 us at K = 4096) for twice
// the work, so it wins unless its last wave is emptier than the prefill
// kernel's by more than that (M = 700, N = 28672: 2 waves against 3, 208
// against 189 us). Where GemmKernel would serve, whose time goes with the
// work, 1.33 prefill waves per full wave of 128 x 256 tiles. Fewer tiles than
// CUs are the prefill kernel's (it splits K). Measured (us, prefill or
// GemmKernel -> wide): K = 4096, N = 28672 at M = 448 / 512 / 1024 / 1280 /
// 1536 / 2048 / 8192 128.8 -> 113.4, 132.8 -> 114.9, 262 -> 226, 369 -> 325,
// 445 -> 329, 448 -> 434, 1877 -> 1675 (with streaming stores, 1 to 6% slower
// than the plain ones that it has); N = 6144 at M = 2048 / 2560 / 8192
// 130 -> 112, 137 -> 127, 422 -> 376; K = 14336, N = 4096 at M = 3584 / 8192
// 431 -> 388, 928 -> 858; K = 8192, N = 8192 at M = 2048 257 -> 235. Below
// K = 2048 the un-overlapped prologue and stores of the larger tile take it
// back (K = 1024, N = 8192, M = 2048: 56.1 -> 57.8).
bool UseWide(const WeightView &w, int64_t M) {
  // 32-bit offsets within a tile's rows.
  if (!PrefillSupportsM(w, M) || w.K < 2048 || w.N >= (int64_t{1} << 21)) return false;
  const int64_t cus = w.num_cus;
  const int64_t tiles = (M + kPTM - 1) / kPTM * ((w.N + kPTN - 1) / kPTN);
  if (tiles < cus) return false;
  const int64_t wide = (M + kWideRows - 1) / kWideRows * ((w.N + kWideCols - 1) / kWideCols);
  const int64_t cost = 7 * ((wide + cus - 1) / cus) * cus;  // a prefill wave: 4 cus
  return UsePrefill(w, M) || w.B == nullptr ? cost <= 4 * ((tiles + cus - 1) / cus) * cus
                                            : cost * 3 <= 16 * tiles;
}

size_t PrefillPartialBytes(const WeightView &w, int64_t M) {
  return static_cast<size_t>(PrefillSplits(w, M) - 1) * static_cast<size_t>(M) * w.N * 4;
}

// 17 to 64 rows. Steps with no even division (a shorter last segment) above
// 32 rows: from 16 Mi weights; smaller ones stay with GemmKernel, whose route
// the tests fix (K = 11008, N = 1024 at M = 33 / 64 streamed 12.6 / 13.7
// against 16.3 / 16.9 us; N = 2048 14.6 / 16.4 against 18.2 / 19.3, N = 4096
// 21.0 / 23.0 against 25.2 / 26.9; K = 2816, N = 20480 at M = 33 / 48 / 64
// 23.0 / 24.8 / 28.9 against 26.8 / 27.9 / 28.9).
bool StreamServes(const WeightView &w, int64_t M) {
  if (!PrefillSupportsShape(w) || w.K > (int64_t{1} << 22) || StreamCrowded(w, M)) return false;
  return M <= 32 || w.K * w.N >= (int64_t{16} << 20) || StreamEven(w);
}

bool StreamSupportsM(const WeightView &w, int64_t M) {
  return M >= 17 && M <= 64 && PickStreamShape(w, M, 0, 0).segs > 0;
}

size_t StreamPartialBytes(const WeightView &w, int64_t M, int segs) {
  return static_cast<size_t>(std::max(segs, 1) - 1) * static_cast<size_t>(M) * w.N * 4;
}

} // namespace

// Without StreamKernel.
static size_t TiledWorkspaceBytes(const WeightView &w, int64_t M) {
  size_t partial = w.B != nullptr ? PartialBytes(w, M, PickShape(w, M)) : 0;
  if (PrefillSupportsM(w, M)) partial = std::max(partial, PrefillPartialBytes(w, M));
  return AImageBytes(w, M) + RowExpBytes(M) + partial;
}

// Its partial sums can be far larger than the tiled kernels' (K = 8320, N =
// 11008 at M = 64 36 MB against 13): with less to be had those serve.
static bool GemmStreams(const WeightView &w, int64_t M, size_t limit) {
  return StreamSupportsM(w, M) &&
         std::max(StreamWorkspaceBytes(w, M, 0, 0), TiledWorkspaceBytes(w, M)) <= limit;
}

size_t GemmWorkspaceBytes(const WeightView &w, int64_t M, size_t limit) {
  const size_t tiled = TiledWorkspaceBytes(w, M);
  return GemmStreams(w, M, limit) ? std::max(tiled, StreamWorkspaceBytes(w, M, 0, 0)) : tiled;
}

bool StreamSupports(const WeightView &w, int64_t M) { return StreamSupportsM(w, M); }

void SetStreamShapes(WeightView *w) {
  // StreamServes and the search answer alike for all rows of a class.
  constexpr int64_t kClassRows[4] = {24, 32, 48, 64};
  for (int i = 0; i < 4; ++i)
    w->stream[i] = StreamServes(*w, kClassRows[i]) ? SearchStreamShape(*w, kClassRows[i])
                                                   : StreamShape{0, 0, 0};
}

size_t StreamWorkspaceBytes(const WeightView &w, int64_t M, int segs, int spw) {
  const StreamShape sh = PickStreamShape(w, M, segs, spw);
  return AImageBytes(w, M) + StreamExpBytes(w, M) + StreamPartialBytes(w, M, sh.segs);
}

// The epilogue finishes fragments wave, wave + wpg, ... up to TG of them per
// wavefront, so it needs wpg >= 4 to reach all 4 TG; at most 8 wavefronts.
bool StreamShapeOk(const WeightView &w, int64_t M, int segs, int spw) {
  const StreamShape sh = PickStreamShape(w, M, segs, spw);
  // every step in a segment, no segment empty (the last may be shorter)
  const int64_t per = static_cast<int64_t>(sh.wpg) * sh.spw, T = w.K / 32;
  return StreamSupportsM(w, M) && sh.segs >= 1 && sh.segs <= kMaxSplits && sh.wpg >= 4 &&
         sh.wpg <= 8 && T % sh.spw == 0 && sh.segs * per >= T && (sh.segs - 1) * per < T;
}

// The chunk conversion, the streaming kernel, and the ordered reduction of the
// segments' partial sums when K is split.
hipError_t LaunchStream(const WeightView &w, int64_t M, const float *A, float *Y, void *work,
                        hipStream_t s, float *H, const float *gamma, float eps, const float *bias,
                        int segs, int spw) {
  const StreamShape sh = PickStreamShape(w, M, segs, spw);
  if (!StreamShapeOk(w, M, segs, spw)) return hipErrorInvalidValue;
  uint4 *Ah = static_cast<uint4 *>(work);
  int *exps = reinterpret_cast<int *>(static_cast<char *>(work) + AImageBytes(w, M));
  float *P = reinterpret_cast<float *>(static_cast<char *>(work) + AImageBytes(w, M) +
                                       StreamExpBytes(w, M));
  const bool cvt = gamma == nullptr && StreamConverts(w, M, sh);
  StreamIn in{Ah, cvt ? A : nullptr, exps, nullptr, eps};
  hipError_t e = hipSuccess;
  if (!cvt) {
    const int m = static_cast<int>(M), K = static_cast<int>(w.K);
    const int groups = static_cast<int>((M + 15) / 16), chunks = (K + kChunkK - 1) / kChunkK;
    float *sq = reinterpret_cast<float *>(exps + chunks * 16 * groups);
    const dim3 grid(chunks * groups * (16 / kChunkRows)), block(256);
    if (gamma != nullptr) {
      in.sq = sq;
      hipLaunchKernelGGL(ConvertChunkKernel<true>, grid, block, 0, s, A, Ah, exps, sq, gamma, m, K,
                         chunks, 16 * groups);
    } else {
      hipLaunchKernelGGL(ConvertChunkKernel<false>, grid, block, 0, s, A, Ah, exps, nullptr, nullptr,
                         m, K, chunks, 16 * groups);
    }
    e = hipGetLastError();
  }
  if (e != hipSuccess) return e;
  float *Hk = sh.segs == 1 ? H : nullptr;
  const float *bk = sh.segs == 1 ? bias : nullptr;
  e = w.has_zp ? LaunchStreamZp<true>(w, M, in, Y, P, Hk, bk, sh, s)
               : LaunchStreamZp<false>(w, M, in, Y, P, Hk, bk, sh, s);
  if (e != hipSuccess || sh.segs == 1) return e;
  return DispatchReduce(sh.segs - 1, Y, P, M * w.N, s, H,
                        std::make_integer_sequence<int, kMaxSplits - 1>{}, bias, w.N);
}

bool PrefillSupports(const WeightView &w, int64_t M) { return PrefillSupportsM(w, M); }


size_t PrefillLayoutBytes(const WeightView &w, size_t *sp_bytes) {
  const int64_t groups = (w.N + kPTN - 1) / kPTN * (kPTN / 64);
  const int64_t steps = w.K / 32;
  if (sp_bytes != nullptr) *sp_bytes = static_cast<size_t>(groups * w.nb * 256);
  return static_cast<size_t>(groups * steps * 1024);
}

bool PrefillLayoutWanted(const WeightView &w) {
  WeightView v = w;
  v.Bp = v.Sp = reinterpret_cast<const uint8_t *>(16);  // the shape checks only
  return PrefillSupportsShape(v) && (w.row_bytes % 16) == 0;
}

hipError_t LaunchPrefillRelayout(const WeightView &w, uint8_t *Bp, uint8_t *Sp, hipStream_t s) {
  size_t sp_bytes = 0;
  const size_t bp_bytes = PrefillLayoutBytes(w, &sp_bytes);
  const int64_t T = w.K / 32;
  const int64_t bw = static_cast<int64_t>(bp_bytes / 4), sw = static_cast<int64_t>(sp_bytes / 4);
  hipLaunchKernelGGL(RelayoutBKernel, StrideGrid(bw), dim3(256), 0, s, w.B,
                     reinterpret_cast<uint32_t *>(Bp), w.N, w.row_bytes, T, bw);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(RelayoutSKernel, StrideGrid(sw), dim3(256), 0, s, w.scales, w.zp,
                     w.col_exp, reinterpret_cast<uint32_t *>(Sp), w.N, w.nb, w.zp_row_bytes, sw);
  return hipGetLastError();
}

// ConvertA, the prefill kernel, and the split reduction when K is split.
static hipError_t LaunchPrefillGemm(const WeightView &w, int64_t M, const float *A, float *Y,
                                    void *work, hipStream_t s, float *H, const float *gamma,
                                    float eps, const float *bias, int splits) {
  uint4 *Ah = static_cast<uint4 *>(work);
  int *row_exp = reinterpret_cast<int *>(static_cast<char *>(work) + AImageBytes(w, M));
  float *partials = reinterpret_cast<float *>(static_cast<char *>(work) + AImageBytes(w, M) +
                                              RowExpBytes(M));
  hipError_t e = gamma != nullptr
                     ? LaunchConvertA<kPTM, true>(w, M, A, Ah, row_exp, s, gamma, eps)
                     : LaunchConvertA<kPTM, false>(w, M, A, Ah, row_exp, s, nullptr, 0.0f);
  if (e != hipSuccess) return e;
  // One split: the kernel's stores apply the gate/up activation or add the
  // bias. Several: the ordered reduction does, after the partial sums.
  float *Hk = splits == 1 ? H : nullptr;
  const float *bk = splits == 1 ? bias : nullptr;
  const bool zp = w.has_zp != 0, bs32 = w.block_size == 32;
  if (zp)
    e = bs32 ? LaunchPrefillT<true, true>(w, M, Ah, Y, partials, splits, s, Hk, row_exp, bk)
             : LaunchPrefillT<true, false>(w, M, Ah, Y, partials, splits, s, Hk, row_exp, bk);
  else
    e = bs32 ? LaunchPrefillT<false, true>(w, M, Ah, Y, partials, splits, s, Hk, row_exp, bk)
             : LaunchPrefillT<false, false>(w, M, Ah, Y, partials, splits, s, Hk, row_exp, bk);
  if (e != hipSuccess || splits == 1) return e;
  return DispatchReduce(splits - 1, Y, partials, M * w.N, s, H,
                        std::make_integer_sequence<int, kMaxSplits - 1>{}, bias, w.N);
}

// ConvertA and the wide kernel, which applies the gate/up activation or adds
// the bias in its stores.
static hipError_t LaunchWideGemm(const WeightView &w, int64_t M, const float *A, float *Y,
                                 void *work, hipStream_t s, float *H, const float *gamma,
                                 float eps, const float *bias) {
  uint4 *Ah = static_cast<uint4 *>(work);
  int *row_exp = reinterpret_cast<int *>(static_cast<char *>(work) + AImageBytes(w, M));
  const hipError_t e = gamma != nullptr
                           ? LaunchConvertA<16, true>(w, M, A, Ah, row_exp, s, gamma, eps)
                           : LaunchConvertA<16, false>(w, M, A, Ah, row_exp, s, nullptr, 0.0f);
  if (e != hipSuccess) return e;
  return LaunchWide(w, M, Ah, Y, H, row_exp, bias, s);
}

size_t GemmShapeWorkspaceBytes(const WeightView &w, int64_t M, int splits) {
  return AImageBytes(w, M) + RowExpBytes(M) + PartialBytes(w, M, MakeShape(w, 32, splits));
}

bool GemmSupports(const WeightView &w, int64_t M) {
  return GemmKernelSupports(w, M) || PrefillSupportsM(w, M);
}

bool GemmKernelSupports(const WeightView &w, int64_t M) {
  // Buffer offsets are 32-bit within one tile of 128 weight rows; up to 16
  // splits of the BM = 32 tiling must fit one grid.
  const int64_t tiles = ((M + 31) / 32) * ((w.N + kBN - 1) / kBN) * 16;
  return w.B != nullptr && M >= 1 && (w.K % kBK) == 0 && w.block_size >= 32 &&
         tiles < (int64_t{1} << 31) &&
         int64_t{kBN} * w.row_bytes < (int64_t{1} << 31) &&
         int64_t{kBN} * w.nb * 4 < (int64_t{1} << 31) && (w.row_bytes % 16) == 0 &&
         (reinterpret_cast<uintptr_t>(w.B) % 16) == 0 && M <= (int64_t{1} << 30) &&
         w.N <= (int64_t{1} << 30) && w.K <= (int64_t{1} << 24);
}

hipError_t LaunchPrefill(const WeightView &w, int64_t M, const float *A, float *Y, void *work,
                         hipStream_t s, float *H, const float *gamma, float eps, const float *bias,
                         bool *bias_done) {
  if (bias_done != nullptr) *bias_done = bias != nullptr;
  return LaunchPrefillGemm(w, M, A, Y, work, s, H, gamma, eps, bias, PrefillSplits(w, M));
}

hipError_t LaunchGemmShape(const WeightView &w, int64_t M, const float *A, float *Y, void *work,
                           hipStream_t s, int bm, int splits, float *H, const float *gamma,
                           float eps) {
  if (bm == kPrefillTileCode) {
    if (!PrefillSupportsShape(w)) return hipErrorInvalidValue;
    const int ktiles = static_cast<int>(w.K / kBK);
    splits = std::max(1, std::min({splits, ktiles, kMaxSplits}));
    const int per = (ktiles + splits - 1) / splits;
    return LaunchPrefillGemm(w, M, A, Y, work, s, H, gamma, eps, nullptr, (ktiles + per - 1) / per);
  }
  if (w.B == nullptr) return hipErrorInvalidValue;  // GemmKernel reads the original layout
  Shape sh = PickShape(w, M);
  if (bm > 0) sh = MakeShape(w, bm, splits > 0 ? splits : 1);
  switch (sh.bm) {
  case 32: return LaunchBM<32>(w, M, A, Y, work, sh, s, H, gamma, eps);
  case 64: return LaunchBM<64>(w, M, A, Y, work, sh, s, H, gamma, eps);
  case 128: return LaunchBM<128>(w, M, A, Y, work, sh, s, H, gamma, eps);
  default: return hipErrorInvalidValue;
  }
}

hipError_t LaunchGemm(const WeightView &w, int64_t M, const float *A, float *Y, void *work,
                      hipStream_t s, float *H, const float *gamma, float eps, const float *bias,
                      bool *bias_done, size_t limit) {
  if (bias_done != nullptr) *bias_done = false;
  if (GemmStreams(w, M, limit)) {
    if (bias_done != nullptr) *bias_done = bias != nullptr;
    return LaunchStream(w, M, A, Y, work, s, H, gamma, eps, bias, 0, 0);
  }
  if (UseWide(w, M)) {
    if (bias_done != nullptr) *bias_done = bias != nullptr;
    return LaunchWideGemm(w, M, A, Y, work, s, H, gamma, eps, bias);
  }
  // A compact plan (no original layout) always takes one of the kernels on the
  // re-laid weights.
  if (UsePrefill(w, M) || w.B == nullptr) {
    if (bias_done != nullptr) *bias_done = bias != nullptr;
    return LaunchPrefillGemm(w, M, A, Y, work, s, H, gamma, eps, bias, PrefillSplits(w, M));
  }
  return LaunchGemmShape(w, M, A, Y, work, s, 0, 0, H, gamma, eps);
}

bool GemmUsesPrefill(const WeightView &w, int64_t M) { return UsePrefill(w, M) || w.B == nullptr; }

bool GemmUsesStream(const WeightView &w, int64_t M) { return StreamSupportsM(w, M); }

bool GemmUsesWide(const WeightView &w, int64_t M) {
  return !StreamSupportsM(w, M) && UseWide(w, M);
}

} // namespace mnb
