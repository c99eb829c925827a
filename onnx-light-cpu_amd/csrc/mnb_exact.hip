// Exact-activation GEMM for MatMulNBits on CDNA4 fp16 MFMA: many rows with
// activations kept to 22 bits or in full instead of the GEMM's 11, over the
// fragment-ordered weights.
//
// It serves the rows that must not take the fp16 GEMM above 16 of them
// (accuracy_level 1), whole groups of 16 at a time, and every K the 64-k
// tiles of the other kernels do not divide. fp32 semantics as the reference
// engine's product (onnx_light_cpu/impl/math/gemm_kernel.cc:1208-1258): q - zp
// is exact, the products are summed in fp32.
//
// Two kernels per call:
//
// 1. SplitRowsKernel: each (row, 256-k unit) of A is scaled by a power of two
//    (largest magnitude in [2^14, 2^15), exact) and split into TERMS fp16
//    terms, written as MFMA operand records [16-row group][32-k step][term]
//    [lane] (lane l: row l & 15, k 8 (l >> 4) .. + 7 of the step in the weight
//    decode's [0,4,1,5,2,6,3,7] order) with the exponents [unit][row]. Values
//    past K and rows past M are zero. TERMS = 2 keeps 22 bits, the operands
//    and exponents of DecodeFragKernel; TERMS = 3 keeps all 24.
//
// 2. ExactKernel. A workgroup of four wavefronts owns 16 MI rows x 256
//    columns and a run of 256-k units; wavefront w owns 64 columns (one weight
//    group) and all of the run. Every operand streams global -> LDS through
//    direct copies into a ring of NS stages of one 64-k tile each (the
//    activation records shared by the four wavefronts, each wavefront's own
//    weight, scale, zero point records and the rows' exponents); two
//    workgroups share a CU so that one multiplies while the other waits. Per
//    step a wavefront decodes its record's four words once (q - zp, 9 VALU
//    per 8 weights) for 4 MI TERMS MFMAs; at each block's end the products
//    are multiplied by the rows' fp32 scales into the unit's sum, at each
//    unit's end that sum, times 2^-e, goes into the sum of `units_per_range`
//    units, and those sums are added in order: with the run and range lengths
//    of DecodeFragKernel's launch every 16-row group gets the bits that the
//    decode path gives it. Runs that do not cover K write partial sums, added
//    in run order by the partial-sum pass; where the row and column tiles
//    alone fill the chip a workgroup takes all runs in turn and adds their
//    sums itself, in the same order.
//
// Bound: the vector ALUs. A step of a wavefront (MI = 2, TERMS = 2) is 16
// MFMAs (256 matrix cycles) against 36 decode + 32 scale VALU at 32-k blocks
// (96 with the zero points and unit sums, 384 cycles; 60 at 128-k blocks).
// Measured per call: accuracy_level 1, K = 4096, N = 6144, M = 256, 32-k blocks
// and a bias 197 -> 51 us (16 groups through the decode kernels before), the
// same bits; K = 2500, N = 5001, M = 333 6338 -> 47 us (GenericKernel before),
// error against 64 bits 1.3e-7 -> 7e-8.
#include "mnb_decode_common.h"

#include <algorithm>

namespace mnb {
namespace ek {

using namespace dec;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kUnitK = 256;     // k per activation exponent
constexpr int kUnitSteps = 8;   // 32-k steps per unit
constexpr int kUnitTiles = 4;   // 64-k tiles per unit
constexpr int kThreads = 256;   // four wavefronts, 64 columns each
constexpr int kCols = 256;
constexpr int kRecord = 64;     // 16-byte units per 1 KiB operand record

// 16-byte units of one stage: activation records, then per wavefront two
// weight records and one 1 KiB record of scales (lanes 0-15 step 0's block,
// 16-31 step 1's), zero points (32-35, 36-39) and exponents (40-55).
template <int MI, int TERMS>
constexpr int AUnits() { return MI * 2 * TERMS * kRecord; }
template <int MI, int TERMS>
constexpr int StageUnits() { return AUnits<MI, TERMS>() + 4 * 3 * kRecord; }
// Stages: four where two workgroups then still fit the 160 KiB of a CU.
template <int MI, int TERMS>
constexpr int Stages() { return StageUnits<MI, TERMS>() * 16 * 4 <= 80 * 1024 ? 4 : 3; }
template <int MI, int TERMS>
constexpr size_t LdsBytes() { return size_t{16} * StageUnits<MI, TERMS>() * Stages<MI, TERMS>(); }

// One workgroup of 8 wavefronts per (256-k unit, group of 16 rows); wavefront
// w takes step w, lane l the 8 values k = 256 u + 32 w + 8 (l >> 4) .. + 7 of
// row l & 15. Rows of K floats need no alignment beyond 4 bytes.
template <int TERMS>
__global__ __launch_bounds__(512) void SplitRowsKernel(const float *__restrict__ A,
                                                       uint4 *__restrict__ img,
                                                       int *__restrict__ exps, int M, int K,
                                                       int units, int rows_padded) {
  __shared__ float red[8][16];
  const int u = static_cast<int>(blockIdx.x) % units;
  const int mt = static_cast<int>(blockIdx.x) / units;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15;
  const int rows = min(16, M - 16 * mt);  // <= 0: a padding group, all zero
  const int k0 = kUnitK * u + 32 * wave + 8 * (lane >> 4);
  const int bytes = max(rows, 0) * K * 4;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(A + static_cast<size_t>(min(16 * mt, M - 1)) * K), 0, bytes, 0x00020000);
  // loads past the buffer give zeros
  const int vo = r < rows && k0 < K ? (r * K + k0) * 4 : bytes;
  float x[8];
  if ((K & 7) == 0) {
    const floatx4 v0 = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ra, vo, 0, 0));
    const floatx4 v1 = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ra, vo + 16, 0, 0));
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = i < 4 ? v0[i & 3] : v1[i & 3];
  } else {
    // the row may end inside the 8: one load per value, those past K beyond the buffer
#pragma unroll
    for (int i = 0; i < 8; ++i)
      x[i] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(ra, k0 + i < K ? vo + 4 * i : bytes, 0, 0));
  }
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(x[i]));
  amax = fmaxf(amax, Xor16(amax));
  amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
  if (lane < 16) red[wave][lane] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 8; ++w) amax = fmaxf(amax, red[w][r]);
  // exact for every e this gives, subnormal inputs included; inf and NaN
  // propagate in their first term
  const int e = SplitExponent(amax, kRowExpTarget);
  if (threadIdx.x < 16) exps[static_cast<size_t>(u) * rows_padded + 16 * mt + lane] = e;
  half8 h[TERMS];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int o = (i & 3) * 2 + (i >> 2);  // k order [0,4,1,5,2,6,3,7]
    float rest = ldexpf(x[i], e);
    const bool finite = __builtin_isfinite(rest);
#pragma unroll
    for (int t = 0; t < TERMS; ++t) {
      const _Float16 term = static_cast<_Float16>(rest);
      h[t][o] = term;
      rest = finite ? rest - static_cast<float>(term) : 0.f;
    }
  }
  uint4 *dst = img + (static_cast<size_t>(mt) * units * kUnitSteps + kUnitSteps * u + wave) *
                         (TERMS * kRecord) + lane;
#pragma unroll
  for (int t = 0; t < TERMS; ++t) dst[t * kRecord] = __builtin_bit_cast(uint4, h[t]);
}

// The launch's K structure (host: MakeShape). Units 0 .. units - 1 form runs
// of run_units, each run's units ranges of range_units.
struct Shape {
  int units, runs, run_units, range_units;
  bool all_runs;  // one workgroup takes every run
};

template <bool HAS_ZP, int SPB, int MI, int TERMS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void ExactKernel(
    const uint4 *__restrict__ img, const int *__restrict__ exps, const uint8_t *__restrict__ Bp,
    const float *__restrict__ Sd, const uint32_t *__restrict__ Zd, float *__restrict__ Y,
    float *__restrict__ partials, float *__restrict__ H, const float *__restrict__ bias, int M,
    int N, int T, int nb, int log2_bs, int groups, int rows_padded, Shape sh) {
  extern __shared__ uint4 lds[];
  constexpr int kNS = Stages<MI, TERMS>();
  constexpr int kStage = StageUnits<MI, TERMS>();
  constexpr int kA = AUnits<MI, TERMS>();
  constexpr int kACopies = (kA / kRecord + 3) / 4;  // activation copies per wavefront and tile
  constexpr int kOps = kACopies + 3;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int c = lane & 15, qd = lane >> 4;

  // Workgroup b -> (run, column tile, row tile): neighbours share the weights.
  const int mtiles = rows_padded / (16 * MI), ntiles = (N + kCols - 1) / kCols;
  int b = static_cast<int>(blockIdx.x);
  const int total = mtiles * ntiles * (sh.all_runs ? 1 : sh.runs);
  if (total % 8 == 0) b = (b & 7) * (total / 8) + (b >> 3);  // an XCD takes a contiguous part
  const int tm = b % mtiles;
  const int tn = b / mtiles % ntiles;
  const int run0 = b / (mtiles * ntiles);
  const int m0 = tm * 16 * MI;
  const int g = 4 * tn + wave;
  const int u_begin = run0 * sh.run_units;
  const int u_end = sh.all_runs ? sh.units : min(sh.units, u_begin + sh.run_units);
  const int tiles = (u_end - u_begin) * kUnitTiles;
  const int t_last = T / 2 - 1;  // last 64-k tile of the weights (T is even)

  // Copy sources. Activations: record p of the stage is (fragment, step,
  // term) of the tile; copies past the last record repeat it.
  const int steps = sh.units * kUnitSteps;
  const uint4 *a_src[kACopies];
  uint32_t a_dst[kACopies];
#pragma unroll
  for (int i = 0; i < kACopies; ++i) {
    const int p = min(4 * i + wave, kA / kRecord - 1);
    const int frag = p / (2 * TERMS), rec = p - frag * 2 * TERMS;
    a_src[i] = img + ((static_cast<size_t>(tm) * MI + frag) * steps * TERMS + rec) * kRecord;
    a_dst[i] = static_cast<uint32_t>(p * kRecord * 16);
  }
  const uint8_t *b_src = Bp + static_cast<size_t>(g) * T * 1024;
  const uint32_t l16 = static_cast<uint32_t>(lane) * 16;
  // The mixed record: lane -> base, byte stride per index and which index.
  // Columns past the last group (N up to a multiple of 256) repeat its scales.
  const int gs = min(g, groups - 1);
  const bool is_e = lane >= 40 && lane < 40 + 4 * MI;
  const bool is_z = HAS_ZP && lane >= 32 && lane < 40;
  const int half = is_z ? (lane >> 2) & 1 : lane < 32 ? lane >> 4 : 0;  // the step of the tile
  const char *m_base;
  uint32_t m_stride;
  if (is_e) {
    m_base = reinterpret_cast<const char *>(exps + m0 + 4 * (lane - 40));
    m_stride = static_cast<uint32_t>(rows_padded) * 4;
  } else if (is_z) {
    m_base = reinterpret_cast<const char *>(Zd + static_cast<size_t>(gs) * nb * 16 + 4 * (lane & 3));
    m_stride = 64;
  } else {
    m_base = reinterpret_cast<const char *>(Sd + static_cast<size_t>(gs) * nb * 64 + 4 * c);
    m_stride = 256;
  }
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const uint32_t b_dst = lds0 + static_cast<uint32_t>((kA + wave * 3 * kRecord) * 16);
  auto issue = [&](int t, int stage) {
    const int tl = min(t, tiles - 1);  // past the run: repeats, into stages nobody reads
    const int kt = u_begin * kUnitTiles + tl;
    const int ktb = min(kt, t_last);   // past K: the activations are zero
    const uint32_t st = static_cast<uint32_t>(stage * kStage * 16);
#pragma unroll
    for (int i = 0; i < kACopies; ++i)
      CopyToLds16S(a_src[i] + static_cast<size_t>(kt) * (2 * TERMS * kRecord), l16,
                   lds0 + st + a_dst[i]);
    CopyToLds16S(b_src + static_cast<size_t>(ktb) * 2048, l16, b_dst + st);
    CopyToLds16S(b_src + static_cast<size_t>(ktb) * 2048 + 1024, l16, b_dst + st + 1024);
    const int blk = min((64 * ktb + 32 * half) >> log2_bs, nb - 1);
    const int idx = is_e ? kt / kUnitTiles : blk;
    CopyToLds16(m_base + static_cast<size_t>(static_cast<uint32_t>(idx)) * m_stride,
                b_dst + st + 2048);
  };

  const Masks mk = MakeMasks();
  // kLow: the terms after the first in accumulators of their own, added to the
  // first's once per block. In one chain every small term would be rounded to
  // the large sum's last place: K = 1003, 128-wide blocks 1.08e-7 off 64 bits
  // instead of 6.2e-8 (GenericKernel 1.06e-7). (Two terms keep DecodeFragKernel's one chain.)
  constexpr bool kLow = TERMS == 3;
  floatx4 tmp[MI][4], low[kLow ? MI : 1][4], racc[MI][4], acc[MI][4], run[MI][4], sum[MI][4];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      tmp[i][j] = racc[i][j] = acc[i][j] = run[i][j] = sum[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

#pragma unroll
  for (int p = 0; p < kNS - 1; ++p) issue(p, p);
  int stage = 0, in_range = 0, in_run = 0;
  for (int u = u_begin; u < u_end; ++u) {
    const uint4 *sb = nullptr;
#pragma unroll
    for (int tt = 0; tt < kUnitTiles; ++tt) {
      const int t = (u - u_begin) * kUnitTiles + tt;
      // Tile t has landed (the copies of the kNS - 2 tiles after it may be
      // outstanding) and every wavefront is past tile t - 1.
      WaitVm<kOps * (kNS - 2)>();
      __syncthreads();
      issue(t + kNS - 1, stage == 0 ? kNS - 1 : stage - 1);
      sb = lds + stage * kStage;
      stage = stage + 1 == kNS ? 0 : stage + 1;
      const uint4 *wb = sb + kA + wave * 3 * kRecord;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        constexpr int kSpb = SPB;
        const int s = 2 * tt + h;  // step of the unit
        half8 a[MI][TERMS];
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int x = 0; x < TERMS; ++x)
            a[i][x] = __builtin_bit_cast(half8, sb[(i * 2 * TERMS + h * TERMS + x) * kRecord + lane]);
        const uint4 w4 = wb[h * kRecord + lane];
        uint32_t neg_lo[4], neg_hi[4];
        uint32_t z = 0;
        if constexpr (HAS_ZP)
          z = reinterpret_cast<const uint32_t *>(wb + 2 * kRecord + 32 + 4 * h)[c];
        const uint32_t wv[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // byte j is the zero point of column 16 j + c: fp16 -(1024 + zp)
          // and -(64 + zp)
          const uint32_t zz = HAS_ZP ? ((z >> (8 * j)) & 0xFu) * 0x10001u : 0x00080008u;
          neg_lo[j] = zz | 0xE400E400u;
          neg_hi[j] = (zz << 4) | 0xD400D400u;
          const half8 q = DecodeQ(wv[j], neg_lo[j], neg_hi[j], mk);
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            if (s % kSpb == 0) tmp[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
            if constexpr (kLow) {
              if (s % kSpb == 0) low[kLow ? i : 0][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int x = TERMS - 1; x > 0; --x)
                low[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][x], q, low[i][j], 0, 0, 0);
              tmp[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][0], q, tmp[i][j], 0, 0, 0);
            } else {
#pragma unroll
              for (int x = 0; x < TERMS; ++x)
                tmp[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][x], q, tmp[i][j], 0, 0, 0);
            }
          }
        }
        if ((s + 1) % kSpb == 0) {
          const floatx4 bsc = __builtin_bit_cast(floatx4, wb[2 * kRecord + 16 * h + c]);
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                racc[i][j][v] = fmaf(bsc[j], kLow ? tmp[i][j][v] + low[kLow ? i : 0][j][v] : tmp[i][j][v],
                                     s + 1 == kSpb ? 0.f : racc[i][j][v]);
        }
      }
    }
    // The unit's sum times 2^-e (exact) into its range's, ranges into the
    // run's and runs into the total, each in order.
    const bool range_start = in_range == 0;
    const bool range_end = ++in_range == sh.range_units || u + 1 == u_end;
    const bool run_start = in_run == 0 || in_run < sh.range_units;
    const bool run_end = ++in_run == sh.run_units || u + 1 == u_end;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int4 e4 = __builtin_bit_cast(
          int4, sb[kA + wave * 3 * kRecord + 2 * kRecord + 40 + 4 * i + qd]);
      const int ev[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float x = __builtin_amdgcn_ldexpf(racc[i][j][v], -ev[v]);
          acc[i][j][v] = range_start ? x : acc[i][j][v] + x;
        }
    }
    if (range_end) {
      in_range = 0;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          run[i][j] = kLow || run_start ? acc[i][j] : run[i][j] + acc[i][j];  // kLow: one range
    }
    if (run_end) {
      const bool first = u < sh.run_units || !sh.all_runs;
      in_run = 0;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[i][j] = first ? run[i][j] : sum[i][j] + run[i][j];
    }
  }
  // No copy into this workgroup's LDS may land after it exits.
  WaitVm<0>();

  // Lane l holds rows m0 + 16 i + 4 qd + v of column 64 g + 16 j + c. Offsets
  // are from this tile's first row (at most 32 rows of N < 2^22 floats); rows
  // past M fall beyond the buffer and columns past N are sent there.
  float *out = run0 == 0 ? Y : partials + static_cast<size_t>(run0 - 1) * M * N;
  const int rows = min(M - m0, 16 * MI);
  if (rows <= 0) return;
  const int width = H != nullptr ? N >> 1 : N;
  const int end = rows * width * 4;
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(
      (H != nullptr ? H : out) + static_cast<size_t>(m0) * width, 0, end, 0x00020000);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = 64 * g + 16 * j + c;
    const float bv = bias != nullptr ? bias[min(n, N - 1)] : 0.f;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * i + 4 * qd + v;
        const float y = sum[i][j][v];
        float val = bias != nullptr ? y + bv : y;
        int off = n < N && row < rows ? (row * N + n) * 4 : end;
        if (H != nullptr) {  // gate/up pairs in lanes c, c ^ 1 (N even)
          val = SiluMul(y, PairSwap(y));
          off = (c & 1) == 0 && n < N && row < rows ? (row * width + (n >> 1)) * 4 : end;
        }
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, val), ry, off, 0, 0);
      }
  }
}

template <bool HAS_ZP, int SPB, int MI, int TERMS>
hipError_t Launch(const WeightView &w, int64_t M, const uint4 *img, const int *exps, float *Y,
                  float *P, float *H, const float *bias, const Shape &sh, int T,
                  int64_t rows_padded, hipStream_t s) {
  const int64_t tiles = rows_padded / (16 * MI) * ((w.N + kCols - 1) / kCols);
  const dim3 grid(static_cast<unsigned>(tiles * (sh.all_runs ? 1 : sh.runs)));
  hipLaunchKernelGGL((ExactKernel<HAS_ZP, SPB, MI, TERMS>), grid, dim3(kThreads),
                     (LdsBytes<MI, TERMS>()), s, img, exps, w.Bp, w.Sd, w.Zd, Y, P, H, bias,
                     static_cast<int>(M), static_cast<int>(w.N), T, static_cast<int>(w.nb),
                     w.log2_bs, static_cast<int>((w.N + 63) / 64), static_cast<int>(rows_padded),
                     sh);
  return hipGetLastError();
}

template <int MI, int TERMS, class... Args>
hipError_t LaunchSpb(const WeightView &w, Args... args) {
  const int spb = std::min(w.block_size / 32, kUnitSteps);
  if (w.has_zp) switch (spb) {
    case 1: return Launch<true, 1, MI, TERMS>(w, args...);
    case 2: return Launch<true, 2, MI, TERMS>(w, args...);
    case 4: return Launch<true, 4, MI, TERMS>(w, args...);
    default: return Launch<true, 8, MI, TERMS>(w, args...);
  }
  switch (spb) {
  case 1: return Launch<false, 1, MI, TERMS>(w, args...);
  case 2: return Launch<false, 2, MI, TERMS>(w, args...);
  case 4: return Launch<false, 4, MI, TERMS>(w, args...);
  default: return Launch<false, 8, MI, TERMS>(w, args...);
  }
}

// Whether the plan holds the ragged-K layout (fp32-exact route of any K)
// rather than the 64-k one (DecodeFragKernel's operands and order).
inline bool Ragged(const WeightView &w) { return (w.K % 64) != 0; }
inline int Steps(const WeightView &w) { return static_cast<int>((w.K + 63) / 64 * 2); }
inline int Units(const WeightView &w) { return static_cast<int>((w.K + kUnitK - 1) / kUnitK); }
inline int Terms(const WeightView &w) { return Ragged(w) ? 3 : 2; }
inline int TileRows(const WeightView &w, int64_t M) { return Ragged(w) && M <= 16 ? 16 : 32; }
inline int64_t PaddedRows(const WeightView &w, int64_t M) {
  const int64_t t = TileRows(w, M);
  return (M + t - 1) / t * t;
}

// Runs of K. 64-k plans take DecodeFragKernel's runs and ranges (its bits);
// ragged ones as many runs of at least two units as keep the launch within
// the two workgroups per CU, one range each. All runs in one workgroup
// where the tiles alone are three quarters of those.
inline Shape MakeShape(const WeightView &w, int64_t M) {
  Shape sh;
  sh.units = Units(w);
  const int64_t tiles =
      PaddedRows(w, M) / TileRows(w, M) * ((w.N + kCols - 1) / kCols);
  const int64_t slots = 2 * static_cast<int64_t>(w.num_cus);
  if (Ragged(w)) {
    const int64_t want = std::max<int64_t>(1, std::min<int64_t>(slots / tiles, sh.units / 2));
    sh.run_units = static_cast<int>((sh.units + want - 1) / want);
    sh.range_units = sh.run_units;
  } else {
    DecodeFragRuns(w, &sh.run_units, &sh.range_units);
  }
  sh.runs = (sh.units + sh.run_units - 1) / sh.run_units;
  sh.all_runs = sh.runs == 1 || tiles * 4 >= slots * 3;
  return sh;
}

inline size_t ImageBytes(const WeightView &w, int64_t M) {
  return static_cast<size_t>(PaddedRows(w, M)) * Units(w) * kUnitK * 2 * Terms(w);
}
inline size_t ExpBytes(const WeightView &w, int64_t M) {
  return (static_cast<size_t>(PaddedRows(w, M)) * Units(w) * 4 + 255) / 256 * 256;
}

__global__ __launch_bounds__(256) void RelayoutRaggedKernel(const uint8_t *__restrict__ B,
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
    const int64_t byte = 16 * s + 4 * (l >> 4);
    Bp[idx] = n < N && byte + 4 <= row_bytes
                  ? *reinterpret_cast<const uint32_t *>(B + n * row_bytes + byte)
                  : 0u;
  }
}

// out[b]: the largest magnitude (its bits; infinite and NaN above all) of
// workgroup b's share of the scales.
__global__ __launch_bounds__(256) void LargestScaleKernel(const float *__restrict__ S, int64_t n,
                                                          uint32_t *__restrict__ out) {
  __shared__ uint32_t red[4];
  uint32_t m = 0;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * 256)
    m = max(m, __float_as_uint(S[i]) & 0x7FFFFFFFu);
  for (int off = 32; off >= 1; off >>= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(m, off, 64)));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = max(max(red[0], red[1]), max(red[2], red[3]));
}

} // namespace ek

hipError_t ExactRaggedScalesOk(const WeightView &w, uint32_t *work, bool *ok) {
  uint32_t top[kScaleCheckWords];
  hipLaunchKernelGGL(ek::LargestScaleKernel, dim3(kScaleCheckWords), dim3(256), 0, nullptr, w.scales,
                     w.N * w.nb, work);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpy(top, work, sizeof(top), hipMemcpyDeviceToHost);
  if (e != hipSuccess) return e;
  constexpr uint32_t kLimit = (127u + 101u) << 23;  // 2^101
  *ok = *std::max_element(top, top + kScaleCheckWords) < kLimit;
  return hipSuccess;
}

bool ExactRaggedLayoutWanted(const WeightView &w) {
  return w.B != nullptr && ek::Ragged(w) && w.block_size >= 32 && w.K <= (int64_t{1} << 24) &&
         w.N < (int64_t{1} << 22) && w.nb * 256 < (int64_t{1} << 31);
}

size_t ExactRaggedLayoutBytes(const WeightView &w) {
  return static_cast<size_t>((w.N + ek::kCols - 1) / ek::kCols * 4) * ek::Steps(w) * 1024;
}

hipError_t LaunchExactRaggedRelayout(const WeightView &w, uint8_t *Bp, hipStream_t s) {
  const int64_t words = static_cast<int64_t>(ExactRaggedLayoutBytes(w) / 4);
  hipLaunchKernelGGL(ek::RelayoutRaggedKernel, StrideGrid(words), dim3(256), 0, s, w.B,
                     reinterpret_cast<uint32_t *>(Bp), w.N, w.row_bytes, ek::Steps(w), words);
  return hipGetLastError();
}

bool ExactSupports(const WeightView &w, int64_t M) {
  if (M < 1 || M > (int64_t{1} << 22) || w.Bp == nullptr || w.Sd == nullptr ||
      (w.has_zp && w.Zd == nullptr))
    return false;
  if (!ek::Ragged(w) && (M % 16 != 0 || !DecodeFragSupports(w, 16))) return false;
  // 32-bit grids and row offsets
  const int64_t tiles = ek::PaddedRows(w, M) / 16 * ((w.N + ek::kCols - 1) / ek::kCols);
  return w.N < (int64_t{1} << 22) && w.K <= (int64_t{1} << 24) &&
         tiles * std::max(16, ek::Units(w)) < (int64_t{1} << 31);
}

// A workgroup multiplies a run of K one unit after the other (2.8 us each) while
// DecodeFragKernel spreads it over wavefronts, so with few rows long runs are
// the decode kernel's. Estimates in us; over 42 weights and two block sizes the
// faster one is taken but for K = 8192, N = 28672 at 48 rows with 128-wide blocks
// (92.9 by groups, 102.8 taken) and some within 4%. us, groups against this, at
// 32 / 48 rows: K = 14336, N = 4096 (runs of 14) 32.4 /
// 49.0 against 50.2 / 51.8; K = N = 4096 (4) 19.3 / 28.4, 23.2 / 23.5; K =
// 4096, N = 28672 (16) 42.1 / 58.7, 56.2 / 55.6; K = 14336, N = 11008 (14, but
// three rounds of decode workgroups) 66.7 / 96.4, 56.4 / 75.5; K = N = 2048 (1)
// 18.1 / 27.1, 14.5 / 14.8.
bool ExactBeatsGroups(const WeightView &w, int64_t M) {
  int run = 1, range = 1;
  DecodeFragRuns(w, &run, &range);
  const int64_t cus = std::max(1, w.num_cus), runs = (ek::Units(w) + run - 1) / run;
  const int64_t tiles = ek::PaddedRows(w, M) / 32 * ((w.N + ek::kCols - 1) / ek::kCols);
  const double exact = 11.5 + 2.8 * run * std::max(1.0, static_cast<double>(tiles * runs) / cus);
  const int64_t rounds = ((w.N + 63) / 64 * runs + cus - 1) / cus;
  const double group = (runs > 1 ? 8.3 : 6.3) + 0.43 * static_cast<double>(rounds * run) +
                       (range > 1 ? 1.0 : 0.0);
  return exact < group * static_cast<double>(M / 16);
}

size_t ExactWorkspaceBytes(const WeightView &w, int64_t M) {
  const ek::Shape sh = ek::MakeShape(w, M);
  const size_t parts = sh.all_runs ? 0 : static_cast<size_t>(sh.runs - 1);
  return ek::ImageBytes(w, M) + ek::ExpBytes(w, M) + parts * static_cast<size_t>(M) * w.N * 4;
}

hipError_t LaunchExact(const WeightView &w, int64_t M, const float *A, float *Y, void *work,
                       hipStream_t s, float *H, const float *bias) {
  if (!ExactSupports(w, M)) return hipErrorInvalidValue;
  const ek::Shape sh = ek::MakeShape(w, M);
  const int64_t rows = ek::PaddedRows(w, M);
  char *base = static_cast<char *>(work);
  uint4 *img = reinterpret_cast<uint4 *>(base);
  int *exps = reinterpret_cast<int *>(base + ek::ImageBytes(w, M));
  float *P = reinterpret_cast<float *>(base + ek::ImageBytes(w, M) + ek::ExpBytes(w, M));
  const dim3 sgrid(static_cast<unsigned>(rows / 16 * sh.units));
  const int m = static_cast<int>(M), k = static_cast<int>(w.K), rp = static_cast<int>(rows);
  if (ek::Terms(w) == 3)
    hipLaunchKernelGGL(ek::SplitRowsKernel<3>, sgrid, dim3(512), 0, s, A, img, exps, m, k, sh.units, rp);
  else
    hipLaunchKernelGGL(ek::SplitRowsKernel<2>, sgrid, dim3(512), 0, s, A, img, exps, m, k, sh.units, rp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // All runs in one workgroup: it applies the activation or adds the bias.
  float *Hk = sh.all_runs ? H : nullptr;
  const float *bk = sh.all_runs ? bias : nullptr;
  const int T = ek::Steps(w);
  if (ek::Terms(w) == 2)
    e = ek::LaunchSpb<2, 2>(w, M, img, exps, Y, P, Hk, bk, sh, T, rows, s);
  else if (ek::TileRows(w, M) == 16)
    e = ek::LaunchSpb<1, 3>(w, M, img, exps, Y, P, Hk, bk, sh, T, rows, s);
  else
    e = ek::LaunchSpb<2, 3>(w, M, img, exps, Y, P, Hk, bk, sh, T, rows, s);
  if (e != hipSuccess || sh.all_runs) return e;
  return LaunchSumPartials(Y, P, M * w.N, sh.runs - 1, H, s, bias, w.N);
}

} // namespace mnb
