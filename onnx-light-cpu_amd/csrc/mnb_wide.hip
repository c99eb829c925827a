// Wide-tile prefill GEMM for MatMulNBits on CDNA4 fp16 MFMA (WideKernel).
//
// PrefillKernel's product (the same fp16 operands, dequantized by DequantWord
// from the fragment-ordered weights) on 256 x 256 output tiles: a wavefront
// multiplies 256 rows x 64 columns, so each dequantized weight fragment feeds
// 16 MFMAs instead of 8. PrefillKernel's k-loop issues 2.4 VALU instructions
// per MFMA, which with the MFMAs' own issue fills 85% of a SIMD's cycles; here
// it is 1.1 (132 -> 111 us at M = 512, K = 4096, N = 28672, one wave of
// tiles; 1.24 PFLOP/s at M = 8192 against 1.09). What bounds it is the MFMAs
// at the clock that their power leaves (65% of the cycles), and per tile the
// prologue and the 256 KiB of stores, which one workgroup per CU does not
// overlap: a 32x32x16 form of the k-loop took as many cycles, and within 3%
// as many without its LDS activation reads, half its copies or the
// dequantization.
//
// A workgroup is four wavefronts, one per SIMD, of 256 fp32 accumulators per
// lane; wavefront cg takes column group cg. With one wavefront per SIMD
// nothing else fills a stall, so the k-loop is laid out by hand, one MFMA per
// slot with the other work of the next step between them (sched_barrier pins
// the slots):
// - an activation fragment is read from LDS in place right behind its last
//   MFMA, 60 slots before its next use;
// - the next step's weight words are dequantized one or two VALU per slot;
// - the barrier that makes the next tile visible sits a quarter into the
//   step, when every LDS read before it has long returned (no wait), and the
//   direct global -> LDS copies of the tile kNS ahead follow one at a time.
#include "mnb_gemm_common.h"

#include <utility>

namespace mnb {
namespace wide {

using namespace gemm;

constexpr int kThreads = 256;
constexpr int kRec = 64;  // 16-byte units per 1 KiB record

constexpr int kMI = kWideRows / 16;  // 16-row blocks per wavefront
constexpr int kCG = kWideCols / 64;  // column groups, one wavefront each
// Copies per wavefront and 64-k tile: activations (two records per 16 rows),
// weights (two per column group), scales (one per two groups).
constexpr int kACopies = kMI / 2, kBCopies = kCG / 2;
constexpr int kOps = kACopies + kBCopies + 1;
constexpr int kARecs = 2 * kMI, kBRecs = 2 * kCG, kSRecs = kCG / 2;
constexpr int kStage = (kARecs + kBRecs + kSRecs) * kRec;
constexpr int kNS = 3;  // stages: 126 KiB of LDS
constexpr size_t kLds = size_t{16} * kStage * kNS;

// s_waitcnt vmcnt(N) lgkmcnt(0) and a workgroup barrier, nothing moved across.
template <int N>
__device__ __forceinline__ void WaitBarrier() {
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  __asm__ volatile("" ::: "memory");
}

template <bool HAS_ZP, bool BS32>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void WideKernel(
    const uint4 *__restrict__ Ah, const uint8_t *__restrict__ Bp, const uint8_t *__restrict__ Sp,
    float *__restrict__ Y, int M, int N, int K, int nb, int log2_bs,
    float *__restrict__ H, const int *__restrict__ row_exp, const int *__restrict__ col_exp,
    const float *__restrict__ bias) {
  extern __shared__ uint4 lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int c = lane & 15, qd = lane >> 4;

  // Workgroup -> tile: an XCD (blockIdx % 8) takes a contiguous run of
  // an order that walks groups of 4 row tiles column tile by column tile.
  const int tiles_m = (M + 16 * kMI - 1) / (16 * kMI);
  const int tiles_n = (N + 64 * kCG - 1) / (64 * kCG);
  const int tiles = tiles_m * tiles_n;
  int tm, tn;
  {
    int L = static_cast<int>(blockIdx.x);
    if (tiles % 8 == 0) L = (L & 7) * (tiles / 8) + (L >> 3);
    constexpr int kGM = 4;
    const int group = L / (kGM * tiles_n);
    const int gm = min(kGM, tiles_m - group * kGM);
    const int rem = L - group * kGM * tiles_n;
    tm = group * kGM + rem % gm;
    tn = rem / gm;
  }
  const int T = K / 32, ktiles = K / kBK, klast = ktiles - 1;

  // Copy sources: record 4 i + wave of each kind. 16-row blocks past the last
  // repeat it (their rows are not stored).
  const uint32_t l16 = static_cast<uint32_t>(lane) * 16;
  const int mt_last = (M - 1) / 16;
  const uint4 *a_src[kACopies];
#pragma unroll
  for (int i = 0; i < kACopies; ++i)
    a_src[i] = Ah + static_cast<size_t>(min(tm * kMI + 2 * i + (wave >> 1), mt_last)) * ktiles *
                    (2 * kRec) + (wave & 1) * kRec;
  const uint8_t *b_src[kBCopies];
#pragma unroll
  for (int i = 0; i < kBCopies; ++i) {
    const int p = 4 * i + wave;
    b_src[i] = Bp + (static_cast<size_t>(tn * kCG + (p >> 1)) * T + (p & 1)) * 1024;
  }
  // Scales: lanes 0-31 the record pair's first group, 32-63 its second; lane
  // bit 4 the step (32-wide blocks: one record per step, else the tile's).
  const int s_pair = wave % kSRecs;
  const uint8_t *s_src = Sp + static_cast<size_t>(tn * kCG + 2 * s_pair) * nb * 256;
  const uint32_t s_off = static_cast<uint32_t>((lane >> 5) * nb * 256 + 16 * c +
                                               (BS32 ? ((lane >> 4) & 1) * 256 : 0));
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  // Copy n (0 .. kOps - 1) of tile kt into the stage at byte st.
  auto copy = [&](auto nc, int kt, uint32_t st) __attribute__((always_inline)) {
    constexpr int n = decltype(nc)::value;
    if constexpr (n < kACopies) {
      CopyToLds16S(a_src[n] + static_cast<size_t>(kt) * (2 * kRec), l16,
                   lds0 + st + static_cast<uint32_t>((4 * n + wave) * kRec * 16));
    } else if constexpr (n < kACopies + kBCopies) {
      constexpr int i = n - kACopies;
      CopyToLds16S(b_src[i] + static_cast<size_t>(kt) * 2048, l16,
                   lds0 + st + static_cast<uint32_t>((kARecs + 4 * i + wave) * kRec * 16));
    } else {
      const int rec = BS32 ? 2 * kt : kt >> (log2_bs - 6);
      CopyToLds16S(s_src + static_cast<size_t>(rec) * 256, s_off,
                   lds0 + st + static_cast<uint32_t>((kARecs + kBRecs + s_pair) * kRec * 16));
    }
  };
  auto issue = [&](int kt, uint32_t st) __attribute__((always_inline)) {
    [&]<int... n>(std::integer_sequence<int, n...>) __attribute__((always_inline)) {
      (copy(std::integral_constant<int, n>{}, kt, st), ...);
    }(std::make_integer_sequence<int, kOps>{});
  };

  const Masks dq = MakeMasks();
  floatx4 acc[kMI][4];
#pragma unroll
  for (int i = 0; i < kMI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // LDS reads of step h of the stage at unit offset su.
  const int a_lane0 = Swz(c, qd), a_lane1 = Swz(c, 4 + qd);
  auto readA = [&](int su, int h, int i) __attribute__((always_inline)) {
    return __builtin_bit_cast(half8, lds[su + i * 2 * kRec + (h == 0 ? a_lane0 : a_lane1)]);
  };
  auto readB = [&](int su, int h) { return lds[su + (kARecs + 2 * wave + h) * kRec + lane]; };
  auto readS = [&](int su, int h) {
    return lds[su + (kARecs + kBRecs + (wave >> 1)) * kRec + 32 * (wave & 1) + 16 * h + c];
  };

  half8 a[kMI];
  uint32_t q0[4][4], q1[4][4];  // dequantized fragments (halves pairs), two sets
  uint4 bw, sw;
  // Dequantization op o (0 .. 63) of word j = o / 16, as DequantWord.
  DequantRow dr;
  uint32_t w8, t16;
  auto dequant_op = [&](auto oc, uint32_t (&q)[4][4]) __attribute__((always_inline)) {
    constexpr int j = decltype(oc)::value / 16, o = decltype(oc)::value % 16;
    const uint32_t w = j == 0 ? bw.x : j == 1 ? bw.y : j == 2 ? bw.z : bw.w;
    const uint32_t sz = j == 0 ? sw.x : j == 1 ? sw.y : j == 2 ? sw.z : sw.w;
    if constexpr (o == 0) dr = RowFromSz<HAS_ZP>(sz);
    else if constexpr (o == 3) w8 = w >> 8;
    else if constexpr (o >= 4) {
      constexpr int v = (o - 4) / 3, step = (o - 4) % 3;
      if constexpr (step == 0)
        t16 = ((v < 2 ? w : w8) & (v % 2 == 0 ? dq.lo : dq.hi)) | (v % 2 == 0 ? dq.e1024 : dq.e64);
      else if constexpr (step == 1)
        t16 = PkAddF16(t16, v % 2 == 0 ? dr.neg_lo : dr.neg_hi);
      else
        q[j][v] = PkMulF16(t16, dr.s);
    }
  };

  // Groups G0 .. G1 - 1 (row blocks, four MFMAs each) of one step: multiplies
  // by qc the fragments in a. From group G0 on it reads step rh of the stage at
  // unit offset su_next into a in place and dequantizes its weights into qn
  // (READ). BAR: groups kB.. of a step whose first kB ran before the barrier:
  // their fragments catch up two per group, and tile t_copy is copied into
  // the stage at byte st_copy, whose tile's last fragments are in a.
  constexpr int kB = kMI / 4;
  auto groups = [&](auto g0_c, auto g1_c, auto read_c, auto bar_c, auto rh_c, uint32_t (&qc)[4][4],
                    uint32_t (&qn)[4][4], int su_next, int t_copy, uint32_t st_copy)
                    __attribute__((always_inline)) {
    constexpr int G0 = decltype(g0_c)::value, G1 = decltype(g1_c)::value;
    constexpr bool READ = decltype(read_c)::value, BAR = decltype(bar_c)::value;
    constexpr int rh = decltype(rh_c)::value;
    constexpr int kS0 = 4 * G0, kS1 = 4 * G1;
    constexpr int kD = kS0 + 12;  // first slot of the dequantization: the words have arrived
    constexpr int kStride = (kS1 - kS0 - 2) / kOps;
    static_assert(!BAR || kStride >= 1, "copies");
    auto slot = [&](auto kc) __attribute__((always_inline)) {
      constexpr int k = kS0 + decltype(kc)::value, i = k / 4, j = k % 4;
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
          __builtin_bit_cast(half8, make_uint4(qc[j][0], qc[j][1], qc[j][2], qc[j][3])), a[i],
          acc[i][j], 0, 0, 0);
      if constexpr (READ) {
        if constexpr (k == kS0) {
          bw = readB(su_next, rh);
          sw = readS(su_next, rh);
        }
        if constexpr (BAR && i < 2 * kB) {
          if constexpr (j == 1) a[2 * (i - kB)] = readA(su_next, rh, 2 * (i - kB));
          if constexpr (j == 3) a[2 * (i - kB) + 1] = readA(su_next, rh, 2 * (i - kB) + 1);
        } else if constexpr (j == 3) {
          a[i] = readA(su_next, rh, i);
        }
        if constexpr (k >= kD) {
          constexpr int o0 = (k - kD) * 64 / (kS1 - kD), o1 = (k + 1 - kD) * 64 / (kS1 - kD);
          [&]<int... o>(std::integer_sequence<int, o...>) __attribute__((always_inline)) {
            (dequant_op(std::integral_constant<int, o0 + o>{}, qn), ...);
          }(std::make_integer_sequence<int, o1 - o0>{});
        }
        if constexpr (BAR && k >= kS0 + 2 && (k - kS0 - 2) % kStride == 0 &&
                      (k - kS0 - 2) / kStride < kOps)
          copy(std::integral_constant<int, (k - kS0 - 2) / kStride>{}, t_copy, st_copy);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    [&]<int... k>(std::integer_sequence<int, k...>) __attribute__((always_inline)) {
      (slot(std::integral_constant<int, k>{}), ...);
    }(std::make_integer_sequence<int, kS1 - kS0>{});
  };

  constexpr uint32_t kStageBytes = kStage * 16;
#pragma unroll
  for (int p = 0; p < kNS; ++p) issue(min(p, klast), p * kStageBytes);
  WaitBarrier<kOps * (kNS - 1)>();
#pragma unroll
  for (int i = 0; i < kMI; ++i) a[i] = readA(0, 0, i);
  bw = readB(0, 0);
  sw = readS(0, 0);
  [&]<int... o>(std::integer_sequence<int, o...>) __attribute__((always_inline)) {
    (dequant_op(std::integral_constant<int, o>{}, q0), ...);
  }(std::make_integer_sequence<int, 64>{});

  // Stage of tile t: t % kNS. At the barrier of tile t's last step tile t's
  // fragments are all in registers, so its stage takes tile t + kNS. The loop
  // turns at that barrier, where no LDS read is outstanding: with a read in
  // flight across the back edge the compiler waits there for all of them.
  int st = 0;
  auto next = [&](int s) { return s + 1 == kNS ? 0 : s + 1; };
  using std::false_type;
  using std::true_type;
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using IB = std::integral_constant<int, kB>;
  using IM = std::integral_constant<int, kMI>;
  auto before = [&](uint32_t (&qc)[4][4]) __attribute__((always_inline)) {
    groups(I0{}, IB{}, false_type{}, false_type{}, I0{}, qc, qc, 0, 0, 0);
    WaitBarrier<kOps * (kNS - 2)>();
  };
  auto after = [&](int t, uint32_t (&qc)[4][4], uint32_t (&qn)[4][4]) __attribute__((always_inline)) {
    const int nx = next(st);
    groups(IB{}, IM{}, true_type{}, true_type{}, I0{}, qc, qn, nx * kStage, min(t + kNS, klast),
           st * kStageBytes);
    st = nx;
  };
  auto first = [&]() __attribute__((always_inline)) {  // step 0 of a tile, reading its step 1
    groups(I0{}, IM{}, true_type{}, false_type{}, I1{}, q0, q1, st * kStage, 0, 0);
  };
  first();
  before(q1);
  for (int t = 0; t < klast; ++t) {
    after(t, q1, q0);
    first();
    before(q1);
  }
  after(klast, q1, q0);

  // The exponents and the bias, all loaded here: between the stores each load
  // waited out the stores before it, a memory round trip per fragment (an
  // eighth of the kernel at M = 512, K = 4096, N = 28672: 131 against 115 us).
  const int m0 = tm * 16 * kMI;
  const int n_first = (tn * kCG + wave) * 64 + 4 * qd;
  int er[kMI];
  int4 ec[4];
  float4 bv[4];
#pragma unroll
  for (int i = 0; i < kMI; ++i) er[i] = row_exp[min(m0 + 16 * i + c, M - 1)];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int nc = min(n_first + 16 * j, N - 4);
    ec[j] = *reinterpret_cast<const int4 *>(col_exp + nc);
    bv[j] = bias != nullptr
                ? make_float4(bias[nc], bias[nc + 1], bias[nc + 2], bias[nc + 3])
                : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // No copy into this workgroup's LDS may land after it exits.
  WaitBarrier<0>();

  const int rows = min(M - m0, 16 * kMI);
  const int width = H != nullptr ? N >> 1 : N;
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(
      (H != nullptr ? H : Y) + static_cast<size_t>(m0) * width, 0, rows * width * 4, 0x00020000);
  // Fragment i: lane l holds row m0 + 16 i + c and, for slice j, columns
  // n_first + 16 j + v, in units of 2^(f_m + e_n).
#pragma unroll
  for (int i = 0; i < kMI; ++i) {
    const int row = 16 * i + c;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n_first + 16 * j;
      const float x0 = __builtin_amdgcn_ldexpf(acc[i][j][0], -(er[i] + ec[j].x));
      const float x1 = __builtin_amdgcn_ldexpf(acc[i][j][1], -(er[i] + ec[j].y));
      const float x2 = __builtin_amdgcn_ldexpf(acc[i][j][2], -(er[i] + ec[j].z));
      const float x3 = __builtin_amdgcn_ldexpf(acc[i][j][3], -(er[i] + ec[j].w));
      const bool ok = row < rows && n < N;
      if (H != nullptr) {
        typedef unsigned int u32x2 __attribute__((vector_size(8)));
        const u32x2 hv = {__float_as_uint(SiluMul(x0, x1)), __float_as_uint(SiluMul(x2, x3))};
        __builtin_amdgcn_raw_buffer_store_b64(hv, ry, ok ? (row * width + (n >> 1)) * 4 : 0x7FFFFFF0,
                                              0, 0);
      } else {
        typedef unsigned int u32x4 __attribute__((vector_size(16)));
        const u32x4 v = {__float_as_uint(x0 + bv[j].x), __float_as_uint(x1 + bv[j].y),
                         __float_as_uint(x2 + bv[j].z), __float_as_uint(x3 + bv[j].w)};
        // Cached: a lane's 16 bytes are an eighth of a line, and the line's
        // other stores come four slices later (as streaming stores, M = 8192,
        // K = 4096, N = 28672: 1552 -> 1580 us; M = 512, K = 2048: 62.4 -> 66.6).
        __builtin_amdgcn_raw_buffer_store_b128(v, ry, ok ? (row * N + n) * 4 : 0x7FFFFFF0, 0, 0);
      }
    }
  }
}

template <bool HAS_ZP, bool BS32>
hipError_t LaunchT(const WeightView &w, int64_t M, const uint4 *Ah, float *Y, float *H,
                   const int *row_exp, const float *bias, hipStream_t s) {
  const int64_t tiles = (M + kWideRows - 1) / kWideRows * ((w.N + kWideCols - 1) / kWideCols);
  hipLaunchKernelGGL((WideKernel<HAS_ZP, BS32>), dim3(static_cast<unsigned>(tiles)),
                     dim3(kThreads), kLds, s, Ah, w.Bp, w.Sp, Y, static_cast<int>(M),
                     static_cast<int>(w.N), static_cast<int>(w.K), static_cast<int>(w.nb), w.log2_bs,
                     H, row_exp, w.col_exp, bias);
  return hipGetLastError();
}

} // namespace wide

hipError_t LaunchWide(const WeightView &w, int64_t M, const uint4 *Ah, float *Y, float *H,
                      const int *row_exp, const float *bias, hipStream_t s) {
  const bool bs32 = w.block_size == 32;
  if (w.has_zp)
    return bs32 ? wide::LaunchT<true, true>(w, M, Ah, Y, H, row_exp, bias, s)
                : wide::LaunchT<true, false>(w, M, Ah, Y, H, row_exp, bias, s);
  return bs32 ? wide::LaunchT<false, true>(w, M, Ah, Y, H, row_exp, bias, s)
              : wide::LaunchT<false, false>(w, M, Ah, Y, H, row_exp, bias, s);
}

} // namespace mnb
