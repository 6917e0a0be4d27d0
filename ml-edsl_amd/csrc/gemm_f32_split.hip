// fp32 dense layer / matmul on the bf16 matrix cores, at fp32 precision, any
// shape, row stride and alignment.
//
// C[M,N] = epilogue(A[M,K] x B[K,N] (+ bias[N])) -- the same op as the fp32
// tiles (reference cpp/src/builders/LinalgBuilder.cpp:106-139, 180-239,
// 301-339), for layers that fp32 MFMA bounds: its dense peak is 157 TFLOP/s,
// that of bf16 MFMA 2500.
//
// Every fp32 value is split exactly into three bf16 values, x = h + m + l (h
// the nearest bf16 of x, m that of x - h, l the rest: 8 + 8 + 8 significand
// bits), and the product takes six of the nine bf16 products, each exact in
// fp32: hh, hm, mh, mm, hl, lh. They are summed in fp32 by
// v_mfma_f32_32x32x16_bf16, hh in one accumulator and the small ones, smallest
// first, in another, so that a step rounds the large sum once. (With all six in
// one accumulator, six times: twice the fp32 chain's error on operands with a
// nonzero value or two per step, 9.4e-7 against 8.1e-7 on X >= 0.)
//
// The products left out, ml, lm and ll, are below 2^-24 of a product together.
// An fp32 chain of n terms is within n 2^-24 sum |ab| of the exact sum and this
// one within 2 2^-24 of it, so only an output of a single term can lose by the
// omission. A workgroup therefore counts the nonzero values of its rows and
// columns in its first 48 or 64 k and, unless the emptiest row and the emptiest
// column must meet at two k there (together two more nonzero values than there
// are k), takes eight products (all but ll, below 2^-33).
//
// Relative 2-norm error against float64, this kernel / the fp32 MFMA chain:
// N(0,1) data at K = 1024, 2048, 4096 1.9e-7 / 5.7e-7, 2.7e-7 / 8.1e-7, 4.0e-7
// / 1.1e-6, after ReLU at K = 4096 3.2e-7 / 8.1e-7; rows with n nonzero values,
// one per step, n = 1 2.5e-8 / 2.5e-8 (largest relative error 5.99e-8 / 5.96e-8),
// n = 2 2.6e-8 / 3.1e-8, n = 8 2.9e-8 / 5.4e-8, n = 32 4.4e-8 / 1.03e-7.
//
// Not every value splits exactly. Below 2^-109 the last remainder may leave
// bf16's range, which cuts at most 2^-134 off the value; near the largest float
// h overflows; and where sums are below 2^-126, rounding is no longer relative
// (2^-150 each; the matrix cores keep subnormal operands and results). A
// workgroup ORs the low halves of all its last remainders (zero exactly when
// they are bf16 values), keeps its largest value, and at the end tests its sums.
// One that is not finite, or is smaller than 2^26 times what may have been lost
// -- K 2^-150 from underflow, and with a value cut K 2^-133 times the largest
// value, unless its row or column is zero throughout -- sends the whole tile to
// v_mfma_f32_16x16x4_f32 and the fp32 operands, with that path's results for
// denormal, huge, infinite and NaN values. So denormals among ordinary values
// are nearly free (one in every row: 4096^3 662 -> 682 us, 2048^3 97 -> 102; 783
// and 105 with rows of zeros as well; sending every tile with a cut value to a
// loop without LDS took 2411 and 542), and a layer whose every tile holds an
// infinity, a NaN or a value near the largest float, or whose sums are all tiny,
// pays for both: 4096^3 1760 us, 2048^3 240, 10000x500x1000 190, twice the fp32
// tiles' time.
//
// Bounds and layout. Splitting costs six VALU operations an element, so it is
// done once per workgroup, on the way into LDS, never per wave: eight k of a
// row of A (two 16-byte loads at any 4-byte alignment) or of a column of B
// (eight 4-byte loads, 64 adjacent columns a wave) become one 16-byte piece of
// each plane, stored in the order the MFMA reads (fragments of 32 rows x 16 k,
// 1 KB, one 16-byte read per lane), rows XORed by the octet so that the eight
// lanes of an LDS cycle never share banks (without it writes ran at a quarter
// of the rate). The stages are double-buffered with one barrier per step; the
// barrier stands before a step's last slice of MFMAs, whose operands are in
// registers, so the next stage's first fragments are read behind those MFMAs.
// Each octet's registers are reloaded with the step after next as soon as it
// has been split, a full step ahead of its use (loading in one burst a slice
// ahead cost 180 of 820 us at 4096^3). The K % BK rows are the first step, the
// only masked one. Rows past M and columns past N read the last row or column;
// their outputs are not stored.
//
// What bounds it is power: the full chip runs this loop at 1.8-1.87 GHz, a
// register-only loop of the same MFMAs takes 491 us at 4096^3. The 256x128 tile
// of four waves, each 128x64, reads LDS least of the tiles whose two sets of
// accumulators fit the registers (a 256x256 tile with one took 580 us at the
// error above). Measured, us, against the fp32 tiles: 4096^3 650-691 / 905
// by box (199-211 TFLOP/s; 700 / 905 on eight products), 4000x1024x4000 178 / 245,
// 2500^3 184 / 277; 2048^3 on eight waves of 64x32 97 / 120, 2001^3 99 / 159;
// 10000x500x1000 on two workgroups of 128x128x16 per CU 75 / 94 (83 on eight
// waves), 3333^3 428 / 681. Counting the first steps and testing the sums cost
// 1 % or less.
#include "common.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace edsl {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// Four floats at any 4-byte aligned address.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kPlanes = 3;

__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  const bf16x2 p = __builtin_convertvector(f32x2{a, b}, bf16x2);
  return __builtin_bit_cast(uint32_t, p);
}
__device__ __forceinline__ float bf_lo(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float bf_hi(uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// Eight floats as three bf16 planes; ORs the bits of the last remainders into
// `lost` and keeps the largest magnitude of the first plane in `big`.
__device__ __forceinline__ void split8(const float (&x)[8], u32x4 (&p)[kPlanes], uint32_t& lost, float& big) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[2 * i], b = x[2 * i + 1];
    const uint32_t h = cvt_pk_bf16(a, b);
    const float ra = a - bf_lo(h), rb = b - bf_hi(h);
    const uint32_t m = cvt_pk_bf16(ra, rb);
    const float qa = ra - bf_lo(m), qb = rb - bf_hi(m);
    p[0][i] = h;
    p[1][i] = m;
    p[2][i] = cvt_pk_bf16(qa, qb);
    lost |= __builtin_bit_cast(uint32_t, qa) | __builtin_bit_cast(uint32_t, qb);
    const f32x2 hf = __builtin_convertvector(__builtin_bit_cast(bf16x2, h), f32x2);
    big = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(hf[0]), __builtin_fabsf(hf[1])), big);
  }
}

// BM x BN outputs per workgroup of WM x WN waves, BK-deep steps of K; WAVES on a
// SIMD, VALU operations scheduled behind an MFMA.
template <int BM_, int BN_, int WM_, int WN_, int BK_, int WAVES_, int VALU_>
struct SplitTile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, BK = BK_;
  static constexpr int kSimdWaves = WAVES_, kValu = VALU_;
  static constexpr int kWaves = WM * WN;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int RB = BM / WM / 32, CB = BN / WN / 32;  // 32x32 blocks of a wave
  static constexpr int KK = BK / 16;                          // MFMA steps of a stage
  static constexpr int OPR = BK / 8;                          // octets per row
  static constexpr int AO = BM * OPR / kThreads;              // octets a thread stages
  static constexpr int BO = BN * OPR / kThreads;
  static constexpr int kFrag = 1024;
  static constexpr int kABytes = BM / 32 * KK * kPlanes * kFrag;
  static constexpr int kBBytes = BN / 32 * KK * kPlanes * kFrag;
  static constexpr int kStage = kABytes + kBBytes;
  static constexpr int kLds = 2 * kStage;
  static_assert(BM * OPR % kThreads == 0 && BN * OPR % kThreads == 0, "octets per thread");
  static_assert(BN % 64 == 0 && BM % 32 == 0, "tile");
};

// The tile from the fp32 operands on v_mfma_f32_16x16x4_f32, for a workgroup
// whose values do not allow the split. `load` fetches a step's octets into
// registers; they are staged in LDS as [k][row] and [k][column], whose pitches
// put the four k of an MFMA operand on different banks.
template <class C, int EPI, class Load>
__device__ __forceinline__ void fp32_tile(const GemmF32Args& args, char* smem, int m0, int n0, int nit,
                                          float (&raw)[C::AO + C::BO][8], Load load) {
  constexpr int R = 2 * C::RB, CC = 2 * C::CB;  // 16x16 blocks of a wave
  constexpr int PA = C::BM + 16, PB = C::BN + 16;
  constexpr int kBuf = C::BK * (PA + PB);
  static_assert(2 * kBuf * 4 <= C::kLds, "two stages of fp32 operands");
  float* lds = reinterpret_cast<float*>(smem);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / C::WN * C::RB * 32, wn = wave % C::WN * C::CB * 32;
  const int g = lane >> 4, r16 = lane & 15;
  auto stage = [&](float* st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::AO; ++i) {
      const int idx = threadIdx.x + i * C::kThreads;
      float* p = st + 8 * (idx % C::OPR) * PA + idx / C::OPR;
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e * PA] = raw[i][e];
    }
#pragma unroll
    for (int i = 0; i < C::BO; ++i) {
      const int idx = wave + i * C::kWaves;
      float* p = st + C::BK * PA + 8 * (idx / (C::BN / 64)) * PB + idx % (C::BN / 64) * 64 + lane;
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e * PB] = raw[C::AO + i][e];
    }
  };
  f32x4 acc[R][CC] = {};
  load(0);
  stage(lds);
  load(1);
  __syncthreads();
#pragma unroll 1
  for (int it = 0; it < nit; ++it) {
    const float* st = lds + (it & 1) * kBuf;
    const float* sa = st + g * PA + wm + r16;
    const float* sb = st + C::BK * PA + g * PB + wn + r16;
#pragma unroll
    for (int k = 0; k < C::BK; k += 4) {
      float a[R], b[CC];
#pragma unroll
      for (int i = 0; i < R; ++i) a[i] = sa[k * PA + 16 * i];
#pragma unroll
      for (int c = 0; c < CC; ++c) b[c] = sb[k * PB + 16 * c];
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int c = 0; c < CC; ++c) acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[c], acc[i][c], 0, 0, 0);
    }
    stage(lds + ((it + 1) & 1) * kBuf);
    load(it + 2);
    __syncthreads();
  }
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    const int n = n0 + wn + 16 * c + r16;
    if (n >= args.N) continue;
    const float bv = epi_has_bias(EPI) ? args.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * g + e;
        if (m < args.M) args.C[(int64_t)m * args.ldc + n] = apply_epilogue_f32<EPI>(acc[i][c][e], bv, args.alpha);
      }
  }
}

template <class C, int EPI>
__global__ void __launch_bounds__(C::kThreads, C::kSimdWaves)
gemm_f32_split_kernel(GemmF32Args args) {
  constexpr int RB = C::RB, CB = C::CB, KK = C::KK;
  __shared__ __align__(16) char smem[C::kLds];
  __shared__ int counts[C::BM + C::BN];  // nonzero values of the tile's rows and columns in the first steps
  __shared__ int fewest[2];              // of a row, of a column
  __shared__ int biggest;
  if (threadIdx.x < 2) fewest[threadIdx.x] = 1 << 30;
  for (int i = threadIdx.x; i < C::BM + C::BN; i += C::kThreads) counts[i] = 0;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN;
  int tm, tn;
  tile_coords(blockIdx.x, args.tiles_m, args.tiles_n, tm, tn);
  const int m0 = tm * C::BM, n0 = tn * C::BN;
  const int M = args.M, N = args.N, K = args.K;

  // Sources of the octets this thread stages.
  const float* pa[C::AO];
  int la[C::AO];
#pragma unroll
  for (int i = 0; i < C::AO; ++i) {
    const int idx = threadIdx.x + i * C::kThreads;
    const int row = idx / C::OPR, o = idx % C::OPR;
    pa[i] = args.A + (int64_t)min(m0 + row, M - 1) * args.lda + 8 * o;
    la[i] = ((row / 32) * KK + o / 2) * kPlanes * C::kFrag + ((o % 2) * 32 + (row % 32 ^ o * (8 / C::OPR))) * 16;
  }
  int cb[C::BO], ob[C::BO], lb[C::BO];
#pragma unroll
  for (int i = 0; i < C::BO; ++i) {
    const int idx = wave + i * C::kWaves;
    const int c64 = idx % (C::BN / 64);
    ob[i] = idx / (C::BN / 64);
    const int col = c64 * 64 + lane;
    cb[i] = min(n0 + col, N - 1);
    lb[i] = C::kABytes + ((col / 32) * KK + ob[i] / 2) * kPlanes * C::kFrag +
            ((ob[i] % 2) * 32 + (col % 32 ^ ob[i] * (8 / C::OPR))) * 16;
  }

  constexpr int kOct = C::AO + C::BO;
  auto line_of = [&](int o) {  // the octet's row, or BM + column, within the tile
    return o < C::AO ? ((int)threadIdx.x + o * C::kThreads) / C::OPR
                     : C::BM + (wave + (o - C::AO) * C::kWaves) % (C::BN / 64) * 64 + lane;
  };
  float raw[kOct][8];
  auto load_octet = [&](float (&raw)[kOct][8], int o, int k0) __attribute__((always_inline)) {
    if (o < C::AO) {
      const float* p = pa[o] + k0;
      const f32x4u v0 = *reinterpret_cast<const f32x4u*>(p), v1 = *reinterpret_cast<const f32x4u*>(p + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        raw[o][e] = v0[e];
        raw[o][4 + e] = v1[e];
      }
    } else {
      const int i = o - C::AO;
      const float* p = args.B + (int64_t)(k0 + 8 * ob[i]) * args.ldb;
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[o][e] = (p + e * args.ldb)[cb[i]];
    }
  };
  auto load_tail = [&](int o, int k0) {
    const int ko = o < C::AO ? 8 * (((int)threadIdx.x + o * C::kThreads) % C::OPR) : 8 * ob[o < C::AO ? 0 : o - C::AO];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = k0 + ko + e, kc = min(k, K - 1);
      const float v = o < C::AO ? pa[o < C::AO ? o : 0][kc - ko] : (args.B + (int64_t)kc * args.ldb)[cb[o < C::AO ? 0 : o - C::AO]];
      raw[o][e] = k < K ? v : 0.0f;
    }
  };
  uint32_t lost = 0;
  float big = 0.0f;
  auto stage_octet = [&](char* st, int o) __attribute__((always_inline)) {
    u32x4 p[kPlanes];
    split8(raw[o], p, lost, big);
    const int at = o < C::AO ? la[o] : lb[o - C::AO];
#pragma unroll
    for (int q = 0; q < kPlanes; ++q) *reinterpret_cast<u32x4*>(st + at + q * C::kFrag) = p[q];
  };

  // Steps: the K % BK rows first, if any, then the full steps.
  const int full = K / C::BK;
  const int has_tail = K % C::BK != 0;
  const int nit = full + has_tail;
  auto k_of = [&](int it) { return (min(it, nit - 1) - has_tail) * C::BK; };  // full steps
  // The first kCheck full steps are loaded here for the count of their nonzero
  // values, behind the first step, which is staged meanwhile.
  constexpr int kCheck = C::BK == 16 ? 3 : 2;
  float first[kCheck][kOct][8];
  if (has_tail) {
#pragma unroll
    for (int o = 0; o < kOct; ++o) load_tail(o, full * C::BK);
  } else {
#pragma unroll
    for (int o = 0; o < kOct; ++o) load_octet(raw, o, 0);
  }
#pragma unroll
  for (int c = 0; c < kCheck; ++c)
#pragma unroll
    for (int o = 0; o < kOct; ++o) load_octet(first[c], o, min(c, full - 1) * C::BK);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int o = 0; o < kOct; ++o) stage_octet(smem, o);
  if (nit > 1) {
#pragma unroll
    for (int o = 0; o < kOct; ++o) load_octet(raw, o, k_of(1));
  }
  __syncthreads();  // counts are zero
#pragma unroll
  for (int o = 0; o < kOct; ++o) {
    int n = 0;
#pragma unroll
    for (int c = 0; c < kCheck; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) n += first[c][o][e] != 0.0f;
    atomicAdd(&counts[line_of(o)], n);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < C::BM + C::BN; i += C::kThreads) {  // whole waves, of rows or of columns
    int n = counts[i];
    n = min(n, __builtin_amdgcn_update_dpp(n, n, 0x121, 0xf, 0xf, false));  // of 16 lanes, by rotation
    n = min(n, __builtin_amdgcn_update_dpp(n, n, 0x122, 0xf, 0xf, false));
    n = min(n, __builtin_amdgcn_update_dpp(n, n, 0x124, 0xf, 0xf, false));
    n = min(n, __builtin_amdgcn_update_dpp(n, n, 0x128, 0xf, 0xf, false));
    if (lane % 16 == 0) atomicMin(&fewest[i >= C::BM], n);
  }
  __syncthreads();
  bool sparse = full < kCheck;  // its last step has been counted more than once
  sparse |= fewest[0] + fewest[1] < kCheck * C::BK + 2;
  // Uniform: take ml and lm. (A vote although all threads agree: with the flag read
  // back by readfirstlane the compiler spills registers in the loop of six
  // products, 10000x500x1000 86 us against 74.)
  const bool eight = __syncthreads_or(sparse) != 0;

  constexpr int BS = KK == 1 ? 2 : KK;  // sets of B fragments
  bf16x8 a[2][kPlanes], b[BS][CB][kPlanes];
  const int oa = wm * RB * KK * kPlanes * C::kFrag;
  const int ob_ = C::kABytes + wn * CB * KK * kPlanes * C::kFrag;
  int lofs[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
    lofs[kk] = ((lane & 32) + (lane % 32 ^ (2 * kk + (lane >> 5)) * (8 / C::OPR))) * 16;
  auto read_a = [&](const char* st, int slice, int set) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < kPlanes; ++q)
      a[set][q] = *reinterpret_cast<const bf16x8*>(st + oa + lofs[slice % KK] + (slice * kPlanes + q) * C::kFrag);
  };
  auto read_b = [&](const char* st, int kk, int set) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int q = 0; q < kPlanes; ++q)
        b[set][j][q] = *reinterpret_cast<const bf16x8*>(st + ob_ + lofs[kk] + ((j * KK + kk) * kPlanes + q) * C::kFrag);
  };
  constexpr int kSlices = RB * KK;
  static_assert(kSlices % 2 == 0, "A sets alternate by slice");
  read_a(smem, 0, 0);
  read_b(smem, 0, 0);
  // Leaves a zero in `counts` only for rows and columns that are zero throughout.
  auto count_zero_lines = [&] {
    for (int r = wave; r < C::BM; r += C::kWaves) {
      if (counts[r] != 0) continue;  // uniform
      const float* p = args.A + (int64_t)min(m0 + r, M - 1) * args.lda;
      uint32_t any = 0;
#pragma unroll 8
      for (int k = 4 * lane; k < K; k += 256) {
        const f32x4u v = *reinterpret_cast<const f32x4u*>(p + min(k, K - 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) any |= __builtin_bit_cast(uint32_t, v[e]);
      }
      if (any & 0x7fffffffu) counts[r] = 1;
    }
    for (int c = 0; c < C::BN; c += 64) {
      if (!__any(counts[C::BM + c + lane] == 0)) continue;  // uniform
      const float* p = args.B + min(n0 + c + lane, N - 1);
      uint32_t any = 0;
#pragma unroll 8
      for (int k = wave; k < K; k += C::kWaves) any |= __builtin_bit_cast(uint32_t, p[(int64_t)k * args.ldb]);
      if (any & 0x7fffffffu) counts[C::BM + c + lane] = 1;
    }
  };
  // The K loop on PRODUCTS (6 or 8) products and the stores; false, with nothing
  // stored, if the tile must be recomputed.
  auto compute = [&](auto products_c) __attribute__((always_inline)) {
    constexpr int PRODUCTS = decltype(products_c)::value;
    f32x16 acc[RB][CB] = {}, low[RB][CB] = {};
    auto step = [&](int it, auto set_c) __attribute__((always_inline)) {
      constexpr int S = decltype(set_c)::value;  // parity of the step
      const char* st = smem + S * C::kStage;
      char* sn = smem + (S ^ 1) * C::kStage;
      const int k2 = k_of(it + 2);
#pragma unroll
      for (int sl = 0; sl < kSlices; ++sl) {
        const int i = sl / KK, kk = sl % KK;
        const int bs = KK == 1 ? S : kk;
        if (sl == kSlices - 1) {
          __syncthreads();
          read_a(sn, 0, (sl + 1) & 1);
          read_b(sn, 0, KK == 1 ? S ^ 1 : 0);
        } else {
          read_a(st, sl + 1, (sl + 1) & 1);
          if (i == 0 && kk + 1 < KK) read_b(st, kk + 1, kk + 1);
        }
        // Smallest products first.
        constexpr int pa_[8] = {1, 2, 2, 0, 1, 1, 0, 0}, pb_[8] = {2, 1, 0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int s = 8 - PRODUCTS; s < 8; ++s)
#pragma unroll
          for (int j = 0; j < CB; ++j) {
            f32x16& t = s < 7 ? low[i][j] : acc[i][j];
            t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[sl & 1][pa_[s]], b[bs][j][pb_[s]], t, 0, 0, 0);
          }
        if (sl < kSlices - 1) {
          // Octets sl, sl + (kSlices - 1), ... of the next stage; each one's
          // registers are then free for the octet of the step after.
#pragma unroll
          for (int o = sl; o < kOct; o += kSlices - 1) {
            stage_octet(sn, o);
            load_octet(raw, o, k2);
          }
        }
        // One MFMA, at most one LDS read, some VALU operations, and so on: the
        // compiler otherwise puts the splitting after the MFMAs.
        constexpr int kReads[2] = {3, 3 + 3 * CB};
        const int reads = kReads[sl == kSlices - 1 || (i == 0 && kk + 1 < KK)];
#pragma unroll
        for (int m = 0; m < PRODUCTS * CB; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (m < reads) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, C::kValu, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int it = 0;
    for (; it + 1 < nit; it += 2) {
      step(it, std::integral_constant<int, 0>{});
      step(it + 1, std::integral_constant<int, 1>{});
    }
    if (it < nit) step(it, std::integral_constant<int, 0>{});

#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) acc[i][j] += low[i][j];
    // `zero` turns NaN if a sum is not finite.
    float zero = 0.0f, least = __builtin_huge_valf();
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          zero = __builtin_fmaf(acc[i][j][e], 0.0f, zero);
          least = __builtin_fminf(least, __builtin_fabsf(acc[i][j][e]));
        }
    const float underflow = 0x1p-124f * (float)K;
    const bool cut = (lost & 0xffffu) != 0;
    if (__syncthreads_or(zero != 0.0f || least < underflow || cut)) {  // uniform
      if (threadIdx.x == 0) biggest = 0;
      __syncthreads();
      atomicMax(&biggest, __builtin_bit_cast(int, big));
      const bool any_cut = __syncthreads_or(cut);
      float limit = underflow;
      if (any_cut) {
        limit = fmaxf(limit, 0x1.02p-105f * (float)K * __builtin_bit_cast(float, biggest));
        count_zero_lines();
        __syncthreads();
      }
      bool bad = zero != 0.0f;
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const bool col = any_cut & (counts[C::BM + (wn * CB + j) * 32 + (lane & 31)] != 0);
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int row = counts[(wm * RB + i) * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3)];
            const float v = __builtin_fabsf(acc[i][j][e]);
            bad |= (v < limit) & ((v != 0.0f) | (col & (row != 0)));
          }
      }
      if (__syncthreads_or(bad)) return false;
    }
    // Lane: rows 8 (r/4) + 4 (lane/32) + r%4 and column lane%32 of a block, so
    // each store writes two 128-byte row segments. The stores go through a
    // descriptor of C's rows m0 .. M-1, whose range check drops rows past M;
    // columns past N are sent out of range. (A branch per store cost an edge
    // tile 20 us; ldc is below 2^21, so a tile's offsets fit 31 bits.)
    const int half = lane >> 5, l32 = lane & 31;
    const int ldc = (int)args.ldc;
    const i32x4 rsrc = buffer_rsrc(args.C + (int64_t)m0 * ldc, (int64_t)(M - m0) * ldc * 4);
    const int col0 = n0 + wn * CB * 32 + l32;
    float bv[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j) bv[j] = epi_has_bias(EPI) && col0 + 32 * j < N ? args.bias[col0 + 32 * j] : 0.0f;
    auto store = [&](auto aux) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const int at = (((wm * RB + i) * 32 + 4 * half) * ldc + col0) * 4;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int dr = 8 * (r >> 2) + (r & 3);
#pragma unroll
          for (int j = 0; j < CB; ++j)
            raw_buffer_store_f32(apply_epilogue_f32<EPI>(acc[i][j][r], bv[j], args.alpha), rsrc,
                                 col0 + 32 * j < N ? at + dr * ldc * 4 + 128 * j : 0x7fffffff, 0, decltype(aux)::value);
          if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    // Rows of C on 128-byte lines are streamed; lines that two segments share stay
    // in the caches until both are there (3310x288x2369 40.4 -> 35.7 us).
    if (ldc % 32 == 0 && reinterpret_cast<uintptr_t>(args.C) % 128 == 0)
      store(std::integral_constant<int, kAuxNonTemporal>{});
    else
      store(std::integral_constant<int, 0>{});
    return true;
  };
  const bool done = eight ? compute(std::integral_constant<int, 8>{}) : compute(std::integral_constant<int, 6>{});
  if (done) return;
  fp32_tile<C, EPI>(args, smem, m0, n0, nit, raw, [&](int it) __attribute__((always_inline)) {
    if (it == 0 && has_tail) {
#pragma unroll
      for (int o = 0; o < kOct; ++o) load_tail(o, full * C::BK);
    } else {
#pragma unroll
      for (int o = 0; o < kOct; ++o) load_octet(raw, o, k_of(it));
    }
  });
}

template <class C>
hipError_t launch_tile(int epi, GemmF32Args a, hipStream_t stream) {
  a.tiles_m = (a.M + C::BM - 1) / C::BM;
  a.tiles_n = (a.N + C::BN - 1) / C::BN;
  const dim3 grid(a.tiles_m * a.tiles_n), block(C::kThreads);
#define EDSL_SPLIT_CASE(E) \
  case E: hipLaunchKernelGGL((gemm_f32_split_kernel<C, E>), grid, block, 0, stream, a); break;
  switch (epi) {
    EDSL_SPLIT_CASE(epi_code(false, ACT_NONE))
    EDSL_SPLIT_CASE(epi_code(true, ACT_NONE))
    EDSL_SPLIT_CASE(epi_code(false, ACT_RELU))
    EDSL_SPLIT_CASE(epi_code(true, ACT_RELU))
    EDSL_SPLIT_CASE(epi_code(false, ACT_LEAKY))
    EDSL_SPLIT_CASE(epi_code(true, ACT_LEAKY))
    EDSL_SPLIT_CASE(epi_code(false, ACT_IF_RELU))
    EDSL_SPLIT_CASE(epi_code(true, ACT_IF_RELU))
    default: return hipErrorInvalidValue;
  }
#undef EDSL_SPLIT_CASE
  return hipGetLastError();
}

}  // namespace

hipError_t launch_gemm_f32_split(int tile, int epi, GemmF32Args a, hipStream_t stream) {
  if (a.M < 1 || a.N < 1 || a.K < 32 || a.ldc >= kF32SplitMaxLdc) return hipErrorInvalidValue;  // a full step of K
  switch (tile) {
    case kSplit256x128: return launch_tile<SplitTile<256, 128, 2, 2, 16, 1, 5>>(epi, a, stream);
    case kSplit128W8: return launch_tile<SplitTile<128, 128, 2, 4, 32, 2, 8>>(epi, a, stream);
    case kSplit128Pair: return launch_tile<SplitTile<128, 128, 2, 2, 16, 2, 8>>(epi, a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace edsl
