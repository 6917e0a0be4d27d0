// fp32 dense layer for small M (M <= 64): a weight-streaming kernel.
//
// Y[M,N] = epilogue(X[M,K] x W[K,N] (+ bias[N])) -- the same op as the tiled
// kernel (reference cpp/src/builders/LinalgBuilder.cpp:106-139, 180-239,
// 301-339), shaped for the HBM-bound case where W dominates the traffic
// (M=16, K=N=8192: W is 256 MiB, X and Y 512 KiB each).
//
// Every W element is read from HBM exactly once and used for all M rows at
// once on the matrix cores:
//  * v_mfma_f32_16x16x4_f32: lane l supplies X[row l%16][k-slot l/16] and
//    W[k-slot l/16][col l%16]. Lane group g = l/16 owns the k rows
//    k0+4g .. k0+4g+3 of each 16-row step: it loads those 4 k of its X row
//    with one 16-byte load and, for each k, CPL consecutive W columns with one
//    4*CPL-byte load. MFMA (step s, column phase c) pairs X[.][k0+4g+s] with
//    W[k0+4g+s][n0 + CPL*(l%16) + c], so lane l%16 accumulates columns
//    n0 + CPL*(l%16) + c: a wave owns 16*CPL columns and stores CPL per row.
//  * A workgroup is NW waves (4 for one row block, 8 for more) covering
//    `cols` adjacent columns: WN waves side by side (cols = 16*CPL*WN), and
//    WK = NW/WN waves splitting the workgroup's K range. The WK slices are
//    summed in LDS, in wave order. Fewer waves per CU keep fewer HBM rows
//    open at once: 16-wave workgroups were 2-3 % slower at M=16, K=N=8192,
//    6-10 % at M=48-64.
//  * Wider column blocks read longer row runs but give fewer workgroups;
//    they split K over `ksplit` workgroups to fill the chip. Each writes its
//    partial tile, and a second small kernel sums the partials in split order
//    and applies bias and activation. (A "last workgroup to arrive reduces"
//    variant, with the partials exchanged through agent-scope atomics, was
//    measured: it costs as much as the extra launch, so it is not used.)
//  * Each K slice starts its walk at a hashed offset (wrapping), so the rows
//    in flight at any moment are spread over the matrix and over the HBM
//    channels instead of every wave hitting the same few rows. Waves side by
//    side share the offset, so a workgroup reads WN*16*CPL*4 contiguous bytes
//    of a row at a time (a per-wave offset was ~2 % slower at M=16).
//  * W registers are reloaded one at a time right after the MFMAs that read
//    them, so a wave's loads stay in flight while it computes.
//    A wave that drained its loads before every batch of MFMAs streamed
//    ~1.5 us slower at M=16, K=N=8192 (~42.7 vs ~41.2 us for the main kernel).
// The summation order is fixed by the shape and the configuration, so
// results are deterministic.
#include "common.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace edsl {
namespace {

// Vectors of floats at any 4-byte aligned address (the vector loads and stores
// of gfx950 need no more than that).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

// Waves per workgroup for MB row blocks of 16 and WN waves side by side.
constexpr int waves_per_wg(int mb, int wn) { return (mb == 1 ? 4 : 8) > wn ? (mb == 1 ? 4 : 8) : wn; }
constexpr int kMaxSplit = 16;
constexpr int kMaxTail = 16;  // rows of the K tail (GemvF32Args::k_end - K)

// WM (GemvF32Args::w_mode): kWVector and kWShared (N >= 4) -- a lane's CPL
// columns are one vector load per row, whatever the alignment of W and its row
// stride; a lane whose columns reach past N loads the last CPL columns instead
// and stores only its own of them. kWScalar (N < 4): a 4-byte load per column,
// columns past N reading column N - 1. X rows are read with one 16-byte load
// per row block and step, at any alignment too.
// kWVector is for W rows that start on 128-byte lines: every line belongs to
// one workgroup and is streamed past the caches (16x8192x8192 44.5 us against
// 50.6 us with plain loads). Otherwise a row's line at a block edge is also
// read by the neighbouring block: plain loads, and neighbours on one XCD and
// its L2 (16x4096x4097 21.4 us against 25.2 us streamed in launch order, and
// 30.2 us for the aligned chunks realigned in registers that this replaced).
template <int MB, int CPL, int WN, int WM, int NS>
__global__ void __launch_bounds__(waves_per_wg(MB, WN) * 64)
gemv_f32_kernel(GemvF32Args a, int epi) {
  using vec = typename std::conditional<CPL == 4, f32x4u, f32x2u>::type;
  constexpr int NW = waves_per_wg(MB, WN);
  static_assert(NW % WN == 0, "waves side by side must divide the workgroup");
  constexpr int WK = NW / WN;
  constexpr int kWaveCols = 16 * CPL;
  constexpr int kGroupCols = kWaveCols * WN;
  // 16-row steps per loop iteration: 8 W loads in flight per lane for one row
  // block, 4 for more. Two row blocks measured faster with one step than with
  // two (M = 32: 21.4 vs 23.5 us at K = N = 4096, 56.5 vs 59.9 us at 8192), and
  // three or four need the registers for their accumulators. Four steps (16
  // loads per lane) with one row block measured no faster, also where each
  // wave's K slice is short (the c4 column shard: 11.3-11.5 against 11.0-11.2 us).
  constexpr int kU = MB == 1 ? 2 : 1;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wn = wave % WN;
  const int wk = wave / WN;
  const int groups = (a.N + kGroupCols - 1) / kGroupCols;  // the last may be partial
  int wg = blockIdx.x;
  if constexpr (WM == kWShared) {
    // Workgroup w runs on XCD w % 8: give each XCD a run of neighbouring
    // column blocks (the first total % 8 XCDs have one more).
    const int total = groups * a.ksplit, x = wg % 8;
    wg = x * (total / 8) + min(x, total % 8) + wg / 8;
  }
  const int g = wg % groups;
  const int split = wg / groups;
  const int n0 = g * kGroupCols + kWaveCols * wn;
  // K, in 16-row chunks, is spread as evenly as possible over the ksplit x WK
  // slices: slice i = split * WK + wk takes chunks [i*C/S, (i+1)*C/S). When S
  // divides C every slice has the same length.
  const int chunks = a.K / 16;
  const int nslices = a.ksplit * WK;
  const int slice = split * WK + wk;
  const int kbeg = 16 * (int)((int64_t)slice * chunks / nslices);
  const int kwave = 16 * (int)((int64_t)(slice + 1) * chunks / nslices) - kbeg;  // multiple of 16
  const int li = lane & 15;
  const int lg = lane >> 4;

  // NS = 2: steps alternate between two sets of accumulators, summed at the
  // end: half the chain, 1/sqrt(2) of its rounding (relative 2-norm error
  // against float64 at 16x4096x4096 2.1e-7 -> 1.5e-7, 16x8192x8192 4.1e-7 ->
  // 2.9e-7). Three and four row blocks pay 3-4 % for it (64x8192x8192 93.5 ->
  // 96.4 us) and take it where the plan splits K into fewer slices
  // (GemvF32Args::two_sets).
  f32x4 sum[NS][MB][CPL] = {};

  const int64_t ldw = a.ldw;
  const int col_lane = n0 + CPL * li;
  const int col_w = WM != kWScalar ? min(col_lane, a.N - CPL) : 0;
  const float* wbase = a.W + (int64_t)(kbeg + 4 * lg) * ldw + col_w;
  int cofs[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) cofs[c] = min(col_lane + c, a.N - 1);
  auto load_row = [&](const float* row) {
    if constexpr (WM == kWVector) {
      return __builtin_nontemporal_load(reinterpret_cast<const vec*>(row));
    } else if constexpr (WM == kWShared) {
      return *reinterpret_cast<const vec*>(row);
    } else {
      vec v;
#pragma unroll
      for (int c = 0; c < CPL; ++c) v[c] = __builtin_nontemporal_load(row + cofs[c]);
      return v;
    }
  };
  // Rows of X past M read row 0 instead: MFMA output row i depends only on
  // A row i, and those output rows are never stored.
  const float* xp[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int row = 16 * mb + li;
    xp[mb] = a.X + (int64_t)(row < a.M ? row : 0) * a.ldx + kbeg + 4 * lg;
  }

  // One step = 16 rows of the wave's K slice: per lane 4 W loads of CPL
  // columns (register q = 4u + s holds row 16u + s of the step) and one X load
  // per row block.
  auto load_w = [&](auto& w, int k) {
    constexpr int U = sizeof(w) / sizeof(w[0]) / 4;
    const float* wp = wbase + (int64_t)k * ldw;
#pragma unroll
    for (int q = 0; q < 4 * U; ++q) w[q] = load_row(wp + (int64_t)(16 * (q / 4) + q % 4) * ldw);
  };
  auto load_x = [&](auto& x, int k) {
    constexpr int U = sizeof(x) / sizeof(x[0]);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const f32x4u v = *reinterpret_cast<const f32x4u*>(xp[mb] + k + 16 * u);
        x[u][mb] = f32x4{v[0], v[1], v[2], v[3]};
      }
  };
  auto mfma_q = [&](f32x4 (&acc)[MB][CPL], const f32x4 (&xu)[MB], int s, const vec& wq) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        acc[mb][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(xu[mb][s], wq[c], acc[mb][c], 0, 0, 0);
  };

  // Main iterations of kU steps, walked from a hashed start. The loads are a
  // rotating pipeline: as soon as the MFMAs of W register q have been issued,
  // q is reloaded with the next iteration's row, so every wave keeps its 4*kU
  // W loads in flight while it computes instead of draining them before each
  // iteration. (The scheduling barrier keeps the compiler from sinking the
  // reloads to the end of the iteration.) For three or four row blocks this
  // also measured faster than loading, waiting and computing one iteration at
  // a time: at K = N = 8192, M = 48 80.5 vs 91.6 us and M = 64 104 vs 115 us;
  // at K = N = 4096 the two measure the same.
  const int nit = kwave / (16 * kU);
  const int r0 = nit > 0 ? (int)(((unsigned)blockIdx.x * 2654435761u >> 8) + (unsigned)wk * 977u) % nit : 0;
  if (nit > 0) {
    vec w[4 * kU];
    f32x4 x[kU][MB], xn[kU][MB];
    int it = r0;
    load_x(x, it * 16 * kU);
    load_w(w, it * 16 * kU);
    auto iteration = [&](auto set) __attribute__((always_inline)) {
      int itn = it + 1;
      if (itn >= nit) itn = 0;
      const int kn = itn * 16 * kU;
      load_x(xn, kn);
      const float* wp = wbase + (int64_t)kn * ldw;
#pragma unroll
      for (int q = 0; q < 4 * kU; ++q) {
        mfma_q(sum[(q / 4 + decltype(set)::value) % NS], x[q / 4], q % 4, w[q]);
        w[q] = load_row(wp + (int64_t)(16 * (q / 4) + q % 4) * ldw);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) x[u][mb] = xn[u][mb];
      it = itn;
    };
    int i = 1;
    // Unrolled only with two sets, which swap from one iteration to the next or
    // within it (16x8192x8192 44.8 -> 44.1 us; with one set it costs:
    // 48x4096x4097 25.4 against 24.7 us, 48x8192x8192 63.9 against 62.2).
    if constexpr (NS > 1)
      for (; i + 1 < nit; i += 2) {
        iteration(std::integral_constant<int, 0>{});
        iteration(std::integral_constant<int, kU % 2>{});
      }
    for (; i < nit; ++i) iteration(std::integral_constant<int, 0>{});
#pragma unroll
    for (int q = 0; q < 4 * kU; ++q) mfma_q(sum[(1 - q / 4) % NS], x[q / 4], q % 4, w[q]);
  }
  // Remaining single steps (kwave not a multiple of 16*kU).
  for (int k = nit * 16 * kU; k < kwave; k += 16) {
    vec w[4];
    f32x4 x[1][MB];
    load_x(x, k);
    load_w(w, k);
#pragma unroll
    for (int q = 0; q < 4; ++q) mfma_q(sum[NS - 1], x[0], q, w[q]);
  }

  f32x4 (&acc)[MB][CPL] = sum[0];
  if constexpr (NS > 1)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int c = 0; c < CPL; ++c) acc[mb][c] += sum[1][mb][c];

  // Sum the WK K-slices of each column block in wave order, one row block at
  // a time to bound LDS.
  __shared__ f32x4 red[WK > 1 ? WK - 1 : 1][WN][CPL][64];
  if constexpr (WK > 1) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      if (wk > 0) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) red[wk - 1][wn][c][lane] = acc[mb][c];
      }
      __syncthreads();
      if (wk == 0) {
#pragma unroll
        for (int w = 0; w < WK - 1; ++w)
#pragma unroll
          for (int c = 0; c < CPL; ++c) acc[mb][c] += red[w][wn][c][lane];
      }
      __syncthreads();
    }
    if (wk != 0) return;
  }

  // Lane holds rows 16*mb + 4*lg + r; register c is column col_lane + c, or
  // col_w + c on a lane whose columns reach past N: such a lane stores its
  // own columns only, one by one (a neighbour's workgroup walks K in another
  // order, so the others could differ in their last bits).
  if (col_lane >= a.N) return;
  const bool full = col_lane + CPL <= a.N;
  const int own = WM != kWScalar ? col_lane - col_w : 0;  // first register of an own column
  auto store = [&](float* row, const vec& v) {
    if (full) {
      *reinterpret_cast<vec*>(row + col_lane) = v;
    } else {
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        if (c >= own && col_lane + c - own < a.N) row[col_lane + c - own] = v[c];
    }
  };
  if (a.ksplit == 1) {
    vec bv;
#pragma unroll
    for (int c = 0; c < CPL; ++c) bv[c] = 0.0f;
    if (epi_has_bias(epi)) {
      if constexpr (WM != kWScalar) {
        bv = *reinterpret_cast<const vec*>(a.bias + col_w);
      } else {
#pragma unroll
        for (int c = 0; c < CPL; ++c) bv[c] = a.bias[cofs[c]];
      }
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * mb + 4 * lg + r;
        if (row < a.M) {
          vec y;
#pragma unroll
          for (int c = 0; c < CPL; ++c) y[c] = epilogue_rt(acc[mb][c][r], bv[c], a.alpha, epi);
          store(a.Y + (int64_t)row * a.ldy, y);
        }
      }
    return;
  }
  const int prow = 16 * MB;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * mb + 4 * lg + r;
      if (row < a.M) {
        vec p;
#pragma unroll
        for (int c = 0; c < CPL; ++c) p[c] = acc[mb][c][r];
        store(a.partials + ((int64_t)split * prow + row) * a.ldp, p);
      }
    }
}

// Y[m, 4j..4j+3] = epilogue(sum over splits s = 0..ksplit-1, in order, plus
// the K tail rows).
// All split loads are issued before the first add so their latencies overlap.
// W, the bias and Y may have any alignment; the last four columns of a row
// that N cuts short are read and written one by one. The partials always have
// an aligned row pitch (ldp, a multiple of 4). FULL: N % 4 == 0, no such columns
// (no load then waits behind a branch: 33x1235x1408 11.2 -> 10.9 us).
// One wave per workgroup spreads the reduction over more CUs than 256-thread
// workgroups (the c4 column shard: 16 workgroups of 256 threads); measured
// 0.2 us faster per layer at c4 and at its column shard.
template <bool FULL>
__global__ void __launch_bounds__(64) gemv_reduce_kernel(GemvF32Args a, int epi, int prow) {
  const int64_t idx = (int64_t)blockIdx.x * 64 + threadIdx.x;  // over M * ceil(N/4)
  const int n4 = (a.N + 3) / 4;
  if (idx >= (int64_t)a.M * n4) return;
  const int row = (int)(idx / n4);
  const int col = 4 * (int)(idx % n4);
  const bool full = FULL || col + 4 <= a.N;
  f32x4 v[kMaxSplit];
#pragma unroll
  for (int sp = 0; sp < kMaxSplit; ++sp)
    if (sp < a.ksplit)
      v[sp] = __builtin_nontemporal_load(
          reinterpret_cast<const f32x4*>(a.partials + ((int64_t)sp * prow + row) * a.ldp + col));
  f32x4 bv = {0.0f, 0.0f, 0.0f, 0.0f};
  if (epi_has_bias(epi)) {
    if (full) {
      const f32x4u v4 = *reinterpret_cast<const f32x4u*>(a.bias + col);
      bv = f32x4{v4[0], v4[1], v4[2], v4[3]};
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) bv[c] = col + c < a.N ? a.bias[col + c] : 0.0f;
    }
  }
  f32x4 s = v[0];
#pragma unroll
  for (int sp = 1; sp < kMaxSplit; ++sp)
    if (sp < a.ksplit) s += v[sp];
  // The K tail (at most 16 rows), after the split sums, in ascending k. All
  // its loads are issued before the first add (rows past k_end read row
  // k_end - 1 and are not added), so their latencies overlap.
  if (a.k_end > a.K) {
    float xt[kMaxTail];
    f32x4 wt[kMaxTail];
#pragma unroll
    for (int t = 0; t < kMaxTail; ++t) {
      const int k = min(a.K + t, a.k_end - 1);
      xt[t] = a.x_tail[(int64_t)row * a.ldx_tail + k];
      const float* wr = a.W + (int64_t)k * a.ldw + col;
      if (full) {
        const f32x4u v4 = *reinterpret_cast<const f32x4u*>(wr);
        wt[t] = f32x4{v4[0], v4[1], v4[2], v4[3]};
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) wt[t][c] = col + c < a.N ? wr[c] : 0.0f;
      }
    }
#pragma unroll
    for (int t = 0; t < kMaxTail; ++t)
      if (a.K + t < a.k_end) s += xt[t] * wt[t];
  }
  f32x4 y;
#pragma unroll
  for (int c = 0; c < 4; ++c) y[c] = epilogue_rt(s[c], bv[c], a.alpha, epi);
  float* dst = a.Y + (int64_t)row * a.ldy + col;
  if (full) {
    *reinterpret_cast<f32x4u*>(dst) = f32x4u{y[0], y[1], y[2], y[3]};
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (col + c < a.N) dst[c] = y[c];
  }
}

template <int MB, int WM, int NS>
hipError_t launch_mb_sets(int cols, int epi, const GemvF32Args& a, hipStream_t stream) {
  const dim3 grid(((a.N + cols - 1) / cols) * a.ksplit);
  auto block = [](int wn) { return dim3(waves_per_wg(MB, wn) * 64); };
  switch (cols) {
    case 32: hipLaunchKernelGGL((gemv_f32_kernel<MB, 2, 1, WM, NS>), grid, block(1), 0, stream, a, epi); break;
    case 64: hipLaunchKernelGGL((gemv_f32_kernel<MB, 4, 1, WM, NS>), grid, block(1), 0, stream, a, epi); break;
    case 128: hipLaunchKernelGGL((gemv_f32_kernel<MB, 4, 2, WM, NS>), grid, block(2), 0, stream, a, epi); break;
    case 256: hipLaunchKernelGGL((gemv_f32_kernel<MB, 4, 4, WM, NS>), grid, block(4), 0, stream, a, epi); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int MB, int WM>
hipError_t launch_mb_w(int cols, int epi, const GemvF32Args& a, hipStream_t stream) {
  if constexpr (MB > 2 && WM != kWScalar)
    if (!a.two_sets) return launch_mb_sets<MB, WM, 1>(cols, epi, a, stream);
  return launch_mb_sets<MB, WM, 2>(cols, epi, a, stream);
}

template <int MB>
hipError_t launch_mb(int cols, int epi, const GemvF32Args& a, hipStream_t stream) {
  switch (a.w_mode) {
    case kWVector: return launch_mb_w<MB, kWVector>(cols, epi, a, stream);
    case kWShared: return launch_mb_w<MB, kWShared>(cols, epi, a, stream);
    case kWScalar: return launch_mb_w<MB, kWScalar>(cols, epi, a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

int gemv_f32_waves_k(int cols, int M) {
  const int wn = cols <= 64 ? 1 : cols / 64;
  return waves_per_wg((M + 15) / 16, wn) / wn;
}

int gemv_f32_w_mode(const float* W, int64_t ldw, int N) {
  if (N < 4) return kWScalar;
  return reinterpret_cast<uintptr_t>(W) % 128 == 0 && ldw % 32 == 0 ? kWVector : kWShared;
}
int gemv_f32_max_ksplit() { return kMaxSplit; }

hipError_t launch_gemv_f32(int epi, int cols, GemvF32Args a, hipStream_t stream) {
  const int mb = (a.M + 15) / 16;
  if (a.k_end < a.K || a.k_end - a.K > kMaxTail || (a.k_end > a.K && a.ksplit < 2)) return hipErrorInvalidValue;
  hipError_t e;
  switch (mb) {
    case 1: e = launch_mb<1>(cols, epi, a, stream); break;
    case 2: e = launch_mb<2>(cols, epi, a, stream); break;
    case 3: e = launch_mb<3>(cols, epi, a, stream); break;
    case 4: e = launch_mb<4>(cols, epi, a, stream); break;
    default: return hipErrorInvalidValue;
  }
  if (e != hipSuccess || a.ksplit == 1) return e;
  const int64_t items = (int64_t)a.M * ((a.N + 3) / 4);
  const dim3 g((unsigned)((items + 63) / 64));
  if (a.N % 4 == 0)
    hipLaunchKernelGGL(gemv_reduce_kernel<true>, g, dim3(64), 0, stream, a, epi, 16 * mb);
  else
    hipLaunchKernelGGL(gemv_reduce_kernel<false>, g, dim3(64), 0, stream, a, epi, 16 * mb);
  return hipGetLastError();
}

}  // namespace edsl
