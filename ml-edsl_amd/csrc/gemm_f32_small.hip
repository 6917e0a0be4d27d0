// fp32 dense layer / matmul for small outputs, any shape, row stride and
// alignment: a 16x16 tile per workgroup of 4 or 8 waves that split K.
//
// C[M,N] = epilogue(A[M,K] x B[K,N] (+ bias[N])) -- the same op as the other
// tiles (reference cpp/src/builders/LinalgBuilder.cpp:106-139, 180-239,
// 301-339), for layers that are bound by latency: their work is microseconds,
// so what counts is how often a wave waits for memory and how many launches
// there are.
//
//  * v_mfma_f32_16x16x4_f32 on 16-deep groups of K: lane l of a wave supplies
//    row l%16 of A and column l%16 of B at k = 16j + 4(l/16) .. +3, one
//    16-byte load of the A row (any 4-byte alignment) and four 4-byte loads of
//    B. A wave issues the loads of up to eight groups before its first MFMA:
//    with K split over enough waves it waits for memory once.
//  * K % 16 rows are one more group, its last k masked, loaded by the last
//    wave before it computes its own groups.
//  * The waves' partial blocks are summed through LDS in wave order (the
//    result depends on the shape only) and written with the epilogue, one
//    output per thread.
// Rows past M and columns past N read the last row or column; their outputs
// are not stored.
#include "common.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace edsl {
namespace {

// Four floats at any 4-byte aligned address.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct Group {
  f32x4 a;  // row l%16, k 4(l/16) .. +3 of the group
  f32x4 b;  // column l%16, the same k
};

template <int WAVES>
__global__ void __launch_bounds__(64 * WAVES) gemm_f32_small_kernel(GemmF32Args args, int epi) {
  __shared__ f32x4 red[WAVES][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  int tm, tn;
  tile_coords(blockIdx.x, args.tiles_m, args.tiles_n, tm, tn);
  const int m0 = tm * 16, n0 = tn * 16;
  const int K = args.K;
  const int64_t ldb = args.ldb;
  const float* pa = args.A + (int64_t)min(m0 + r16, args.M - 1) * args.lda + 4 * g;
  const float* pb = args.B + 4 * g * ldb + min(n0 + r16, args.N - 1);
  const int ng = K / 16;
  const int jb = (int)((int64_t)wave * ng / WAVES), je = (int)((int64_t)(wave + 1) * ng / WAVES);

  auto load = [&](Group& f, int j) __attribute__((always_inline)) {
    const f32x4u v = *reinterpret_cast<const f32x4u*>(pa + 16 * j);
    f.a = f32x4{v[0], v[1], v[2], v[3]};
    const float* p = pb + 16 * j * ldb;
#pragma unroll
    for (int s = 0; s < 4; ++s) f.b[s] = p[s * ldb];
  };
  f32x4 acc[8] = {};
  auto mfmas = [&](const Group& f, f32x4& c) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f32_16x16x4f32(f.a[s], f.b[s], c, 0, 0, 0);
  };

  Group tail;
  const bool has_tail = wave == WAVES - 1 && (K & 15) != 0;  // uniform per wave
  if (has_tail) {
    const int k0 = 16 * ng;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 4 * g + s, kc = min(k, K - 1);
      const float av = pa[kc - 4 * g], bv = pb[(kc - 4 * g) * ldb];
      tail.a[s] = k < K ? av : 0.0f;
      tail.b[s] = k < K ? bv : 0.0f;
    }
  }
  // Up to U groups of loads, then their MFMAs; loads past the wave's last
  // group repeat it.
  auto batch = [&](int j, auto uc) __attribute__((always_inline)) {
    constexpr int U = decltype(uc)::value;
    Group f[U];
#pragma unroll
    for (int u = 0; u < U; ++u) load(f[u], min(j + u, je - 1));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (j + u < je) mfmas(f[u], acc[u]);
  };
  const int n = je - jb;
  if (n > 4) {
    for (int j = jb; j < je; j += 8) batch(j, std::integral_constant<int, 8>{});
  } else if (n > 2) {
    batch(jb, std::integral_constant<int, 4>{});
  } else if (n > 0) {
    batch(jb, std::integral_constant<int, 2>{});
  }
  if (has_tail) mfmas(tail, acc[7]);

  const int e = threadIdx.x >> 6;
  const int row = m0 + 4 * g + e, col = n0 + r16;
  const bool out = e < 4 && row < args.M && col < args.N;
  const float bias = out && epi_has_bias(epi) ? args.bias[col] : 0.0f;
  red[wave][lane] = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  __syncthreads();
  if (!out) return;
  const float* p = reinterpret_cast<const float*>(red) + lane * 4 + e;
  float v[WAVES];
#pragma unroll
  for (int w = 0; w < WAVES; ++w) v[w] = p[w * 256];
  float s = v[0];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) s += v[w];
  args.C[(int64_t)row * args.ldc + col] = epilogue_rt(s, bias, args.alpha, epi);
}

}  // namespace

hipError_t launch_gemm_f32_small(int waves, int epi, GemmF32Args a, hipStream_t stream) {
  if (a.M < 1 || a.N < 1 || a.K < 1) return hipErrorInvalidValue;
  a.tiles_m = (a.M + 15) / 16;
  a.tiles_n = (a.N + 15) / 16;
  const dim3 grid(a.tiles_m * a.tiles_n), block(64 * waves);
  switch (waves) {
    case 4: hipLaunchKernelGGL(gemm_f32_small_kernel<4>, grid, block, 0, stream, a, epi); break;
    case 8: hipLaunchKernelGGL(gemm_f32_small_kernel<8>, grid, block, 0, stream, a, epi); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace edsl
