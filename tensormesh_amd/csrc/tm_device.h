// Device helpers shared by the element kernels (HIP translation units only).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tmh {

// Node pairs an element kernel computes: all B*B (i, j) in row-major order,
// or with `upper` the B(B+1)/2 pairs i <= j (row-major as well).  Entry p of
// the LDS table packs (i << 8) | j; returns the number of pairs.
template <int B>
__device__ __forceinline__ int fill_pairs(uint16_t* pairs, bool upper) {
  if (!upper) {
    for (int p = threadIdx.x; p < B * B; p += blockDim.x) pairs[p] = (uint16_t)(((p / B) << 8) | (p % B));
    return B * B;
  }
  for (int p = threadIdx.x; p < B * (B + 1) / 2; p += blockDim.x) {
    int i = 0, r = p;
    while (r >= B - i) {  // row i holds B - i pairs
      r -= B - i;
      ++i;
    }
    pairs[p] = (uint16_t)((i << 8) | (i + r));
  }
  return B * (B + 1) / 2;
}

// Orders a wavefront's LDS accesses before and after it for lanes that read
// each other's words (the hardware runs one wave's LDS accesses in order, so
// this costs nothing; a workgroup barrier would make four waves wait for the
// slowest of them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Stores one block of N values per lane (acc, bound for out + dst * N; dst < 0:
// none).  Float64 blocks go through LDS, kStageBlocks at a time, so that
// consecutive lanes write consecutive words of a block: stores of whole
// 72-byte blocks from each lane keep the address unit busy for about 160
// cycles per 64 lanes of 16 bytes (Neo-Hookean tetra10: 1.75e8 of its cycles
// against 1.20e8 staged, 60 M write requests to L2 against 23 M, kernel
// 398 -> 360 us).  Float32 blocks are half that and leave the lanes directly:
// staged, the same kernel went from 133 to 141 us at 24^3 x 6 elements.  STAGE
// = false: callers whose lanes hold few blocks, or small ones, at a time.
// stage: stage_bytes<T, N>() bytes of LDS of this wavefront.
constexpr int kStageBlocks = 32;
template <typename T, int N, bool STAGE = sizeof(T) == 8>
constexpr int stage_bytes() {
  return STAGE ? kStageBlocks * (N * (int)sizeof(T) + 4) : 0;
}

// transposed: the D x D block (N = D * D) is stored transposed.
template <typename T, int N, bool STAGE = sizeof(T) == 8>
__device__ __forceinline__ void store_blocks(char* stage, const double (&acc)[N], int32_t dst, bool transposed,
                                             T* __restrict__ out) {
  constexpr int D = N == 9 ? 3 : N == 4 ? 2 : 1;
  T v[N];
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = (T)acc[k];
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int c = a + 1; c < D; ++c) {
      const T up = v[a * D + c], lo = v[c * D + a];
      v[a * D + c] = transposed ? lo : up;
      v[c * D + a] = transposed ? up : lo;
    }
  if constexpr (!STAGE) {
    if (dst >= 0) {
#pragma unroll
      for (int k = 0; k < N; ++k) out[(int64_t)dst * N + k] = v[k];
    }
    return;
  }
  T* const val = reinterpret_cast<T*>(stage);
  int32_t* const at = reinterpret_cast<int32_t*>(val + kStageBlocks * N);
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 0; h < 64 / kStageBlocks; ++h) {
    wave_sync();
    if (lane / kStageBlocks == h) {
#pragma unroll
      for (int k = 0; k < N; ++k) val[(lane % kStageBlocks) * N + k] = v[k];
      at[lane % kStageBlocks] = dst;
    }
    wave_sync();
#pragma unroll
    for (int f0 = 0; f0 < kStageBlocks * N; f0 += 64) {
      const int f = f0 + lane;
      if (f < kStageBlocks * N) {
        const int b = f / N;
        const int32_t d = at[b];
        if (d >= 0) out[(int64_t)d * N + (f - b * N)] = val[f];
      }
    }
  }
}

// Bijection from the hardware dispatch order (workgroup b of a launch runs on
// XCD b mod 8) to a logical order in which every XCD owns one contiguous
// range of [0, nb): neighbouring logical workgroups then share that XCD's L2,
// and so do launches that map the same logical workgroup to the same rows.
__device__ __forceinline__ int64_t xcd_block(int64_t b, int64_t nb) {
  const int64_t q = nb / 8, r = nb % 8;
  const int64_t x = b % 8, y = b / 8;
  return x < r ? x * (q + 1) + y : r * (q + 1) + (x - r) * q + y;
}

// a * b + c rounded once, whatever the file's contraction mode.
template <typename T>
__device__ __forceinline__ T fma_t(T a, T b, T c) {
  if constexpr (sizeof(T) == 8)
    return __builtin_fma(a, b, c);
  else
    return __builtin_fmaf(a, b, c);
}

// v of lane f(l) for the cross-lane pattern CTRL of a DPP move.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Sum of v over the wavefront, in every lane: the bits of the butterfly
// v += v(lane ^ 32), v(lane ^ 16), .. v(lane ^ 1).  After step m all lanes that
// agree modulo m hold the same value, so a rotation by m within a row of 16
// (DPP, a few cycles) serves steps 8 to 1 and the 32- and 16-lane swaps the
// first two, in place of six LDS-pipe permutes of two words each (ds_bpermute,
// ~100 cycles).
__device__ __forceinline__ double wave_sum(double v) {
  {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  }
  {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  }
  v += dpp_move<0x128>(v);  // row_ror:8
  v += dpp_move<0x124>(v);  // row_ror:4
  v += dpp_move<0x122>(v);  // row_ror:2
  v += dpp_move<0x121>(v);  // row_ror:1
  return v;
}

// A value that is the same in every lane, moved to scalar registers.
__device__ __forceinline__ double uniform(double v) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                          __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Float32 geometry of a P1 simplex, and when it must be redone in float64.
// With edges e_k = x_{k+1} - x_0 and det = det[e_0 .. e_{D-1}], the shape
// quality q = |det| / prod_k |e_k| (the volume over that of the box on the
// edges: 1 for right angles, -> 0 for slivers and needles) bounds the float32
// cancellation: the rounding error of the local matrix, relative to its
// largest entry, grows like eps / q (measured over 300,000 random tetrahedra
// and triangles with q down to 1e-4: at most 7.8e-7 for q >= 0.1).  Elements
// with q < kSliverQ, and degenerate ones, are flagged for float64.  Evaluated
// as a product of O(h) ratios, so that no term under- or overflows for edge
// lengths h within float32's exponent range.
constexpr float kSliverQ = 0.1f;

template <int D>
__device__ __forceinline__ bool sliver_f32(const float (&e)[D][D], float det) {
  float l[D];
#pragma unroll
  for (int k = 0; k < D; ++k) {
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < D; ++j) s += e[k][j] * e[k][j];
    l[k] = s;
  }
  const float r0 = det * __builtin_amdgcn_rcpf(l[0]);
  float lhs, rhs;
  if constexpr (D == 3) {
    lhs = r0 * (det * __builtin_amdgcn_rcpf(l[1]));  // det^2 / (l0 l1)
    rhs = kSliverQ * kSliverQ * l[2];
  } else {
    lhs = r0 * det;  // det^2 / l0
    rhs = kSliverQ * kSliverQ * l[1];
  }
  return !(lhs >= rhs);  // NaN (a zero edge) counts as a sliver
}

// Per-point D x D sums of one element, spread over the element's L lanes:
//   out[q][r * D + c] = (diag && r == c) + sum_{b < B} a(q, r, b) * m(q, b, c)
// One (q, r, c) per lane when the MQ D D entries (MQ >= Q, the instance's
// largest rule) fit in one pass of the lanes, else one row (q, r) per lane.
// Both take the nodes in order, so they give the same bits.
template <int D, int B, int L, int MQ, typename A, typename M, typename Out>
__device__ __forceinline__ void point_sums(int lane, int Q, bool diag, A a, M m, Out out) {
  if constexpr (MQ * D * D <= L) {
    if (lane < Q * D * D) {
      const int q = lane / (D * D), r = (lane / D) % D, c = lane % D;
      double s = (diag && r == c) ? 1.0 : 0.0;
      for (int b = 0; b < B; ++b) s += a(q, r, b) * m(q, b, c);
      out(q, r, c) = s;
    }
    return;
  }
  for (int t = lane; t < Q * D; t += L) {
    const int q = t / D, r = t % D;
    double s[D];
#pragma unroll
    for (int c = 0; c < D; ++c) s[c] = (diag && r == c) ? 1.0 : 0.0;
    for (int b = 0; b < B; ++b) {
      const double ab = a(q, r, b);
#pragma unroll
      for (int c = 0; c < D; ++c) s[c] += ab * m(q, b, c);
    }
#pragma unroll
    for (int c = 0; c < D; ++c) out(q, r, c) = s[c];
  }
}

}  // namespace tmh
