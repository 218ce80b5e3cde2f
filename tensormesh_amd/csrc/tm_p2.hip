// Stage G for every cell but the scalar P1 forms: element matrices
// (wave_element_kernel) and the Neo-Hookean residual and tangent
// (hyper_wave_kernel), one or more elements per wavefront.
//
// Replaces the same reference chain as tm_p1.hip -- eval_shape_grad
// (tensormesh/element/element.py:956-968), jxw (transformation.py:1265-1272),
// the vmap'd forward and _integrate (element_assembler.py:190-209,416-438) --
// for triangle6 / tetra10 and larger cells and for
// LinearElasticityElementAssembler (builtin.py:172-178), where the Jacobian
// varies per quadrature point and a local matrix has up to 81 x 81 entries.
//
// Work split among an element's lanes:
//   1. lanes load the element's B*D coordinates into LDS;
//   2. J_q[i][j] = sum_b x[b][j] dphi_q[i][b], its inverse and
//      jxw_q = w_q |det J_q|, by point q's lane or with the sums spread over
//      the lanes;
//   3. grad_q[b][d] = sum_i dphi_q[i][b] Jinv_q[d][i] into LDS;
//   4. lanes take tiles of node pairs (i, j); a pair's H x H block, from sums
//      over the points, is written to slot (e*B + i)*B + j -- the flattening of
//      the reference's [E, B, B, H, H] element tensor -- or packed, or in
//      contribution order (TM_FLAG_UPPER, slot_dest).
// Linear elasticity uses Ba^T C Bb in closed form:
//   (Ba^T C Bb)[a][c] = lam g_i[a] g_j[c] + mu g_i[c] g_j[a] + mu delta_ac g_i.g_j
// which is the product of the Voigt matrices of functional/elasticity.py:132-284.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "tm_device.h"
#include "tm_internal.h"

namespace {

constexpr int kWave = 64;
constexpr int kWavesPerBlock = 4;
constexpr int kMaxQ = 16;      // Neo-Hookean kernel
constexpr int kMaxQWave = 32;  // element-matrix kernel (a 3 x 3 x 3 hexahedron rule has 27 points)

// Dispatch order with chunks of kChunk logical workgroups on one XCD, 8 chunks
// in flight at a time; a last part group keeps the dispatch order.
constexpr int kChunk = 64;
__device__ __forceinline__ int64_t xcd_chunks(int64_t b, int64_t nb) {
  const int64_t g = b / (8 * kChunk), r = b % (8 * kChunk);
  return (g + 1) * 8 * kChunk > nb ? b : g * 8 * kChunk + (r % 8) * kChunk + r / 8;
}

// Nodes per side of the tile of node pairs that a lane owns, for B nodes on L
// lanes and rules of at most MQ points.  A 2 x 2 tile reads four gradients for
// four pairs where single pairs read eight, so it is the better one where
// there are tiles for most lanes (as many elements per wavefront as that).
// With one or two elements (rules of many points, whose gradients fill LDS)
// most lanes would have no tile: single pairs as long as they take at most
// twice the rounds of the lanes.  Float32 blocks leave the lanes directly, and
// a tile's are two blocks apart: single pairs there as well while the sums are
// short.  Element kernel of linear elasticity, upper blocks, 2 x 2 / single
// (us): 36^3 x 6 tetra, 5 points, float64, 353 / 137, 400^2 quads, 9 points,
// 137 / 61 (59 before there were tiles); whole blocks with their reduction,
// 12^3 x 6 tetra20, 4 points, float32, 138 / 116 (119), 24 points 253 / 270.
constexpr int tile_side(int B, int L, int MQ, bool blocks_f32) {
  const int nt = (B + 1) / 2, tiles = nt * (nt + 1) / 2, pairs = B * (B + 1) / 2;
  const int r1 = (pairs + L - 1) / L, r2 = (tiles + L - 1) / L;
  return r1 <= (L >= 32 ? 2 : 1) * r2 || (blocks_f32 && L >= 32 && MQ <= 16) ? 1 : 2;
}

// MQ: largest number of quadrature points the LDS arrays hold.  upper: only
// the blocks i <= j (symmetric forms, TM_FLAG_UPPER); block (j, i) is always
// stored as the exact transpose of block (i, j).  EPW elements per wavefront
// on L = 64 / EPW lanes each, WPB wavefronts per workgroup; an element's
// stages stay within its wavefront and need no workgroup barrier.
//
// Linear elasticity: a lane owns a tile of node pairs, 2 x 2 or a single one
// (tile_side), and accumulates, per pair, S[a][c] = sum_q jxw_q g_i[a] g_j[c]; the block is
//   lam S[a][c] + mu S[c][a] + mu delta_ac tr S,
// 12 float64 operations per pair and point instead of 42 when the block is
// formed at every point, and four gradients read from LDS for four pairs
// instead of eight.  Measured: hexahedra 40^3 float32 84 -> 62 us, tetra10
// 17^3 x 6 float64 59 -> 48.5 us.  Half of that is the block stores (41 and 30 us
// without them), the rest latency: an element's stages depend on each other
// and its gradients (1.5 KB) limit the wavefronts in flight.
//
// Scalar forms use the same tiles (upper ones only, a value stands for (i, j)
// and (j, i)) and write the element's matrix from LDS, or single pairs of one
// round from the lanes (mass on tetra10, 24 points, 57 -> 49 us): Laplace and diffusion
// on hexahedra 40^3 float64 66 -> 46 us, tetra10 20^3 x 6 float32 44 -> 29 us.
template <typename T, int D, int B, int H, int FORM, int MQ, int EPW, int WPB>
__global__ void __launch_bounds__(kWave * WPB)
    wave_element_kernel(const int32_t* __restrict__ conn, const T* __restrict__ pts,
                        const T* __restrict__ coeff, const double* __restrict__ tab, int Q,
                        double lam, double mu, int64_t n_elem, int upper, T* __restrict__ slot,
                        const int32_t* __restrict__ slot_dest) {
  constexpr int L = kWave / EPW;   // lanes per element
  constexpr int kEpb = WPB * EPW;  // elements per workgroup
  constexpr bool kBlock = FORM == TM_FORM_LINEAR_ELASTICITY;
  constexpr int TS = tile_side(B, L, MQ, kBlock && sizeof(T) == 4);  // nodes per side of a tile
  constexpr int NT = (B + TS - 1) / TS;                               // tiles per side
  constexpr int NP = TS * TS;                                         // pairs per tile
  __shared__ double s_tab[MQ * (1 + B + D * B)];
  __shared__ uint16_t s_tile[NT * NT];
  // odd strides between many elements: with even ones (192 doubles for
  // hexahedra) the elements of a wavefront met in the same banks, half of all
  // LDS cycles.  With one or two elements even ones, which keep the reads of
  // two gradient components 16-byte aligned (quads 400^2, 9 points, 70 -> 51 us).
  constexpr int kOdd = EPW > 2 ? 1 : 0;
  __shared__ double s_jxw[kEpb][MQ | kOdd];
  __shared__ double s_kq[kBlock ? 1 : kEpb][MQ | kOdd];
  // a scalar form of one round of single pairs stores its values from the lanes
  constexpr bool kDirect = !kBlock && TS == 1 && NT * (NT + 1) / 2 <= L;
  // gradients (none for the mass form), then a scalar form's matrix
  constexpr int kGrad = FORM == TM_FORM_MASS ? 1 : MQ * B * D, kMat = kBlock || kDirect ? 1 : B * B;
  __shared__ double s_g[kEpb][(kGrad > kMat ? kGrad : kMat) | kOdd];
  __shared__ uint16_t s_pair[kBlock || kDirect ? 1 : B * B];
  __shared__ int s_v[FORM == TM_FORM_DIFFUSION_NODE ? kEpb : 1][B];
  // with many elements per wavefront and points for more than half of an
  // element's lanes, a point's lane goes from the coordinates to its gradients
  // in registers; else the sums and the gradients are spread over the lanes,
  // through inv (Laplace, us, in registers / spread: hexahedra 40^3, 27 points
  // on 64 lanes, 237 / 198; tetra10 18^3 x 6 with the reduction, 5 points on 16
  // lanes, 46.9 / 44.3)
  constexpr bool kFused = 2 * MQ > L && EPW > 2;
  constexpr int kInv = kFused ? 0 : MQ * D * D;
  // what the blocks no longer need: each wavefront stages their stores there
  struct Early {
    double x[(B * D + kInv) % 2 == kOdd ? B * D : B * D + 1], inv[kFused ? 1 : MQ][kFused ? 1 : D * D];
  };
  // Float64 blocks are stored through LDS, except a few per wavefront (36^3 x 6
  // tetra, 5 points, two elements, 137 -> 110 us) and the 32-byte ones of four
  // elements or less (quads of 9 nodes, whole blocks, two elements, 71 -> 64)
  constexpr bool kStage = sizeof(T) == 8 && !(TS == 1 && B * (B + 1) <= L) && !(D == 2 && EPW <= 4);
  constexpr int kEarly = EPW * (int)sizeof(Early), kBlocks = kBlock ? tmh::stage_bytes<T, H * H, kStage>() : 0;
  __shared__ __align__(16) char s_mem[WPB][kEarly > kBlocks ? kEarly : kBlocks];

  const int lane = threadIdx.x % kWave % L;          // lane within the element's group
  const int sub = threadIdx.x % kWave / L;           // element within the wavefront (EPW: a lane left over)
  const int wv = threadIdx.x / kWave * EPW + (sub < EPW ? sub : 0);  // element slot within the workgroup
  // Chunks of consecutive workgroups on one XCD: neighbours write neighbouring
  // contribution-ordered slots, which then merge in one L2, and the elements
  // are still taken nearly in order, so that the slots written last are the
  // ones the reduction reads first.  Element kernel + reduction (float64, us)
  // in dispatch order, in one contiguous range per XCD and in chunks of 16, 64,
  // 256: 64^3 hexahedra 697, 702, 679, 672, 671; 30^3 x 6 tetra10 636, 613, 607,
  // 588, 597; 17^3 x 6 102.5, 100.1, 100.0, 99.3, 103.3.  (The Neo-Hookean
  // launch, which has other work per block, gains nothing: 385-404 without,
  // 390, 392, 405 with chunks of 4, 16, 64.)
  const int64_t e = xcd_chunks(blockIdx.x, gridDim.x) * kEpb + wv;
  const bool active = sub < EPW && e < n_elem;
  char* const mem = s_mem[threadIdx.x / kWave];
  Early& el = reinterpret_cast<Early*>(mem)[sub < EPW ? sub : 0];

  const int tab_len = Q + Q * B + Q * D * B;
  for (int t = threadIdx.x; t < tab_len; t += blockDim.x) s_tab[t] = tab[t];
  // scalar forms compute the upper tiles only and store each value twice
  const int n_tiles = tmh::fill_pairs<NT>(s_tile, !kBlock || upper != 0);
  const int n_pairs = upper ? B * (B + 1) / 2 : B * B;
  if constexpr (!kBlock && !kDirect) tmh::fill_pairs<B>(s_pair, upper != 0);
  const double* w = s_tab;
  const double* phi = s_tab + Q;
  const double* dphi = s_tab + Q + Q * B;

  // a lane loads whole nodes: the two dependent loads of an element are one
  // round trip each
  if (active)
    for (int b = lane; b < B; b += L) {
      const int64_t v = conn[e * B + b];
      if constexpr (FORM == TM_FORM_DIFFUSION_NODE) s_v[wv][b] = (int)v;
#pragma unroll
      for (int d = 0; d < D; ++d) el.x[b * D + d] = (double)pts[v * D + d];
    }
  __syncthreads();
  // the slots of the pairs of the lane's first tile (contribution order),
  // loaded now so that their latency hides behind the per-point stages.
  // Pair p of the table is block (i, j): full blocks at p = i*B + j, upper
  // blocks packed at their index among the pairs i <= j
  constexpr int HH = H * H;
  auto pair_slot = [&](int i, int j) -> int32_t {
    if (i >= B || j >= B || (upper && i > j)) return -1;
    const int p = upper ? i * B - i * (i - 1) / 2 + j - i : i * B + j;
    return slot_dest ? slot_dest[e * n_pairs + p] : (int32_t)(e * n_pairs + p);
  };
  auto tile_slots = [&](int t, int32_t (&d)[NP], bool (&has)[NP]) {
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int i = TS * (s_tile[t] >> 8) + k / TS, j = TS * (s_tile[t] & 255) + k % TS;
      has[k] = i < B && j < B && (!upper || i <= j);
      d[k] = has[k] ? pair_slot(i, j) : 0;
    }
  };
  int32_t dst[NP] = {};
  bool has[NP] = {};
  if constexpr (kBlock)
    if (active && lane < n_tiles) tile_slots(lane, dst, has);
  tmh::wave_sync();
  // Jacobian J[i][j] = sum_b dphi_b[i] x_b[j], inverse, weight and gradients
  // g_b[d] = sum_i dphi_b[i] inv[d][i] of every point
  auto point = [&](int q, const double (&J)[D][D], double (&inv)[D][D]) {
    double det;
    if constexpr (D == 2) {
      det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
      inv[0][0] = J[1][1] / det;
      inv[0][1] = -J[0][1] / det;
      inv[1][0] = -J[1][0] / det;
      inv[1][1] = J[0][0] / det;
    } else {
      const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
      const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
      const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
      det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
      const double r = 1.0 / det;
      inv[0][0] = c00 * r;
      inv[1][0] = c01 * r;
      inv[2][0] = c02 * r;
      inv[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * r;
      inv[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * r;
      inv[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * r;
      inv[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * r;
      inv[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * r;
      inv[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * r;
    }
    s_jxw[wv][q] = w[q] * fabs(det);
    if constexpr (!kBlock) {
      double kq = 1.0;
      if constexpr (FORM == TM_FORM_DIFFUSION_ELEM) kq = (double)coeff[e];
      if constexpr (FORM == TM_FORM_DIFFUSION_NODE) {
        kq = 0.0;
        for (int b = 0; b < B; ++b) kq += (double)coeff[s_v[wv][b]] * phi[q * B + b];
      }
      s_kq[wv][q] = kq;
    }
  };
  auto gradient = [&](int q, int b, const double (&inv)[D][D]) {
    if constexpr (FORM == TM_FORM_MASS) return;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < D; ++i) s += dphi[(q * D + i) * B + b] * inv[d][i];
      s_g[wv][(q * B + b) * D + d] = s;
    }
  };
  if constexpr (kFused) {
    if (active)
      for (int q = lane; q < Q; q += L) {
        double J[D][D], inv[D][D];
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
          for (int j = 0; j < D; ++j) {
            double s = 0.0;
#pragma unroll
            for (int b = 0; b < B; ++b) s += dphi[(q * D + i) * B + b] * el.x[b * D + j];
            J[i][j] = s;
          }
        point(q, J, inv);
#pragma unroll
        for (int b = 0; b < B; ++b) gradient(q, b, inv);
      }
  } else {
    // (J into inv, which point q's lane then overwrites with the inverse)
    if (active)
      tmh::point_sums<D, B, L, MQ>(
          lane, Q, false, [&](int q, int i, int b) { return dphi[(q * D + i) * B + b]; },
          [&](int, int b, int j) { return el.x[b * D + j]; },
          [&](int q, int i, int j) -> double& { return el.inv[q][i * D + j]; });
    tmh::wave_sync();
    if (active)
      for (int q = lane; q < Q; q += L) {
        double J[D][D], inv[D][D];
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
          for (int j = 0; j < D; ++j) J[i][j] = el.inv[q][i * D + j];
        point(q, J, inv);
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
          for (int j = 0; j < D; ++j) el.inv[q][i * D + j] = inv[i][j];
      }
    tmh::wave_sync();
    if (active)
      for (int t = lane; t < Q * B; t += L) {
        const int q = t / B, b = t - q * B;
        double inv[D][D];
#pragma unroll
        for (int d = 0; d < D; ++d)
#pragma unroll
          for (int i = 0; i < D; ++i) inv[d][i] = el.inv[q][d * D + i];
        gradient(q, b, inv);
      }
  }
  tmh::wave_sync();
  if constexpr (kBlock) {
#pragma unroll 1
    for (int t0 = 0; t0 < n_tiles; t0 += L) {
      const int t = t0 + lane;
      const bool mine = active && t < n_tiles;
      // tile (I, J) of the lower half is formed as (J, I) and transposed
      int I = mine ? s_tile[t] >> 8 : 0, J = mine ? s_tile[t] & 255 : 0;
      const bool low = I > J;
      if (t0 > 0) {
        if (mine) {
          tile_slots(t, dst, has);
        } else {
#pragma unroll
          for (int k = 0; k < NP; ++k) has[k] = false;
        }
      }
      if (low) {
        const int u = I;
        I = J;
        J = u;
      }
      // the tile's nodes, those past the last one standing in as the last
      int ti[TS], tj[TS];
#pragma unroll
      for (int k = 0; k < TS; ++k) {
        ti[k] = TS * I + k < B ? TS * I + k : B - 1;
        tj[k] = TS * J + k < B ? TS * J + k : B - 1;
      }
      double S[NP][HH];
#pragma unroll
      for (int k = 0; k < NP; ++k)
#pragma unroll
        for (int n = 0; n < HH; ++n) S[k][n] = 0.0;
      for (int q = 0; q < Q; ++q) {
        const double* g = &s_g[wv][q * B * D];
        const double wq = s_jxw[wv][q];
        double gi[TS][D], gj[TS][D];
#pragma unroll
        for (int k = 0; k < TS; ++k)
#pragma unroll
          for (int d = 0; d < D; ++d) {
            gi[k][d] = g[ti[k] * D + d] * wq;
            gj[k][d] = g[tj[k] * D + d];
          }
#pragma unroll
        for (int k = 0; k < NP; ++k)
#pragma unroll
          for (int a = 0; a < D; ++a)
#pragma unroll
            for (int c = 0; c < D; ++c) S[k][a * D + c] += gi[k / TS][a] * gj[k % TS][c];
      }
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        // pair k of the tile as stored, (TS I + k/TS, TS J + k%TS) before the
        // swap: sums of pair (lo, hi), the diagonal tile's (1, 0) from its (0, 1)
        constexpr int kTurn = TS == 2 ? 2 : -1;
        const int mirror = (k % TS) * TS + k / TS;
        const bool turned = k == kTurn && I == J;
        double s[HH];
#pragma unroll
        for (int n = 0; n < HH; ++n) s[n] = low || turned ? S[mirror][n] : S[k][n];
        const bool flip = low || turned;
        // pair (i, i): the sums above the diagonal stand for those below
        const bool self = I == J && k % TS == k / TS;
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
          for (int c = 0; c < a; ++c) s[a * D + c] = self ? s[c * D + a] : s[a * D + c];
        double tr = 0.0;
#pragma unroll
        for (int a = 0; a < D; ++a) tr += s[a * D + a];
        double blk[HH];
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
          for (int c = 0; c < D; ++c) {
            double v = lam * s[a * D + c] + mu * s[c * D + a];
            if (a == c) v += mu * tr;
            blk[a * D + c] = v;
          }
        const bool neg = slot_dest && dst[k] < 0;   // contribution order: read as (j, i)
        tmh::store_blocks<T, HH, kStage>(mem, blk, has[k] ? dst[k] & INT32_MAX : -1, flip != neg, slot);
      }
    }
    return;
  }
  static_assert(kBlock || H == 1, "scalar forms have one value per pair");
  // the values of the lane's tiles, then the element's B x B matrix in the
  // place of its gradients, then contiguous stores
  constexpr int kRounds = (NT * (NT + 1) / 2 + L - 1) / L;
  double S[kRounds][NP];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int t = lane + r * L;
#pragma unroll
    for (int k = 0; k < NP; ++k) S[r][k] = 0.0;
    if (active && t < n_tiles) {
      int ti[TS], tj[TS];
#pragma unroll
      for (int k = 0; k < TS; ++k) {
        const int i = TS * (s_tile[t] >> 8) + k, j = TS * (s_tile[t] & 255) + k;
        ti[k] = i < B ? i : B - 1;
        tj[k] = j < B ? j : B - 1;
      }
      for (int q = 0; q < Q; ++q) {
        const double wq = s_jxw[wv][q];
        if constexpr (FORM == TM_FORM_MASS) {
          const double* ph = phi + q * B;
          double pi[TS], pj[TS];
#pragma unroll
          for (int k = 0; k < TS; ++k) {
            pi[k] = ph[ti[k]];
            pj[k] = ph[tj[k]];
          }
#pragma unroll
          for (int k = 0; k < NP; ++k) S[r][k] += (pi[k / TS] * pj[k % TS]) * wq;
        } else {
          const double* g = &s_g[wv][q * B * D];
          const double kq = s_kq[wv][q];
          double gi[TS][D], gj[TS][D];
#pragma unroll
          for (int k = 0; k < TS; ++k)
#pragma unroll
            for (int d = 0; d < D; ++d) {
              gi[k][d] = g[ti[k] * D + d];
              gj[k][d] = g[tj[k] * D + d];
            }
#pragma unroll
          for (int k = 0; k < NP; ++k) {
            double dot = 0.0;
#pragma unroll
            for (int d = 0; d < D; ++d) dot += gi[k / TS][d] * gj[k % TS][d];
            S[r][k] += (kq * dot) * wq;
          }
        }
      }
    }
  }
  T* out = slot + e * (int64_t)n_pairs;
  if constexpr (kDirect) {
    if (active && lane < n_tiles) {
      const int i = s_tile[lane] >> 8, j = s_tile[lane] & 255;
      const T v = (T)S[0][0];
      if (!upper) {
        out[i * B + j] = v;
        out[j * B + i] = v;
      } else if (slot_dest) {
        slot[slot_dest[e * n_pairs + lane] & INT32_MAX] = v;
      } else {
        out[lane] = v;
      }
    }
    return;
  }
  tmh::wave_sync();
  double* const mat = s_g[wv];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int t = lane + r * L;
    if (active && t < n_tiles) {
      const int i0 = TS * (s_tile[t] >> 8), j0 = TS * (s_tile[t] & 255);
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        const int i = i0 + k / TS, j = j0 + k % TS;
        if (i < B && j < B) {
          mat[i * B + j] = S[r][k];
          mat[j * B + i] = S[r][k];
        }
      }
    }
  }
  tmh::wave_sync();
  if (!active) return;
  for (int p = lane; p < n_pairs; p += L) {
    const T v = (T)mat[upper ? (s_pair[p] >> 8) * B + (s_pair[p] & 255) : p];
    if (slot_dest)
      slot[slot_dest[e * n_pairs + p] & INT32_MAX] = v;
    else
      out[p] = v;
  }
}

// Neo-Hookean residual and consistent tangent, one wavefront per element.
// Replaces autograd of NeoHookeanModel.energy (builtin.py:301-333,
// element_assembler.py:631-657): psi = mu/2 (I1 - d) - mu ln J + lam/2 (ln J)^2
// with F = I + grad u, grad u[a][d] = sum_b u[n_b][a] dphi_b/dx_d.
//   P   = mu F + (lam ln J - mu) F^-T
//   R_i[a]       = sum_q jxw_q sum_A P_q[a][A] g_q,i[A]
//   K_ij[a][b]   = sum_q jxw_q ( mu delta_ab g_i.g_j + lam h_i[a] h_j[b] - c2 h_i[b] h_j[a] )
// with h_i = F^-T g_i  (h_i[a] = sum_A g_i[A] Finv[A][a]) and c2 = lam ln J - mu:
// the 9x9 tangent dP/dF = mu I + lam F^-T (x) F^-T - c2 (F^-1 swapped) contracted
// with the shape gradients on both sides.  At u = 0 it equals the linear
// elasticity block.  Tangent layout as the block forms: ((e*B+i)*B+j)*D*D + a*D + b;
// residual slots [e][i][a] summed into [N][D] by the node incidence reduction.
typedef float tm_floatx16 __attribute__((ext_vector_type(16)));

// MQ: largest number of quadrature points the LDS arrays hold.  Slot row
// (e, i) (B blocks of D x D values) goes to e*B + i, or with inc_inv to its
// position inc_inv[e*B + i] in the node-sorted incidence list.  In the VALU
// tangent a lane forms a whole D x D block; float64 blocks are stored through
// LDS (kViaLds), float32 ones from the lane (tmh::store_blocks).  The MFMA tile spreads a
// row over lanes, so that variant is staged in LDS and written as whole slot
// rows with vector stores.
// upper (TM_FLAG_UPPER): only the pairs i <= j.
// EPW elements per wavefront, each on L = 64 / EPW lanes: the VALU path packs
// two, so that the per-quadrature-point stages (Q active lanes) serve two
// elements at once (tetra10 f64 1.15 -> 1.07 ms per Newton assembly).
// BIG (tetra20, hexahedron27: element tangents of 60 x 60 and 81 x 81): one
// wavefront per workgroup and the rule tables read through the caches instead
// of LDS, so that a wave needs LDS only for its gradients (2 Q B D doubles).
template <typename T, int D, int B, bool MFMA, int MQ, bool BIG, int EPW, bool TAN>
__global__ void __launch_bounds__(kWave * (BIG ? 1 : kWavesPerBlock), TAN && !MFMA && MQ == 4 && EPW <= 2 ? 5 : 1)
    hyper_wave_kernel(const int32_t* __restrict__ conn, const T* __restrict__ pts, const T* __restrict__ disp,
                      const double* __restrict__ tab, int Q, double lam, double mu, int64_t n_elem, int upper,
                      T* __restrict__ tslot, T* __restrict__ rslot, const int32_t* __restrict__ inc_inv,
                      double* __restrict__ energy_e, const int32_t* __restrict__ slot_dest) {
  // TAN: the launch forms the tangent (ts == tslot); energy and residual
  // launches compile without the h arrays, the tangent stage and its
  // registers
  T* const ts = TAN ? tslot : nullptr;
  constexpr int kMaxQ = MQ;
  constexpr int kRowVals = B * D * D;  // values of one slot row
  constexpr int kWpb = BIG ? 1 : kWavesPerBlock;  // waves per workgroup
  static_assert(!(BIG && MFMA), "the MFMA tile holds at most 32 x 32");
  static_assert(EPW == 1 || !(MFMA || BIG), "the MFMA tile and BIG cells take a whole wavefront");
  constexpr int L = kWave / EPW;  // lanes per element
  constexpr int kEpb = kWpb * EPW;  // elements per workgroup
  constexpr bool kStage = MFMA;  // the MFMA tile spreads a row over lanes: staged row stores
  __shared__ double s_tab[BIG ? 1 : MQ * (1 + B + D * B)];
  // what the tangent's stores no longer need: each wave stages its blocks there
  struct Early {
    double x[B * D], u[B * D], inv[MQ][D * D], P[MQ][D * D], Fi[MQ][D * D];
  };
  // Float64 blocks are stored through LDS, except few per wavefront and the
  // large cells', whose lone wavefront waits for each of its rounds (assembly
  // of residual and tangent, us, through LDS / from the lanes: 36^3 x 6 tetra,
  // 4 points, 299 / 273; 12^3 x 6 tetra20, 24 points, 417 / 386; 18^3
  // hexahedra of 27 nodes, 27 points, 487 / 449)
  constexpr bool kViaLds = sizeof(T) == 8 && !BIG && B * (B + 1) > L;
  constexpr int kEarly = EPW * (int)sizeof(Early), kBlocks = TAN && !MFMA ? tmh::stage_bytes<T, D * D, kViaLds>() : 0;
  __shared__ __align__(16) char s_mem[kWpb][kEarly > kBlocks ? kEarly : kBlocks];
  __shared__ double s_jxw[kEpb][kMaxQ];
  __shared__ double s_g[kEpb][kMaxQ * B * D];
  __shared__ double s_h[kEpb][TAN ? kMaxQ * B * D : 1];
  __shared__ double s_c2[kEpb][kMaxQ];
  __shared__ double s_psi[kEpb][kMaxQ];   // psi * jxw per point (energy launches)
  __shared__ int s_v[kEpb][B];
  __shared__ T s_out[kEpb][kStage ? B * kRowVals : 1];
  __shared__ uint16_t s_pair[B * B];

  static_assert(B <= L && MQ <= L, "an element's lanes index its nodes and its quadrature points");
  const int lane = threadIdx.x % L;   // lane within the element's group
  const int wv = threadIdx.x / L;     // element slot within the workgroup
  char* const mem = s_mem[threadIdx.x / kWave];
  Early& el = reinterpret_cast<Early*>(mem)[wv % EPW];
  const int64_t e = (int64_t)blockIdx.x * kEpb + wv;
  const bool active = e < n_elem;
  const int tab_len = Q + Q * B + Q * D * B;
  if constexpr (!BIG)
    for (int t = threadIdx.x; t < tab_len; t += blockDim.x) s_tab[t] = tab[t];
  const int n_pairs = tmh::fill_pairs<B>(s_pair, upper != 0);
  const double* tb = BIG ? tab : s_tab;
  const double* w = tb;
  const double* dphi = tb + Q + Q * B;
  if (active && lane < B) s_v[wv][lane] = conn[e * B + lane];
  // the lane's first tangent block destination (contribution order), loaded
  // now so that its latency hides behind the per-point stages
  const int32_t dst = (!MFMA && slot_dest && ts && active && lane < n_pairs) ? slot_dest[e * n_pairs + lane] : 0;
  __syncthreads();
  if (active) {
    for (int t = lane; t < B * D; t += L) {
      const int b = t / D, d = t % D;
      el.x[t] = (double)pts[(int64_t)s_v[wv][b] * D + d];
      el.u[t] = (double)disp[(int64_t)s_v[wv][b] * D + d];
    }
  }
  tmh::wave_sync();
  // the Jacobians J[i][j] = sum_b dphi_b[i] x_b[j] (into el.inv, which
  // point q's lane then overwrites with the inverse)
  if (active)
    tmh::point_sums<D, B, L, MQ>(
        lane, Q, false, [&](int q, int i, int b) { return dphi[(q * D + i) * B + b]; },
        [&](int, int b, int j) { return el.x[b * D + j]; },
        [&](int q, int i, int j) -> double& { return el.inv[q][i * D + j]; });
  tmh::wave_sync();
  if (active && lane < Q) {
    const int q = lane;
    double J[D][D];
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
      for (int j = 0; j < D; ++j) J[i][j] = el.inv[q][i * D + j];
    double inv[D][D];
    double det;
    if constexpr (D == 2) {
      det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
      inv[0][0] = J[1][1] / det;
      inv[0][1] = -J[0][1] / det;
      inv[1][0] = -J[1][0] / det;
      inv[1][1] = J[0][0] / det;
    } else {
      const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
      const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
      const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
      det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
      const double r = 1.0 / det;
      inv[0][0] = c00 * r;
      inv[1][0] = c01 * r;
      inv[2][0] = c02 * r;
      inv[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * r;
      inv[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * r;
      inv[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * r;
      inv[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * r;
      inv[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * r;
      inv[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * r;
    }
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
      for (int j = 0; j < D; ++j) el.inv[q][i * D + j] = inv[i][j];
    s_jxw[wv][q] = w[q] * fabs(det);
  }
  tmh::wave_sync();
  if (active) {
    // a lane per (point, node): its D components share the reads of dphi
    for (int t = lane; t < Q * B; t += L) {
      const int q = t / B, b = t % B;
      double dp[D];
#pragma unroll
      for (int i = 0; i < D; ++i) dp[i] = dphi[(q * D + i) * B + b];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < D; ++i) s += dp[i] * el.inv[q][d * D + i];
        s_g[wv][t * D + d] = s;
      }
    }
  }
  tmh::wave_sync();
  // the deformation gradients F[a][d] = delta_ad + sum_b u_b[a] g_b[d] (into
  // el.Fi, which the per-point stage below overwrites with F^-1)
  if (active)
    tmh::point_sums<D, B, L, MQ>(
        lane, Q, true, [&](int, int a, int b) { return el.u[b * D + a]; },
        [&](int q, int b, int d) { return s_g[wv][(q * B + b) * D + d]; },
        [&](int q, int a, int d) -> double& { return el.Fi[q][a * D + d]; });
  tmh::wave_sync();
  if (active && lane < Q) {
    const int q = lane;
    double F[D][D];
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
      for (int d = 0; d < D; ++d) F[a][d] = el.Fi[q][a * D + d];
    double Fi[D][D];
    double Jd;
    if constexpr (D == 2) {
      Jd = F[0][0] * F[1][1] - F[0][1] * F[1][0];
      Fi[0][0] = F[1][1] / Jd;
      Fi[0][1] = -F[0][1] / Jd;
      Fi[1][0] = -F[1][0] / Jd;
      Fi[1][1] = F[0][0] / Jd;
    } else {
      const double c00 = F[1][1] * F[2][2] - F[1][2] * F[2][1];
      const double c01 = F[1][2] * F[2][0] - F[1][0] * F[2][2];
      const double c02 = F[1][0] * F[2][1] - F[1][1] * F[2][0];
      Jd = F[0][0] * c00 + F[0][1] * c01 + F[0][2] * c02;
      const double r = 1.0 / Jd;
      Fi[0][0] = c00 * r;
      Fi[1][0] = c01 * r;
      Fi[2][0] = c02 * r;
      Fi[0][1] = (F[0][2] * F[2][1] - F[0][1] * F[2][2]) * r;
      Fi[1][1] = (F[0][0] * F[2][2] - F[0][2] * F[2][0]) * r;
      Fi[2][1] = (F[0][1] * F[2][0] - F[0][0] * F[2][1]) * r;
      Fi[0][2] = (F[0][1] * F[1][2] - F[0][2] * F[1][1]) * r;
      Fi[1][2] = (F[0][2] * F[1][0] - F[0][0] * F[1][2]) * r;
      Fi[2][2] = (F[0][0] * F[1][1] - F[0][1] * F[1][0]) * r;
    }
    const double lj = log(Jd);
    const double c2 = lam * lj - mu;
    s_c2[wv][q] = c2;
    if (energy_e) {
      // psi = mu/2 (I1 - d) - mu ln J + lam/2 (ln J)^2, I1 = sum F_aA^2 (builtin.py:301-314)
      double I1 = 0.0;
#pragma unroll
      for (int a = 0; a < D; ++a)
#pragma unroll
        for (int A = 0; A < D; ++A) I1 += F[a][A] * F[a][A];
      s_psi[wv][q] = (0.5 * mu * (I1 - (double)D) - mu * lj + 0.5 * lam * lj * lj) * s_jxw[wv][q];
    }
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
      for (int A = 0; A < D; ++A) {
        el.P[q][a * D + A] = mu * F[a][A] + c2 * Fi[A][a];
        el.Fi[q][a * D + A] = Fi[a][A];
      }
  }
  tmh::wave_sync();
  if (energy_e && active && lane == 0) {
    // the element's energy, its points summed in order
    double s = 0.0;
    for (int q = 0; q < Q; ++q) s += s_psi[wv][q];
    energy_e[e] = s;
  }
  if (active && ts) {
    // h = F^-T g, read by the tangent only
    for (int t = lane; t < Q * B * D; t += L) {
      const int q = t / (B * D), b = (t / D) % B, a = t % D;
      const double* g = &s_g[wv][(q * B + b) * D];
      double s = 0.0;
#pragma unroll
      for (int A = 0; A < D; ++A) s += g[A] * el.Fi[q][A * D + a];
      s_h[wv][t] = s;
    }
  }
  tmh::wave_sync();
  if (rslot && active) {
    // one component per lane, and without a tangent, where LDS reads are most
    // of the kernel, a node per lane, whose components share g (82,944 tetra10,
    // energy + residual, float64: 50.8 -> 45.3 us with the gradients' part; with a
    // tangent 402 -> 408 us: too few lanes)
    constexpr int V = TAN ? 1 : D;
    for (int t = lane; t < B * D / V; t += L) {
      const int i = t * V / D, a0 = t * V % D;
      double acc[V];
#pragma unroll
      for (int v = 0; v < V; ++v) acc[v] = 0.0;
      for (int q = 0; q < Q; ++q) {
        double g[D];
#pragma unroll
        for (int A = 0; A < D; ++A) g[A] = s_g[wv][(q * B + i) * D + A];
        const double wq = s_jxw[wv][q];
#pragma unroll
        for (int v = 0; v < V; ++v) {
          double s = 0.0;
#pragma unroll
          for (int A = 0; A < D; ++A) s += el.P[q][(a0 + v) * D + A] * g[A];
          acc[v] += s * wq;
        }
      }
      // element order: row (e, i) at e*B + i; incidence order: at inc_inv[e*B + i]
      const int64_t row = inc_inv ? (int64_t)inc_inv[e * B + i] : e * B + i;
#pragma unroll
      for (int v = 0; v < V; ++v) rslot[row * D + a0 + v] = (T)acc[v];
    }
  }
  if constexpr (MFMA) {
    // K_e = sum_q L_q^T R_q as one 32 x 32 tile (rows (i, a), columns (j, b),
    // B*D <= 32) with inner index (q, c, A), two per v_mfma_f32_32x32x2f32:
    //   L^T[(i,a)][(q,c,A)] = delta_ac g_q,i[A]
    //   R[(q,c,A)][(j,b)]   = jxw_q (mu delta_cb g_q,j[A] + lam Finv[A][c] h_j[b] - c2 Finv[A][b] h_j[c])
    // Lane l supplies A[m = l%32][k = l/32] and B[k = l/32][n = l%32]; the
    // accumulator register r of lane l holds row (r/4)*8 + (l/32)*4 + r%4,
    // column l%32.
    if (ts) {
      constexpr int DD = D * D;
      constexpr int M = B * D;
      static_assert(M <= 32, "tile holds at most 32 rows");
      const int m = lane % 32, kh = lane / 32;
      const int i = m / D, a = m % D;
      const int j = m / D, b = m % D;  // n == m for the B operand column
      tm_floatx16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
      const int steps = (Q * DD) / 2;
      for (int st = 0; st < steps; ++st) {
        const int kk = 2 * st + kh;
        const int q = kk / DD, c = (kk % DD) / D, A = kk % D;
        float av = 0.0f, bv = 0.0f;
        if (m < M) {
          const double* g = &s_g[wv][q * B * D];
          const double* h = &s_h[wv][q * B * D];
          const double* Fi = el.Fi[q];
          if (a == c) av = (float)g[i * D + A];
          double v = lam * Fi[A * D + c] * h[j * D + b] - s_c2[wv][q] * Fi[A * D + b] * h[j * D + c];
          if (c == b) v += mu * g[j * D + A];
          bv = (float)(v * s_jxw[wv][q]);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc, 0, 0, 0);
      }
      const int n = m;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = (r / 4) * 8 + kh * 4 + (r % 4);
        if (row < M && n < M && active) {
          const int ii = row / D, aa = row % D, jj = n / D, bb = n % D;
          s_out[wv][(ii * B + jj) * DD + aa * D + bb] = (T)acc[r];
        }
      }
    }
  } else if (ts) {
    // one lane per node pair (i, j): the whole D x D block from one read of
    // g_i, g_j, h_i, h_j per quadrature point
    constexpr int DD = D * D;
    int32_t d_next = dst;
#pragma unroll 1
    for (int p0 = 0; p0 < n_pairs; p0 += L) {
      const int p = p0 + lane;
      const int32_t d = d_next;
      if (p + L < n_pairs && slot_dest && active) d_next = slot_dest[e * n_pairs + p + L];
      int32_t at = -1;
      double acc[DD];
#pragma unroll
      for (int k = 0; k < DD; ++k) acc[k] = 0.0;
      if (active && p < n_pairs) {
        int i = s_pair[p] >> 8, j = s_pair[p] & 255;
        // element order: block p of the element's pairs (packed when upper);
        // incidence order (full blocks only): slot row inc_inv[e*B + i];
        // contribution order (upper): slot slot_dest[e*P + p], transposed
        // when its id is negative -- formed as block (j, i), which is the
        // exact transpose of (i, j) (the same products, commuted)
        if (slot_dest) {
          at = d & INT32_MAX;
          if (d < 0) {
            const int t = i;
            i = j;
            j = t;
          }
        } else {
          at = inc_inv ? inc_inv[e * B + i] * B + j : (int32_t)(e * n_pairs + p);
        }
        for (int q = 0; q < Q; ++q) {
          const double* gi = &s_g[wv][(q * B + i) * D];
          const double* gj = &s_g[wv][(q * B + j) * D];
          const double* hi = &s_h[wv][(q * B + i) * D];
          const double* hj = &s_h[wv][(q * B + j) * D];
          double vgi[D], vgj[D], vhi[D], vhj[D];
#pragma unroll
          for (int d = 0; d < D; ++d) {
            vgi[d] = gi[d];
            vgj[d] = gj[d];
            vhi[d] = hi[d];
            vhj[d] = hj[d];
          }
          const double w = s_jxw[wv][q];
          const double lw = lam * w, cw = s_c2[wv][q] * w;
          double dot = 0.0;
#pragma unroll
          for (int d = 0; d < D; ++d) dot += vgi[d] * vgj[d];
          const double mw = mu * dot * w;
#pragma unroll
          for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) {
              double t = lw * (vhi[a] * vhj[b]) - cw * (vhi[b] * vhj[a]);
              if (a == b) t += mw;
              acc[a * D + b] += t;
            }
        }
      }
      tmh::store_blocks<T, DD, kViaLds>(mem, acc, at, false, ts);
    }
  }
  if constexpr (kStage) {
    tmh::wave_sync();
    if (ts && active) {
      // whole slot rows with vector stores: 16 bytes when a row's size allows,
      // else 8 (slot buffers are 256-byte aligned)
      constexpr int kRowBytes = kRowVals * (int)sizeof(T);
      constexpr int kVec = kRowBytes % 16 == 0 ? 16 : 8;
      static_assert(kRowBytes % kVec == 0, "slot rows are whole vectors");
      constexpr int kPerRow = kRowBytes / kVec;
      typedef int32_t vec_t __attribute__((ext_vector_type(kVec / 4)));
      for (int v = lane; v < B * kPerRow; v += L) {
        const int i = v / kPerRow, o = v % kPerRow;
        const int64_t srow = inc_inv ? (int64_t)inc_inv[e * B + i] : e * B + i;
        const vec_t x = reinterpret_cast<const vec_t*>(&s_out[wv][i * kRowVals])[o];
        reinterpret_cast<vec_t*>(ts + srow * kRowVals)[o] = x;
      }
    }
  }
}

template <typename T, int D, int B>
int launch_hyper(const tm_mesh_view* m, const tm_form_desc* f, const void* disp, void* tslot, void* rslot,
                 const int32_t* inc_inv, double* energy_e, const int32_t* slot_dest, hipStream_t stream) {
  // more than 32 element dofs (tetra20: 60, hexahedron27: 81), or a rule of
  // more than 16 points (the 24-point tetrahedron rule): one element per
  // workgroup, the BIG variant, with rules of up to 32 points
  constexpr bool kBigCell = B * D > 32;
  const int Q = f->n_quad;
  const bool big = kBigCell || Q > kMaxQ;
  const int wpb = big ? 1 : kWavesPerBlock;
  if (Q <= 0 || Q > kMaxQWave) return tmh::fail(TM_ERR_UNSUPPORTED, "quadrature rule has too many points");
  if (!f->tab_dev) return tmh::fail(TM_ERR_ARG, "device form tables missing");
  const double mu = f->young / (2.0 * (1.0 + f->poisson));
  const double lam = f->young * f->poisson / ((1.0 + f->poisson) * (1.0 - 2.0 * f->poisson));
  const bool mfma = (f->flags & TM_FLAG_MFMA) != 0;
  if (mfma && !(std::is_same<T, float>::value && B * D <= 32))
    return tmh::fail(TM_ERR_UNSUPPORTED, "the MFMA tangent path is float32 only");
  if (mfma && Q > kMaxQ) return tmh::fail(TM_ERR_UNSUPPORTED, "the MFMA tangent path takes rules of <= 16 points");
  if (mfma && (Q * D * D) % 2 != 0) return tmh::fail(TM_ERR_UNSUPPORTED, "MFMA path needs an even Q*D*D");
  // two elements per wavefront (32 lanes each) on the VALU path by default:
  // the per-quadrature-point stages, which use Q lanes, then serve two
  // elements; four (16 lanes each) without a tangent, whose pair loop wants
  // no lanes (tetra10 energy + residual 185 -> 146 us per call, f64); form->epw
  // asks for 1, 2 or 4 (4: 16 lanes, rules of <= 4 points)
  int epw = (mfma || big) ? 1 : (!tslot && Q <= 4 && B <= 16) ? 4 : 2;
  if (f->epw != 0) {
    const bool ok = f->epw == 1 || (!mfma && !big && (f->epw == 2 || (f->epw == 4 && Q <= 4 && B <= 16)));
    if (!ok) return tmh::fail(TM_ERR_ARG, "elements per wavefront not admitted for this cell / rule / tangent");
    epw = f->epw;
  }
  const int64_t per_block = (int64_t)wpb * epw;
  const int64_t grid = (m->n_elem + per_block - 1) / per_block;
  if (grid == 0) return TM_OK;
  const dim3 g((unsigned)grid), blk(kWave * wpb);
  const int upper = (f->flags & TM_FLAG_UPPER) != 0;
  if (upper && (mfma || inc_inv))
    return tmh::fail(TM_ERR_ARG, "TM_FLAG_UPPER needs the element-ordered VALU tangent (no MFMA, no block rows)");
#define TM_HYPER_T(MF, MQ, BG, EPW, TAN)                                                            \
  hyper_wave_kernel<T, D, B, MF, MQ, BG, EPW, TAN><<<g, blk, 0, stream>>>(                          \
      m->conn, (const T*)m->points, (const T*)disp, f->tab_dev, Q, lam, mu, m->n_elem, upper,     \
      (T*)tslot, (T*)rslot, inc_inv, energy_e, upper ? slot_dest : nullptr)
#define TM_HYPER_V(MF, MQ, BG, EPW) TM_HYPER_T(MF, MQ, BG, EPW, true)
  // the VALU instances come without the tangent machinery for energy and
  // residual launches (fewer registers and LDS: more waves per SIMD)
#define TM_HYPER(MF, MQ, EPW)                                \
  do {                                                       \
    if constexpr (MF) TM_HYPER_T(MF, MQ, false, EPW, true);  \
    else if (tslot) TM_HYPER_T(MF, MQ, false, EPW, true);    \
    else TM_HYPER_T(MF, MQ, false, EPW, false);              \
  } while (0)
  if constexpr (kBigCell) {
    if (Q <= 16) TM_HYPER_V(false, 16, true, 1); else TM_HYPER_V(false, 32, true, 1);
  } else if (big) {
    TM_HYPER_V(false, 32, true, 1);
  } else if (mfma) {
    if constexpr (std::is_same<T, float>::value) {  // float64 was rejected above
      if (Q <= 4) TM_HYPER(true, 4, 1); else TM_HYPER(true, 16, 1);
    }
  } else if (Q <= 4) {
    if (epw == 1) TM_HYPER(false, 4, 1);
    else if (epw == 2) TM_HYPER(false, 4, 2);
    else if constexpr (B <= 16) TM_HYPER(false, 4, 4);
  } else if (Q <= 8) {
    if (epw == 1) TM_HYPER(false, 8, 1); else TM_HYPER(false, 8, 2);
  } else {
    if (epw == 1) TM_HYPER(false, 16, 1); else TM_HYPER(false, 16, 2);
  }
#undef TM_HYPER
#undef TM_HYPER_V
#undef TM_HYPER_T
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    tmh::set_error("neo-hookean kernel launch: %s", hipGetErrorString(err));
    return TM_ERR_HIP;
  }
  return TM_OK;
}

template <typename T>
int dispatch_hyper(const tm_mesh_view* m, const tm_form_desc* f, const void* disp, void* tslot, void* rslot,
                   const int32_t* inc_inv, double* energy_e, hipStream_t s, const int32_t* slot_dest = nullptr) {
  switch (m->cell) {
#define TM_CASE(C, D, B) \
  case C: return launch_hyper<T, D, B>(m, f, disp, tslot, rslot, inc_inv, energy_e, slot_dest, s);
    TM_ALL_CELLS(TM_CASE)
#undef TM_CASE
    default: return tmh::fail(TM_ERR_ARG, "unknown cell");
  }
}

template <typename T, int D, int B, int MQ>
int launch_wave(const tm_mesh_view* m, const tm_form_desc* f, void* slot_ws, hipStream_t stream, int* hh_out,
                const int32_t* slot_dest) {
  const int Q = f->n_quad;
  const T* pts = static_cast<const T*>(m->points);
  const T* coeff = static_cast<const T*>(f->coeff);
  T* slot = static_cast<T*>(slot_ws);
  // By default as many elements per wavefront as have a lane for every tile
  // of the upper triangle (at most 16), where a wavefront's arrays fit 20 KB,
  // in workgroups of two wavefronts where four would take more than 40 KB;
  // else two where their gradients fit 40 KB, else one.  form->epw: 1, two where
  // that holds, or the default (0)
  constexpr int kElemBytes = 8 * (B * D + MQ * (D * D + 2) + B * (MQ * D > B ? MQ * D : B)) + 4 * B;
  // without a scalar form's matrix, which only the 27 nodes of a one-point rule
  // outgrow the gradients by (59 KB of LDS for a workgroup of two elements)
  constexpr int kGradBytes = 8 * (B * D + MQ * (D * D + 2 + B * D)) + 4 * B;
  constexpr int kTwo = (2 * kWavesPerBlock * kGradBytes <= 40960 && MQ <= kWave / 2 && B <= kWave / 2) ? 2 : 1;
  constexpr int NT = (B + 1) / 2, kTiles = NT * (NT + 1) / 2;
  constexpr int kMost = kTiles >= kWave ? 1 : kWave / kTiles < 16 ? kWave / kTiles : 16;
  constexpr int kMany = kMost * kElemBytes <= 20480 ? kMost : kTwo;
  const int upper = (f->flags & TM_FLAG_UPPER) != 0;
  // Whole blocks of the cells of 8 to 10 nodes: consecutive lanes on single
  // pairs write consecutive blocks (element kernel and reduction, kMany / two:
  // 18^3 x 6 tetra10 float32 109 / 90 us, hexahedra 40^3 119 / 97, float64
  // 178 / 174 and 225 / 214).  Smaller cells lose by it (tetra 128 / 152).
  constexpr int kWhole = B >= 8 && kMany > kTwo ? kTwo : kMany;
  const int epw = f->epw != 0 ? f->epw : f->form == TM_FORM_LINEAR_ELASTICITY && !upper ? kWhole : kMany;
  if (epw != 1 && epw != kTwo && epw != kMany)
    return tmh::fail(TM_ERR_ARG, "elements per wavefront not admitted for this cell / rule");
  *hh_out = 1;
  double lam = 0.0, mu = 0.0;
#define TM_WAVE_E(H, FORM, EPW)                                                                                    \
  do {                                                                                                            \
    constexpr int kWpb = EPW * kWavesPerBlock * kElemBytes <= 40960 || EPW <= 2 ? kWavesPerBlock : 2;              \
    const int64_t grid = (m->n_elem + kWpb * EPW - 1) / (kWpb * EPW);                                             \
    if (grid == 0) return TM_OK;                                                                                  \
    wave_element_kernel<T, D, B, H, FORM, MQ, EPW, kWpb><<<grid, kWave * kWpb, 0, stream>>>(                       \
        m->conn, pts, coeff, f->tab_dev, Q, lam, mu, m->n_elem, upper, slot, upper ? slot_dest : nullptr);       \
  } while (0)
#define TM_WAVE(H, FORM)                                \
  do {                                                  \
    if (epw == kMany) TM_WAVE_E(H, FORM, kMany);        \
    else if (epw == kTwo) TM_WAVE_E(H, FORM, kTwo);     \
    else TM_WAVE_E(H, FORM, 1);                         \
  } while (0)
  switch (f->form) {
    case TM_FORM_LAPLACE:
      TM_WAVE(1, TM_FORM_LAPLACE);
      break;
    case TM_FORM_DIFFUSION_ELEM:
      if (!coeff) return tmh::fail(TM_ERR_ARG, "diffusion form needs a coefficient");
      TM_WAVE(1, TM_FORM_DIFFUSION_ELEM);
      break;
    case TM_FORM_DIFFUSION_NODE:
      if (!coeff) return tmh::fail(TM_ERR_ARG, "diffusion form needs a coefficient");
      TM_WAVE(1, TM_FORM_DIFFUSION_NODE);
      break;
    case TM_FORM_MASS:
      TM_WAVE(1, TM_FORM_MASS);
      break;
    case TM_FORM_LINEAR_ELASTICITY:
      mu = f->young / (2.0 * (1.0 + f->poisson));
      lam = f->young * f->poisson / ((1.0 + f->poisson) * (1.0 - 2.0 * f->poisson));
      *hh_out = D * D;
      TM_WAVE(D, TM_FORM_LINEAR_ELASTICITY);
      break;
    default:
      return tmh::fail(TM_ERR_UNSUPPORTED, "unknown form");
  }
#undef TM_WAVE
#undef TM_WAVE_E
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    tmh::set_error("element kernel launch: %s", hipGetErrorString(err));
    return TM_ERR_HIP;
  }
  return TM_OK;
}

template <typename T, int D, int B>
int launch_scalar_or_block(const tm_mesh_view* m, const tm_form_desc* f, void* slot_ws, hipStream_t stream,
                           int* hh_out, const int32_t* sd) {
  const int Q = f->n_quad;
  if (Q <= 0 || Q > kMaxQWave) return tmh::fail(TM_ERR_UNSUPPORTED, "quadrature rule has too many points");
  if (!f->tab_dev) return tmh::fail(TM_ERR_ARG, "device form tables missing");
  if (Q <= 4) return launch_wave<T, D, B, 4>(m, f, slot_ws, stream, hh_out, sd);
  if (Q <= 8) return launch_wave<T, D, B, 8>(m, f, slot_ws, stream, hh_out, sd);
  if (Q <= 16) return launch_wave<T, D, B, 16>(m, f, slot_ws, stream, hh_out, sd);
  return launch_wave<T, D, B, kMaxQWave>(m, f, slot_ws, stream, hh_out, sd);
}

template <typename T>
int dispatch_cell(const tm_mesh_view* m, const tm_form_desc* f, void* slot_ws, hipStream_t stream, int* hh,
                  const int32_t* sd) {
  switch (m->cell) {
#define TM_CASE(C, D, B) \
  case C: return launch_scalar_or_block<T, D, B>(m, f, slot_ws, stream, hh, sd);
    TM_ALL_CELLS(TM_CASE)
#undef TM_CASE
    default: return tmh::fail(TM_ERR_ARG, "unknown cell");
  }
}

}  // namespace

int tm_hyper_element_rows(const tm_mesh_view* mesh, const tm_form_desc* form, const void* disp, void* tslot,
                          void* rslot, const int32_t* inc_inv, hipStream_t stream) {
  return mesh->dtype == TM_F64 ? dispatch_hyper<double>(mesh, form, disp, tslot, rslot, inc_inv, nullptr, stream)
                               : dispatch_hyper<float>(mesh, form, disp, tslot, rslot, inc_inv, nullptr, stream);
}

int tm_p2_element_matrices(const tm_mesh_view* mesh, const tm_form_desc* form, void* slot_ws,
                           hipStream_t stream, int* hh_out, const int32_t* slot_dest) {
  if (mesh->dtype == TM_F64) return dispatch_cell<double>(mesh, form, slot_ws, stream, hh_out, slot_dest);
  return dispatch_cell<float>(mesh, form, slot_ws, stream, hh_out, slot_dest);
}

extern "C" int tm_assemble_neohookean(const tm_mesh_view* mesh, const tm_form_desc* form, const void* disp,
                                      const tm_pattern_view* pat, const tm_incidence_view* inc, void* tslot_ws,
                                      void* tangent, void* rslot_ws, void* residual, tm_stream_t stream_) {
  TM_TRY_BEGIN
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (!mesh || !form || !disp) return tmh::fail(TM_ERR_ARG, "NULL argument");
  if (tmh::cell_basis(mesh->cell) < 0) return tmh::fail(TM_ERR_ARG, "unknown cell");
  const int64_t B = tmh::cell_basis(mesh->cell), D = tmh::cell_dim(mesh->cell);
  if (mesh->n_elem * B * B >= tmh::kMaxIndex) return tmh::fail(TM_ERR_SIZE, "mesh too large");
  if (tangent && (!pat || !tslot_ws)) return tmh::fail(TM_ERR_ARG, "tangent needs a pattern and a slot workspace");
  if (residual && (!inc || !rslot_ws)) return tmh::fail(TM_ERR_ARG, "residual needs incidence and a workspace");
  void* ts = tangent ? tslot_ws : nullptr;
  void* rs = residual ? rslot_ws : nullptr;
  if (tangent && pat->slot_dest && !(form->flags & TM_FLAG_UPPER))
    return tmh::fail(TM_ERR_ARG, "slot_dest needs TM_FLAG_UPPER (symmetric element blocks)");
  const int32_t* sd = tangent ? pat->slot_dest : nullptr;
  int st = mesh->dtype == TM_F64 ? dispatch_hyper<double>(mesh, form, disp, ts, rs, nullptr, nullptr, stream, sd)
                                 : dispatch_hyper<float>(mesh, form, disp, ts, rs, nullptr, nullptr, stream, sd);
  if (st) return st;
  // the residual reduction first: part of its slots (tens of MB) still sits in
  // the caches after the element kernel, and would not after the tangent
  // reduction has streamed the much larger tangent slots (measured faster)
  if (residual) {
    st = tm_segmented_reduce(mesh->dtype, mesh->n_points, (int32_t)D, inc->inc_ptr, inc->inc, inc->n_blocks,
                             inc->blk_ptr, rslot_ws, residual, stream_);
    if (st) return st;
  }
  if (tangent) {
    st = tmh::reduce_view(mesh->dtype, pat, (int32_t)(D * D), tslot_ws, tangent, stream_);
    if (st) return st;
  }
  return TM_OK;
  TM_TRY_END
}

extern "C" int tm_neohookean_energy(const tm_mesh_view* mesh, const tm_form_desc* form, const void* disp,
                                    void* energy_ws, void* energy, const tm_incidence_view* inc, void* rslot_ws,
                                    void* residual, tm_stream_t stream_) {
  TM_TRY_BEGIN
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (!mesh || !form || !disp || !energy || !energy_ws) return tmh::fail(TM_ERR_ARG, "NULL argument");
  if (mesh->dtype != TM_F64 && mesh->dtype != TM_F32) return tmh::fail(TM_ERR_ARG, "unknown dtype");
  const int64_t B = tmh::cell_basis(mesh->cell), D = tmh::cell_dim(mesh->cell);
  if (B < 0) return tmh::fail(TM_ERR_ARG, "unknown cell");
  if (mesh->n_elem < 0 || mesh->n_elem * B * D >= tmh::kMaxIndex) return tmh::fail(TM_ERR_SIZE, "mesh too large");
  if (mesh->n_elem > 0 && (!mesh->conn || !mesh->points)) return tmh::fail(TM_ERR_ARG, "NULL buffer");
  if (residual && (!inc || !rslot_ws)) return tmh::fail(TM_ERR_ARG, "residual needs incidence and a workspace");
  // energy launches form no tangent: the tangent flags do not apply
  tm_form_desc f = *form;
  f.flags = 0;
  double* e_out = static_cast<double*>(energy_ws);
  void* rs = residual ? rslot_ws : nullptr;
  int st = mesh->dtype == TM_F64 ? dispatch_hyper<double>(mesh, &f, disp, nullptr, rs, nullptr, e_out, stream)
                                 : dispatch_hyper<float>(mesh, &f, disp, nullptr, rs, nullptr, e_out, stream);
  if (st) return st;
  st = tmh::sum_fixed(e_out, mesh->n_elem, e_out + mesh->n_elem, mesh->dtype, energy, stream_);
  if (st) return st;
  if (residual) {
    st = tm_segmented_reduce(mesh->dtype, mesh->n_points, (int32_t)D, inc->inc_ptr, inc->inc, inc->n_blocks,
                             inc->blk_ptr, rslot_ws, residual, stream_);
    if (st) return st;
  }
  return TM_OK;
  TM_TRY_END
}
