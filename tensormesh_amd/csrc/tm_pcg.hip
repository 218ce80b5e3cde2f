// Whole solves of the two-launch Jacobi-PCG (tm_solve.hip) in one launch.
//
// The recurrences, every rounding and the order of every sum are those of
// cg2_vec_kernel / cg2_spmv_kernel, so the iterates, the iteration counts and
// the solution are bit for bit the same (behavioural reference:
// tensormesh/sparse/solve/torch_solve.py:54-128).  What changes is where the
// state lives.  The two launches of a step re-read the matrix and seven
// vectors (25-29 MB each at 261,121 rows) and pay dispatch and drain twice.
// Here a workgroup of 1,024 threads keeps its rows' matrix entries, x, r, p, s,
// w and the inverse diagonal in registers (the entries past the first few in
// LDS) for the whole solve; a step moves only u = M r and three partial sums
// per 256 rows between workgroups, and is bound by the latency of those two
// exchanges through memory (about 1.3 us each between XCDs), not by bytes.
// Measured per step, float64, two launches -> here: 261,121 rows of a triangle
// mesh (256 workgroups) 16.9 -> 5.0 us, 89,401 rows 12.4 -> 4.3 us, 516,961 rows
// (two rows per thread) 29.3 -> 8.0 us, 205,379 rows of a tetrahedral mesh
// 23.6 -> 8.0 us, 361 rows (SOLO) 11.0 -> 1.2 us; 256 uneven systems of
// 1.7 M rows together 43 -> 12.5 ms per solve.
//
// A system inside one workgroup (SOLO) exchanges both through LDS with two
// barriers per step.  A system over several workgroups exchanges them through
// device memory without flags or grid barriers: every word is its own flag.
// A word is reset to a bit pattern that no published value has (a NaN no
// arithmetic produces; a computed NaN of that pattern is published as the
// default NaN) and readers poll until it changes.  Three buffers rotate: step
// k publishes in buffer k mod 3 and resets buffer (k + 1) mod 3, last read in
// step k - 2; a workgroup publishes its sums of step k only after its reset
// has reached memory, and nobody reads buffer (k + 1) before it has
// everybody's sums of step k.  The accesses are relaxed at agent scope: on this
// chip they go past the caches of one XCD, and a store counted off by
// s_waitcnt vmcnt has reached the memory that all XCDs read.  That property,
// not the language's memory model, orders the reset before the sums; a release
// store would order it too, but writes the whole L2 back (10 of the 21.6 us
// that a step then took).  u of other workgroups' rows (the halo) is
// read once per workgroup into LDS: gathered from memory per matrix entry it
// took 11.8 us.  Every workgroup adds its system's partial sums itself, in
// workgroup order, so all of them take the same decisions without a broadcast
// (one workgroup per sum and a second exchange: 6.3 us).
//
// The workgroups of a launch that exchange through memory are co-resident by
// a cooperative launch, and every wait is bounded: after kGiveUpTicks a
// workgroup raises the abort word and leaves, as do all that see it or time
// out themselves; the caller then solves with the two-launch kernels.  So does
// a workgroup that cannot hold what it was given: too many halo columns, a row
// of more entries than the instance's, a column of another system.
#include <hip/hip_runtime.h>

#include "tm_device.h"
#include "tm_internal.h"

// no implicit contraction: the same rounding steps as tm_solve.hip
#pragma clang fp contract(off)

namespace {

constexpr int kBlock = 256;                    // rows per partial sum (workgroup size of tm_solve.hip)
constexpr int kGroups = 4;                     // blocks a workgroup works on at a time
constexpr int kThreads = kGroups * kBlock;
constexpr int kHalo = 4096;                    // columns of other workgroups that a workgroup may read
constexpr int kTable = 2 * kHalo;              // hash table that numbers them
constexpr int kPoll = 4;                       // partial sums a thread reads at once
constexpr int kNS2 = 16;                       // scalars per system (tm_solve.hip)
constexpr uint64_t kGiveUpTicks = 200000000;   // 2 s of the 100 MHz counter

template <typename T>
struct Word;
template <>
struct Word<double> {
  typedef uint64_t type;
  static constexpr uint64_t kEmpty = ~0ull, kNan = 0x7ff8000000000000ull;
};
template <>
struct Word<float> {
  typedef uint32_t type;
  static constexpr uint32_t kEmpty = ~0u, kNan = 0x7fc00000u;
};

template <typename T>
__device__ __forceinline__ typename Word<T>::type to_word(T v) {
  const auto w = __builtin_bit_cast(typename Word<T>::type, v);
  return w == Word<T>::kEmpty ? Word<T>::kNan : w;
}

template <typename W>
__device__ __forceinline__ W peek(const W* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename W>
__device__ __forceinline__ void post(W* p, W v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// peek at a 32-bit byte offset from a uniform base (one address register)
template <typename W>
__device__ __forceinline__ W peek_at(const W* base, uint32_t off) {
  return peek(reinterpret_cast<const W*>(reinterpret_cast<const char*>(base) + off));
}

struct RunArgs {
  const int32_t *wg_sys, *wg_blk0, *sys_blk, *blk_row0, *blk_row1, *rp, *ci;
  const void *av, *dinv, *r, *w;
  void* x;
  const double* part;   // gamma (2 slots), |r|^2, delta, |b|^2 as tm_pcg_init leaves them
  double* sc;
  int32_t nb, parity, n_iter;
  double tol2;
  void* ubuf;           // [3][n_rows] words of u
  uint64_t* pbuf;       // [3][nb][4] words: each block's gamma, |r|^2, delta (one unused)
  int32_t* abort;
  int64_t n_rows;
};

__device__ __forceinline__ uint32_t hash(int32_t col) { return ((uint32_t)col * 2654435769u) >> 19; }
static_assert(kTable == 1 << 13, "hash() gives 13 bits");

// Spins of one wait: true while the wait may go on.
struct Patience {
  uint64_t t0 = 0;
  uint32_t n = 0;
  __device__ __forceinline__ bool more(int32_t* abort) {
    if ((++n & 63u) != 0) return true;
    const uint64_t t = wall_clock64();
    if (t0 == 0) t0 = t;
    if (t - t0 > kGiveUpTicks) {
      post(abort, 1);
      return false;
    }
    return peek(abort) == 0;
  }
};

// Matrix values a thread holds in registers: what fits beside its vectors in
// the 128 registers of a 1,024-thread workgroup; the others lie in LDS.
template <typename T, int K, int PER>
constexpr int reg_values() {
  const int most = sizeof(T) == 4 ? 16 : PER == 24 ? 12 : 8;
  return K * PER < most ? K * PER : most;
}

// K rows per thread, rows of at most PER entries.
template <typename T, int K, int PER, bool SOLO>
__global__ void __launch_bounds__(kThreads) cg2_run_kernel(RunArgs a) {
  typedef typename Word<T>::type W;
  constexpr int kOwn = kThreads * K;
  __shared__ T s_u[SOLO ? 2 * kOwn : kOwn + kHalo];           // u of the own rows, then of the halo
  __shared__ double s_wave[SOLO ? 2 : 1][3][kGroups * K][4];  // wave sums of gamma, |r|^2, delta
  __shared__ double s_red[3][4];
  // matrix values past the first kReg of a thread; before them, the tables
  // that number the halo
  constexpr int kReg = reg_values<T, K, PER>(), kLds = K * PER - kReg;
  constexpr int kTables = SOLO ? 0 : 4 * kTable + 4 * kHalo + 2 * kTable, kVals = kLds * kThreads * (int)sizeof(T);
  __shared__ __align__(16) char s_mem[kTables > kVals ? kTables : kVals > 0 ? kVals : 16];
  int32_t* const s_key = reinterpret_cast<int32_t*>(s_mem);
  int32_t* const s_hcol = s_key + kTable;
  uint16_t* const s_hidx = reinterpret_cast<uint16_t*>(s_hcol + kHalo);
  T* const s_val = reinterpret_cast<T*>(s_mem);
  __shared__ int s_abort, s_halo;
  const int tid = threadIdx.x, lane = tid & 63, grp = tid / kBlock, gw = (tid / 64) & 3, gt = tid & (kBlock - 1);
  const int sy = a.wg_sys[blockIdx.x];
  const int32_t b0 = a.sys_blk[sy], b1 = a.sys_blk[sy + 1], wb0 = a.wg_blk0[blockIdx.x];
  double* const c = a.sc + (int64_t)sy * kNS2;
  if (c[6] == 0.0) return;  // stopped at its initial residual; cleared later only after every workgroup took part
  if (tid == 0) s_abort = s_halo = 0;
  const int32_t own = a.blk_row0[wb0];  // the workgroup's rows are consecutive
  const int32_t sys_row0 = a.blk_row0[b0], sys_rows = a.blk_row1[b1 - 1] - sys_row0;

  T av[kReg], x[K], r[K], p[K], s[K], w[K], d[K], u[K];
  int32_t row[K], ra[K], len[K];  // row -1: none
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int32_t blk = wb0 + k * kGroups + grp;
    row[k] = -1;
    ra[k] = len[k] = 0;
    x[k] = r[k] = p[k] = s[k] = w[k] = d[k] = T(0);
    if (blk < b1) {
      const int32_t i = a.blk_row0[blk] + gt;
      if (i < a.blk_row1[blk]) {
        row[k] = i;
        ra[k] = a.rp[i];
        len[k] = a.rp[i + 1] - ra[k];
        x[k] = ((const T*)a.x)[i];
        r[k] = ((const T*)a.r)[i];
        w[k] = ((const T*)a.w)[i];
        d[k] = ((const T*)a.dinv)[i];
      }
    }
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (k * PER + j < kReg) av[k * PER + j] = j < len[k] ? ((const T*)a.av)[ra[k] + j] : T(0);
    u[k] = d[k] * r[k];
  }
  if constexpr (!SOLO) {
    // the halo: every column outside the own rows, numbered once (in no
    // particular order) through a hash table
    for (int i = tid; i < kTable; i += kThreads) s_key[i] = -1;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k)
      for (int j = 0; j < len[k]; ++j) {
        const int32_t col = a.ci[ra[k] + j];
        if ((uint32_t)(col - own) < (uint32_t)kOwn || *(volatile int*)&s_halo > kHalo) continue;
        for (uint32_t h = hash(col);; h = (h + 1) % kTable) {
          const int32_t old = atomicCAS(&s_key[h], -1, col);
          if (old == col) break;
          if (old == -1) {
            const int n = atomicAdd(&s_halo, 1);
            if (n < kHalo) {
              s_hcol[n] = col;
              s_hidx[h] = (uint16_t)n;
            }
            break;
          }
        }
      }
  }
  // gamma and delta of the initial state, summed over the system's workgroups
  if (grp == 0) {
#pragma unroll
    for (int n = 0; n < 3; n += 2) {
      double v = 0.0;
      const double* src = a.part + (int64_t)(n == 0 ? (a.parity ^ 1) : 3) * a.nb;
      for (int32_t b = b0 + gt; b < b1; b += kBlock) v += src[b];
      v = tmh::wave_sum(v);
      if (lane == 0) s_red[n][gw] = v;
    }
  }
  __syncthreads();
  const int n_halo = SOLO ? 0 : s_halo;
  if (n_halo > kHalo) {  // uniform per workgroup
    if (tid == 0) post(a.abort, 2);
    return;
  }
  // byte offsets into s_u of the columns, two to a word; past the row's end
  // (and without a row) the workgroup's first row.  A row of more entries than
  // a thread holds, or a column of another system, ends the launch: the first
  // would be cut short, the second has no place in s_u.
  uint32_t cj[K][PER / 2];
  bool unfit = false;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    unfit |= len[k] > PER;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      uint32_t at = 0;
      if (j < len[k]) {
        const int32_t col = a.ci[ra[k] + j];
        unfit |= (uint32_t)(col - sys_row0) >= (uint32_t)sys_rows;
        at = (uint32_t)(col - own);
        if (!SOLO && at >= (uint32_t)kOwn) {
          uint32_t h = hash(col);
          while (s_key[h] != col) h = (h + 1) % kTable;
          at = kOwn + s_hidx[h];
        }
      }
      at *= (uint32_t)sizeof(T);
      cj[k][j / 2] = j % 2 ? cj[k][j / 2] | (at << 16) : at;
    }
  }
  if (unfit) s_abort = 1;
  // this thread's halo columns, as byte offsets into a buffer of u
  constexpr int kHaloPer = SOLO ? 1 : kHalo / kThreads;
  uint32_t hc[kHaloPer];
#pragma unroll
  for (int m = 0; m < kHaloPer; ++m) {
    const int i = tid + m * kThreads;
    hc[m] = SOLO || n_halo == 0 ? 0u : (uint32_t)s_hcol[i < n_halo ? i : 0] * (uint32_t)sizeof(T);
  }
  // the first wave publishes the workgroup's sums
  const bool poster = tid / 64 == 0 && lane < 16 * K && (lane & 3) < 3 && wb0 + (lane >> 2) < b1;
  const int64_t my_word = (int64_t)wb0 * 4 + lane;
  double gamma = tmh::uniform(((s_red[0][0] + s_red[0][1]) + s_red[0][2]) + s_red[0][3]);
  double delta = tmh::uniform(((s_red[2][0] + s_red[2][1]) + s_red[2][2]) + s_red[2][3]);
  double rr = 0.0;
  const double bb = c[5];
  const double* prev = c + 8 + 4 * (a.parity ^ 1);
  double iter = prev[2], alpha0 = prev[0], gamma0 = prev[1];
  bool active = true;
  int buf = 0;
  __syncthreads();  // s_red and the tables are read
  if (s_abort) {    // uniform per workgroup
    if (tid == 0) post(a.abort, 3);
    return;
  }
#pragma unroll
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (k * PER + j >= kReg)
        s_val[(k * PER + j - kReg) * kThreads + tid] = j < len[k] ? ((const T*)a.av)[ra[k] + j] : T(0);
  for (int32_t it = 0; it < a.n_iter && active; ++it) {
    const int next = buf == 2 ? 0 : buf + 1;
    const int par = SOLO ? it & 1 : 0;
    T* const su = s_u + (SOLO ? par * kOwn : 0);
    W* const ub = (W*)a.ubuf + (int64_t)buf * a.n_rows;
    W* const un = (W*)a.ubuf + (int64_t)next * a.n_rows;
    double alpha, beta;
    if (iter == 0.0) {
      beta = 0.0;
      alpha = delta != 0.0 ? gamma / delta : 0.0;
    } else {
      beta = gamma0 != 0.0 ? gamma / gamma0 : 0.0;
      const double den = delta - beta * gamma / alpha0;
      alpha = den != 0.0 ? gamma / den : 0.0;
    }
    const T al = (T)alpha, be = (T)beta;
    double g[K], q[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      g[k] = q[k] = 0.0;
      if (row[k] >= 0) {
        // u leaves first: the other workgroups wait for it
        const T u0 = u[k];
        s[k] = tmh::fma_t(be, s[k], w[k]);
        r[k] = tmh::fma_t(-al, s[k], r[k]);
        u[k] = d[k] * r[k];
        if constexpr (!SOLO) post(ub + row[k], to_word<T>(u[k]));
        su[row[k] - own] = u[k];
        p[k] = tmh::fma_t(be, p[k], u0);
        x[k] = tmh::fma_t(al, p[k], x[k]);
        g[k] = (double)r[k] * (double)u[k];
        q[k] = (double)r[k] * (double)r[k];
      }
    }
    W hv[kHaloPer];
    auto read_halo = [&] {
#pragma unroll
      for (int m = 0; m < kHaloPer; ++m)
        if (m * kThreads < n_halo) hv[m] = peek_at(ub, hc[m]);
    };
    if constexpr (!SOLO) {
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (row[k] >= 0) post(un + row[k], (W)Word<T>::kEmpty);
      if (poster) post(a.pbuf + (int64_t)next * a.nb * 4 + my_word, (uint64_t)~0ull);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const double gs = tmh::wave_sum(g[k]), qs = tmh::wave_sum(q[k]);
      if (lane == 0) {
        s_wave[par][0][k * kGroups + grp][gw] = gs;
        s_wave[par][1][k * kGroups + grp][gw] = qs;
      }
    }
    Patience wait;
    if constexpr (!SOLO) {
      // a first look that comes too early costs more than it finds: the polls
      // queue before the words they wait for (5.4 -> 5.0 us per step at 256
      // workgroups, no change at 40)
      __builtin_amdgcn_s_sleep(8);
      read_halo();
      for (;;) {
        bool bad = false;
#pragma unroll
        for (int m = 0; m < kHaloPer; ++m) bad |= m * kThreads < n_halo && hv[m] == Word<T>::kEmpty;
        if (!bad) break;
        if (!wait.more(a.abort)) {
          s_abort = 1;
          break;
        }
        read_halo();
      }
#pragma unroll
      for (int m = 0; m < kHaloPer; ++m)
        if (tid + m * kThreads < n_halo) su[kOwn + tid + m * kThreads] = __builtin_bit_cast(T, hv[m]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      T acc = T(0);
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const T uj = *reinterpret_cast<const T*>(reinterpret_cast<const char*>(su) +
                                                 (j % 2 ? cj[k][j / 2] >> 16 : cj[k][j / 2] & 0xffffu));
        const T aj = k * PER + j < kReg ? av[k * PER + j < kReg ? k * PER + j : 0]
                                        : s_val[(k * PER + j - kReg) * kThreads + tid];
        acc = j < len[k] ? acc + aj * uj : acc;
      }
      w[k] = acc;
      const double ds = tmh::wave_sum(row[k] >= 0 ? (double)acc * (double)u[k] : 0.0);
      if (lane == 0) s_wave[par][2][k * kGroups + grp][gw] = ds;
    }
    double sum[3];
    if constexpr (SOLO) {
      __syncthreads();
#pragma unroll
      for (int n = 0; n < 3; ++n) {
        // at most eight sums: of the butterfly over 64 lanes and the other
        // waves of the 256-thread sum, all but three steps add zeros
        const int at = lane & 7;
        const double* t = s_wave[par][n][at < kGroups * K ? at : 0];
        double v = 0.0;
        if (at < b1 - b0) v += ((t[0] + t[1]) + t[2]) + t[3];
        v += tmh::dpp_move<0x124>(v);
        v += tmh::dpp_move<0x122>(v);
        v += tmh::dpp_move<0x121>(v);
        sum[n] = v;
      }
    } else {
      // this wave's words (u, and the resets) have reached memory before any
      // sum of the workgroup is published
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (poster) {
        const double* t = s_wave[0][lane & 3][lane >> 2];
        post(a.pbuf + (int64_t)buf * a.nb * 4 + my_word, to_word<double>(((t[0] + t[1]) + t[2]) + t[3]));
      }
      if (grp < 3) {
        // every workgroup adds the system's sums itself, one quantity to a
        // group of 256 threads, kPoll words at a time: one round trip for the
        // 1,024 sums of a system of 262,144 rows
        const uint64_t* src = a.pbuf + (int64_t)buf * a.nb * 4 + grp;
        double v = 0.0;
        __builtin_amdgcn_s_sleep(16);  // as above: 5.8 -> 5.5 us at 256 workgroups, 4.6 -> 4.2 at 88
        for (int32_t b = b0 + gt; b < b1; b += kPoll * kBlock) {
          uint64_t t[kPoll];
          for (;;) {
            bool bad = false;
#pragma unroll
            for (int n = 0; n < kPoll; ++n) t[n] = peek(src + (int64_t)(b + n * kBlock < b1 ? b + n * kBlock : b) * 4);
#pragma unroll
            for (int n = 0; n < kPoll; ++n) bad |= t[n] == Word<double>::kEmpty;
            if (!bad) break;
            if (!wait.more(a.abort)) {
              s_abort = 1;
              break;
            }
          }
#pragma unroll
          for (int n = 0; n < kPoll; ++n)
            if (b + n * kBlock < b1) v += __builtin_bit_cast(double, t[n]);
        }
        v = tmh::wave_sum(v);
        if (lane == 0) s_red[grp][gw] = v;
      }
      __syncthreads();
      if (s_abort) return;  // x untouched
#pragma unroll
      for (int n = 0; n < 3; ++n) sum[n] = ((s_red[n][0] + s_red[n][1]) + s_red[n][2]) + s_red[n][3];
    }
    alpha0 = tmh::uniform(alpha);
    gamma0 = gamma;
    iter += 1.0;
    gamma = tmh::uniform(sum[0]);
    rr = tmh::uniform(sum[1]);
    delta = tmh::uniform(sum[2]);
    active = rr > a.tol2 * bb && bb > 0.0;
    buf = next;
  }
#pragma unroll
  for (int k = 0; k < K; ++k)
    if (row[k] >= 0) ((T*)a.x)[row[k]] = x[k];
  if (tid == 0 && wb0 == b0) {
    c[4] = rr;
    c[6] = active ? 1.0 : 0.0;
    c[7] = iter;
  }
}

// Every word of the buffers that iteration 0 reads, and the abort word.
template <typename T>
__global__ void __launch_bounds__(kBlock) cg2_run_reset_kernel(typename Word<T>::type* __restrict__ ubuf, int64_t n,
                                                               uint64_t* __restrict__ pbuf, int64_t np,
                                                               int32_t* __restrict__ abort) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) ubuf[i] = Word<T>::kEmpty;
  if (i < np) pbuf[i] = ~0ull;
  if (i == 0) *abort = 0;
}

template <typename T>
const void* kernel_of(int k, int per, bool solo) {
#define TM_RUN(K, PER) \
  if (k == K && per == PER) return solo ? (const void*)cg2_run_kernel<T, K, PER, true> : (const void*)cg2_run_kernel<T, K, PER, false>
  TM_RUN(1, 8);
  TM_RUN(1, 16);
  TM_RUN(1, 24);
  TM_RUN(2, 8);
#undef TM_RUN
  return nullptr;
}

const void* kernel_of(int dtype, int k, int per, bool solo) {
  return dtype == TM_F64 ? kernel_of<double>(k, per, solo) : dtype == TM_F32 ? kernel_of<float>(k, per, solo) : nullptr;
}

int64_t up16(int64_t v) { return (v + 15) / 16 * 16; }

}  // namespace

extern "C" int64_t tm_pcg_run_workgroups(int32_t dtype, int32_t rows_per_thread, int32_t row_entries) {
  const void* f = kernel_of(dtype, rows_per_thread, row_entries, false);
  if (!f) return 0;
  int dev = 0, cus = 0, coop = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, kThreads, 0) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return coop ? (int64_t)cus * per_cu : 0;
}

extern "C" int64_t tm_pcg_run_bytes(const tm_pcg_view* v) {
  if (!v || v->n_rows < 0 || v->n_blocks < 0) return 0;
  return up16(3 * v->n_rows * (v->dtype == TM_F64 ? 8 : 4)) + 12 * 8 * v->n_blocks + 16;
}

extern "C" int tm_pcg_run(const tm_pcg_view* v, const tm_pcg_run_plan* plan, void* x, int32_t n_iter,
                          tm_stream_t stream_) {
  TM_TRY_BEGIN
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (!v || !plan || !x || n_iter < 1) return tmh::fail(TM_ERR_ARG, "NULL view / plan / x or no steps");
  if (v->two_launch != 1) return tmh::fail(TM_ERR_ARG, "tm_pcg_run continues the two-launch iteration");
  if (v->n_rows <= 0 || v->n_rows >= tmh::kMaxIndex / 8 || v->n_blocks <= 0 || v->n_blocks >= tmh::kMaxIndex ||
      v->n_sys <= 0 || plan->n_wg <= 0 || plan->n_wg > v->n_blocks)
    return tmh::fail(TM_ERR_SIZE, "bad system or workgroup counts");
  if (!v->row_ptr || !v->col_idx || !v->values || !v->dinv || !v->r || !v->q || !v->partials || !v->scalars ||
      !v->blk_row0 || !v->blk_row1 || !v->sys_blk || !plan->wg_sys || !plan->wg_blk0 || !plan->ws)
    return tmh::fail(TM_ERR_ARG, "NULL buffer");
  const void* f = kernel_of(v->dtype, plan->rows_per_thread, plan->row_entries, false);
  const void* f_solo = kernel_of(v->dtype, plan->rows_per_thread, plan->row_entries, true);
  if (!f) return tmh::fail(TM_ERR_UNSUPPORTED, "no kernel for these rows per thread and row entries");
  if (plan->ws_bytes < tm_pcg_run_bytes(v)) return tmh::fail(TM_ERR_SIZE, "workspace too small");
  if (plan->n_solo > 0 && (plan->solo_blocks < 1 || plan->solo_blocks > kGroups * plan->rows_per_thread))
    return tmh::fail(TM_ERR_ARG, "one-workgroup systems of more blocks than a workgroup takes");
  if (plan->n_solo < 0 || plan->n_solo > plan->n_wg || plan->n_launch < 0 || (plan->n_launch > 0 && !plan->launch_end))
    return tmh::fail(TM_ERR_ARG, "bad launch groups");
  const int64_t most_wg = plan->n_launch ? tm_pcg_run_workgroups(v->dtype, plan->rows_per_thread, plan->row_entries) : 0;
  int64_t at = plan->n_solo;
  for (int32_t i = 0; i < plan->n_launch; ++i) {
    const int64_t n = plan->launch_end[i] - at;
    if (n <= 0) return tmh::fail(TM_ERR_ARG, "empty launch group");
    if (n > most_wg) return tmh::fail(TM_ERR_UNSUPPORTED, "more workgroups than can run at once");
    at += n;
  }
  if (at != plan->n_wg) return tmh::fail(TM_ERR_ARG, "launch groups do not cover the workgroups");
  const int64_t ubytes = up16(3 * v->n_rows * (v->dtype == TM_F64 ? 8 : 4));
  char* ws = static_cast<char*>(plan->ws);
  RunArgs a{};
  a.wg_sys = plan->wg_sys;
  a.wg_blk0 = plan->wg_blk0;
  a.sys_blk = v->sys_blk;
  a.blk_row0 = v->blk_row0;
  a.blk_row1 = v->blk_row1;
  a.rp = v->row_ptr;
  a.ci = v->col_idx;
  a.av = v->values;
  a.dinv = v->dinv;
  a.r = v->r;
  a.w = v->q;
  a.x = x;
  a.part = v->partials;
  a.sc = v->scalars;
  a.nb = (int32_t)v->n_blocks;
  a.parity = v->parity & 1;
  a.n_iter = n_iter;
  a.tol2 = v->rtol * v->rtol;
  a.ubuf = ws;
  a.pbuf = reinterpret_cast<uint64_t*>(ws + ubytes);
  a.abort = reinterpret_cast<int32_t*>(a.pbuf + 12 * v->n_blocks);
  a.n_rows = v->n_rows;
  const bool solo = plan->n_launch == 0;  // nothing is exchanged through memory
  const int64_t words = solo ? 1 : v->n_rows, pwords = solo ? 1 : 4 * v->n_blocks;
  const int64_t grid = ((words > pwords ? words : pwords) + kBlock - 1) / kBlock;
  if (v->dtype == TM_F64)
    cg2_run_reset_kernel<double><<<grid, kBlock, 0, stream>>>((uint64_t*)ws, words, a.pbuf, pwords, a.abort);
  else
    cg2_run_reset_kernel<float><<<grid, kBlock, 0, stream>>>((uint32_t*)ws, words, a.pbuf, pwords, a.abort);
  void* args[] = {&a};
  hipError_t err = hipGetLastError();
  if (err == hipSuccess && plan->n_solo > 0)
    err = hipLaunchKernel(f_solo, dim3((unsigned)plan->n_solo), dim3(kBlock * (plan->solo_blocks < kGroups ? plan->solo_blocks : kGroups)), args, 0, stream);
  for (int32_t i = 0; i < plan->n_launch && err == hipSuccess; ++i) {
    const int64_t lo = i ? plan->launch_end[i - 1] : plan->n_solo;
    a.wg_sys = plan->wg_sys + lo;
    a.wg_blk0 = plan->wg_blk0 + lo;
    err = hipLaunchCooperativeKernel(const_cast<void*>(f), dim3((unsigned)(plan->launch_end[i] - lo)), dim3(kThreads),
                                     args, 0, stream);
  }
  if (err != hipSuccess) {
    (void)hipGetLastError();
    tmh::set_error("pcg run launch: %s", hipGetErrorString(err));
    return TM_ERR_HIP;
  }
  return TM_OK;
  TM_TRY_END
}
