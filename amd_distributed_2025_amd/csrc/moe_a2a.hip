// MoE dispatch/combine for one rank on MI355X (gfx950, wave64).
//
// Stages 1-3 are "ranked row moves". A workgroup owns a group of ROWS
// consecutive rows of its stage's input stream, one wave64 per row. Each wave
// first issues the 16-byte loads of its whole row (up to 16 vectors per lane
// in flight), then the workgroup finds the destination slot of all its rows
// with ONE pass over the stage's keys: a slot is the number of keys that
// precede the row in the stage's stable order, so every lane counts, for each
// of the group's rows, the keys it scanned that precede that row; the counts
// are reduced with a wave64 butterfly and a small LDS exchange; then each wave
// stores its row. The keys are a few KB and stay in L2. There are no atomics
// on global memory, no counters to clear and no dependencies between
// workgroups, so results do not depend on scheduling and nothing has to be
// zeroed between calls.
//
// Stage 4 (combine) gives a workgroup one token: it finds the rows addressed to
// the token, orders them by arrival, and accumulates them with the reference's
// per-addend rounding.
//
// Reference behaviour reproduced here: all2all/reference.py:68-148 (dispatch),
// :151-234 (combine), :262 (simulated expert).

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <limits.h>
#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>

#include "moe_a2a.h"
#include "stream_rules.h"
#include "tile_rules.h"

// Device memory of moe_a2a_dispatch_recv_static: the send-back plan of one call, held by the
// library so that the caller brings no buffer for it. Every GPU the library runs on has its own
// copy at its own address; host code reaches it only through the address that
// hipGetSymbolAddress returned for that GPU (static_plan_buffer below), never through this name.
#define MOE_A2A_STATIC_PLAN_EXPERTS 4096  /* world_size <= 64 times num_local_experts <= 64 */
static __device__ __align__(256) int32_t scratch[2 * MOE_A2A_STATIC_PLAN_EXPERTS];

namespace {

constexpr int META = MOE_A2A_META_DIM;
constexpr int NWAVES = BLOCK / 64;
constexpr int COMBINE_CAP = 64;       // addends per token handled by the fast path
constexpr int COMBINE_WEIGHTS = 128;  // weights of one token staged in LDS
constexpr int COMBINE_BATCH = 8;      // addend rows loaded before accumulating
constexpr int MAX_LOCAL_EXPERTS = 4096;  // LDS prefix table of the expert-major walkers
constexpr int NUM_XCD = 8;

// 16 bytes as a native clang vector: loads and stores of it are single
// global_load/store_dwordx4 and the value lives in registers. (HIP's uint4 is a
// struct whose copies become memcpy calls that can pin a local in memory.)
typedef unsigned int b128 __attribute__((ext_vector_type(4)));

// How a row is stored.
// STREAM (nontemporal) does not write-allocate in L2, which makes the writing kernel about a quarter faster, but a
// kernel that reads the rows right afterwards then fetches them from HBM and loses more than the writer gained. So
// the row movers use it only for the two buffers whose next reader is the exchange (in a multi-GPU job: the
// fabric), not for expert_x / expert_y, which the expert computation reads next on the same device.
// THROUGH (device scope) writes on past L2 while the kernel runs. What a plain store leaves dirty there is written
// back when the kernel ends, with nothing else going on: the 29 MB that stage 2 writes at the headline shape
// (8 ranks, 2048 rows of 14 KB) cost 15.8 us plain, 14.7 through; the stand-in's rows of a whole job 44.5 and 42.9.
// The readers lose nothing: the L2s of the XCDs do not serve each other, so they come from behind L2 either way.
// With little to write back the longer way of each store costs more. Where the line lies, us of the kernel in a graph, plain
// / through, and of the kernels of a job around it where that tells more:
//  - stage 2, whose waves write whole rows: about 1000 of them, whatever their length, or 8 MB (10 rows of 5.8 KB 3.45 / 3.98,
//    715 4.43 / 4.62, 1010 4.96 / 4.93, 1422 6.08 / 5.46; 483 of 14 KB 5.15 / 5.34, 715 5.88 / 5.86, 1010 6.68 / 6.09; 494 of
//    2 KB 3.71 / 3.92, 2042 6.71 / 6.32; with stages 2 and 3 around the expert 1010 of 8 KB 16.3 / 17.3, 1169 16.8 / 16.5,
//    1422 of 5.8 KB 16.6 / 15.9, 2042 of 2 KB 13.9 / 12.9).
//  - stand-in expert and the dispatch of a job whose ranks share the GPU: 1 MB of rows (dispatch: 64 rows of 512 B 3.76 /
//    3.92, 1.0 MB of them 4.37 / 4.59, 3.9 MB 7.80 / 7.70; 1 MB of 2 KB 3.95 / 4.04, 4 MB 4.77 / 4.63; 7 MB of 14 KB 5.09 /
//    4.73. Expert: 0.5 MB of 512 B 2.25 / 2.18, 28 MB of 14 KB 9.84 / 7.21. One rank's dispatch, expert and combine: 0.1 MB
//    of 5.8 KB 10.46 / 10.77, 0.7 MB 10.99 / 11.11, 1.4 MB 11.68 / 11.37, 2.8 MB 13.10 / 12.54).
//  - exchange: 8 MB of rows for a rank (0.03 MB of 512 B 2.25 / 2.41, 3.9 MB 6.30 / 7.31; 8 MB of 2 KB 5.01 / 5.27, 16 MB 8.46
//    / 7.80; 3.9 MB of 8 KB 3.18 / 3.31, 6.2 MB 3.67 / 3.61).
enum Store { PLAIN, THROUGH, STREAM };
//  - results of a job whose ranks share the GPU, past the cache behind L2, where they and the rows they are added up from are 80 MB, with several ranks
//    128 MB: what is left dirty there goes out line by line among the reads of whatever comes next. us of the whole call, plain / stream: layer of 32
//    experts, 2048 x 4096, 2048 tokens, 4 per token (84 MB) 337 / 333, of 64, 1024 x 4096, 2048 tokens, 8 per token (151 MB) 413 / 410; 8 ranks of
//    256 tokens, 8 per token of 14 KB (264 MB) 92.5 / 91.4, of 8 KB (151 MB) 55.7 / 55.4, but of 189, 4 per token of 11 KB (84 MB) 38.1 / 38.7.
//    Nontemporal loads of the rows as well: 330, 410; 94.3, 54.6.
constexpr long long JOB_STREAM_BYTES = 80ll << 20, JOB_RANKS_STREAM_BYTES = 128ll << 20;
constexpr long long JOB_THROUGH_BYTES = 1 << 20, EXCHANGE_THROUGH_BYTES = 8 << 20;  // (stage 2's: recv_through)
// (a kernel for each kind: chosen inside one, the stores of 5.5 MB of rows took 0.3 us longer than either)
template <typename V> constexpr Store THROUGH_OF = sizeof(V) == sizeof(b128) ? THROUGH : PLAIN;  // (of 16 bytes only)
#ifndef MOE_A2A_STORE_SEND   /* stage 1 -> send buffer */
#define MOE_A2A_STORE_SEND STREAM
#endif
#ifndef MOE_A2A_STORE_CSEND  /* stage 3 -> send-back buffer */
#define MOE_A2A_STORE_CSEND STREAM
#endif
template <Store HOW, typename V>
__device__ __forceinline__ void row_store(V* p, const V& v) {
  if constexpr (HOW == STREAM) __builtin_nontemporal_store(v, p);
  else if constexpr (HOW == THROUGH && sizeof(V) == sizeof(b128))
    __builtin_amdgcn_global_store_b128((__attribute__((address_space(1))) b128*)p, v, "agent");
  else *p = v;
}
// PAST: nontemporal, for rows of streams that the caches do not hold (csrc/stream_rules.h).
template <bool PAST, typename P>
__device__ __forceinline__ auto row_load(P p) {
  if constexpr (PAST) return __builtin_nontemporal_load(p);
  else return *p;
}

// ---------------------------------------------------------------- wave / block primitives

// Workgroup barrier that orders LDS traffic only. __syncthreads() also waits
// for every global load in flight, which would drain a row's prefetched payload
// in the middle of the slot computation; the waves here exchange data through
// LDS alone, so waiting for the LDS counter is enough.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Inclusive prefix sum across the 64 lanes of a wave, in the VALU's
// data-parallel-primitive (DPP) lane network: four row_shr steps scan each row
// of 16 lanes, row_bcast15 / row_bcast31 carry the row totals across rows.
// Six dependent VALU ops; a __shfl-based scan would take six round trips through
// the LDS crossbar, which is what dominates a slot computation of a few hundred
// cycles.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_add(int v) {
  // lanes whose source lies outside the row, or whose row is masked off, add 0
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xf, false);
}

__device__ __forceinline__ int wave_inclusive_scan(int v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1
  v = dpp_add<0x112, 0xf>(v);  // row_shr:2
  v = dpp_add<0x114, 0xf>(v);  // row_shr:4
  v = dpp_add<0x118, 0xf>(v);  // row_shr:8
  v = dpp_add<0x142, 0xa>(v);  // row_bcast15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast31 into rows 2 and 3
  return v;
}

// Sum over the wave, returned to every lane.
__device__ __forceinline__ int wave_sum(int v) {
  return __builtin_amdgcn_readlane(wave_inclusive_scan(v), 63);
}

// Sum over a workgroup of NW waves; every lane gets the total. `red` is NW ints
// of LDS and may be reused right after the call returns.
template <int NW>
__device__ __forceinline__ int block_sum(int v, int* red) {
  v = wave_sum(v);
  if (NW == 1) return v;
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  lds_barrier();
  int s = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) s += red[w];
  lds_barrier();
  return s;
}

// A value that was loaded early, handed on at the place where the program first needs it. The
// compiler moves arithmetic on a loaded value (a clamp, a compare) up to the load, out of loops
// and branches, and then waits for the load right there: a whole memory round trip ahead of
// everything issued after it. An empty volatile asm statement cannot be moved, so the wait lands
// where this is called.
__device__ __forceinline__ int first_use(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// A float32 value that counts as computed and rounded at this point: the compiler may not fuse the
// multiplication that made it with the conversion that follows. (Fused, a product rounded to fp16
// becomes v_fma_mixlo_f16 with an addend of +0, and -0 * scale + 0 is +0 where the product is -0.)
__device__ __forceinline__ float rounded_here(float v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Loads through a pointer that went through unknown_origin() and were issued before issued_here()
// stay before it. The compiler otherwise sinks a load whose value is only used under a condition
// into that condition's block, behind whatever the condition waits for; an asm statement that
// may write memory stops that only for pointers that it cannot prove untouched by the statement
// (a __restrict__ parameter is proven, the same address out of an asm statement is not).
// The pointer must be the same for every lane of the wave (it is kept in scalar registers).
template <typename T>
using global_ptr = const T __attribute__((address_space(1)))*;  // (still known to point into global memory)
template <typename T>
__device__ __forceinline__ global_ptr<T> unknown_origin(const T* p) {
  uint64_t a = (uint64_t)p;
  asm volatile("" : "+s"(a));
  return (global_ptr<T>)a;
}
__device__ __forceinline__ void issued_here() { asm volatile("" ::: "memory"); }

// Workgroups are handed to the 8 XCDs round-robin by blockIdx. This bijection
// on [0, grid) gives each XCD one contiguous run of logical items, so items
// that share a source row are served by the same L2.
__device__ __forceinline__ int xcd_contiguous(int b, int grid) {
  const int x = b % NUM_XCD;
  const int base = grid / NUM_XCD, rem = grid % NUM_XCD;
  return x * base + min(x, rem) + b / NUM_XCD;
}

// floor-mod (Python's %) by a positive divisor. `magic` = ceil(2^32 / d) gives
// an exact quotient for 0 <= e < 65536 and d <= 65536; other values take the
// slow path.
__device__ __forceinline__ int floormod(int e, int d, uint32_t magic) {
  if (d == 1) return 0;
  if ((uint32_t)e < 65536u) {
    uint32_t q = __umulhi((uint32_t)e, magic);
    return e - (int)q * d;
  }
  int m = e % d;
  return m < 0 ? m + d : m;
}

// As a kernel's first argument: a structure passed by value ends the arguments that waves start with in registers. Setting those
// up costs some 3 cycles per wave wherever waves are started, which shows where a launch is many waves with little to do. (Two
// words: a structure of one travels as that word.)
struct ArgumentsLoaded {
  int unused[2];
};

// key[u] = floormod(key[u], d, magic), with one branch for all of them.
template <int U>
__device__ __forceinline__ void floormod_each(int (&key)[U], int d, uint32_t magic) {
  int all = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) all |= key[u];
  if (__ballot((uint32_t)all >= 65536u) != 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) key[u] = floormod(key[u], d, magic);
    return;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) key[u] = d == 1 ? 0 : key[u] - (int)__umulhi((uint32_t)key[u], magic) * d;
}

// Inclusive [lo, hi] range of expert ids owned by the same destination as `e`.
// Ids outside [0, E) name no destination: they form one class after all ranks
// (compared as unsigned numbers, a negative id is just a large one), so the
// classes still partition the integers, slots stay a permutation, the rows of
// the real destinations sit where the counts say, and the stray rows end up
// behind them, where no exchange looks.
__device__ __forceinline__ void dest_class(int e, int nle, int E, uint32_t magic, uint32_t& lo,
                                           uint32_t& hi) {
  if ((uint32_t)e >= (uint32_t)E) {
    lo = (uint32_t)E; hi = UINT_MAX;
  } else {
    const uint32_t d = (nle == 1) ? (uint32_t)e : __umulhi((uint32_t)e, magic);
    lo = d * nle; hi = lo + nle - 1;
  }
}

// Rows cut into `per_row` pieces each; pieces are numbered along the stream.
struct Pieces {
  int per_row;
  uint32_t magic, shift;  // q / per_row of 0 <= q < 2^31 is the high word of q * magic, shifted
  __device__ __forceinline__ int row_of(int q) const { return per_row == 1 ? q : (int)(__umulhi((uint32_t)q, magic) >> shift); }
};

// NV vectors of one row chunk held in registers. Loads are unconditional
// (lanes past the end of the row re-read its last vector), so all of them are
// in flight at once; only the stores are predicated.
template <typename V, int NV>
struct Payload {
  V v[NV];
  __device__ __forceinline__ void load(const V* __restrict__ row, int base, int row_vecs) {
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = row[min(base + j * BLOCK + (int)threadIdx.x, row_vecs - 1)];
  }
  template <Store HOW>
  __device__ __forceinline__ void store(V* __restrict__ row, int base, int row_vecs) const {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int idx = base + j * BLOCK + threadIdx.x;
      if (idx < row_vecs) row_store<HOW>(row + idx, v[j]);
    }
  }
  template <typename F>
  __device__ __forceinline__ void map(F f) {
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = f(v[j]);
  }
};

// Sum of max(counts[i], 0) over i < n, computed by every wave on its own: the
// lanes load the counts side by side (one memory round trip instead of n
// dependent scalar loads) and reduce with the wave butterfly.
// Every count is also cut to `cap`; callers make sure n * cap fits an int, so
// the sum cannot wrap whatever the counts hold.
__device__ __forceinline__ int sum_counts(const int* __restrict__ counts, int n, int cap) {
  const int lane = threadIdx.x & 63;
  int s = 0;
  for (int i = lane; i < n; i += 64) s += min(max(counts[i], 0), cap);
  return __builtin_amdgcn_readfirstlane(wave_sum(s));
}

// Number of keys i in [0, n) that pass `test(key_i, i)`, summed over the lanes
// of this thread only (reduce with block_sum). `keys.fetch(idx, key)` loads
// SCAN_UNROLL keys at once (indices already clamped to [0, n)), so that all
// loads are in flight before the first compare; lanes past n are masked out.
#ifndef MOE_A2A_SCAN_UNROLL
#define MOE_A2A_SCAN_UNROLL 8
#endif
constexpr int SCAN_UNROLL = MOE_A2A_SCAN_UNROLL;
template <int BLK, typename Keys, typename Test>
__device__ __forceinline__ int count_keys(int n, const Keys& keys, Test test) {
  int cnt = 0;
  // the trip count is the same for every lane: fetch() may use wave shuffles
  for (int b = 0; b < n; b += SCAN_UNROLL * BLK) {
    const int i = b + threadIdx.x;
    int idx[SCAN_UNROLL], key[SCAN_UNROLL];
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) idx[u] = min(i + u * BLK, n - 1);
    keys.fetch(idx, key);
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) {
      if (b + u * BLK >= n) break;
      cnt += (i + u * BLK < n) ? (int)test(key[u], i + u * BLK) : 0;
    }
  }
  return cnt;
}

// Keys stored `stride` ints apart, key i at base[i * stride].
struct StridedKeys {
  const int* __restrict__ base;
  int stride;
  template <int U>
  __device__ __forceinline__ void fetch(const int (&idx)[U], int (&key)[U]) const {
#pragma unroll
    for (int u = 0; u < U; ++u) key[u] = base[(size_t)idx[u] * stride];
  }
};

// One row chunk held by one wave: NVW vectors per lane, vector j of lane l is
// element base + j*64 + l of the row. Loads are unconditional and clamped, so
// all NVW of them are in flight at once; stores are predicated.
template <typename V, int NVW>
struct WavePayload {
  V v[NVW];
  template <bool PAST = false, typename P>  // const V* or global_ptr<V>
  __device__ __forceinline__ void load(P row, int base, int row_vecs, int lane) {
#pragma unroll
    for (int j = 0; j < NVW; ++j) v[j] = row_load<PAST>(row + min(base + j * 64 + lane, row_vecs - 1));
  }
  template <Store HOW>
  __device__ __forceinline__ void store(V* __restrict__ row, int base, int row_vecs, int lane) const {
#pragma unroll
    for (int j = 0; j < NVW; ++j) {
      const int idx = base + j * 64 + lane;
      if (idx < row_vecs) row_store<HOW>(row + idx, v[j]);
    }
  }
};

// For each of the ROWS rows r of a group: this lane's share of the number of
// keys i in [0, n) with test(r, key_i, i). Split in two so that the first
// batch of key loads can be issued BEFORE the row payload (loads return in
// issue order, so the keys arrive first and the slot is ready while the payload
// is still in flight):  RowsScan scan(n, keys);  ...issue payload...;
// scan.finish(keys, test, cnt);
// SHORT: scans that mostly end inside a batch leave it there. That pays while a unit has another workgroup to go on with (stage 2
// with / without, 1422 rows of 14 KB 8.15 / 8.41 us, of 8 KB 6.05 / 6.25); with one workgroup on a unit the waits at the branches
// cost more (900 rows of 14 KB 6.35 / 5.42), and so they do where batches are full (the 4800 rows of a skewed job in the
// compact layout 20.2 / 19.2).
template <typename Keys, bool SHORT = false, int UNROLL = SCAN_UNROLL>
struct RowsScan {
  static constexpr int STEP = 64 * ROWS;
  int n, b;  // keys that may be loaded; first key of the batch in flight (same for every lane)
  int key[UNROLL];
  // `n_load` keys are known to be readable; how many of them count is told to finish().
  __device__ __forceinline__ RowsScan(int n_load, const Keys& keys) : n(n_load), b(0) {
    if (n > 0) issue(keys);
  }
  // Every lane of the workgroup takes part (fetch() may use wave shuffles);
  // lanes whose keys fall past n load key n-1 and are masked in consume().
  __device__ __forceinline__ void issue(const Keys& keys) {
    const int i = b + threadIdx.x;
    int idx[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) idx[u] = min(i + u * STEP, n - 1);
    keys.fetch(idx, key);
  }
  template <typename Test>
  __device__ __forceinline__ void consume(Test test, int (&cnt)[ROWS]) const {
    const int i = b + threadIdx.x;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if (SHORT && b + u * STEP >= n) break;
      const int i2 = i + u * STEP;
      if (i2 < n) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) cnt[r] += (int)test(r, key[u], i2);
      }
    }
  }
  // Counts over keys [0, n_valid), n_valid <= n_load. The first batch is consumed
  // in straight-line code, apart from the loop over later batches: inside a loop
  // the compiler must assume the keys were the last loads issued and would wait
  // for the payload as well.
  template <typename Test>
  __device__ __forceinline__ void finish(const Keys& keys, int n_valid, Test test, int (&cnt)[ROWS]) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) cnt[r] = 0;
    const bool first = n > 0;
    n = min(n, n_valid);
    if (first) consume(test, cnt);
    for (b += UNROLL * STEP; b < n; b += UNROLL * STEP) {
      issue(keys);
      consume(test, cnt);
    }
  }
  // Adds the counts over keys [from, to): keys past the n_load the scan began with, readable now
  // that the caller knows the stream is that long (a stream longer than the hint it was launched with).
  template <typename Test>
  __device__ __forceinline__ void extend(const Keys& keys, int from, int to, Test test, int (&cnt)[ROWS]) {
    n = to;
    for (b = from; b < to; b += UNROLL * STEP) {
      issue(keys);
      consume(test, cnt);
    }
  }
};

// Total of cnt[wave] over the workgroup, returned to the lanes of that wave:
// wave w gets the count that belongs to the group's row w. `part` is
// 2*ROWS*ROWS ints of LDS used in halves by alternate calls (`parity` flips per
// call), so one barrier per call is enough: a wave can only overwrite a half
// after every wave has passed the barrier of the call in between.
__device__ __forceinline__ int rows_reduce(const int (&cnt)[ROWS], int* part, int parity, int wave,
                                           int lane) {
  if (ROWS == 1) return wave_sum(cnt[0]);
  int* half = part + (parity & 1) * (ROWS * ROWS);
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int s = wave_sum(cnt[r]);
    if (lane == 0) half[wave * ROWS + r] = s;
  }
  lds_barrier();
  int mine = 0;
#pragma unroll
  for (int w = 0; w < ROWS; ++w) mine += half[w * ROWS + wave];
  return mine;
}

// ---------------------------------------------------------------- stage 1: dispatch, send side
//
// grid = W counting workgroups (rows per destination rank) followed by one
// workgroup per (group of ROWS entries, chunk). Entry i = t*K + k goes to slot
//   #{entries of a lower destination} + #{earlier entries of the same destination}.

template <typename V, int NVW>
__global__ __launch_bounds__(64 * ROWS) void dispatch_send_kernel(
    const V* __restrict__ x, const int* __restrict__ indices, int S, int K, int W, int movers, int chunks, int row_vecs,
    int nle, int E, uint32_t magic, int rank, V* __restrict__ send_buf,
    int* __restrict__ send_meta, int* __restrict__ send_counts, int* __restrict__ send_slot) {
  __shared__ int part[2 * ROWS * ROWS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const StridedKeys key{indices, 1};

  if ((int)blockIdx.x < W) {
    const int lo = blockIdx.x * nle, hi = lo + nle - 1;
    int c = count_keys<64 * ROWS>(S, key, [lo, hi](int e, int) { return (e >= lo) & (e <= hi); });
    c = block_sum<ROWS>(c, part);
    if (tid == 0) send_counts[blockIdx.x] = c;
    return;
  }

  const int groups = (S + ROWS - 1) / ROWS;
  const int items = groups * chunks;
  int parity = 0;
  for (int q = xcd_contiguous(blockIdx.x - W, movers); q < items; q += movers, ++parity) {
    const int grp = chunks == 1 ? q : q / chunks, c = q - grp * chunks;
    const int i0 = grp * ROWS, i = i0 + wave;
    const bool valid = i < S;
    const int base = c * (64 * NVW);

    // every wave reads the expert ids of all rows of the group (the same few
    // words for every lane), so no exchange between the waves is needed
    int re[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) re[r] = indices[min(i0 + r, S - 1)];
    RowsScan<StridedKeys> scan(S, key);
    const int ic = min(i, S - 1);
    const int t = ic / K, k = ic - t * K;
    WavePayload<V, NVW> p;
    p.load(x + (size_t)t * row_vecs, base, row_vecs, lane);

    uint32_t rlo[ROWS], rhi[ROWS];
    int e = 0;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      dest_class(re[r], nle, E, magic, rlo[r], rhi[r]);
      if (r == wave) e = re[r];
    }
    int cnt[ROWS];
    scan.finish(key, S, [&](int r, int e2, int i2) {
      const uint32_t u2 = (uint32_t)e2;
      return (u2 < rlo[r]) | ((u2 <= rhi[r]) & (u2 >= rlo[r]) & (i2 < i0 + r));
    }, cnt);
    const int slot = rows_reduce(cnt, part, parity, wave, lane);

    if (valid) {
      p.template store<MOE_A2A_STORE_SEND>(send_buf + (size_t)slot * row_vecs, base, row_vecs, lane);
      if (c == 0) {
        if (lane < META) {
          int m = lane == 0 ? e : lane == 1 ? rank : lane == 2 ? t : lane == 3 ? k : 0;
          send_meta[(size_t)slot * META + lane] = m;
        }
        if (lane == 0 && send_slot) send_slot[i] = slot;
      }
    }
  }
}

// Stage 1 with one workgroup per (token, row chunk): the token's row is loaded
// once, its K entries are ranked together (FAN at a time) in one pass over the
// keys, and the row held in registers is stored to each of their slots. Compared
// with a wave per entry this reads every source row once instead of K times and
// issues an eighth of the key loads. The order is carried by one composite key
// per entry, class * S + i with class = destination, or W for an id outside
// [0, E): entry a precedes entry b exactly when its composite key is smaller.
// The host uses this kernel when (W + 2) * S fits an int.

// FAN: entries of a token that are ranked in one pass over the keys and then stored (2, 4 or 8).
// Fewer per pass means more passes over the keys and more barriers, but the first rows leave sooner
// and the ranking of the next entries runs while they drain; a compute unit has nothing else to
// do meanwhile, because all its workgroups rank at the same time. That pays while a pass is short.
// Measured at K = 8, H = 7168, the chain of four kernels (stage 1 alone in brackets), us, with
// 2 / 4 / 8: S = 2048 entries 36.5 / 36.9 / 37.4; S = 4096 73.9 / 75.4 / 74.5 (15.7 / 14.2 / 15.2);
// S = 8192 168.7 / 167.9 / 164.4 (31.6 / 31.8 / 29.0); S = 12288 233.2 / 230.5 / 222.6 (50.3 / 42.9 /
// 38.8); S = 32768 693.6 / 615.0 / 567.7 (245.4 / 169.4 / 130.6). The host takes 2 up to
// MOE_A2A_FAN2_MAX_ENTRIES entries and 8 above.
#ifndef MOE_A2A_FAN2_MAX_ENTRIES
#define MOE_A2A_FAN2_MAX_ENTRIES 4096
#endif
inline int fan_of(long long S) { return S <= MOE_A2A_FAN2_MAX_ENTRIES ? 2 : 8; }

template <typename V, int NV, int FAN>
__global__ __launch_bounds__(BLOCK) void dispatch_fanout_kernel(
    const V* __restrict__ x, const int* __restrict__ indices, int T, int K, int W, int chunks, int row_vecs, int nle,
    int E, uint32_t magic, int rank, V* __restrict__ send_buf,
    int* __restrict__ send_meta, int* __restrict__ send_counts, int* __restrict__ send_slot) {
  __shared__ int part[2 * NWAVES * FAN];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int S = T * K;
  // destination rank, or W for an id outside [0, E)
  auto klass = [&](int e) {
    return (uint32_t)e >= (uint32_t)E ? W : nle == 1 ? e : (int)__umulhi((uint32_t)e, magic);
  };

  if ((int)blockIdx.x < W) {
    const int want = blockIdx.x;
    int c = count_keys<BLOCK>(S, StridedKeys{indices, 1}, [&](int e, int) { return klass(e) == want; });
    c = block_sum<NWAVES>(c, part);
    if (tid == 0) send_counts[blockIdx.x] = c;
    return;
  }

  const int items = T * chunks, movers = gridDim.x - W;
  int parity = 0;
  for (int q = blockIdx.x - W; q < items; q += movers) {
    const int t = chunks == 1 ? q : q / chunks, c = q - t * chunks;
    const int base = c * (BLOCK * NV);
    const int i0 = t * K;

    // first batch of keys, then the row: the keys come back first
    int key[SCAN_UNROLL];
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) key[u] = indices[min(tid + u * BLOCK, S - 1)];
    Payload<V, NV> p;
    p.load(x + (size_t)t * row_vecs, base, row_vecs);

    for (int g0 = 0; g0 < K; g0 += FAN) {
      int mine[FAN];
#pragma unroll
      for (int g = 0; g < FAN; ++g) {
        const int i = i0 + min(g0 + g, K - 1);
        mine[g] = klass(indices[i]) * S + i;
      }
      int cnt[FAN];
#pragma unroll
      for (int g = 0; g < FAN; ++g) cnt[g] = 0;
      auto consume = [&](const int (&k)[SCAN_UNROLL], int b) {
#pragma unroll
        for (int u = 0; u < SCAN_UNROLL; ++u) {
          const int i2 = b + tid + u * BLOCK;
          const int ck = i2 < S ? klass(k[u]) * S + i2 : INT_MAX;
#pragma unroll
          for (int g = 0; g < FAN; ++g) cnt[g] += (int)(ck < mine[g]);
        }
      };
      consume(key, 0);
      for (int b = SCAN_UNROLL * BLOCK; b < S; b += SCAN_UNROLL * BLOCK) {
        int more[SCAN_UNROLL];
#pragma unroll
        for (int u = 0; u < SCAN_UNROLL; ++u) more[u] = indices[min(b + tid + u * BLOCK, S - 1)];
        consume(more, b);
      }

      int* half = part + (parity++ & 1) * (NWAVES * FAN);
#pragma unroll
      for (int g = 0; g < FAN; ++g) {
        const int sum = wave_sum(cnt[g]);
        if (lane == 0) half[wave * FAN + g] = sum;
      }
      lds_barrier();
      const int live = min(FAN, K - g0);
#pragma unroll
      for (int g = 0; g < FAN; ++g) {
        if (g < live) {
          int slot = 0;
#pragma unroll
          for (int w = 0; w < NWAVES; ++w) slot += half[w * FAN + g];
          p.template store<MOE_A2A_STORE_SEND>(send_buf + (size_t)slot * row_vecs, base, row_vecs);
        }
      }
      if (c == 0 && tid < live * META) {
        const int g = tid / META, f = tid - g * META;
        int slot = 0;
#pragma unroll
        for (int w = 0; w < NWAVES; ++w) slot += half[w * FAN + g];
        const int i = i0 + g0 + g;
        const int m = f == 0 ? indices[i] : f == 1 ? rank : f == 2 ? t : f == 3 ? g0 + g : 0;
        send_meta[(size_t)slot * META + f] = m;
        if (f == 0 && send_slot) send_slot[i] = slot;
      }
    }
  }
}

// The same fan-out for rows longer than 256 vectors: a workgroup of BLK = 512
// lanes holds NV vectors per lane (BLK lanes apart), so a row is cut into fewer
// chunks and its K entries are ranked less often. A lane compares 2048 / BLK keys per
// batch; the per-wave counts travel as 16-bit pairs (entry g with entry g + 4),
// are summed across the waves by the DPP row scan of one wave (a row of 16
// lanes per pair) and come back through LDS. Needs S < 65536 for the pairs not
// to carry into each other (a slot is below S). The composite key here is
// class << order_bits | i with S <= 1 << order_bits (no multiply per key). Measured at K = 8, H = 7168:
// the whole step 0.3 us shorter than with 256 lanes; 1024 lanes (one chunk per
// row) 0.5 us longer.

template <typename V, int BLK, int NV, bool POW2, int FAN>
__global__ __launch_bounds__(BLK) void dispatch_fanout_wide_kernel(
    const V* __restrict__ x, const int* __restrict__ indices, int T, int K, int W, int chunks, int row_vecs, int E,
    uint32_t magic, int nle_shift, int order_bits, int rank,
    V* __restrict__ send_buf, int* __restrict__ send_meta, int* __restrict__ send_counts,
    int* __restrict__ send_slot) {
  constexpr int NW = BLK / 64;
  constexpr int KEYS = SCAN_UNROLL * BLOCK / BLK;  // a batch stays SCAN_UNROLL * BLOCK keys
  constexpr int PAIRS = FAN / 2;
  static_assert(FAN == 2 || FAN == 4 || FAN == 8, "pairs of 16-bit counts, one DPP row of 16 lanes per pair");
  static_assert(NW <= 16 && KEYS >= 1, "one DPP row of 16 lanes sums the waves");
  __shared__ int part[NW * PAIRS];
  __shared__ int total[PAIRS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int S = T * K;
  // destination rank, or W for an id outside [0, E). POW2: nle is a power of two and the division
  // is a shift (the multiply-high it replaces runs at a quarter of the rate)
  auto klass = [&](int e) {
    const int d = POW2 ? e >> nle_shift : (int)__umulhi((uint32_t)e, magic);
    return (uint32_t)e >= (uint32_t)E ? W : d;
  };
  // the composite key of entry i: class in the high bits, i below (S <= 1 << order_bits)
  auto composite = [&](int e, int i) { return (klass(e) << order_bits) | i; };

  if ((int)blockIdx.x < W) {
    const int want = blockIdx.x;
    int c = count_keys<BLK>(S, StridedKeys{indices, 1}, [&](int e, int) { return klass(e) == want; });
    c = block_sum<NW>(c, part);
    if (tid == 0) send_counts[blockIdx.x] = c;
    return;
  }

  const int items = T * chunks, movers = gridDim.x - W;
  for (int q = blockIdx.x - W; q < items; q += movers) {
    const int t = chunks == 1 ? q : q / chunks, c = q - t * chunks;
    const int col = c * (BLK * NV) + tid;  // this lane's first vector; the others BLK apart
    const int i0 = t * K;

    // the token's own expert ids: lane l of every wave holds entry l, or entry g0 + l % FAN of a token with more than
    // 64 and where eight are ranked per pass, which is mostly the only one (1500 tokens of 5 KB, 4 per token, 16 ranks 13.4 us
    // with entries picked by their number, 13.0 here). One vector load issued ahead of the keys (as uniform loads they become scalar loads that are
    // waited for one by one in the middle of the ranking)
    const bool all_own = FAN < 8 && K <= 64;
    const int own0 = indices[i0 + min(all_own ? lane : lane & (FAN - 1), K - 1)];
    int key[KEYS];
#pragma unroll
    for (int u = 0; u < KEYS; ++u) key[u] = indices[min(tid + u * BLK, S - 1)];
    V v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = x[(size_t)t * row_vecs + min(col + j * BLK, row_vecs - 1)];

    for (int g0 = 0; g0 < K; g0 += FAN) {
      // (a later group waits for its ids inside the branch: a wait at the place where the two paths
      // meet would cover the first group's row as well, which is requested behind its ids)
      int own = own0;
      if (!all_own && g0 > 0) own = first_use(indices[i0 + min(g0 + (lane & (FAN - 1)), K - 1)]);
      int mine[FAN];
#pragma unroll
      for (int g = 0; g < FAN; ++g) {
        const int k = min(g0 + g, K - 1);
        mine[g] = composite(__builtin_amdgcn_readlane(own, all_own ? k : g), i0 + k);
      }
      int cnt[FAN];
#pragma unroll
      for (int g = 0; g < FAN; ++g) cnt[g] = 0;
      auto consume = [&](const int (&k)[KEYS], int b) {
#pragma unroll
        for (int u = 0; u < KEYS; ++u) {
          // Keys past the end of the stream are left out where a lane has two vectors of the row: 188 tokens of 14 KB, 8 per
          // token 5.57 us, 6.49 with them. With one, the branches cost more than the compares: 400 of 5 KB, 4 per token, 16 ranks
          // 4.44 with branches, 4.25 here; 1000 8.38 / 8.06.
          if (NV > 1 && b + u * BLK >= S) break;
          const int i2 = b + tid + u * BLK;
          const int ck = i2 < S ? composite(k[u], i2) : INT_MAX;
#pragma unroll
          for (int g = 0; g < FAN; ++g) cnt[g] += (int)(ck < mine[g]);
        }
      };
      consume(key, 0);
      for (int b = KEYS * BLK; b < S; b += KEYS * BLK) {
        int more[KEYS];
#pragma unroll
        for (int u = 0; u < KEYS; ++u) more[u] = indices[min(b + tid + u * BLK, S - 1)];
        consume(more, b);
      }

#pragma unroll
      for (int h = 0; h < PAIRS; ++h) {
        const int sum = wave_sum(cnt[h] | (cnt[h + PAIRS] << 16));
        if (lane == 0) part[wave * PAIRS + h] = sum;
      }
      lds_barrier();
      if (wave == 0) {  // row h of 16 lanes adds up pair h of every wave
        const int h = lane >> 4, w = lane & 15;
        int sum = w < NW && h < PAIRS ? part[w * PAIRS + h] : 0;
        sum = dpp_add<0x111, 0xf>(sum);
        sum = dpp_add<0x112, 0xf>(sum);
        sum = dpp_add<0x114, 0xf>(sum);
        sum = dpp_add<0x118, 0xf>(sum);
        if (w == 15 && h < PAIRS) total[h] = sum;
      }
      lds_barrier();
      // no third barrier: `part` is next written before a barrier that wave 0 only reaches after
      // it has read `part`, and `total` after a barrier every wave reaches after reading it
      int slot[FAN];
#pragma unroll
      for (int h = 0; h < PAIRS; ++h) {
        const int both = total[h];
        slot[h] = both & 0xffff;
        slot[h + PAIRS] = (int)((unsigned)both >> 16);
      }
      const int live = min(FAN, K - g0);
#pragma unroll
      for (int g = 0; g < FAN; ++g) {
#pragma unroll
        for (int j = 0; j < NV; ++j)
          if (g < live && col + j * BLK < row_vecs)
            row_store<MOE_A2A_STORE_SEND>(send_buf + (size_t)slot[g] * row_vecs + col + j * BLK, v[j]);
      }
      if (c == 0 && tid < live * META) {
        const int g = tid / META, f = tid - g * META;
        int mine_slot = 0, e = 0;
#pragma unroll
        for (int gg = 0; gg < FAN; ++gg) {
          mine_slot = gg == g ? slot[gg] : mine_slot;
          if (FAN < 8) e = gg == g ? __builtin_amdgcn_readlane(own, all_own ? min(g0 + gg, K - 1) : gg) : e;
        }
        if (FAN == 8) e = __shfl(own, g, 64);  // (lanes 0 .. FAN-1 of wave 0 are among the active ones)
        const int i = i0 + g0 + g;
        const int m = f == 0 ? e : f == 1 ? rank : f == 2 ? t : f == 3 ? g0 + g : 0;
        send_meta[(size_t)mine_slot * META + f] = m;
        if (f == 0 && send_slot) send_slot[i] = mine_slot;
      }
    }
  }
}

// The fan-out of a job with few entries: every wave holds all their keys (KEYS per lane) and ranks entries of its own
// (wave, wave + 4, ...), so that one barrier makes the slots known, where the kernels above add partial counts over the
// waves, for two entries at a time. Such a job is bound by the chain of steps from the launch to the last store, and what
// counts in it is the code that a wave runs through: KEYS is the smallest of 2, 4, 8, 12 and 16 that holds the entries, and
// nothing in the scan is skipped by a branch (with up to 16 keys per lane skipped in this way 3.23 us instead of 2.57 for
// the 32 entries of 12 KB below, 2.83 with up to 8). us, one launch after another in a graph, before / here: 72 entries
// of 1 KB, 6 per token 4.38 / 2.77, 32 of 12 KB, 2 per token 3.92 / 2.57, 500 of 5.8 KB, 4 per token 3.85 / 3.30, 720 of
// 2 KB, 8 per token 5.27 / 3.61, 800 of 14 KB, 8 per token 6.17 / 4.66. With more keys, or more pieces of rows that each hold
// them, they go through the unit's one path to L1 too often (send_way).
template <typename V, int KEYS, bool POW2>
__global__ __launch_bounds__(BLOCK) void dispatch_few_kernel(
    const V* __restrict__ x, const int* __restrict__ indices, int T, int K, int W, int chunks, int row_vecs, int E,
    uint32_t magic, int nle_shift, int order_bits, int rank,
    V* __restrict__ send_buf, int* __restrict__ send_meta, int* __restrict__ send_counts,
    int* __restrict__ send_slot) {
  __shared__ int slots[FEW_MAX_K], ids[FEW_MAX_K];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int S = T * K;
  auto klass = [&](int e) {
    const int d = POW2 ? e >> nle_shift : (int)__umulhi((uint32_t)e, magic);
    return (uint32_t)e >= (uint32_t)E ? W : d;
  };
  // (as above)
  auto composite = [&](int e, int i) { return (klass(e) << order_bits) | i; };
  int key[KEYS];
  auto fetch = [&] {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) key[u] = indices[min(lane + u * 64, S - 1)];
  };

  if ((int)blockIdx.x < W) {
    if (wave > 0) return;
    fetch();
    int n = 0;
#pragma unroll
    for (int u = 0; u < KEYS; ++u) n += __popcll(__ballot(lane + u * 64 < S && klass(key[u]) == (int)blockIdx.x));
    if (lane == 0) send_counts[blockIdx.x] = n;
    return;
  }

  const int q = blockIdx.x - W;
  const int t = chunks == 1 ? q : q / chunks, c = q - t * chunks;
  const int i0 = t * K, col = c * BLOCK + tid;
  const int own = indices[i0 + min(lane, K - 1)];
  fetch();
  const V v = x[(size_t)t * row_vecs + min(col, row_vecs - 1)];
#pragma unroll
  for (int u = 0; u < KEYS; ++u)
    key[u] = lane + u * 64 < S ? composite(key[u], lane + u * 64) : INT_MAX;
  for (int k = wave; k < K; k += NWAVES) {
    const int mine = composite(__builtin_amdgcn_readlane(own, k), i0 + k);
    int slot = 0;
#pragma unroll
    for (int u = 0; u < KEYS; ++u) slot += __popcll(__ballot(key[u] < mine));
    if (lane == 0) slots[k] = slot;
  }
  if (wave == 0 && lane < K) ids[lane] = own;
  lds_barrier();
  const int slot_of = slots[min(lane, K - 1)];
  for (int k = 0; k < K; ++k) {
    const int slot = __builtin_amdgcn_readlane(slot_of, k);
    if (col < row_vecs) row_store<MOE_A2A_STORE_SEND>(send_buf + (size_t)slot * row_vecs + col, v);
  }
  if (c == 0) {
    for (int m = tid; m < K * META; m += BLOCK) {
      const int k = m / META, f = m - k * META;
      const int slot = slots[k];
      send_meta[(size_t)slot * META + f] = f == 0 ? ids[k] : f == 1 ? rank : f == 2 ? t : f == 3 ? k : 0;
      if (f == 0 && send_slot) send_slot[i0 + k] = slot;
    }
  }
}

// The fan-out of a long stream: a workgroup owns ROWS consecutive tokens, a wave each, and ranks all of their entries in one
// pass over the keys, which costs the same for one entry as for 64: a lane counts its keys by destination in bytes packed
// into two words (up to 8 destinations, up to 255 keys per lane), apart for the keys ahead of the workgroup's first entry
// and the others. From these come where every destination's rows begin and how many of them lie ahead; the workgroup's own
// entries, one per lane of every wave, add the lanes before them with the same destination. The kernels above compare every
// key with every entry of one token, which grows with the square of the stream. What bounds this one is the stores of the
// rows, below some 4 KB per token the passes over the keys (4 bytes and nine instructions each, 2 KB ahead). us, before / here:
// 2787 tokens of 4 KB, 4 per token 33.4 / 14.6 (the rows alone 10.4 at 5.3 TB/s), 4096 of 14 KB, 8 per token 118.9 / 102.5
// (99.7), 4096 of 512 bytes, 8 per token 109 / 23.6, 1500 of 1 KB, 6 per token 17.6 / 7.3, 700 of 3.4 KB, 5 per token 8.1 / 5.6,
// 3626 of 8150 bytes, moved by elements, 3 per token 109 / 37.
template <typename V, int NVW, bool POW2>
__global__ __launch_bounds__(64 * ROWS) void dispatch_block_kernel(
    const V* __restrict__ x, const int* __restrict__ indices, int T, int K, int W, int chunks, int row_vecs, int E,
    uint32_t magic, int nle_shift, int rank,
    V* __restrict__ send_buf, int* __restrict__ send_meta, int* __restrict__ send_counts,
    int* __restrict__ send_slot) {
  static_assert(64 * ROWS == BLOCK, "a wave per token");
  constexpr int KEYS = 8, BATCH = KEYS * BLOCK, WORDS = 4;  // 16-bit pairs: destinations 0 and 2, 1 and 3, 4 and 6, 5 and 7
  __shared__ int part[ROWS][2 * WORDS];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int S = T * K;
  const int q = xcd_contiguous(blockIdx.x, gridDim.x);
  const int grp = chunks == 1 ? q : q / chunks, c = q - grp * chunks;
  const int t0 = grp * ROWS, i0 = t0 * K, own = min(ROWS, T - t0) * K;  // (own <= 64)
  auto klass = [&](int e) {
    const int d = POW2 ? e >> nle_shift : (int)__umulhi((uint32_t)e, magic);
    return (uint32_t)e >= (uint32_t)E ? BLOCK_RANKS : d;
  };
  const int mine = indices[i0 + min(lane, own - 1)];
  int key[KEYS];
  auto fetch = [&](int b) {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) key[u] = indices[min(b + tid + u * BLOCK, S - 1)];
  };
  fetch(0);
  issued_here();
  const int t = t0 + wave, base = c * (64 * NVW);
  WavePayload<V, NVW> p;
  p.load(x + (size_t)min(t, T - 1) * row_vecs, base, row_vecs, lane);

  uint32_t ahead[2] = {}, others[2] = {};  // destinations 0..3 and 4..7, a byte each
  auto count = [&](uint32_t (&n)[2], int b, int from, int to) {  // the batch's keys in [from, to)
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      const int i = b + tid + u * BLOCK;
      const int d = (i >= from) & (i < to) ? klass(key[u]) : BLOCK_RANKS;
      const uint32_t one = 1u << ((d & 3) * 8);
      n[0] += d < 4 ? one : 0;
      n[1] += (uint32_t)(d - 4) < 4u ? one : 0;
    }
  };
  for (int b = 0; b < S; b += BATCH) {
    if (b > 0) fetch(b);
    if (b < i0) count(ahead, b, 0, i0);
    if (b + BATCH > i0) count(others, b, i0, S);
  }
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int a0 = wave_sum((int)(ahead[w] & 0x00ff00ffu)), a1 = wave_sum((int)((ahead[w] >> 8) & 0x00ff00ffu));
    const int o0 = wave_sum((int)(others[w] & 0x00ff00ffu)), o1 = wave_sum((int)((others[w] >> 8) & 0x00ff00ffu));
    if (lane == 0) {
      part[wave][w * 2] = a0;
      part[wave][w * 2 + 1] = a1;
      part[wave][WORDS + w * 2] = o0;
      part[wave][WORDS + w * 2 + 1] = o1;
    }
  }
  lds_barrier();
  // lane d: entries of destination d ahead of the workgroup's, and all of them
  const int word = (lane >> 2 & 1) * 2 + (lane & 1), half = (lane >> 1 & 1) * 16;
  int before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < ROWS; ++w) {
    before += part[w][word] >> half & 0xffff;
    total += part[w][WORDS + word] >> half & 0xffff;
  }
  const bool is_rank = lane < W;
  before = is_rank ? before : 0;
  total = is_rank ? total + before : 0;
  const int upto = wave_inclusive_scan(total), all_before = wave_inclusive_scan(before);
  // (entries without a destination come last: in lane BLOCK_RANKS, behind all ranks)
  const int first = lane < BLOCK_RANKS ? upto - total + before : upto + i0 - all_before;
  if (blockIdx.x == 0 && wave == 0 && is_rank) send_counts[lane] = total;
  const int d = lane < own ? klass(mine) : -1;
  int slot = __shfl(first, d < 0 ? 0 : d, 64);
#pragma unroll
  for (int r = 0; r <= BLOCK_RANKS; ++r) {
    const unsigned long long same = __ballot(d == r);
    slot += d == r ? __popcll(same & ((1ull << lane) - 1)) : 0;
  }

  if (t >= T) return;
  for (int k = 0; k < K; ++k) {
    const int to = __builtin_amdgcn_readlane(slot, wave * K + k);
    p.template store<MOE_A2A_STORE_SEND>(send_buf + (size_t)to * row_vecs, base, row_vecs, lane);
  }
  if (c == 0) {
    for (int b = 0; b < K * META; b += 64) {
      const int m = b + lane, k = min(m / META, K - 1), f = m - k * META;
      const int to = __shfl(slot, wave * K + k, 64), e = __shfl(mine, wave * K + k, 64);
      if (m < K * META) {
        send_meta[(size_t)to * META + f] = f == 0 ? e : f == 1 ? rank : f == 2 ? t : f == 3 ? k : 0;
        if (f == 0 && send_slot) send_slot[t * K + k] = to;
      }
    }
  }
}

// The same for longer streams yet: a workgroup of sixteen waves owns `own_tokens` tokens (of at most 64 entries), so that fewer of them
// pass over all keys, and its waves take pieces of 64 vectors of the tokens' rows in turn, along the stream, so that few places of
// the send buffer are open at a time. What bounds it is the stores of the rows, of short ones the keys. us, dispatch_block_kernel /
// here: 3090 tokens of 1.1 KB, 4 per token 13.5 / 8.8; 3123 of 1 KB, 2 each 9.9 / 6.8; 3630 of 1.5 KB, 8 each 24.8 / 19.4; 3554 of 8.6 KB, 2
// each 21.4 / 18.0; 3001 of 12 KB, 5 each 42.9 / 38.7; 4096 of 14 KB, 8 each, behind the other stages, 118 / 111.
template <bool POW2>
__global__ __launch_bounds__(LONG_BLOCK) void dispatch_long_kernel(
    const b128* __restrict__ x, const int* __restrict__ indices, int T, int K, int W, int own_tokens, Pieces pieces, int row_vecs,
    int E, uint32_t magic, int nle_shift, int rank,
    b128* __restrict__ send_buf, int* __restrict__ send_meta, int* __restrict__ send_counts,
    int* __restrict__ send_slot) {
  constexpr int KEYS = 8, BATCH = KEYS * LONG_BLOCK, WORDS = 4, NW = LONG_BLOCK / 64;
  __shared__ int part[2 * WORDS][NW];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int S = T * K;
  const int t0 = blockIdx.x * own_tokens, i0 = t0 * K, tokens = min(own_tokens, T - t0), own = tokens * K;  // (own <= 64)
  auto klass = [&](int e) {
    const int d = POW2 ? e >> nle_shift : (int)__umulhi((uint32_t)e, magic);
    return (uint32_t)e >= (uint32_t)E ? BLOCK_RANKS : d;
  };
  const int mine = indices[i0 + min(lane, own - 1)];
  int key[KEYS];
  auto fetch = [&](int b) {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) key[u] = indices[min(b + tid + u * LONG_BLOCK, S - 1)];
  };
  fetch(0);
  issued_here();
  const int items = tokens * pieces.per_row;
  auto vector_of = [&](int q) {
    const int tl = pieces.row_of(q), at = (q - tl * pieces.per_row) * 64 + lane;
    return x[(size_t)(t0 + tl) * row_vecs + min(at, row_vecs - 1)];
  };
  b128 v{};
  if (wave < items) v = vector_of(wave);

  uint32_t ahead[2] = {}, others[2] = {};
  auto count = [&](uint32_t (&n)[2], int b, int from, int to) {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      const int i = b + tid + u * LONG_BLOCK;
      const int d = (i >= from) & (i < to) ? klass(key[u]) : BLOCK_RANKS;
      const uint32_t one = 1u << ((d & 3) * 8);
      n[0] += d < 4 ? one : 0;
      n[1] += (uint32_t)(d - 4) < 4u ? one : 0;
    }
  };
  for (int b = 0; b < S; b += BATCH) {
    if (b > 0) fetch(b);
    if (b < i0) count(ahead, b, 0, i0);
    if (b + BATCH > i0) count(others, b, i0, S);
  }
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int a0 = wave_sum((int)(ahead[w] & 0x00ff00ffu)), a1 = wave_sum((int)((ahead[w] >> 8) & 0x00ff00ffu));
    const int o0 = wave_sum((int)(others[w] & 0x00ff00ffu)), o1 = wave_sum((int)((others[w] >> 8) & 0x00ff00ffu));
    if (lane == 0) {
      part[w * 2][wave] = a0;
      part[w * 2 + 1][wave] = a1;
      part[WORDS + w * 2][wave] = o0;
      part[WORDS + w * 2 + 1][wave] = o1;
    }
  }
  lds_barrier();
  const int word = (lane >> 2 & 1) * 2 + (lane & 1), half = (lane >> 1 & 1) * 16;
  int before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    before += part[word][w] >> half & 0xffff;
    total += part[WORDS + word][w] >> half & 0xffff;
  }
  const bool is_rank = lane < W;
  before = is_rank ? before : 0;
  total = is_rank ? total + before : 0;
  const int upto = wave_inclusive_scan(total), all_before = wave_inclusive_scan(before);
  const int first = lane < BLOCK_RANKS ? upto - total + before : upto + i0 - all_before;
  if (blockIdx.x == 0 && wave == 0 && is_rank) send_counts[lane] = total;
  const int d = lane < own ? klass(mine) : -1;
  int slot = __shfl(first, d < 0 ? 0 : d, 64);
#pragma unroll
  for (int r = 0; r <= BLOCK_RANKS; ++r) {
    const unsigned long long same = __ballot(d == r);
    slot += d == r ? __popcll(same & ((1ull << lane) - 1)) : 0;
  }

  for (int b = wave * 64; b < own * META; b += LONG_BLOCK) {
    const int m = b + lane, k = min(m / META, own - 1), f = m - k * META;
    const int to = __shfl(slot, k, 64), e = __shfl(mine, k, 64);
    if (m < own * META) {
      const int tl = k / K;
      send_meta[(size_t)to * META + f] = f == 0 ? e : f == 1 ? rank : f == 2 ? t0 + tl : f == 3 ? k - tl * K : 0;
      if (f == 0 && send_slot) send_slot[i0 + k] = to;
    }
  }
  for (int q = wave; q < items;) {
    const int tl = pieces.row_of(q), at = (q - tl * pieces.per_row) * 64 + lane;
    const b128 out = v;
    q += NW;
    if (q < items) v = vector_of(q);
    for (int k = 0; k < K; ++k) {
      const int to = __builtin_amdgcn_readlane(slot, tl * K + k);
      if (at < row_vecs) row_store<MOE_A2A_STORE_SEND>(send_buf + (size_t)to * row_vecs + at, out);
    }
  }
}

// ---------------------------------------------------------------- send plan (counts, offsets, maps)
//
// The stable counting sort of stage 1 made explicit, for callers that want the
// plan without moving rows (a sender that writes into a peer's buffer, a
// debugger): rows per destination rank and per expert, the exclusive offsets
// of the destinations, and both index maps. One workgroup of 16 waves walks
// the (t, k) stream in tiles of 1024 entries:
//   pass 1  per-wave privatised LDS histograms of the destinations (no two
//           waves touch the same counters), one shared LDS histogram of the
//           expert ids; a wave64 exclusive scan turns the destination totals
//           into offsets;
//   pass 2  inside a wave, an entry's rank among the earlier lanes with the
//           same destination comes from a ballot per destination present in
//           the wave; the waves of a tile are ordered by a prefix over their
//           per-destination counts, tiles by a running base per destination.
// slot(i) = offset[d] + #earlier entries with destination d — the order of
// all2all/reference.py:79-86,93.

constexpr int PLAN_BLOCK = 1024;
constexpr int PLAN_WAVES = PLAN_BLOCK / 64;
constexpr int PLAN_MAX_RANKS = 64;      // destinations kept per wave in LDS
constexpr int PLAN_MAX_EXPERTS = 8192;  // shared expert histogram in LDS

__global__ __launch_bounds__(PLAN_BLOCK) void plan_send_kernel(
    const int* __restrict__ indices, int S, int nle, int E, int W, uint32_t magic,
    int* __restrict__ rank_counts, int* __restrict__ rank_offsets, int* __restrict__ expert_counts,
    int* __restrict__ dst_slot, int* __restrict__ src_entry) {
  __shared__ int wave_hist[PLAN_WAVES][PLAN_MAX_RANKS];
  __shared__ int base[PLAN_MAX_RANKS];        // next free slot of each destination
  __shared__ int expert_hist[PLAN_MAX_EXPERTS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const unsigned long long lanes_below = lane == 0 ? 0ull : (~0ull >> (64 - lane));

  auto dest_of = [&](int e) { return nle == 1 ? e : (int)__umulhi((uint32_t)e, magic); };
  auto in_range = [&](int e) { return (e >= 0) & (e < E); };

  // ---- pass 1: histograms
  for (int i = tid; i < PLAN_WAVES * PLAN_MAX_RANKS; i += PLAN_BLOCK) (&wave_hist[0][0])[i] = 0;
  for (int i = tid; i < E; i += PLAN_BLOCK) expert_hist[i] = 0;
  lds_barrier();
  for (int b = 0; b < S; b += PLAN_BLOCK) {
    const int i = b + tid;
    const int e = i < S ? indices[i] : -1;
    if (in_range(e)) {
      atomicAdd(&expert_hist[e], 1);
      // lanes of one wave that share a destination add their count once
      const int d = dest_of(e);
      unsigned long long todo = __ballot(1);
      while (todo) {
        const int leader = __builtin_amdgcn_readfirstlane(d);
        const unsigned long long same = __ballot(d == leader);
        if (d == leader) {
          if ((same & lanes_below) == 0) wave_hist[wave][leader] += __popcll(same);
          break;
        }
        todo &= ~same;
      }
    }
  }
  lds_barrier();
  for (int i = tid; i < E; i += PLAN_BLOCK) expert_counts[i] = expert_hist[i];
  if (wave == 0) {  // destination totals -> exclusive offsets with a wave64 scan
    int total = 0;
    if (lane < W) {
#pragma unroll
      for (int w = 0; w < PLAN_WAVES; ++w) total += wave_hist[w][lane];
    }
    const int incl = wave_inclusive_scan(total);
    if (lane < W) {
      rank_counts[lane] = total;
      rank_offsets[lane] = incl - total;
      base[lane] = incl - total;
    }
    if (lane == W - 1 || (W == 64 && lane == 63)) rank_offsets[W] = incl;
  }
  lds_barrier();

  // ---- pass 2: stable slots, tile by tile
  for (int b = 0; b < S; b += PLAN_BLOCK) {
    for (int i = tid; i < PLAN_WAVES * PLAN_MAX_RANKS; i += PLAN_BLOCK) (&wave_hist[0][0])[i] = 0;
    lds_barrier();
    const int i = b + tid;
    const int e = i < S ? indices[i] : -1;
    const bool ok = in_range(e);
    const int d = ok ? dest_of(e) : -1;
    int rank_in_wave = 0;
    unsigned long long todo = __ballot(ok);
    while (todo) {  // every lane of the wave runs the same number of rounds
      const int first = __ffsll((long long)todo) - 1;
      const int leader = __builtin_amdgcn_readlane(d, first);
      const unsigned long long same = __ballot(ok && d == leader);
      if (ok && d == leader) {
        rank_in_wave = __popcll(same & lanes_below);
        if (rank_in_wave == 0) wave_hist[wave][leader] = __popcll(same);
      }
      todo &= ~same;
    }
    lds_barrier();
    if (ok) {
      int before = base[d];
      for (int w = 0; w < wave; ++w) before += wave_hist[w][d];
      const int slot = before + rank_in_wave;
      dst_slot[i] = slot;
      src_entry[slot] = i;
    }
    lds_barrier();
    if (tid < W) {
      int t = 0;
#pragma unroll
      for (int w = 0; w < PLAN_WAVES; ++w) t += wave_hist[w][tid];
      base[tid] += t;
    }
    lds_barrier();
  }
}

// ---------------------------------------------------------------- stage 2: dispatch, receive side
//
// grid = nle counting workgroups (rows per local expert) followed by one
// workgroup per (group of ROWS received rows, chunk). Row i goes to expert
// le = e % nle at position #{earlier rows of the same expert}.
//
// `hint_rows` rows of recv_buf / recv_meta are readable whatever the counts
// say. A workgroup whose rows lie below that bound issues all its loads before
// it knows the true row count R (the counts are loaded at the same time) and
// only the stores wait for R; rows at or past R are loaded and dropped. Counts
// that add up to more than `capacity_rows` (what the buffers hold) are cut off there.

//
// PLAN (W <= 64): the counting workgroup of expert le also splits its rows by
// source rank and writes, for every source s, two ints at plan[(le*W + s)*2]:
//   [0] the position inside expert le at which the rows from s start (inside an
//       expert, rows lie in arrival order, that is by source rank), and
//   [1] the row of the send-back stream of stage 3 that the first of them goes
//       to: #{rows from lower sources} + #{rows from s in lower experts}.
// Stage 3 then places a row without scanning any keys.

constexpr int PLAN_INTS = 2;  // ints per (local expert, source rank) of the send-back plan

// Long streams. The movers below rank a row by counting the keys ahead of it, and every
// workgroup of four rows repeats that pass: the key loads grow with the square of the row count
// (at 8192 rows they are two thirds of the payload). For long streams the positions are worked
// out by a launch of their own, one workgroup of 1024 lanes per tile of 1024 rows: an LDS
// histogram (atomics; the order of the adds does not matter) of the experts of all rows ahead of
// the tile, then inside the tile a row's rank among the earlier lanes of its wave with the same
// expert (the set of those lanes from one ballot per bit of the expert number), the waves ordered
// by a prefix over their per-expert counts. row_pos[i] = #{rows before i with the same local expert}, which is
// the slot the reference's running counter hands out (all2all/reference.py:140-146). The movers
// then read one int per row instead of scanning. COMPACT: plus where the row's expert starts, from the same counts
// of all rows. Stage 2, us with scans / planned: 10000 rows of 512 bytes, padded 22.0 / 15.5, compact 43.6 / 16.6; 20000 of 3 KB 67.6 /
// 31.8 and 147 / 33; 7500 of 14 KB 42.5 / 33.3 and 53.5 / 34.5; 4096 of 3 KB 8.9 / 9.6 and 12.9 / 10.4, of 14 KB 19.3 / 21.9 and 23.0 / 23.0;
// 3000 of 1.3 KB compact 9.7 / 9.7, of 14 KB 14.6 / 19.2.
constexpr int RPLAN_BLOCK = 1024;
constexpr int RPLAN_WAVES = RPLAN_BLOCK / 64;
constexpr int RPLAN_MAX_EXPERTS = 256;  // local experts with a counter per wave in LDS
constexpr int RPLAN_SPREAD = 32;

template <bool COMPACT>
__global__ __launch_bounds__(RPLAN_BLOCK) void plan_recv_kernel(
    const int* __restrict__ recv_meta, const int* __restrict__ recv_counts, int W, int hint_rows,
    int capacity_rows, int nle, uint32_t magic, int expert_bits, int* __restrict__ row_pos) {
  __shared__ int ahead[RPLAN_MAX_EXPERTS];                 // rows of each expert before the tile, in several copies and then summed
  __shared__ int all[COMPACT ? RPLAN_MAX_EXPERTS : 1];      // rows of each expert, likewise, and then where they start
  __shared__ int in_wave[RPLAN_WAVES][RPLAN_MAX_EXPERTS];   // rows of each expert in each wave of the tile
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const unsigned long long lanes_below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  int R = -1;  // not known yet
  // Lanes of a wave that count for the same expert do so one after the other, so few experts get several copies of their counters.
  // Stage 2 of 7500 rows of 512 bytes, us with one copy / these: one expert, padded 16.0 / 12.6, compact 22.8 / 13.6; copies beyond that
  // only have to be summed (32 experts with 32 copies, 4096 rows 9.3 / 10.5).
  int copies = 1;
  while (copies * nle < RPLAN_SPREAD) copies *= 2;
  const int my_copy = (lane & (copies - 1)) * nle;
  auto rows = [&] { return min(sum_counts(recv_counts, W, capacity_rows), capacity_rows); };
  for (int first = blockIdx.x * RPLAN_BLOCK;; first += gridDim.x * RPLAN_BLOCK) {
    // A tile that lies wholly below the readable bound sends its loads off before the row
    // count is known: the counts travel at the same time (one round trip instead of three).
    const bool early = R < 0 && first + RPLAN_BLOCK <= hint_rows;
    if (!early) {
      if (R < 0) R = rows();
      if (first >= R) break;
    }
    const int last = early ? first + RPLAN_BLOCK - 1 : R - 1;  // last row that may be read
    const int i = first + tid;
    const int mine = recv_meta[(size_t)min(i, last) * META];
    // the first keys: of rows ahead, or (COMPACT) of all that may be read
    constexpr int BATCH = SCAN_UNROLL * RPLAN_BLOCK;
    const int got = min(BATCH, COMPACT ? (early ? hint_rows : R) : first);
    int e2[SCAN_UNROLL];
    auto fetch = [&](int from, int to) {
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) e2[u] = recv_meta[(size_t)min(from + tid + u * RPLAN_BLOCK, max(to - 1, 0)) * META];
    };
    fetch(0, got);
    for (int j = tid; j < copies * nle; j += RPLAN_BLOCK) {
      ahead[j] = 0;
      if constexpr (COMPACT) all[j] = 0;
    }
    for (int j = tid; j < RPLAN_WAVES * RPLAN_MAX_EXPERTS; j += RPLAN_BLOCK) (&in_wave[0][0])[j] = 0;
    if (R < 0) R = rows();
    lds_barrier();
    if (first >= R) break;  // (uniform over the workgroup)
    const bool ok = i < R;
    const int le = floormod(mine, nle, magic);
    auto count = [&](int from, int to) {
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) {
        const int at = from + tid + u * RPLAN_BLOCK;
        if (at < to) {
          const int le2 = floormod(e2[u], nle, magic);
          if (!COMPACT || at < first) atomicAdd(&ahead[my_copy + le2], 1);
          if constexpr (COMPACT) atomicAdd(&all[my_copy + le2], 1);
        }
      }
    };
    const int end = COMPACT ? R : first;
    count(0, min(got, end));
    for (int b = got; b < end; b += BATCH) {
      fetch(b, end);
      count(b, end);
    }
    // the lanes of this wave with the same expert, from one ballot per bit of the expert number
    // (a loop over the experts present in the wave costs a round per expert: 3.8 us of issue
    // slots with 32 experts and four waves per SIMD)
    unsigned long long same = __ballot(ok);
    for (int b = 0; b < expert_bits; ++b) {
      const bool set = (le >> b) & 1;
      const unsigned long long with_bit = __ballot(set);
      same &= set ? with_bit : ~with_bit;
    }
    const int rank_in_wave = __popcll(same & lanes_below);
    if (ok && rank_in_wave == 0) in_wave[wave][le] = __popcll(same);
    lds_barrier();
    if (copies > 1) {
      if (tid < nle) {
        int n = 0, n_all = 0;
        for (int c = tid; c < copies * nle; c += nle) {
          n += ahead[c];
          if constexpr (COMPACT) n_all += all[c];
        }
        ahead[tid] = n;
        if constexpr (COMPACT) all[tid] = n_all;
      }
      lds_barrier();
    }
    if constexpr (COMPACT) {  // where each expert's rows start: a prefix by one wave, four experts per lane
      if (wave == 0) {
        int n[RPLAN_MAX_EXPERTS / 64], sum = 0;
#pragma unroll
        for (int j = 0; j < RPLAN_MAX_EXPERTS / 64; ++j) {
          const int x = lane * (RPLAN_MAX_EXPERTS / 64) + j;
          n[j] = x < nle ? all[x] : 0;
          sum += n[j];
        }
        int before = wave_inclusive_scan(sum) - sum;
#pragma unroll
        for (int j = 0; j < RPLAN_MAX_EXPERTS / 64; ++j) {
          const int x = lane * (RPLAN_MAX_EXPERTS / 64) + j;
          if (x < nle) all[x] = before;
          before += n[j];
        }
      }
      lds_barrier();
    }
    if (ok) {
      int pos = ahead[le] + rank_in_wave;
      if constexpr (COMPACT) pos += all[le];
      for (int w = 0; w < wave; ++w) pos += in_wave[w][le];
      row_pos[i] = pos;
    }
    lds_barrier();  // the tables are cleared again by the next tile
  }
}

// COMPACT: the compact layout, the experts' rows back to back, row pos of expert le at offset[le] + pos with offset =
// exclusive prefix of the rows per expert (padded: row pos of expert le at le * max_recv + pos, all2all/reference.py:127-136).
// A row's place is then the number of rows of lower experts anywhere in the stream plus the earlier rows of its own
// expert (one pass over all keys); `max_recv` is the number of rows the compact buffers hold, and the counting
// workgroups also write the offsets.

// A workgroup that plans expert blockIdx.x: its rows, where every source's run of them starts inside the expert and in the
// send-back stream, and in the compact layout where the expert starts.
template <bool COMPACT, int UNROLL>
__device__ __forceinline__ void plan_expert(
    const int* __restrict__ recv_meta, const int* __restrict__ recv_counts, int W, int hint_rows, int nle, int capacity_rows,
    uint32_t magic, int* __restrict__ expert_num_tokens, int* __restrict__ plan, int* __restrict__ expert_offsets) {
  // Its keys go out with the counts, as far as the hint says that they can be read. A lane per source counts by the
  // ballots of 64 rows, cut to the rows of its source.
  __shared__ int sums[ROWS][2][64];  // per wave and source: rows of this expert, rows of lower experts
  constexpr int BLK = 64 * ROWS;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int me = blockIdx.x, first_of_wave = __builtin_amdgcn_readfirstlane(wave) * 64;
  const int raw_count = recv_counts[min(lane, W - 1)];
  int e2[UNROLL];
  auto fetch = [&](int b, int end) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) e2[u] = recv_meta[(size_t)min(b + tid + u * BLK, end - 1) * META];
  };
  const int early = min(hint_rows, UNROLL * BLK);
  if (early > 0) fetch(0, early);
  const int mine = lane < W ? min(max(first_use(raw_count), 0), capacity_rows) : 0;
  const int incl = wave_inclusive_scan(mine);
  const int R = min(__builtin_amdgcn_readlane(incl, 63), capacity_rows);
  int here = 0, below = 0;
  auto count = [&](int b, int end) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int row0 = b + u * BLK + first_of_wave;
      if (row0 >= end) break;
      const int le2 = floormod(e2[u], nle, magic);
      const bool there = row0 + lane < end;
      auto lanes_from = [&](int row) {
        const int n = row - row0;
        return n <= 0 ? ~0ull : n >= 64 ? 0ull : ~0ull << n;
      };
      const unsigned long long own = lanes_from(incl - mine) & ~lanes_from(incl);
      here += __popcll(__ballot(there && le2 == me) & own);
      below += __popcll(__ballot(there && le2 < me) & own);
    }
  };
  count(0, min(early, R));
  for (int b = early; b < R; b += UNROLL * BLK) {
    fetch(b, R);
    count(b, R);
  }
  sums[wave][0][lane] = here;
  sums[wave][1][lane] = below;
  lds_barrier();
  if (wave == 0) {
#pragma unroll
    for (int w = 1; w < ROWS; ++w) {
      here += sums[w][0][lane];
      below += sums[w][1][lane];
    }
    const int upto = wave_inclusive_scan(here);
    if (lane < W) {
      int* out = plan + ((size_t)me * W + lane) * PLAN_INTS;
      out[0] = upto - here;
      out[1] = (incl - mine) + below;
    }
    if (lane == 63) expert_num_tokens[me] = upto;
    if constexpr (COMPACT) {  // rows of lower experts, from every source: where this expert's rows start
      const int lower = wave_sum(below), mine_all = __builtin_amdgcn_readlane(upto, 63);
      if (lane == 0) {
        expert_offsets[me] = lower;
        if (me == nle - 1) expert_offsets[nle] = lower + mine_all;
      }
    }
  }
}

// A workgroup that only counts the rows of expert blockIdx.x. `red` is ROWS ints of LDS.
template <bool COMPACT>
__device__ __forceinline__ void count_expert(
    const int* __restrict__ recv_meta, const int* __restrict__ recv_counts, int W, int nle, int capacity_rows, uint32_t magic,
    int* red, int* __restrict__ expert_num_tokens, int* __restrict__ expert_offsets) {
  const StridedKeys key{recv_meta, META};
  const int R = min(sum_counts(recv_counts, W, capacity_rows), capacity_rows);
  const int me = blockIdx.x, tid = threadIdx.x;
  int c = count_keys<64 * ROWS>(R, key, [=](int e, int) { return floormod(e, nle, magic) == me; });
  c = block_sum<ROWS>(c, red);
  if (tid == 0) expert_num_tokens[me] = c;
  if constexpr (COMPACT) {
    int lower = count_keys<64 * ROWS>(R, key, [=](int e, int) { return floormod(e, nle, magic) < me; });
    lower = block_sum<ROWS>(lower, red);
    if (tid == 0) {
      expert_offsets[me] = lower;
      if (me == nle - 1) expert_offsets[nle] = lower + c;
    }
  }
}

template <typename V, int NVW, bool PLAN, bool COMPACT, Store HOW, bool SHORT>
__global__ __launch_bounds__(64 * ROWS) void dispatch_recv_kernel(
    const V* __restrict__ recv_buf, const int* __restrict__ recv_meta,
    const int* __restrict__ recv_counts, int W, int hint_rows, int movers, int chunks, int row_vecs, int nle,
    int capacity_rows, uint32_t magic, int max_recv, int* __restrict__ expert_num_tokens,
    V* __restrict__ expert_x, int* __restrict__ expert_meta, int* __restrict__ plan, int* __restrict__ expert_offsets) {
  constexpr int UNROLL = HOW == PLAIN ? 4 : SCAN_UNROLL;  // (PLAIN: up to 1024 rows of elements, or of more than 64 experts)
  __shared__ int part[2 * ROWS * ROWS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const StridedKeys key{recv_meta, META};

  if constexpr (PLAN) {
    if ((int)blockIdx.x < nle) {
      plan_expert<COMPACT, UNROLL>(recv_meta, recv_counts, W, hint_rows, nle, capacity_rows, magic, expert_num_tokens, plan,
                                   expert_offsets);
      return;
    }
  }

  if ((int)blockIdx.x < nle) {
    count_expert<COMPACT>(recv_meta, recv_counts, W, nle, capacity_rows, magic, part, expert_num_tokens, expert_offsets);
    return;
  }

  int parity = 0;
  // One (group, chunk) item. `limit` rows may be read; R is evaluated after the
  // loads are issued (it is already known on every pass but the first).
  auto move = [&](int q, int limit, auto&& rows_known) {
    const int grp = chunks == 1 ? q : q / chunks, c = q - grp * chunks;
    const int i0 = grp * ROWS, i = i0 + wave;
    const int ic = min(i, limit - 1);
    const int base = c * (64 * NVW);

    int re[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) re[r] = recv_meta[(size_t)min(i0 + r, limit - 1) * META];
    int m = 0;
    if (c == 0 && lane < META) m = recv_meta[(size_t)ic * META + lane];
    // only rows before the group's last row can precede any of its rows in its expert; the rows of
    // lower experts, which the compact layout puts ahead of it, lie anywhere in the stream
    RowsScan<StridedKeys, SHORT, UNROLL> scan(COMPACT ? limit : min(i0 + ROWS - 1, limit), key);
    WavePayload<V, NVW> p;
    p.load(recv_buf + (size_t)ic * row_vecs, base, row_vecs, lane);

    const int R = rows_known();
    int rle[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) rle[r] = floormod(re[r], nle, magic);
    int cnt[ROWS];
    auto precedes = [&](int r, int e2, int i2) {
      const int le2 = floormod(e2, nle, magic);
      if constexpr (COMPACT) return (le2 < rle[r]) | ((le2 == rle[r]) & (i2 < i0 + r));
      else return (le2 == rle[r]) & (i2 < i0 + r);
    };
    scan.finish(key, COMPACT ? R : min(i0 + ROWS - 1, R), precedes, cnt);
    if constexpr (COMPACT) {
      // the scan began with the `limit` keys that were known to be readable; a stream longer than
      // that (a hint below the row count) has rows of lower experts behind them as well
      if (R > limit) scan.extend(key, limit, R, precedes, cnt);
    }
    const int pos = rows_reduce(cnt, part, parity++, wave, lane);

    if (i < R && pos < max_recv) {
      int le = 0;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) le = r == wave ? rle[r] : le;
      const size_t row = COMPACT ? (size_t)pos : (size_t)le * max_recv + pos;
      p.template store<HOW>(expert_x + row * row_vecs, base, row_vecs, lane);
      if (c == 0 && lane < META) expert_meta[row * META + lane] = m;
    }
    return R;
  };

  // Back to front: the workgroups launched first take the last rows. A compute unit serves the
  // memory requests of its workgroups in launch order, and the later a row lies in the stream
  // the more keys its group scans; the workgroups a unit serves last should be the cheap ones
  // (measured at 2048 rows of 14 KB: 11.7 -> 11.1 us; with a few workgroups more than two per
  // unit, which are then the ones with next to nothing to scan, 13.2 -> 11.6 us).
  int q = movers - 1 - ((int)blockIdx.x - nle);
  int R;
  // only groups that lie wholly below the bound: their rows can be read as they are
  const int hint_items = hint_rows / ROWS * chunks;
  if (W <= 64 && q < hint_items) {
    // The count travels with the rows: nothing touches the loaded value before the key and row
    // loads have been issued (first_use).
    const int raw_count = recv_counts[min(lane, W - 1)];
    R = move(q, hint_rows, [&] {
      const int my_count = lane < W ? min(max(first_use(raw_count), 0), capacity_rows) : 0;
      return min(wave_sum(my_count), capacity_rows);
    });
    q += movers;
  } else {
    R = min(sum_counts(recv_counts, W, capacity_rows), capacity_rows);
  }
  const int items = (R + ROWS - 1) / ROWS * chunks;
  for (; q < items; q += movers) move(q, R, [&] { return R; });
}

// The movers of a long stream, with the positions that plan_recv_kernel left: a wave per piece of 64 * NVW vectors of a row, in
// the order of the stream. Memory bounds it, and what shaped it is how few places of the streams are open at a time (planned_recv_vecs and
// RECV_PAST_BYTES, csrc/stream_rules.h): 32768 rows of 14 KB between the other stages 160 us with a workgroup on the same piece of four rows and plain
// loads of four vectors, 137 here (6.9 TB/s); what a graph of stages 1 to 4 loses without stage 2, its plan with it, 192 / 192 (203 with two vectors per
// lane); with a stage before and behind it 12000 rows of 4 KB 53.6 / 47.0.
template <typename V, int NVW, bool PLAN, bool COMPACT, Store HOW, bool PAST>
__global__ __launch_bounds__(64 * ROWS) void dispatch_recv_planned_kernel(
    const int* __restrict__ recv_meta, const int* __restrict__ row_pos, const int* __restrict__ recv_counts,
    const V* __restrict__ recv_buf, int W, int hint_rows, int movers, Pieces pieces, int row_vecs, int nle, int capacity_rows,
    uint32_t magic, int max_recv, V* __restrict__ expert_x, int* __restrict__ expert_meta,
    int* __restrict__ expert_num_tokens, int* __restrict__ plan, int* __restrict__ expert_offsets) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if ((int)blockIdx.x < nle) {
    if constexpr (PLAN) {
      plan_expert<COMPACT, SCAN_UNROLL>(recv_meta, recv_counts, W, hint_rows, nle, capacity_rows, magic, expert_num_tokens, plan,
                                        expert_offsets);
    } else {
      __shared__ int red[ROWS];
      count_expert<COMPACT>(recv_meta, recv_counts, W, nle, capacity_rows, magic, red, expert_num_tokens, expert_offsets);
    }
    return;
  }
  const bool lanes_hold_counts = W <= 64;
  const int raw_count = recv_counts[min(lane, W - 1)];
  int R = -1;  // not known yet
  auto rows = [&] {
    const int my_count = lane < W ? min(max(first_use(raw_count), 0), capacity_rows) : 0;
    return min(lanes_hold_counts ? wave_sum(my_count) : sum_counts(recv_counts, W, capacity_rows), capacity_rows);
  };
  for (int q = ((int)blockIdx.x - nle) * ROWS + wave;; q += movers * ROWS) {
    const int i = pieces.row_of(q), c = q - i * pieces.per_row, base = c * (64 * NVW);
    if (R >= 0 || i >= hint_rows) {  // (rows below the hint can be read before the count is known)
      if (R < 0) R = rows();
      if (i >= R) return;
    }
    const int e = recv_meta[(size_t)i * META], pos = row_pos[i];
    int m = 0;
    if (c == 0 && lane < META) m = recv_meta[(size_t)i * META + lane];
    WavePayload<V, NVW> p;
    p.template load<PAST>(unknown_origin(recv_buf + (size_t)i * row_vecs), base, row_vecs, lane);
    issued_here();
    if (R < 0) R = rows();
    if (i >= R) return;
    if ((uint32_t)pos < (uint32_t)max_recv) {
      const size_t row = COMPACT ? (size_t)pos : (size_t)floormod(e, nle, magic) * max_recv + pos;
      p.template store<HOW>(expert_x + row * row_vecs, base, row_vecs, lane);
      if (c == 0 && lane < META) expert_meta[row * META + lane] = m;
    }
  }
}

// The same for a short stream: every wave ranks a row of its own against all keys it needs (KEYS per lane, the fewest that
// hold hint_rows), with nothing to wait for but its own loads. As in dispatch_few_kernel the code that a wave runs through is
// what counts. us, one launch after another in a graph, before / here: 72 rows of 1 KB 3.33 / 2.54, 32 of 12 KB 3.87 / 3.09,
// 500 of 5.8 KB 4.11 / 3.44, 600 of 8 KB 4.45 / 4.11, 800 of 14 KB 6.17 / 5.75.
template <typename V, int NVW, int KEYS, bool COMPACT, Store HOW>
__global__ __launch_bounds__(64 * ROWS) void dispatch_recv_few_kernel(
    const V* __restrict__ recv_buf, const int* __restrict__ recv_meta,
    const int* __restrict__ recv_counts, int W, int hint_rows, int movers, int chunks, int row_vecs, int nle,
    int capacity_rows, uint32_t magic, int max_recv, int* __restrict__ expert_num_tokens,
    V* __restrict__ expert_x, int* __restrict__ expert_meta, int* __restrict__ plan, int* __restrict__ expert_offsets) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((int)blockIdx.x < nle) {
    plan_expert<COMPACT, KEYS / ROWS>(recv_meta, recv_counts, W, hint_rows, nle, capacity_rows, magic, expert_num_tokens, plan,
                            expert_offsets);
    return;
  }
  int R = -1;  // not known yet
  const int raw_count = recv_counts[min(lane, W - 1)];
  auto rows_arrived = [&] {
    const int my_count = lane < W ? min(max(first_use(raw_count), 0), capacity_rows) : 0;
    return min(wave_sum(my_count), capacity_rows);
  };
  for (int q = ((int)blockIdx.x - nle) * ROWS + wave;; q += movers * ROWS) {
    const int i = chunks == 1 ? q : q / chunks, c = q - i * chunks;
    if (R < 0 && i >= hint_rows) R = rows_arrived();
    if (R >= 0 && i >= R) return;
    const int base = c * (64 * NVW);
    const int e = recv_meta[(size_t)i * META];
    // keys that may be read, and of them the ones that can precede the row
    const int limit = R < 0 ? hint_rows : R;
    int n = COMPACT ? limit : min(i + 1, limit);
    int key[KEYS];
    auto fetch = [&](int b) {
#pragma unroll
      for (int u = 0; u < KEYS; ++u) key[u] = recv_meta[(size_t)min(b + u * 64 + lane, n - 1) * META];
    };
    fetch(0);
    int m = 0;
    if (c == 0 && lane < META) m = recv_meta[(size_t)i * META + lane];
    WavePayload<V, NVW> p;
    p.load(recv_buf + (size_t)i * row_vecs, base, row_vecs, lane);
    if (R < 0) R = rows_arrived();
    if (i >= R) return;
    const int le = floormod(e, nle, magic);
    int pos = 0;
    auto count = [&](int b, int end) {
      floormod_each(key, nle, magic);
#pragma unroll
      for (int u = 0; u < KEYS; ++u) {
        const int j = b + u * 64 + lane, le2 = key[u];
        pos += __popcll(__ballot(((le2 == le) & (j < i)) | (COMPACT && (le2 < le) & (j < end))));
      }
    };
    count(0, min(n, R));
    int b = min(n, 64 * KEYS);
    if constexpr (COMPACT) n = R;
    for (; b < n; b += 64 * KEYS) {
      fetch(b);
      count(b, n);
    }
    if (pos < max_recv) {
      const size_t row = COMPACT ? (size_t)pos : (size_t)le * max_recv + pos;
      p.template store<HOW>(expert_x + row * row_vecs, base, row_vecs, lane);
      if (c == 0 && lane < META) expert_meta[row * META + lane] = m;
    }
  }
}

// ---------------------------------------------------------------- expert-major stream helpers

// pre[0..nle] = exclusive prefix of value_of(le); returns the total. Each lane
// owns a contiguous run of experts; runs are combined by a wave64 scan and a
// scan over the wave totals.
template <int NW, class ValueOf>
__device__ __forceinline__ int expert_prefix_of(int nle, int* pre, int* red, ValueOf value_of) {
  const int tid = threadIdx.x;
  const int per = (nle + 64 * NW - 1) / (64 * NW);
  const int b = min(tid * per, nle), e = min(b + per, nle);
  int s = 0;
  for (int i = b; i < e; ++i) s += value_of(i);
  const int inc = wave_inclusive_scan(s);
  if ((tid & 63) == 63) red[tid >> 6] = inc;
  lds_barrier();
  int off = 0, total = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    if (w < (tid >> 6)) off += red[w];
    total += red[w];
  }
  int run = off + inc - s;
  for (int i = b; i < e; ++i) {
    pre[i] = run;
    run += value_of(i);
  }
  if (tid == 0) pre[nle] = total;
  lds_barrier();
  return total;
}

// The prefix of the rows per expert, min(cnt[le], max_recv).
template <int NW>
__device__ __forceinline__ int expert_prefix(const int* __restrict__ cnt, int nle, int max_recv,
                                             int* pre, int* red) {
  return expert_prefix_of<NW>(nle, pre, red, [=](int le) { return min(max(cnt[le], 0), max_recv); });
}

// Largest le in [0, nle) with pre[le] <= g, for g < pre[nle] (so empty experts
// are skipped). Fixed-trip binary lifting: `top` is the largest power of two
// below nle (0 when nle == 1), so several searches can run interleaved.
__device__ __forceinline__ int expert_of(const int* pre, int nle, int top, int g) {
  int lo = 0;
  for (int step = top; step > 0; step >>= 1) {
    const int c = lo + step;
    if (c < nle && pre[c] <= g) lo = c;
  }
  return lo;
}

__device__ __forceinline__ int top_step(int nle) {
  int top = 0;
  for (int s = 1; s < nle; s <<= 1) top = s;
  return top;
}

// Keys (int FIELD of the meta row) of rows of the expert-major stream, row g
// being the g-th valid row in (le, j) order. The SCAN_UNROLL searches of one
// fetch advance in lock step, so their LDS reads overlap instead of chaining.
template <int FIELD>
struct ExpertStreamKeys {
  const int* pre;  // LDS, nle + 1 entries, pre[nle] = number of rows
  const int* __restrict__ meta;
  int nle, top, max_recv;
  bool compact;  // the experts' rows lie back to back: stream row g is buffer row g
  __device__ __forceinline__ void fetch(const int* g, int* key) const {
    if (compact) {
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) key[u] = meta[(size_t)g[u] * META + FIELD];
      return;
    }
    int le[SCAN_UNROLL];
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) le[u] = 0;
    for (int step = top; step > 0; step >>= 1) {
      // all reads of a step first, then all updates: the reads stay in flight together
      int c[SCAN_UNROLL], v[SCAN_UNROLL];
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) c[u] = min(le[u] + step, nle);  // pre[nle] > g: never taken
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) v[u] = pre[c[u]];
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) le[u] = v[u] <= g[u] ? c[u] : le[u];
    }
    int first[SCAN_UNROLL];
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) first[u] = pre[le[u]];
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) {
      const size_t row = (size_t)le[u] * max_recv + (g[u] - first[u]);
      key[u] = meta[row * META + FIELD];
    }
  }
};

// The same stream when there are at most 64 local experts: lane l of every wave
// keeps the prefix of expert l in a register, so there is no LDS table, no
// barrier and the row a wave owns is found with one ballot. Lanes at or past
// nle hold the total, which no row index reaches.
struct WaveExpertPrefix {
  int excl, incl;  // rows before / up to and including expert `lane`
  int total;
  __device__ __forceinline__ WaveExpertPrefix(const int* __restrict__ cnt, int nle, int max_recv) {
    const int lane = threadIdx.x & 63;
    const int c = lane < nle ? min(max(cnt[lane], 0), max_recv) : 0;
    incl = wave_inclusive_scan(c);
    excl = incl - c;
    total = __builtin_amdgcn_readlane(incl, 63);
  }
  // expert holding row g (wave-uniform g < total) and the number of rows before it
  __device__ __forceinline__ void locate(int g, int& le, int& first) const {
    le = __popcll(__ballot(incl <= g));
    first = __builtin_amdgcn_readlane(excl, le);
  }
};

template <int FIELD>
struct WaveStreamKeys {
  int excl;  // this lane's WaveExpertPrefix::excl
  const int* __restrict__ meta;
  int nle, top, max_recv;
  bool compact;  // the experts' rows lie back to back: stream row g is buffer row g
  __device__ __forceinline__ void fetch(const int* g, int* key) const {
    if (compact) {  // (the same for every lane: no lane leaves the shuffles below behind)
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) key[u] = meta[(size_t)g[u] * META + FIELD];
      return;
    }
    int le[SCAN_UNROLL];
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) le[u] = 0;
    for (int step = top; step > 0; step >>= 1) {
      int c[SCAN_UNROLL], v[SCAN_UNROLL];
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) c[u] = le[u] + step;  // at most 32+16+...+1 = 63
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) v[u] = __shfl(excl, c[u], 64);
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) le[u] = v[u] <= g[u] ? c[u] : le[u];
    }
    int first[SCAN_UNROLL];
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) first[u] = __shfl(excl, le[u], 64);
#pragma unroll
    for (int u = 0; u < SCAN_UNROLL; ++u) {
      const size_t row = (size_t)le[u] * max_recv + (g[u] - first[u]);
      key[u] = meta[row * META + FIELD];
    }
  }
};

// ---------------------------------------------------------------- stage 3: combine, send side
//
// grid = W counting workgroups (rows per origin rank) followed by one workgroup
// per (group of ROWS valid expert rows, chunk), rows numbered g in (le, j)
// order. Row g with origin d goes to slot
//   #{rows of a lower origin} + #{earlier rows of origin d}.

//
// PLAN (needs SMALL and W <= 64): stage 2 left, for every (local expert, source
// rank), where that run of rows starts inside the expert and in the send-back
// stream (see dispatch_recv_kernel). A wave then finds the run its row lies in
// with one ballot over W lanes and needs no key scan and no exchange with the
// other waves. The plan counts every received row, so it only describes the
// buffers when no expert overflowed max_recv; if one did, every workgroup sees
// it in the counts and takes the scan instead.

template <typename V, int NVW, bool SMALL, bool PLAN, bool PAST, typename... Loaded>
__global__ __launch_bounds__(64 * ROWS) void combine_send_kernel(
    Loaded..., const int* __restrict__ expert_num_tokens, const int* __restrict__ plan,
    const int* __restrict__ expert_meta, const V* __restrict__ expert_y, int nle, int W, int chunks, int max_recv,
    int compact_rows, int row_vecs, int capacity_rows, V* __restrict__ send_buf, int* __restrict__ send_meta,
    int* __restrict__ send_counts) {
  static_assert(!PLAN || SMALL, "the planned path keeps the expert prefix in registers");
  __shared__ int part[2 * ROWS * ROWS];
  __shared__ int pre[SMALL ? 1 : MAX_LOCAL_EXPERTS + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  // compact_rows > 0: expert_y / expert_meta hold the experts' rows back to back (stream row g is
  // buffer row g) in buffers of compact_rows rows, and max_recv is that number too
  const bool compact = compact_rows > 0;

  if constexpr (PLAN) {
    const int raw = lane < nle ? expert_num_tokens[lane] : 0;
    const int have = max(raw, 0);
    const int incl = wave_inclusive_scan(have), excl = incl - have;
    const int R = __builtin_amdgcn_readlane(incl, 63);
    // (the plan also counts rows that found no room; with such rows the scan below is taken)
    if (__ballot(raw > max_recv) == 0 && !(compact && R > compact_rows)) {

      if ((int)blockIdx.x < W) {
        // rows that go back to origin `me`: the lengths of its runs, one expert per lane
        const int me = blockIdx.x;
        int len = 0;
        if (lane < nle) {
          const int* run = plan + ((size_t)lane * W + me) * PLAN_INTS;
          len = (me + 1 < W ? run[PLAN_INTS] : have) - run[0];
        }
        const int total = wave_sum(len);
        if (tid == 0) send_counts[me] = total;
        return;
      }

      const int items = R * chunks, movers = (gridDim.x - W) * ROWS;
      for (int qv = (blockIdx.x - W) * ROWS + wave; qv < items; qv += movers) {
        const int q = __builtin_amdgcn_readfirstlane(qv);  // the same for every lane of a wave
        const int g = chunks == 1 ? q : q / chunks, c = q - g * chunks;
        const int base = c * (64 * NVW);
        const int le = __popcll(__ballot(incl <= g));
        const int j = g - __builtin_amdgcn_readlane(excl, le);
        const size_t row = compact ? (size_t)g : (size_t)le * max_recv + j;
        int run[PLAN_INTS] = {INT_MAX, 0};
        if (lane < W) __builtin_memcpy(run, plan + ((size_t)le * W + lane) * PLAN_INTS, sizeof(run));
        int m = 0;
        if (c == 0 && lane < META) m = expert_meta[row * META + lane];
        WavePayload<V, NVW> p;
        p.template load<PAST>(unknown_origin(expert_y + row * row_vecs), base, row_vecs, lane);
        // (the row is only used by the stores below, which depend on the slot: without this the
        // compiler moves the loads down behind the plan's round trip)
        issued_here();
        // the run starts are ascending in the source rank: the last one at or below j is ours
        const int src = max((int)__popcll(__ballot(run[0] <= j)) - 1, 0);
        const int slot = __builtin_amdgcn_readlane(run[1], src) + (j - __builtin_amdgcn_readlane(run[0], src));
        if (slot >= 0 && slot < capacity_rows) {
          p.template store<MOE_A2A_STORE_CSEND>(send_buf + (size_t)slot * row_vecs, base, row_vecs, lane);
          if (c == 0 && lane < META) send_meta[(size_t)slot * META + lane] = m;
        }
      }
      return;
    }
  }

  // SMALL (nle <= 64): prefix in registers; otherwise the LDS table
  using Keys = typename std::conditional<SMALL, WaveStreamKeys<1>, ExpertStreamKeys<1>>::type;
  int R, my_excl = 0, my_incl = 0;
  if constexpr (SMALL) {
    const WaveExpertPrefix wp(expert_num_tokens, nle, max_recv);
    R = wp.total; my_excl = wp.excl; my_incl = wp.incl;
  } else {
    R = expert_prefix<ROWS>(expert_num_tokens, nle, max_recv, pre, part);
  }
  if (compact) R = min(R, compact_rows);
  Keys key;
  if constexpr (SMALL) key = Keys{my_excl, expert_meta, nle, 32, max_recv, compact};
  else key = Keys{pre, expert_meta, nle, top_step(nle), max_recv, compact};
  // buffer row of stream row g (wave-uniform g < R)
  auto padded_row = [&](int g) -> size_t {
    if (compact) return (size_t)g;
    int le, first;
    if constexpr (SMALL) {
      le = __popcll(__ballot(my_incl <= g));
      first = __builtin_amdgcn_readlane(my_excl, le);
    } else {
      le = expert_of(pre, nle, key.top, g);
      first = pre[le];
    }
    return (size_t)le * max_recv + (g - first);
  };

  if ((int)blockIdx.x < W) {
    const int me = blockIdx.x;
    int c = count_keys<64 * ROWS>(R, key, [me](int d, int) { return d == me; });
    c = block_sum<ROWS>(c, part);
    if (tid == 0) send_counts[me] = c;
    return;
  }

  const int groups = (R + ROWS - 1) / ROWS;
  const int items = groups * chunks, movers = gridDim.x - W;
  int parity = 0;
  for (int q = blockIdx.x - W; q < items; q += movers, ++parity) {
    const int grp = chunks == 1 ? q : q / chunks, c = q - grp * chunks;
    const int g0 = grp * ROWS, g = g0 + wave;
    const bool valid = g < R;
    const int base = c * (64 * NVW);

    // origin rank of every row of the group, read by every wave (no exchange)
    int rd[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) rd[r] = expert_meta[padded_row(min(g0 + r, R - 1)) * META + 1];
    const size_t row = padded_row(min(g, R - 1));
    int m = 0;
    if (c == 0 && lane < META) m = expert_meta[row * META + lane];
    RowsScan<Keys> scan(R, key);
    WavePayload<V, NVW> p;
    p.load(expert_y + row * row_vecs, base, row_vecs, lane);

    int cnt[ROWS];
    // origins compared as unsigned numbers: a row whose meta names no rank (negative, or W and
    // above) sorts behind the rows of every real origin instead of shifting their segments
    scan.finish(key, R, [&](int r, int d2, int g2) {
      return ((uint32_t)d2 < (uint32_t)rd[r]) | ((d2 == rd[r]) & (g2 < g0 + r));
    }, cnt);
    const int slot = rows_reduce(cnt, part, parity, wave, lane);

    if (valid && slot < capacity_rows) {
      p.template store<MOE_A2A_STORE_CSEND>(send_buf + (size_t)slot * row_vecs, base, row_vecs, lane);
      if (c == 0 && lane < META) send_meta[(size_t)slot * META + lane] = m;
    }
  }
}

// ---------------------------------------------------------------- 16-bit float helpers
//
// Element arithmetic works on 32-bit words holding two 16-bit elements (low
// half = even element), so that the gfx950 pair conversion v_cvt_pk_bf16_f32
// (round to nearest even) does the rounding of both in one instruction.
// A NaN keeps whatever payload the hardware gives it while it is being
// accumulated; bf16 results are canonicalised to 0x7fc0 (what torch stores for
// any NaN) where they are written out.

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <int DT> struct Pair16;
template <> struct Pair16<MOE_A2A_BF16> {
  static __device__ __forceinline__ float lo(uint32_t w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
  static __device__ __forceinline__ uint32_t round(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
  }
  static __device__ __forceinline__ uint32_t canonical(uint32_t w) {
    if ((w & 0x7fffu) > 0x7f80u) w = (w & 0xffff0000u) | 0x7fc0u;
    if ((w & 0x7fff0000u) > 0x7f800000u) w = (w & 0x0000ffffu) | 0x7fc00000u;
    return w;
  }
};
template <> struct Pair16<MOE_A2A_F16> {
  static __device__ __forceinline__ float lo(uint32_t w) {
    return (float)__builtin_bit_cast(f16x2, w).x;
  }
  static __device__ __forceinline__ float hi(uint32_t w) {
    return (float)__builtin_bit_cast(f16x2, w).y;
  }
  static __device__ __forceinline__ uint32_t round(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
  }
  static __device__ __forceinline__ uint32_t canonical(uint32_t w) { return w; }
};

template <typename V> struct Words;  // 32-bit words (element pairs) per vector
template <> struct Words<b128> { static constexpr int N = 4; };
template <> struct Words<uint16_t> { static constexpr int N = 1; };  // one element, high half unused

template <typename V>
__device__ __forceinline__ uint32_t get_word(const V& v, int i) {
  if constexpr (Words<V>::N == 1) return v;
  else return v[i];
}

template <typename V>
__device__ __forceinline__ V from_words(const uint32_t* w) {
  if constexpr (Words<V>::N == 1) {
    return (uint16_t)w[0];
  } else {
    b128 v;
    v.x = w[0]; v.y = w[1]; v.z = w[2]; v.w = w[3];
    return v;
  }
}

// ---------------------------------------------------------------- stage 4: combine, receive side

// A running row sum: two floats per word, each always exactly representable in
// the 16-bit type. step() is one `out[t] += row.float() * w` of the reference:
//   p = RN32(f32(v) * w);  a = RN32(acc + p);  acc = RN16(a)
template <int DT>
struct PairAcc {
  float lo, hi;
  __device__ __forceinline__ void set(uint32_t w) { lo = Pair16<DT>::lo(w); hi = Pair16<DT>::hi(w); }
  __device__ __forceinline__ void step(uint32_t v, float w) {
    const float a = __fadd_rn(lo, __fmul_rn(Pair16<DT>::lo(v), w));
    const float b = __fadd_rn(hi, __fmul_rn(Pair16<DT>::hi(v), w));
    set(Pair16<DT>::round(a, b));
  }
  __device__ __forceinline__ uint32_t word() const {
    return Pair16<DT>::canonical(Pair16<DT>::round(lo, hi));
  }
};

// Workgroup of BLK lanes per (token, chunk); each lane owns NV vector columns.
// The workgroup finds the rows addressed to its token by scanning the src_token
// column of the arriving meta rows, orders them by arrival index, then walks
// them in that order with all rows of a batch loaded up front.
//
// `hint_rows` rows of recv_meta are readable whatever the counts say: the first
// batch of the scan is loaded before the true row count R is known (the counts
// are loaded at the same time); rows at or past R are ignored.

// Long streams: every workgroup of a token scanning the whole arriving stream makes the meta
// reads grow with tokens x rows. return_map_kernel turns the stream into a table first: one
// thread per arriving row writes its row number at entry_row[src_token * K + src_k]. A token's
// workgroup then looks its K entries up instead of scanning (MAPPED below). An entry is taken
// only if the meta row it points to names this token and this k NOW, so whatever an earlier
// call left in the table can never be mistaken for an arrival; the table needs no clearing.
// The one assumption is that no (token, k) pair arrives twice, which holds for every stream
// the dispatch produced: with duplicates the table keeps one of them.
__global__ __launch_bounds__(BLOCK) void return_map_kernel(
    const int* __restrict__ recv_meta, const int* __restrict__ recv_counts, int W, int hint_rows,
    int capacity_rows, int T, int K, int* __restrict__ entry_row) {
  // the first row of a thread is loaded before the row count is known when it lies below the
  // readable bound (the counts travel at the same time)
  int i = blockIdx.x * BLOCK + threadIdx.x;
  int tk[2] = {-1, -1};
  bool loaded = i < hint_rows;
  if (loaded) __builtin_memcpy(tk, recv_meta + (size_t)i * META + 2, 8);
  const int R = min(sum_counts(recv_counts, W, capacity_rows), capacity_rows);
  for (; i < R; i += gridDim.x * BLOCK) {
    if (!loaded) __builtin_memcpy(tk, recv_meta + (size_t)i * META + 2, 8);
    loaded = false;
    if ((uint32_t)tk[0] < (uint32_t)T && (uint32_t)tk[1] < (uint32_t)K) entry_row[(size_t)tk[0] * K + tk[1]] = i;
  }
}

template <typename V, int DT, int BLK, int NV, bool MAPPED, int UNROLL>
__global__ __launch_bounds__(BLK) void combine_recv_kernel(
    const int* __restrict__ recv_meta, const int* __restrict__ recv_counts, const float* __restrict__ weights, int W,
    int hint_rows, int T, int K, int chunks, int capacity_rows, const V* __restrict__ recv_buf, int row_vecs,
    int accumulate, V* __restrict__ out, const int* __restrict__ entry_row) {
  constexpr int N = Words<V>::N;
  constexpr int FAST = 8;  // addends ordered in registers
  __shared__ int hit_row[COMBINE_CAP], hit_k[COMBINE_CAP];
  __shared__ int ord_row[COMBINE_CAP];
  __shared__ float ord_w[COMBINE_CAP];
  __shared__ float wts[COMBINE_WEIGHTS];
  __shared__ int nhit;
  const int tid = threadIdx.x, lane = tid & 63;
  const int kw = min(K, COMBINE_WEIGHTS);
  const bool lanes_hold_counts = W <= 64;
  // in flight with the first batch of the scan (first_use)
  const int raw_count = recv_counts[min(lane, W - 1)];
  int R = -1;  // not known yet
  auto rows_arrived = [&] {
    const int my_count = lane < W ? min(max(first_use(raw_count), 0), capacity_rows) : 0;
    return min(lanes_hold_counts ? wave_sum(my_count) : sum_counts(recv_counts, W, capacity_rows), capacity_rows);
  };

  // rows [lo, hi) of the arriving stream: note the ones addressed to token t
  auto scan = [&](int t, int lo, int hi) {
    for (int b = lo; b < hi; b += UNROLL * BLK) {
      int key[UNROLL], kk[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        // src_token and src_k with one 8-byte load (4-byte aligned, which global loads accept);
        // fetching src_k for the hits alone with a dependent load costs more than it saves
        int tk[2];
        __builtin_memcpy(tk, recv_meta + (size_t)min(b + tid + u * BLK, hi - 1) * META + 2, 8);
        key[u] = tk[0];
        kk[u] = tk[1];
      }
      if (R < 0) R = rows_arrived();
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int row = b + tid + u * BLK;
        // (an arriving row whose k names no weight of the token is not an addend)
        if (row < min(hi, R) && key[u] == t && (uint32_t)kk[u] < (uint32_t)K) {
          const int p = atomicAdd(&nhit, 1);
          if (p < COMBINE_CAP) {
            hit_row[p] = row;
            hit_k[p] = kk[u];
          }
        }
      }
    }
  };

  const int items = T * chunks;
  for (int q = blockIdx.x; q < items; q += gridDim.x) {
    const int t = chunks == 1 ? q : q / chunks, c = q - t * chunks;
    const int base = c * (BLK * NV);
    V* __restrict__ orow = out + (size_t)t * row_vecs;

    // the token's weights travel to LDS while the scan's loads are in flight
    float wreg = 0.0f;
    if (tid < kw) wreg = weights[(size_t)t * K + tid];

    PairAcc<DT> acc[NV][N];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      V o{};
      if (accumulate) o = orow[min(base + j * BLK + tid, row_vecs - 1)];
#pragma unroll
      for (int e = 0; e < N; ++e) acc[j][e].set(get_word(o, e));
    }

    if (tid == 0) nhit = 0;
    lds_barrier();
    if constexpr (MAPPED) {
      if (R < 0) R = rows_arrived();
      for (int k = tid; k < K; k += BLK) {
        const int i = entry_row[(size_t)t * K + k];
        if ((uint32_t)i < (uint32_t)R) {
          int tk[2];
          __builtin_memcpy(tk, recv_meta + (size_t)i * META + 2, 8);
          if (tk[0] == t && tk[1] == k) {
            const int p = atomicAdd(&nhit, 1);
            if (p < COMBINE_CAP) {
              hit_row[p] = i;
              hit_k[p] = k;
            }
          }
        }
      }
    } else if (R < 0) {
      // first item: one batch below the readable bound goes out before R is known
      const int spec = min(hint_rows, UNROLL * BLK);
      scan(t, 0, spec);
      if (R < 0) R = rows_arrived();
      scan(t, spec, R);
    } else {
      scan(t, 0, R);
    }
    if (tid < kw) wts[tid] = wreg;
    lds_barrier();
    const int n = nhit;

    if (n <= FAST && K <= COMBINE_WEIGHTS) {  // (every weight of the token is in LDS)
      if (n > 0) {
        // Order the (at most 8) hits by arrival index. Lane l of every wave takes hit l % 8; its
        // place in the order is the number of hits that arrived earlier, counted with seven
        // rotations of a 16-lane DPP row (lanes 8..15 of a row hold the same eight hits again, so
        // rotating by 1..7 shows a lane every other hit once). Each lane then pushes its hit to
        // the lane of its place, and the ordered rows and weights are read lane by lane into
        // scalar registers. About 45 vector instructions per wave; a sorting network on the
        // hits as uniform values becomes some 150 scalar instructions, and the sixteen waves of a
        // compute unit share one scalar unit.
        const int p = lane & (FAST - 1);
        const int hr = p < n ? hit_row[p] : INT_MAX;
        const int hk = p < n ? hit_k[p] : 0;  // (0 <= k < K: checked when the hit was noted)
        const float hw = wts[hk];
        int place = 0;
#define MOE_A2A_ROT(S) place += (int)(__builtin_amdgcn_update_dpp(0, hr, 0x120 + S, 0xf, 0xf, false) < hr)
        MOE_A2A_ROT(1); MOE_A2A_ROT(2); MOE_A2A_ROT(3); MOE_A2A_ROT(4); MOE_A2A_ROT(5); MOE_A2A_ROT(6); MOE_A2A_ROT(7);
#undef MOE_A2A_ROT
        // (lanes without a hit all get place n, which nothing reads)
        const int to = ((lane & ~(FAST - 1)) | place) << 2;
        const int ordered_row = __builtin_amdgcn_ds_permute(to, hr);
        const int ordered_w = __builtin_amdgcn_ds_permute(to, __float_as_int(hw));
        V v[FAST][NV];
        float w[FAST];
#pragma unroll
        for (int u = 0; u < FAST; ++u) {
          // row 0 exists (n > 0): loaded for the places past n and not used
          const int row = u < n ? __builtin_amdgcn_readlane(ordered_row, u) : 0;
          w[u] = __int_as_float(__builtin_amdgcn_readlane(ordered_w, u));
#pragma unroll
          for (int j = 0; j < NV; ++j)
            v[u][j] = recv_buf[(size_t)row * row_vecs + min(base + j * BLK + tid, row_vecs - 1)];
        }
#pragma unroll
        for (int u = 0; u < FAST; ++u) {
          if (u < n) {
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
              for (int e = 0; e < N; ++e) acc[j][e].step(get_word(v[u][j], e), w[u]);
          }
        }
      }
    } else if (n <= COMBINE_CAP) {
      if (tid < n) {  // order the hits by arrival index
        const int me = hit_row[tid];
        int r = 0;
        for (int b = 0; b < n; ++b) r += hit_row[b] < me;
        const int k = hit_k[tid];
        const bool ok = (k >= 0) & (k < K);
        ord_row[r] = ok ? me : -1;
        ord_w[r] = !ok ? 0.0f : k < kw ? wts[k] : weights[(size_t)t * K + k];
      }
      lds_barrier();
      for (int a0 = 0; a0 < n; a0 += COMBINE_BATCH) {
        V v[COMBINE_BATCH][NV];
#pragma unroll
        for (int u = 0; u < COMBINE_BATCH; ++u) {
          // clamped, unconditional loads keep the whole batch in flight
          const int row = max(ord_row[min(a0 + u, n - 1)], 0);
#pragma unroll
          for (int j = 0; j < NV; ++j)
            v[u][j] = recv_buf[(size_t)row * row_vecs + min(base + j * BLK + tid, row_vecs - 1)];
        }
#pragma unroll
        for (int u = 0; u < COMBINE_BATCH; ++u) {
          if (a0 + u < n && ord_row[a0 + u] >= 0) {
            const float w = ord_w[a0 + u];
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
              for (int e = 0; e < N; ++e) acc[j][e].step(get_word(v[u][j], e), w);
          }
        }
      }
    } else {
      // More addends than the LDS list holds: walk the stream in order.
      for (int i = 0; i < R; ++i) {
        if (recv_meta[(size_t)i * META + 2] != t) continue;
        const int k = recv_meta[(size_t)i * META + 3];
        if (k < 0 || k >= K) continue;
        const float w = weights[(size_t)t * K + k];
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          const int idx = base + j * BLK + tid;
          if (idx < row_vecs) {
            const V v = recv_buf[(size_t)i * row_vecs + idx];
#pragma unroll
            for (int e = 0; e < N; ++e) acc[j][e].step(get_word(v, e), w);
          }
        }
      }
    }

#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int idx = base + j * BLK + tid;
      if (idx < row_vecs) {
        uint32_t h[N];
#pragma unroll
        for (int e = 0; e < N; ++e) h[e] = acc[j][e].word();
        orow[idx] = from_words<V>(h);
      }
    }
    lds_barrier();  // the LDS lists are reused by the next item
  }
}

// Stage 4 of a long stream with its table (return_map_kernel), for up to eight entries per token: a wave per (token, piece
// of 64 * NV vectors), with nothing to wait for but its own loads. Lane k (and those 8, 16, .. on) holds entry k: the rows that the
// table names are ordered by arrival and asked for while the meta rows that say whether they are the token's are on their way. Memory
// bounds it, on short rows the two dependent trips. us with the launch that makes the table, a workgroup of 256 lanes per piece that takes
// these steps one after the other with barriers between them / here: 2500 tokens of 2 KB, 1 per token 14.3 / 10.4, 1600 of 2 KB, 2 each 13.1 / 10.2,
// 4096 of 8 KB, 2 each 34.3 / 24.5, 3 each 37.4 / 29.7, 4096 of 14 KB, 8 each 109.5 / 96.0 (5.8 TB/s).
template <int DT, int NV, int ADDENDS, bool PAST>
__global__ __launch_bounds__(BLOCK) void combine_recv_mapped_kernel(
    const int* __restrict__ entry_row, const int* __restrict__ recv_counts, const float* __restrict__ weights,
    const int* __restrict__ recv_meta, int W, int T, int K, Pieces pieces, int capacity_rows,
    const b128* __restrict__ recv_buf, int row_vecs, int accumulate, b128* __restrict__ out) {
  constexpr int N = Words<b128>::N, FAST = 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int items = T * pieces.per_row, waves = gridDim.x * NWAVES;
  const int raw_count = recv_counts[min(lane, W - 1)];
  int R = -1;
  for (int q = blockIdx.x * NWAVES + wave; q < items; q += waves) {
    const int t = pieces.row_of(q), base = (q - t * pieces.per_row) * (64 * NV);
    const int k = lane & (FAST - 1), kc = min(k, K - 1);
    const int i = entry_row[(size_t)t * K + kc];
    const float w = weights[(size_t)t * K + kc];
    b128* __restrict__ orow = out + (size_t)t * row_vecs;
    PairAcc<DT> acc[NV][N];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      b128 o{};
      if (accumulate) o = orow[min(base + j * 64 + lane, row_vecs - 1)];
#pragma unroll
      for (int e = 0; e < N; ++e) acc[j][e].set(get_word(o, e));
    }
    if (R < 0) {
      const int my_count = lane < W ? min(max(first_use(raw_count), 0), capacity_rows) : 0;
      R = min(W <= 64 ? wave_sum(my_count) : sum_counts(recv_counts, W, capacity_rows), capacity_rows);
    }
    const bool named = k < K && (uint32_t)i < (uint32_t)R;
    int tk[2] = {-1, -1};
    if (named) __builtin_memcpy(tk, recv_meta + (size_t)i * META + 2, 8);
    // (as in combine_recv_kernel; a stale entry may name a row that another one names as well: the entry decides between them)
    const uint32_t key = named ? (uint32_t)i << 3 | k : UINT_MAX;
    int place = 0;
#define MOE_A2A_ROT(S) place += (int)((uint32_t)__builtin_amdgcn_update_dpp(0, (int)key, 0x120 + S, 0xf, 0xf, false) < key)
    MOE_A2A_ROT(1); MOE_A2A_ROT(2); MOE_A2A_ROT(3); MOE_A2A_ROT(4); MOE_A2A_ROT(5); MOE_A2A_ROT(6); MOE_A2A_ROT(7);
#undef MOE_A2A_ROT
    const int to = ((lane & ~(FAST - 1)) | place) << 2;
    const int ordered_row = __builtin_amdgcn_ds_permute(to, i), ordered_w = __builtin_amdgcn_ds_permute(to, __float_as_int(w));
    const int n = __popcll(__ballot(named) & 0xff);
    b128 v[ADDENDS][NV];
#pragma unroll
    for (int u = 0; u < ADDENDS; ++u) {
      if (u < n) {
        const b128* row = recv_buf + (size_t)__builtin_amdgcn_readlane(ordered_row, u) * row_vecs;
#pragma unroll
        for (int j = 0; j < NV; ++j) v[u][j] = row_load<PAST>(unknown_origin(row) + min(base + j * 64 + lane, row_vecs - 1));
      }
    }
    issued_here();
    // which of the ordered rows are addends: those whose meta row names this token and entry
    const int ordered_ok = __builtin_amdgcn_ds_permute(to, (int)(named && tk[0] == t && tk[1] == k));
    const unsigned long long ok = __ballot(ordered_ok != 0);
#pragma unroll
    for (int u = 0; u < ADDENDS; ++u) {
      if (u < n && (ok >> u & 1)) {
        const float wu = __int_as_float(__builtin_amdgcn_readlane(ordered_w, u));
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
          for (int e = 0; e < N; ++e) acc[j][e].step(get_word(v[u][j], e), wu);
      }
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int idx = base + j * 64 + lane;
      if (idx < row_vecs) {
        uint32_t h[N];
#pragma unroll
        for (int e = 0; e < N; ++e) h[e] = acc[j][e].word();
        row_store<THROUGH>(orow + idx, from_words<b128>(h));
      }
    }
  }
}

// Stage 4 for up to eight entries per token without a table: one pass of sixteen waves over the arriving meta rows notes what is addressed to any
// of the workgroup's tokens, in whatever order; then a wave per (token, piece of 64 vectors) orders the token's rows by arrival and has all of
// them under way at once. A token with more than ADDENDS rows (pairs that arrive twice) is added up from another walk over the stream.
// Bound by the trips (counts and metas, rows) and, with many tokens, by the rows: a workgroup per token and 256 vectors, each of which reads all
// metas, spent most of its time on those. us, that / here: 885 tokens of 5.8 KB, 4 per token 10.8 / 7.2, 939 of 8.4 KB, 2 each 10.2 / 6.8, 1428
// of 7.6 KB, 2 each 11.7 / 7.8, 1622 of 1 KB, 1 each 6.2 / 4.3, 377 of 10 KB, 6 each 8.4 / 7.4. Results stored plainly 0.1 to 0.4 us longer.
template <int DT, int ADDENDS>
__global__ __launch_bounds__(COMBINE_BLOCK) void combine_recv_block_kernel(
    const int* __restrict__ recv_meta, const int* __restrict__ recv_counts, const float* __restrict__ weights, int W, int hint_rows, int T,
    int K, int tokens, Pieces pieces, int capacity_rows, const b128* __restrict__ recv_buf, int row_vecs, int accumulate,
    b128* __restrict__ out) {
  constexpr int N = Words<b128>::N, FAST = 8, UNROLL = 4, WAVES = COMBINE_BLOCK / 64;
  __shared__ int hits[COMBINE_TOKENS], hit[COMBINE_TOKENS * FAST];  // rows of a token; their numbers * 8 + entry
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int t0 = blockIdx.x * tokens, here = min(tokens, T - t0);
  const int raw_count = recv_counts[min(lane, W - 1)];
  if (tid < COMBINE_TOKENS) hits[tid] = 0;
  int tk[UNROLL][2];
  auto fetch = [&](int b, int end) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
      __builtin_memcpy(tk[u], recv_meta + (size_t)min(b + tid + u * COMBINE_BLOCK, end - 1) * META + 2, 8);
  };
  auto note = [&](int b, int end) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int row = b + tid + u * COMBINE_BLOCK, t = tk[u][0] - t0;
      if (row < end && (uint32_t)t < (uint32_t)here && (uint32_t)tk[u][1] < (uint32_t)K) {
        const int p = atomicAdd(&hits[t], 1);
        if (p < FAST) hit[t * FAST + p] = row << 3 | tk[u][1];
      }
    }
  };
  const int ahead = min(hint_rows, UNROLL * COMBINE_BLOCK);  // (readable whatever the counts say; more than none)
  fetch(0, ahead);
  lds_barrier();
  const int my_count = lane < W ? min(max(first_use(raw_count), 0), capacity_rows) : 0;
  const int R = min(W <= 64 ? wave_sum(my_count) : sum_counts(recv_counts, W, capacity_rows), capacity_rows);
  note(0, min(ahead, R));
  for (int b = ahead; b < R; b += UNROLL * COMBINE_BLOCK) {
    fetch(b, R);
    note(b, R);
  }
  lds_barrier();

  const int items = here * pieces.per_row;
  for (int q = wave; q < items; q += WAVES) {
    const int item = pieces.row_of(q), at = (q - item * pieces.per_row) * 64 + lane, col = min(at, row_vecs - 1), t = t0 + item;
    const int n = __builtin_amdgcn_readfirstlane(hits[item]);
    const float* const w_row = weights + (size_t)t * K;
    b128* __restrict__ orow = out + (size_t)t * row_vecs;
    PairAcc<DT> acc[N];
    b128 o{};
    if (accumulate) o = orow[col];
#pragma unroll
    for (int e = 0; e < N; ++e) acc[e].set(get_word(o, e));
    if (n <= ADDENDS) {
      const int p = lane & (FAST - 1);
      const int mine = p < n ? hit[item * FAST + p] : INT_MAX;
      const float w = w_row[p < n ? mine & 7 : 0];
      int place = 0;
#define MOE_A2A_ROT(S) place += (int)(__builtin_amdgcn_update_dpp(0, mine, 0x120 + S, 0xf, 0xf, false) < mine)
      MOE_A2A_ROT(1); MOE_A2A_ROT(2); MOE_A2A_ROT(3); MOE_A2A_ROT(4); MOE_A2A_ROT(5); MOE_A2A_ROT(6); MOE_A2A_ROT(7);
#undef MOE_A2A_ROT
      const int to = ((lane & ~(FAST - 1)) | place) << 2;  // (lanes without a row all get place n, which nothing reads)
      const int ordered = __builtin_amdgcn_ds_permute(to, mine);
      b128 v[ADDENDS];
#pragma unroll
      for (int u = 0; u < ADDENDS; ++u)
        if (u < n) v[u] = *(unknown_origin(recv_buf + (size_t)(__builtin_amdgcn_readlane(ordered, u) >> 3) * row_vecs) + col);
      issued_here();
      const int ordered_w = __builtin_amdgcn_ds_permute(to, __float_as_int(w));
#pragma unroll
      for (int u = 0; u < ADDENDS; ++u) {
        if (u < n) {
          const float wu = __int_as_float(__builtin_amdgcn_readlane(ordered_w, u));
#pragma unroll
          for (int e = 0; e < N; ++e) acc[e].step(get_word(v[u], e), wu);
        }
      }
    } else {
      for (int b = 0; b < R; b += 64) {
        int key[2];
        __builtin_memcpy(key, recv_meta + (size_t)min(b + lane, R - 1) * META + 2, 8);
        unsigned long long mine = __ballot(b + lane < R && key[0] == t && (uint32_t)key[1] < (uint32_t)K);
        for (; mine; mine &= mine - 1) {
          const int l = __builtin_ctzll(mine);
          const float wu = w_row[__builtin_amdgcn_readlane(key[1], l)];
          const b128 v = recv_buf[(size_t)(b + l) * row_vecs + col];
#pragma unroll
          for (int e = 0; e < N; ++e) acc[e].step(get_word(v, e), wu);
        }
      }
    }
    if (at < row_vecs) {
      uint32_t h[N];
#pragma unroll
      for (int e = 0; e < N; ++e) h[e] = acc[e].word();
      row_store<THROUGH>(orow + at, from_words<b128>(h));
    }
  }
}

// The same for a short stream (hint_rows <= 64 * KEYS): every wave looks through all of it by itself. The rows of 64 keys
// that are the token's come out of a ballot in arrival order, so there is nothing to sort and no other wave to wait for.
// ADDENDS: rows under way at a time. us, one launch after another in a graph, before / here: 72 rows of 1 KB, 6 per token
// 3.73 / 3.06, 32 of 12 KB 3.62 / 2.79, 240 of 2 KB 3.69 / 2.92, 500 of 5.8 KB 4.37 / 3.88.
constexpr int COMBINE_FEW_ROWS = 64 * 8;
template <int DT, int NV, int KEYS, int ADDENDS>
__global__ __launch_bounds__(BLOCK) void combine_recv_few_kernel(
    const int* __restrict__ recv_meta, const int* __restrict__ recv_counts, const float* __restrict__ weights, int W,
    int hint_rows, int K, int chunks, int capacity_rows, const b128* __restrict__ recv_buf, int row_vecs,
    int accumulate, b128* __restrict__ out) {
  constexpr int N = Words<b128>::N, LIST = 64;
  __shared__ int hits[NWAVES][LIST][2];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int t = chunks == 1 ? (int)blockIdx.x : (int)blockIdx.x / chunks, c = (int)blockIdx.x - t * chunks;
  const int base = c * (BLOCK * NV);
  const int raw_count = recv_counts[min(lane, W - 1)];
  const float my_weight = weights[(size_t)t * K + min(lane, K - 1)];
  int tk[KEYS][2];
  auto fetch = [&](int b, int end) {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) __builtin_memcpy(tk[u], recv_meta + (size_t)min(b + u * 64 + lane, end - 1) * META + 2, 8);
  };
  fetch(0, hint_rows);
  b128* __restrict__ orow = out + (size_t)t * row_vecs;
  PairAcc<DT> acc[NV][N];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    b128 o{};
    if (accumulate) o = orow[min(base + j * BLOCK + tid, row_vecs - 1)];
#pragma unroll
    for (int e = 0; e < N; ++e) acc[j][e].set(o[e]);
  }
  const int my_count = lane < W ? min(max(first_use(raw_count), 0), capacity_rows) : 0;
  const int R = min(wave_sum(my_count), capacity_rows);
  int n = 0;
  auto note = [&](int b, int end) {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      const int row = b + u * 64 + lane;
      // (an arriving row whose k names no weight of the token is not an addend)
      const bool hit = row < end && tk[u][0] == t && (uint32_t)tk[u][1] < (uint32_t)K;
      const unsigned long long all = __ballot(hit);
      const int at = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(all >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)all, 0));
      if (hit && at < LIST) {
        hits[wave][at][0] = row;
        hits[wave][at][1] = tk[u][1];
      }
      n += __popcll(all);
    }
  };
  note(0, min(hint_rows, R));
  for (int b = hint_rows; b < R; b += KEYS * 64) {
    fetch(b, R);
    note(b, R);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (n <= LIST) {
    for (int a0 = 0; a0 < n; a0 += ADDENDS) {
      const int p = min(a0 + (lane & (ADDENDS - 1)), n - 1);
      const int hit_row = hits[wave][p][0];
      const int hit_weight = __builtin_amdgcn_ds_bpermute(hits[wave][p][1] << 2, __float_as_int(my_weight));
      b128 v[ADDENDS][NV];
      float w[ADDENDS];
#pragma unroll
      for (int u = 0; u < ADDENDS; ++u) {
        // (row 0 exists: loaded for the places past n and not used)
        const int row = a0 + u < n ? __builtin_amdgcn_readlane(hit_row, u) : 0;
        w[u] = __int_as_float(__builtin_amdgcn_readlane(hit_weight, u));
#pragma unroll
        for (int j = 0; j < NV; ++j) v[u][j] = recv_buf[(size_t)row * row_vecs + min(base + j * BLOCK + tid, row_vecs - 1)];
      }
#pragma unroll
      for (int u = 0; u < ADDENDS; ++u) {
        if (a0 + u < n) {
#pragma unroll
          for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < N; ++e) acc[j][e].step(v[u][j][e], w[u]);
        }
      }
    }
  } else {  // more addends than the list holds: walk the stream in order
    for (int i = 0; i < R; ++i) {
      if (recv_meta[(size_t)i * META + 2] != t) continue;
      const int k = recv_meta[(size_t)i * META + 3];
      if (k < 0 || k >= K) continue;
      const float w = weights[(size_t)t * K + k];
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const b128 v = recv_buf[(size_t)i * row_vecs + min(base + j * BLOCK + tid, row_vecs - 1)];
#pragma unroll
        for (int e = 0; e < N; ++e) acc[j][e].step(v[e], w);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int idx = base + j * BLOCK + tid;
    if (idx < row_vecs) {
      uint32_t h[N];
#pragma unroll
      for (int e = 0; e < N; ++e) h[e] = acc[j][e].word();
      orow[idx] = from_words<b128>(h);
    }
  }
}

// ---------------------------------------------------------------- simulated expert

// .to(out_dtype), then times `scale` = (1 + rank) in float32, rounded once (all2all/reference.py:262)
template <typename V, int DIN, int DOUT>
__device__ __forceinline__ V standin_expert(V v, float scale) {
  constexpr int N = Words<V>::N;
  uint32_t h[N];
#pragma unroll
  for (int e = 0; e < N; ++e) {
    const uint32_t w = get_word(v, e);
    const uint32_t o = Pair16<DOUT>::round(Pair16<DIN>::lo(w), Pair16<DIN>::hi(w));
    const float lo = rounded_here(__fmul_rn(Pair16<DOUT>::lo(o), scale));
    const float hi = rounded_here(__fmul_rn(Pair16<DOUT>::hi(o), scale));
    h[e] = Pair16<DOUT>::canonical(Pair16<DOUT>::round(lo, hi));
  }
  return from_words<V>(h);
}

template <typename V, int NV, int DIN, int DOUT, Store HOW>
__global__ __launch_bounds__(BLOCK) void expert_scale_kernel(
    const V* __restrict__ expert_x, const int* __restrict__ expert_num_tokens, int nle,
    int max_recv, float scale, int row_vecs, int chunks, V* __restrict__ expert_y, int compact_rows) {
  __shared__ int red[NWAVES];
  __shared__ int pre[MAX_LOCAL_EXPERTS + 1];
  // compact_rows > 0: the experts' rows lie back to back in buffers of that many rows (= max_recv)
  int R = expert_prefix<NWAVES>(expert_num_tokens, nle, max_recv, pre, red);
  if (compact_rows > 0) R = min(R, compact_rows);
  const int top = top_step(nle);
  const int items = R * chunks;
  for (int q = blockIdx.x; q < items; q += gridDim.x) {
    const int g = chunks == 1 ? q : q / chunks, c = q - g * chunks;
    const int base = c * (BLOCK * NV);
    const int le = compact_rows > 0 ? 0 : expert_of(pre, nle, top, g);
    const size_t row = compact_rows > 0 ? (size_t)g : (size_t)le * max_recv + (g - pre[le]);
    Payload<V, NV> p;
    p.load(expert_x + row * row_vecs, base, row_vecs);
    p.map([scale](V v) { return standin_expert<V, DIN, DOUT>(v, scale); });
    p.template store<HOW>(expert_y + row * row_vecs, base, row_vecs);
  }
}

// The same for at most 64 local experts and 16-byte vectors: a wave per (row,
// chunk of 64 * NVW vectors), the expert prefix in one register per lane, the
// row found with one ballot. No LDS table, no barrier. Long streams take two vectors per lane and nontemporal loads (PAST; EXPERT_PAST_BYTES,
// csrc/stream_rules.h): 470 MB of rows among the other stages 170 -> 153 us, 29 MB 13.4 -> 12.8 (between events).
template <int NVW, int DIN, int DOUT, Store HOW, bool PAST>
__global__ __launch_bounds__(64 * ROWS) void expert_scale_wave_kernel(
    const b128* __restrict__ expert_x, const int* __restrict__ expert_num_tokens, int nle,
    int max_recv, float scale, int row_vecs, int chunks, b128* __restrict__ expert_y, int compact_rows) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const WaveExpertPrefix wp(expert_num_tokens, nle, max_recv);
  const int R = compact_rows > 0 ? min(wp.total, compact_rows) : wp.total;
  const int items = R * chunks, waves = gridDim.x * ROWS;
  for (int q = blockIdx.x * ROWS + wave; q < items; q += waves) {
    const int g = chunks == 1 ? q : q / chunks, c = q - g * chunks;
    const int base = c * (64 * NVW);
    int le, first;
    wp.locate(g, le, first);
    const size_t row = compact_rows > 0 ? (size_t)g : (size_t)le * max_recv + (g - first);
    WavePayload<b128, NVW> p;
    p.template load<PAST>(expert_x + row * row_vecs, base, row_vecs, lane);
#pragma unroll
    for (int j = 0; j < NVW; ++j) p.v[j] = standin_expert<b128, DIN, DOUT>(p.v[j], scale);
    p.template store<HOW>(expert_y + row * row_vecs, base, row_vecs, lane);
  }
}

// ---------------------------------------------------------------- expert computation: grouped GEMM
//
// expert_y[le, j, :] = expert_x[le, j, :] @ W[le]^T for the valid rows j < expert_num_tokens[le] of
// the padded expert-major buffers: what stands where all2all/reference.py:262 has the simulated
// expert. W[le] is [H_out = H, H_in = H] with the input index contiguous (the layout of a linear
// layer's weight).
//
// With a few dozen rows per expert the problem is bound by streaming the weights (C4: 3.3 GB of
// them for 0.2 PFLOP), so the kernel is built to keep weight bytes in flight and to ask for them in
// whole cache lines. A workgroup of GW waves (4, or 5 to 8 for blocks of 128 tokens) owns GW * 32
// output columns x one block of TJ*32 tokens of one expert; a wave owns 32 of the columns for all
// tokens of the block (TJ tiles of
// v_mfma_f32_32x32x16, fp32 accumulators in registers) and walks the input dimension 64 elements
// (128 bytes of every row) at a time.
//
// Weights: the MFMA wants a lane to hold inputs of ONE output column, which read from memory as
// it lies makes every load instruction touch 32 different lines, a quarter of each (measured: 4.0
// TB/s against 5.6 with the same bytes requested line by line). So a wave loads its 32 x 128 bytes
// of a step with 8 lanes per line, drops them into 4 KB of LDS of its own, and picks the operands
// up from there in MFMA layout. No barrier is involved: a wave's LDS operations execute in order.
// Tokens: the rows of the block are what the waves share. Each step's 128 bytes of every token
// are loaded once per workgroup, parked in LDS and read from there by all of them: one LDS barrier per
// step. Both kinds of loads are issued DEPTH steps ahead of their use; the vector memory counter
// retires in order, so the token loads run one step ahead of the weights: waiting for the tokens
// that are parked next never waits for the weights issued after them.
// LDS layout of both: row-major 128-byte rows, the eight 16-byte vectors of a row XORed with bits
// 1..3 of the row number, which makes the parking writes (8 lanes per row) and the operand reads
// (16 rows, same vector) hit all 64 banks once per 16 lanes.
//
// The MFMA computes the tile transposed (weights as the A operand, tokens as B), which leaves a lane
// holding four consecutive output columns of one token: 8-byte stores. MFMA q of a step takes inputs
// 16 q .. 16 q + 15 of the step (a lane's half kb of them: the 16-byte vector 2 q + kb of the row), the
// order in which dense_gemm_kernel walks K too: which of the two kernels a row count selects changes no
// bit of the result.
//
// Tiles are numbered over (expert, block of tokens) by a prefix over the device-side counts, so a
// hot expert is spread over as many workgroups as it has blocks and an empty one costs nothing.
// Every block of an expert re-reads the expert's weights: TJ = 4 (128 tokens) is used when the
// caller's row count says blocks of 64 would not hold most experts, TJ = 1 (32 tokens, 64 columns per
// workgroup) when experts have a handful of rows or there are few workgroups.

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int DT> struct Mfma32x32x16;
template <> struct Mfma32x32x16<MOE_A2A_BF16> {
  static __device__ __forceinline__ f32x16 mma(b128 a, b128 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma32x32x16<MOE_A2A_F16> {
  static __device__ __forceinline__ f32x16 mma(b128 a, b128 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

#ifndef MOE_A2A_GEMM_OCC
#define MOE_A2A_GEMM_OCC 3
#endif
#ifndef MOE_A2A_GEMM_OCC4
#define MOE_A2A_GEMM_OCC4 2  // workgroups per compute unit with blocks of 128 tokens
#endif
#ifndef MOE_A2A_GEMM_DEPTH
#define MOE_A2A_GEMM_DEPTH 2
#endif
constexpr int BUFFER_RAW_32BIT = 0x00020000;  // word 3 of a gfx9 buffer descriptor: raw buffer of 32-bit data
constexpr int BUFFER_STREAM = 2;  // cache policy of a buffer load: nontemporal
constexpr int GEMM_COLS = 128;   // output columns per workgroup (of four waves), 32 per wave
constexpr int GEMM_KSTEP = 64;   // input elements per step: 8 vectors of 16 bytes per row
#ifndef MOE_A2A_GEMM_DEPTH4
#define MOE_A2A_GEMM_DEPTH4 3  // with blocks of 128 tokens (two workgroups per unit: 655 against 675 us at C4)
#endif
constexpr int GEMM_DEPTH = MOE_A2A_GEMM_DEPTH;  // steps between a load and its use

// The step of K at which the product of group g starts (it goes round from there). Rows a multiple of 4 KB
// apart put the same step of every row on the same few memory channels, and workgroups that walk K side by
// side then all ask those: 256-row panels read at 4.6 TB/s with rows of 8 KB and 4.3 with 12 KB, at 6.1 with
// the panels started apart (5.1 and 5.6 with 4 KB; nothing between with 2, 6 and 14 KB). A function of the
// group alone, so every kernel adds up a group's products in the same order.
__device__ __forceinline__ int first_kstep(int g, int groups, int K) {
  return K % 2048 ? 0 : (int)((long long)g * (K / GEMM_KSTEP) / groups);
}

// x [groups, max_rows, K], w [groups, N, K], bias [groups, N] or null, y [groups, max_rows, N];
// rows_of_group null: every group has max_rows rows (a plain dense product when groups == 1).
// GW waves per workgroup, 32 output columns each: every workgroup of an expert pulls the expert's
// token rows through its own L1, so wider workgroups halve that traffic (GW = 8: one workgroup of
// 512 lanes per compute unit instead of two of 256).
// STREAMED: the weights leave nothing behind in the caches (weights_past_the_cache, csrc/tile_rules.h).
// TJ = 1: two waves per workgroup, and either many of those per unit (D = 2) or few with twice the lookahead.
template <int DT, int TJ, int GW, int D, bool STREAMED>
__global__ __launch_bounds__(64 * GW, GW > 4 || D > 3 ? 1 : TJ == 1 ? 4 : TJ == 2 ? MOE_A2A_GEMM_OCC : MOE_A2A_GEMM_OCC4) void expert_gemm_kernel(
    const b128* __restrict__ expert_x, const int* __restrict__ expert_num_tokens,
    const b128* __restrict__ weights, const uint16_t* __restrict__ bias, uint16_t* __restrict__ expert_y,
    int nle, int max_recv, int N, int K, int col_tiles, int compact) {
  constexpr int TOK = TJ * 32;               // tokens per block
  __shared__ b128 xs[D][TOK * 8];            // D steps of TOK tokens x 8 vectors
  constexpr int THREADS = 64 * GW;
  // the token rows of a step are fetched and parked by all lanes when their number divides the
  // block's vectors, else by the first four waves
  constexpr int LOADERS = (TOK * 8) % THREADS == 0 ? THREADS : 256;
  constexpr int XL = TOK * 8 / LOADERS;       // token loads of a loading lane per step (LOADERS / 8 rows each)
  static_assert(XL >= 1 && XL * LOADERS == TOK * 8 && LOADERS <= THREADS, "whole loads");
  __shared__ b128 ws[GW][32 * 8];            // per wave: one step of its 32 weight rows x 8 vectors
  __shared__ int red[GW], red_rows[GW];
  __shared__ int home[4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int row_vecs = K / 8, steps = (K + GEMM_KSTEP - 1) / GEMM_KSTEP;
  const int tail_vecs = row_vecs - (steps - 1) * 8;  // vectors of a row in the last step, 1..8
  auto rows_of = [=](int le) { return expert_num_tokens ? min(max(expert_num_tokens[le], 0), max_recv) : max_recv; };

  // Blocks of tokens per expert, summed over the run of experts this thread owns and scanned over
  // the workgroup: block number g of the launch belongs to the thread with begin <= g < begin + mine.
  const int per = (nle + THREADS - 1) / THREADS;
  const int run_b = min(tid * per, nle), run_e = min(run_b + per, nle);
  // compact: x and y hold the experts' rows back to back in buffers of max_recv rows. The rows
  // ahead of an expert are a prefix over the counts, and an expert only has the rows that still
  // fit the buffers (counts that add up to more never send a load or a store past their end).
  int mine_rows = 0;
  for (int le = run_b; le < run_e; ++le) mine_rows += rows_of(le);
  int rows_begin;
  {
    const int inc_rows = wave_inclusive_scan(mine_rows);
    if (lane == 63) red_rows[wave] = inc_rows;
    lds_barrier();
    int off_rows = 0;
#pragma unroll
    for (int w = 0; w < GW; ++w) off_rows += w < wave ? red_rows[w] : 0;
    rows_begin = off_rows + inc_rows - mine_rows;
  }
  // rows of expert le that are there: all of them in the padded layout
  auto kept_of = [=](int le, int ahead) {
    const int n = rows_of(le);
    return compact ? min(ahead + n, max_recv) - min(ahead, max_recv) : n;
  };
  auto blocks_for = [=](int rows) { return (rows + TOK - 1) / TOK; };
  int mine = 0;
  for (int le = run_b, ahead = rows_begin; le < run_e; ahead += rows_of(le), ++le) mine += blocks_for(kept_of(le, ahead));
  int begin, row_blocks;
  {
    const int inc = wave_inclusive_scan(mine);
    if (lane == 63) red[wave] = inc;
    lds_barrier();
    int off = 0, total = 0;
#pragma unroll
    for (int w = 0; w < GW; ++w) {
      off += w < wave ? red[w] : 0;
      total += red[w];
    }
    begin = off + inc - mine;
    row_blocks = total;
  }

  // Loads are 8 lanes per 128-byte row: lane l of a wave takes row l/8 (+ 8 per further load) and
  // the vector of that row that belongs in physical slot l%8.
  const int sub = lane >> 3, slot = lane & 7;
  // operand reads: row r of the tile, logical vector 2*q + kb of the step (q: the MFMA, kb: the lane's half)
  const int r = lane & 31, kb = lane >> 5, read_swz = (r >> 1) & 7;

  const int tiles = row_blocks * col_tiles, stride = gridDim.x;
  for (int tile = blockIdx.x; tile < tiles; tile += stride) {
    const int rb = tile / col_tiles, ct = tile - rb * col_tiles;
    if (begin <= rb && rb < begin + mine) {  // one thread: walk its run to the expert of block rb
      int le = run_b, first = begin, rows_ahead = rows_begin;
      for (;; ++le) {
        const int n = blocks_for(kept_of(le, rows_ahead));
        if (rb < first + n) break;
        first += n;
        rows_ahead += rows_of(le);
      }
      home[0] = le;
      home[1] = first;
      home[2] = min(rows_ahead, max_recv);
      home[3] = kept_of(le, rows_ahead);
    }
    lds_barrier();  // (the next write to `home` comes after the barriers of the steps below)
    // (uniform values are pinned to scalar registers: the bases below then cost no vector registers)
    const int le = __builtin_amdgcn_readfirstlane(home[0]);
    const int rows = __builtin_amdgcn_readfirstlane(home[3]);
    const int t0 = (rb - __builtin_amdgcn_readfirstlane(home[1])) * TOK;  // first token of the block (t0 < rows)
    const int first_step = first_kstep(le, nle, K);
    auto k_bytes = [=](int at) {  // byte of a row at which step number `at` of the walk begins
      const int k = at + first_step;
      return (k >= steps ? k - steps : k) * (GEMM_KSTEP * 2);
    };
    // buffer row of the expert's first row
    const size_t row0 = compact ? (size_t)__builtin_amdgcn_readfirstlane(home[2]) : (size_t)le * max_recv;
    const int n0 = ct * (GW * 32) + __builtin_amdgcn_readfirstlane(wave) * 32;  // first output column of this wave
    const bool cols_valid = n0 < N;                      // the last tile of columns may be partly empty
    const int nw = min(n0, N - 32);                      // (a wave without columns reads valid memory)

    // weights: load i takes rows sub + 8*i of the wave's 32; tokens: load i takes tokens tid/8 + 32*i.
    // Both go through buffer descriptors (base and extent in scalar registers, a 32-bit byte offset
    // per lane, the step's offset as the scalar operand). The extent of the token buffer ends with
    // the expert's last valid row: lanes that would load tokens past it get zeros and cause no
    // traffic. Tiles of 32 tokens with no valid token are skipped altogether. When K is not a
    // multiple of 64, the lanes that hold vectors past the end of a row in the last step are sent
    // out of range there the same way (both operands: a zero times a stray NaN would not be zero).
    const int live = rows - t0;  // valid tokens of this block, > 0
    const int row_bytes = K * 2;
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(weights + ((size_t)le * N + nw) * row_vecs), 0, 32 * row_bytes, BUFFER_RAW_32BIT);
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(expert_x + (row0 + t0) * row_vecs), 0, min(live, TOK) * row_bytes, BUFFER_RAW_32BIT);
    int woff[4], wslot[4], xoff[XL], wpast[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = sub + 8 * i, vec = slot ^ ((row >> 1) & 7);
      woff[i] = row * row_bytes + vec * 16;
      wslot[i] = row * 8 + slot;
      if (i < 2) wpast[i] = vec >= tail_vecs ? OUT_OF_RANGE : 0;  // (loads i and i + 2 take the same vector)
    }
    constexpr int XROWS = LOADERS / 8;  // token rows one load of the workgroup covers: 16, 32 or 64
    const bool loader = LOADERS == THREADS || tid < LOADERS;  // (whole waves)
    const int xrow = tid >> 3, xvec = slot ^ ((xrow >> 1) & 7);  // (XROWS * i does not change bits 1..3)
    const int xpast = xvec >= tail_vecs ? OUT_OF_RANGE : 0;
#pragma unroll
    for (int i = 0; i < XL; ++i) xoff[i] = (xrow + XROWS * i) * row_bytes + xvec * 16;

    f32x16 acc[TJ] = {};
    b128 wv[D][4], xv[D][XL];
    auto load_w = [&](int set, int step) {
      const int at = min(step, steps - 1);  // past the end: the last step again, unused
      const bool last = at == steps - 1;  // (rows of whole steps, the only ones that start elsewhere, have nothing past their end)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        wv[set][i] = __builtin_amdgcn_raw_buffer_load_b128(wbuf, woff[i] + (last ? wpast[i & 1] : 0),
                                                           k_bytes(at), STREAMED ? BUFFER_STREAM : 0);
    };
    auto load_x = [&](int set, int step) {
      const int at = min(step, steps - 1);
      const bool last = at == steps - 1;
      // (load i holds tokens XROWS * i .. of the block: a load without a valid token is neither
      // issued nor parked, and a tile of 32 tokens without one is not multiplied; what is left in the place
      // of a token that was not parked only reaches the results of that token, which are not stored)
#pragma unroll
      for (int i = 0; i < XL; ++i)
        if (loader && i * XROWS < live)
          xv[set][i] = __builtin_amdgcn_raw_buffer_load_b128(xbuf, xoff[i] + (last ? xpast : 0),
                                                             k_bytes(at), 0);
    };
    auto park_x = [&](int set) {
#pragma unroll
      for (int i = 0; i < XL; ++i)
        if (loader && i * XROWS < live) xs[set][tid + LOADERS * i] = xv[set][i];
    };
    auto compute = [&](int set) {
#pragma unroll
      for (int i = 0; i < 4; ++i) ws[wave][wslot[i]] = wv[set][i];
      b128 a[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] = ws[wave][r * 8 + ((q * 2 + kb) ^ read_swz)];
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          if (j * 32 < live) {
            const b128 tok = xs[set][(j * 32 + r) * 8 + ((q * 2 + kb) ^ read_swz)];
            acc[j] = Mfma32x32x16<DT>::mma(a[q], tok, acc[j]);
          }
        }
    };
    auto step = [&](int u, int at) {  // step `at`, which lives in register set and LDS buffer u = at % D
      compute(u);
      load_w(u, at + D);
      park_x((u + 1) % D);            // step at + 1, loaded one step before the weights now in flight
      load_x((u + 1) % D, at + 1 + D);
      lds_barrier();
    };

#pragma unroll
    for (int i = 0; i < D; ++i) {
      load_x(i, i);
      load_w(i, i);
    }
    park_x(0);
    load_x(0, D);
    lds_barrier();
    // D steps per trip, so that the register sets have fixed names in the loop body; the last
    // steps % D are peeled (inside the loop they would be paths on which set 0 follows set 0, and
    // the compiler would have to wait for the weights as if that happened)
    int at = 0;
    for (; at + D <= steps; at += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) step(u, at + u);
    }
#pragma unroll
    for (int u = 0; u < D - 1; ++u)
      if (at + u < steps) step(u, at + u);

    // D[n][token] of a 32x32 tile: this lane holds token r and output columns g*8 + kb*4 + 0..3, g < 4.
    // With a bias the sum is rounded to the 16-bit type first and the bias added to that, as
    // `matmul(x, w.T) + bias` on 16-bit tensors does (gemm-rs/reference.py:54-57).
    if (cols_valid) {
      uint32_t bias2[4][2] = {};
      if (bias) {
#pragma unroll
        for (int g = 0; g < 4; ++g) __builtin_memcpy(bias2[g], bias + (size_t)le * N + n0 + kb * 4 + g * 8, 8);
      }
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int token = t0 + j * 32 + r;
        if (token < rows) {
          uint16_t* out = expert_y + (row0 + token) * N + n0 + kb * 4;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x16& c = acc[j];
            uint32_t two[2] = {Pair16<DT>::canonical(Pair16<DT>::round(c[g * 4 + 0], c[g * 4 + 1])),
                               Pair16<DT>::canonical(Pair16<DT>::round(c[g * 4 + 2], c[g * 4 + 3]))};
            if (bias) {
#pragma unroll
              for (int h = 0; h < 2; ++h)
                two[h] = Pair16<DT>::canonical(Pair16<DT>::round(
                    __fadd_rn(Pair16<DT>::lo(two[h]), Pair16<DT>::lo(bias2[g][h])),
                    __fadd_rn(Pair16<DT>::hi(two[h]), Pair16<DT>::hi(bias2[g][h]))));
            }
            __builtin_memcpy(out + g * 8, two, 8);
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------- product with few rows
//
// Y[M, N] = X[M, K] @ W[N, K]^T where larger tiles would leave compute units without work (M = 64,
// N = 7168: 56 tiles of 128 columns; M = 255, N = 1728: 56 of 64 x 128). Here a
// workgroup owns only 32 output columns x one block of 32 or 64 tokens, and its KW waves (four,
// eight for long K) split K: wave w takes steps w, w + KW, ... of 64 elements, streams
// its own slices of the 32 weight rows and of the token rows (both 8 lanes per 128-byte line,
// turned into MFMA layout through LDS private to the wave: no barrier in the loop), and keeps
// partial sums in registers. At the end the partial sums meet in LDS and are added in a fixed
// order (wave 0 + 1 + 2 + ...), so results do not depend on scheduling.
// What bounds it: with more than 32 rows, what a unit can take in (a workgroup of 64 x 7168 x 2304 fetches 442 KB,
// two thirds of it token rows out of L2, and passes them all through LDS); with fewer, HBM or, on few columns, the
// trips of a wave. Of both, what it does not have to do counts: with waits that leave the younger step under way (the
// order of the loads is pinned, or the compiler waits for all of them), no loads past the last step, fragments read
// ahead of the MFMAs, and the final sums shared out over all waves: 64 x 7168 x 2304 11.1 -> 9.7 us, x 4608 23.5 -> 19.8,
// 64 x 2048 x 4608 16.2 -> 13.1, 16 x 7168 x 2304 8.8 -> 7.5, 1 x 4096 x 4096 9.4 -> 7.9, 64 x 8192 x 8192 36.5 -> 31.7.
// (16 x 16384 x 2048 15.4 -> 15.6: one workgroup per unit instead of two, for the registers.) A third step under way
// does not fit the registers beside 64 rows, and changes nothing with fewer.

template <int DT, int TJ, int KW, bool APART>
__global__ __launch_bounds__(64 * KW) void skinny_gemm_kernel(
    const b128* __restrict__ X, const b128* __restrict__ Wt, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ Y, int M, int N, int K, int row_units, uint32_t row_magic) {
  constexpr int TOK = TJ * 32;
  constexpr int XL = TJ * 4;  // token loads per lane and step: TOK rows x 8 vectors over 64 lanes
  extern __shared__ b128 skinny_lds[];  // per wave: 32 weight rows, then TOK token rows, of 8 vectors
  b128(*wsl)[32 * 8] = reinterpret_cast<b128(*)[32 * 8]>(skinny_lds);
  b128(*xsl)[TOK * 8] = reinterpret_cast<b128(*)[TOK * 8]>(skinny_lds + KW * 32 * 8);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int row_vecs = K / 8, row_bytes = K * 2, steps = (K + GEMM_KSTEP - 1) / GEMM_KSTEP;
  const int tail_vecs = row_vecs - (steps - 1) * 8;
  // Row blocks of the same columns run beside each other on one XCD: its L2 then has the weights for all but the first
  // (us, row blocks numbered last / first: 140 x 3008 x 4680 28.3 / 21.1, 37 x 3968 x 936 5.7 / 4.75, 81 x 2176 x 7488
  // 15.2 / 13.7). row_magic = ceil(2^32 / row_units): exact for the up to 10240 workgroups, and a division less to wait for.
  int rb = 0, cu = blockIdx.x;
  if (row_units > 1) {
    const int logical = xcd_contiguous(blockIdx.x, N / 32 * row_units);
    cu = __umulhi((uint32_t)logical, row_magic);
    rb = logical - cu * row_units;
  }
  const int t0 = rb * TOK, n0 = cu * 32, live = M - t0;
  // APART: where rows lie a multiple of 4 KB apart (see first_kstep) workgroups start apart too, by whole turns of
  // the waves, so that a wave keeps its steps: 8 x 8192 x 8192 34.1 -> 25.6 us, 1 x 4096 x 4096 12.4 -> 9.5, 64 x
  // 8192 x 8192 41 -> 38, 16 x 16384 x 2048 16.0 -> 14.6. Elsewhere going round costs 0.8 % (64 x 7168 x 2304 11.29 us,
  // 11.20 without).
  static_assert(32 % KW == 0, "whole turns in the steps of 2048 inputs");
  const int first_step = APART ? (int)((uint32_t)cu * (steps / KW) / ((uint32_t)N / 32)) * KW : 0;

  const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(Wt + (size_t)n0 * row_vecs), 0, 32 * row_bytes, BUFFER_RAW_32BIT);
  const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(X + (size_t)t0 * row_vecs), 0, min(live, TOK) * row_bytes, BUFFER_RAW_32BIT);
  // load i of a lane: row sub + 8 * i, the vector that belongs in physical slot `slot` of that row
  const int sub = lane >> 3, slot = lane & 7;
  auto vec_of = [&](int row) { return slot ^ ((row >> 1) & 7); };
  const int r = lane & 31, kb = lane >> 5, read_swz = (r >> 1) & 7;

  f32x16 acc[TJ] = {};
  b128 wv[2][4], xv[2][XL];
  int woff[2];  // (rows 16 apart take the same vector)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = sub + 8 * i;
    woff[i] = row * row_bytes + vec_of(row) * 16;
  }
  auto load = [&](int set, int step) __attribute__((always_inline)) {
    const int k = step + first_step, soff = (APART && k >= steps ? k - steps : k) * (GEMM_KSTEP * 2);
    int off[2];  // (past the end of the rows in the last step: out of range, zeros)
#pragma unroll
    for (int i = 0; i < 2; ++i) off[i] = woff[i] + (step == steps - 1 && vec_of(sub + 8 * i) >= tail_vecs ? OUT_OF_RANGE : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      wv[set][i] = __builtin_amdgcn_raw_buffer_load_b128(wbuf, off[i & 1] + (i >> 1) * 16 * row_bytes, soff, 0);
#pragma unroll
    for (int i = 0; i < XL; ++i)
      xv[set][i] = __builtin_amdgcn_raw_buffer_load_b128(xbuf, off[i & 1] + (i >> 1) * 16 * row_bytes, soff, 0);
  };
  auto compute = [&](int set) {
#pragma unroll
    for (int i = 0; i < 4; ++i) wsl[wave][(sub + 8 * i) * 8 + slot] = wv[set][i];
#pragma unroll
    for (int i = 0; i < XL; ++i) xsl[wave][(sub + 8 * i) * 8 + slot] = xv[set][i];
    b128 a[4], tok[TJ][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a[q] = wsl[wave][r * 8 + ((kb * 4 + q) ^ read_swz)];
#pragma unroll
      for (int j = 0; j < TJ; ++j) tok[j][q] = xsl[wave][(j * 32 + r) * 8 + ((kb * 4 + q) ^ read_swz)];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < TJ; ++j) acc[j] = Mfma32x32x16<DT>::mma(a[q], tok[j][q], acc[j]);
    __builtin_amdgcn_sched_barrier(0);
  };

  // The wave's n steps (two at least: the launch sees to it), two of them under way. Nothing is asked for past the
  // last one (a load out of range takes its turn in the address unit all the same: 0.7 us for the eight waves' loads of
  // a step), and no load in the loop is conditional (the wait for a step has to know how many are younger).
  const int n = (steps - wave + KW - 1) / KW;
  auto load_step = [&](int set, int i) __attribute__((always_inline)) {
    load(set, wave + i * KW);
    __builtin_amdgcn_sched_barrier(0);  // (in this order, which the waits count on)
  };
  load_step(0, 0);
  load_step(1, 1);
  int i = 0;
  for (; i + 4 <= n; i += 2) {
    compute(0);
    load_step(0, i + 2);
    compute(1);
    load_step(1, i + 3);
  }
  compute(0);
  if (n - i == 3) {
    load_step(0, i + 2);
    compute(1);
    compute(0);
  } else {
    compute(1);
  }

  // Partial sums to LDS (a wave's region holds exactly its TJ x 16 floats per lane), 16 bytes at a time; then every wave
  // adds up a share of the four quarters of the token tiles, each in the order of the waves, and writes it out.
  f32x4* mine = reinterpret_cast<f32x4*>(xsl[wave]);
#pragma unroll
  for (int j = 0; j < TJ; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) mine[(j * 4 + g) * 64 + lane] = f32x4{acc[j][g * 4], acc[j][g * 4 + 1], acc[j][g * 4 + 2], acc[j][g * 4 + 3]};
  __syncthreads();
#pragma unroll
  for (int p = 0; p < (TJ * 4 + KW - 1) / KW; ++p) {
    const int share = p * KW + wave, j = share % TJ, g = share / TJ;
    if (g >= 4 || j * 32 >= live) continue;
    f32x4 c = reinterpret_cast<const f32x4*>(xsl[0])[(j * 4 + g) * 64 + lane];
#pragma unroll
    for (int w = 1; w < KW; ++w) {
      const f32x4 more = reinterpret_cast<const f32x4*>(xsl[w])[(j * 4 + g) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) c[e] = __fadd_rn(c[e], more[e]);
    }
    // this lane: token r of tile j, output columns n0 + g*8 + kb*4 + 0..3
    const int token = t0 + j * 32 + r;
    if (token < M) {
      uint32_t two[2] = {Pair16<DT>::canonical(Pair16<DT>::round(c[0], c[1])), Pair16<DT>::canonical(Pair16<DT>::round(c[2], c[3]))};
      if (bias) {
        uint32_t b2[2];
        __builtin_memcpy(b2, bias + n0 + kb * 4 + g * 8, 8);
#pragma unroll
        for (int h = 0; h < 2; ++h)
          two[h] = Pair16<DT>::canonical(Pair16<DT>::round(
              __fadd_rn(Pair16<DT>::lo(two[h]), Pair16<DT>::lo(b2[h])),
              __fadd_rn(Pair16<DT>::hi(two[h]), Pair16<DT>::hi(b2[h]))));
      }
      __builtin_memcpy(Y + (size_t)token * N + n0 + kb * 4 + g * 8, two, 8);
    }
  }
}

// ---------------------------------------------------------------- dense product (many rows)
//
// C[M, N] = A[M, K] @ B[N, K]^T for outputs that tiles of 256 columns (phased_gemm_kernel) would spread over
// too few compute units, and for experts' rows (GROUPED) also where those would leave much of a last round idle. A
// workgroup of four waves owns a BM x BN tile of C (128 x 128; 64 x 128 and products of one round are sliced_gemm_kernel's) and walks K in steps of
// 64 elements. Per step the workgroup copies BM + BN rows of 128 bytes into LDS once (through registers, two LDS
// buffers, one barrier per step), and every wave reads each operand fragment it needs once per 16-element slice
// of the step for a whole row or column of its MFMA tiles, issued one slice ahead.
// The loop body is laid out by hand (sched_group_barrier): memory instructions spread over the MFMAs, and every
// slice of a step carries the same mix. Loads or stores issued back to back make the wave wait for the queues of
// the memory pipes, which its neighbours fill at the same moment, and the matrix core idles meanwhile.
// LDS rows are 128 bytes with the eight 16-byte vectors of a row XORed with bits 1..3 of the
// row number (reads of 32 rows at one vector hit every bank equally); a thread stores linearly and
// picks the global vector that belongs at its place, so the stores are conflict-free too.
// The tile is computed transposed (B rows as the first MFMA operand): a lane then holds four
// consecutive columns of one row of C.
// Tiles are numbered so that each XCD (blockIdx % 8) works on a run of consecutive tile numbers,
// and consecutive numbers walk GROUP_M tile rows down before they step to the next tile column:
// the 32 workgroups an XCD runs at a time share 4 row panels of A and 8 of B in its L2.

template <int DT, int WM, int WN, int TM, int TN, bool GROUPED, bool STREAMED = false>
__global__ __launch_bounds__(64 * WM * WN, 2) void dense_gemm_kernel(
    const b128* __restrict__ A, const b128* __restrict__ B, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n,
    const int* __restrict__ rows_of_group, int groups, int max_rows, int compact) {
  constexpr int NT = 64 * WM * WN, BM = WM * TM * 32, BN = WN * TN * 32;
  constexpr int LA = BM * 8 / NT, LB = BN * 8 / NT;  // 16-byte vectors a thread copies per step
  constexpr int GROUP_M = 4;
  extern __shared__ b128 tile_lds[];  // [2][(BM + BN) * 8]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = __builtin_amdgcn_readfirstlane(wave / WN), wn = __builtin_amdgcn_readfirstlane(wave % WN);
  const int row_vecs = K / 8, row_bytes = K * 2, steps = (K + GEMM_KSTEP - 1) / GEMM_KSTEP;
  const int tail_vecs = row_vecs - (steps - 1) * 8;

  // GROUPED: A is [groups, max_rows, K], B [groups, N, K], bias [groups, N] or null, C [groups,
  // max_rows, N], and group g has rows_of_group[g] rows (read here, clamped to max_rows). Row
  // tiles are numbered over the groups by a prefix over their counts: every thread sums the row
  // tiles of a run of groups, a scan over the workgroup places the runs, and the thread whose run
  // holds a row tile walks it to find the group. The launch strides over (row tile, column tile)
  // pairs, column tile fastest, so its size is a matter of speed only.
  __shared__ int grp_red[NT / 64], grp_red_rows[NT / 64];
  __shared__ int grp_home[4];
  [[maybe_unused]] auto rows_of = [=](int g) { return min(max(rows_of_group[g], 0), max_rows); };
  // compact: A and C hold the groups' rows back to back in buffers of max_rows rows. The rows
  // ahead of a group are a prefix over the counts, and a group only has the rows that still fit
  // the buffers (counts that add up to more never send a load or a store past their end).
  [[maybe_unused]] auto kept_of = [=](int g, int ahead) {
    const int n = rows_of(g);
    return compact ? min(ahead + n, max_rows) - min(ahead, max_rows) : n;
  };
  [[maybe_unused]] auto tiles_for = [=](int rows) { return (rows + BM - 1) / BM; };
  [[maybe_unused]] int run_first = 0, run_end = 0, run_begin = 0, run_tiles = 0, total_tiles = 0, run_rows_begin = 0;
  if constexpr (GROUPED) {
    const int per = (groups + NT - 1) / NT;
    run_first = min(tid * per, groups);
    run_end = min(run_first + per, groups);
    int run_rows = 0;
    for (int g = run_first; g < run_end; ++g) run_rows += rows_of(g);
    const int inc_rows = wave_inclusive_scan(run_rows);
    if (lane == 63) grp_red_rows[wave] = inc_rows;
    lds_barrier();
    int off_rows = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) off_rows += w < wave ? grp_red_rows[w] : 0;
    run_rows_begin = off_rows + inc_rows - run_rows;
    for (int g = run_first, ahead = run_rows_begin; g < run_end; ahead += rows_of(g), ++g)
      run_tiles += tiles_for(kept_of(g, ahead));
    const int inc = wave_inclusive_scan(run_tiles);
    if (lane == 63) grp_red[wave] = inc;
    lds_barrier();
    int off = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
      off += w < wave ? grp_red[w] : 0;
      total += grp_red[w];
    }
    run_begin = off + inc - run_tiles;
    total_tiles = total * tiles_n;
    if ((int)blockIdx.x >= total_tiles) return;
  }
  int tile = blockIdx.x;
  do {  // (one pass unless GROUPED)
  int n0, rows_left;          // first column of the tile; rows of A and C from the tile's first row on
  const b128* a_tile;         // the tile's first row of A
  const b128* b_tile;         // the tile's first row of B (column n0 of the product)
  uint16_t* c_tile;           // the tile's first row of C
  const uint16_t* bias_row;   // the bias of the tile's group, or null
  [[maybe_unused]] int k_first = 0;  // the step of K at which the tile starts
  if constexpr (GROUPED) {
    // whole rounds of the launch are renumbered so that an XCD works on consecutive pairs
    // (the column tiles of one row tile share its rows in that XCD's L2)
    const int round = tile / (int)gridDim.x;
    int logical = tile;
    if ((round + 1) * (int)gridDim.x <= total_tiles)
      logical = round * (int)gridDim.x + xcd_contiguous(blockIdx.x, gridDim.x);
    const int rb = logical / tiles_n, tn = logical - rb * tiles_n;
    lds_barrier();  // the tile before is out of LDS, and its grp_home has been read
    if (run_begin <= rb && rb < run_begin + run_tiles) {
      int g = run_first, first = run_begin, rows_ahead = run_rows_begin;
      for (;; ++g) {
        const int n = tiles_for(kept_of(g, rows_ahead));
        if (rb < first + n) break;
        first += n;
        rows_ahead += rows_of(g);
      }
      grp_home[0] = g;
      grp_home[1] = first;
      grp_home[2] = min(rows_ahead, max_rows);
      grp_home[3] = kept_of(g, rows_ahead);
    }
    lds_barrier();
    const int g = __builtin_amdgcn_readfirstlane(grp_home[0]);
    const int t0 = (rb - __builtin_amdgcn_readfirstlane(grp_home[1])) * BM;
    const size_t row0 = compact ? (size_t)__builtin_amdgcn_readfirstlane(grp_home[2]) : (size_t)g * max_rows;
    n0 = tn * BN;
    rows_left = __builtin_amdgcn_readfirstlane(grp_home[3]) - t0;
    a_tile = A + (row0 + t0) * row_vecs;
    b_tile = B + ((size_t)g * N + n0) * row_vecs;
    k_first = first_kstep(g, groups, K);
    c_tile = C + (row0 + t0) * N;
    bias_row = bias ? bias + (size_t)g * N : nullptr;
  } else {
    const int logical = xcd_contiguous(blockIdx.x, gridDim.x);
    const int per_group = GROUP_M * tiles_n, group = logical / per_group, in = logical - group * per_group;
    const int rows = min(GROUP_M, tiles_m - group * GROUP_M);
    const int tn = in / rows, tm = group * GROUP_M + in - tn * rows;
    n0 = tn * BN;
    rows_left = M - tm * BM;
    a_tile = A + (size_t)tm * BM * row_vecs;
    b_tile = B + (size_t)n0 * row_vecs;
    c_tile = C + (size_t)tm * BM * N;
    bias_row = bias;
  }

  // Loads go through buffer descriptors whose extent ends with the last row of the matrix: rows of
  // a tile past it read as zeros. Vectors past the end of a row in the last step are sent out of
  // range the same way.
  const __amdgpu_buffer_rsrc_t abuf = __builtin_amdgcn_make_buffer_rsrc(
      (void*)a_tile, 0, min(BM, rows_left) * row_bytes, BUFFER_RAW_32BIT);
  const __amdgpu_buffer_rsrc_t bbuf = __builtin_amdgcn_make_buffer_rsrc(
      (void*)b_tile, 0, min(BN, N - n0) * row_bytes, BUFFER_RAW_32BIT);
  // copy i of a thread: LDS place p = tid + i * NT, that is row p / 8 (rows NT / 8 apart, which
  // leaves bits 1..3 of the row number alone) and the vector that belongs in physical slot p % 8
  const int crow = tid >> 3, cvec = (tid & 7) ^ ((crow >> 1) & 7);
  const int coff = crow * row_bytes + cvec * 16;
  const int cpast = cvec >= tail_vecs ? OUT_OF_RANGE : 0;
  const int rstep = (NT / 8) * row_bytes;

  b128 ga[LA], gb[LB];
  // A thread's LA + LB vectors of a step in four quarters: A[0..LA/2), A[LA/2..LA), B[0..LB/2), B[LB/2..LB)
  static_assert(LA % 2 == 0 && LB % 2 == 0, "quarters");
  auto load_quarter = [&](int q, int step) __attribute__((always_inline)) {
    const int at = min(step, steps - 1);  // (past the end: the last step again, never used)
    const int k = GROUPED && at + k_first >= steps ? at + k_first - steps : at + k_first;
    const int soff = k * (GEMM_KSTEP * 2), off = coff + (at == steps - 1 ? cpast : 0);
    if (q < 2) {
#pragma unroll
      for (int i = q * (LA / 2); i < (q + 1) * (LA / 2); ++i)
        ga[i] = __builtin_amdgcn_raw_buffer_load_b128(abuf, off + i * rstep, soff, 0);
    } else {
#pragma unroll
      for (int i = (q - 2) * (LB / 2); i < (q - 1) * (LB / 2); ++i)
        gb[i] = __builtin_amdgcn_raw_buffer_load_b128(bbuf, off + i * rstep, soff, STREAMED ? BUFFER_STREAM : 0);
    }
  };
  auto store_quarter = [&](int q, int buf) __attribute__((always_inline)) {
    b128* as = tile_lds + buf * ((BM + BN) * 8);
    b128* bs = as + BM * 8;
    if (q < 2) {
#pragma unroll
      for (int i = q * (LA / 2); i < (q + 1) * (LA / 2); ++i) as[tid + i * NT] = ga[i];
    } else {
#pragma unroll
      for (int i = (q - 2) * (LB / 2); i < (q - 1) * (LB / 2); ++i) bs[tid + i * NT] = gb[i];
    }
  };

  const int r = lane & 31, h = lane >> 5, swz = (r >> 1) & 7;
  f32x16 acc[TM][TN] = {};
  // Operand fragments of one 16-element slice of a step: two register sets, so that the reads of
  // the next slice are in flight while the matrix cores work on this one.
  b128 af[2][TM], bf[2][TN];
  auto read_frags = [&](int set, int buf, int kk) __attribute__((always_inline)) {
    const b128* as = tile_lds + buf * ((BM + BN) * 8) + (wm * TM * 32 + r) * 8;
    const b128* bs = tile_lds + buf * ((BM + BN) * 8) + BM * 8 + (wn * TN * 32 + r) * 8;
    const int v = (kk * 2 + h) ^ swz;
#pragma unroll
    for (int i = 0; i < TM; ++i) af[set][i] = as[i * 256 + v];
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[set][j] = bs[j * 256 + v];
  };
  // (GROUPED) bands of 32 rows of this wave's part of the tile that hold rows of the group: the
  // last row tile of a group computes only those, in a copy of the loop with that one condition
  constexpr bool SKIP_BANDS = GROUPED;
  [[maybe_unused]] const int live_bands = min(max((rows_left - wm * TM * 32 + 31) / 32, 0), TM);
  auto mfmas = [&](int set, auto ragged) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (decltype(ragged)::value && i >= live_bands) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = Mfma32x32x16<DT>::mma(bf[set][j], af[set][i], acc[i][j]);
    }
  };

  // Step s computes from LDS buffer s & 1. During it the rows of step s + 1 (in registers since
  // the step before) go to the other buffer, the rows of step s + 2 are requested from memory,
  // and the one barrier of the step sits before its last slice: behind it the first fragments
  // of step s + 1 are read while the matrix cores finish step s.
  // State at the start of step s: LDS buffer s & 1 holds the rows of step s; the other buffer
  // holds quarter 0 of step s + 1; the registers hold quarter 0 of step s + 2 and quarters 1..3
  // of step s + 1. Every slice of a step stores one quarter and requests its replacement, so
  // that the memory pipes see an even stream (four waves issuing all their loads in the same
  // slice oversubscribe the address unit while it idles in the others). Writes into a buffer
  // are legal from the barrier of the step that last read it to the barrier before the step that
  // reads it next: the last slice of step s - 1 and the first three of step s.
#pragma unroll
  for (int q = 0; q < 4; ++q) load_quarter(q, 0);
#pragma unroll
  for (int q = 0; q < 4; ++q) store_quarter(q, 0);
#pragma unroll
  for (int q = 0; q < 4; ++q) load_quarter(q, 1);
  store_quarter(0, 1);
  load_quarter(0, 2);
  __syncthreads();
  read_frags(0, 0, 0);
  // A wave that issues its loads or stores back to back waits for the queues of the memory pipes and issues no
  // MFMA meanwhile: a slice's TM + TN fragment reads and one quarter's stores and loads are spread over its
  // TM * TN MFMAs.
  constexpr int N_MFMA = TM * TN, N_QUARTER = (LA > LB ? LA : LB) / 2;
  constexpr int READS_EACH = (TM + TN + N_MFMA - 1) / N_MFMA, MOVES_EACH = (N_QUARTER + N_MFMA - 1) / N_MFMA;
#define MOE_A2A_INTERLEAVE()                                            \
    _Pragma("unroll") for (int q = 0; q < N_MFMA; ++q) {                \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                \
      __builtin_amdgcn_sched_group_barrier(0x100, READS_EACH, 0);       \
      __builtin_amdgcn_sched_group_barrier(0x200, MOVES_EACH, 0);       \
      __builtin_amdgcn_sched_group_barrier(0x020, MOVES_EACH, 0);       \
    }                                                                   \
  __builtin_amdgcn_sched_barrier(0);
  auto one_step = [&](int step, int cur, auto ragged) __attribute__((always_inline)) {  // cur = step & 1, a constant where this is called
    read_frags(1, cur, 1);
    store_quarter(1, cur ^ 1);
    load_quarter(1, step + 2);
    mfmas(0, ragged);
    MOE_A2A_INTERLEAVE()
    read_frags(0, cur, 2);
    store_quarter(2, cur ^ 1);
    load_quarter(2, step + 2);
    mfmas(1, ragged);
    MOE_A2A_INTERLEAVE()
    read_frags(1, cur, 3);
    store_quarter(3, cur ^ 1);
    load_quarter(3, step + 2);
    mfmas(0, ragged);
    MOE_A2A_INTERLEAVE()
    lds_barrier();
    read_frags(0, cur ^ 1, 0);
    store_quarter(0, cur);
    load_quarter(0, step + 3);
    mfmas(1, ragged);
    MOE_A2A_INTERLEAVE()
  };
  auto walk_k = [&](auto ragged) __attribute__((always_inline)) {
    int step = 0;
    for (; step + 2 <= steps; step += 2) {
      one_step(step, 0, ragged);
      one_step(step + 1, 1, ragged);
    }
    if (step < steps) one_step(step, 0, ragged);
  };
  // (both copies hold the same barriers, so the waves of a workgroup may take different ones)
  if (!SKIP_BANDS || live_bands == TM) walk_k(std::false_type{});
  else if constexpr (SKIP_BANDS) walk_k(std::true_type{});

  // Results leave through LDS so that they reach memory in whole lines. acc[i][j] holds row
  // i*32 + r of the wave's tile and columns j*32 + g*8 + h*4 + 0..3 (g < 4): a lane's own values
  // are 8-byte pieces of 32 different rows. Each wave parks one band of 32 rows at a time in a
  // region of its own (rows padded by 16 bytes so that they start in different banks; a wave's
  // LDS operations execute in order, so no barrier is needed inside it) and reads it back with
  // 16 lanes per row: a store instruction then writes four 256-byte row segments. They write through (Store):
  // 1500 x 2304 x 360 8.7 -> 7.9 us, 1586 x 2432 x 1536 16.8 -> 15.8, with a kernel behind it that reads the result
  // 21.2 -> 20.1; experts' products, plain / through / streaming: 7 x 57 rows, 2656 x 1152 13.4 / 13.2 / 13.3 and with
  // the reader 18.7 / 18.5 / 19.6; 32 x 100 rows, 2720 x 1024 52.4 / 51.9 / 50.2 and 61.2 / 60.2 / 60.8.
  __syncthreads();  // every wave has read its last fragments: the operand tiles can be overwritten
  {
    constexpr int VR = TN * 4;            // 16-byte vectors per row of the wave's tile
    constexpr int PITCH = TN * 64 + 16;   // bytes per parked row
    constexpr int ROWS_PER_READ = 64 / VR;
    char* park = (char*)tile_lds + wave * (32 * PITCH);
    const int ncol = n0 + wn * TN * 32;
    uint32_t bias2[TN][4][2] = {};
    if (bias_row) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (ncol + j * 32 < N) __builtin_memcpy(bias2[j][g], bias_row + ncol + j * 32 + g * 8 + h * 4, 8);
    }
    const int rrow = lane / VR, rvec = lane % VR;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (SKIP_BANDS && i >= live_bands) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const f32x16& c = acc[i][j];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          uint32_t two[2] = {Pair16<DT>::canonical(Pair16<DT>::round(c[g * 4 + 0], c[g * 4 + 1])),
                             Pair16<DT>::canonical(Pair16<DT>::round(c[g * 4 + 2], c[g * 4 + 3]))};
          if (bias_row) {
#pragma unroll
            for (int e = 0; e < 2; ++e)
              two[e] = Pair16<DT>::canonical(Pair16<DT>::round(
                  __fadd_rn(Pair16<DT>::lo(two[e]), Pair16<DT>::lo(bias2[j][g][e])),
                  __fadd_rn(Pair16<DT>::hi(two[e]), Pair16<DT>::hi(bias2[j][g][e]))));
          }
          __builtin_memcpy(park + r * PITCH + (j * 32 + g * 8 + h * 4) * 2, two, 8);
        }
      }
#pragma unroll
      for (int p = 0; p < 32 / ROWS_PER_READ; ++p) {
        const int row = p * ROWS_PER_READ + rrow;
        const b128 v = *(const b128*)(park + row * PITCH + rvec * 16);
        const int m = (wm * TM + i) * 32 + row, n = ncol + rvec * 8;
        if (m < rows_left && n < N) row_store<THROUGH>((b128*)(c_tile + (size_t)m * N + n), v);
      }
    }
  }
  tile += gridDim.x;
  } while (GROUPED && tile < total_tiles);
}

#undef MOE_A2A_INTERLEAVE

// ---------------------------------------------------------------- dense product, 256 columns per tile
//
// The same product for tiles large enough to keep the matrix cores busy. A workgroup of eight waves
// (two per SIMD) owns 32 * TM rows x 64 * TN columns; a wave owns TM bands of 16 rows (every second band
// of the tile) x TN columns of 16 and uses v_mfma_f32_16x16x32. What shaped it:
//  - Power. With every matrix core busy on ordinary data the clock, not the pipe, sets the rate: from
//    registers alone 32x32x16 runs at 1.80 PFLOP/s and 16x16x32 at 2.06 (2.4 of either on zeros), because it
//    reads and writes an accumulator half as often per product.
//  - Rows go from memory to LDS directly (buffer_load ... lds): no registers, no ds_write, and what is
//    saved there is clock for the matrix cores.
//  - Two groups of four waves take turns ("phases", a barrier apart): while one group multiplies, the other
//    reads its next fragments (32 elements of K) and asks for rows. A wave thus needs one set of fragments,
//    and no memory instruction ever stands between two MFMAs of the group that owns the matrix cores.
//  - Phases have to be even: rows of one operand are requested in the first slice of a step and rows of the
//    other in the second. All of them in one phase cost 12 % (324 against 363 us at 8192 x 8192 x 3712).
//  - Lookahead: 160 KB hold five half-steps of 32 KB. One operand gets three buffers and is asked for two steps
//    ahead, the other two buffers and one step; with two of each, rows that start off the 128-byte lines
//    (K = 3696) ran 17 % longer (399 against 340 us). Steps of 32 elements in a ring of five buffers look
//    farther ahead but ask for half lines: 425 against 380 us at K = 4096.
//  - Rows that start off the lines take one and three quarter times the line requests: AHEAD then brings the
//    lines into L2 before (operands out of HBM, K = 3696: 390 -> 372 us; on aligned rows it costs 1 to 2 %).
//  - GROUPED (the experts' products): a group's weights are read for a few hundred rows only, most lines come
//    from HBM, and the loads bound it. The fewer tiles the better: up to 320 rows per tile, spread evenly over the
//    tiles of a group, and only the bands of 32 rows that there are get fetched and multiplied. Beside two buffers
//    of 320 rows of A there is room for five halves of B (128 columns each): the ring of halves keeps half a
//    step of weights under way while the rows of the next step are waited for, and rows of A have a whole step to
//    arrive. 32 groups x 256 rows, 2048 x 4096: 208 us with dense_gemm_kernel's 128 x 128 tiles, 151 with two whole
//    buffers of either operand, which leave nothing under way then, 137 here (131 without the MFMAs, 99 without the
//    loads, 107 with the weights alone, which is their rate out of HBM in this pattern); 4096 x 2048 161 -> 147.
// Measured at 8192 x 8192 (bf16, uniform values, clocks settled): K = 3696 395 us with dense_gemm_kernel's
// 256 x 256 tile, 340 here (1.46 PFLOP/s); K = 4096 x 4096 x 4096 107 and 90; K = 8192 795 and 702.
//
// Order of K: MFMA q of a step takes inputs 32 q .. 32 q + 31. The instruction adds them as two runs of 16 in
// that order, so a row count that selects this kernel or another changes no bit of the result.
// LDS rows are 128 bytes, the eight 16-byte vectors of a row XORed with bits 1..3 of the row number, as above;
// a direct load writes 1 KB (eight rows) in lane order, so the lane picks the vector that belongs at its place.

// 16 bytes per lane from a buffer into LDS at `base` + OFF + 16 * lane. The place travels in m0, which the compiler
// sets (so that it knows what m0 holds); the instruction is written out, as the wait for it, through vmcnt, is the
// caller's. One wait state between the two.
template <int OFF, bool STREAMED = false>
__device__ __forceinline__ void load_to_lds(unsigned base, int voffset, b128 rsrc, int soffset) {
  if constexpr (STREAMED)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 ::"{m0}"(base + OFF), "v"(voffset), "s"(rsrc), "s"(soffset) : "memory");
  else
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"{m0}"(base + OFF), "v"(voffset), "s"(rsrc), "s"(soffset) : "memory");
}
// the descriptor of such a load, as __builtin_amdgcn_make_buffer_rsrc lays it out
__device__ __forceinline__ b128 buffer_words(const void* p, int bytes) {
  const uint64_t a = (uint64_t)p;
  return b128{(unsigned)a, (unsigned)(a >> 32) & 0xffffu, (unsigned)bytes, (unsigned)BUFFER_RAW_32BIT};
}

template <int I, int END, typename F>
__device__ __forceinline__ void unrolled(F&& f) {  // f(0), f(1), ... with constants
  if constexpr (I < END) {
    f(std::integral_constant<int, I>{});
    unrolled<I + 1, END>(f);
  }
}

constexpr int WAIT_LDS_ONLY = 0xC07F;  // s_waitcnt lgkmcnt(0), the other counters left alone

template <int DT> struct Mfma16x16x32;
template <> struct Mfma16x16x32<MOE_A2A_BF16> {
  static __device__ __forceinline__ f32x4 mma(b128 a, b128 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma16x16x32<MOE_A2A_F16> {
  static __device__ __forceinline__ f32x4 mma(b128 a, b128 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

constexpr int phased_rows(int TM) { return 32 * TM; }
constexpr int phased_cols(int TN) { return 64 * TN; }
constexpr size_t phased_lds_bytes(int TM, int TN, int NA, int HB) {  // NA buffers of A, HB half buffers of B
  return (size_t)(NA * phased_rows(TM) + HB * phased_cols(TN) / 2) * 128;
}

// Tiles of a grouped product: A is [groups, max_rows, K], B [groups, N, K], C [groups, max_rows, N], and group g
// has rows_of_group[g] rows (read here, clamped to max_rows). A group's rows are spread evenly over the fewest
// tiles of BM rows, in whole bands of 32; tiles are numbered by group, column tile and row tile, so that
// neighbours share the group's weights. compact: A and C hold the groups' rows back to back in buffers of
// max_rows rows. The rows ahead of a group are a prefix over the counts, and a group only has the rows that
// still fit the buffers (counts that add up to more never send a load or a store past their end).
struct GroupTile {
  int total;       // tiles of the product; the rest holds for a tile below that
  int group, tn;   // group and column tile
  int rows;        // rows of the tile, at least 1
  size_t row_at;   // its first row in A and C
};

// Every thread sums the tiles of a run of groups, a scan over the workgroup (NT lanes) places the runs, and the
// thread whose run holds the tile walks it to find the group. `lds` is 20 ints that nobody else uses until the
// barrier after the call.
template <int NT, int BM>
__device__ __forceinline__ GroupTile find_group_tile(int tile, const int* __restrict__ rows_of_group, int groups,
                                                     int max_rows, int tiles_n, bool compact, int* lds) {
  constexpr int NW = NT / 64;
  static_assert(NW <= 8, "20 ints");
  int* const red = lds;
  int* const red_rows = lds + 8;
  int* const home = lds + 16;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  auto rows_of = [=](int g) { return min(max(rows_of_group[g], 0), max_rows); };
  auto kept_of = [=](int g, int ahead) {
    const int n = rows_of(g);
    return compact ? min(ahead + n, max_rows) - min(ahead, max_rows) : n;
  };
  auto tiles_for = [=](int rows) { return (rows + BM - 1) / BM * tiles_n; };
  const int per = (groups + NT - 1) / NT, run_first = min(tid * per, groups), run_end = min(run_first + per, groups);
  int run_rows = 0, run_tiles = 0;
  for (int g = run_first; g < run_end; ++g) run_rows += rows_of(g);
  const int inc_rows = wave_inclusive_scan(run_rows);
  if (lane == 63) red_rows[wave] = inc_rows;
  lds_barrier();
  int run_ahead = inc_rows - run_rows;
#pragma unroll
  for (int w = 0; w < NW; ++w) run_ahead += w < wave ? red_rows[w] : 0;
  for (int g = run_first, ahead = run_ahead; g < run_end; ahead += rows_of(g), ++g) run_tiles += tiles_for(kept_of(g, ahead));
  const int inc = wave_inclusive_scan(run_tiles);
  if (lane == 63) red[wave] = inc;
  lds_barrier();
  int run_begin = inc - run_tiles, total = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    run_begin += w < wave ? red[w] : 0;
    total += red[w];
  }
  GroupTile at;
  at.total = __builtin_amdgcn_readfirstlane(total);
  if (tile >= at.total) return at;
  // (an XCD works on a run of consecutive tiles)
  const int logical = xcd_contiguous(tile, at.total);
  if (run_begin <= logical && logical < run_begin + run_tiles) {
    int g = run_first, first = run_begin, ahead = run_ahead;
    for (;; ++g) {
      const int n = tiles_for(kept_of(g, ahead));
      if (logical < first + n) break;
      first += n;
      ahead += rows_of(g);
    }
    const int kept = kept_of(g, ahead), n = (kept + BM - 1) / BM, height = ((kept + n - 1) / n + 31) / 32 * 32;
    const int tn = (logical - first) / n, t0 = (logical - first - tn * n) * height;
    home[0] = g;
    home[1] = tn;
    home[2] = (compact ? min(ahead, max_rows) : 0) + t0;
    home[3] = min(height, kept - t0);
  }
  lds_barrier();
  at.group = __builtin_amdgcn_readfirstlane(home[0]);
  at.tn = __builtin_amdgcn_readfirstlane(home[1]);
  at.row_at = (compact ? 0 : (size_t)at.group * max_rows) + __builtin_amdgcn_readfirstlane(home[2]);
  at.rows = __builtin_amdgcn_readfirstlane(home[3]);
  return at;
}

// ---------------------------------------------------------------- products of few tiles
//
// The experts' product of few rows per expert, on tiles of 32 x 32 or 32 x 64, where they leave a unit with one or two workgroups (and some with long
// walks of K, grouped_ring): nothing then hides the way of a step's rows from memory but the steps that are already under way. Four waves fetch the
// rows of a tile of 32 TM x 32 TN straight into a ring of DEPTH steps in LDS (64 to 72 KB of them) and multiply a quarter of the tile each. One barrier per step:
// behind it step s + 1 is there for everybody, and everybody holds the fragments of step s, so that its place is free for
// step s + DEPTH, and the fragments of step s + 1 are read beside the MFMAs of step s (without that, and with all of a tile's
// 32 columns on one wave, 1 row in 1024 x 7168 took 27.6 us instead of 17.1).
// LDS rows, fragments and the order of K are those of phased_gemm_kernel.
// What bounds it: with few tiles the chain of a step (barrier, fragments, two MFMAs: 0.14 us), with more HBM (5 to 6 TB/s
// from 400 tiles on). us, expert_gemm_kernel / here: 7 of 48
// groups with a row, 832 x 3840 21.7 / 11.3; 2 of 8, 2048 x 4096 23.0 / 11.8; 4 groups of 1 row, 2048 x 7168 38.1 / 22.5; 19 of 2, 6272 x
// 3360 157.0 / 120.6. (Larger tiles are sliced_gemm_kernel's. On these it is up to 7 % behind: 101 products of 32 x 64 1.02 of the time here.)

constexpr size_t ring_lds_bytes(int TM, int TN, int DEPTH) { return (size_t)DEPTH * (TM + TN) * 32 * 128; }

template <int DT, int TM, int TN, int DEPTH, bool STREAMED>
__global__ __launch_bounds__(256, 1) void ring_gemm_kernel(
    const b128* __restrict__ A, const b128* __restrict__ B, const int* __restrict__ rows_of_group,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ C, int N, int K, int tiles_n, int groups, int max_rows, int compact) {
  constexpr int BM = 32 * TM, BN = 32 * TN, LA = TM, LB = TN;  // direct loads (8 rows each) of a wave per step
  constexpr int STEP_BYTES = (BM + BN) * 128, B_AT = BM * 128, RING_BYTES = DEPTH * STEP_BYTES;
  constexpr int YOUNGER = (LA + LB) * (DEPTH - 2);  // a wave's loads that may be under way when step s + 1 has to be there
  static_assert(DEPTH >= 3 && YOUNGER + LA + LB < 64, "loads that the wait can count");
  extern __shared__ b128 tile_lds[];  // [DEPTH][(BM + BN) * 8]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int row_vecs = K / 8, row_bytes = K * 2, steps = (K + GEMM_KSTEP - 1) / GEMM_KSTEP;
  const int tail_vecs = row_vecs - (steps - 1) * 8;
  // load i of a wave takes rows i * 32 + wave * 8 .. + 7 of an operand, a lane the vector that belongs at its place
  const int vec = (lane & 7) ^ ((wave * 4 + (lane >> 4)) & 7);
  const int off = (wave * 8 + (lane >> 3)) * row_bytes + vec * 16;
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) b128*)tile_lds + wave * 1024;
  // fragment of a slice of 32 inputs: row r of a band of 16, vector 4 * slice + q of the step
  const int r = lane & 15, q = lane >> 4, swz = (r >> 1) & 7;

  for (int tile = blockIdx.x;; tile += gridDim.x) {
    const GroupTile at = find_group_tile<256, BM>(tile, rows_of_group, groups, max_rows, tiles_n, compact, (int*)tile_lds);
    if (tile >= at.total) return;
    lds_barrier();
    const int n0 = at.tn * BN;
    const int k_first = first_kstep(at.group, groups, K) * (GEMM_KSTEP * 2);
    const b128 abuf = buffer_words(A + at.row_at * row_vecs, min(BM, at.rows) * row_bytes);
    const b128 bbuf = buffer_words(B + ((size_t)at.group * N + n0) * row_vecs, min(BN, N - n0) * row_bytes);
    int past = 0, soff = k_first;  // past the end of the rows in their last step, and everywhere behind it: out of range
    unsigned fill = 0, use = 0;
    auto range = [&](int step) __attribute__((always_inline)) {  // before a step near the end is asked for
      if (step == steps - 1) past = vec >= tail_vecs ? OUT_OF_RANGE : 0;
      else if (step >= steps) past = OUT_OF_RANGE;
    };
    auto load = [&]() __attribute__((always_inline)) {
      unrolled<0, LA>([&](auto c) __attribute__((always_inline)) {
        constexpr int i = decltype(c)::value;
        load_to_lds<i * 4096>(base + fill, off + i * 32 * row_bytes + past, abuf, soff);
      });
      unrolled<0, LB>([&](auto c) __attribute__((always_inline)) {
        constexpr int i = decltype(c)::value;
        load_to_lds<B_AT + i * 4096, STREAMED>(base + fill, off + i * 32 * row_bytes + past, bbuf, soff);
      });
      fill = fill == RING_BYTES - STEP_BYTES ? 0u : fill + STEP_BYTES;
      soff += GEMM_KSTEP * 2;
      if (k_first && soff == row_bytes) soff = 0;
    };
#pragma unroll 1
    for (int step = 0; step < DEPTH; ++step) {
      range(step);
      load();
    }
    f32x4 acc[TM][TN] = {};
    b128 af[2][2][TM], bf[2][2][TN];  // [set][slice]
    const bool multiplies = wm * (BM / 2) < at.rows && n0 + wn * (BN / 2) < N;  // (the same for the whole wave)
    auto read_frags = [&](auto set) __attribute__((always_inline)) {  // of the step in `use`
      constexpr int f = decltype(set)::value;
      const char* as = (const char*)tile_lds + use + (wm * (BM / 2) + r) * 128;
      const char* bs = (const char*)tile_lds + use + B_AT + (wn * (BN / 2) + r) * 128;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int v = ((s * 4 + q) ^ swz) * 16;
#pragma unroll
        for (int j = 0; j < TN; ++j) bf[f][s][j] = *(const b128*)(bs + j * (16 * 128) + v);
#pragma unroll
        for (int i = 0; i < TM; ++i) af[f][s][i] = *(const b128*)(as + i * (16 * 128) + v);
      }
      use = use == RING_BYTES - STEP_BYTES ? 0u : use + STEP_BYTES;
      __builtin_amdgcn_sched_barrier(0);
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    auto one_step = [&](auto set, auto other) __attribute__((always_inline)) {
      constexpr int f = decltype(set)::value;
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
      load();
      if (multiplies) {
        read_frags(other);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = Mfma16x16x32<DT>::mma(bf[f][s][j], af[f][s][i], acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER + LA + LB) : "memory");
    lds_barrier();
    if (multiplies) read_frags(even);
    int step = 0;
    for (; step + DEPTH + 2 < steps; step += 2) {  // (what these ask for lies before the last step)
      one_step(even, odd);
      one_step(odd, even);
    }
    for (; step < steps; step += 2) {
      range(step + DEPTH);
      one_step(even, odd);
      if (step + 1 == steps) break;
      range(step + 1 + DEPTH);
      one_step(odd, even);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the loads past the last step write zeros)
    __syncthreads();

    // this lane: row r of a band, columns q * 4 + 0..3 of 16
    if (multiplies) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn * (BN / 2) + j * 16 + q * 4;
        if (n >= N) continue;
        uint32_t bias2[2] = {};
        if (bias) __builtin_memcpy(bias2, bias + (size_t)at.group * N + n, 8);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int m = wm * (BM / 2) + i * 16 + r;
          const f32x4& c = acc[i][j];
          uint32_t two[2] = {Pair16<DT>::canonical(Pair16<DT>::round(c[0], c[1])),
                             Pair16<DT>::canonical(Pair16<DT>::round(c[2], c[3]))};
          if (bias) {
#pragma unroll
            for (int e = 0; e < 2; ++e)
              two[e] = Pair16<DT>::canonical(Pair16<DT>::round(
                  __fadd_rn(Pair16<DT>::lo(two[e]), Pair16<DT>::lo(bias2[e])),
                  __fadd_rn(Pair16<DT>::hi(two[e]), Pair16<DT>::hi(bias2[e]))));
          }
          if (m < at.rows) __builtin_memcpy(C + (at.row_at + m) * N + n, two, 8);
        }
      }
    }
  }
}

// ---------------------------------------------------------------- products of a few hundred tiles
//
// The experts' product or a plain one where its tiles make for about one workgroup per unit, or two. WM x WN waves, two or four of them on a SIMD,
// fetch the rows of a tile straight into a ring of DEPTH steps in LDS. A wave holds the fragments of one slice of 32 inputs while those of the
// next are on their way, so that its reads are behind MFMAs and the waves of a SIMD fill each other's gaps; one barrier per step, in its
// middle. LDS rows, fragments, results and the order of K are those of phased_gemm_kernel, so among kernels that walk K whole the choice changes no
// bit (products that were split over K before round their sums elsewhere: a single one instead of one per wave).
// What bounds it: rows out of L2, some 17 TB/s over the chip on any tile (32 x 64 to 192 x 128: 0.2 to 0.67 us a step), and 3.5 to 5 us around
// the walk (launch, first rows, results). us, the kernel that had the product / here:
//   plain, on one group of ring_gemm_kernel, whose workgroups search the groups for their tile: 77 x 7360 x 768 7.84 / 5.74, 351 x 1728 x 832
//     8.19 / 6.04, 202 x 2432 x 6272 26.7 / 21.7, 24 x 2176 x 384 5.31 / 4.38; on 64 x 128 of dense_gemm_kernel, whose rows go through registers
//     into two buffers: 786 x 1984 x 4608 28.4 / 25.5, 297 x 1152 x 408 5.79 / 4.77, 37 x 7808 x 8 4.33 / 3.75; split over K, in calls: 64 x 7168 x 2304
//     9.1 / 8.7 (on 64 x 32), 88 x 5056 x 2432 10.4 / 8.7
//   experts': 15 of 400 rows, 576 x 640 (dense_gemm_kernel, 64 x 128) 23.9 / 16.8; 5 of 253, 896 x 1856 (a ring of 64 x 128) 17.3 / 14.0; 11 of 50,
//     1248 x 6240 69.4 / 45.0; 22 of 239, 640 x 1280 (dense_gemm_kernel, 128 x 128) 25.0 / 17.2; 13 of 377, 1024 x 4032
//     (phased_gemm_kernel, 192 x 256) 72.0 / 52.6; 18 of 39, 960 x 1408 (expert_gemm_kernel) 22.2 / 13.0
template <int WM_, int WN_, int TM_, int TN_, int DEPTH_, int ON_UNIT_>
struct Slices {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, DEPTH = DEPTH_, ON_UNIT = ON_UNIT_;  // (workgroups on a unit)
  static constexpr int ROWS = WM * TM * 16, COLS = WN * TN * 16, LANES = 64 * WM * WN;
  static constexpr size_t LDS_BYTES = (size_t)DEPTH * (ROWS + COLS) * 128;
};
using Slices32x64 = Slices<2, 2, 1, 2, 6, 2>;
using Slices64x32 = Slices<4, 1, 1, 2, 6, 2>;
using Slices64x64 = Slices<4, 2, 1, 2, 4, 2>;
using Slices64x128 = Slices<2, 4, 2, 2, 3, 2>;
using Slices128x128 = Slices<4, 2, 2, 4, 4, 1>;
using Slices192x128 = Slices<4, 2, 3, 4, 3, 1>;

// (Rings of twice the depth where every unit has a tile at most, of 144 KB of LDS: 0.4 to 1.2 us longer, as two launches in a row do not overlap then; with
// weights that HBM has to deliver as well, 64 x 7168 x 2304 12.0 / 13.0, 85 x 5376 x 1856 9.6 / 10.6, 200 x 4096 x 4096 18.8 / 17.7.)
template <int DT, typename TILE, bool GROUPED, bool STREAMED>
__global__ __launch_bounds__(64 * TILE::WM * TILE::WN, TILE::ON_UNIT * TILE::WM * TILE::WN / 4) void sliced_gemm_kernel(
    const b128* __restrict__ A, const b128* __restrict__ B, const uint16_t* __restrict__ bias, uint16_t* __restrict__ C, int M, int N, int K,
    int tiles_m, int tiles_n, const int* __restrict__ rows_of_group, int groups, int max_rows, int compact) {
  constexpr int WM = TILE::WM, WN = TILE::WN, TM = TILE::TM, TN = TILE::TN, DEPTH = TILE::DEPTH;
  constexpr int NW = WM * WN, NT = 64 * NW, BM = TILE::ROWS, BN = TILE::COLS, GROUP_M = 4;
  constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW;  // direct loads (8 rows each) of a wave per step
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "whole loads");
  constexpr int STEP_BYTES = (BM + BN) * 128, B_AT = BM * 128, RING_BYTES = DEPTH * STEP_BYTES;
  constexpr int YOUNGER = (LA + LB) * (DEPTH - 2);  // a wave's loads that may be under way when step s + 1 has to be there
  static_assert(DEPTH >= 2 && YOUNGER + LA + LB < 64, "loads that the wait can count");
  extern __shared__ b128 tile_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int row_vecs = K / 8, row_bytes = K * 2, steps = (K + GEMM_KSTEP - 1) / GEMM_KSTEP;
  const int tail_vecs = row_vecs - (steps - 1) * 8;
  // load i of a wave takes rows (i * NW + wave) * 8 .. + 7 of an operand, a lane the vector that belongs at its place
  const int lrow = wave * 8 + (lane >> 3);
  const int vec = (lane & 7) ^ ((lrow >> 1) & 7);
  const int off = lrow * row_bytes + vec * 16;
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) b128*)tile_lds + wave * 1024;
  // fragment of a slice of 32 inputs: row r of a band of 16, vector 4 * slice + q of the step
  const int r = lane & 15, q = lane >> 4, swz = (r >> 1) & 7;
  [[maybe_unused]] const int total_tiles = tiles_m * tiles_n;  // (GROUPED: counted by find_group_tile)

  for (int tile = blockIdx.x;; tile += gridDim.x) {
    int n0, rows_left;         // first column of the tile; rows of the matrix from the tile's first one on
    size_t row_at, b_at;       // the tile's first rows of A and C, and of B
    const uint16_t* bias_row;  // the bias of the tile's group, or null
    [[maybe_unused]] int k_first = 0;
    if constexpr (GROUPED) {
      const GroupTile at = find_group_tile<NT, BM>(tile, rows_of_group, groups, max_rows, tiles_n, compact, (int*)tile_lds);
      if (tile >= at.total) return;
      lds_barrier();
      n0 = at.tn * BN;
      rows_left = at.rows;
      row_at = at.row_at;
      b_at = (size_t)at.group * N + n0;
      k_first = first_kstep(at.group, groups, K) * (GEMM_KSTEP * 2);
      bias_row = bias ? bias + (size_t)at.group * N : nullptr;
    } else {
      if (tile >= total_tiles) return;
      const int logical = xcd_contiguous(tile, total_tiles);
      const int per_group = GROUP_M * tiles_n, group = logical / per_group, in = logical - group * per_group;
      const int group_rows = min(GROUP_M, tiles_m - group * GROUP_M);
      const int tn = in / group_rows, tm = group * GROUP_M + in - tn * group_rows;
      n0 = tn * BN;
      rows_left = M - tm * BM;
      row_at = (size_t)tm * BM;
      b_at = n0;
      bias_row = bias;
    }
    const b128 abuf = buffer_words(A + row_at * row_vecs, min(BM, rows_left) * row_bytes);
    const b128 bbuf = buffer_words(B + b_at * row_vecs, min(BN, N - n0) * row_bytes);
    int past = 0, soff = k_first;  // past the end of the rows in their last step, and everywhere behind it: out of range
    unsigned fill = 0, use = 0;
    auto range = [&](int step) __attribute__((always_inline)) {  // before a step near the end is asked for
      if (step == steps - 1) past = vec >= tail_vecs ? OUT_OF_RANGE : 0;
      else if (step >= steps) past = OUT_OF_RANGE;
    };
    auto load = [&]() __attribute__((always_inline)) {
      unrolled<0, LA>([&](auto c) __attribute__((always_inline)) {
        constexpr int i = decltype(c)::value;
        load_to_lds<i * NW * 1024>(base + fill, off + i * 8 * NW * row_bytes + past, abuf, soff);
      });
      unrolled<0, LB>([&](auto c) __attribute__((always_inline)) {
        constexpr int i = decltype(c)::value;
        load_to_lds<B_AT + i * NW * 1024, STREAMED>(base + fill, off + i * 8 * NW * row_bytes + past, bbuf, soff);
      });
      fill = fill == RING_BYTES - STEP_BYTES ? 0u : fill + STEP_BYTES;
      soff += GEMM_KSTEP * 2;
      if (GROUPED && k_first && soff == row_bytes) soff = 0;
    };
#pragma unroll 1
    for (int step = 0; step < DEPTH; ++step) {
      range(step);
      load();
    }
    f32x4 acc[TM][TN] = {};
    b128 af[2][TM], bf[2][TN];  // [slice]
    auto read_frags = [&](auto slice) __attribute__((always_inline)) {  // of the step in `use`
      constexpr int s = decltype(slice)::value;
      const int v = ((s * 4 + q) ^ swz) * 16;
      const char* as = (const char*)tile_lds + use + (wm * TM * 16 + r) * 128 + v;
      const char* bs = (const char*)tile_lds + use + B_AT + (wn * TN * 16 + r) * 128 + v;
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[s][j] = *(const b128*)(bs + j * (16 * 128));
#pragma unroll
      for (int i = 0; i < TM; ++i) af[s][i] = *(const b128*)(as + i * (16 * 128));
    };
    auto mfmas = [&](auto slice) __attribute__((always_inline)) {
      constexpr int s = decltype(slice)::value;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = Mfma16x16x32<DT>::mma(bf[s][j], af[s][i], acc[i][j]);
    };
    constexpr std::integral_constant<int, 0> first{};
    constexpr std::integral_constant<int, 1> second{};
    auto one_step = [&]() __attribute__((always_inline)) {
      read_frags(second);  // (the first slice is in registers)
      __builtin_amdgcn_sched_barrier(0);
      mfmas(first);
      __builtin_amdgcn_sched_barrier(0);
      // everybody has read this step's rows, whose place the step DEPTH on takes, and the next one's are there for everybody
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
      __builtin_amdgcn_sched_barrier(0);
      load();
      use = use == RING_BYTES - STEP_BYTES ? 0u : use + STEP_BYTES;
      read_frags(first);
      __builtin_amdgcn_sched_barrier(0);
      mfmas(second);
      __builtin_amdgcn_sched_barrier(0);
    };
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER + LA + LB) : "memory");
    lds_barrier();
    read_frags(first);
    int step = 0;
    for (; step + DEPTH + 1 < steps; ++step) one_step();  // (what these ask for lies before the last step)
    for (; step < steps; ++step) {
      range(step + DEPTH);
      one_step();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the loads past the last step write zeros)
    __syncthreads();

    // Out through LDS as in phased_gemm_kernel, a band of 16 rows at a time.
    constexpr int VR = TN * 2, PITCH = TN * 32 + 16, ROWS_PER_READ = 64 / VR;
    static_assert(ROWS_PER_READ <= 16 && NW * 16 * PITCH <= RING_BYTES, "bands that a wave reads in whole turns");
    char* park = (char*)tile_lds + wave * (16 * PITCH);
    uint16_t* const c_tile = C + row_at * N;
    const int ncol = n0 + wn * TN * 16;
    uint32_t bias2[TN][2] = {};
    if (bias_row) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
        if (ncol + j * 16 < N) __builtin_memcpy(bias2[j], bias_row + ncol + j * 16 + q * 4, 8);
    }
    const int rrow = lane / VR, rvec = lane % VR;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const f32x4& c = acc[i][j];
        uint32_t two[2] = {Pair16<DT>::canonical(Pair16<DT>::round(c[0], c[1])), Pair16<DT>::canonical(Pair16<DT>::round(c[2], c[3]))};
        if (bias_row) {
#pragma unroll
          for (int e = 0; e < 2; ++e)
            two[e] = Pair16<DT>::canonical(Pair16<DT>::round(__fadd_rn(Pair16<DT>::lo(two[e]), Pair16<DT>::lo(bias2[j][e])),
                                                             __fadd_rn(Pair16<DT>::hi(two[e]), Pair16<DT>::hi(bias2[j][e]))));
        }
        __builtin_memcpy(park + r * PITCH + (j * 16 + q * 4) * 2, two, 8);
      }
#pragma unroll
      for (int p = 0; p < 16 / ROWS_PER_READ; ++p) {
        const int row = p * ROWS_PER_READ + rrow;
        const b128 v = *(const b128*)(park + row * PITCH + rvec * 16);
        const int m = (wm * TM + i) * 16 + row, n = ncol + rvec * 8;
        if (m < rows_left && n < N) row_store<THROUGH>((b128*)(c_tile + (size_t)m * N + n), v);
      }
    }
    lds_barrier();  // the results are out of LDS
  }
}

template <int DT, int TM, int TN, int NA, int HB, bool AHEAD, bool GROUPED, bool STREAMED = false>
__global__ __launch_bounds__(512, 1) void phased_gemm_kernel(
    const b128* __restrict__ A, const b128* __restrict__ B, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n,
    const int* __restrict__ rows_of_group, int groups, int max_rows, int compact) {
  constexpr int BM = phased_rows(TM), BN = phased_cols(TN), GROUP_M = 4;
  constexpr int LA = BM / 64, LB = BN / 64;  // direct loads (8 rows each) of a wave per step
  constexpr bool HALVES = HB % 2 != 0;  // B goes to a ring of HB halves (BN / 2 columns each) instead of NB whole buffers
  constexpr int NB = HB / 2;
  static_assert(BM % 64 == 0 && (HALVES ? NA == 2 && HB == 5 && !AHEAD : NA >= 2 && NB >= 2 && NA + NB == 5),
                "whole loads, and a schedule for the buffers");
  static_assert(!(AHEAD && GROUPED), "tiles that share rows across an XCD");
  constexpr bool EARLY = !GROUPED && TM == 8;   // a workgroup has several tiles of 256 x 256,
  constexpr bool ONE_TILE = !GROUPED && !EARLY;  // and one of the lower ones, of which there are fewer (linear_way)
  constexpr bool B_FIRST = NB <= NA;  // the operand with fewer buffers is asked for in the first slice of a step
  constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128, HALF_BYTES = B_BYTES / 2, B_AT = NA * A_BYTES;
  extern __shared__ b128 tile_lds[];  // [NA][BM * 8], [HB][BN * 4]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int row_vecs = K / 8, row_bytes = K * 2, steps = (K + GEMM_KSTEP - 1) / GEMM_KSTEP;
  const int tail_vecs = row_vecs - (steps - 1) * 8;
  const bool first_group = wave < 4;

  // A workgroup strides over the tiles (the size of the launch is a matter of speed only). EARLY: the first loads of
  // its next tile go out before the results of the last one do, so that they arrive while those are written, and the
  // accumulators are cleared meanwhile. A workgroup per tile / this: 8192 x 8192 x 512 84.5 / 79.0 us, x 3696 370.6 /
  // 368.3, 4096 x 4096 x 4096 93.5 / 92.4. Experts' products have
  // a workgroup per tile in general, and the registers for it would be spilled at 320 rows: 140 -> 146 us.
  int tile = blockIdx.x, total_tiles = tiles_m * tiles_n;  // (GROUPED: counted by find_tile)
  int n0, rows_left;         // first column of the tile; rows of the matrix from the tile's first one on
  size_t row_at, b_at;       // the tile's first rows of A and C, and of B
  const uint16_t* bias_row;  // the bias of the tile's group, or null
  [[maybe_unused]] int tn, tm, k_first = 0;
  auto find_tile = [&]() __attribute__((always_inline)) {  // (GROUPED: nobody uses LDS, and there is a tile if tile < total_tiles)
    if constexpr (GROUPED) {
      const GroupTile at = find_group_tile<512, BM>(tile, rows_of_group, groups, max_rows, tiles_n, compact, (int*)tile_lds);
      total_tiles = at.total;
      if (tile >= at.total) return;
      lds_barrier();
      n0 = at.tn * BN;
      rows_left = at.rows;
      row_at = at.row_at;
      b_at = (size_t)at.group * N + n0;
      k_first = first_kstep(at.group, groups, K) * (GEMM_KSTEP * 2);
      bias_row = bias ? bias + (size_t)at.group * N : nullptr;
    } else {
      const int logical = xcd_contiguous(tile, total_tiles);
      const int per_group = GROUP_M * tiles_n, group = logical / per_group, in = logical - group * per_group;
      const int group_rows = min(GROUP_M, tiles_m - group * GROUP_M);
      tn = in / group_rows, tm = group * GROUP_M + in - tn * group_rows;
      n0 = tn * BN;
      rows_left = M - tm * BM;
      row_at = (size_t)tm * BM;
      b_at = n0;
      bias_row = bias;
    }
  };

  // As in dense_gemm_kernel: rows past the end of a matrix read as zeros (they lie past the extent), and
  // so do the vectors past the end of a row in the last step and everything past the last step.
  b128 abuf, bbuf;
  // Load i of a wave takes rows i * 64 + wave * 8 .. + 7, and a lane the vector that belongs at its place: the same for all i.
  auto vec_of = [=](int l) { return (l & 7) ^ (((wave * 8 + (l >> 3)) >> 1) & 7); };
  int aoff[LA], boff[LB];
  auto a_range = [&](int step) __attribute__((always_inline)) {  // before the rows of a step near the end are asked for
    if (step == steps - 1) {
#pragma unroll
      for (int i = 0; i < LA; ++i) aoff[i] += vec_of(lane) >= tail_vecs ? OUT_OF_RANGE : 0;
    } else if (step >= steps) {
#pragma unroll
      for (int i = 0; i < LA; ++i) aoff[i] = OUT_OF_RANGE;
    }
  };
  auto b_range = [&](int step, int from, int to) __attribute__((always_inline)) {
    if (step == steps - 1) {
#pragma unroll
      for (int i = from; i < to; ++i) boff[i] += vec_of(lane) >= tail_vecs ? OUT_OF_RANGE : 0;
    } else if (step >= steps) {
#pragma unroll
      for (int i = from; i < to; ++i) boff[i] = OUT_OF_RANGE;
    }
  };

  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) b128*)tile_lds;
  const unsigned a_base = lds0 + wave * 1024, b_base = lds0 + B_AT + wave * 1024;
  // byte of a row at which the next requested step begins
  int a_soff, b_soff;
  [[maybe_unused]] int half_soff[2];
  unsigned a_fill, b_fill;  // buffer (as a byte offset) that the next requested step goes to
  unsigned a_use, b_use;    // buffer of the step being multiplied (HALVES: the place of the half that holds this wave's columns)
  auto next_a = [](unsigned at) { return at == (NA - 1) * A_BYTES ? 0u : at + A_BYTES; };
  auto next_b = [](unsigned at) {
    return at + B_BYTES < HB * HALF_BYTES ? at + B_BYTES : at + B_BYTES - HB * HALF_BYTES;
  };
  auto load_a = [&]() __attribute__((always_inline)) {
    unrolled<0, LA>([&](auto c) __attribute__((always_inline)) {
      constexpr int i = decltype(c)::value;
      load_to_lds<i * 8192>(a_base + a_fill, aoff[i], abuf, a_soff);
    });
    a_fill = next_a(a_fill);
    a_soff += GEMM_KSTEP * 2;
    if (GROUPED && k_first && a_soff == row_bytes) a_soff = 0;
  };
  auto load_b = [&]() __attribute__((always_inline)) {
    unrolled<0, LB>([&](auto c) __attribute__((always_inline)) {
      constexpr int i = decltype(c)::value;
      load_to_lds<i * 8192, STREAMED>(b_base + b_fill, boff[i], bbuf, b_soff);
    });
    b_fill = next_b(b_fill);
    b_soff += GEMM_KSTEP * 2;
    if (GROUPED && k_first && b_soff == row_bytes) b_soff = 0;
  };

  auto load_half = [&](auto half) __attribute__((always_inline)) {  // the next step's columns of a half
    constexpr int h = decltype(half)::value;
    unrolled<0, LB / 2>([&](auto c) __attribute__((always_inline)) {
      constexpr int i = decltype(c)::value;
      load_to_lds<i * 8192, STREAMED>(b_base + b_fill, boff[h * (LB / 2) + i], bbuf, half_soff[h]);
    });
    b_fill = b_fill == (HB - 1) * HALF_BYTES ? 0u : b_fill + HALF_BYTES;
    half_soff[h] += GEMM_KSTEP * 2;
    if (GROUPED && k_first && half_soff[h] == row_bytes) half_soff[h] = 0;
  };
  constexpr std::integral_constant<int, 0> lower{};
  constexpr std::integral_constant<int, 1> upper{};

  // AHEAD: a wave touches, four steps ahead, one line each of the rows this workgroup fetches into L2 for its
  // neighbours as well: of the GROUP_M x 8 tiles that an XCD works on at a time, the 8 with the same rows of
  // A share those out, and the GROUP_M with the same rows of B. What comes back is not used. The load is one that
  // the compiler knows, which keeps anything else out of its register until it has returned, and a volatile one, so
  // that it stays between the two waits that count it. (Only lanes with a row of their own ask: with the others
  // repeating a row, 8192 x 8192 x 3696 took 2 % longer.)
  constexpr int AHEAD_STEPS = 4;
  typedef const __attribute__((address_space(1))) char* global_bytes;
  [[maybe_unused]] global_bytes touch_base = nullptr;
  [[maybe_unused]] unsigned touch_off = 0;
  [[maybe_unused]] uint32_t touched = 0;
  [[maybe_unused]] bool touches = false;
  auto aim_touches = [&]() __attribute__((always_inline)) {
    constexpr int A_EACH = BM / 8 / 4, B_EACH = BN / GROUP_M / 4;  // rows of a wave of either group
    touch_base = (global_bytes)(first_group ? A + row_at * row_vecs : B + b_at * row_vecs);
    const int a_row = min((tn & 7) * (BM / 8) + wave * A_EACH + lane, rows_left - 1);
    const int b_row = min((tm & (GROUP_M - 1)) * (BN / GROUP_M) + (wave - 4) * B_EACH + lane, N - n0 - 1);
    touches = lane < (first_group ? A_EACH : B_EACH);  // (lanes of every wave: its waits count the load)
    touch_off = (unsigned)(first_group ? a_row : b_row) * row_bytes;
  };
  auto touch = [&](int step) __attribute__((always_inline)) {
    if constexpr (AHEAD) {
      global_bytes at = touch_base + min(step, steps - 1) * (GEMM_KSTEP * 2);
      asm("" : "+s"(at));  // (a scalar base and the lane's offset: no vector register to write anew)
      if (touches) {
        asm("" : "+v"(touch_off));
        touched = __scoped_atomic_load_n((const volatile __attribute__((address_space(1))) uint32_t*)(at + touch_off),
                                         __ATOMIC_RELAXED, __MEMORY_SCOPE_WVFRNT);
      }
    }
  };

  // fragment of a slice: row r of the band, vector 4 * slice + q of the step
  const int r = lane & 15, q = lane >> 4, swz = (r >> 1) & 7;
  const char* const lds = (const char*)tile_lds;
  const char* a_frag[2];
  const char* b_frag[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    a_frag[s] = lds + (wm * 16 + r) * 128 + ((s * 4 + q) ^ swz) * 16;
    b_frag[s] = lds + B_AT + ((HALVES ? wn & 1 : wn) * TN * 16 + r) * 128 + ((s * 4 + q) ^ swz) * 16;
  }
  b128 af[TM], bf[TN];
  f32x4 acc[TM][TN];
  auto read_frags = [&](auto bands, int slice) __attribute__((always_inline)) {
    const char* ap = a_frag[slice] + a_use;
    const char* bp = b_frag[slice] + b_use;
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[j] = *(const b128*)(bp + j * (16 * 128));
#pragma unroll
    for (int i = 0; i < decltype(bands)::value; ++i) af[i] = *(const b128*)(ap + i * (32 * 128));
    __builtin_amdgcn_sched_barrier(0);
  };
  // this wave's turn at the matrix cores; `begin` and `end` are what it does first and last in it
  auto multiply = [&](auto bands, auto begin, auto end) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(WAIT_LDS_ONLY);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    begin();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < decltype(bands)::value; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = Mfma16x16x32<DT>::mma(bf[j], af[i], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
    end();
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // Step s reads its buffers in both of its slices. In the first it asks for the operand with fewer buffers, n
  // of them: step s + n - 1, into the buffer of step s - 1 (the other group has read its last slice in the phase
  // before); in the second likewise for the other operand. Before the barrier that ends the second reading phase
  // the wave waits for everything that step s + 1 needs, which is all but the youngest loads: step s + 1 is then
  // in LDS for everybody one barrier later, when the first group gets there.
  auto nothing = []() __attribute__((always_inline)) {};
  auto one_slice_pair = [&](auto bands, int step) __attribute__((always_inline)) {
    read_frags(bands, 0);
    if constexpr (B_FIRST) load_b(); else load_a();
    multiply(bands, nothing, nothing);
    read_frags(bands, 1);
    if constexpr (B_FIRST) load_a(); else load_b();
    touch(step + AHEAD_STEPS);
    a_use = next_a(a_use);
    b_use = next_b(b_use);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((B_FIRST ? LA : LB) + (AHEAD ? 1 : 0)) : "memory");
    multiply(bands, nothing, nothing);
  };
  // With five halves of B, step s + 1's upper half and step s + 2's lower one go to the places of step s - 1's halves,
  // and step s + 1's rows of A to the buffer of step s - 1. Step s + 1 has to be there when the first group has
  // multiplied step s: both groups wait in the phase before that, the first behind its MFMAs, the second behind its
  // last reads, for all but the lower half of step s + 2, the youngest loads.
  auto one_step_of_halves = [&](auto bands) __attribute__((always_inline)) {
    constexpr int YOUNGER = LB / 2;  // loads of a wave that may be under way when a step ends
    read_frags(bands, 0);
    load_half(upper);
    load_a();
    multiply(bands, nothing, nothing);
    read_frags(bands, 1);
    load_half(lower);
    a_use = next_a(a_use);
    b_use = next_b(b_use);
    if (!first_group) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
    multiply(bands, nothing, [&]() __attribute__((always_inline)) {
      if (first_group) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
    });
  };
  constexpr int FIRST_YOUNGER = HALVES ? LB / 2 : (NA - 2) * LA + (NB - 2) * LB;  // of a tile's first loads, what its first step does without
  auto begin_tile = [&]() __attribute__((always_inline)) {
    abuf = buffer_words(A + row_at * row_vecs, min(BM, rows_left) * row_bytes);
    bbuf = buffer_words(B + b_at * row_vecs, min(BN, N - n0) * row_bytes);
    int at = lane;  // (worked out anew for each tile: kept over the loop the offsets would take registers that it needs)
    asm volatile("" : "+v"(at));
    const int off = (wave * 8 + (at >> 3)) * row_bytes + vec_of(at) * 16;
#pragma unroll
    for (int i = 0; i < LA; ++i) aoff[i] = off + i * 64 * row_bytes;
#pragma unroll
    for (int i = 0; i < LB; ++i) boff[i] = off + i * 64 * row_bytes;
    a_soff = b_soff = half_soff[0] = half_soff[1] = GROUPED ? k_first : 0;
    a_fill = b_fill = a_use = 0;
    b_use = HALVES ? (wn >> 1) * HALF_BYTES : 0;
    if constexpr (AHEAD) aim_touches();
    if constexpr (HALVES) {
      b_range(0, 0, LB);
      load_half(lower);
      load_half(upper);
      a_range(0);
      load_a();
      b_range(1, 0, LB / 2);
      load_half(lower);
    } else {
      unrolled<0, 2>([&](auto c) __attribute__((always_inline)) {
        constexpr int at = decltype(c)::value;
        if constexpr (at < NA - 1) { a_range(at); load_a(); }
        if constexpr (at < NB - 1) { b_range(at, 0, LB); load_b(); }
      });
    }
  };
  auto walk_k = [&](auto bands) __attribute__((always_inline)) {
    int step = 0;
    if constexpr (HALVES) {
      for (; step + 3 < steps; ++step) one_step_of_halves(bands);
      for (; step < steps; ++step) {
        a_range(step + 1);
        b_range(step + 1, LB / 2, LB);
        b_range(step + 2, 0, LB / 2);
        one_step_of_halves(bands);
      }
    } else {
      for (; step + 3 < steps; ++step) one_slice_pair(bands, step);  // (what it asks for lies before the last step)
      for (; step < steps; ++step) {
        a_range(step + NA - 1);
        b_range(step + NB - 1, 0, LB);
        one_slice_pair(bands, step);
      }
    }
  };
  find_tile();
  if (tile >= total_tiles) return;
  begin_tile();
  auto clear = [&]() __attribute__((always_inline)) {  // (while the first loads are under way)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        acc[i][j] = f32x4{};
        asm volatile("" : "+v"(acc[i][j]));
      }
  };
  clear();
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FIRST_YOUNGER) : "memory");
  for (;;) {
  asm volatile("s_barrier" ::: "memory");
  if (!first_group) asm volatile("s_barrier" ::: "memory");  // one phase behind
  // A group's tile multiplies only the bands of 32 rows that it has: a copy of the loop per number of them (a
  // condition on every band inside one loop takes registers that the loop needs)
  if constexpr (GROUPED) {
    const int live = (min(rows_left, BM) + 31) / 32;
    unrolled<1, TM + 1>([&](auto bands) __attribute__((always_inline)) { if (live == decltype(bands)::value) walk_k(bands); });
  } else {
    walk_k(std::integral_constant<int, TM>{});
  }
  if (first_group) asm volatile("s_barrier" ::: "memory");
  // (the loads past the last step write zeros)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (AHEAD) asm volatile("" ::"v"(touched));
  __syncthreads();

  // Out through LDS as in dense_gemm_kernel, a band of 16 rows at a time: a lane holds columns
  // j * 16 + q * 4 + 0..3 of row r, and a store instruction writes whole 128-byte pieces of rows.
  // How they are stored (Store), measured as us of the product alone, plain / through / streaming, and with a kernel
  // behind it that reads the result. Results of up to 64 MB go through: 2048 x 4096 x 256 9.8 / 8.3 / 9.1, with the
  // reader 15.8 / 14.6 / 16.6; 4096 x 6144 x 512 32.2 / 30.6 / 31.0, 47.5 / 46.1 / 48.1. Larger ones are streamed
  // where there is work to write them behind (8192 x 8192 x 3696 375 / 372 / 369, 416 / 413 / 415), and plain where
  // that would cost the reader more than it gains (8192 x 8192 x 512 83 / 87 / 72, 123 / 127 / 128). Experts' results
  // are streamed, which leaves L2 to the operands: 32 x 256 rows, 4096 x 2048 145 / 144 / 137, 180 / 183 / 177.
  // (Tiles of one per workgroup make no results of more than 21 MB: linear_way.)
  const bool large = !ONE_TILE && (long long)M * N > (32ll << 20), streams = GROUPED || (large && K >= 2048);
  constexpr int VR = TN * 2, PITCH = TN * 32 + 16, ROWS_PER_READ = 64 / VR, BAND_STORES = 16 / ROWS_PER_READ;
  static_assert(8 * 16 * PITCH <= A_BYTES, "results leave through the last buffer of A, which a tile's first loads leave alone");
  char* park = (char*)tile_lds + (NA - 1) * A_BYTES + wave * (16 * PITCH);
  uint16_t* const c_tile = C + row_at * N;
  const int ncol = n0 + wn * TN * 16, rows_out = rows_left;
  const bool whole_columns = n0 + BN <= N, with_bias = bias_row != nullptr;
  uint32_t bias2[TN][2] = {};
  if (with_bias) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
      if (ncol + j * 16 < N) __builtin_memcpy(bias2[j], bias_row + ncol + j * 16 + q * 4, 8);
#pragma unroll
    for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(bias2[j][0]), "+v"(bias2[j][1]));  // (waited for here, ahead of the loads below)
  }
  bool more = false;
  if constexpr (!ONE_TILE) {
    tile += gridDim.x;
    more = tile < total_tiles;
  }
  if (EARLY && more) {
    find_tile();
    begin_tile();
  }
  {
    int rrow = lane / VR, rvec = lane % VR;
    // (the places of all bands are worked out here: ahead of the loop over tiles they would take 60 registers)
    asm volatile("" : "+v"(rrow), "+v"(rvec));
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const f32x4& c = acc[i][j];
        uint32_t two[2] = {Pair16<DT>::canonical(Pair16<DT>::round(c[0], c[1])),
                           Pair16<DT>::canonical(Pair16<DT>::round(c[2], c[3]))};
        if (with_bias) {
#pragma unroll
          for (int e = 0; e < 2; ++e)
            two[e] = Pair16<DT>::canonical(Pair16<DT>::round(
                __fadd_rn(Pair16<DT>::lo(two[e]), Pair16<DT>::lo(bias2[j][e])),
                __fadd_rn(Pair16<DT>::hi(two[e]), Pair16<DT>::hi(bias2[j][e]))));
        }
        __builtin_memcpy(park + r * PITCH + (j * 16 + q * 4) * 2, two, 8);
      }
#pragma unroll
      for (int p = 0; p < 16 / ROWS_PER_READ; ++p) {
        const int row = p * ROWS_PER_READ + rrow;
        const b128 v = *(const b128*)(park + row * PITCH + rvec * 16);
        const int m = i * 32 + wm * 16 + row, n = ncol + rvec * 8;
        if (m < rows_out && n < N) {
          b128* const to = (b128*)(c_tile + (size_t)m * N + n);
          if (streams) row_store<STREAM>(to, v);
          else if (large) row_store<PLAIN>(to, v);
          else row_store<THROUGH>(to, v);
        }
      }
    }
  }
  if (!more) return;
  if constexpr (!EARLY) {
    lds_barrier();  // the results are out of LDS
    find_tile();
    begin_tile();
    clear();
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FIRST_YOUNGER) : "memory");
    continue;
  }
  clear();
  // The first step's rows: all but the youngest first loads and the stores behind them, of which there are as many as
  // whole bands. (Loads and stores are counted in the order in which they were issued.)
  constexpr int STORES = TM * BAND_STORES;
  if (whole_columns && rows_out >= BM) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FIRST_YOUNGER + STORES) : "memory");
  else if (whole_columns && rows_out >= BM / 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FIRST_YOUNGER + STORES / 2) : "memory");
  else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FIRST_YOUNGER) : "memory");
  }
}

// ---------------------------------------------------------------- exchange stand-in

// (ArgumentsLoaded: nothing waits for these arguments that the counts would not be waited for as well. A leg of 64 rows of 1 KB 2.12 / 2.01 us.)
template <typename V, int NV, Store HOW>
__global__ __launch_bounds__(BLOCK) void exchange_local_kernel(
    ArgumentsLoaded, const V* __restrict__ send_buf, const int* __restrict__ send_meta,
    const int* __restrict__ send_counts, int dst_rank, V* __restrict__ recv_buf,
    int* __restrict__ recv_meta, const int* __restrict__ recv_counts, int src_rank, int row_vecs,
    int chunks, int send_capacity_rows, int recv_capacity_rows) {
  const int tid = threadIdx.x;
  const int src_off = sum_counts(send_counts, dst_rank, send_capacity_rows);
  const int dst_off = sum_counts(recv_counts, src_rank, recv_capacity_rows);
  int n = min(max(send_counts[dst_rank], 0), max(recv_counts[src_rank], 0));
  // never past what either buffer holds, whatever the counts claim
  n = max(min(n, min(send_capacity_rows - src_off, recv_capacity_rows - dst_off)), 0);
  const int items = n * chunks;
  for (int q = blockIdx.x; q < items; q += gridDim.x) {
    const int i = chunks == 1 ? q : q / chunks, c = q - i * chunks;
    const int base = c * (BLOCK * NV);
    Payload<V, NV> p;
    p.load(send_buf + (size_t)(src_off + i) * row_vecs, base, row_vecs);
    p.template store<HOW>(recv_buf + (size_t)(dst_off + i) * row_vecs, base, row_vecs);
    if (c == 0 && tid < META)
      recv_meta[(size_t)(dst_off + i) * META + tid] = send_meta[(size_t)(src_off + i) * META + tid];
  }
}

// All source legs of one destination in one launch: blockIdx.y is the source rank. The W source
// buffers are separate allocations (one per rank object), so their addresses travel by value in
// the kernel arguments. Every wave works out both offsets of its leg from the W counts the
// sources hold for this destination (one lane per source, a wave scan) and the kernel also
// writes those counts to recv_counts, which an exchange of counts would have delivered
// (all2all/reference.py:88-91,181-185).
constexpr int GATHER_MAX_RANKS = 64;
struct GatherSources {
  const void* buf[GATHER_MAX_RANKS];
  const int* meta[GATHER_MAX_RANKS];
  const int* counts[GATHER_MAX_RANKS];
};

template <typename V, int NV, Store HOW>
__global__ __launch_bounds__(BLOCK) void exchange_gather_kernel(
    GatherSources src, int W, int dst_rank, V* __restrict__ recv_buf, int* __restrict__ recv_meta,
    int* __restrict__ recv_counts, int row_vecs, int chunks, int send_capacity_rows,
    int recv_capacity_rows) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int s = blockIdx.y;
  // rows every source holds for this destination (lane l: source l)
  const int held = lane < W ? min(max(src.counts[lane][dst_rank], 0), send_capacity_rows) : 0;
  const int upto = wave_inclusive_scan(held);
  if (blockIdx.x == 0 && s == 0 && tid < W) recv_counts[tid] = held;
  const int dst_off = __builtin_amdgcn_readlane(upto - held, s);
  const int* __restrict__ my_counts = src.counts[s];
  const int src_off = sum_counts(my_counts, dst_rank, send_capacity_rows);
  int n = __builtin_amdgcn_readlane(held, s);
  // never past what either buffer holds, whatever the counts claim
  n = max(min(n, min(send_capacity_rows - src_off, recv_capacity_rows - dst_off)), 0);
  const V* __restrict__ send_buf = (const V*)src.buf[s];
  const int* __restrict__ send_meta = src.meta[s];
  const int items = n * chunks;
  for (int q = blockIdx.x; q < items; q += gridDim.x) {
    const int i = chunks == 1 ? q : q / chunks, c = q - i * chunks;
    const int base = c * (BLOCK * NV);
    Payload<V, NV> p;
    p.load(send_buf + (size_t)(src_off + i) * row_vecs, base, row_vecs);
    p.template store<HOW>(recv_buf + (size_t)(dst_off + i) * row_vecs, base, row_vecs);
    if (c == 0 && tid < META)
      recv_meta[(size_t)(dst_off + i) * META + tid] = send_meta[(size_t)(src_off + i) * META + tid];
  }
}

// ---------------------------------------------------------------- jobs whose ranks share the GPU
//
// Where every rank of a job lives on this GPU there is nothing to exchange: a token's row can go straight
// to its experts' rows and come straight back. Three kernels replace the five stages and two exchanges:
//   local_plan_kernel      the expert-buffer row of every (rank, token, k) entry (entry_row), in the order in
//                          which the stages would have put it there: by source rank, token and k inside an
//                          expert. Left out for up to LOCAL_FEW_RANKS ranks with LOCAL_RANK_ENTRIES entries
//                          between them, whose mover ranks them itself (local_dispatch_few_kernel), and for up to
//                          32768 entries of whole vectors (local_dispatch_long_kernel).
//   local_dispatch_kernel  one workgroup per (token, chunk of its row) reads the chunk once and stores it to
//                          all of the token's expert rows, as it is or through the stand-in expert.
//   local_combine_kernel   one workgroup per (token, chunk): gathers the token's expert rows and adds them up
//                          in arrival order. Rows come back by destination rank, expert and position, so
//                          arrival order is the order of the expert-buffer rows themselves, in both layouts.
// Bound by memory: a row is written once to its expert and read once from there, where the stages and
// copies moved it six times.

constexpr int LOCAL_MAX_RANKS = 64;
constexpr int LOCAL_MAX_EXPERTS = 1024;     // counters of the plan in LDS
constexpr int LOCAL_MAX_K = 64;             // entries of a token, one per lane
constexpr int LOCAL_FEW_RANKS = 8;          // a table that a wave holds in scalar registers
// Up to here in a launch. Picking costs each wave some fifty scalar instructions, which many short waves take longer for than for the
// dependent load that lanes of other waves hide: us, job's way back with compares / loads by rank, 4792 tokens of 512 bytes, 2 per token 8.49 /
// 8.03, 7944 of 640 bytes, 5 each 17.7 / 16.6, 2256 of 768 bytes, 3 each 5.97 / 5.63; planned dispatch of 18768 of 512 bytes 35.0 / 33.8.
constexpr int LOCAL_FEW_WORKGROUPS = 2048;
constexpr int LOCAL_RANK_BITS = 11;
constexpr int LOCAL_RANK_ENTRIES = 1 << LOCAL_RANK_BITS;  // 32 keys per lane of a wave

// Tables of R ranks, passed by value. Jobs of up to eight ranks pass eight entries: a launch with 1.3 KB of arguments takes
// the host 4.6 us where one with a few words takes 3.0, and eight entries are read at once and picked from by compares,
// where a table of 64 costs each wave a load of `first` by lane and then one by rank.
template <int R>
struct LocalSources {
  const void* x[R];
  const int* indices[R];
  int first[R + 1];  // number of the rank's first token, counted over all ranks (up to [W]; INT_MAX behind it)
};
template <int R>
struct LocalResults {
  const float* weights[R];
  void* out[R];
  int first[R + 1];
};

// the rank that token number t (the same for every lane of the wave) belongs to
template <int R>
__device__ __forceinline__ int rank_of_token(const int (&first)[R + 1], int W, int t) {
  if constexpr (R <= LOCAL_FEW_RANKS) {
    int r = 0;
#pragma unroll
    for (int s = 1; s < R; ++s) r += (int)(first[s] <= t);
    return r;
  } else {
    const int lane = threadIdx.x & 63;
    return __popcll(__ballot(lane < W && first[lane] <= t)) - 1;
  }
}
// table[r], with r the same for every lane
template <int R, typename T>
__device__ __forceinline__ T of_rank(const T* table, int r) {
  if constexpr (R <= LOCAL_FEW_RANKS) {
    T v = table[0];
#pragma unroll
    for (int s = 1; s < R; ++s) v = s == r ? table[s] : v;
    return v;
  } else {
    return table[r];
  }
}

constexpr int LPLAN_BLOCK = 1024, LPLAN_WAVES = LPLAN_BLOCK / 64;

// One workgroup per 1024 entries. Entries before the tile go through an LDS histogram per expert; inside the
// tile an entry's place among the lanes of its wave with the same expert comes from one ballot per bit of
// the expert number, the waves are ordered by a prefix over their counts (as in plan_recv_kernel).
//   compact        row = rows of lower experts + position, else expert * max_recv + position
//   expert_limit   entries at or past that position in their expert are dropped (row -1), as the padded
//                  buffers of all2all/reference.py:123-136 have no room for them
//   rank_limit     > 0: entries past that many of their destination rank are dropped (what its receive
//                  buffer holds). Reached only by tokens that name an expert more than once.
// Entries with an expert outside [0, E) have no row. The last workgroup writes the rows per expert.
// Here: the row of the lane's entry, of up to one per lane from `begin` to before `end`; `entry_expert` is what the entry names.
template <int R>
__device__ __forceinline__ int local_plan(
    const LocalSources<R>& src, int W, int S, int K, int E, int nle, int expert_bits, int rank_bits, bool compact, int max_recv,
    int expert_limit, int rank_limit, int begin, int end, int* __restrict__ expert_num_tokens,
    int* __restrict__ expert_offsets, int& entry_expert) {
  extern __shared__ int plan_lds[];            // before[E], total[E], in_wave[LPLAN_WAVES][E]
  int* const before = plan_lds;
  int* const total = plan_lds + E;
  int* const in_wave = plan_lds + 2 * E;
  __shared__ int first_entry[LOCAL_MAX_RANKS + 1];
  __shared__ const int* keys_of[LOCAL_MAX_RANKS];
  __shared__ int rank_in_wave_of[LPLAN_WAVES][LOCAL_MAX_RANKS];
  __shared__ int rank_before[LOCAL_MAX_RANKS];
  __shared__ int red[LPLAN_WAVES];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const unsigned long long lanes_below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const bool last = blockIdx.x == gridDim.x - 1;
  if (tid <= W) first_entry[tid] = src.first[tid] * K;
  if (tid < W) keys_of[tid] = src.indices[tid];
  for (int j = tid; j < (2 + LPLAN_WAVES) * E; j += LPLAN_BLOCK) plan_lds[j] = 0;
  for (int j = tid; j < LPLAN_WAVES * LOCAL_MAX_RANKS; j += LPLAN_BLOCK) (&rank_in_wave_of[0][0])[j] = 0;
  __syncthreads();
  auto rank_of = [&](int i) {  // of entry i < S
    int r = 0;
    for (int step = rank_bits ? 1 << (rank_bits - 1) : 0; step > 0; step >>= 1)
      if (r + step < W && first_entry[r + step] <= i) r += step;
    return r;
  };
  auto key_at = [&](int i) {  // its expert id
    const int r = rank_of(i);
    return keys_of[r][i - first_entry[r]];
  };
  const int i = begin + tid;
  const int e = i < end ? key_at(i) : -1;
  entry_expert = e;
  const int scanned = compact ? S : begin;
  // compact: both counts of an expert in one word where they fit, all entries below, those before the tile above
  const bool packed = compact && S <= 0xffff;
  auto before_of = [&](int j) { return packed ? (int)((uint32_t)before[j] >> 16) : before[j]; };
  auto total_of = [&](int j) { return packed ? before[j] & 0xffff : total[j]; };
  auto count = [&](int key, int i2) __attribute__((always_inline)) {
    if (i2 >= scanned || (uint32_t)key >= (uint32_t)E) return;
    if (packed) {
      atomicAdd(&before[key], i2 < begin ? 0x10001 : 1);
    } else {
      if (compact) atomicAdd(&total[key], 1);
      if (i2 < begin) atomicAdd(&before[key], 1);
    }
  };
  if (W == 1) {
    for (int b = 0; b < scanned; b += SCAN_UNROLL * LPLAN_BLOCK) {
      int e2[SCAN_UNROLL];
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) e2[u] = keys_of[0][min(b + tid + u * LPLAN_BLOCK, scanned - 1)];
#pragma unroll
      for (int u = 0; u < SCAN_UNROLL; ++u) count(e2[u], b + tid + u * LPLAN_BLOCK);
    }
  } else {
    // Four entries of a rank with one search for it and one load: the searches were a third of the time (16384 entries
    // of 8 ranks, 256 experts: 11.2 us, of which the second counter took another; 7.9 with both).
    constexpr int VEC = 4, UNROLL = 4;
    const int vecs = (scanned + VEC - 1) / VEC;
    for (int b = 0; b < vecs; b += UNROLL * LPLAN_BLOCK) {
      int e2[UNROLL][VEC];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int i2 = min(b + tid + u * LPLAN_BLOCK, vecs - 1) * VEC, r = rank_of(i2);
        const int* from = keys_of[r] + (i2 - first_entry[r]);
        if (i2 + VEC <= min(first_entry[r + 1], scanned)) {
          __builtin_memcpy(e2[u], from, sizeof e2[u]);  // (4-byte aligned, which global loads accept)
        } else {
#pragma unroll
          for (int v = 0; v < VEC; ++v) e2[u][v] = key_at(min(i2 + v, scanned - 1));
        }
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
#pragma unroll
        for (int v = 0; v < VEC; ++v) count(e2[u][v], (b + tid + u * LPLAN_BLOCK) * VEC + v);
    }
  }
  const bool ok = (uint32_t)e < (uint32_t)E;
  unsigned long long same = __ballot(ok);
  for (int b = 0; b < expert_bits; ++b) {
    const bool set = (e >> b) & 1;
    const unsigned long long with_bit = __ballot(set);
    same &= set ? with_bit : ~with_bit;
  }
  const int in_wave_before = __popcll(same & lanes_below);
  if (ok && in_wave_before == 0) in_wave[wave * E + e] = __popcll(same);
  const int dst = ok ? e / nle : 0;
  int rank_lane_before = 0;
  if (rank_limit > 0) {
    unsigned long long peers = __ballot(ok);
    for (int b = 0; b < rank_bits; ++b) {
      const bool set = (dst >> b) & 1;
      const unsigned long long with_bit = __ballot(set);
      peers &= set ? with_bit : ~with_bit;
    }
    rank_lane_before = __popcll(peers & lanes_below);
    if (ok && rank_lane_before == 0) rank_in_wave_of[wave][dst] = __popcll(peers);
  }
  __syncthreads();
  int pos = 0;
  if (ok) {
    pos = before_of(e) + in_wave_before;
    for (int w = 0; w < wave; ++w) pos += in_wave[w * E + e];
  }
  bool keep = ok && pos < expert_limit;
  if (rank_limit > 0) {
    if (tid < W) {
      int n = 0;
      for (int j = 0; j < nle; ++j) n += before_of(tid * nle + j);
      rank_before[tid] = n;
    }
    __syncthreads();
    if (ok) {
      int n = rank_before[dst] + rank_lane_before;
      for (int w = 0; w < wave; ++w) n += rank_in_wave_of[w][dst];
      keep = keep && n < rank_limit;
    }
  }
  if (compact) {  // exclusive prefix of the rows per expert (E <= 1024: one expert per lane)
    const int mine = tid < E ? total_of(tid) : 0;
    const int incl = wave_inclusive_scan(mine);
    if (lane == 63) red[wave] = incl;
    __syncthreads();
    int off = incl - mine;
    for (int w = 0; w < wave; ++w) off += red[w];
    if (tid < E) total[tid] = off;
    if (last && tid < E && expert_offsets) {
      expert_offsets[tid] = off;
      if (tid == E - 1) expert_offsets[E] = off + mine;
    }
    if (last && tid < E && expert_num_tokens) expert_num_tokens[tid] = mine;
    __syncthreads();
  } else if (last && expert_num_tokens) {
    for (int j = tid; j < E; j += LPLAN_BLOCK) {
      int n = before_of(j);
      for (int w = 0; w < LPLAN_WAVES; ++w) n += in_wave[w * E + j];
      expert_num_tokens[j] = n;
    }
  }
  return !keep ? -1 : compact ? total[e] + pos : e * max_recv + pos;
}

template <int R>
__global__ __launch_bounds__(LPLAN_BLOCK) void local_plan_kernel(
    LocalSources<R> src, int W, int S, int K, int E, int nle, int expert_bits, int rank_bits, bool compact, int max_recv,
    int expert_limit, int rank_limit, int* __restrict__ entry_row, int* __restrict__ expert_num_tokens,
    int* __restrict__ expert_offsets) {
  const int begin = blockIdx.x * LPLAN_BLOCK, i = begin + threadIdx.x;
  int e;
  const int row = local_plan<R>(src, W, S, K, E, nle, expert_bits, rank_bits, compact, max_recv, expert_limit, rank_limit, begin,
                                min(S, begin + LPLAN_BLOCK), expert_num_tokens, expert_offsets, e);
  if (i < S) entry_row[i] = row;
}

// The token's row, held by the workgroup, to its K places: row_of and own hold the places and experts of entries, one per
// lane. DIN / DOUT >= 0: rows leave as `row.to(out) * (1 + rank of the expert)` (all2all/reference.py:262).
template <int DIN, int DOUT, Store HOW, typename V, int NV>
__device__ __forceinline__ void local_rows_out(const Payload<V, NV>& p, int base, int row_vecs, int K, int row_of, int own, int nle,
                                               uint32_t magic, V* __restrict__ rows) {
  for (int k = 0; k < K; ++k) {
    const int row = __builtin_amdgcn_readlane(row_of, k);
    if (row < 0) continue;
    V* __restrict__ to = rows + (size_t)row * row_vecs;
    if constexpr (DIN >= 0) {
      const int e = __builtin_amdgcn_readlane(own, k);
      const float scale = (float)(1 + (nle == 1 ? e : (int)__umulhi((uint32_t)e, magic)));
      Payload<V, NV> y = p;
      y.map([scale](V v) { return standin_expert<V, DIN, DOUT>(v, scale); });
      y.template store<HOW>(to, base, row_vecs);
    } else {
      p.template store<HOW>(to, base, row_vecs);
    }
  }
}
__device__ __forceinline__ void local_meta_out(int K, int row_of, int own, int r, int local_t, int* __restrict__ meta) {
  for (int m0 = 0; m0 < K * META; m0 += BLOCK) {  // (the same trips for every lane: they shuffle)
    const int m = m0 + threadIdx.x, k = min(m / META, K - 1), f = m - k * META;
    const int row = __shfl(row_of, k, 64), e = __shfl(own, k, 64);
    if (m < K * META && row >= 0) meta[(size_t)row * META + f] = f == 0 ? e : f == 1 ? r : f == 2 ? local_t : f == 3 ? k : 0;
  }
}

template <typename V, int NV, int DIN, int DOUT, Store HOW, int R>
__global__ __launch_bounds__(BLOCK) void local_dispatch_kernel(
    const int* __restrict__ entry_row, V* __restrict__ rows, int* __restrict__ meta, int W, int K, int chunks, int row_vecs,
    int nle, uint32_t magic, LocalSources<R> src) {
  const int lane = threadIdx.x & 63;
  const int q = blockIdx.x;
  const int t = chunks == 1 ? q : q / chunks, c = q - t * chunks;
  const int row_of = entry_row[(size_t)t * K + min(lane, K - 1)];
  const int r = rank_of_token<R>(src.first, W, t), local_t = t - of_rank<R>(src.first, r);
  const int base = c * (BLOCK * NV);
  const int own = of_rank<R>(src.indices, r)[(size_t)local_t * K + min(lane, K - 1)];
  Payload<V, NV> p;
  p.load((const V*)of_rank<R>(src.x, r) + (size_t)local_t * row_vecs, base, row_vecs);
  local_rows_out<DIN, DOUT, HOW>(p, base, row_vecs, K, row_of, own, nle, magic, rows);
  if (c == 0 && meta) local_meta_out(K, row_of, own, r, local_t, meta);
}

// The same with the plan in it: a workgroup ranks the entries of `tokens` tokens and its waves move their rows, pieces of 64 * NV vectors, the first
// ones of which are on their way while it counts. Every workgroup counts up to all keys, at once and about as long as the last one of a plan, whose
// launch is saved. Bound by memory, on small jobs by that count. us of both launches / here: 8 ranks, 2048 tokens of 14 KB, 8 per token 49.3 /
// 47.6 (6.4 TB/s in the rows), 1920 of 11 KB, 7 each 34.9 / 31.9, 1528 of 7 KB, 4 each 16.0 / 14.1, 520 of 8.6 KB, 5 each 13.8 / 11.2; one rank, 2048 of 8 KB,
// 4 each 20.2 / 17.7, 3084 of 1.6 KB, 2 each 9.9 / 7.2.
template <int NV, int DIN, int DOUT, int R>
__global__ __launch_bounds__(LPLAN_BLOCK) void local_dispatch_long_kernel(
    LocalSources<R> src, int W, int S, int K, int E, int nle, uint32_t magic, int expert_bits, int rank_bits, bool compact, int max_recv,
    int expert_limit, int rank_limit, int tokens, Pieces pieces, int row_vecs, int* __restrict__ entry_row,
    int* __restrict__ expert_num_tokens, int* __restrict__ expert_offsets, b128* __restrict__ rows, int* __restrict__ meta) {
  __shared__ int places[LOCAL_LONG_ENTRIES], experts[LOCAL_LONG_ENTRIES];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int t0 = blockIdx.x * tokens, begin = t0 * K, end = min(S, begin + tokens * K);
  const int items = (end - begin) / K * pieces.per_row;
  WavePayload<b128, NV> p;
  auto load = [&](int q) __attribute__((always_inline)) {
    const int item = pieces.row_of(q), r = rank_of_token<R>(src.first, W, t0 + item), local_t = t0 + item - of_rank<R>(src.first, r);
    p.load((const b128*)of_rank<R>(src.x, r) + (size_t)local_t * row_vecs, (q - item * pieces.per_row) * (64 * NV), row_vecs, lane);
  };
  if (wave < items) load(wave);
  int e;
  const int row = local_plan<R>(src, W, S, K, E, nle, expert_bits, rank_bits, compact, max_recv, expert_limit, rank_limit, begin, end,
                                expert_num_tokens, expert_offsets, e);
  if (begin + tid < end) {
    entry_row[begin + tid] = row;
    places[tid] = row;
    experts[tid] = e;
  }
  lds_barrier();
  for (int q = wave; q < items; q += LPLAN_WAVES) {
    if (q != wave) load(q);
    const int item = pieces.row_of(q), base = (q - item * pieces.per_row) * (64 * NV);
    const int row_of = places[item * K + min(lane, K - 1)], own = experts[item * K + min(lane, K - 1)];
    for (int k = 0; k < K; ++k) {
      const int to = __builtin_amdgcn_readlane(row_of, k);
      if (to < 0) continue;
      WavePayload<b128, NV> y = p;
      if constexpr (DIN >= 0) {
        const int of = __builtin_amdgcn_readlane(own, k);
        const float scale = (float)(1 + (nle == 1 ? of : (int)__umulhi((uint32_t)of, magic)));
#pragma unroll
        for (int j = 0; j < NV; ++j) y.v[j] = standin_expert<b128, DIN, DOUT>(p.v[j], scale);
      }
      y.template store<THROUGH>(rows + (size_t)to * row_vecs, base, row_vecs, lane);
    }
    if (base == 0 && meta) {
      const int t = t0 + item, r = rank_of_token<R>(src.first, W, t), local_t = t - of_rank<R>(src.first, r);
      for (int m0 = 0; m0 < K * META; m0 += 64) {  // (the same trips for every lane: they shuffle)
        const int m = m0 + lane, k = min(m / META, K - 1), f = m - k * META;
        const int to = __shfl(row_of, k, 64), of = __shfl(own, k, 64);
        if (m < K * META && to >= 0) meta[(size_t)to * META + f] = f == 0 ? of : f == 1 ? r : f == 2 ? local_t : f == 3 ? k : 0;
      }
    }
  }
}

// The same without a plan, for few entries of few ranks: every wave holds all keys (KEYS per lane) and ranks entries of its own
// (wave, wave + 4, ...), as dispatch_few_kernel does; workgroup 0 counts the rows per expert where the caller wants
// to know them. x0 and indices0 are rank 0's, which is all that a job of one rank has (R = 1).
// A plan's launch costs more than the scan, and the chain from launch to last store is what bounds these jobs. us of a whole
// job in a graph with partial counts added up over the waves and tables of 64 ranks / here: 8 ranks x 16 tokens x 2, hidden
// 6144 10.9 / 7.9, x 30 x 4, 2880 11.9 / 10.3, x 7 x 6, 7168 13.5 / 9.3, x 24 x 8, 4096 13.0 / 12.4 (16.2 with keys that every
// wave picks up by itself); one rank's dispatch, expert and combine, 16 tokens x 2, hidden 256 10.5 / 9.3, 180 x 8, 4096 18.9 /
// 17.7. NV: vectors of the row that a lane moves (local_few_vecs).
template <typename V, int DIN, int DOUT, Store HOW, int R, int KEYS, int NV>
__global__ __launch_bounds__(BLOCK) void local_dispatch_few_kernel(
    const void* x0, const int* indices0, int T, int K, int E, int chunks, int row_vecs, bool counts, bool compact, int max_recv,
    int expert_limit, int nle, uint32_t magic, int W, int* __restrict__ entry_row, int* __restrict__ expert_num_tokens,
    int* __restrict__ expert_offsets, V* __restrict__ rows, int* __restrict__ meta, LocalSources<R> src) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int S = T * K;
  // expert id of entry i, counted over all ranks
  auto key_at = [&](int i) {
    const int* from = indices0;
    if constexpr (R > 1) {
      int first = 0;
#pragma unroll
      for (int r = 1; r < R; ++r) {
        const int f = r < W ? src.first[r] * K : INT_MAX;
        from = f <= i ? src.indices[r] : from;
        first = f <= i ? f : first;
      }
      from -= first;
    }
    return from[i];
  };
  int q = blockIdx.x;
  if (counts) {
    if (q == 0) {
      __shared__ int hist[LOCAL_MAX_EXPERTS];
      __shared__ int red[NWAVES];
      constexpr int EACH = LOCAL_MAX_EXPERTS / BLOCK, MINE = KEYS / NWAVES;
      int key[MINE];
#pragma unroll
      for (int u = 0; u < MINE; ++u) key[u] = key_at(min(tid + u * BLOCK, S - 1));
      for (int j = tid; j < E; j += BLOCK) hist[j] = 0;
      lds_barrier();
#pragma unroll
      for (int u = 0; u < MINE; ++u)
        if (tid + u * BLOCK < S && (uint32_t)key[u] < (uint32_t)E) atomicAdd(&hist[key[u]], 1);
      lds_barrier();
      int own[EACH], sum = 0;
#pragma unroll
      for (int j = 0; j < EACH; ++j) {
        own[j] = tid * EACH + j < E ? hist[tid * EACH + j] : 0;
        sum += own[j];
      }
      const int incl = wave_inclusive_scan(sum);
      if (lane == 63) red[wave] = incl;
      lds_barrier();
      int off = incl - sum;
      for (int w = 0; w < wave; ++w) off += red[w];
#pragma unroll
      for (int j = 0; j < EACH; ++j) {
        const int e = tid * EACH + j;
        if (e < E) {
          if (expert_num_tokens) expert_num_tokens[e] = own[j];
          if (expert_offsets) {
            expert_offsets[e] = off;
            if (e == E - 1) expert_offsets[E] = off + own[j];
          }
        }
        off += own[j];
      }
      return;
    }
    --q;
  }
  const int t = chunks == 1 ? q : q / chunks, c = q - t * chunks;
  int r = 0, local_t = t;
  const void* x = x0;
  const int* indices = indices0;
  if constexpr (R > 1) {
    r = rank_of_token<R>(src.first, W, t);
    local_t = t - of_rank<R>(src.first, r);
    x = of_rank<R>(src.x, r);
    indices = of_rank<R>(src.indices, r);
  }
  const int base = c * (BLOCK * NV);
  const int own = indices[(size_t)local_t * K + min(lane, K - 1)];
  // The waves load a quarter of the keys each and share them through LDS where the ranks' pointers have to be picked from
  // for every key, and where there are many
  constexpr bool SHARED = R > 1 || KEYS > 4;
  constexpr int LOADED = SHARED ? KEYS / NWAVES : KEYS;
  int loaded[LOADED], key[KEYS];
  const int mine0 = SHARED ? tid : lane;
#pragma unroll
  for (int u = 0; u < LOADED; ++u) loaded[u] = key_at(min(mine0 + u * (SHARED ? BLOCK : 64), S - 1));
  Payload<V, NV> p;
  p.load((const V*)x + (size_t)local_t * row_vecs, base, row_vecs);

  // a key's place in (expert, entry) order; ids outside [0, E) come last
  __shared__ int places[LOCAL_MAX_K];
  auto composite = [&](int e, int i) { return ((uint32_t)e < (uint32_t)E ? e : E) << LOCAL_RANK_BITS | i; };
#pragma unroll
  for (int u = 0; u < LOADED; ++u) {
    const int i = mine0 + u * (SHARED ? BLOCK : 64);
    loaded[u] = i < S ? composite(loaded[u], i) : INT_MAX;
  }
  if constexpr (SHARED) {  // (in whatever order: a key holds its place)
    __shared__ b128 all[KEYS * 16];
#pragma unroll
    for (int u = 0; u < LOADED; ++u) ((int*)all)[tid + u * BLOCK] = loaded[u];
    lds_barrier();
#pragma unroll
    for (int u = 0; u < KEYS / 4; ++u) {
      const b128 four = all[lane + u * 64];
#pragma unroll
      for (int v = 0; v < 4; ++v) key[u * 4 + v] = (int)four[v];
    }
  } else {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) key[u] = loaded[u];
  }
  for (int k = wave; k < K; k += NWAVES) {
    const int e = __builtin_amdgcn_readlane(own, k);
    const int mine = composite(e, t * K + k), from = mine & ~(LOCAL_RANK_ENTRIES - 1);
    int pos = 0, lower = 0;  // entries ahead of it in its expert, and of lower experts
#pragma unroll
    for (int u = 0; u < KEYS; ++u) pos += __popcll(__ballot((uint32_t)(key[u] - from) < (uint32_t)(mine - from)));
    if (compact) {
#pragma unroll
      for (int u = 0; u < KEYS; ++u) lower += __popcll(__ballot(key[u] < from));
    }
    const bool keep = (uint32_t)e < (uint32_t)E && pos < expert_limit;
    if (lane == 0) places[k] = !keep ? -1 : compact ? lower + pos : e * max_recv + pos;
  }
  lds_barrier();
  const int row_of = places[min(lane, K - 1)];
  local_rows_out<DIN, DOUT, HOW>(p, base, row_vecs, K, row_of, own, nle, magic, rows);
  if (c == 0) {
    if (wave == 0 && lane < K) entry_row[(size_t)t * K + lane] = row_of;
    if (meta) local_meta_out(K, row_of, own, r, local_t, meta);
  }
}

// ADDENDS: 2, 4, 6 or 8, no fewer than a token's entries, whose rows are all under way at once; 0 for more of them, in batches of 8. Past the last one
// its row is loaded again, which costs as much as another (us, all with 8 / as many as here, 3 per token: 3907 tokens of 4.3 KB 15.4 / 14.2; 2 per token:
// 2987 of 6.4 KB 17.4 / 13.2; 1: 3683 of 7.2 KB 17.4 / 13.2; 6, of 8 ranks: 238 of 4.5 KB 13.7 / 12.4).
// weights0 and out0 are rank 0's, which is all that a job of one rank has (R = 1).
template <typename V, int DT, int NV, int ADDENDS, Store HOW, int R>
__global__ __launch_bounds__(BLOCK) void local_combine_kernel(
    const int* __restrict__ entry_row, const float* weights0, const V* __restrict__ rows, void* out0, int K, int chunks,
    int row_vecs, int first_token, int accumulate, int W, LocalResults<R> dst) {
  constexpr int N = Words<V>::N, BATCH = ADDENDS ? ADDENDS : 8, RUN = BATCH > 4 ? 8 : 4;
  constexpr bool MANY = ADDENDS == 0;
  const int tid = threadIdx.x, lane = tid & 63;
  const int q = blockIdx.x;
  const int item = chunks == 1 ? q : q / chunks, c = q - item * chunks;
  const int t = first_token + item;
  int local_t = t;
  const float* weights = weights0;
  void* out = out0;
  if constexpr (R > 1) {
    const int r = rank_of_token<R>(dst.first, W, t);
    local_t = t - of_rank<R>(dst.first, r);
    weights = of_rank<R>(dst.weights, r);
    out = of_rank<R>(dst.out, r);
  }
  const int base = c * (BLOCK * NV);
  V* __restrict__ orow = (V*)out + (size_t)local_t * row_vecs;
  // entry of this lane; lanes repeat the entries in runs of 4 or 8 unless there are more
  const int k = MANY ? lane : lane & (RUN - 1);
  const bool there = k < K;
  const int loaded = entry_row[(size_t)t * K + min(k, K - 1)];
  const float w_loaded = weights[(size_t)local_t * K + min(k, K - 1)];
  PairAcc<DT> acc[NV][N];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    V o{};
    if (accumulate) o = orow[min(base + j * BLOCK + tid, row_vecs - 1)];
#pragma unroll
    for (int e = 0; e < N; ++e) acc[j][e].set(get_word(o, e));
  }
  const int mine = there && loaded >= 0 ? loaded : INT_MAX;
  const int n = __popcll(__ballot(mine != INT_MAX && lane < (MANY ? 64 : RUN)));
  // place of this lane's row among the token's rows (all different), then rows and weights in order
  int place = 0;
  if constexpr (MANY) {
    for (int b = 0; b < K; ++b) place += (int)(__builtin_amdgcn_readlane(mine, b) < mine);
  } else {
#define MOE_A2A_ROT(S) place += (int)(__builtin_amdgcn_update_dpp(0, mine, 0x120 + S, 0xf, 0xf, false) < mine)
    MOE_A2A_ROT(1); MOE_A2A_ROT(2); MOE_A2A_ROT(3);
    if constexpr (RUN > 4) { MOE_A2A_ROT(4); MOE_A2A_ROT(5); MOE_A2A_ROT(6); MOE_A2A_ROT(7); }
#undef MOE_A2A_ROT
  }
  const int to = (MANY ? place : (lane & ~(RUN - 1)) | place) << 2;  // (lanes without a row all get place n, which nothing reads)
  const int ordered_row = __builtin_amdgcn_ds_permute(to, mine);
  const int ordered_w = __builtin_amdgcn_ds_permute(to, __float_as_int(w_loaded));
  for (int a0 = 0; a0 < n; a0 += BATCH) {
    V v[BATCH][NV];
    float w[BATCH];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const int from = min(a0 + u, n - 1);  // (loaded again past the last one, and not used)
      const int row = __builtin_amdgcn_readlane(ordered_row, from);
      w[u] = __int_as_float(__builtin_amdgcn_readlane(ordered_w, from));
#pragma unroll
      for (int j = 0; j < NV; ++j)
        v[u][j] = rows[(size_t)row * row_vecs + min(base + j * BLOCK + tid, row_vecs - 1)];
    }
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      if (a0 + u < n) {
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
          for (int e = 0; e < N; ++e) acc[j][e].step(get_word(v[u][j], e), w[u]);
      }
    }
    if (!MANY) break;
  }
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int idx = base + j * BLOCK + tid;
    if (idx < row_vecs) {
      uint32_t h[N];
#pragma unroll
      for (int e = 0; e < N; ++e) h[e] = acc[j][e].word();
      row_store<HOW>(orow + idx, from_words<V>(h));
    }
  }
}

// ---------------------------------------------------------------- host side

struct Geometry {
  bool vec16;     // 16-byte vectors usable for every row buffer of the call
  int row_vecs;   // vectors (or 2-byte elements) per row
  int nv;         // block-per-row kernels: vectors per lane (1, 2 or 4)
  int chunks;     //   and workgroups per row = ceil(row_vecs / (BLOCK * nv))
  int nvw;        // wave-per-row kernels: vectors per lane of the row's wave
  int wchunks;    //   and chunks per row = ceil(row_vecs / (64 * nvw))
  int nle;
  int max_recv;
  uint32_t magic; // ceil(2^32 / nle)
};

bool shape_ok(const moe_a2a_shape* s) {
  return s && s->world_size >= 1 && s->rank >= 0 && s->rank < s->world_size &&
         s->num_experts >= s->world_size && s->num_experts <= 65536 &&
         s->num_experts % s->world_size == 0 && s->experts_per_token >= 1 && s->hidden_dim >= 1 &&
         s->max_num_tokens >= 1 &&
         (long long)s->max_num_tokens * s->world_size <= INT_MAX / 8;
}

bool aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

template <typename... P>
bool all_aligned(size_t a, P... ptrs) { return (aligned(ptrs, a) && ...); }

void row_geometry(Geometry& g, int hidden_dim, bool ptrs_16B) {
  const long long row_bytes = 2ll * hidden_dim;
  g.vec16 = (row_bytes % 16 == 0) && ptrs_16B;
  g.row_vecs = g.vec16 ? (int)(row_bytes / 16) : hidden_dim;
  g.nv = g.row_vecs <= BLOCK ? 1 : g.row_vecs <= 2 * BLOCK ? 2 : 4;
  g.chunks = (g.row_vecs + BLOCK * g.nv - 1) / (BLOCK * g.nv);
  g.nvw = 16;
  if (g.vec16) {
    const int need = (g.row_vecs + 63) / 64;
    for (int c : {14, 12, 8, 6, 4, 2, 1})
      if (need <= c) g.nvw = c;
  }
  g.wchunks = (g.row_vecs + 64 * g.nvw - 1) / (64 * g.nvw);
}

template <typename... P>
Geometry geometry(const moe_a2a_shape* s, P... row_ptrs) {
  Geometry g;
  row_geometry(g, s->hidden_dim, all_aligned(16, row_ptrs...));
  g.nle = s->num_experts / s->world_size;
  g.max_recv = s->max_num_tokens * s->world_size;
  g.magic = g.nle == 1 ? 0u : (uint32_t)(0xffffffffu / (uint32_t)g.nle) + 1u;
  return g;
}

// Workgroups that move rows: one per item up to a cap the kernels stride over.
// `items` beyond INT_MAX are rejected by the callers before this is reached.
int mover_blocks(long long items) {
  const long long cap = 1 << 20;
  long long g = items < cap ? items : cap;
  return (int)(g < 1 ? 1 : g);
}

int launch_status() { return hipGetLastError() == hipSuccess ? MOE_A2A_OK : MOE_A2A_ELAUNCH; }

// Picks the <vector type, vectors per lane> instantiation for a geometry.
#define MOE_A2A_FOR_ROW_KERNEL(G, LAUNCH)                  \
  do {                                                     \
    if ((G).vec16) {                                       \
      if ((G).nv == 1) { LAUNCH(b128, 1); }                \
      else if ((G).nv == 2) { LAUNCH(b128, 2); }           \
      else { LAUNCH(b128, 4); }                            \
    } else {                                               \
      if ((G).nv == 1) { LAUNCH(uint16_t, 1); }            \
      else if ((G).nv == 2) { LAUNCH(uint16_t, 2); }       \
      else { LAUNCH(uint16_t, 4); }                        \
    }                                                      \
  } while (0)

// Same for the wave-per-row kernels: <vector type, vectors per lane of a wave>.
#define MOE_A2A_FOR_WAVE_KERNEL(G, LAUNCH)        \
  do {                                            \
    if ((G).vec16) {                              \
      switch ((G).nvw) {                          \
        case 1: LAUNCH(b128, 1); break;           \
        case 2: LAUNCH(b128, 2); break;           \
        case 4: LAUNCH(b128, 4); break;           \
        case 6: LAUNCH(b128, 6); break;           \
        case 8: LAUNCH(b128, 8); break;           \
        case 12: LAUNCH(b128, 12); break;         \
        case 14: LAUNCH(b128, 14); break;         \
        default: LAUNCH(b128, 16); break;         \
      }                                           \
    } else {                                      \
      LAUNCH(uint16_t, 16);                       \
    }                                             \
  } while (0)

Pieces pieces_of(int per_row) {
  Pieces p{per_row, 0, 0};
  if (per_row > 1) {
    int bits = 1;  // per_row <= 1 << bits
    while ((1ll << bits) < per_row) ++bits;
    p.magic = (uint32_t)((1ull << (31 + bits)) / (uint32_t)per_row + 1);
    p.shift = bits - 1;
  }
  return p;
}

// The send-back plan is kept by the lanes of one wave: one lane per source rank
// in stage 2, one lane per local expert in stage 3.
bool plan_supported(const moe_a2a_shape* s) {
  return s->world_size <= 64 && s->num_experts / s->world_size <= 64;
}

// Address of `scratch` on the GPU that is current for the calling thread, looked up once per
// GPU with that GPU current and kept. Returns nullptr if the runtime cannot name it.
constexpr int MAX_GPUS = 64;
std::mutex static_plan_mutex;
int32_t* static_plan_address[MAX_GPUS] = {};

int32_t* static_plan_buffer() {
  int gpu = -1;
  if (hipGetDevice(&gpu) != hipSuccess || gpu < 0 || gpu >= MAX_GPUS) return nullptr;
  std::lock_guard<std::mutex> lock(static_plan_mutex);
  if (!static_plan_address[gpu]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    static_plan_address[gpu] = static_cast<int32_t*>(p);
  }
  return static_plan_address[gpu];
}

// W counts, each cut to `capacity_rows` on the device, must add up inside an int.
bool counts_fit(long long capacity_rows, int world_size) {
  return capacity_rows * world_size <= INT_MAX;
}

// Workgroups of a ranked row move over `rows` rows.
long long group_items(long long rows, const Geometry& g) {
  return (rows + ROWS - 1) / ROWS * g.wchunks;
}

}  // namespace

extern "C" {

const char* moe_a2a_version(void) { return "moe_a2a 0.7 gfx950"; }

#ifndef MOE_A2A_BUILD_ID
#define MOE_A2A_BUILD_ID "unknown"
#endif
const char* moe_a2a_build_id(void) { return MOE_A2A_BUILD_ID; }

const char* moe_a2a_strerror(int status) {
  switch (status) {
    case MOE_A2A_OK: return "ok";
    case MOE_A2A_EINVAL: return "invalid argument (null pointer, bad shape or unsupported size)";
    case MOE_A2A_EALIGN: return "row buffer is not aligned to its 2-byte elements";
    case MOE_A2A_ELAUNCH: return "kernel launch failed";
    case MOE_A2A_ESCRATCH:
      return "shape beyond the library's static buffer (world_size <= 64 and num_local_experts <= 64), "
             "or the buffer's address is unavailable";
    default: return "unknown status";
  }
}

int moe_a2a_dispatch_send(const moe_a2a_shape* s, const void* x, const int32_t* indices,
                          int32_t num_tokens, void* send_buf, int32_t* send_meta,
                          int32_t* send_counts, int32_t* send_slot, void* stream) {
  if (!shape_ok(s) || num_tokens < 0 || num_tokens > s->max_num_tokens || !send_counts)
    return MOE_A2A_EINVAL;
  const long long S = (long long)num_tokens * s->experts_per_token;
  if (S > 0 && (!x || !indices || !send_buf || !send_meta)) return MOE_A2A_EINVAL;
  if (!all_aligned(2, x, send_buf)) return MOE_A2A_EALIGN;
  const Geometry g = geometry(s, x, send_buf);
  if (!items_fit(S, g.wchunks)) return MOE_A2A_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  Geometry f = g;
  f.nv = 1;
  f.chunks = (f.row_vecs + BLOCK - 1) / BLOCK;
  const SendWay way = send_way(num_tokens, s->experts_per_token, s->world_size, g.row_vecs, g.vec16);
  if (way == SEND_FEW) {
    int order_bits = 1, nle_shift = 0;
    while ((1 << order_bits) < S) ++order_bits;
    while ((1 << nle_shift) < g.nle) ++nle_shift;
    const int few_grid = s->world_size + num_tokens * f.chunks, keys = few_keys(S);
#define LAUNCH_K(V, KEYS, POW2)                                                                  \
  dispatch_few_kernel<V, KEYS, POW2><<<few_grid, BLOCK, 0, st>>>(                                \
      (const V*)x, indices, num_tokens, s->experts_per_token, s->world_size, f.chunks,           \
      f.row_vecs, s->num_experts, g.magic, nle_shift, order_bits, s->rank,                       \
      (V*)send_buf, send_meta, send_counts, send_slot)
#define LAUNCH(V, POW2)                                  \
  do {                                                   \
    if (keys == 2) LAUNCH_K(V, 2, POW2);                 \
    else if (keys == 4) LAUNCH_K(V, 4, POW2);            \
    else if (keys == 8) LAUNCH_K(V, 8, POW2);            \
    else if (keys == 12) LAUNCH_K(V, 12, POW2);          \
    else LAUNCH_K(V, 16, POW2);                          \
  } while (0)
    if ((g.nle & (g.nle - 1)) == 0) { if (f.vec16) LAUNCH(b128, true); else LAUNCH(uint16_t, true); }
    else { if (f.vec16) LAUNCH(b128, false); else LAUNCH(uint16_t, false); }
#undef LAUNCH
#undef LAUNCH_K
    return launch_status();
  }
  if (const int own = long_tokens(way, num_tokens, s->experts_per_token, s->world_size, g.row_vecs, g.vec16)) {
    int nle_shift = 0;
    while ((1 << nle_shift) < g.nle) ++nle_shift;
    const int long_grid = (num_tokens + own - 1) / own;
#define LAUNCH(POW2)                                                                             \
  dispatch_long_kernel<POW2><<<long_grid, LONG_BLOCK, 0, st>>>(                                  \
      (const b128*)x, indices, num_tokens, s->experts_per_token, s->world_size, own,             \
      pieces_of((g.row_vecs + 63) / 64), g.row_vecs, s->num_experts, g.magic, nle_shift, s->rank, \
      (b128*)send_buf, send_meta, send_counts, send_slot)
    if ((g.nle & (g.nle - 1)) == 0) LAUNCH(true);
    else LAUNCH(false);
#undef LAUNCH
    return launch_status();
  }
  if (way == SEND_BLOCK) {
    Geometry b = g;
    b.nvw = block_piece(num_tokens, s->experts_per_token, b.nvw, b.vec16);
    b.wchunks = (b.row_vecs + 64 * b.nvw - 1) / (64 * b.nvw);
    int nle_shift = 0;
    while ((1 << nle_shift) < g.nle) ++nle_shift;
    const bool pow2 = (g.nle & (g.nle - 1)) == 0;
    const int block_grid = (num_tokens + ROWS - 1) / ROWS * b.wchunks;
#define LAUNCH_B(V, NVW, POW2)                                                                \
  dispatch_block_kernel<V, NVW, POW2><<<block_grid, 64 * ROWS, 0, st>>>(                      \
      (const V*)x, indices, num_tokens, s->experts_per_token, s->world_size, b.wchunks,       \
      b.row_vecs, s->num_experts, g.magic, nle_shift, s->rank, (V*)send_buf, send_meta,       \
      send_counts, send_slot)
#define LAUNCH(V, NVW)                            \
  do {                                            \
    if (pow2) LAUNCH_B(V, NVW, true);             \
    else LAUNCH_B(V, NVW, false);                 \
  } while (0)
    MOE_A2A_FOR_WAVE_KERNEL(b, LAUNCH);
#undef LAUNCH
#undef LAUNCH_B
    return launch_status();
  }
  if (way == SEND_FANOUT || way == SEND_FANOUT_WIDE) {
    const int fan = fan_of(S);
    constexpr int WIDE = 2 * BLOCK;  // 512-lane workgroups
    if (way == SEND_FANOUT_WIDE) {
      // Rows of more than 512 vectors: two vectors per lane, so that a row of up to 1024 vectors
      // is one workgroup's and its entries are ranked once, not once per chunk (measured at
      // H = 7168: the whole step 0.4 us shorter; 256 lanes x 4 and 1024 lanes x 1 were slower).
      const int fnv = f.row_vecs > WIDE ? 2 : 1;
      const int wchunks = (f.row_vecs + WIDE * fnv - 1) / (WIDE * fnv);
      const int wgrid = s->world_size + mover_blocks((long long)num_tokens * wchunks);
      int order_bits = 1;  // S <= 1 << order_bits <= 65536, so (W + 1) << order_bits fits an int
      while ((1ll << order_bits) < S) ++order_bits;
      const bool pow2 = (g.nle & (g.nle - 1)) == 0;
      int nle_shift = 0;
      while ((1 << nle_shift) < g.nle) ++nle_shift;
#define LAUNCH_W(V, NV, POW2, FAN)                                                             \
  dispatch_fanout_wide_kernel<V, WIDE, NV, POW2, FAN><<<wgrid, WIDE, 0, st>>>(                 \
      (const V*)x, indices, num_tokens, s->experts_per_token, s->world_size, wchunks,          \
      f.row_vecs, s->num_experts, g.magic, nle_shift, order_bits, s->rank,                     \
      (V*)send_buf, send_meta, send_counts, send_slot)
#define LAUNCH_WF(V, NV, POW2)                       \
  do {                                               \
    if (fan == 2) LAUNCH_W(V, NV, POW2, 2);          \
    else LAUNCH_W(V, NV, POW2, 8);                   \
  } while (0)
#define LAUNCH_WV(V)                                                  \
  do {                                                                \
    if (fnv == 2) { if (pow2) LAUNCH_WF(V, 2, true); else LAUNCH_WF(V, 2, false); } \
    else { if (pow2) LAUNCH_WF(V, 1, true); else LAUNCH_WF(V, 1, false); }          \
  } while (0)
      if (f.vec16) LAUNCH_WV(b128);
      else LAUNCH_WV(uint16_t);
#undef LAUNCH_WV
#undef LAUNCH_WF
#undef LAUNCH_W
      return launch_status();
    }
    const int fgrid = s->world_size + mover_blocks((long long)num_tokens * f.chunks);
#define LAUNCH_F(V, FAN)                                                                       \
  dispatch_fanout_kernel<V, 1, FAN><<<fgrid, BLOCK, 0, st>>>(                                  \
      (const V*)x, indices, num_tokens, s->experts_per_token, s->world_size, f.chunks,         \
      f.row_vecs, g.nle, s->num_experts, g.magic, s->rank, (V*)send_buf, send_meta,            \
      send_counts, send_slot)
#define LAUNCH(V)                         \
  do {                                    \
    if (fan == 2) LAUNCH_F(V, 2);         \
    else LAUNCH_F(V, 8);                  \
  } while (0)
    if (f.vec16) LAUNCH(b128);  // one vector per lane is the only shape this kernel is launched with
    else LAUNCH(uint16_t);
#undef LAUNCH
#undef LAUNCH_F
    return launch_status();
  }
  const int grid = s->world_size + mover_blocks(group_items(S, g));
#define LAUNCH(V, NVW)                                                                         \
  dispatch_send_kernel<V, NVW><<<grid, 64 * ROWS, 0, st>>>(                                    \
      (const V*)x, indices, (int)S, s->experts_per_token, s->world_size, grid - s->world_size, \
      g.wchunks, g.row_vecs, g.nle, s->num_experts, g.magic, s->rank, (V*)send_buf, send_meta, \
      send_counts, send_slot)
  MOE_A2A_FOR_WAVE_KERNEL(g, LAUNCH);
#undef LAUNCH
  return launch_status();
}

int moe_a2a_plan_send(const moe_a2a_shape* s, const int32_t* indices, int32_t num_tokens,
                      int32_t* rank_counts, int32_t* rank_offsets, int32_t* expert_counts,
                      int32_t* dst_slot, int32_t* src_entry, void* stream) {
  if (!shape_ok(s) || num_tokens < 0 || num_tokens > s->max_num_tokens || !rank_counts ||
      !rank_offsets || !expert_counts)
    return MOE_A2A_EINVAL;
  if (s->world_size > PLAN_MAX_RANKS || s->num_experts > PLAN_MAX_EXPERTS) return MOE_A2A_EINVAL;
  const long long S = (long long)num_tokens * s->experts_per_token;
  if (S > INT_MAX / 2) return MOE_A2A_EINVAL;
  if (S > 0 && (!indices || !dst_slot || !src_entry)) return MOE_A2A_EINVAL;
  const Geometry g = geometry(s);
  plan_send_kernel<<<1, PLAN_BLOCK, 0, (hipStream_t)stream>>>(
      indices, (int)S, g.nle, s->num_experts, s->world_size, g.magic, rank_counts, rank_offsets,
      expert_counts, dst_slot, src_entry);
  return launch_status();
}

}  // extern "C"

namespace {

// Stage 2; with `row_position` (capacity_rows ints of workspace) the positions come from a
// planning launch and the movers scan nothing.
int launch_dispatch_recv(const moe_a2a_shape* s, const void* recv_buf, const int32_t* recv_meta,
                         const int32_t* recv_counts, int32_t rows_hint, int32_t capacity_rows,
                         int32_t* expert_num_tokens, void* expert_x, int32_t* expert_meta,
                         int32_t* send_back_plan, int32_t* row_position, void* stream,
                         int32_t compact_rows = 0, int32_t* expert_offsets = nullptr) {
  if (!shape_ok(s) || rows_hint < 0 || capacity_rows < 0 || !recv_counts || !expert_num_tokens ||
      !expert_x || !expert_meta)
    return MOE_A2A_EINVAL;
  if (compact_rows > 0 && !expert_offsets) return MOE_A2A_EINVAL;
  if (!counts_fit(capacity_rows, s->world_size)) return MOE_A2A_EINVAL;
  if (rows_hint > capacity_rows) rows_hint = capacity_rows;
  if (capacity_rows > 0 && (!recv_buf || !recv_meta)) return MOE_A2A_EINVAL;
  if (!all_aligned(2, recv_buf, expert_x)) return MOE_A2A_EALIGN;
  Geometry g = geometry(s, recv_buf, expert_x);
  hipStream_t st = (hipStream_t)stream;
  const bool planned = send_back_plan && plan_supported(s);
  // the stream can hold at most nle * max_recv rows that fit the expert buffers
  if (!items_fit((long long)g.nle * g.max_recv, g.wchunks)) return MOE_A2A_EINVAL;
  // no scan to repeat per piece: a row is split among more waves, as in the planned stage 3
  const long long stream_bytes = (long long)rows_hint * s->hidden_dim * 2;
  const int piece_vecs = g.vec16 ? planned_recv_vecs(stream_bytes, g.row_vecs) : g.nvw, pieces = (g.row_vecs + 64 * piece_vecs - 1) / (64 * piece_vecs);
  // (what a launch numbers are the pieces of the rows that arrive, however many the experts could take; more than it can number are scanned for)
  if (row_position && g.nle <= RPLAN_MAX_EXPERTS && capacity_rows > 0 && items_fit(capacity_rows, pieces)) {
    g.nvw = piece_vecs;
    g.wchunks = pieces;
    const int tiles = (int)std::min<long long>(((long long)rows_hint + RPLAN_BLOCK - 1) / RPLAN_BLOCK + 1, 1 << 16);
    int expert_bits = 0;  // nle <= 1 << expert_bits
    while ((1 << expert_bits) < g.nle) ++expert_bits;
    auto plan_rows = compact_rows > 0 ? plan_recv_kernel<true> : plan_recv_kernel<false>;
    plan_rows<<<tiles, RPLAN_BLOCK, 0, st>>>(recv_meta, recv_counts, s->world_size, rows_hint, capacity_rows, g.nle, g.magic,
                                             expert_bits, row_position);
    const int movers = mover_blocks(((long long)rows_hint * g.wchunks + ROWS - 1) / ROWS);
    const bool past = stream_bytes >= RECV_PAST_BYTES;
#define LAUNCH_C(V, NVW, PLAN, COMPACT, PAST)                                                                  \
  dispatch_recv_planned_kernel<V, NVW, PLAN, COMPACT, THROUGH, PAST><<<g.nle + movers, 64 * ROWS, 0, st>>>(    \
      recv_meta, row_position, recv_counts, (const V*)recv_buf, s->world_size, rows_hint, movers,              \
      pieces_of(g.wchunks), g.row_vecs, g.nle, capacity_rows, g.magic,                                         \
      COMPACT ? compact_rows : g.max_recv, (V*)expert_x, expert_meta, expert_num_tokens, send_back_plan,       \
      expert_offsets)
#define LAUNCH_L(V, NVW, PLAN, PAST)                            \
  do {                                                          \
    if (compact_rows > 0) LAUNCH_C(V, NVW, PLAN, true, PAST);   \
    else LAUNCH_C(V, NVW, PLAN, false, PAST);                   \
  } while (0)
#define LAUNCH_P(V, NVW, PLAN)                        \
  do {                                                \
    if constexpr (sizeof(V) == sizeof(b128)) {        \
      if (past) {                                     \
        LAUNCH_L(V, NVW, PLAN, true);                 \
        break;                                        \
      }                                               \
    }                                                 \
    LAUNCH_L(V, NVW, PLAN, false);                    \
  } while (0)
#define LAUNCH(V, NVW)                     \
  do {                                     \
    if (planned) LAUNCH_P(V, NVW, true);   \
    else LAUNCH_P(V, NVW, false);          \
  } while (0)
    if (!g.vec16) LAUNCH(uint16_t, 16);
    else if (g.nvw == 1) LAUNCH(b128, 1);
    else LAUNCH(b128, 2);
#undef LAUNCH
#undef LAUNCH_P
#undef LAUNCH_L
#undef LAUNCH_C
    return launch_status();
  }
  const RecvFew few = planned ? recv_few(rows_hint, g.row_vecs, g.nvw, g.vec16, compact_rows > 0) : RECV_NOT_FEW;
  if (few != RECV_NOT_FEW) {  // (planned: at most 64 ranks)
    const int few_grid = g.nle + mover_blocks(((long long)rows_hint * g.wchunks + ROWS - 1) / ROWS);
#define LAUNCH_H(V, NVW, KEYS, COMPACT, HOW)                                                 \
  dispatch_recv_few_kernel<V, NVW, KEYS, COMPACT, HOW><<<few_grid, 64 * ROWS, 0, st>>>(      \
      (const V*)recv_buf, recv_meta, recv_counts, s->world_size, rows_hint,                  \
      few_grid - g.nle, g.wchunks, g.row_vecs, g.nle, capacity_rows, g.magic,                \
      compact_rows > 0 ? compact_rows : g.max_recv, expert_num_tokens, (V*)expert_x,         \
      expert_meta, send_back_plan, expert_offsets)
#define LAUNCH_K(V, NVW, KEYS, COMPACT)                                                         \
  do {                                                                                          \
    /* (a lane's vectors of a whole row of 8 MB in 1024: 6 and more) */                         \
    constexpr Store LARGE = NVW == 8 || NVW == 12 || NVW == 16 ? THROUGH_OF<V> : PLAIN;         \
    if (few == RECV_FEW_THROUGH) LAUNCH_H(V, NVW, KEYS, COMPACT, LARGE);                        \
    else LAUNCH_H(V, NVW, KEYS, COMPACT, PLAIN);                                                \
  } while (0)
#define LAUNCH_C(V, NVW, COMPACT)                                       \
  do {                                                                  \
    if (rows_hint <= 64 * 4) LAUNCH_K(V, NVW, 4, COMPACT);              \
    else if (rows_hint <= 64 * 8) LAUNCH_K(V, NVW, 8, COMPACT);         \
    else if (rows_hint <= 64 * 12) LAUNCH_K(V, NVW, 12, COMPACT);       \
    else LAUNCH_K(V, NVW, 16, COMPACT);                                 \
  } while (0)
#define LAUNCH(V, NVW)                                   \
  do {                                                   \
    if (compact_rows > 0) LAUNCH_C(V, NVW, true);        \
    else LAUNCH_C(V, NVW, false);                        \
  } while (0)
    MOE_A2A_FOR_WAVE_KERNEL(g, LAUNCH);
#undef LAUNCH
#undef LAUNCH_C
#undef LAUNCH_K
#undef LAUNCH_H
    return launch_status();
  }
  const int grid = g.nle + mover_blocks(group_items(rows_hint, g));
  const bool through = recv_through(rows_hint, 2ll * s->hidden_dim);  // (Store)
#define LAUNCH_S(V, NVW, PLAN, COMPACT, HOW, SHORT)                                         \
  dispatch_recv_kernel<V, NVW, PLAN, COMPACT, HOW, SHORT><<<grid, 64 * ROWS, 0, st>>>(      \
      (const V*)recv_buf, recv_meta, recv_counts, s->world_size, rows_hint, grid - g.nle,    \
      g.wchunks, g.row_vecs, g.nle, capacity_rows, g.magic,                                  \
      compact_rows > 0 ? compact_rows : g.max_recv,                                          \
      expert_num_tokens, (V*)expert_x, expert_meta, send_back_plan, expert_offsets)
#define LAUNCH_P(V, NVW, PLAN, COMPACT)                                                        \
  do {                                                                                      \
    /* (planned rows of vectors that come here are more than 1024, or 8 MB of 14 per lane,  \
       a workgroup per unit: recv_few) */                                                   \
    constexpr bool VECTORS = PLAN && sizeof(V) == sizeof(b128), SHORT = !COMPACT;           \
    constexpr bool SHORT_FEW = SHORT && !(VECTORS && NVW == 14);                            \
    if (!through) LAUNCH_S(V, NVW, PLAN, COMPACT, (VECTORS ? THROUGH : PLAIN), SHORT);         \
    else if (rows_hint > FEW_ENTRIES) LAUNCH_S(V, NVW, PLAN, COMPACT, THROUGH, SHORT);         \
    else LAUNCH_S(V, NVW, PLAN, COMPACT, THROUGH, SHORT_FEW);                                  \
  } while (0)
#define LAUNCH(V, NVW)                                         \
  do {                                                         \
    if (compact_rows > 0) {                                    \
      if (planned) LAUNCH_P(V, NVW, true, true);               \
      else LAUNCH_P(V, NVW, false, true);                      \
    } else {                                                   \
      if (planned) LAUNCH_P(V, NVW, true, false);              \
      else LAUNCH_P(V, NVW, false, false);                     \
    }                                                          \
  } while (0)
  MOE_A2A_FOR_WAVE_KERNEL(g, LAUNCH);
#undef LAUNCH
#undef LAUNCH_P
#undef LAUNCH_S
  return launch_status();
}

}  // namespace

extern "C" {

int moe_a2a_dispatch_recv(const moe_a2a_shape* s, const void* recv_buf, const int32_t* recv_meta,
                          const int32_t* recv_counts, int32_t rows_hint, int32_t capacity_rows,
                          int32_t* expert_num_tokens, void* expert_x, int32_t* expert_meta,
                          int32_t* send_back_plan, void* stream) {
  return launch_dispatch_recv(s, recv_buf, recv_meta, recv_counts, rows_hint, capacity_rows,
                              expert_num_tokens, expert_x, expert_meta, send_back_plan, nullptr, stream);
}

int moe_a2a_dispatch_recv_long(const moe_a2a_shape* s, const void* recv_buf, const int32_t* recv_meta,
                               const int32_t* recv_counts, int32_t rows_hint, int32_t capacity_rows,
                               int32_t* expert_num_tokens, void* expert_x, int32_t* expert_meta,
                               int32_t* send_back_plan, int32_t* row_position, void* stream) {
  if (!row_position) return MOE_A2A_EINVAL;
  return launch_dispatch_recv(s, recv_buf, recv_meta, recv_counts, rows_hint, capacity_rows,
                              expert_num_tokens, expert_x, expert_meta, send_back_plan, row_position, stream);
}

int moe_a2a_dispatch_recv_static(const moe_a2a_shape* s, const void* recv_buf,
                                 const int32_t* recv_meta, const int32_t* recv_counts,
                                 int32_t rows_hint, int32_t capacity_rows, int32_t* expert_num_tokens,
                                 void* expert_x, int32_t* expert_meta,
                                 const int32_t** send_back_plan, void* stream) {
  if (!shape_ok(s) || !send_back_plan) return MOE_A2A_EINVAL;
  *send_back_plan = nullptr;
  // the plan needs a lane per source rank and per local expert, and 2 * num_experts ints
  if (!plan_supported(s) || s->num_experts > MOE_A2A_STATIC_PLAN_EXPERTS) return MOE_A2A_ESCRATCH;
  int32_t* plan = static_plan_buffer();
  if (!plan) return MOE_A2A_ESCRATCH;
  // every int of the plan that this shape uses is written by the call: nothing to clear
  const int rc = moe_a2a_dispatch_recv(s, recv_buf, recv_meta, recv_counts, rows_hint, capacity_rows,
                                       expert_num_tokens, expert_x, expert_meta, plan, stream);
  if (rc == MOE_A2A_OK) *send_back_plan = plan;
  return rc;
}

}  // extern "C"

namespace {

constexpr int LOADED_MIN_ROWS = 4096;

// Stage 3; compact_rows > 0: the expert buffers hold the experts' rows back to back.
int launch_combine_send(const moe_a2a_shape* s, const void* expert_y, const int32_t* expert_meta,
                        const int32_t* expert_num_tokens, int32_t rows_hint, int32_t capacity_rows,
                        void* send_buf, int32_t* send_meta, int32_t* send_counts,
                        const int32_t* send_back_plan, int32_t compact_rows, void* stream) {
  if (!shape_ok(s) || rows_hint < 0 || capacity_rows < 0 || compact_rows < 0 || !expert_y || !expert_meta ||
      !expert_num_tokens || !send_counts)
    return MOE_A2A_EINVAL;
  if (capacity_rows > 0 && (!send_buf || !send_meta)) return MOE_A2A_EINVAL;
  if (!all_aligned(2, expert_y, send_buf)) return MOE_A2A_EALIGN;
  Geometry g = geometry(s, expert_y, send_buf);
  if (g.nle > MAX_LOCAL_EXPERTS) return MOE_A2A_EINVAL;
  if (compact_rows > 0) {
    if (!counts_fit(compact_rows, g.nle)) return MOE_A2A_EINVAL;  // counts cut to the capacity add up in an int
    g.max_recv = compact_rows;  // no expert has more rows than the buffers hold
  }
  const bool planned = send_back_plan && plan_supported(s);
  // (the planned path has no scan to repeat per piece, so a row can be split among more waves)
  const long long stream_bytes = (long long)rows_hint * s->hidden_dim * 2;
  const bool past = stream_bytes >= EXPERT_PAST_BYTES;
  const int planned_nvw = planned_send_vecs(stream_bytes, g.row_vecs);
  if (planned && g.vec16 && g.nvw > planned_nvw) {
    g.nvw = planned_nvw;
    g.wchunks = (g.row_vecs + 64 * g.nvw - 1) / (64 * g.nvw);
  }
  if (!items_fit(compact_rows > 0 ? (long long)compact_rows : (long long)g.nle * g.max_recv, g.wchunks))
    return MOE_A2A_EINVAL;
  const int grid = s->world_size + mover_blocks(group_items(rows_hint, g));
  hipStream_t st = (hipStream_t)stream;
  // (ArgumentsLoaded) Rows of up to 1 KB, a wave each. us with arguments in registers / loaded: 5056 rows of 512 bytes 3.67 / 3.29, 35928
  // of 512 14.0 / 12.8, 32102 of 1 KB 16.3 / 15.1, its scan 391 / 372; some 3000 the same, fewer are better off with registers.
#define LAUNCH_A(V, NVW, SMALL, PLAN, PAST, ...)                                               \
  do {                                                                                         \
    auto kernel = combine_send_kernel<V, NVW, SMALL, PLAN, PAST __VA_OPT__(,) __VA_ARGS__>;    \
    kernel<<<grid, 64 * ROWS, 0, st>>>(                                                        \
        __VA_OPT__(__VA_ARGS__{},) expert_num_tokens, send_back_plan, expert_meta,             \
        (const V*)expert_y, g.nle, s->world_size, g.wchunks, g.max_recv, compact_rows,         \
        g.row_vecs, capacity_rows, (V*)send_buf, send_meta, send_counts);                      \
  } while (0)
#define LAUNCH_R(V, NVW, SMALL, PLAN, PAST)                                                    \
  do {                                                                                         \
    if constexpr (NVW == 1) {                                                                  \
      if (rows_hint > LOADED_MIN_ROWS) {                                                       \
        LAUNCH_A(V, NVW, SMALL, PLAN, PAST, ArgumentsLoaded);                                  \
        break;                                                                                 \
      }                                                                                        \
    }                                                                                          \
    LAUNCH_A(V, NVW, SMALL, PLAN, PAST);                                                       \
  } while (0)
#define LAUNCH_S(V, NVW, SMALL, PLAN)                                                          \
  do {                                                                                         \
    if constexpr (PLAN && sizeof(V) == sizeof(b128) && NVW <= 8) {                             \
      if (past) {                                                                              \
        LAUNCH_R(V, NVW, SMALL, PLAN, true);                                                   \
        break;                                                                                 \
      }                                                                                        \
    }                                                                                          \
    LAUNCH_R(V, NVW, SMALL, PLAN, false);                                                      \
  } while (0)
#define LAUNCH(V, NVW)                                   \
  do {                                                   \
    if (planned) LAUNCH_S(V, NVW, true, true);           \
    else if (g.nle <= 64) LAUNCH_S(V, NVW, true, false); \
    else LAUNCH_S(V, NVW, false, false);                 \
  } while (0)
  MOE_A2A_FOR_WAVE_KERNEL(g, LAUNCH);
#undef LAUNCH
#undef LAUNCH_S
#undef LAUNCH_R
#undef LAUNCH_A
  return launch_status();
}

// Stage 4; with `entry_row` (num_tokens * K ints of workspace) a launch of its own first maps
// every (token, k) to its arriving row and the workgroups look their rows up instead of scanning.
int launch_combine_recv(const moe_a2a_shape* s, const void* recv_buf, const int32_t* recv_meta,
                        const int32_t* recv_counts, int32_t rows_hint, int32_t capacity_rows,
                        const float* weights, int32_t num_tokens, void* out_tokens,
                        int32_t accumulate, int32_t dtype, int32_t* entry_row, void* stream) {
  if (!shape_ok(s) || num_tokens < 0 || num_tokens > s->max_num_tokens || !recv_counts ||
      rows_hint < 0 || capacity_rows < 0)
    return MOE_A2A_EINVAL;
  if (!counts_fit(capacity_rows, s->world_size)) return MOE_A2A_EINVAL;
  if (rows_hint > capacity_rows) rows_hint = capacity_rows;
  if (dtype != MOE_A2A_F16 && dtype != MOE_A2A_BF16) return MOE_A2A_EINVAL;
  if (num_tokens == 0) return MOE_A2A_OK;
  if (!recv_buf || !recv_meta || !weights || !out_tokens) return MOE_A2A_EINVAL;
  if (!all_aligned(2, recv_buf, out_tokens)) return MOE_A2A_EALIGN;
  const Geometry g = geometry(s, recv_buf, out_tokens);
  // 256 lanes per (token, chunk), one vector column each; rows of at most 512
  // vectors are not split, their lanes take two columns
  // 256 lanes per (token, chunk) with one vector column each for rows up to 256 vectors and two
  // columns beyond. Every workgroup of a token repeats the scan of the arrivals, so fewer, fatter
  // chunks win until the registers of a lane (8 addends x columns in flight) run out.
#ifndef MOE_A2A_COMBINE_NV_WIDE
#define MOE_A2A_COMBINE_NV_WIDE 1
#endif
  const int nv = g.row_vecs > 2 * BLOCK ? MOE_A2A_COMBINE_NV_WIDE : g.row_vecs > BLOCK ? 2 : 1;
  const int chunks = (g.row_vecs + BLOCK * nv - 1) / (BLOCK * nv);
  if (!items_fit(num_tokens, chunks)) return MOE_A2A_EINVAL;
  const int grid = mover_blocks((long long)num_tokens * chunks);
  hipStream_t st = (hipStream_t)stream;
  const int K = s->experts_per_token, W = s->world_size;
  const bool mapped = entry_row != nullptr && capacity_rows > 0;
  if (mapped) {
    const int mgrid = (int)std::min<long long>(((long long)rows_hint + BLOCK - 1) / BLOCK + 1, 1 << 16);
    return_map_kernel<<<mgrid, BLOCK, 0, st>>>(recv_meta, recv_counts, W, rows_hint, capacity_rows,
                                               num_tokens, K, entry_row);
  }
  // Up to eight entries per token a wave has the rows of its piece in one go (combine_recv_mapped_kernel).
  if (mapped && g.vec16 && K <= 8 && capacity_rows < 1 << 28) {
    const bool past = ((long long)rows_hint + num_tokens) * s->hidden_dim * 2 >= COMBINE_PAST_BYTES;
    const int mnv = mapped_vecs(K, g.row_vecs, past), pieces = (g.row_vecs + 64 * mnv - 1) / (64 * mnv);
    if (items_fit(num_tokens, pieces)) {
      const int fgrid = mover_blocks(((long long)num_tokens * pieces + NWAVES - 1) / NWAVES);
#define LAUNCH_P(DT, NV, ADDENDS, PAST)                                                                          \
  combine_recv_mapped_kernel<DT, NV, ADDENDS, PAST><<<fgrid, BLOCK, 0, st>>>(                                    \
      entry_row, recv_counts, weights, recv_meta, W, num_tokens, K, pieces_of(pieces), capacity_rows,            \
      (const b128*)recv_buf, g.row_vecs, accumulate, (b128*)out_tokens)
#define LAUNCH_A(DT, NV, ADDENDS)                          \
  do {                                                     \
    if (past) LAUNCH_P(DT, NV, ADDENDS, true);             \
    else LAUNCH_P(DT, NV, ADDENDS, false);                 \
  } while (0)
#define LAUNCH(DT)                                                                                               \
  do {                                                                                                           \
    if (K <= 2) { if (mnv == 2) LAUNCH_A(DT, 2, 2); else LAUNCH_A(DT, 1, 2); }                                   \
    else if (K <= 4) { if (mnv == 2) LAUNCH_A(DT, 2, 4); else LAUNCH_A(DT, 1, 4); }                              \
    else LAUNCH_A(DT, 1, 8);                                                                                     \
  } while (0)
      if (dtype == MOE_A2A_BF16) LAUNCH(MOE_A2A_BF16);
      else LAUNCH(MOE_A2A_F16);
#undef LAUNCH
#undef LAUNCH_A
#undef LAUNCH_P
      return launch_status();
    }
  }
  // Up to 512 rows every wave looks through the stream by itself (combine_recv_few_kernel); above that the waves share the
  // scan (601 rows of 8 KB: 4.17 us shared, 4.68 by each wave), with code for what there is of it up to 1024.
  if (!mapped && g.vec16 && rows_hint > 0 && rows_hint <= COMBINE_FEW_ROWS && W <= 64 && K <= FEW_MAX_K &&
      (long long)num_tokens * chunks <= 1 << 20) {
    const int few_grid = num_tokens * chunks;
#define LAUNCH_A(DT, NV, KEYS, ADDENDS)                                                         \
  combine_recv_few_kernel<DT, NV, KEYS, ADDENDS><<<few_grid, BLOCK, 0, st>>>(                \
      recv_meta, recv_counts, weights, W, rows_hint, K, chunks, capacity_rows, (const b128*)recv_buf, \
      g.row_vecs, accumulate, (b128*)out_tokens)
#define LAUNCH_K(DT, NV, KEYS)                                                                  \
  do {                                                                                       \
    if (K <= 4) LAUNCH_A(DT, NV, KEYS, 4);                                                   \
    else LAUNCH_A(DT, NV, KEYS, 8);                                                          \
  } while (0)
#define LAUNCH(DT, NV)                                                                       \
  do {                                                                                       \
    if (rows_hint <= 64 * 4) LAUNCH_K(DT, NV, 4);                                            \
    else LAUNCH_K(DT, NV, 8);                                                                \
  } while (0)
    if (dtype == MOE_A2A_BF16) { if (nv == 1) LAUNCH(MOE_A2A_BF16, 1); else LAUNCH(MOE_A2A_BF16, 2); }
    else { if (nv == 1) LAUNCH(MOE_A2A_F16, 1); else LAUNCH(MOE_A2A_F16, 2); }
#undef LAUNCH
#undef LAUNCH_K
#undef LAUNCH_A
    return launch_status();
  }
  // Above one token per unit a workgroup looks through the stream for several at once (combine_block).
  const int block_pieces = (g.row_vecs + 63) / 64;
  const int block_tokens = mapped || !g.vec16 || capacity_rows >= 1 << 28 || block_pieces > INT_MAX / 2 / COMBINE_TOKENS
                               ? 0 : combine_block(num_tokens, rows_hint, K);
  if (block_tokens) {
    const int block_grid = (num_tokens + block_tokens - 1) / block_tokens;
#define LAUNCH_A(DT, ADDENDS)                                                                                    \
  combine_recv_block_kernel<DT, ADDENDS><<<block_grid, COMBINE_BLOCK, 0, st>>>(                                  \
      recv_meta, recv_counts, weights, W, rows_hint, num_tokens, K, block_tokens, pieces_of(block_pieces),       \
      capacity_rows, (const b128*)recv_buf, g.row_vecs, accumulate, (b128*)out_tokens)
#define LAUNCH(DT)                   \
  do {                               \
    if (K <= 2) LAUNCH_A(DT, 2);     \
    else if (K <= 4) LAUNCH_A(DT, 4); \
    else LAUNCH_A(DT, 8);            \
  } while (0)
    if (dtype == MOE_A2A_BF16) LAUNCH(MOE_A2A_BF16);
    else LAUNCH(MOE_A2A_F16);
#undef LAUNCH
#undef LAUNCH_A
    return launch_status();
  }
#define LAUNCH(V, DT, BLK, NV)                                                               \
  do {                                                                                       \
    if (mapped)                                                                              \
      combine_recv_kernel<V, DT, BLK, NV, true, SCAN_UNROLL><<<grid, BLK, 0, st>>>(          \
          recv_meta, recv_counts, weights, W, rows_hint, num_tokens, K, chunks,              \
          capacity_rows, (const V*)recv_buf, g.row_vecs, accumulate, (V*)out_tokens, entry_row); \
    else if (rows_hint <= 4 * BLK)                                                              \
      combine_recv_kernel<V, DT, BLK, NV, false, 4><<<grid, BLK, 0, st>>>(                   \
          recv_meta, recv_counts, weights, W, rows_hint, num_tokens, K, chunks,              \
          capacity_rows, (const V*)recv_buf, g.row_vecs, accumulate, (V*)out_tokens, nullptr); \
    else                                                                                     \
      combine_recv_kernel<V, DT, BLK, NV, false, SCAN_UNROLL><<<grid, BLK, 0, st>>>(         \
          recv_meta, recv_counts, weights, W, rows_hint, num_tokens, K, chunks,              \
          capacity_rows, (const V*)recv_buf, g.row_vecs, accumulate, (V*)out_tokens, nullptr); \
  } while (0)
#define PICK_SHAPE(V, DT)                       \
  do {                                          \
    if (nv == 1) { LAUNCH(V, DT, BLOCK, 1); }   \
    else { LAUNCH(V, DT, BLOCK, 2); }           \
  } while (0)
  if (g.vec16) {
    if (dtype == MOE_A2A_BF16) PICK_SHAPE(b128, MOE_A2A_BF16);
    else PICK_SHAPE(b128, MOE_A2A_F16);
  } else {
    if (dtype == MOE_A2A_BF16) PICK_SHAPE(uint16_t, MOE_A2A_BF16);
    else PICK_SHAPE(uint16_t, MOE_A2A_F16);
  }
#undef PICK_SHAPE
#undef LAUNCH
  return launch_status();
}

}  // namespace

extern "C" {

int moe_a2a_dispatch_recv_compact(const moe_a2a_shape* s, const void* recv_buf, const int32_t* recv_meta,
                                  const int32_t* recv_counts, int32_t rows_hint, int32_t capacity_rows,
                                  int32_t* expert_num_tokens, int32_t* expert_offsets, void* expert_x,
                                  int32_t* expert_meta, int32_t compact_capacity_rows,
                                  int32_t* send_back_plan, void* stream) {
  if (compact_capacity_rows < 1 || !expert_offsets) return MOE_A2A_EINVAL;
  return launch_dispatch_recv(s, recv_buf, recv_meta, recv_counts, rows_hint, capacity_rows, expert_num_tokens,
                              expert_x, expert_meta, send_back_plan, nullptr, stream, compact_capacity_rows,
                              expert_offsets);
}

int moe_a2a_dispatch_recv_compact_long(const moe_a2a_shape* s, const void* recv_buf, const int32_t* recv_meta,
                                       const int32_t* recv_counts, int32_t rows_hint, int32_t capacity_rows,
                                       int32_t* expert_num_tokens, int32_t* expert_offsets, void* expert_x,
                                       int32_t* expert_meta, int32_t compact_capacity_rows,
                                       int32_t* send_back_plan, int32_t* row_position, void* stream) {
  if (compact_capacity_rows < 1 || !expert_offsets || !row_position) return MOE_A2A_EINVAL;
  return launch_dispatch_recv(s, recv_buf, recv_meta, recv_counts, rows_hint, capacity_rows, expert_num_tokens,
                              expert_x, expert_meta, send_back_plan, row_position, stream, compact_capacity_rows,
                              expert_offsets);
}

int moe_a2a_combine_send(const moe_a2a_shape* s, const void* expert_y, const int32_t* expert_meta,
                         const int32_t* expert_num_tokens, int32_t rows_hint,
                         int32_t capacity_rows, void* send_buf, int32_t* send_meta, int32_t* send_counts,
                         const int32_t* send_back_plan, void* stream) {
  return launch_combine_send(s, expert_y, expert_meta, expert_num_tokens, rows_hint, capacity_rows, send_buf,
                             send_meta, send_counts, send_back_plan, 0, stream);
}

int moe_a2a_combine_send_compact(const moe_a2a_shape* s, const void* expert_y, const int32_t* expert_meta,
                                 const int32_t* expert_num_tokens, int32_t rows_hint,
                                 int32_t compact_capacity_rows, int32_t capacity_rows, void* send_buf,
                                 int32_t* send_meta, int32_t* send_counts, const int32_t* send_back_plan,
                                 void* stream) {
  if (compact_capacity_rows < 1) return MOE_A2A_EINVAL;
  return launch_combine_send(s, expert_y, expert_meta, expert_num_tokens, rows_hint, capacity_rows, send_buf,
                             send_meta, send_counts, send_back_plan, compact_capacity_rows, stream);
}

int moe_a2a_combine_recv(const moe_a2a_shape* s, const void* recv_buf, const int32_t* recv_meta,
                         const int32_t* recv_counts, int32_t rows_hint, int32_t capacity_rows,
                         const float* weights, int32_t num_tokens, void* out_tokens,
                         int32_t accumulate, int32_t dtype, void* stream) {
  return launch_combine_recv(s, recv_buf, recv_meta, recv_counts, rows_hint, capacity_rows, weights,
                             num_tokens, out_tokens, accumulate, dtype, nullptr, stream);
}

int moe_a2a_combine_recv_long(const moe_a2a_shape* s, const void* recv_buf, const int32_t* recv_meta,
                              const int32_t* recv_counts, int32_t rows_hint, int32_t capacity_rows,
                              const float* weights, int32_t num_tokens, void* out_tokens,
                              int32_t accumulate, int32_t dtype, int32_t* entry_row, void* stream) {
  if (!entry_row) return MOE_A2A_EINVAL;
  return launch_combine_recv(s, recv_buf, recv_meta, recv_counts, rows_hint, capacity_rows, weights,
                             num_tokens, out_tokens, accumulate, dtype, entry_row, stream);
}

}  // extern "C"

namespace {

// The stand-in expert; compact_rows > 0: the expert buffers hold the experts' rows back to back.
int launch_expert_scale(const moe_a2a_shape* s, const void* expert_x, const int32_t* expert_num_tokens,
                        int32_t rows_hint, int32_t in_dtype, int32_t out_dtype, void* expert_y,
                        int32_t compact_rows, void* stream) {
  if (!shape_ok(s) || rows_hint < 0 || compact_rows < 0 || !expert_x || !expert_num_tokens || !expert_y)
    return MOE_A2A_EINVAL;
  if ((in_dtype != MOE_A2A_F16 && in_dtype != MOE_A2A_BF16) ||
      (out_dtype != MOE_A2A_F16 && out_dtype != MOE_A2A_BF16))
    return MOE_A2A_EINVAL;
  if (!all_aligned(2, expert_x, expert_y)) return MOE_A2A_EALIGN;
  Geometry g = geometry(s, expert_x, expert_y);
  if (g.nle > MAX_LOCAL_EXPERTS) return MOE_A2A_EINVAL;
  if (compact_rows > 0) {
    if (!counts_fit(compact_rows, g.nle)) return MOE_A2A_EINVAL;
    g.max_recv = compact_rows;
  }
  const long long most_rows = compact_rows > 0 ? (long long)compact_rows : (long long)g.nle * g.max_recv;
  if (!items_fit(most_rows, g.chunks)) return MOE_A2A_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  const float scale = (float)(1 + s->rank);
  const bool through = (long long)rows_hint * s->hidden_dim * 2 >= JOB_THROUGH_BYTES;  // (Store)
#ifndef MOE_A2A_SCALE_WAVES
#define MOE_A2A_SCALE_WAVES 1
#endif
  if (MOE_A2A_SCALE_WAVES && g.vec16 && g.nle <= 64) {
    const long long stream_bytes = (long long)rows_hint * s->hidden_dim * 2;
    const bool past = stream_bytes >= EXPERT_PAST_BYTES;
    const int nvw = std::min(g.nvw, past ? 2 : 4);  // 1, 2 or 4 vectors per lane
    const int wchunks = (g.row_vecs + 64 * nvw - 1) / (64 * nvw);
    if (!items_fit(most_rows, wchunks)) return MOE_A2A_EINVAL;
    const int wgrid = mover_blocks(((long long)rows_hint * wchunks + ROWS - 1) / ROWS);
#define LAUNCH_WH(NVW, DI, DO, HOW, PAST)                                                      \
  expert_scale_wave_kernel<NVW, DI, DO, HOW, PAST><<<wgrid, 64 * ROWS, 0, st>>>(                     \
      (const b128*)expert_x, expert_num_tokens, g.nle, g.max_recv, scale, g.row_vecs, wchunks,  \
      (b128*)expert_y, compact_rows)
#define LAUNCH_WT(NVW, DI, DO)                                                                 \
  do {                                                                                         \
    if constexpr (NVW <= 2) {                                                                  \
      if (past) {                                                                              \
        if (stream_bytes >= EXPERT_STREAM_BYTES) LAUNCH_WH(NVW, DI, DO, STREAM, true);         \
        else LAUNCH_WH(NVW, DI, DO, THROUGH, true);                                            \
        break;                                                                                 \
      }                                                                                        \
    }                                                                                          \
    if (through) LAUNCH_WH(NVW, DI, DO, THROUGH, false);                                       \
    else LAUNCH_WH(NVW, DI, DO, PLAIN, false);                                                 \
  } while (0)
#define LAUNCH_W(NVW)                                                                          \
  do {                                                                                         \
    if (in_dtype == MOE_A2A_BF16 && out_dtype == MOE_A2A_BF16)                                 \
      LAUNCH_WT(NVW, MOE_A2A_BF16, MOE_A2A_BF16);                                              \
    else if (in_dtype == MOE_A2A_F16 && out_dtype == MOE_A2A_F16)                              \
      LAUNCH_WT(NVW, MOE_A2A_F16, MOE_A2A_F16);                                                \
    else if (in_dtype == MOE_A2A_F16)                                                          \
      LAUNCH_WT(NVW, MOE_A2A_F16, MOE_A2A_BF16);                                               \
    else                                                                                       \
      LAUNCH_WT(NVW, MOE_A2A_BF16, MOE_A2A_F16);                                               \
  } while (0)
    if (nvw == 1) LAUNCH_W(1);
    else if (nvw == 2) LAUNCH_W(2);
    else LAUNCH_W(4);
#undef LAUNCH_W
#undef LAUNCH_WT
#undef LAUNCH_WH
    return launch_status();
  }
  const int grid = mover_blocks((long long)rows_hint * g.chunks);
#define LAUNCH_H(V, NV, DI, DO, HOW)                                                         \
  expert_scale_kernel<V, NV, DI, DO, HOW><<<grid, BLOCK, 0, st>>>(                           \
      (const V*)expert_x, expert_num_tokens, g.nle, g.max_recv, scale, g.row_vecs, g.chunks, \
      (V*)expert_y, compact_rows)
#define LAUNCH_T(V, NV, DI, DO)                                                              \
  do {                                                                                       \
    if (through) LAUNCH_H(V, NV, DI, DO, THROUGH_OF<V>);                                     \
    else LAUNCH_H(V, NV, DI, DO, PLAIN);                                                     \
  } while (0)
#define LAUNCH(V, NV)                                                                         \
  do {                                                                                        \
    if (in_dtype == MOE_A2A_BF16 && out_dtype == MOE_A2A_BF16)                                \
      LAUNCH_T(V, NV, MOE_A2A_BF16, MOE_A2A_BF16);                                            \
    else if (in_dtype == MOE_A2A_F16 && out_dtype == MOE_A2A_F16)                             \
      LAUNCH_T(V, NV, MOE_A2A_F16, MOE_A2A_F16);                                              \
    else if (in_dtype == MOE_A2A_F16)                                                         \
      LAUNCH_T(V, NV, MOE_A2A_F16, MOE_A2A_BF16);                                             \
    else                                                                                      \
      LAUNCH_T(V, NV, MOE_A2A_BF16, MOE_A2A_F16);                                             \
  } while (0)
  MOE_A2A_FOR_ROW_KERNEL(g, LAUNCH);
#undef LAUNCH
#undef LAUNCH_T
#undef LAUNCH_H
  return launch_status();
}

}  // namespace

extern "C" {

int moe_a2a_expert_scale(const moe_a2a_shape* s, const void* expert_x,
                         const int32_t* expert_num_tokens, int32_t rows_hint, int32_t in_dtype,
                         int32_t out_dtype, void* expert_y, void* stream) {
  return launch_expert_scale(s, expert_x, expert_num_tokens, rows_hint, in_dtype, out_dtype, expert_y, 0, stream);
}

int moe_a2a_expert_scale_compact(const moe_a2a_shape* s, const void* expert_x,
                                 const int32_t* expert_num_tokens, int32_t rows_hint,
                                 int32_t compact_capacity_rows, int32_t in_dtype, int32_t out_dtype,
                                 void* expert_y, void* stream) {
  if (compact_capacity_rows < 1) return MOE_A2A_EINVAL;
  return launch_expert_scale(s, expert_x, expert_num_tokens, rows_hint, in_dtype, out_dtype, expert_y,
                             compact_capacity_rows, stream);
}

#ifndef MOE_A2A_GEMM_ROWS_FOR_128
#define MOE_A2A_GEMM_ROWS_FOR_128 48  // rows per group (mean, from the hint) above which blocks hold 128 tokens
#endif

}  // extern "C"

namespace {

// y[g, :rows(g), :] = x[g, :rows(g), :] @ w[g]^T (+ bias[g]) for `groups` groups of at most max_rows
// rows; rows_of_group null means max_rows rows in every group.
int launch_grouped_gemm(const void* x, const int32_t* rows_of_group, const void* w, const void* bias,
                        void* y, int groups, long long max_rows, long long rows_hint, int N, int K,
                        int dtype, hipStream_t st, int compact = 0) {
  if (dtype != MOE_A2A_F16 && dtype != MOE_A2A_BF16) return MOE_A2A_EINVAL;
  if (N % 32 != 0 || K % 8 != 0) return MOE_A2A_EINVAL;  // whole wave tiles of columns, whole 16-byte vectors
  if (!all_aligned(16, x, w, y) || !all_aligned(8, bias)) return MOE_A2A_EALIGN;
  // per-lane byte offsets inside a block of tokens and inside a wave's 32 weight rows are 32-bit
  if (!tile_rows_in_range(128, K) || max_rows > INT_MAX / 2) return MOE_A2A_EINVAL;
  // Blocks of 32 rows on workgroups of 64 columns where they do better than 64 x 128. (1) Up to eight rows per
  // group: twice as many workgroups share the stream of weights out more evenly. (2) Too few workgroups to keep
  // that stream in flight, at most two per unit: each then looks four steps ahead (streams_far_ahead). Measured, us, blocks
  // of 64 on 128 columns / of 32 on 64, two steps / four (rows per group, groups, N x K): 2.25, 64, 2048 x 1024 52.6
  // / 44.4 / -; the same, 1024 x 2048 44.8 / 44.5 / -; 4, 8, 7168 x 2048 45.6 / 42.2 / -; 2, 64, 512 x 7168 98.1 /
  // 89.4 / 71.6; 1, 4, 2048 x 7168 85.8 / 73.0 / 38.2; 4, 8, 1024 x 2048 21.6 / 18.5 / 14.1; 20, 4, 2048 x 7168 86.3 /
  // - / 39.7; 30, 8, 1024 x 4096 45.1 / - / 23.9; 40, 8, 2048 x 7168 101.5 / - / 58.8; but 24, 64, 1024 x 2048 53.4 /
  // 56.2 / 62.1 and 40, 32, 1024 x 512 11.5 / - / 12.4.
  // (Some of these are ring_gemm_kernel's by now: grouped_ring.)
  const bool counts_fit_32 = (max_rows / 32 + 1) * groups * ((N + 63) / 64) <= INT_MAX / 2;
  const bool far_ahead = counts_fit_32 && streams_far_ahead(rows_hint, groups, N);
  const bool few = counts_fit_32 && (far_ahead || rows_hint <= 8ll * groups);
  const int tj = few ? 1 : rows_hint > (long long)MOE_A2A_GEMM_ROWS_FOR_128 * groups ? 4 : 2;
  // every group can end in a partly filled block of tokens; the kernel strides over what the hint misses
  const long long row_blocks = rows_hint / (tj * 32) + groups;
  // Workgroups of up to 256 columns (8 waves, one workgroup per compute unit) pull an expert's
  // token rows through half as many L1s as workgroups of 128; taken when blocks hold 128 tokens and
  // there are tiles for every unit. One workgroup per unit makes the launch a number of rounds over
  // the units, and half a round at the end leaves half the chip idle (measured: 0.66 of HBM peak at
  // 3.5 rounds, 0.71 at 7.0), so the width is the widest of 8..5 waves whose last round is nearly
  // full, judged from the blocks the row count promises (every group at least one).
#ifndef MOE_A2A_GEMM_WIDE_MIN_TILES
#define MOE_A2A_GEMM_WIDE_MIN_TILES 512
#endif
  constexpr int UNITS = 256;  // compute units of an MI355X
  int gw = few ? 2 : 4;
  if (tj == 4 && row_blocks * ((N + 255) / 256) >= MOE_A2A_GEMM_WIDE_MIN_TILES) {
    const long long blocks = std::max<long long>(groups, (rows_hint + 127) / 128);
    double best = -1.0;
    for (int w = 8; w >= 5; --w) {
      const long long tiles = blocks * ((N + 32 * w - 1) / (32 * w));
      const double rounds = (double)tiles / UNITS, fill = rounds / std::ceil(rounds);
      if (fill >= 0.95) { gw = w; break; }
      if (fill > best) { best = fill; gw = w; }
    }
  }
  const int cols = 32 * gw;
  const int col_tiles = (N + cols - 1) / cols;
  if ((max_rows / 64 + 1) * groups * col_tiles > INT_MAX / 2) return MOE_A2A_EINVAL;
  const int grid = mover_blocks(row_blocks * col_tiles);
  const bool streamed = weights_past_the_cache(groups, rows_hint, N, K);
#define LAUNCH_GS(DT, TJ, GW, D, S)                                                                   \
  expert_gemm_kernel<DT, TJ, GW, D, S><<<grid, 64 * GW, 0, st>>>((const b128*)x, rows_of_group, (const b128*)w, \
                                                                 (const uint16_t*)bias, (uint16_t*)y, groups,  \
                                                                 (int)max_rows, N, K, col_tiles, compact)
#define LAUNCH_G(DT, TJ, GW, D)                       \
  do {                                                \
    if (streamed) LAUNCH_GS(DT, TJ, GW, D, true);     \
    else LAUNCH_GS(DT, TJ, GW, D, false);             \
  } while (0)
#define LAUNCH_GW(DT)                                             \
  do {                                                            \
    if (far_ahead) LAUNCH_G(DT, 1, 2, 4);                         \
    else if (few) LAUNCH_G(DT, 1, 2, 2);                          \
    else if (tj == 2) LAUNCH_G(DT, 2, 4, GEMM_DEPTH);             \
    else if (gw == 8) LAUNCH_G(DT, 4, 8, MOE_A2A_GEMM_DEPTH4);    \
    else if (gw == 7) LAUNCH_G(DT, 4, 7, MOE_A2A_GEMM_DEPTH4);    \
    else if (gw == 6) LAUNCH_G(DT, 4, 6, MOE_A2A_GEMM_DEPTH4);    \
    else if (gw == 5) LAUNCH_G(DT, 4, 5, MOE_A2A_GEMM_DEPTH4);    \
    else LAUNCH_G(DT, 4, 4, MOE_A2A_GEMM_DEPTH4);                 \
  } while (0)
  if (dtype == MOE_A2A_BF16) LAUNCH_GW(MOE_A2A_BF16);
  else LAUNCH_GW(MOE_A2A_F16);
#undef LAUNCH_GW
#undef LAUNCH_G
#undef LAUNCH_GS
  return launch_status();
}

constexpr int MOE_A2A_NOT_DENSE = 1;  // (internal) the shape is left to the next kernel

constexpr size_t local_plan_lds_bytes(int experts) { return (size_t)(2 + LPLAN_WAVES) * experts * sizeof(int); }
constexpr size_t dense_lds_bytes(int BM, int BN) { return 2 * (size_t)(BM + BN) * 8 * sizeof(b128); }
constexpr size_t skinny_lds_bytes(int tj, int waves) { return (size_t)waves * (32 + 32 * tj) * 8 * sizeof(b128); }

// The tile buffers can be more LDS than a kernel gets by default: allowed once per GPU, for every
// tile and type at once, so that only the first dense call on a GPU touches kernel attributes.
int allow_large_lds() {
  static bool allowed[MAX_GPUS] = {};
  int gpu = -1;
  if (hipGetDevice(&gpu) != hipSuccess || gpu < 0 || gpu >= MAX_GPUS) return MOE_A2A_ELAUNCH;
  std::lock_guard<std::mutex> lock(static_plan_mutex);
  if (allowed[gpu]) return MOE_A2A_OK;
  bool ok = true;
  auto allow = [&](const void* kernel, size_t bytes) {
    ok = ok && hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
  };
  auto allow_grouped = [&](auto dtype, auto streamed) {
    constexpr int DT = decltype(dtype)::value;
    constexpr bool S = decltype(streamed)::value;
    allow((const void*)phased_gemm_kernel<DT, 10, 4, 2, 5, false, true, S>, phased_lds_bytes(10, 4, 2, 5));
    allow((const void*)phased_gemm_kernel<DT, 8, 4, 2, 6, false, true, S>, phased_lds_bytes(8, 4, 2, 6));
    allow((const void*)phased_gemm_kernel<DT, 6, 4, 2, 6, false, true, S>, phased_lds_bytes(6, 4, 2, 6));
    allow((const void*)dense_gemm_kernel<DT, 2, 2, 2, 2, true, S>, dense_lds_bytes(128, 128));
    allow((const void*)ring_gemm_kernel<DT, 1, 1, 8, S>, ring_lds_bytes(1, 1, 8));
    allow((const void*)ring_gemm_kernel<DT, 1, 2, 6, S>, ring_lds_bytes(1, 2, 6));
    allow((const void*)sliced_gemm_kernel<DT, Slices64x64, true, S>, Slices64x64::LDS_BYTES);
    allow((const void*)sliced_gemm_kernel<DT, Slices64x128, true, S>, Slices64x128::LDS_BYTES);
    allow((const void*)sliced_gemm_kernel<DT, Slices128x128, true, S>, Slices128x128::LDS_BYTES);
    allow((const void*)sliced_gemm_kernel<DT, Slices192x128, true, S>, Slices192x128::LDS_BYTES);
    if constexpr (!S) {
      allow((const void*)sliced_gemm_kernel<DT, Slices64x32, false, false>, Slices64x32::LDS_BYTES);
      allow((const void*)sliced_gemm_kernel<DT, Slices32x64, false, false>, Slices32x64::LDS_BYTES);
      allow((const void*)sliced_gemm_kernel<DT, Slices64x64, false, false>, Slices64x64::LDS_BYTES);
      allow((const void*)sliced_gemm_kernel<DT, Slices64x128, false, false>, Slices64x128::LDS_BYTES);
    }
  };
  allow((const void*)phased_gemm_kernel<MOE_A2A_BF16, 8, 4, 3, 4, false, false>, phased_lds_bytes(8, 4, 3, 4));
  allow((const void*)phased_gemm_kernel<MOE_A2A_F16, 8, 4, 3, 4, false, false>, phased_lds_bytes(8, 4, 3, 4));
  allow((const void*)phased_gemm_kernel<MOE_A2A_BF16, 8, 4, 3, 4, true, false>, phased_lds_bytes(8, 4, 3, 4));
  allow((const void*)phased_gemm_kernel<MOE_A2A_F16, 8, 4, 3, 4, true, false>, phased_lds_bytes(8, 4, 3, 4));
  allow((const void*)phased_gemm_kernel<MOE_A2A_BF16, 4, 2, 3, 4, false, false>, phased_lds_bytes(4, 2, 3, 4));
  allow((const void*)phased_gemm_kernel<MOE_A2A_BF16, 6, 2, 3, 4, false, false>, phased_lds_bytes(6, 2, 3, 4));
  allow((const void*)phased_gemm_kernel<MOE_A2A_F16, 4, 2, 3, 4, false, false>, phased_lds_bytes(4, 2, 3, 4));
  allow((const void*)phased_gemm_kernel<MOE_A2A_F16, 6, 2, 3, 4, false, false>, phased_lds_bytes(6, 2, 3, 4));
  allow((const void*)dense_gemm_kernel<MOE_A2A_BF16, 2, 2, 2, 2, false>, dense_lds_bytes(128, 128));
  allow((const void*)dense_gemm_kernel<MOE_A2A_F16, 2, 2, 2, 2, false>, dense_lds_bytes(128, 128));
  allow_grouped(std::integral_constant<int, MOE_A2A_BF16>{}, std::false_type{});
  allow_grouped(std::integral_constant<int, MOE_A2A_BF16>{}, std::true_type{});
  allow_grouped(std::integral_constant<int, MOE_A2A_F16>{}, std::false_type{});
  allow_grouped(std::integral_constant<int, MOE_A2A_F16>{}, std::true_type{});
  allow((const void*)skinny_gemm_kernel<MOE_A2A_BF16, 2, 8, true>, skinny_lds_bytes(2, 8));
  allow((const void*)skinny_gemm_kernel<MOE_A2A_BF16, 2, 8, false>, skinny_lds_bytes(2, 8));
  allow((const void*)skinny_gemm_kernel<MOE_A2A_F16, 2, 8, true>, skinny_lds_bytes(2, 8));
  allow((const void*)skinny_gemm_kernel<MOE_A2A_F16, 2, 8, false>, skinny_lds_bytes(2, 8));
  allow((const void*)local_plan_kernel<1>, local_plan_lds_bytes(LOCAL_MAX_EXPERTS));
  allow((const void*)local_plan_kernel<LOCAL_FEW_RANKS>, local_plan_lds_bytes(LOCAL_MAX_EXPERTS));
  allow((const void*)local_plan_kernel<LOCAL_MAX_RANKS>, local_plan_lds_bytes(LOCAL_MAX_EXPERTS));
  if (!ok) return MOE_A2A_ELAUNCH;
  allowed[gpu] = true;
  return MOE_A2A_OK;
}

// A product on ring_gemm_kernel, in the tiles that grouped_ring has chosen. MOE_A2A_NOT_DENSE where it has too many.
int launch_grouped_ring(const void* x, const int32_t* rows_of_group, const void* w, const void* bias, void* y, int groups,
                        long long max_rows, long long rows_hint, int N, int K, int dtype, hipStream_t st, int compact, RingTile way) {
  const int BM = 32, BN = way == RING_32x32 ? 32 : 64;
  const long long tiles_n = (N + BN - 1) / BN;
  // Every group that has a row can end in a partly filled row tile; the kernel strides over what the hint misses. (Workgroups
  // without a tile are not free with so much LDS: 6 rows of 95 groups, 1152 x 192 9.7 us with one for every group.)
  const long long pairs = (rows_hint / BM + (rows_hint > 0 ? std::min<long long>(groups, rows_hint) : groups)) * tiles_n;
  if ((max_rows / BM + 1) * groups * tiles_n > INT_MAX / 2) return MOE_A2A_NOT_DENSE;
  const int grid = mover_blocks((pairs + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
  if (const int rc = allow_large_lds()) return rc;
  const bool streamed = weights_past_the_cache(groups, rows_hint, N, K) && rows_hint <= (long long)groups * BM;
  auto launch = [&](auto dtype_const, auto streamed_const) {
    constexpr int DT = decltype(dtype_const)::value;
    constexpr bool S = decltype(streamed_const)::value;
    auto start = [&](auto kernel, int depth) {
      kernel<<<grid, 256, ring_lds_bytes(BM / 32, BN / 32, depth), st>>>((const b128*)x, (const b128*)w, rows_of_group, (const uint16_t*)bias,
                                                                         (uint16_t*)y, N, K, (int)tiles_n, groups, (int)max_rows, compact);
    };
    if (way == RING_32x32) start(ring_gemm_kernel<DT, 1, 1, 8, S>, 8);
    else start(ring_gemm_kernel<DT, 1, 2, 6, S>, 6);
  };
  auto launch_of = [&](auto dtype_const) {
    if (streamed) launch(dtype_const, std::true_type{});
    else launch(dtype_const, std::false_type{});
  };
  if (dtype == MOE_A2A_BF16) launch_of(std::integral_constant<int, MOE_A2A_BF16>{});
  else launch_of(std::integral_constant<int, MOE_A2A_F16>{});
  return launch_status();
}

// A product on sliced_gemm_kernel, in the tiles that grouped_slices or linear_slices has chosen. MOE_A2A_NOT_DENSE where it has too many.
int launch_slices(const void* x, const int32_t* rows_of_group, const void* w, const void* bias, void* y, int groups, long long max_rows,
                  long long rows_hint, int N, int K, int dtype, hipStream_t st, int compact, SlicedTile way) {
  const int BM = sliced_rows(way), BN = sliced_cols(way);
  const long long tiles_m = (max_rows + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  if (tiles_m * groups * tiles_n > INT_MAX / 2) return MOE_A2A_NOT_DENSE;
  // (GROUPED: every group that has a row can end in a partly filled row tile; the kernel strides over what the hint misses)
  const long long pairs = rows_of_group ? (rows_hint / BM + std::min<long long>(groups, std::max(rows_hint, 1ll))) * tiles_n : tiles_m * tiles_n;
  const int grid = mover_blocks(pairs);
  if (const int rc = allow_large_lds()) return rc;
  const bool streamed = rows_of_group && weights_past_the_cache(groups, rows_hint, N, K) && rows_hint <= (long long)groups * BM;
  auto start = [&](auto dtype_const, auto tile, auto grouped, auto streamed_const) {
    using TILE = decltype(tile);
    sliced_gemm_kernel<decltype(dtype_const)::value, TILE, decltype(grouped)::value, decltype(streamed_const)::value>
        <<<grid, TILE::LANES, TILE::LDS_BYTES, st>>>((const b128*)x, (const b128*)w, (const uint16_t*)bias, (uint16_t*)y, (int)max_rows, N, K,
                                                     (int)tiles_m, (int)tiles_n, rows_of_group, groups, (int)max_rows, compact);
  };
  auto launch_of = [&](auto dtype_const) {
    auto grouped = [&](auto tile) {
      if (streamed) start(dtype_const, tile, std::true_type{}, std::true_type{});
      else start(dtype_const, tile, std::true_type{}, std::false_type{});
    };
    auto plain = [&](auto tile) { start(dtype_const, tile, std::false_type{}, std::false_type{}); };
    if (rows_of_group) {
      if (way == SLICES_64x64) grouped(Slices64x64{});
      else if (way == SLICES_64x128) grouped(Slices64x128{});
      else if (way == SLICES_128x128) grouped(Slices128x128{});
      else grouped(Slices192x128{});
    } else {
      if (way == SLICES_64x32) plain(Slices64x32{});
      else if (way == SLICES_32x64) plain(Slices32x64{});
      else if (way == SLICES_64x64) plain(Slices64x64{});
      else plain(Slices64x128{});
    }
  };
  if (dtype == MOE_A2A_BF16) launch_of(std::integral_constant<int, MOE_A2A_BF16>{});
  else launch_of(std::integral_constant<int, MOE_A2A_F16>{});
  return launch_status();
}

// A plain product on tiles that workgroups own whole, as linear_way has chosen.
int launch_linear_tiles(const void* a, const void* b, const void* bias, void* c, int M, int N, int K, int dtype,
                        LinearWay way, hipStream_t st) {
  const int BM = way == PHASED_256 ? 256 : way == PHASED_192 ? 192 : 128;
  const int BN = way == PHASED_256 ? 256 : 128;
  const long long tiles_m = ((long long)M + BM - 1) / BM, tiles_n = ((long long)N + BN - 1) / BN;
  if (tiles_m * tiles_n > INT_MAX / 2) return MOE_A2A_NOT_DENSE;
  const int grid = (int)(tiles_m * tiles_n);
  const int phased_grid = way == PHASED_256 ? std::min(grid, 256) : grid;  // (one per unit, which strides over its tiles)
  if (const int rc = allow_large_lds()) return rc;
#define LAUNCH_P(DT, TM, TN, AHEAD)                                                              \
  phased_gemm_kernel<DT, TM, TN, 3, 4, AHEAD, false><<<phased_grid, 512, phased_lds_bytes(TM, TN, 3, 4), st>>>( \
      (const b128*)a, (const b128*)b, (const uint16_t*)bias, (uint16_t*)c, M, N, K, (int)tiles_m, (int)tiles_n, \
      nullptr, 0, 0, 0)
#define LAUNCH_D(DT, TM, TN, LDS)                                                                \
  dense_gemm_kernel<DT, 2, 2, TM, TN, false><<<grid, 256, LDS, st>>>(                            \
      (const b128*)a, (const b128*)b, (const uint16_t*)bias, (uint16_t*)c, M, N, K, (int)tiles_m, (int)tiles_n, \
      nullptr, 0, 0, 0)
#define LAUNCH_DT(DT)                                                                            \
  do {                                                                                           \
    if (way == PHASED_256 && K * 2 % 128 != 0) LAUNCH_P(DT, 8, 4, true);                         \
    else if (way == PHASED_256) LAUNCH_P(DT, 8, 4, false);                                       \
    else if (way == PHASED_192) LAUNCH_P(DT, 6, 2, false);                                       \
    else if (way == PHASED_128) LAUNCH_P(DT, 4, 2, false);                                       \
    else LAUNCH_D(DT, 2, 2, dense_lds_bytes(128, 128));                                          \
  } while (0)
  if (dtype == MOE_A2A_BF16) LAUNCH_DT(MOE_A2A_BF16);
  else LAUNCH_DT(MOE_A2A_F16);
#undef LAUNCH_DT
#undef LAUNCH_D
#undef LAUNCH_P
  return launch_status();
}

#ifndef MOE_A2A_GROUPED_DENSE_MIN_ROWS
#define MOE_A2A_GROUPED_DENSE_MIN_ROWS 56  // rows per group (from the caller's row count) from which tiles are used
#endif
// The grouped product where its tiles are few (launch_grouped_ring), and from some dozens of rows per group: the dense kernels' tiles (each weight row read once per 64
// to 320 rows, operands shared by the workgroup's waves through LDS) do as well as or better than the kernel that is
// built around streaming the weights. MOE_A2A_NOT_DENSE otherwise.
int launch_grouped_dense(const void* x, const int32_t* rows_of_group, const void* w, const void* bias, void* y,
                         int groups, long long max_rows, long long rows_hint, int N, int K, int dtype,
                         hipStream_t st, int compact = 0) {
  if (dtype != MOE_A2A_F16 && dtype != MOE_A2A_BF16) return MOE_A2A_EINVAL;
  if (N % 32 != 0 || K % 8 != 0) return MOE_A2A_EINVAL;
  if (!all_aligned(16, x, w, y) || !all_aligned(8, bias)) return MOE_A2A_EALIGN;
  if (max_rows > INT_MAX / 2) return MOE_A2A_NOT_DENSE;
  const RingTile ring = grouped_ring(rows_hint, groups, N, K);
  if (ring == RING_32x32 || ring == RING_32x64) {
    const int rc = launch_grouped_ring(x, rows_of_group, w, bias, y, groups, max_rows, rows_hint, N, K, dtype, st, compact, ring);
    if (rc != MOE_A2A_NOT_DENSE) return rc;
  }
  const bool tiled = rows_hint >= (long long)MOE_A2A_GROUPED_DENSE_MIN_ROWS * groups;
  const int bands = tiled && !ring ? grouped_tile_bands(rows_hint, groups, N, K) : 0;
  if (const SlicedTile slices = grouped_slices(ring, bands, rows_hint, groups, N)) {
    const int rc = launch_slices(x, rows_of_group, w, bias, y, groups, max_rows, rows_hint, N, K, dtype, st, compact, slices);
    if (rc != MOE_A2A_NOT_DENSE) return rc;
  }
  if (!bands || bands == 2) return MOE_A2A_NOT_DENSE;
  const int BM = bands * 32, BN = bands <= 4 ? 128 : 256;
  const long long tiles_n = (N + BN - 1) / BN;
  // every group can end in a partly filled row tile; the kernel strides over what the hint misses
  const long long pairs = (rows_hint / BM + groups) * tiles_n;
  if ((max_rows / BM + 1) * groups * tiles_n > INT_MAX / 2) return MOE_A2A_NOT_DENSE;
  const int grid = mover_blocks((pairs + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
  if (const int rc = allow_large_lds()) return rc;
  // (tiles of one row of tiles per group ask for its weights once; neighbours that ask for them too find them in L2)
  const bool streamed = weights_past_the_cache(groups, rows_hint, N, K) && rows_hint <= (long long)groups * BM;
  auto launch = [&](auto dtype_const, auto streamed_const) {
    constexpr int DT = decltype(dtype_const)::value;
    constexpr bool S = decltype(streamed_const)::value;
    auto start = [&](auto kernel, int lanes, size_t lds_bytes) {
      kernel<<<grid, lanes, lds_bytes, st>>>((const b128*)x, (const b128*)w, (const uint16_t*)bias, (uint16_t*)y, 0, N, K,
                                             0, (int)tiles_n, rows_of_group, groups, (int)max_rows, compact);
    };
    auto phased = [&](auto kernel, size_t lds_bytes) { start(kernel, 512, lds_bytes); };
    auto dense = [&](auto kernel, size_t lds_bytes) { start(kernel, 256, lds_bytes); };
    if (bands == 10) phased(phased_gemm_kernel<DT, 10, 4, 2, 5, false, true, S>, phased_lds_bytes(10, 4, 2, 5));
    else if (bands == 8) phased(phased_gemm_kernel<DT, 8, 4, 2, 6, false, true, S>, phased_lds_bytes(8, 4, 2, 6));
    else if (bands == 6) phased(phased_gemm_kernel<DT, 6, 4, 2, 6, false, true, S>, phased_lds_bytes(6, 4, 2, 6));
    else dense(dense_gemm_kernel<DT, 2, 2, 2, 2, true, S>, dense_lds_bytes(128, 128));
  };
  auto launch_of = [&](auto dtype_const) {
    if (streamed) launch(dtype_const, std::true_type{});
    else launch(dtype_const, std::false_type{});
  };
  if (dtype == MOE_A2A_BF16) launch_of(std::integral_constant<int, MOE_A2A_BF16>{});
  else launch_of(std::integral_constant<int, MOE_A2A_F16>{});
  return launch_status();
}

// A plain product on workgroups of 32 columns whose waves split K among them, tj x 32 rows each.
int launch_linear_split(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, int dtype, int tj,
                        hipStream_t st) {
  const int steps = (K + GEMM_KSTEP - 1) / GEMM_KSTEP;
  const int row_units = (M + 32 * tj - 1) / (32 * tj), grid = N / 32 * row_units;
  const uint32_t row_magic = row_units > 1 ? (uint32_t)(((1ull << 32) + row_units - 1) / row_units) : 0;
  // eight waves keep more of the stream in flight (measured 10 to 13 % less time from 28 steps
  // on); with few steps the four extra partial sums cost more than that
  const int waves = steps >= 24 ? 8 : 4;
  if (const int rc = allow_large_lds()) return rc;
#define LAUNCH_KA(DT, TJ, KW, APART)                                                      \
  skinny_gemm_kernel<DT, TJ, KW, APART><<<grid, 64 * KW, skinny_lds_bytes(TJ, KW), st>>>( \
      (const b128*)x, (const b128*)w, (const uint16_t*)bias, (uint16_t*)y, M, N, K, row_units, row_magic)
#define LAUNCH_K(DT, TJ, KW)                               \
  do {                                                     \
    if (K % 2048 == 0) LAUNCH_KA(DT, TJ, KW, true);        \
    else LAUNCH_KA(DT, TJ, KW, false);                     \
  } while (0)
#define LAUNCH_KW(DT)                                      \
  do {                                                     \
    if (waves == 8 && tj == 2) LAUNCH_K(DT, 2, 8);         \
    else if (waves == 8) LAUNCH_K(DT, 1, 8);               \
    else if (tj == 2) LAUNCH_K(DT, 2, 4);                  \
    else LAUNCH_K(DT, 1, 4);                               \
  } while (0)
  if (dtype == MOE_A2A_BF16) LAUNCH_KW(MOE_A2A_BF16);
  else LAUNCH_KW(MOE_A2A_F16);
#undef LAUNCH_KW
#undef LAUNCH_K
#undef LAUNCH_KA
  return launch_status();
}

int launch_linear(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, int dtype, hipStream_t st) {
  if (dtype != MOE_A2A_F16 && dtype != MOE_A2A_BF16) return MOE_A2A_EINVAL;
  if (N % 32 != 0 || K % 8 != 0) return MOE_A2A_EINVAL;
  if (!all_aligned(16, x, w, y) || !all_aligned(8, bias)) return MOE_A2A_EALIGN;
  const RingTile ring = linear_ring(M, N, K);
  const LinearWay way = ring ? STREAM_WEIGHTS : linear_way(M, N, K);
  if (const SlicedTile slices = linear_slices(ring, way, M, N, K)) {
    const int rc = launch_slices(x, nullptr, w, bias, y, 1, M, M, N, K, dtype, st, 0, slices);
    if (rc != MOE_A2A_NOT_DENSE) return rc;
  }
  int rc = MOE_A2A_NOT_DENSE;
  if (way == SPLIT_32 || way == SPLIT_64) rc = launch_linear_split(x, w, bias, y, M, N, K, dtype, way == SPLIT_32 ? 1 : 2, st);
  else if (way != STREAM_WEIGHTS && way != TILES_64x128) rc = launch_linear_tiles(x, w, bias, y, M, N, K, dtype, way, st);
  if (rc != MOE_A2A_NOT_DENSE) return rc;
  return launch_grouped_gemm(x, nullptr, w, bias, y, 1, M, M, N, K, dtype, st);
}

}  // namespace

extern "C" {

int moe_a2a_expert_gemm(const moe_a2a_shape* s, const void* expert_x,
                        const int32_t* expert_num_tokens, int32_t rows_hint, const void* weights,
                        const void* bias, int32_t in_dim, int32_t out_dim, int32_t dtype,
                        void* expert_y, void* stream) {
  if (!shape_ok(s) || rows_hint < 0 || in_dim < 1 || out_dim < 1 || !expert_x || !expert_num_tokens ||
      !weights || !expert_y)
    return MOE_A2A_EINVAL;
  const int nle = s->num_experts / s->world_size;
  const long long max_recv = (long long)s->max_num_tokens * s->world_size;
  const int dense = launch_grouped_dense(expert_x, expert_num_tokens, weights, bias, expert_y, nle, max_recv,
                                         rows_hint, out_dim, in_dim, dtype, (hipStream_t)stream);
  if (dense != MOE_A2A_NOT_DENSE) return dense;
  return launch_grouped_gemm(expert_x, expert_num_tokens, weights, bias, expert_y, nle, max_recv, rows_hint,
                             out_dim, in_dim, dtype, (hipStream_t)stream);
}

int moe_a2a_expert_gemm_compact(const moe_a2a_shape* s, const void* expert_x,
                                const int32_t* expert_num_tokens, int32_t rows_hint,
                                int32_t compact_capacity_rows, const void* weights, const void* bias,
                                int32_t in_dim, int32_t out_dim, int32_t dtype, void* expert_y,
                                void* stream) {
  if (!shape_ok(s) || rows_hint < 0 || compact_capacity_rows < 1 || in_dim < 1 || out_dim < 1 || !expert_x ||
      !expert_num_tokens || !weights || !expert_y)
    return MOE_A2A_EINVAL;
  const int nle = s->num_experts / s->world_size;
  if (!counts_fit(compact_capacity_rows, nle)) return MOE_A2A_EINVAL;
  // (every count is cut to the rows the buffers hold; counts that dispatch_recv_compact wrote add up to at most that)
  const int dense = launch_grouped_dense(expert_x, expert_num_tokens, weights, bias, expert_y, nle,
                                         compact_capacity_rows, rows_hint, out_dim, in_dim, dtype,
                                         (hipStream_t)stream, 1);
  if (dense != MOE_A2A_NOT_DENSE) return dense;
  return launch_grouped_gemm(expert_x, expert_num_tokens, weights, bias, expert_y, nle, compact_capacity_rows,
                             rows_hint, out_dim, in_dim, dtype, (hipStream_t)stream, 1);
}

int moe_a2a_linear(const void* input, const void* weight, const void* bias, int32_t m, int32_t n,
                   int32_t k, int32_t dtype, void* output, void* stream) {
  if (m < 0 || n < 1 || k < 1 || !weight || (m > 0 && (!input || !output))) return MOE_A2A_EINVAL;
  if (m == 0) return MOE_A2A_OK;
  return launch_linear(input, weight, bias, output, m, n, k, dtype, (hipStream_t)stream);
}

int moe_a2a_exchange_local(int32_t world_size, int32_t hidden_dim, const void* send_buf,
                           const int32_t* send_meta, const int32_t* send_counts, int32_t dst_rank,
                           void* recv_buf, int32_t* recv_meta, const int32_t* recv_counts,
                           int32_t src_rank, int32_t rows_hint, int32_t send_capacity_rows,
                           int32_t recv_capacity_rows, void* stream) {
  if (world_size < 1 || hidden_dim < 1 || dst_rank < 0 || dst_rank >= world_size ||
      src_rank < 0 || src_rank >= world_size || rows_hint < 0 || send_capacity_rows < 0 ||
      recv_capacity_rows < 0 || !send_counts || !recv_counts ||
      !counts_fit(send_capacity_rows, world_size) || !counts_fit(recv_capacity_rows, world_size))
    return MOE_A2A_EINVAL;
  if (send_capacity_rows == 0 || recv_capacity_rows == 0) return MOE_A2A_OK;  // nothing can move
  if (!send_buf || !send_meta || !recv_buf || !recv_meta) return MOE_A2A_EINVAL;
  if (!all_aligned(2, send_buf, recv_buf)) return MOE_A2A_EALIGN;
  Geometry g{};
  row_geometry(g, hidden_dim, all_aligned(16, send_buf, recv_buf));
  if (!items_fit(rows_hint, g.chunks)) return MOE_A2A_EINVAL;
  const int grid = mover_blocks((long long)rows_hint * g.chunks);
  const bool through = (long long)rows_hint * hidden_dim * 2 >= EXCHANGE_THROUGH_BYTES;  // (Store)
  hipStream_t st = (hipStream_t)stream;
#define LAUNCH_H(V, NV, HOW)                                                                  \
  exchange_local_kernel<V, NV, HOW><<<grid, BLOCK, 0, st>>>(                                  \
      ArgumentsLoaded{}, (const V*)send_buf, send_meta, send_counts, dst_rank, (V*)recv_buf, recv_meta,          \
      recv_counts, src_rank, g.row_vecs, g.chunks, send_capacity_rows, recv_capacity_rows)
#define LAUNCH(V, NV)                                    \
  do {                                                   \
    if (through) LAUNCH_H(V, NV, THROUGH_OF<V>);         \
    else LAUNCH_H(V, NV, PLAIN);                         \
  } while (0)
  MOE_A2A_FOR_ROW_KERNEL(g, LAUNCH);
#undef LAUNCH
#undef LAUNCH_H
  return launch_status();
}

int moe_a2a_exchange_gather_local(int32_t world_size, int32_t hidden_dim, const void* const* send_bufs,
                                  const int32_t* const* send_metas, const int32_t* const* send_counts,
                                  int32_t dst_rank, void* recv_buf, int32_t* recv_meta,
                                  int32_t* recv_counts, int32_t rows_hint, int32_t send_capacity_rows,
                                  int32_t recv_capacity_rows, void* stream) {
  if (world_size < 1 || world_size > GATHER_MAX_RANKS || hidden_dim < 1 || dst_rank < 0 ||
      dst_rank >= world_size || rows_hint < 0 || send_capacity_rows < 0 || recv_capacity_rows < 0 ||
      !send_bufs || !send_metas || !send_counts || !recv_counts ||
      !counts_fit(send_capacity_rows, world_size) || !counts_fit(recv_capacity_rows, world_size))
    return MOE_A2A_EINVAL;
  GatherSources src{};
  bool all16 = aligned(recv_buf, 16);
  for (int r = 0; r < world_size; ++r) {
    if (!send_counts[r]) return MOE_A2A_EINVAL;
    if (send_capacity_rows > 0 && (!send_bufs[r] || !send_metas[r])) return MOE_A2A_EINVAL;
    if (!aligned(send_bufs[r], 2)) return MOE_A2A_EALIGN;
    all16 = all16 && aligned(send_bufs[r], 16);
    src.buf[r] = send_bufs[r];
    src.meta[r] = send_metas[r];
    src.counts[r] = send_counts[r];
  }
  if (send_capacity_rows > 0 && recv_capacity_rows > 0 && (!recv_buf || !recv_meta)) return MOE_A2A_EINVAL;
  if (!aligned(recv_buf, 2)) return MOE_A2A_EALIGN;
  Geometry g{};
  row_geometry(g, hidden_dim, all16);
  if (!items_fit(rows_hint, g.chunks)) return MOE_A2A_EINVAL;
  // (the launch also delivers the counts, so it is made even when no row can move)
  const dim3 grid(std::min(mover_blocks((long long)rows_hint * g.chunks), 1 << 16), world_size);
  const bool through = (double)rows_hint * world_size * hidden_dim * 2 >= EXCHANGE_THROUGH_BYTES;  // (Store)
  hipStream_t st = (hipStream_t)stream;
#define LAUNCH_H(V, NV, HOW)                                                                   \
  exchange_gather_kernel<V, NV, HOW><<<grid, BLOCK, 0, st>>>(src, world_size, dst_rank, (V*)recv_buf, \
                                                             recv_meta, recv_counts, g.row_vecs, g.chunks, \
                                                             send_capacity_rows, recv_capacity_rows)
#define LAUNCH(V, NV)                                    \
  do {                                                   \
    if (through) LAUNCH_H(V, NV, THROUGH_OF<V>);         \
    else LAUNCH_H(V, NV, PLAIN);                         \
  } while (0)
  MOE_A2A_FOR_ROW_KERNEL(g, LAUNCH);
#undef LAUNCH
#undef LAUNCH_H
  return launch_status();
}


}  // extern "C"

namespace {

bool local_supported(const moe_a2a_shape* s) {
  return s->world_size <= LOCAL_MAX_RANKS && s->num_experts <= LOCAL_MAX_EXPERTS && s->experts_per_token <= LOCAL_MAX_K;
}

}  // namespace

extern "C" {

int moe_a2a_local_dispatch(const moe_a2a_shape* s, const void* const* x, const int32_t* const* indices,
                           const int32_t* num_tokens, int32_t compact_rows, int32_t in_dtype, int32_t out_dtype,
                           int32_t* entry_row, int32_t* expert_num_tokens, int32_t* expert_offsets,
                           void* expert_rows, int32_t* expert_meta, void* stream) {
  if (!shape_ok(s) || !local_supported(s) || !x || !indices || !num_tokens || compact_rows < 0 || !expert_rows)
    return MOE_A2A_EINVAL;
  const bool standin = in_dtype >= 0 || out_dtype >= 0;
  if (standin && ((in_dtype != MOE_A2A_F16 && in_dtype != MOE_A2A_BF16) ||
                  (out_dtype != MOE_A2A_F16 && out_dtype != MOE_A2A_BF16)))
    return MOE_A2A_EINVAL;
  const int W = s->world_size, K = s->experts_per_token, E = s->num_experts;
  bool all16 = aligned(expert_rows, 16);
  long long tokens = 0;
  for (int r = 0; r < W; ++r) {
    if (num_tokens[r] < 0 || num_tokens[r] > s->max_num_tokens || (num_tokens[r] > 0 && (!x[r] || !indices[r])))
      return MOE_A2A_EINVAL;
    if (!aligned(x[r], 2)) return MOE_A2A_EALIGN;
    all16 = all16 && aligned(x[r], 16);
    tokens += num_tokens[r];
    if (tokens * K > INT_MAX / 2) return MOE_A2A_EINVAL;
  }
  auto sources = [&](auto table) {
    int first = 0;
    for (int r = 0; r < W; ++r) {
      table.x[r] = x[r];
      table.indices[r] = indices[r];
      table.first[r] = first;
      first += num_tokens[r];
    }
    table.first[W] = first;
    for (int r = W + 1; r < (int)(sizeof(table.first) / sizeof(int)); ++r) table.first[r] = INT_MAX;
    return table;
  };
  const int S = (int)(tokens * K);
  if (!aligned(expert_rows, 2)) return MOE_A2A_EALIGN;
  if (S > 0 && !entry_row) return MOE_A2A_EINVAL;
  const bool compact = compact_rows > 0;
  if (compact && compact_rows < S) return MOE_A2A_EINVAL;
  Geometry g;
  row_geometry(g, s->hidden_dim, all16);
  g.nle = E / W;
  g.max_recv = s->max_num_tokens * W;
  g.magic = g.nle == 1 ? 0u : (uint32_t)(0xffffffffu / (uint32_t)g.nle) + 1u;
  if ((long long)E * g.max_recv > INT_MAX || !items_fit(tokens, g.chunks)) return MOE_A2A_EINVAL;
  // what the padded expert buffers and a rank's receive buffer have room for (the second only matters
  // where a token can have more entries on a rank than the rank has experts)
  const int expert_limit = compact && !standin ? INT_MAX : g.max_recv;
  const int rank_limit = K > g.nle && g.nle > 1 ? (int)std::min<long long>((long long)g.max_recv * g.nle, INT_MAX) : 0;
  hipStream_t st = (hipStream_t)stream;
  const bool through = (long long)S * s->hidden_dim * 2 >= JOB_THROUGH_BYTES;  // (Store)
  // Few ranks with few entries: the mover ranks them
  const int few_nv = local_few_vecs(tokens, S, W, g.row_vecs, g.vec16);
  const int few_chunks = (g.row_vecs + BLOCK * few_nv - 1) / (BLOCK * few_nv);
  if (W <= LOCAL_FEW_RANKS && S > 0 && S <= LOCAL_RANK_ENTRIES && rank_limit == 0 && items_fit(tokens, few_chunks)) {
    const bool counts = expert_num_tokens || expert_offsets;
    const int grid = (counts ? 1 : 0) + (int)(tokens * few_chunks);
#define LAUNCH_H(V, DI, DO, HOW, R, KEYS, NV)                                                              \
  local_dispatch_few_kernel<V, DI, DO, HOW, R, KEYS, NV><<<grid, BLOCK, 0, st>>>(                          \
      x[0], indices[0], (int)tokens, K, E, few_chunks, g.row_vecs, counts, compact, g.max_recv, expert_limit, \
      g.nle, g.magic, W, entry_row, expert_num_tokens, expert_offsets, (V*)expert_rows, expert_meta,       \
      sources(LocalSources<R>{}))
#define LAUNCH_T(V, DI, DO, R, KEYS, NV)                                                                   \
  do {                                                                                                     \
    /* (rows cut for several vectors per lane are 1 MB and more) */                                        \
    constexpr Store SMALL = NV > 1 ? THROUGH_OF<V> : PLAIN;                                                \
    if (through) LAUNCH_H(V, DI, DO, THROUGH_OF<V>, R, KEYS, NV);                                          \
    else LAUNCH_H(V, DI, DO, SMALL, R, KEYS, NV);                                                          \
  } while (0)
#define LAUNCH_S(V, R, KEYS, NV)                                                                           \
  do {                                                                                                     \
    if (!standin) LAUNCH_T(V, -1, -1, R, KEYS, NV);                                                        \
    else if (in_dtype == MOE_A2A_BF16 && out_dtype == MOE_A2A_BF16) LAUNCH_T(V, MOE_A2A_BF16, MOE_A2A_BF16, R, KEYS, NV); \
    else if (in_dtype == MOE_A2A_F16 && out_dtype == MOE_A2A_F16) LAUNCH_T(V, MOE_A2A_F16, MOE_A2A_F16, R, KEYS, NV); \
    else if (in_dtype == MOE_A2A_F16) LAUNCH_T(V, MOE_A2A_F16, MOE_A2A_BF16, R, KEYS, NV);                 \
    else LAUNCH_T(V, MOE_A2A_BF16, MOE_A2A_F16, R, KEYS, NV);                                              \
  } while (0)
#define LAUNCH_N(V, R, KEYS)                                                                               \
  do {                                                                                                     \
    constexpr int MORE = sizeof(V) == sizeof(b128) ? 2 : 4;  /* (local_few_vecs) */                        \
    if (few_nv == 1) LAUNCH_S(V, R, KEYS, 1);                                                              \
    else if (few_nv == MORE) LAUNCH_S(V, R, KEYS, MORE);                                                   \
    else LAUNCH_S(V, R, KEYS, 2 * MORE);                                                                   \
  } while (0)
#define LAUNCH_K(V, R)                                                                                     \
  do {                                                                                                     \
    if (S <= 64 * 4 && few_nv == 1) LAUNCH_S(V, R, 4, 1);                                                  \
    else if (S <= 64 * 16) LAUNCH_N(V, R, 16);                                                             \
    else LAUNCH_N(V, R, 32);                                                                               \
  } while (0)
#define LAUNCH(V)                                                                                          \
  do {                                                                                                     \
    if (W == 1) LAUNCH_K(V, 1);                                                                            \
    else LAUNCH_K(V, LOCAL_FEW_RANKS);                                                                     \
  } while (0)
    if (g.vec16) LAUNCH(b128);
    else LAUNCH(uint16_t);
#undef LAUNCH
#undef LAUNCH_K
#undef LAUNCH_N
#undef LAUNCH_S
#undef LAUNCH_T
#undef LAUNCH_H
    return launch_status();
  }
  int expert_bits = 0, rank_bits = 0;
  while ((1 << expert_bits) < E) ++expert_bits;
  while ((1 << rank_bits) < W) ++rank_bits;
  if (const int rc = allow_large_lds()) return rc;
  if (const int each = g.vec16 ? local_long_tokens(tokens, K, W, E) : 0) {  // the movers rank theirs themselves
    const int nv = local_long_vecs((long long)S * s->hidden_dim * 2, g.row_vecs), pieces = (g.row_vecs + 64 * nv - 1) / (64 * nv);
    const int grid = (int)((tokens + each - 1) / each);
    auto start = [&](auto table) {
      constexpr int R = sizeof(table.x) / sizeof(table.x[0]);
#define LAUNCH_H(NV, DI, DO)                                                                               \
  local_dispatch_long_kernel<NV, DI, DO, R><<<grid, LPLAN_BLOCK, local_plan_lds_bytes(E), st>>>(           \
      table, W, S, K, E, g.nle, g.magic, expert_bits, rank_bits, compact, g.max_recv, expert_limit, rank_limit, each, \
      pieces_of(pieces), g.row_vecs, entry_row, expert_num_tokens, expert_offsets, (b128*)expert_rows, expert_meta)
#define LAUNCH(NV)                                                                                         \
  do {                                                                                                     \
    if (!standin) LAUNCH_H(NV, -1, -1);                                                                    \
    else if (in_dtype == MOE_A2A_BF16 && out_dtype == MOE_A2A_BF16) LAUNCH_H(NV, MOE_A2A_BF16, MOE_A2A_BF16); \
    else if (in_dtype == MOE_A2A_F16 && out_dtype == MOE_A2A_F16) LAUNCH_H(NV, MOE_A2A_F16, MOE_A2A_F16);  \
    else if (in_dtype == MOE_A2A_F16) LAUNCH_H(NV, MOE_A2A_F16, MOE_A2A_BF16);                             \
    else LAUNCH_H(NV, MOE_A2A_BF16, MOE_A2A_F16);                                                          \
  } while (0)
      if (nv == 1) LAUNCH(1);
      else if (nv == 2) LAUNCH(2);
      else LAUNCH(4);
#undef LAUNCH
#undef LAUNCH_H
    };
    if (W == 1) start(sources(LocalSources<1>{}));
    else start(sources(LocalSources<LOCAL_FEW_RANKS>{}));
    return launch_status();
  }
  const int tiles = std::max(1, (S + LPLAN_BLOCK - 1) / LPLAN_BLOCK);
  auto launch = [&](auto table) {
    constexpr int R = sizeof(table.x) / sizeof(table.x[0]);
    local_plan_kernel<R><<<tiles, LPLAN_BLOCK, local_plan_lds_bytes(E), st>>>(
        table, W, S, K, E, g.nle, expert_bits, rank_bits, compact, g.max_recv, expert_limit, rank_limit, entry_row,
        expert_num_tokens, expert_offsets);
    if (S == 0) return;
    const int grid = (int)(tokens * g.chunks);
#define LAUNCH_H(V, NV, DI, DO)                                                                            \
  local_dispatch_kernel<V, NV, DI, DO, THROUGH_OF<V>, R><<<grid, BLOCK, 0, st>>>(                          \
      entry_row, (V*)expert_rows, expert_meta, W, K, g.chunks, g.row_vecs, g.nle, g.magic, table)
#define LAUNCH(V, NV)                                                                                      \
  do {                                                                                                     \
    if (!standin) LAUNCH_H(V, NV, -1, -1);                                                                 \
    else if (in_dtype == MOE_A2A_BF16 && out_dtype == MOE_A2A_BF16) LAUNCH_H(V, NV, MOE_A2A_BF16, MOE_A2A_BF16); \
    else if (in_dtype == MOE_A2A_F16 && out_dtype == MOE_A2A_F16) LAUNCH_H(V, NV, MOE_A2A_F16, MOE_A2A_F16); \
    else if (in_dtype == MOE_A2A_F16) LAUNCH_H(V, NV, MOE_A2A_F16, MOE_A2A_BF16);                          \
    else LAUNCH_H(V, NV, MOE_A2A_BF16, MOE_A2A_F16);                                                       \
  } while (0)
    MOE_A2A_FOR_ROW_KERNEL(g, LAUNCH);
#undef LAUNCH
#undef LAUNCH_H
  };
  // (one rank: nothing to pick from. us, planned, with a table of eight / one: 13694 tokens of 1.2 KB 19.2 / 15.4, 5452 of 2019
  // elements, 2 each, 22.5 / 19.3, 1753 of 6.5 KB, 2 each 10.4 / 9.9)
  if (W == 1) launch(sources(LocalSources<1>{}));
  else if (W <= LOCAL_FEW_RANKS && tokens * g.chunks <= LOCAL_FEW_WORKGROUPS) launch(sources(LocalSources<LOCAL_FEW_RANKS>{}));
  else launch(sources(LocalSources<LOCAL_MAX_RANKS>{}));
  return launch_status();
}

int moe_a2a_local_combine(const moe_a2a_shape* s, const void* expert_rows, const int32_t* entry_row,
                          const float* const* weights, const int32_t* num_tokens, void* const* out_tokens,
                          int32_t only_rank, int32_t accumulate, int32_t dtype, void* stream) {
  if (!shape_ok(s) || !local_supported(s) || !weights || !num_tokens || !out_tokens || only_rank >= s->world_size ||
      (dtype != MOE_A2A_F16 && dtype != MOE_A2A_BF16))
    return MOE_A2A_EINVAL;
  const int W = s->world_size, K = s->experts_per_token;
  bool all16 = aligned(expert_rows, 16);
  long long tokens = 0;
  int first = 0;  // token that the launch starts with
  for (int r = 0; r < W; ++r) {
    if (num_tokens[r] < 0 || num_tokens[r] > s->max_num_tokens) return MOE_A2A_EINVAL;
    const bool wanted = (only_rank < 0 || r == only_rank) && num_tokens[r] > 0;
    if (wanted && (!weights[r] || !out_tokens[r])) return MOE_A2A_EINVAL;
    if (wanted && !aligned(out_tokens[r], 2)) return MOE_A2A_EALIGN;
    all16 = all16 && (!wanted || aligned(out_tokens[r], 16));
    if (r == only_rank) first = (int)tokens;
    tokens += num_tokens[r];
    if (tokens * K > INT_MAX / 2) return MOE_A2A_EINVAL;
  }
  auto results = [&](auto table) {
    int at = 0;
    for (int r = 0; r < W; ++r) {
      table.weights[r] = weights[r];
      table.out[r] = out_tokens[r];
      table.first[r] = at;
      at += num_tokens[r];
    }
    table.first[W] = at;
    for (int r = W + 1; r < (int)(sizeof(table.first) / sizeof(int)); ++r) table.first[r] = INT_MAX;
    return table;
  };
  const long long items = only_rank < 0 ? tokens : num_tokens[only_rank];
  if (items == 0) return MOE_A2A_OK;
  if (!expert_rows || !entry_row) return MOE_A2A_EINVAL;
  if (!aligned(expert_rows, 2)) return MOE_A2A_EALIGN;
  Geometry g;
  row_geometry(g, s->hidden_dim, all16);
  // one column of vectors per lane (eight rows of it in flight), two for rows of 257 to 512 vectors
  const int nv = g.row_vecs > 2 * BLOCK ? 1 : g.row_vecs > BLOCK ? 2 : 1;
  const int chunks = (g.row_vecs + BLOCK * nv - 1) / (BLOCK * nv);
  if (!items_fit(items, chunks)) return MOE_A2A_EINVAL;
  const int grid = (int)(items * chunks);
  hipStream_t st = (hipStream_t)stream;
  const bool few_ranks = W <= LOCAL_FEW_RANKS && grid <= LOCAL_FEW_WORKGROUPS;
  const bool streams = g.vec16 && (items * K + items) * s->hidden_dim * 2 >= (W == 1 ? JOB_STREAM_BYTES : JOB_RANKS_STREAM_BYTES);
  // (of rows in several chunks three entries and more stay with eight, whose workgroups, fewer on a unit, have fewer rows open at once: 8 ranks, us
  // with 8 / as many as there are, 193 tokens of 12 KB, 3 per token 13.7 / 14.0, 184 of 10.7 KB, 4 per token 14.5 / 15.0, 162 of 11 KB, 6 17.2 / 17.6)
  const bool long_rows = g.row_vecs > 2 * BLOCK;
#define LAUNCH_R(V, DT, NV, ADDENDS, HOW, R)                                                               \
  local_combine_kernel<V, DT, NV, ADDENDS, HOW, R><<<grid, BLOCK, 0, st>>>(                                \
      entry_row, weights[0], (const V*)expert_rows, out_tokens[0], K, chunks, g.row_vecs, first, accumulate, W, \
      results(LocalResults<R>{}))
#define LAUNCH(V, DT, NV, ADDENDS, HOW)                                                                    \
  do {                                                                                                     \
    if (W == 1) LAUNCH_R(V, DT, NV, ADDENDS, HOW, 1);                                                      \
    else if (few_ranks) LAUNCH_R(V, DT, NV, ADDENDS, HOW, LOCAL_FEW_RANKS);                                \
    else LAUNCH_R(V, DT, NV, ADDENDS, HOW, LOCAL_MAX_RANKS);                                               \
  } while (0)
#define LAUNCH_N(V, DT, ADDENDS, HOW)                                                                      \
  do {                                                                                                     \
    if (nv == 1) LAUNCH(V, DT, 1, ADDENDS, HOW);                                                           \
    else LAUNCH(V, DT, 2, ADDENDS, HOW);                                                                   \
  } while (0)
#define LAUNCH_H(DT, ADDENDS)                                                                              \
  do {                                                                                                     \
    if (streams) LAUNCH_N(b128, DT, ADDENDS, STREAM);                                                      \
    else LAUNCH_N(b128, DT, ADDENDS, PLAIN);                                                               \
  } while (0)
#define PICK(DT)                                                                                           \
  do {                                                                                                     \
    if (!g.vec16 && K <= 8) LAUNCH_N(uint16_t, DT, 8, PLAIN);                                              \
    else if (!g.vec16) LAUNCH_N(uint16_t, DT, 0, PLAIN);                                                   \
    else if (K <= 2) LAUNCH_H(DT, 2);                                                                      \
    else if (K <= 4 && !long_rows) LAUNCH_H(DT, 4);                                                        \
    else if (K <= 6 && !long_rows) LAUNCH_H(DT, 6);                                                        \
    else if (K <= 8) LAUNCH_H(DT, 8);                                                                      \
    else LAUNCH_H(DT, 0);                                                                                  \
  } while (0)
  if (dtype == MOE_A2A_BF16) PICK(MOE_A2A_BF16);
  else PICK(MOE_A2A_F16);
#undef LAUNCH_H
#undef LAUNCH_N
#undef PICK
#undef LAUNCH
#undef LAUNCH_R
  return launch_status();
}

}  // extern "C"
