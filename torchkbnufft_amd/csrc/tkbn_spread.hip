// Adjoint table interpolation (spread) for gfx950: binned, tile-owned, LDS-accumulated.
//
// Restates torchkbnufft/_nufft/interp.py:587-726 (table_interp_adjoint: the conjugate
// transpose of the forward gather, accumulated with index_add_ per (batch, coil) row).
//
// Plan (per call, per trajectory):
//   1. bin_count   : from each sample's base grid cell (the forward's base-offset rule)
//                    the tiles its J-window reaches (per dimension the tiles of cells
//                    base .. base+J-1, wrapping); one count per reached tile.
//   2. plan_scan   : exclusive scan of the counts; per tile its split count; the work
//                    list of (tile, split) items.
//   3. bin_scatter : per tile, the list of samples that reach it.
// Same-address atomics on hot tiles are aggregated per wave (one atomic per distinct
// tile per wave).
// Spread: one work-group per (tile, split, chunk of coil rows).  The group owns the
// tile's cells: it zeroes an LDS accumulator, walks its candidate samples, adds every
// tap that lands inside the tile with an LDS atomic, and stores each owned cell once.
// Every tile is a work item (empty tiles store zeros), so the output grid needs no
// zero-fill.  Tiles whose candidate list exceeds `target` are split over several
// groups; those tiles are zeroed first and the groups add their partial tiles with
// global atomics.
// Deterministic mode accumulates 64-bit fixed point (integer adds are associative, so
// the result does not depend on the order samples arrive in) and never splits tiles:
// the output is bitwise repeatable.  The fixed-point scale is 2^e with
// e = 60 - ceil(log2(2 * max|kdata| * candidates * wraps)), wraps = prod_d ceil(J_d / K_d),
// so no tile sum can overflow for tables of modulus <= 1 (the Kaiser-Bessel tables are
// normalised to 1).  Complex128 data keeps ~60 bits per tile sum: a quantum of
// 2 max|kdata| V 2^-60 (about 1e-13 relative for a 5e4-entry tile).
#include <mutex>
#include <type_traits>
#include <vector>

#include "tkbn_geom.h"
#include "tkbn_plancache.h"

namespace tkbn {

struct TileGeom {
  int K[3];        // grid size per dimension
  int J[3];        // numpoints per dimension
  int T[3];        // tile size (cells) per dimension
  int nb[3];       // tiles per dimension
  int bstride[3];  // tile index strides
  int lstride[3];  // cell strides inside a tile
  int NB;          // tiles
  int tcells;      // cells per tile
  int target;      // candidate samples per split
  int CC;          // coil rows per work-group
  int64_t maxwork; // work items per trajectory (upper bound)
  int rec_entry;   // separable spread: a record per entry, else one per sample
  int64_t maxent;  // (sample, tile) entries per trajectory (upper bound)
  int own_only;    // forward plans: each sample only in the tile of its base cell
  int R[3];        // forward: staged region per dimension (T + J - 1)
  int rstride[3];  // forward: cell strides of the staged region
  int rcells;      // forward: cells of the staged region
  // workspace offsets (in int32 units) of one trajectory's plan
  int64_t o_key, o_perm, o_count, o_start, o_cursor, o_wstart, o_work, o_nwork, plan_ints;
  int64_t o_maxabs_bytes;  // byte offset of the max|kdata| slot (8 bytes)
  FastDiv fT[3], fl[3], fR[3], ftc, frc;  // dividers by T, lstride, R, tcells, rcells
  FastDiv ftarget;         // separable plan: divider by target
  int64_t o_rec_bytes;     // separable plan: byte offset of the records
  int64_t plan_stride;     // separable plan: ints from one trajectory's plan to the next
  int64_t o_hot;                             // 3-D register-tile plan: list of split tiles
  int64_t o_meta, o_tmp, o_sort, o_scratch;  // 3-D register-tile plan: counts, scan scratch, sort
  int64_t o_sw, o_sb;                        // 3-D register-tile plan: per-sample tap weights, bases
  int64_t pool_off_bytes, pool_slots;        // 3-D register-tile plan: piece partials
  int nchunk;                                // 3-D register-tile plan: chunks of coil rows
};

// dynamic LDS per group; with the ~350 bytes of static LDS the total stays under 64 KiB
constexpr int kLdsBudget = 60 * 1024;

// Threads per group of the sample-lane kernels (single-problem and batched).  The gather
// stages one region per group (at most two groups per CU), so 1024 lanes hide its LDS and
// tap latency best (8-coil 320^3 kooshball forward 4.0 -> 2.8 ms, 64 uneven 2-D problems
// 4.4 -> 4.0 ms per batched pair, 1-coil 256^2 pair 0.17 -> 0.15 ms).  The spread keeps
// 256: more lanes per tile contend for the same LDS accumulators (the batched pair
// 4.4 -> 5.4-6.0 ms with 512-1024).
// (complex128 and numpoints above 6 keep 256: at 1024 threads their registers spill.)
constexpr int spread_tiles_threads(int) { return 256; }
// (The 3-D gather's registers leave a CU six waves per SIMD: one group of 1024 threads, which
// then waits for its own 60 KB of staging, or three of 512, of which LDS holds two, one
// gathering while the other stages.  320^3, 8 rows, 1.6 M radial samples: 256 threads 2.95 ms,
// 512 2.47 ms, 1024 2.59 ms.)
template <typename T, int JM, int D>
constexpr int fwd_tiled_threads() { return sizeof(T) == 4 && JM <= 6 ? (D == 3 ? 512 : 1024) : 256; }

template <typename T>
__device__ __forceinline__ int64_t sample_base_wrapped(const Geom<T>& g, int d, T omega) {
#pragma clang fp contract(off)
  const T tm = omega / g.gam[d];
  const bool ok = (fabs(tm) < (T)1.0e15);
  const T fb = floor(tm - g.halfJ[d]);
  const int64_t base = ok ? (int64_t)fb + 1 : 0;
  int64_t bm = base % g.K[d];
  if (bm < 0) bm += g.K[d];
  return bm;
}

// ---------------------------------------------------------------------------
// plan kernels
// ---------------------------------------------------------------------------
// Tiles reached along dimension d by a sample whose wrapped base cell is bm: the tiles
// of cells bm .. bm+J-1 (mod K); at most 3 (2 unless the last tile is shorter than J-1).
__device__ __forceinline__ int dim_tiles(const TileGeom& tg, int d, int bm, int* tl) {
  if (tg.own_only) {
    tl[0] = bm / tg.T[d];
    return 1;
  }
  int n = 0;
  for (int j = 0; j < tg.J[d]; ++j) {
    int c = bm + j;
    while (c >= tg.K[d]) c -= tg.K[d];
    const int tile = c / tg.T[d];
    bool seen = false;
    for (int q = 0; q < n; ++q) seen = seen || tl[q] == tile;
    if (!seen && n < 3) tl[n++] = tile;
  }
  return n;
}

// Groups the wave's valid lanes by key (ballots and shuffles only): the lowest lane of
// each group is its leader; `rank` is the lane's position inside its group and `cnt`
// (leaders only) the group size.
__device__ __forceinline__ void wave_group_by_key(int key, bool valid, int& leader_of, int& rank, int& cnt) {
  const int lane = threadIdx.x & 63;
  unsigned long long pending = __ballot(valid);
  leader_of = lane;
  rank = 0;
  cnt = 0;
  while (pending) {
    const int leader = __ffsll((unsigned long long)pending) - 1;
    const int lkey = __shfl(key, leader, 64);
    // keys of earlier groups differ from lkey, so `mine` only selects pending lanes
    const bool mine = valid && key == lkey;
    const unsigned long long same = __ballot(mine) & pending;
    if (lane == leader) cnt = __popcll(same);
    if (mine) {
      leader_of = leader;
      rank = __popcll(same & ((1ull << lane) - 1ull));
    }
    pending &= ~same;
  }
}

// atomicAdd(ptr + key, 1) for every lane with `valid`: one atomic per distinct key in
// the wave, all issued by one instruction.  Returns the value this lane's increment
// would have seen (lanes with equal keys are ranked in lane order), -1 if not valid.
// Every active lane of the wave must call it.
// Work-group barrier that orders LDS accesses only.  __syncthreads() also waits for
// the group's outstanding global loads and stores (its workgroup-scope fence), which
// would serialise a loop of store rounds on their completion.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ int wave_aggregated_inc(int* ptr, int key, bool valid) {
  const int lane = threadIdx.x & 63;
  int leader_of, rank, cnt;
  wave_group_by_key(key, valid, leader_of, rank, cnt);
  int old = 0;
  if (valid && leader_of == lane) old = atomicAdd(ptr + key, cnt);
  old = __shfl(old, leader_of, 64);
  return valid ? old + rank : -1;
}

// the same increments when the old values are not needed (no return trip)
__device__ __forceinline__ void wave_aggregated_add(int* ptr, int key, bool valid) {
  const int lane = threadIdx.x & 63;
  int leader_of, rank, cnt;
  wave_group_by_key(key, valid, leader_of, rank, cnt);
  if (valid && leader_of == lane) atomicAdd(ptr + key, cnt);
}

template <typename T, int D>
__device__ __forceinline__ void sample_tiles(const Geom<T>& g, const TileGeom& tg, const T* om, int64_t m, bool live,
                                             int tl[3][3], int* ntl) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    ntl[d] = 1;
    tl[d][0] = 0;
  }
  if (!live) return;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const int bm = (int)sample_base_wrapped<T>(g, d, om[d * g.M + m]);
    ntl[d] = dim_tiles(tg, d, bm, tl[d]);
  }
}

// Walks the (up to 27) reached tiles of each lane's sample in a wave-uniform loop and
// applies fn(key, valid) to each; lanes past the end pass valid = false.
template <int D, typename F>
__device__ __forceinline__ void for_each_tile(const TileGeom& tg, int tl[3][3], const int* ntl, bool live, F fn) {
  for (int a = 0; a < (D > 0 ? 3 : 1); ++a)
    for (int c = 0; c < (D > 1 ? 3 : 1); ++c)
      for (int e = 0; e < (D > 2 ? 3 : 1); ++e) {
        const bool valid = live && a < ntl[0] && c < ntl[1] && e < ntl[2];
        int key = 0;
        if (valid) {
          key = tl[0][a] * tg.bstride[0];
          if (D > 1) key += tl[1][c] * tg.bstride[1];
          if (D > 2) key += tl[2][e] * tg.bstride[2];
        }
        if (__ballot(valid)) fn(key, valid);
      }
}

// Grid-stride over the samples (whole blocks step together, so the wave-aggregated
// atomics see full waves); the grid is capped (bin_grid) so that the launch costs
// little when a cached plan makes it exit at once.
template <typename T, int D>
__global__ void __launch_bounds__(256)
    bin_count_kernel(const Geom<T> g, const TileGeom tg, const T* __restrict__ omega, int* __restrict__ ws,
                     const CacheHdr* cache) {
  if (cache_hit(cache)) return;  // cached plan reused
  const int64_t b = blockIdx.z;
  const T* om = omega + (g.batched ? b * D * g.M : 0);
  int* count = ws + b * tg.plan_ints + tg.o_count;
  for (int64_t m0 = (int64_t)blockIdx.x * blockDim.x; m0 < g.M; m0 += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = m0 + threadIdx.x;
    const bool live = m < g.M;
    int tl[3][3], ntl[3];
    sample_tiles<T, D>(g, tg, om, m, live, tl, ntl);
    for_each_tile<D>(tg, tl, ntl, live, [&](int key, bool valid) { wave_aggregated_add(count, key, valid); });
  }
}

template <typename T, int D>
__global__ void __launch_bounds__(256)
    bin_scatter_kernel(const Geom<T> g, const TileGeom tg, const T* __restrict__ omega, int* __restrict__ ws,
                       const CacheHdr* cache) {
  if (cache_hit(cache)) return;  // cached plan reused
  const int64_t b = blockIdx.z;
  const T* om = omega + (g.batched ? b * D * g.M : 0);
  int* plan = ws + b * tg.plan_ints;
  for (int64_t m0 = (int64_t)blockIdx.x * blockDim.x; m0 < g.M; m0 += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = m0 + threadIdx.x;
    const bool live = m < g.M;
    int tl[3][3], ntl[3];
    sample_tiles<T, D>(g, tg, om, m, live, tl, ntl);
    for_each_tile<D>(tg, tl, ntl, live, [&](int key, bool valid) {
      const int pos = wave_aggregated_inc(plan + tg.o_cursor, key, valid);
      if (valid) plan[tg.o_perm + pos] = (int)m;
    });
  }
}

// blocks of 256 for a grid-stride pass over n items: at most 2048
inline unsigned bin_grid(int64_t n) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 256), 2048)); }

// Block-wide exclusive scan of n ints (in place into out[0..n]), 1024 threads.
__device__ void block_exclusive_scan(const int* in, int* out, int n, int* sbuf) {
  const int tid = threadIdx.x, nt = blockDim.x;
  const int per = (n + nt - 1) / nt;
  const int lo = tid * per, hi = min(lo + per, n);
  int sum = 0;
  for (int i = lo; i < hi; ++i) sum += in[i];
  sbuf[tid] = sum;
  __syncthreads();
  // Hillis-Steele over the per-thread sums
  for (int off = 1; off < nt; off <<= 1) {
    const int v = tid >= off ? sbuf[tid - off] : 0;
    __syncthreads();
    sbuf[tid] += v;
    __syncthreads();
  }
  int run = sbuf[tid] - sum;
  for (int i = lo; i < hi; ++i) {
    const int v = in[i];
    out[i] = run;
    run += v;
  }
  if (tid == nt - 1) out[n] = sbuf[nt - 1];
  __syncthreads();
}

__global__ void __launch_bounds__(1024) plan_scan_kernel(const TileGeom tg, int* __restrict__ ws,
                                                        const CacheHdr* cache = nullptr) {
  if (cache && cache_hit(cache)) return;  // cached plan reused
  __shared__ int sbuf[1024];
  int* plan = ws + (int64_t)blockIdx.x * tg.plan_ints;
  const int* count = plan + tg.o_count;
  int* start = plan + tg.o_start;
  int* cursor = plan + tg.o_cursor;
  int* wstart = plan + tg.o_wstart;
  int* work = plan + tg.o_work;
  block_exclusive_scan(count, start, tg.NB, sbuf);
  for (int i = threadIdx.x; i < tg.NB; i += blockDim.x) cursor[i] = start[i];
  // split counts per tile (stored temporarily in wstart[t + 1])
  for (int t = threadIdx.x; t < tg.NB; t += blockDim.x) {
    const int v = count[t];
    wstart[t + 1] = v <= tg.target ? 1 : (v + tg.target - 1) / tg.target;
  }
  __syncthreads();
  // scan of split counts: reuse cursor-free area (work list) as scratch input
  int* splits = work;  // NB ints, then overwritten by the work list below
  for (int t = threadIdx.x; t < tg.NB; t += blockDim.x) splits[t] = wstart[t + 1];
  __syncthreads();
  block_exclusive_scan(splits, wstart, tg.NB, sbuf);
  // work list: work[wstart[t] + s] = t
  const int cap = (int)tg.maxwork;  // cannot be exceeded (see make_tile_geom); guards memory
  for (int t = threadIdx.x; t < tg.NB; t += blockDim.x) {
    const int a = wstart[t], e = min(wstart[t + 1], cap);
    for (int w = a; w < e; ++w) work[w] = t;
  }
  if (threadIdx.x == 0) plan[tg.o_nwork] = min(wstart[tg.NB], cap);
}

// ---------------------------------------------------------------------------
// max |re|, |im| of kdata (deterministic mode's fixed-point scale)
// ---------------------------------------------------------------------------
template <typename T>
struct uint_of;
template <>
struct uint_of<float> {
  using type = unsigned int;
};
template <>
struct uint_of<double> {
  using type = unsigned long long;
};

// max |re|, |im| over kdata, or +inf when kdata or omega holds a non-finite value
// (fixed-point accumulation cannot carry those; the float-atomic kernel then runs)
// Block `blk` of `nblk` (256 threads) of the max-|kdata| pass.
template <typename T>
__device__ __forceinline__ void maxabs_block(const T* __restrict__ x, int64_t n, const T* __restrict__ om, int64_t nom,
                                             void* slot, int64_t blk, int64_t nblk) {
  using U = typename uint_of<T>::type;
  T mx = 0;
  for (int64_t i = blk * blockDim.x + threadIdx.x; i < n; i += nblk * blockDim.x) {
    const T v = fabs(x[i]);
    mx = isfinite(v) ? (v > mx ? v : mx) : (T)INFINITY;
  }
  for (int64_t i = blk * blockDim.x + threadIdx.x; i < nom; i += nblk * blockDim.x)
    if (!isfinite(om[i])) mx = (T)INFINITY;
  // wave reduce, block reduce in LDS, then one atomic per block (few blocks: the
  // atomics all hit one address)
  for (int off = 32; off > 0; off >>= 1) {
    const T o = __shfl_down(mx, off, 64);
    mx = o > mx ? o : mx;
  }
  __shared__ T wmax[4];  // 256 threads = 4 waves
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) mx = wmax[w] > mx ? wmax[w] : mx;
    U bits;
    memcpy(&bits, &mx, sizeof(T));
    atomicMax(static_cast<U*>(slot), bits);  // non-negative floats order like their bits
  }
}

template <typename T>
__global__ void __launch_bounds__(256) maxabs_kernel(const T* __restrict__ x, int64_t n, const T* __restrict__ om,
                                                     int64_t nom, void* slot) {
  maxabs_block<T>(x, n, om, nom, slot, blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------------
// zero the cells of split tiles (fast mode), before their partial sums arrive
// ---------------------------------------------------------------------------
template <typename T, int D>
__device__ __forceinline__ void zero_hot_tiles_item(const Geom<T>& g, const TileGeom& tg, const int* __restrict__ ws,
                                                    cplx<T>* __restrict__ grid, int t, int64_t yc, int64_t b) {
  const int* plan = ws + b * tg.plan_ints;
  const int* wstart = plan + tg.o_wstart;
  if (wstart[t + 1] - wstart[t] <= 1) return;
  const int64_t nrows = g.batched ? g.C : g.B * g.C;
  const int64_t rowbase = g.batched ? b * g.C : 0;
  const int64_t r0 = yc * tg.CC;
  const int64_t r1 = r0 + tg.CC < nrows ? r0 + tg.CC : nrows;
  int origin[3] = {0, 0, 0};
  for (int d = 0; d < D; ++d) origin[d] = ((t / tg.bstride[d]) % tg.nb[d]) * tg.T[d];
  for (int cell = threadIdx.x; cell < tg.tcells; cell += blockDim.x) {
    int64_t gi = 0;
    bool in = true;
    for (int d = 0; d < D; ++d) {
      const int l = (int)fmodd(fdiv(cell, tg.fl[d]), tg.fT[d]);
      const int k = origin[d] + l;
      in = in && k < g.K[d];
      gi += (int64_t)k * g.stride[d];
    }
    if (!in) continue;
    for (int64_t r = r0; r < r1; ++r) grid[(rowbase + r) * g.G + gi] = make_c<T>(0, 0);
  }
}

template <typename T, int D>
__global__ void __launch_bounds__(256)
    zero_hot_tiles_kernel(const Geom<T> g, const TileGeom tg, const int* __restrict__ ws, cplx<T>* __restrict__ grid) {
  zero_hot_tiles_item<T, D>(g, tg, ws, grid, blockIdx.x, blockIdx.y, blockIdx.z);
}

// The zero pass of split tiles and the max-|kdata| pass as one launch (both must finish
// before the spread; one launch saves the host a few microseconds per call): blocks
// [0, NB * ychunks * zdim) zero, the last `nmax` blocks take the max.
template <typename T, int D>
__global__ void __launch_bounds__(256)
    zero_hot_maxabs_kernel(const Geom<T> g, const TileGeom tg, const int* __restrict__ ws, cplx<T>* __restrict__ grid,
                           int64_t ychunks, const T* __restrict__ x, int64_t n, const T* __restrict__ om, int64_t nom,
                           void* slot, int64_t nmax) {
  const int64_t nzero = (int64_t)tg.NB * ychunks * (g.batched ? g.B : 1);
  const int64_t blk = blockIdx.x;
  if (blk >= nzero) {
    maxabs_block<T>(x, n, om, nom, slot, blk - nzero, nmax);
    return;
  }
  const int64_t t = blk % tg.NB, rest = blk / tg.NB;
  zero_hot_tiles_item<T, D>(g, tg, ws, grid, (int)t, rest % ychunks, rest / ychunks);
}

// ---------------------------------------------------------------------------
// the spread
// ---------------------------------------------------------------------------
template <typename T, bool DET>
struct AccOf;
template <>
struct AccOf<float, false> {
  using type = float;
};
template <>
struct AccOf<double, false> {
  using type = double;
};
template <typename T>
struct AccOf<T, true> {
  using type = unsigned long long;
};

// x * scale as a two's-complement 64-bit integer.  float: the product is exact (scale is
// a power of two, |x * scale| < 2^61), and its magnitude a splits exactly into
// 2^32 * hi + lo with hi = floor(a / 2^32) and lo in [0, 2^32) (a's 24 significant bits
// either all lie below 2^32, hi = 0, or lo holds those of them below 2^32), so two 32-bit
// conversions replace a double round trip; rounded toward zero.  double: to nearest.
__device__ __forceinline__ unsigned long long to_fixed(float x, float scale) {
  const float v = x * scale;
  const float a = fabsf(v);
  const float hi = floorf(a * 0x1p-32f);
  const float lo = fmaf(hi, -0x1p32f, a);
  const unsigned long long u =
      ((unsigned long long)(unsigned int)hi << 32) + (unsigned long long)(unsigned int)lo;
  return v < 0.f ? 0ull - u : u;
}
__device__ __forceinline__ unsigned long long to_fixed(double x, double scale) {
  return (unsigned long long)llrint(x * scale);
}

// FIXED: 64-bit fixed-point LDS accumulation (LDS integer atomics are much faster
// than float ones; the sum is also order independent).  It exits when the max|kdata|
// slot says a non-finite value is present; the float kernel launched with
// `fallback` = 1 runs only in that case, so NaN and inf still propagate.
// One work item: tile piece wi, chunk yc of tg.CC coil rows, per-batch plan b (blockIdx
// of spread_tiles_kernel, or a batch kernel's decoded item).
template <typename T, bool FIXED, int D, int JM>
__device__ __forceinline__ void spread_tiles_item(const Geom<T>& g, const TileGeom& tg, const cplx<T>* __restrict__ kdata,
                                                  const T* __restrict__ omega, const int* __restrict__ ws,
                                                  const void* __restrict__ maxabs_slot, cplx<T>* __restrict__ grid,
                                                  const int fallback, int64_t wi, int64_t yc, int64_t b,
                                                  unsigned char* smem_raw) {
  using C2 = cplx<T>;
  using A = typename AccOf<T, FIXED>::type;
  T amax = 0;
  if (FIXED || fallback) {
    memcpy(&amax, maxabs_slot, sizeof(T));
    if (FIXED != (bool)isfinite(amax)) return;  // the other kernel of the pair handles this call
  }
  A* acc = reinterpret_cast<A*>(smem_raw);

  const int* plan = ws + b * tg.plan_ints;
  if (wi >= plan[tg.o_nwork]) return;
  const int* wstart = plan + tg.o_wstart;
  const int t = plan[tg.o_work + wi];
  const int split = (int)(wi - wstart[t]);
  const int nsplit = wstart[t + 1] - wstart[t];

  const int64_t nrows = g.batched ? g.C : g.B * g.C;
  const int64_t rowbase = g.batched ? b * g.C : 0;
  const int64_t r0 = yc * tg.CC;
  const int ncc = (int)((r0 + tg.CC < nrows ? r0 + tg.CC : nrows) - r0);

  int origin[3] = {0, 0, 0};
#pragma unroll
  for (int d = 0; d < D; ++d) origin[d] = ((t / tg.bstride[d]) % tg.nb[d]) * tg.T[d];

  const int cstart = plan[tg.o_start + t];
  const int V = plan[tg.o_start + t + 1] - cstart;  // (counts are cleared each call)
  const int i0 = split * tg.target;
  const int i1 = min(i0 + tg.target, V);

  const int nacc = ncc * 2 * tg.tcells;
  for (int i = threadIdx.x; i < nacc; i += blockDim.x) acc[i] = A(0);
  __syncthreads();

  double scale = 1.0;
  if constexpr (FIXED) {
    // |re|, |im| of one tap <= 2 max(|re|, |im|) of the data times |w_0 .. w_{D-1}| <= 1
    // (tables normalised to 1); a cell meets at most V entries, each up to
    // prod_d ceil(J_d / K_d) times (footprints wider than a tiny grid wrap onto it)
    double mult = 1.0;
#pragma unroll
    for (int d = 0; d < D; ++d) mult *= (double)((g.J[d] + g.K[d] - 1) / g.K[d]);
    const double bound = 2.0 * (double)amax * (double)(V > 0 ? V : 1) * mult;
    int e = 50;
    if (bound > 0) e = 60 - (ilogb(bound) + 1);  // amax is finite here (the float kernel takes the rest)
    e = e > 100 ? 100 : e;
    scale = ldexp(1.0, e);
  }
  const T fscale = (T)scale;  // a power of two: x * fscale is exact (|x * fscale| < 2^61)

  const int* perm = plan + tg.o_perm;
  const T* om = omega + (g.batched ? b * D * g.M : 0);
  for (int i = i0 + (int)threadIdx.x; i < i1; i += blockDim.x) {
    const int m = perm[cstart + i];
    C2 w[D][JM];
    int loc[D][JM];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      int mdx[JM];
      sample_taps_md<T, JM>(g, d, om[d * g.M + m], w[d], mdx);
#pragma unroll
      for (int j = 0; j < JM; ++j) {
        const int l = mdx[j] - origin[d];
        loc[d][j] = (mdx[j] >= 0 && l >= 0 && l < tg.T[d]) ? l * tg.lstride[d] : -1;
      }
    }
    const T theta = sample_theta<T, D>(g, om, m);
    const C2 phase = make_c<T>(cos(theta), sin(theta));
    // the next row's sample is loaded while this row's taps are added
    const C2* kp = kdata + (rowbase + r0) * g.M + m;
    C2 knext = ncc > 0 ? kp[0] : make_c<T>(0, 0);
    for (int c = 0; c < ncc; ++c) {
      const C2 kc = knext;
      if (c + 1 < ncc) knext = kp[(int64_t)(c + 1) * g.M];
      C2 v = cmul_conj(kc, phase);
      if constexpr (FIXED) {
        // the fixed-point scale (a power of two) applied once per row: every tap
        // product is then the scaled one exactly
        v.x *= fscale;
        v.y *= fscale;
      }
      A* are = acc + (int64_t)(2 * c) * tg.tcells;
      A* aim = are + tg.tcells;
      auto add = [&](int cell, C2 x) {
        if constexpr (FIXED) {
          atomicAdd(are + cell, to_fixed(x.x, (T)1));
          atomicAdd(aim + cell, to_fixed(x.y, (T)1));
        } else {
          atomicAdd(are + cell, x.x);
          atomicAdd(aim + cell, x.y);
        }
      };
      if constexpr (D == 1) {
#pragma unroll
        for (int j0 = 0; j0 < JM; ++j0)
          if (loc[0][j0] >= 0) add(loc[0][j0], cmul_conj(v, w[0][j0]));
      } else if constexpr (D == 2) {
#pragma unroll
        for (int j0 = 0; j0 < JM; ++j0) {
          if (loc[0][j0] >= 0) {
            const C2 v0 = cmul_conj(v, w[0][j0]);
#pragma unroll
            for (int j1 = 0; j1 < JM; ++j1)
              if (loc[1][j1] >= 0) add(loc[0][j0] + loc[1][j1], cmul_conj(v0, w[1][j1]));
          }
        }
      } else {
#pragma unroll 1
        for (int j0 = 0; j0 < JM; ++j0) {
          if (loc[0][j0] >= 0) {
            const C2 v0 = cmul_conj(v, w[0][j0]);
#pragma unroll
            for (int j1 = 0; j1 < JM; ++j1) {
              if (loc[1][j1] >= 0) {
                const C2 v1 = cmul_conj(v0, w[1][j1]);
                const int base = loc[0][j0] + loc[1][j1];
#pragma unroll
                for (int j2 = 0; j2 < JM; ++j2)
                  if (loc[2][j2] >= 0) add(base + loc[2][j2], cmul_conj(v1, w[2][j2]));
              }
            }
          }
        }
      }
    }
  }
  __syncthreads();

  // store the owned cells
  const double inv = 1.0 / scale;
  for (int idx = threadIdx.x; idx < ncc * tg.tcells; idx += blockDim.x) {
    const int c = (int)fdiv(idx, tg.ftc);
    const int cell = idx - c * tg.tcells;
    int64_t gi = 0;
    bool in = true;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int l = (int)fmodd(fdiv(cell, tg.fl[d]), tg.fT[d]);
      const int kk = origin[d] + l;
      in = in && kk < g.K[d];
      gi += (int64_t)kk * g.stride[d];
    }
    if (!in) continue;
    C2 val;
    if constexpr (FIXED) {
      val.x = (T)((double)(long long)acc[(2 * c) * tg.tcells + cell] * inv);
      val.y = (T)((double)(long long)acc[(2 * c + 1) * tg.tcells + cell] * inv);
    } else {
      val.x = acc[(2 * c) * tg.tcells + cell];
      val.y = acc[(2 * c + 1) * tg.tcells + cell];
    }
    C2* dst = grid + (rowbase + r0 + c) * g.G + gi;
    if (nsplit == 1) {
      *dst = val;
    } else {
      unsafeAtomicAdd(&dst->x, val.x);
      unsafeAtomicAdd(&dst->y, val.y);
    }
  }
}

template <typename T, bool FIXED, int D, int JM>
__global__ void __launch_bounds__(spread_tiles_threads(D))
    spread_tiles_kernel(const Geom<T> g, const TileGeom tg, const cplx<T>* __restrict__ kdata,
                        const T* __restrict__ omega, const int* __restrict__ ws, const void* __restrict__ maxabs_slot,
                        cplx<T>* __restrict__ grid, const int fallback) {
  // 16-byte aligned: 8-byte LDS atomics (double / int64 accumulators) need natural
  // alignment, and the static LDS above this array is not a multiple of 8 bytes
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  spread_tiles_item<T, FIXED, D, JM>(g, tg, kdata, omega, ws, maxabs_slot, grid, fallback, blockIdx.x, blockIdx.y,
                                     blockIdx.z, smem_raw);
}

// Fixed point, or (when the max slot says kdata or omega holds a non-finite value) the
// float-atomic pass, in one launch: the two items return at once unless the slot selects
// them (the LDS is sized for the fixed-point accumulators, the larger of the two).
template <typename T, int D, int JM>
__global__ void __launch_bounds__(spread_tiles_threads(D))
    spread_tiles_either_kernel(const Geom<T> g, const TileGeom tg, const cplx<T>* __restrict__ kdata,
                               const T* __restrict__ omega, const int* __restrict__ ws,
                               const void* __restrict__ maxabs_slot, cplx<T>* __restrict__ grid) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  spread_tiles_item<T, true, D, JM>(g, tg, kdata, omega, ws, maxabs_slot, grid, 0, blockIdx.x, blockIdx.y, blockIdx.z,
                                    smem_raw);
  spread_tiles_item<T, false, D, JM>(g, tg, kdata, omega, ws, maxabs_slot, grid, 1, blockIdx.x, blockIdx.y,
                                     blockIdx.z, smem_raw);
}

// ---------------------------------------------------------------------------
// separable spread geometry (2-D, complex64, J <= 6; the kernel is spread_sep_kernel):
//   entries (sample, 16 x 16 tile its footprint meets).  Footprints are contiguous inside a
//   tile when every grid extent is at least tile + J - 1 cells (a wrapped footprint then
//   never meets one tile twice); smaller grids use the sample-lane kernel.
// ---------------------------------------------------------------------------
constexpr int kRegT0 = 16, kRegT1 = 16;
constexpr int kRegMinC0 = -5;  // first footprint column relative to the tile, J <= 6
constexpr int kRegKeys = kRegT1 - kRegMinC0;  // c0 values per tile: -5 .. 15

// Tiles met along one dimension by the footprint bm .. bm+J-1 (mod K), in footprint
// order, with the footprint's first cell relative to each tile's origin.  The runs of
// one tile are contiguous because K >= T + J - 1.
__device__ __forceinline__ int coil_dim_tiles(int K, int J, int T, int bm, int* tl, int* off) {
  int n = 0;
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    if (j < J) {
      int c = bm + j;
      if (c >= K) c -= K;  // bm < K and J < K
      const int tile = c / T;
      if (n == 0 || tl[n - 1] != tile) {
        tl[n] = tile;
        off[n] = c - tile * T - j;
        ++n;
      }
    }
  }
  return n;
}

// Walks a sample's (tile0, tile1) pairs in a wave-uniform loop; fn(key, pair0, pair1, valid).
template <typename F>
__device__ __forceinline__ void coil_for_each_entry(const TileGeom& tg, const int (&tl)[2][3], const int (&off)[2][3],
                                                    const int (&n)[2], bool live, F fn) {
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const bool valid = live && a < n[0] && c < n[1];
      const int key = valid ? ((tl[0][a] * tg.nb[1] + tl[1][c]) * kRegKeys + off[1][c] - kRegMinC0) : 0;
      if (__ballot(valid)) fn(key, a, c, valid);
    }
}

__device__ __forceinline__ void coil_sample_tiles(const Geom<float>& g, const TileGeom& tg, const float* om, int m,
                                                  bool live, int (&tl)[2][3], int (&off)[2][3], int (&n)[2]) {
  n[0] = n[1] = 0;
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int q = 0; q < 3; ++q) tl[d][q] = off[d][q] = 0;
  if (!live) return;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const int bm = (int)sample_base_wrapped<float>(g, d, om[d * g.M + m]);
    n[d] = coil_dim_tiles(g.K[d], g.J[d], tg.T[d], bm, tl[d], off[d]);
  }
}

// ---------------------------------------------------------------------------
// separable forward gather geometry (2-D, complex64, J <= 6; the kernel is
// gather_sep_kernel)
//   The plan bins every sample once, into the tile of its base cell (the footprint's
//   first cell), keeping trajectory order inside a tile.  One group per (16 x 16 tile,
//   split, chunk of coil rows) stages the tile and its J-1 halo (21 x 21 cells, wrapped) in
//   LDS with the coil row fastest; the lanes of an entry are the chunk's rows, so a tap
//   read by a wave is a few runs of consecutive LDS words.
// ---------------------------------------------------------------------------
constexpr int kGatT0 = 16, kGatT1 = 16;     // tile edges
constexpr int kGatR0 = kGatT0 + 5;          // staged region edges (J <= 6)
constexpr int kGatR1 = kGatT1 + 5;
constexpr int kGatCells = kGatR0 * kGatR1;  // 441
constexpr int kGatTarget = 512;             // entries per work item

__device__ __forceinline__ int gat_base_tile(const Geom<float>& g, const TileGeom& tg, const float* om, int m, int* l) {
  int key = 0;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const int T = d == 0 ? kGatT0 : kGatT1;
    const int bm = (int)sample_base_wrapped<float>(g, d, om[d * g.M + m]);
    const int tile = bm / T;
    l[d] = bm - tile * T;
    key += tile * tg.bstride[d];
  }
  return key;
}

// Work item of group b.  Consecutive groups go to different XCDs (round robin), so
// group b runs on XCD x = b mod 8 as that XCD's k-th group, k = b / 8.  Items are
// dealt to the XCDs in runs of `run` consecutive items (run r -> XCD r mod 8).  The
// gather makes a run kXcdTiles neighbouring work items times all their coil chunks:
// the chunks of a tile share its plan records, and neighbouring tiles the cache lines
// of their common halo columns, through one L2, while the hot tiles at the head of the
// list spread over all XCDs.  A bijection of [0, n) for n a multiple of 8 * run.
constexpr int kXcdTiles = 4;
__device__ __forceinline__ int64_t xcd_work_item(int64_t b, int run) {
  const int64_t x = b % 8, k = b / 8;
  return run * (x + 8 * (k / run)) + k % run;
}

// ---------------------------------------------------------------------------
// forward gather from an LDS-staged tile (standard grid layout)
//   one group per (tile, split, coil chunk): stage the tile plus its J-1 halo cells
//   (wrapped) for the chunk's rows, then every sample based in the tile reads its
//   J^d neighbourhood from LDS.
// ---------------------------------------------------------------------------
// acc += a * b with four fused multiply-adds into the accumulator
template <typename C>
__device__ __forceinline__ void cmac_fma(C& acc, const C a, const C b) {
  acc.x = fma(a.x, b.x, acc.x);
  acc.x = fma(-a.y, b.y, acc.x);
  acc.y = fma(a.x, b.y, acc.y);
  acc.y = fma(a.y, b.x, acc.y);
}

// Sum over the J^D taps of one sample from the staged region L (nested: the last
// dimension's row first).  FULL: every numpoints is JM, so the loads of a row carry no
// guards and are issued together.
template <typename T, int D, int JM, bool FULL>
__device__ __forceinline__ cplx<T> fwd_taps(const Geom<T>& g, const TileGeom& tg, const cplx<T>* L,
                                            const cplx<T> (&w)[D][JM], const int (&loc0)[D]) {
  using C2 = cplx<T>;
  const C2 zero = make_c<T>(0, 0);
  C2 acc = zero;
  if constexpr (D == 1) {
    C2 v[JM];
#pragma unroll
    for (int j = 0; j < JM; ++j) v[j] = (FULL || j < g.J[0]) ? L[loc0[0] + j] : zero;
#pragma unroll
    for (int j = 0; j < JM; ++j) cmac_fma(acc, w[0][j], v[j]);
  } else if constexpr (D == 2) {
#pragma unroll
    for (int j0 = 0; j0 < JM; ++j0) {
      if (FULL || j0 < g.J[0]) {
        const C2* rp = L + (loc0[0] + j0) * tg.rstride[0] + loc0[1];
        C2 v[JM];
#pragma unroll
        for (int j1 = 0; j1 < JM; ++j1) v[j1] = (FULL || j1 < g.J[1]) ? rp[j1] : zero;
        C2 part = zero;
#pragma unroll
        for (int j1 = 0; j1 < JM; ++j1) cmac_fma(part, w[1][j1], v[j1]);
        cmac_fma(acc, w[0][j0], part);
      }
    }
  } else {
    auto plane = [&](int j0) {  // sum over the (j1, j2) taps of plane j0
      C2 p0 = zero;
#pragma unroll
      for (int j1 = 0; j1 < JM; ++j1) {
        if (FULL || j1 < g.J[1]) {
          const C2* rp = L + (loc0[0] + j0) * tg.rstride[0] + (loc0[1] + j1) * tg.rstride[1] + loc0[2];
          C2 v[JM];
#pragma unroll
          for (int j2 = 0; j2 < JM; ++j2) v[j2] = (FULL || j2 < g.J[2]) ? rp[j2] : zero;
          C2 p1 = zero;
#pragma unroll
          for (int j2 = 0; j2 < JM; ++j2) cmac_fma(p1, w[2][j2], v[j2]);
          cmac_fma(p0, w[1][j1], p1);
        }
      }
      return p0;
    };
    if constexpr (JM <= 6) {
#pragma unroll
      for (int j0 = 0; j0 < JM; ++j0)
        if (FULL || j0 < g.J[0]) cmac_fma(acc, w[0][j0], plane(j0));
    } else {
#pragma unroll 1
      for (int j0 = 0; j0 < JM; ++j0)
        if (FULL || j0 < g.J[0]) cmac_fma(acc, w[0][j0], plane(j0));
    }
  }
  return acc;
}

constexpr int kFwdStageU = 8;  // staging loads in flight per thread

// One work item: tile piece wi, chunk yc of tg.CC coil rows, per-batch plan b (blockIdx
// of interp_fwd_tiled_kernel, or a batch kernel's decoded item).
template <typename T, int D, int JM>
__device__ __forceinline__ void fwd_tiled_item(const Geom<T>& g, const TileGeom& tg, const cplx<T>* __restrict__ grid,
                                               const T* __restrict__ omega, const int* __restrict__ ws,
                                               cplx<T>* __restrict__ kdata, int64_t wi, int64_t yc, int64_t b,
                                               unsigned char* smem_raw) {
  using C2 = cplx<T>;
  C2* lds = reinterpret_cast<C2*>(smem_raw);
  const int* plan = ws + b * tg.plan_ints;
  if (wi >= plan[tg.o_nwork]) return;
  const int* wstart = plan + tg.o_wstart;
  const int t = plan[tg.o_work + wi];
  const int split = (int)(wi - wstart[t]);
  const int V = plan[tg.o_start + t + 1] - plan[tg.o_start + t];  // (counts are cleared each call)
  const int i0 = split * tg.target;
  const int i1 = min(i0 + tg.target, V);
  if (i0 >= i1) return;  // empty tile: nothing to gather

  const int64_t nrows = g.batched ? g.C : g.B * g.C;
  const int64_t rowbase = g.batched ? b * g.C : 0;
  const int64_t r0 = yc * tg.CC;
  const int ncc = (int)((r0 + tg.CC < nrows ? r0 + tg.CC : nrows) - r0);

  int origin[3] = {0, 0, 0};
#pragma unroll
  for (int d = 0; d < D; ++d) origin[d] = ((t / tg.bstride[d]) % tg.nb[d]) * tg.T[d];

  // stage: lds[c * rcells + cell] = grid[row c][(origin + l) mod K], kFwdStageU loads in
  // flight per thread before their LDS stores (one load per wait would pay a memory
  // latency per element); the loads past the end read the last element again
  const int rc = tg.rcells;
  const int nstage = ncc * rc;
  auto stage_src = [&](int idx) {
    const int c = (int)fdiv(idx, tg.frc);
    int cell = idx - c * rc;
    int64_t gi = 0;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const int q = (int)fdiv(cell, tg.fR[d]);
      const int l = cell - q * tg.R[d];
      cell = q;
      int k = origin[d] + l;
      while (k >= g.K[d]) k -= g.K[d];
      gi += (int64_t)k * g.stride[d];
    }
    return grid + (rowbase + r0 + c) * g.G + gi;
  };
  for (int base = threadIdx.x; base < nstage; base += kFwdStageU * blockDim.x) {
    C2 v[kFwdStageU];
#pragma unroll
    for (int u = 0; u < kFwdStageU; ++u) v[u] = *stage_src(min(base + u * (int)blockDim.x, nstage - 1));
#pragma unroll
    for (int u = 0; u < kFwdStageU; ++u)
      if (base + u * (int)blockDim.x < nstage) lds[base + u * blockDim.x] = v[u];
  }
  __syncthreads();

  const int* perm = plan + tg.o_perm;
  const int cstart = plan[tg.o_start + t];
  const T* om = omega + (g.batched ? b * D * g.M : 0);
  bool full = true;  // every numpoints is JM: unguarded taps
#pragma unroll
  for (int d = 0; d < D; ++d) full = full && g.J[d] == JM;
  for (int i = i0 + (int)threadIdx.x; i < i1; i += blockDim.x) {
    const int m = perm[cstart + i];
    C2 w[D][JM];
    int loc0[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      int mdx[JM];
      sample_taps_md<T, JM>(g, d, om[d * g.M + m], w[d], mdx);
      int l = mdx[0] - origin[d];  // base cell lies in this tile
      l = l < 0 ? 0 : (l >= tg.T[d] ? tg.T[d] - 1 : l);
      loc0[d] = l;
    }
    const T theta = sample_theta<T, D>(g, om, m);
    const C2 phase = make_c<T>(cos(theta), sin(theta));
    for (int c = 0; c < ncc; ++c) {
      const C2* L = lds + c * rc;
      const C2 acc = full ? fwd_taps<T, D, JM, true>(g, tg, L, w, loc0) : fwd_taps<T, D, JM, false>(g, tg, L, w, loc0);
      kdata[(rowbase + r0 + c) * g.M + m] = cmul(acc, phase);
    }
  }
}

template <typename T, int D, int JM>
__global__ void __launch_bounds__((fwd_tiled_threads<T, JM, D>()))
    interp_fwd_tiled_kernel(const Geom<T> g, const TileGeom tg, const cplx<T>* __restrict__ grid,
                            const T* __restrict__ omega, const int* __restrict__ ws, cplx<T>* __restrict__ kdata) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  fwd_tiled_item<T, D, JM>(g, tg, grid, omega, ws, kdata, blockIdx.x, blockIdx.y, blockIdx.z, smem_raw);
}

// ---------------------------------------------------------------------------
// separable kernels (2-D, complex64, J <= 6)
//   The reference's table for dimension d holds t[i] = KB(u) exp(-i pi (N-1) u / K)
//   at u = (i - J L / 2) / L (_nufft/utils.py:122-179), and the taps j of one sample
//   read t[i_0 - j L] (the float32 index arithmetic of _nufft/interp.py:129-131 gives
//   i_j = i_0 - j L except in rare rounding cases).  So along every dimension a tap
//   weight is R[i_j] (the real KB value) times a factor B shared by the sample's taps
//   in one tile, times P(k) = exp(i pi (N-1) k / K) of the tap's cell k.  The kernels
//   work on the grid multiplied by P_0 P_1 (the forward stages its tile rotated; the
//   adjoint rotates its tile accumulator back when it flushes), with real tap weights:
//   two FMAs per tap and coil row instead of four.  Entries whose taps break the form
//   (a table of another form, N unknown, a non-finite sample, or a rounding case) are
//   flagged by the plan and applied with complex weights in the rotated frame, so the
//   result is the reference's for every table.
//   Every phase of the frame is evaluated in double and rounded once at the end: with float
//   phases the results of few-row problems were further from 64-bit sums than those of the
//   complex-weight kernels (12 rows, 256^2 adjoint, sums in float32: 1.26e-7 against 1.12e-7,
//   with double phases 1.07e-7).
// ---------------------------------------------------------------------------
struct SepGeom {
  int L[2];            // table oversampling
  // int offsets of what the trajectories of a call share (behind their plans):
  int64_t o_rtab[2];   // the real tables
  int64_t o_ptab[2];   // the cell phases P_d(k), k < K_d (double2)
  int64_t o_nm1;       // N_d - 1 (2 ints), found from the tables
  int64_t o_flag;      // set where a table is not of the form
  int64_t end;         // ints of the plans and this in all
};

// N - 1 of the table's phase, read off its first entry past the centre:
// t[c + 1] = KB(1 / L) exp(-i pi (N - 1) / (K L)), so N - 1 = -arg(t[c + 1]) K L / pi
// (the float32 argument is good to far better than one unit of N - 1); the plan then
// checks every entry against the form, so a wrong estimate only costs speed.
__device__ __forceinline__ int sep_nm1_estimate(const Geom<float>& g, int d) {
  const float2 t = g.table[d][g.center[d] + 1];
  const double ang = (double)atan2f(t.y, t.x);
  return (int)llrint(-ang * (double)g.K[d] * g.Lf[d] / 3.141592653589793);
}

// exp(i pi a / q) for an integer a of any sign and q > 0; a is reduced modulo 2q first.
// In double: a float angle in [0, 2 pi) is off by up to 1.9e-7, which was the largest error
// of the rotated frame (only plans evaluate phases).
__device__ __forceinline__ double2 pi_phase_d(int64_t a, int64_t q) {
  int64_t r = a % (2 * q);
  if (r < 0) r += 2 * q;
  double s, c;
  sincospi((double)r / (double)q, &s, &c);
  return make_double2(c, s);
}

// P(p) = exp(i pi (N - 1) p / K) for a cell coordinate p >= 0 that may run past the
// grid's end (the gather's staged halo): P(p) = P(p - K) (-1)^(N - 1), from the plan's
// table of P(k), k < K.
__device__ __forceinline__ float2 sep_cell_phase(const double2* P, int K, int nm1, int p) {
  bool flip = false;
  while (p >= K) {
    p -= K;
    flip = flip != ((nm1 & 1) != 0);
  }
  const double2 v = P[p];
  return flip ? make_float2((float)-v.x, (float)-v.y) : make_float2((float)v.x, (float)v.y);
}

// Plan record of one sample (64 bytes).  The forward keeps them in tile order; the adjoint,
// whose samples have an entry in every tile that they reach, in sample order, and lists a
// tile's samples in perm (80 bytes a sample; a record per entry took up to 272, and was
// written 1.7 times).
struct SepRec {
  int me;      // forward: sample index; adjoint: first cell of the footprint along dimension 0;
               // exception flag << 31
  int rc;      // forward: base cell relative to the tile, (p0 + 8) | (p1 + 8) << 8; adjoint:
               // first cell along dimension 1
  float2 F;    // forward: shift phase * B_0 * B_1 (exceptions: the shift phase alone);
               // adjoint: the conjugate, for the wrapped footprint's first cell
  float w0[6]; // R_0 of taps 0..5 along dimension 0
  float w1[6]; // R_1 along dimension 1
};
static_assert(sizeof(SepRec) == 64, "plan record is 64 bytes");


// Exact reference arithmetic of one sample along dimension d: the unwrapped base cell,
// the table index of tap 0, and whether every tap j < J uses index i_0 - j L.
struct SepTaps {
  int64_t base;
  int ti0;
  bool regular;
};
__device__ __forceinline__ SepTaps sep_taps(const Geom<float>& g, int d, float omega) {
#pragma clang fp contract(off)
  SepTaps r;
  const float tm = omega / g.gam[d];
  const bool ok = fabsf(tm) < 1.0e15f;
  const float fb = floorf(tm - g.halfJ[d]);
  r.base = ok ? (int64_t)fb + 1 : 0;
  r.regular = ok;
  r.ti0 = 0;
  const int L = (int)g.Lf[d];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    if (j < g.J[d]) {
      const float u = tm - (float)(r.base + j);
      int ti = (int)rintf(u * g.Lf[d]) + g.center[d];
      ti = ti < 0 ? 0 : (ti > g.tmax[d] ? g.tmax[d] : ti);
      if (j == 0) r.ti0 = ti;
      else r.regular = r.regular && ti == r.ti0 - j * L;
    }
  }
  return r;
}

// Table weight of tap j along dimension d exactly as the reference indexes it (NaN
// for a non-finite sample), for the complex-weight entries.
__device__ __forceinline__ float2 sep_tap_weight(const Geom<float>& g, int d, float omega, int j) {
#pragma clang fp contract(off)
  const float tm = omega / g.gam[d];
  if (!(fabsf(tm) < 1.0e15f)) return make_float2(NAN, NAN);
  if (j >= g.J[d]) return make_float2(0.f, 0.f);
  const int64_t base = (int64_t)floorf(tm - g.halfJ[d]) + 1;
  const float u = tm - (float)(base + j);
  int ti = (int)rintf(u * g.Lf[d]) + g.center[d];
  ti = ti < 0 ? 0 : (ti > g.tmax[d] ? g.tmax[d] : ti);
  return g.table[d][ti];
}

// Angle of a tap's phase B_d = exp(-i pi (N-1) n / (L K)) over pi, n = (i_0 - J L / 2) + L p
// (p: tap 0's cell in the tile frame), reduced modulo 2
__device__ __forceinline__ double sep_turn(const Geom<float>& g, const SepGeom& sg, int nm1, int d, int ti0, int64_t p) {
  const int64_t q = (int64_t)sg.L[d] * g.K[d];
  return (double)((int64_t)nm1 * ((int64_t)(ti0 - g.center[d]) + (int64_t)sg.L[d] * p) % (2 * q)) / (double)q;
}
// exp(i (theta - pi turns)), evaluated in double and rounded once
__device__ __forceinline__ float2 sep_factor(float theta, double turns) {
  double s, c;
  sincos((double)theta - turns * 3.14159265358979323846, &s, &c);
  return make_float2((float)c, (float)s);
}

// Real tables R_d[i] = Re(t_d[i] exp(i pi (N-1)(i - J L / 2) / (L K))) and cell phases, once
// for all trajectories (the blocks of the first one; 12 000 values in double for the usual
// tables); sets the flag when any imaginary part is not negligible (the table does not have
// the form, or N is unknown for a complex table).  Grid-stride over both tables.
__device__ __forceinline__ void sep_table_prep(const Geom<float>& g, const SepGeom& sg, int* tabs) {
  if (blockIdx.y != 0) return;
  const int nm1[2] = {sep_nm1_estimate(g, 0), sep_nm1_estimate(g, 1)};
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    tabs[sg.o_nm1] = nm1[0];
    tabs[sg.o_nm1 + 1] = nm1[1];
  }
  const int64_t n0 = g.tmax[0] + 1, n1 = g.tmax[1] + 1;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n0 + n1;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int d = i < n0 ? 0 : 1;
    const int m = (int)(d == 0 ? i : i - n0);
    const float2 t = g.table[d][m];
    const double2 p = pi_phase_d((int64_t)nm1[d] * (m - g.center[d]), (int64_t)sg.L[d] * g.K[d]);
    const float re = (float)((double)t.x * p.x - (double)t.y * p.y);
    const float im = (float)((double)t.x * p.y + (double)t.y * p.x);
    reinterpret_cast<float*>(tabs + sg.o_rtab[d])[m] = re;
    if (!(fabsf(im) <= 0x1p-19f * (fabsf(t.x) + fabsf(t.y)))) atomicOr(tabs + sg.o_flag, 1);
  }
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (int64_t)g.K[0] + g.K[1];
       i += (int64_t)gridDim.x * blockDim.x) {
    const int d = i < g.K[0] ? 0 : 1;
    const int k = (int)(d == 0 ? i : i - g.K[0]);
    reinterpret_cast<double2*>(tabs + sg.o_ptab[d])[k] = pi_phase_d((int64_t)nm1[d] * k, g.K[d]);
  }
}

// ---- plans -------------------------------------------------------------------------
__device__ __forceinline__ void sep_gat_record(const Geom<float>& g, const TileGeom& tg, const SepGeom& sg,
                                               const float* __restrict__ omega, int* __restrict__ plan,
                                               const int* __restrict__ tabs, int m, int key,
                                               const int (&l)[2], int pos);
__device__ __forceinline__ void sep_spr_scatter_item(const Geom<float>& g, const TileGeom& tg, const SepGeom& sg,
                                                     const float* __restrict__ omega, int* __restrict__ plan,
                                                     const int* __restrict__ tabs, int m);

// Scan of per-tile counts into tile starts and the work list, longest work first: tiles
// above `target` entries, cut into pieces of `target`, then the others by size class (above
// 1/2, 1/4, 1/8 of the target, the rest), so that no long tile starts late (16 coils x 4,
// 320^2 radial: the spread's waves were 1.2 per SIMD on average with the tiles in grid
// order, 2 fit).  Empty tiles get no item when `skip_empty`.
// One block does it, so it is bound by its own chain of loads and barriers: one pass adds the
// classes up, one scans entries, pieces and classes together, 2048 tiles a round, the next
// round's counts loaded ahead (16384 tiles, 4000 samples: the count kernel with its scan 65 us,
// 368 with a block scan each of entries, pieces and four classes; 1024 tiles, 206 k samples: 39
// and 62 us).
constexpr int kSepClasses = 4;
constexpr int kScanTiles = 8;  // tiles of a thread per round
struct SepSums {
  int ent, pieces;
  unsigned long long cls;  // classes 1 .. 4, 16 bits each (a round has at most 2048 tiles)
};
__device__ __forceinline__ SepSums sep_add(SepSums a, SepSums b) {
  return SepSums{a.ent + b.ent, a.pieces + b.pieces, a.cls + b.cls};
}
struct SepScanLds {
  SepSums wave[4];
  int total[kSepClasses + 1];
};
__device__ __forceinline__ void sep_plan_scan(const TileGeom& tg, int* __restrict__ plan, bool skip_empty,
                                              SepScanLds& lds) {
  const int target = tg.target, NB = tg.NB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;  // 256 threads
  const int* count = plan + tg.o_count;
  int* start = plan + tg.o_start;
  int* cursor = plan + tg.o_cursor;
  int* wstart = plan + tg.o_wstart;
  int* work = plan + tg.o_work;
  const auto size_class = [&](int v) {  // 0: split; kSepClasses + 1: no item
    if (v > target) return 0;
    if (v == 0 && skip_empty) return kSepClasses + 1;
    return 2 * v > target ? 1 : 4 * v > target ? 2 : 8 * v > target ? 3 : 4;
  };
  const auto sums_of = [&](int v) {
    const int c = size_class(v);
    return SepSums{v, c == 0 ? (int)fdiv(v + target - 1, tg.ftarget) : 0, c >= 1 && c <= kSepClasses ? 1ull << (16 * (c - 1)) : 0ull};
  };
  if (tid <= kSepClasses) lds.total[tid] = 0;
  __syncthreads();
  int mine[kSepClasses + 1] = {0, 0, 0, 0, 0};
  for (int t0 = tid; t0 < NB; t0 += kScanTiles * 256) {
    int v[kScanTiles];
    SepSums a{0, 0, 0};
#pragma unroll
    for (int i = 0; i < kScanTiles; ++i) v[i] = count[min(t0 + i * 256, NB - 1)];
#pragma unroll
    for (int i = 0; i < kScanTiles; ++i)
      if (t0 + i * 256 < NB) a = sep_add(a, sums_of(v[i]));
    mine[0] += a.pieces;
#pragma unroll
    for (int c = 0; c < kSepClasses; ++c) mine[c + 1] += (int)((a.cls >> (16 * c)) & 0xffff);
  }
#pragma unroll
  for (int c = 0; c <= kSepClasses; ++c) {
    for (int off = 32; off > 0; off >>= 1) mine[c] += __shfl_down(mine[c], off, 64);
    if (lane == 0 && mine[c] != 0) atomicAdd(&lds.total[c], mine[c]);
  }
  __syncthreads();
  // next item of each class, entries so far
  int next[kSepClasses + 1], ent = 0;
  next[0] = 0;
#pragma unroll
  for (int c = 1; c <= kSepClasses; ++c) next[c] = next[c - 1] + lds.total[c - 1];
  const int cap = (int)tg.maxwork;
  if (tid == 0) plan[tg.o_nwork] = min(next[kSepClasses] + lds.total[kSepClasses], cap);

  int ahead[kScanTiles];  // the next round's counts
#pragma unroll
  for (int i = 0; i < kScanTiles; ++i) ahead[i] = count[min(kScanTiles * tid + i, NB - 1)];
  for (int t0 = 0; t0 < NB; t0 += kScanTiles * 256) {
    const int t = t0 + kScanTiles * tid;
    int v[kScanTiles];
    SepSums sum{0, 0, 0};
#pragma unroll
    for (int i = 0; i < kScanTiles; ++i) {
      v[i] = ahead[i];
      ahead[i] = count[min(t + kScanTiles * 256 + i, NB - 1)];
    }
#pragma unroll
    for (int i = 0; i < kScanTiles; ++i)
      if (t + i < NB) sum = sep_add(sum, sums_of(v[i]));
    SepSums incl = sum;
    for (int off = 1; off < 64; off <<= 1) {
      const SepSums o{__shfl_up(incl.ent, off, 64), __shfl_up(incl.pieces, off, 64), __shfl_up(incl.cls, off, 64)};
      if (lane >= off) incl = sep_add(incl, o);
    }
    if (lane == 63) lds.wave[wave] = incl;
    __syncthreads();
    SepSums run{incl.ent - sum.ent, incl.pieces - sum.pieces, incl.cls - sum.cls}, all{0, 0, 0};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wave) run = sep_add(run, lds.wave[w]);
      all = sep_add(all, lds.wave[w]);
    }
    __syncthreads();  // the next round overwrites the waves' sums
#pragma unroll
    for (int i = 0; i < kScanTiles; ++i) {
      if (t + i < NB) {
        const int c = size_class(v[i]);
        const SepSums one = sums_of(v[i]);
        start[t + i] = cursor[t + i] = ent + run.ent;
        int at = 0;  // (a select each: an indexed register array would go through memory)
#pragma unroll
        for (int k = 0; k <= kSepClasses; ++k)
          if (c == k) at = next[k] + (k == 0 ? run.pieces : (int)((run.cls >> (16 * (k - 1))) & 0xffff));
        if (c <= kSepClasses) {
          wstart[t + i] = at;
          const int e = min(at + (c == 0 ? one.pieces : 1), cap);
          for (int w = at; w < e; ++w) work[w] = t + i;
        }
        run = sep_add(run, one);
      }
    }
    ent += all.ent;
    next[0] += all.pieces;
#pragma unroll
    for (int k = 1; k <= kSepClasses; ++k) next[k] += (int)((all.cls >> (16 * (k - 1))) & 0xffff);
  }
  if (tid == 0) start[NB] = ent;
}

// The count kernels' end: the last block of a trajectory to finish scans its counts (its
// own launch for the scan cost 5 us of every call, also where the plan is kept).  The
// counts are device-scope atomics, and each wave waits for its own before its block signs
// off; nothing else is read here (a release fence by every block wrote the L2 back 800
// times: 69 instead of 62 us for 206 000 new samples).
__device__ __forceinline__ void sep_scan_if_last(const TileGeom& tg, int* __restrict__ plan, bool skip_empty) {
  __shared__ SepScanLds lds;
  __shared__ bool last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) last = atomicAdd(plan + tg.o_count + tg.NB, 1) == (int)gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  __threadfence();
  sep_plan_scan(tg, plan, skip_empty, lds);
}

// Forward: each sample once, in the 16 x 16 tile of its base cell (trajectory order
// within a tile as far as the building atomics keep it); count[NB] counts finished blocks.
// blockIdx.y: the trajectory (one plan each).
__global__ void __launch_bounds__(256)
    sep_gat_count_kernel(const Geom<float> g, const TileGeom tg, const SepGeom sg, const float* __restrict__ omega,
                         int* __restrict__ ws, const CacheHdr* cache) {
  if (cache_hit(cache)) return;  // cached plan reused
  sep_table_prep(g, sg, ws);
  omega += (int64_t)blockIdx.y * 2 * g.M;
  ws += (int64_t)blockIdx.y * tg.plan_stride;
  for (int m0 = blockIdx.x * blockDim.x; m0 < g.M; m0 += gridDim.x * blockDim.x) {
    const int m = m0 + threadIdx.x;
    const bool live = m < g.M;
    int l[2];
    const int key = live ? gat_base_tile(g, tg, omega, m, l) : 0;
    wave_aggregated_add(ws + tg.o_count, key, live);
  }
  sep_scan_if_last(tg, ws, true);
}

__global__ void __launch_bounds__(256)
    sep_gat_scatter_kernel(const Geom<float> g, const TileGeom tg, const SepGeom sg, const float* __restrict__ omega,
                           int* __restrict__ ws, const CacheHdr* cache) {
  if (cache_hit(cache)) return;  // cached plan reused
  omega += (int64_t)blockIdx.y * 2 * g.M;
  int* const plan = ws + (int64_t)blockIdx.y * tg.plan_stride;
  for (int m0 = blockIdx.x * blockDim.x; m0 < g.M; m0 += gridDim.x * blockDim.x) {
    const int m = m0 + threadIdx.x;
    const bool live = m < g.M;
    int l[2] = {0, 0};
    const int key = live ? gat_base_tile(g, tg, omega, m, l) : 0;
    const int pos = wave_aggregated_inc(plan + tg.o_cursor, key, live);
    if (live) sep_gat_record(g, tg, sg, omega, plan, ws, m, key, l, pos);
  }
}

// the forward record of sample m (tile `key`, base cell l inside it) at plan position pos
__device__ __forceinline__ void sep_gat_record(const Geom<float>& g, const TileGeom& tg, const SepGeom& sg,
                                               const float* __restrict__ omega, int* __restrict__ plan,
                                               const int* __restrict__ tabs, int m, int key,
                                               const int (&l)[2], int pos) {
  const bool tab_ok = tabs[sg.o_flag] == 0;
  const int nm10 = tabs[sg.o_nm1], nm11 = tabs[sg.o_nm1 + 1];
  const float om0 = omega[m], om1 = omega[g.M + m];
  const SepTaps a = sep_taps(g, 0, om0), b = sep_taps(g, 1, om1);
  const float theta = sample_theta<float, 2>(g, omega, m);
  double turns = 0.;
  SepRec rec;
  const bool exc = !(tab_ok && a.regular && b.regular);
  const float* R0 = reinterpret_cast<const float*>(tabs + sg.o_rtab[0]);
  const float* R1 = reinterpret_cast<const float*>(tabs + sg.o_rtab[1]);
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    rec.w0[j] = (!exc && j < g.J[0]) ? R0[a.ti0 - j * sg.L[0]] : 0.f;
    rec.w1[j] = (!exc && j < g.J[1]) ? R1[b.ti0 - j * sg.L[1]] : 0.f;
  }
  if (!exc) {
    // tap 0's cell in the tile frame is the wrapped base (the staged region continues
    // past the grid's end without wrapping its coordinates)
    const int o0 = (key / tg.bstride[0]) % tg.nb[0] * kGatT0, o1 = (key / tg.bstride[1]) % tg.nb[1] * kGatT1;
    turns = sep_turn(g, sg, nm10, 0, a.ti0, o0 + l[0]) + sep_turn(g, sg, nm11, 1, b.ti0, o1 + l[1]);
  }
  rec.me = m | (exc ? (int)0x80000000u : 0);
  rec.rc = (l[0] + 8) | ((l[1] + 8) << 8);
  rec.F = sep_factor(theta, turns);
  reinterpret_cast<SepRec*>(reinterpret_cast<char*>(plan) + tg.o_rec_bytes)[pos] = rec;
}

// Adjoint: one entry per (sample, 16 x 16 tile its footprint meets), count[NB] as above.  The
// sample index goes to perm; the record, with the exception flag, to the same position or (not
// rec_entry) to the sample's.
__global__ void __launch_bounds__(256)
    sep_spr_count_kernel(const Geom<float> g, const TileGeom tg, const SepGeom sg, const float* __restrict__ omega,
                         int* __restrict__ ws, const CacheHdr* cache) {
  if (cache_hit(cache)) return;  // cached plan reused
  sep_table_prep(g, sg, ws);
  omega += (int64_t)blockIdx.y * 2 * g.M;
  ws += (int64_t)blockIdx.y * tg.plan_stride;
  for (int m0 = blockIdx.x * blockDim.x; m0 < g.M; m0 += gridDim.x * blockDim.x) {
    const int m = m0 + threadIdx.x;
    const bool live = m < g.M;
    int tl[2][3], off[2][3], n[2];
    coil_sample_tiles(g, tg, omega, m, live, tl, off, n);
    int* count = ws + tg.o_count;
    coil_for_each_entry(tg, tl, off, n, live, [&](int key, int, int c, bool valid) {
      const int tkey = valid ? (key - (off[1][c] - kRegMinC0)) / kRegKeys : 0;
      wave_aggregated_add(count, tkey, valid);
    });
  }
  sep_scan_if_last(tg, ws, false);
}

// Zeroes tile t of rows [r0, r1) if its pieces add into the grid
__device__ __forceinline__ void sep_zero_hot_item(const Geom<float>& g, const TileGeom& tg, const int* plan,
                                                  float2* __restrict__ grid, int t, int64_t r0, int64_t r1);

// Blocks x < nscatter write the records of a new plan (trajectory blockIdx.y), the others
// clear what the spread adds into, on every call: block nscatter + t + NB * y, tile t and
// rows [64 y, 64 y + 64).
__global__ void __launch_bounds__(256)
    sep_spr_scatter_kernel(const Geom<float> g, const TileGeom tg, const SepGeom sg, const float* __restrict__ omega,
                           int* __restrict__ ws, const CacheHdr* cache, int nscatter, float2* __restrict__ grid) {
  if ((int)blockIdx.x >= nscatter) {
    const int64_t b = blockIdx.y;
    const int x = (int)blockIdx.x - nscatter, y = x / tg.NB;
    const int64_t nrows = g.batched ? g.C : g.B * g.C, rowbase = g.batched ? b * g.C : 0;
    const int64_t r0 = (int64_t)y * 64;
    const int64_t r1 = r0 + 64 < nrows ? r0 + 64 : nrows;
    sep_zero_hot_item(g, tg, ws + b * tg.plan_stride, grid, x - y * tg.NB, rowbase + r0, rowbase + r1);
    return;
  }
  if (cache_hit(cache)) return;  // cached plan reused
  omega += (int64_t)blockIdx.y * 2 * g.M;
  int* const plan = ws + (int64_t)blockIdx.y * tg.plan_stride;
  for (int m0 = blockIdx.x * blockDim.x; m0 < g.M; m0 += nscatter * blockDim.x)
    sep_spr_scatter_item(g, tg, sg, omega, plan, ws, m0 + threadIdx.x);
}

// the adjoint's record and entries of sample m (m >= M: a dead lane that still takes part in the
// wave-aggregated cursor increments)
__device__ __forceinline__ void sep_spr_scatter_item(const Geom<float>& g, const TileGeom& tg, const SepGeom& sg,
                                                     const float* __restrict__ omega, int* __restrict__ plan,
                                                     const int* __restrict__ tabs, int m) {
  const bool live = m < g.M;
  int tl[2][3], off[2][3], n[2];
  coil_sample_tiles(g, tg, omega, m, live, tl, off, n);
  SepTaps a{}, b{};
  float theta = 0.f;
  bool regular = false;
  if (live) {
    a = sep_taps(g, 0, omega[m]);
    b = sep_taps(g, 1, omega[g.M + m]);
    theta = sample_theta<float, 2>(g, omega, m);
    regular = tabs[sg.o_flag] == 0 && a.regular && b.regular;
  }
  const float* R0 = reinterpret_cast<const float*>(tabs + sg.o_rtab[0]);
  const float* R1 = reinterpret_cast<const float*>(tabs + sg.o_rtab[1]);
  const int nm10 = tabs[sg.o_nm1], nm11 = tabs[sg.o_nm1 + 1];
  SepRec* recs = reinterpret_cast<SepRec*>(reinterpret_cast<char*>(plan) + tg.o_rec_bytes);
  const int c0 = live ? (int)sample_base_wrapped<float>(g, 0, omega[m]) : 0;
  const int c1 = live ? (int)sample_base_wrapped<float>(g, 1, omega[g.M + m]) : 0;
  SepRec rec;
  const float2 F = sep_factor(
      theta, regular ? sep_turn(g, sg, nm10, 0, a.ti0, c0) + sep_turn(g, sg, nm11, 1, b.ti0, c1) : 0.);
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    rec.w0[j] = (regular && j < g.J[0]) ? R0[a.ti0 - j * sg.L[0]] : 0.f;
    rec.w1[j] = (regular && j < g.J[1]) ? R1[b.ti0 - j * sg.L[1]] : 0.f;
  }
  rec.me = c0 | (regular ? 0 : (int)0x80000000u);
  rec.rc = c1;
  rec.F = make_float2(F.x, -F.y);
  coil_for_each_entry(tg, tl, off, n, live, [&](int key, int, int c, bool valid) {
    const int tkey = valid ? (key - (off[1][c] - kRegMinC0)) / kRegKeys : 0;
    const int pos = wave_aggregated_inc(plan + tg.o_cursor, tkey, valid);
    if (!valid) return;
    plan[tg.o_perm + pos] = m;
    if (tg.rec_entry) recs[pos] = rec;
  });
  if (live && !tg.rec_entry) recs[m] = rec;
}

// ---- forward gather ------------------------------------------------------------------
// A group per 16 x 16 tile, piece and chunk of ROWS coil rows; the tile and its halo are
// staged in LDS with the coil row fastest, rotated: region = grid * P_0 * P_1; ROWS lanes
// per entry compute
//   y = F * sum_i w0[i] sum_j w1[j] region[l0 + i][l1 + j]
// with real w0, w1; exception entries use the table's complex weights and the cells
// rotated back.
// ROWS: 16 from 9 coil rows on (the records are read once per 16 rows), else the smallest of
// 8, 4, 2, 1 that holds them: fewer idle lanes, and 64 / ROWS entries share a wave.
template <int ROWS>
struct GatShape {
  static constexpr int kPitch = ROWS > 1 ? ROWS + 1 : 1;  // float2 per staged cell (odd: stores spread over banks)
  static constexpr int kThreads = ROWS == 16 ? 512 : 256;
};

template <int ROWS>
__device__ __forceinline__ float2 sep_gat_real(const float (&w0)[6], const float (&w1)[6], const float2* L0, int J0,
                                               int J1, bool fixed6) {
  constexpr int kPitch = GatShape<ROWS>::kPitch;
  if (fixed6) {
    // J = 6: all 36 taps are read before any is used (a scheduling barrier keeps the
    // sums behind the reads, so the LDS latency is paid once per entry)
    float2 X[6][6];
#pragma unroll
    for (int j0 = 0; j0 < 6; ++j0)
#pragma unroll
      for (int j1 = 0; j1 < 6; ++j1) X[j0][j1] = L0[j0 * (kGatR1 * kPitch) + j1 * kPitch];
    __builtin_amdgcn_sched_barrier(0);
    float2 acc = make_float2(0.f, 0.f);
#pragma unroll
    for (int j0 = 0; j0 < 6; ++j0) {
      float2 p = make_float2(0.f, 0.f);
#pragma unroll
      for (int j1 = 0; j1 < 6; ++j1) {
        p.x = fmaf(w1[j1], X[j0][j1].x, p.x);
        p.y = fmaf(w1[j1], X[j0][j1].y, p.y);
      }
      acc.x = fmaf(w0[j0], p.x, acc.x);
      acc.y = fmaf(w0[j0], p.y, acc.y);
    }
    return acc;
  }
  float2 acc = make_float2(0.f, 0.f);
#pragma unroll
  for (int j0 = 0; j0 < 6; ++j0) {
    if (j0 < J0) {
      const float2* L = L0 + j0 * (kGatR1 * kPitch);
      float2 p = make_float2(0.f, 0.f);
#pragma unroll
      for (int j1 = 0; j1 < 6; ++j1) {
        if (j1 < J1) {
          const float2 x = L[j1 * kPitch];
          p.x = fmaf(w1[j1], x.x, p.x);
          p.y = fmaf(w1[j1], x.y, p.y);
        }
      }
      acc.x = fmaf(w0[j0], p.x, acc.x);
      acc.y = fmaf(w0[j0], p.y, acc.y);
    }
  }
  return acc;
}

// exception entry: the table's weights on the cells rotated back by conj(P_0 P_1)
template <int ROWS>
__device__ __forceinline__ float2 sep_gat_complex(const Geom<float>& g, float om0, float om1, const float2* L0,
                                                  const float2* p0, const float2* p1) {
  constexpr int kPitch = GatShape<ROWS>::kPitch;
  float2 acc = make_float2(0.f, 0.f);
  for (int j0 = 0; j0 < g.J[0]; ++j0) {
    const float2* L = L0 + j0 * (kGatR1 * kPitch);
    float2 p = make_float2(0.f, 0.f);
    for (int j1 = 0; j1 < g.J[1]; ++j1) cmac(p, sep_tap_weight(g, 1, om1, j1), cmul_conj(L[j1 * kPitch], p1[j1]));
    cmac(acc, sep_tap_weight(g, 0, om0, j0), cmul_conj(p, p0[j0]));
  }
  return acc;
}

// One work item: tile piece wi, chunk of ROWS coil rows; `plan`, `omega` and rows
// [rowbase, rowbase + nrows) belong to one trajectory, `tabs` to all.  `region`: kGatCells * kPitch cells,
// `ph`: the phases P_0 of the region's rows and P_1 of its columns.
template <int JF, int ROWS>
__device__ __forceinline__ void gather_sep_item(const Geom<float>& g, const TileGeom& tg, const SepGeom& sg,
                                                const float2* __restrict__ grid, const float* __restrict__ omega,
                                                const int* plan, const int* tabs, float2* kdata, int64_t rowbase,
                                                int64_t nrows, int64_t wi, int chunk, float2* region, float2* ph) {
  constexpr int kPitch = GatShape<ROWS>::kPitch, kThreads = GatShape<ROWS>::kThreads;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int slot = lane / ROWS, row = lane % ROWS;  // entry slot, coil row
  if (wi >= plan[tg.o_nwork]) return;
  const int t = plan[tg.o_work + wi];
  const int split = (int)(wi - plan[tg.o_wstart + t]);
  const int V = plan[tg.o_start + t + 1] - plan[tg.o_start + t];
  const int i0 = split * tg.target;
  const int i1 = min(i0 + tg.target, V);
  if (i0 >= i1) return;
  const int64_t rbase = (int64_t)chunk * ROWS;
  const int ncc = (int)((rbase + ROWS < nrows ? rbase + ROWS : nrows) - rbase);
  const int64_t row0 = rowbase + rbase;
  const int o0 = ((t / tg.bstride[0]) % tg.nb[0]) * kGatT0;
  const int o1 = ((t / tg.bstride[1]) % tg.nb[1]) * kGatT1;
  float2* const p0 = ph;
  float2* const p1 = ph + kGatR0;
  const auto phases = [&](int i) {  // i-th of the kGatR0 + kGatR1 phases
    const int d = i < kGatR0 ? 0 : 1;
    const int nm1 = tabs[sg.o_nm1 + d];
    const double2* P = reinterpret_cast<const double2*>(tabs + sg.o_ptab[d]);
    ph[i] = sep_cell_phase(P, g.K[d], nm1, d == 0 ? o0 + i : o1 + i - kGatR0);
  };

  if constexpr (ROWS == 16) {
    // Stage: thread (coil row sr, region column sl1) of the first 16 x 21 threads loads
    // that column's 21 region rows (consecutive threads read consecutive grid columns;
    // the row index steps by one and wraps), while the other threads look up the phases;
    // then every loaded value is stored rotated.
    constexpr int kStageThreads = ROWS * kGatR1;  // 336
    static_assert(kStageThreads + kGatR0 + kGatR1 <= kThreads, "spare threads look up the phases");
    const int sr = (int)threadIdx.x / kGatR1, sl1 = (int)threadIdx.x - sr * kGatR1;
    float2 v[kGatR0];
    if ((int)threadIdx.x < kStageThreads) {
      int k1 = o1 + sl1;
      while (k1 >= g.K[1]) k1 -= g.K[1];
      int k0 = o0;  // a tile origin lies inside the grid
      const bool live = sr < ncc;
      const float2* src = grid + (row0 + (live ? sr : 0)) * g.G + k1;
#pragma unroll
      for (int l0 = 0; l0 < kGatR0; ++l0) {
        v[l0] = live ? src[(int64_t)k0 * g.stride[0]] : make_float2(0.f, 0.f);
        k0 = k0 + 1 == g.K[0] ? 0 : k0 + 1;
      }
    } else if ((int)threadIdx.x - kStageThreads < kGatR0 + kGatR1) {
      phases((int)threadIdx.x - kStageThreads);
    }
    lds_barrier();
    if ((int)threadIdx.x < kStageThreads) {
      const float2 pc = p1[sl1];
#pragma unroll
      for (int l0 = 0; l0 < kGatR0; ++l0)
        region[(l0 * kGatR1 + sl1) * kPitch + sr] = cmul(v[l0], cmul(p0[l0], pc));
    }
  } else {
    // cell by cell: all of a thread's loads in flight before their stores
    constexpr int kN = ROWS * kGatCells, kU = (kN + kThreads - 1) / kThreads;
    float2 v[kU];
    const auto place = [&](int i, int& r, int& l0, int& l1) {
      r = i / kGatCells;
      const int c = i - r * kGatCells;
      l0 = c / kGatR1;
      l1 = c - l0 * kGatR1;
    };
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      int r, l0, l1;
      place(min((int)threadIdx.x + u * kThreads, kN - 1), r, l0, l1);
      int k0 = o0 + l0, k1 = o1 + l1;
      while (k0 >= g.K[0]) k0 -= g.K[0];
      while (k1 >= g.K[1]) k1 -= g.K[1];
      v[u] = grid[(row0 + min(r, ncc - 1)) * g.G + (int64_t)k0 * g.stride[0] + k1];
    }
    if ((int)threadIdx.x < kGatR0 + kGatR1) phases((int)threadIdx.x);
    lds_barrier();
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      int r, l0, l1;
      const int i = (int)threadIdx.x + u * kThreads;
      place(min(i, kN - 1), r, l0, l1);
      if (i < kN) region[(l0 * kGatR1 + l1) * kPitch + r] = cmul(v[u], cmul(p0[l0], p1[l1]));
    }
  }
  __syncthreads();

  // Records one entry ahead, alternating between two register sets (unconditional,
  // clamped loads).  Slot h of wave w takes entries i0 + kPer w + h, stepping by kStep.
  constexpr int kPer = 64 / ROWS, kStep = kPer * (kThreads / 64);
  const float4* recs = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(plan) + tg.o_rec_bytes) +
                       (int64_t)plan[tg.o_start + t] * 4;
  const int J0 = g.J[0], J1 = g.J[1];
  float4 ra[4], rb[4];
  auto load_rec = [&](float4 (&r)[4], int e) {
    const int ec = e < i1 ? e : i1 - 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = recs[(int64_t)ec * 4 + q];
  };
  auto finish = [&](const float4 (&r)[4], int e) {
    if (e < i1) {
      const int me = __float_as_int(r[0].x), rc = __float_as_int(r[0].y);
      const int m = me & 0x7fffffff;
      const int l0 = (rc & 255) - 8, l1 = ((rc >> 8) & 255) - 8;
      const float2 F = make_float2(r[0].z, r[0].w);
      const float2* L0 = region + (l0 * kGatR1 + l1) * kPitch + row;
      float2 acc;
      if (me >= 0) {
        const float w0[6] = {r[1].x, r[1].y, r[1].z, r[1].w, r[2].x, r[2].y};
        const float w1[6] = {r[2].z, r[2].w, r[3].x, r[3].y, r[3].z, r[3].w};
        acc = sep_gat_real<ROWS>(w0, w1, L0, J0, J1, JF == 6);
      } else {
        acc = sep_gat_complex<ROWS>(g, omega[m], omega[g.M + m], L0, p0 + l0, p1 + l1);
      }
      if (row < ncc) kdata[(row0 + row) * g.M + m] = cmul(acc, F);
    }
  };
  load_rec(ra, i0 + kPer * wave + slot);
  for (int eb = i0 + kPer * wave; eb < i1; eb += 2 * kStep) {
    const int e = eb + slot;
    load_rec(rb, e + kStep);
    finish(ra, e);
    load_rec(ra, e + 2 * kStep);
    finish(rb, e + kStep);
  }
}

template <int JF, int ROWS>
__global__ void __launch_bounds__(GatShape<ROWS>::kThreads)
    gather_sep_kernel(const Geom<float> g, const TileGeom tg, const SepGeom sg, const float2* __restrict__ grid,
                      const float* __restrict__ omega, const int* ws, float2* kdata, int nchunk) {
  __shared__ __attribute__((aligned(16))) float2 region[kGatCells * GatShape<ROWS>::kPitch];
  __shared__ float2 ph[kGatR0 + kGatR1];
  const int64_t b = blockIdx.y;  // trajectory
  const int64_t item = xcd_work_item(blockIdx.x, kXcdTiles * nchunk);
  const int64_t wi = item / nchunk;
  gather_sep_item<JF, ROWS>(g, tg, sg, grid, omega + b * 2 * g.M, ws + b * tg.plan_stride, ws, kdata,
                            g.batched ? b * g.C : 0, g.batched ? g.C : g.B * g.C, wi, (int)(item - wi * nchunk), region,
                            ph);
}

// ---- adjoint spread --------------------------------------------------------------------
// On the matrix cores: in the rotated frame every tap of an entry adds s * w0[i] * w1[j]
// with real w0, w1 (s = kdata * F), so a tile's sum over its entries is a matrix product
// with the entries as the inner dimension.  A wave takes four entries of a 16 x 16 tile per
// 16x16x4 MFMA; their weights and data pass through its own part of LDS, without
// work-group barriers.  A tile (or a piece of its entries) belongs to one wave, or, where
// tiles are dense, to the four waves of a group, which split its entries and add their sums
// through LDS at the end: a tile's entries are a serial chain, and cutting it into more
// pieces would cost atomics (about 160 G lanes a second: with 128-entry pieces nearly every
// tile of a 434 x 362 grid with 130 000 entries and 39 rows was split, 153 us).
//   rows form (G = 8, 16 coil rows): per tile row r and 8 coil rows,  D_r[component][column]
//     += s[component][entry] * (w0[entry][r] w1[entry][column]); the 16 components are the
//     real and imaginary parts of the 8 rows, and tile rows that none of the four entries
//     reaches are skipped (neighbouring samples of a trajectory share most rows);
//   outer form (G = 1, 2, 4 coil rows): per row and component, D[row][column] +=
//     (w0[entry][row] s[entry]) * w1[entry][column].
// Every cell of the tile has one owner, so nothing is added atomically except the pieces of
// split tiles.  The flush multiplies each cell by conj(P_0 P_1).
// Entries with complex weights, and entries whose data are not finite (0 * inf would reach
// the whole tile), are left out of the products and added with atomics after the flush,
// tap by tap over their own footprint.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kMmBatch = 32;   // entries staged at once by a wave
constexpr int kMmWaves = 4;    // waves per work-group
constexpr int kMmWPitch = 20;  // floats per staged row of 16 weights (+4: spreads the banks, takes what falls outside)
constexpr int kMmExc = 32;     // entries left to the atomic pass that a wave remembers
// rows per chunk of a form, and waves per SIMD of its kernel
__host__ __device__ constexpr int mm_rows(int G) { return G; }
constexpr int mm_waves(int G) { return G >= 8 ? 2 : G > 2 ? 3 : 4; }
// floats per staged entry's data (two components a row; +2 spreads the banks)
constexpr int mm_spitch(int G) { return 2 * G + 2; }

// Sums.  Chunks of up to 8 rows: in double, on the float64 MFMA (half the float32 rate), the
// weights' products too, so that a cell is rounded once however many entries it meets, as with
// the 64-bit integer sums of the sample-lane kernel.  Against 64-bit sums of random data, 900
// samples in one tile: 6.0e-8, the integer sums 6.8e-8; float32 chains of 32 entries added up
// in double 8.4e-8, one float32 chain 1.6e-7 (and 4e-7 on a cell of one-sign data, now 6e-8).
// 256^2, 402 x 512 radial, adjoint interpolation of 1 / 8 / 12 rows: 29 / 64 / 107 us, 25 /
// 53 / 70 with float32 sums, 44 / 163 / 223 with the integer sums.  Chunks of 16 rows, which
// only problems of 32 rows on one trajectory and more take, stay in float32, as their sums
// have always been.
template <int G>
struct MmSum {
  typedef f64x4 vec;
  typedef double one;
};
template <>
struct MmSum<16> {
  typedef f32x4 vec;
  typedef float one;
};
__device__ __forceinline__ f32x4 mm_mfma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f64x4 mm_mfma(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// Row of the first operand that lane n16 brings, so that register v of lane group k4 holds row
// 4 k4 + v of the product (the float32 form's own order; the float64 one holds row 4 v + k4)
template <int G>
__device__ __forceinline__ int mm_arow(int n16) {
  return sizeof(typename MmSum<G>::one) == 4 ? n16 : 4 * (n16 & 3) + (n16 >> 2);
}

template <int G>
struct __attribute__((aligned(16))) MmLds {  // one wave's staging
  float w0[kMmBatch * kMmWPitch];  // weights of the tile's rows (zero outside the footprint)
  float w1[kMmBatch * kMmWPitch];  // weights of the tile's columns
  float s[kMmBatch * mm_spitch(G)];
  int exc[kMmExc];
};

// a tile of more than `target` entries is cut into pieces of `target`, listed first
__host__ __device__ inline int mm_splits(int v, int target) { return v <= target ? 1 : (v + target - 1) / target; }

// LDS writes of this wave's lanes are visible to its other lanes after this
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}


// a b with nearly one rounding a component (the rounding of each second product is added back)
__device__ __forceinline__ float2 cmul_once(float2 a, float2 b) {
  const float p = a.y * b.y, q = a.y * b.x;
  return make_float2(fmaf(a.x, b.x, -p) - fmaf(a.y, b.y, -p), fmaf(a.x, b.y, q) + fmaf(a.y, b.x, -q));
}

// One work item: tile piece wi, chunk of coil rows, for one wave (ks = 1) or the whole group
// (ks = kMmWaves, this wave its part `part`); `plan`, `omega` and rows [rowbase, rowbase +
// nrows) belong to one trajectory, `tabs` to all.
template <int G>
__device__ __forceinline__ void spread_sep_item(const Geom<float>& g, const TileGeom& tg, const SepGeom& sg,
                                                const float2* __restrict__ kdata, const float* __restrict__ omega,
                                                const int* __restrict__ plan, const int* __restrict__ tabs,
                                                float2* __restrict__ grid, int64_t rowbase, int64_t nrows, int64_t wi,
                                                int chunk, int ks, int part,
                                                MmLds<G>* group_lds, MmLds<G>& lds) {
  constexpr int kRows = mm_rows(G), kSP = mm_spitch(G);
  constexpr int kGroups = G >= 8 ? G / 8 : 0;  // rows form: 8 coil rows each
  constexpr int kLoads = kRows > 1 ? kRows / 2 : 1;  // rows staged by a half-wave
  const int lane = threadIdx.x & 63;
  const int n16 = lane & 15, k4 = lane >> 4;  // matrix operands: outer index, inner index (entry)
  if (wi >= plan[tg.o_nwork]) return;
  const int t = plan[tg.o_work + wi];
  const int split = (int)(wi - plan[tg.o_wstart + t]);
  const int64_t rbase = (int64_t)chunk * kRows;
  const int ncc = (int)((rbase + kRows < nrows ? rbase + kRows : nrows) - rbase);
  const int64_t row0 = rowbase + rbase;
  const int o0 = ((t / tg.bstride[0]) % tg.nb[0]) * kRegT0;
  const int o1 = ((t / tg.bstride[1]) % tg.nb[1]) * kRegT1;
  const int cstart = plan[tg.o_start + t];
  const int V = plan[tg.o_start + t + 1] - cstart;
  const int nsplit = mm_splits(V, tg.target);
  int i0 = nsplit > 1 ? split * tg.target : 0;
  int i1 = nsplit > 1 ? min(i0 + tg.target, V) : V;
  if (ks > 1) {  // this wave's batches
    const int nb = (i1 - i0 + kMmBatch - 1) / kMmBatch;
    const int b0 = i0 + (nb * part / kMmWaves) * kMmBatch, b1 = i0 + (nb * (part + 1) / kMmWaves) * kMmBatch;
    i0 = min(b0, i1);
    i1 = min(b1, i1);
  }
  const SepRec* recs = reinterpret_cast<const SepRec*>(reinterpret_cast<const char*>(plan) + tg.o_rec_bytes);
  const int* perm = plan + tg.o_perm + cstart;
  const int odd0 = tabs[sg.o_nm1] & 1, odd1 = tabs[sg.o_nm1 + 1] & 1;
  // a footprint's first cell relative to the tile, below 0 where it starts before the tile
  // or past the grid's end
  const auto rel = [](int cell, int o, int T, int K) { return cell - o < T ? cell - o : cell - o - K; };
  const int J0 = g.J[0];

  // phases of the tile's rows (lane n16: row n16) and of this lane's column, for the flush
  const double2 pr16 = reinterpret_cast<const double2*>(tabs + sg.o_ptab[0])[min(o0 + n16, g.K[0] - 1)];
  const double2 pc = reinterpret_cast<const double2*>(tabs + sg.o_ptab[1])[min(o1 + n16, g.K[1] - 1)];

  constexpr int kAcc = kGroups > 0 ? kGroups * kRegT0 : 2 * kRows;
  typedef typename MmSum<G>::vec Sum;
  typedef typename MmSum<G>::one Sum1;
  const int arow = mm_arow<G>(n16);
  Sum sum[kAcc];
#pragma unroll
  for (int c = 0; c < kAcc; ++c) sum[c] = Sum{0, 0, 0, 0};

  // Staging: lane (entry e, half h) holds the sample's header, its weights along dimension h
  // and its data for the half's rows.  The sample indices are loaded two batches ahead, the
  // records and the data one, so that all are in flight during a walk.
  const int e = lane & (kMmBatch - 1), h = lane / kMmBatch;
  int mnext = 0;
  float4 head = make_float4(0.f, 0.f, 0.f, 0.f);  // me, rc, F
  float2 wv[3], kd[kLoads];
  const auto stage_row = [&](int c) { return kRows > 1 ? h * kLoads + c : 0; };
  int at = 0;  // position of the entry that mnext belongs to
  const auto load_index = [&](int base) {
    at = min(base + e, i1 - 1);
    mnext = perm[at];
  };
  const auto load_sample = [&] {
    const int m = mnext;
    const float2* r = reinterpret_cast<const float2*>(recs + (tg.rec_entry ? cstart + at : m));
    head = *reinterpret_cast<const float4*>(r);
#pragma unroll
    for (int q = 0; q < 3; ++q) wv[q] = r[2 + 3 * h + q];
#pragma unroll
    for (int c = 0; c < kLoads; ++c) kd[c] = kdata[(row0 + min(stage_row(c), ncc - 1)) * g.M + m];
  };
  int nexc = 0;  // entries left to the atomic pass
  // operands of entries 4 k .. 4 k + 3: rows form: the tile's 16 row weights, outer form: the
  // weight of row arow; the weight of column n16; the data
  struct Operands {
    f32x4 w0[kGroups > 0 ? 4 : 1];
    float w1, a[kGroups > 0 ? kGroups : 2 * kRows];
  };
  const auto read_ops = [&](int k) {
    Operands o;
    const int en = 4 * k + k4;
    o.w1 = lds.w1[en * kMmWPitch + n16];
    if constexpr (kGroups > 0) {
#pragma unroll
      for (int u = 0; u < kGroups; ++u) o.a[u] = lds.s[en * kSP + 16 * u + arow];
#pragma unroll
      for (int q = 0; q < 4; ++q) o.w0[q] = *reinterpret_cast<const f32x4*>(&lds.w0[en * kMmWPitch + 4 * q]);
    } else {
      o.w0[0][0] = lds.w0[en * kMmWPitch + arow];
#pragma unroll
      for (int c = 0; c < kRows; ++c) {
        const float2 sv = *reinterpret_cast<const float2*>(&lds.s[en * kSP + 2 * c]);
        o.a[2 * c] = sv.x;
        o.a[2 * c + 1] = sv.y;
      }
    }
    return o;
  };
  if (i0 < i1) {  // loads past the end read the last entry again
    load_index(i0);
    load_sample();
    load_index(i0 + kMmBatch);
  }
  for (int base = i0; base < i1; base += kMmBatch) {
    const bool live = base + e < i1;
    const int me = __float_as_int(head.x);
    const int b0 = me & 0x7fffffff, b1 = __float_as_int(head.y);
    const int r0 = rel(b0, o0, kRegT0, g.K[0]), c0 = rel(b1, o1, kRegT1, g.K[1]);
    // one grid period before the wrapped cell: F times (-1)^(N - 1)
    const bool flip = ((b0 - o0 >= kRegT0 ? odd0 : 0) ^ (b1 - o1 >= kRegT1 ? odd1 : 0)) != 0;
    const float2 F = flip ? make_float2(-head.z, -head.w) : make_float2(head.z, head.w);
    const bool use = live && me >= 0;  // others get zero weights
    float2 s[kLoads];
    float probe = 0.f;  // NaN once any value is not finite
#pragma unroll
    for (int c = 0; c < kLoads; ++c) {
      s[c] = cmul_once(kd[c], F);
      probe = fmaf(s[c].x, 0.f, probe);
      probe = fmaf(s[c].y, 0.f, probe);
    }
    const bool finite = probe == 0.f;
    const bool bad = live && (me < 0 || !finite);
    const unsigned long long bb = __ballot(bad || !finite);
    if (bb) {  // rare: zero what is not finite, remember the first kMmExc entries left out
#pragma unroll
      for (int c = 0; c < kLoads; ++c)
        if (!(isfinite(s[c].x) && isfinite(s[c].y))) s[c] = make_float2(0.f, 0.f);
      const unsigned long long bb = __ballot(bad);
      const unsigned both = (unsigned)bb | (unsigned)(bb >> 32);
      const int at = nexc + __popc(both & ((1u << e) - 1u));
      if (h == 0 && ((both >> e) & 1u) && at < kMmExc) lds.exc[at] = base + e;
      nexc += __popc(both);
    }
    {
      // the row's zeros, then its six weights; what falls outside the tile goes to slot 16
      float* w = (h == 0 ? lds.w0 : lds.w1) + e * kMmWPitch;
      const int off = use ? (h == 0 ? r0 : c0) : 16;
#pragma unroll
      for (int q = 0; q < 4; ++q) reinterpret_cast<float4*>(w)[q] = make_float4(0.f, 0.f, 0.f, 0.f);
      const float wj[6] = {wv[0].x, wv[0].y, wv[1].x, wv[1].y, wv[2].x, wv[2].y};
#pragma unroll
      for (int j = 0; j < 6; ++j) w[min((unsigned)(off + j), 16u)] = wj[j];
    }
#pragma unroll
    for (int c = 0; c < kLoads; ++c)
      if (kRows > 1 || h == 0) *reinterpret_cast<float2*>(&lds.s[e * kSP + 2 * stage_row(c)]) = s[c];
    // tile rows that entries 4 k .. 4 k + 3 reach, in lane 4 k
    unsigned mask = use ? ((((1u << J0) - 1u) << (r0 + 5)) >> 5) & 0xffffu : 0u;
    mask |= (unsigned)__builtin_amdgcn_mov_dpp((int)mask, 0xb1, 0xf, 0xf, true);  // lane ^ 1
    mask |= (unsigned)__builtin_amdgcn_mov_dpp((int)mask, 0x4e, 0xf, 0xf, true);  // lane ^ 2
    wave_lds_sync();
    load_sample();
    load_index(base + 2 * kMmBatch);
    // Four entries at a time; the operands of the next four are read from LDS (all of them,
    // before the branches that skip rows) while this four's products run.
    Operands op = read_ops(0);
#pragma unroll
    for (int k = 0; k < kMmBatch / 4; ++k) {
      const unsigned mk = __builtin_amdgcn_readlane(mask, 4 * k);
      Operands nxt = op;
      if (k + 1 < kMmBatch / 4) nxt = read_ops(k + 1);
      asm volatile("" ::: "memory");  // keeps the reads here
      if constexpr (kGroups > 0) {
#pragma unroll
        for (int r = 0; r < kRegT0; ++r) {
          if ((mk >> r) & 1u) {
            const Sum1 w = (Sum1)op.w0[r / 4][r % 4] * (Sum1)op.w1;
#pragma unroll
            for (int u = 0; u < kGroups; ++u) sum[u * kRegT0 + r] = mm_mfma((Sum1)op.a[u], w, sum[u * kRegT0 + r]);
          }
        }
      } else if (mk != 0) {
#pragma unroll
        for (int c = 0; c < kRows; ++c) {
          sum[2 * c] = mm_mfma((Sum1)op.w0[0][0] * (Sum1)op.a[2 * c], (Sum1)op.w1, sum[2 * c]);
          sum[2 * c + 1] = mm_mfma((Sum1)op.w0[0][0] * (Sum1)op.a[2 * c + 1], (Sum1)op.w1, sum[2 * c + 1]);
        }
      }
      op = nxt;
    }
    wave_lds_sync();  // the next batch overwrites the staging
  }

  const int exc = lane < kMmExc ? lds.exc[lane] : 0;  // (the staging is reused)

  // A group's waves add their sums, in wave order: wave q collects the q-th kQ accumulators.
  constexpr int kQ = kAcc / kMmWaves > 2 ? kAcc / kMmWaves : 2, kRounds = kAcc / kQ;
  static_assert((kMmWaves - 1) * kQ * 64 * sizeof(Sum) <= kMmWaves * sizeof(MmLds<G>), "the sums fit the staging");
  if (ks > 1) {
    Sum* const sums = reinterpret_cast<Sum*>(group_lds);  // [wave, the collecting one left out][kQ][lane]
#pragma unroll
    for (int q = 0; q < kRounds; ++q) {
      lds_barrier();  // the staging, or the last round's sums, are read
      if (part != q) {
        Sum* const mine = sums + (part - (part > q ? 1 : 0)) * (kQ * 64) + lane;
#pragma unroll
        for (int i = 0; i < kQ; ++i) mine[i * 64] = sum[q * kQ + i];
      }
      lds_barrier();
      if (part == q) {
#pragma unroll
        for (int i = 0; i < kQ; ++i) {
          Sum s = q == 0 ? sum[i] : sums[i * 64 + lane];
#pragma unroll
          for (int w = 1; w < kMmWaves; ++w) s += w == q ? sum[q * kQ + i] : sums[((w - (w > q ? 1 : 0)) * kQ + i) * 64 + lane];
          sum[q * kQ + i] = s;
        }
      }
    }
  }
  const auto mine = [&](int a) { return ks == 1 || a / kQ == part; };  // accumulators this wave flushes

  // Flush: lane n16 holds column n16 of the tile; every cell inside the grid is written
  // (split tiles were zeroed first and add), 128 contiguous bytes of a row per 16 lanes.
  const int k1 = o1 + n16;
  const auto phase = [&](int r) {  // of this lane's cell in tile row r
    return cmul(make_double2(__shfl(pr16.x, r, 64), __shfl(pr16.y, r, 64)), pc);
  };
  const auto put = [&](int row, int r, double2 p, Sum1 re, Sum1 im) {  // the rotated cell of tile row r
    const int k0 = o0 + r;
    if (row < ncc && k0 < g.K[0] && k1 < g.K[1]) {
      const double2 vd = cmul_conj(make_double2((double)re, (double)im), p);
      const float2 v = make_float2((float)vd.x, (float)vd.y);
      float2* dst = grid + (row0 + row) * g.G + (int64_t)k0 * g.stride[0] + k1;
      if (nsplit == 1) {
        *dst = v;
      } else {
        unsafeAtomicAdd(&dst->x, v.x);
        unsafeAtomicAdd(&dst->y, v.y);
      }
    }
  };
  if constexpr (kGroups > 0) {
#pragma unroll
    for (int r = 0; r < kRegT0; ++r) {
      const double2 p = phase(r);
#pragma unroll
      for (int u = 0; u < kGroups; ++u) {
        if (!mine(u * kRegT0 + r)) continue;
        const Sum a = sum[u * kRegT0 + r];
        put(8 * u + 2 * k4, r, p, a[0], a[1]);
        put(8 * u + 2 * k4 + 1, r, p, a[2], a[3]);
      }
    }
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const double2 p = phase(4 * k4 + v);
#pragma unroll
      for (int c = 0; c < kRows; ++c)
        if (mine(2 * c)) put(c, 4 * k4 + v, p, sum[2 * c][v], sum[2 * c + 1][v]);
    }
  }

  // Entries left out of the products: lane (tap row i, coil row) adds
  // kdata * conj(phase) * conj(t0[i] t1[j]) over the row's taps inside the tile.  The
  // remembered ones, or (more than fit) a walk over all entries of the item.
  // The tile's stores come first: they and the atomics meet in this XCD's L2 (a device-scope
  // fence would write the whole L2 back).
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (ks > 1) __syncthreads();
  if (nexc == 0) return;
  const bool listed = nexc <= kMmExc;
  const int n = listed ? nexc : i1 - i0;
  for (int x = 0; x < n; ++x) {
    const int ei = listed ? __shfl(exc, x, 64) : i0 + x;
    const int m = perm[ei];
    const SepRec& rec = recs[tg.rec_entry ? cstart + ei : m];
    const int me = rec.me;
    const int i = lane >> 3;
    const int r = rel(me & 0x7fffffff, o0, kRegT0, g.K[0]) + i, c0 = rel(rec.rc, o1, kRegT1, g.K[1]);
    if (i >= J0 || r < 0 || r >= kRegT0 || o0 + r >= g.K[0]) continue;
    const float2 F = rec.F;
    for (int row = lane & 7; row < ncc; row += 8) {
      const float2 kv = kdata[(row0 + row) * g.M + m];
      const float2 s = cmul(kv, F);
      if (me >= 0 && isfinite(s.x) && isfinite(s.y)) continue;
      const float om0 = omega[m], om1 = omega[g.M + m];
      const float theta = sample_theta<float, 2>(g, omega, m);
      const float2 u = cmul_conj(cmul_conj(kv, make_float2(cosf(theta), sinf(theta))), sep_tap_weight(g, 0, om0, i));
      for (int j = 0; j < g.J[1]; ++j) {
        const int c = c0 + j;
        if (c >= 0 && c < kRegT1 && o1 + c < g.K[1]) {
          const float2 v = cmul_conj(u, sep_tap_weight(g, 1, om1, j));
          float2* dst = grid + (row0 + row) * g.G + (int64_t)(o0 + r) * g.stride[0] + (o1 + c);
          unsafeAtomicAdd(&dst->x, v.x);
          unsafeAtomicAdd(&dst->y, v.y);
        }
      }
    }
  }
}

// (At least two waves per SIMD asked for: the accumulators then stay in VGPRs.  With the
// larger register budget the compiler keeps them in AGPRs and moves them to VGPRs and back
// around every skipped row.)
template <int G>
__global__ void __launch_bounds__(64 * kMmWaves) __attribute__((amdgpu_waves_per_eu(mm_waves(G))))
    spread_sep_kernel(const Geom<float> g, const TileGeom tg, const SepGeom sg, const float2* __restrict__ kdata,
                      const float* __restrict__ omega, const int* __restrict__ ws, float2* __restrict__ grid,
                      int nchunk, int ks) {
  __shared__ MmLds<G> lds[kMmWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t b = blockIdx.y;  // trajectory
  const int64_t item = ks == 1 ? (int64_t)blockIdx.x * kMmWaves + wave : (int64_t)blockIdx.x;
  const int64_t wi = item / nchunk;
  spread_sep_item<G>(g, tg, sg, kdata, omega + b * 2 * g.M, ws + b * tg.plan_stride, ws, grid, g.batched ? b * g.C : 0,
                     g.batched ? g.C : g.B * g.C, wi, (int)(item - wi * nchunk), ks, wave, lds, lds[wave]);
}

__device__ __forceinline__ void sep_zero_hot_item(const Geom<float>& g, const TileGeom& tg, const int* plan,
                                                  float2* __restrict__ grid, int t, int64_t r0, int64_t r1) {
  const int* start = plan + tg.o_start;
  if (mm_splits(start[t + 1] - start[t], tg.target) <= 1) return;
  const int o0 = ((t / tg.bstride[0]) % tg.nb[0]) * kRegT0;
  const int o1 = ((t / tg.bstride[1]) % tg.nb[1]) * kRegT1;
  for (int cell = threadIdx.x; cell < kRegT0 * kRegT1; cell += blockDim.x) {
    const int k0 = o0 + cell / kRegT1, k1 = o1 + cell % kRegT1;
    if (k0 >= g.K[0] || k1 >= g.K[1]) continue;
    for (int64_t r = r0; r < r1; ++r) grid[r * g.G + (int64_t)k0 * g.stride[0] + k1] = make_float2(0.f, 0.f);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Tile shapes tried in order (largest first): the first whose LDS staging holds
// min(rows, 3) coil rows at once is used.  Larger tiles keep more samples (lanes)
// busy per group; the row floor keeps 3-D tiles from holding a single row.
static const int* tile_shape(int D, bool fwd, int64_t nrows, int64_t numpoints_max, bool f32) {
  static const int spread2[2][3] = {{32, 32, 1}, {16, 16, 1}};
  static const int spread3[3][3] = {{16, 16, 12}, {8, 8, 8}, {8, 8, 4}};
  static const int fwd2[2][3] = {{32, 32, 1}, {16, 16, 1}};
  static const int fwd3[2][3] = {{16, 16, 12}, {8, 8, 8}};
  static const int one[1][3] = {{1024, 1, 1}};
  const int(*cand)[3] = one;
  int n = 1;
  if (D == 2) {
    cand = fwd ? fwd2 : spread2;
    n = 2;
  } else if (D == 3) {
    cand = fwd ? fwd3 : spread3;
    n = fwd ? 2 : 3;
  }
  // 2-D: a tile that holds min(rows, 3) rows per group; 3-D: the largest tile that
  // holds one row (fewer replicated entries: (16+5)^2 (12+5) / (16^2 12) = 2.4 against
  // 4.3 for 8^3, which more than pays for the entries' weights being computed per row)
  const int64_t want = D == 3 ? 1 : (nrows < 3 ? (nrows > 0 ? nrows : 1) : 3);
  for (int c = 0; c < n; ++c) {
    int64_t cells = 1;
    for (int i = 0; i < D; ++i) cells *= fwd ? cand[c][i] + numpoints_max - 1 : cand[c][i];
    const int64_t per_row = fwd ? cells * (f32 ? 8 : 16) : 2 * cells * 8;
    if (per_row * want <= kLdsBudget) return cand[c];
  }
  return cand[n - 1];
}

static TileGeom make_tile_geom(const tkbn_interp_desc* d, bool det, bool fwd = false) {
  TileGeom tg{};
  const int D = d->ndim;
  const int64_t rows0 = d->omega_batched ? d->coils : d->batch * d->coils;
  int64_t jmax = 1;
  for (int i = 0; i < D; ++i) jmax = d->numpoints[i] > jmax ? d->numpoints[i] : jmax;
  const int* shape = tile_shape(D, fwd, rows0, jmax, d->dtype == TKBN_F32);
  int tcells = 1;
  for (int i = 0; i < 3; ++i) {
    tg.T[i] = 1;
    tg.nb[i] = 1;
    tg.K[i] = 1;
    tg.J[i] = 1;
  }
  bool tuned = false;  // caller's tile edges (validated to fit one row in LDS)
  for (int i = 0; i < D; ++i) tuned = tuned || d->tile[i] > 0;
  for (int i = 0; i < D; ++i) {
    int T = tuned ? (d->tile[i] > 0 ? d->tile[i] : 1) : shape[i];
    const int need = (int)d->numpoints[i] - 1;
    if (T < need) T = need;
    if (T > d->grid_size[i]) T = (int)d->grid_size[i];
    if (T < 1) T = 1;
    tg.T[i] = T;
    tg.nb[i] = (int)ceil_div(d->grid_size[i], T);
    tg.K[i] = (int)d->grid_size[i];
    tg.J[i] = (int)d->numpoints[i];
    tcells *= T;
  }
  int bs = 1, ls = 1;
  for (int i = D - 1; i >= 0; --i) {
    tg.bstride[i] = bs;
    bs *= tg.nb[i];
    tg.lstride[i] = ls;
    ls *= tg.T[i];
  }
  tg.NB = bs;
  tg.tcells = tcells;
  tg.own_only = fwd ? 1 : 0;
  int rcells = 1;
  for (int i = 0; i < 3; ++i) tg.R[i] = 1;
  for (int i = 0; i < D; ++i) tg.R[i] = tg.T[i] + (int)d->numpoints[i] - 1;
  int rs = 1;
  for (int i = D - 1; i >= 0; --i) {
    tg.rstride[i] = rs;
    rs *= tg.R[i];
  }
  rcells = rs;
  tg.rcells = rcells;
  const int accb = 8;  // 64-bit fixed point (float data, deterministic) or double
  const int64_t nrows = d->omega_batched ? d->coils : d->batch * d->coils;
  int cc = fwd ? (int)(kLdsBudget / ((int64_t)rcells * (d->dtype == TKBN_F32 ? 8 : 16)))
               : (int)(kLdsBudget / (2LL * tcells * accb));
  cc = cc < 1 ? 1 : (cc > 8 ? 8 : cc);
  if (cc > nrows) cc = (int)(nrows > 0 ? nrows : 1);
  tg.CC = cc;
  // entries per work item: hot tiles are cut into pieces of `target` (measured: 512 for
  // the spread, against 1024 / 2048, is 10-20 % faster on a 12-coil 256^2 spiral; for the
  // 3-D gather, whose pieces each re-stage a 60 KB region per row, 2048 against 1024 is
  // ~1.5 % faster on the 8-coil 320^3 kooshball)
  tg.target = det ? 0x3fffffff
                  : (d->work_target > 0 ? d->work_target : (fwd ? (D == 3 ? 2048 : 1024) : 512));
  const int64_t M = d->klength;
  // a sample reaches at most maxt_d tiles along dimension d: 1 with a single tile,
  // 2 when every tile is at least J-1 long, 3 when the last tile is shorter
  int64_t per_sample = 1;
  for (int i = 0; i < D && !fwd; ++i) {
    int mt = 1;
    if (tg.nb[i] > 1) {
      const int last = tg.K[i] - (tg.nb[i] - 1) * tg.T[i];
      mt = last >= tg.J[i] - 1 ? 2 : 3;
    }
    per_sample *= mt;
  }
  tg.maxent = per_sample * M;
  // sum_t ceil(V_t / target) <= NB + (sum_t V_t) / target
  tg.maxwork = det ? tg.NB : tg.NB + tg.maxent / tg.target + 1;
  int64_t o = 0;
  tg.o_key = o;
  tg.o_perm = o; o += tg.maxent;
  tg.o_count = o; o += tg.NB;
  tg.o_start = o; o += tg.NB + 1;
  tg.o_cursor = o; o += tg.NB;
  tg.o_wstart = o; o += tg.NB + 1;
  tg.o_work = o; o += (tg.maxwork > tg.NB ? tg.maxwork : tg.NB);
  tg.o_nwork = o; o += 1;
  o = (o + 3) & ~3LL;  // 16-byte align each plan
  tg.plan_ints = o;
  // dimensions >= D keep extent 1 (their strides are unused and may be 0)
  for (int i = 0; i < 3; ++i) {
    tg.fT[i] = make_fastdiv((uint32_t)std::max(tg.T[i], 1));
    tg.fl[i] = make_fastdiv((uint32_t)std::max(tg.lstride[i], 1));
    tg.fR[i] = make_fastdiv((uint32_t)std::max(tg.R[i], 1));
  }
  tg.ftc = make_fastdiv((uint32_t)std::max(tg.tcells, 1));
  tg.frc = make_fastdiv((uint32_t)std::max(tg.rcells, 1));
  return tg;
}

static int64_t spread_workspace_bytes(const tkbn_interp_desc* d, const TileGeom& tg) {
  const int64_t nplans = d->omega_batched ? d->batch : 1;
  return nplans * tg.plan_ints * 4 + 16;
}

// the sample-lane spread's workspace
static int64_t adj_lane_bytes(const tkbn_interp_desc* d, bool det) {
  return plan_cache_bytes(d) + spread_workspace_bytes(d, make_tile_geom(d, det));
}

static size_t spread_lds_bytes(const tkbn_interp_desc* d, const TileGeom& tg, bool det) {
  (void)d;
  (void)det;
  return (size_t)tg.CC * 2 * tg.tcells * 8;  // 8-byte accumulators (make_tile_geom)
}

template <typename T, int D, int JM>
int spread_launch(const Geom<T>& g, const TileGeom& tg, bool det, const void* kdata, const void* omega, int* ws,
                  void* maxabs_slot, void* grid, size_t lds, hipStream_t s, const CacheHdr* cache) {
  const int64_t nrows = g.batched ? g.C : g.B * g.C;
  const int64_t zdim = g.batched ? g.B : 1;
  if (cache && g.M > 0) {  // no header: the caller reuses the plan
    dim3 gc(bin_grid(g.M), 1, (unsigned)zdim);
    bin_count_kernel<T, D><<<gc, dim3(256), 0, s>>>(g, tg, static_cast<const T*>(omega), ws, cache);
    TKBN_LAUNCH_CHECK("bin_count_kernel");
  }
  if (cache) {
    plan_scan_kernel<<<dim3((unsigned)zdim), dim3(1024), 0, s>>>(tg, ws, cache);
    TKBN_LAUNCH_CHECK("plan_scan_kernel");
  }
  if (cache && g.M > 0) {
    dim3 gc(bin_grid(g.M), 1, (unsigned)zdim);
    bin_scatter_kernel<T, D><<<gc, dim3(256), 0, s>>>(g, tg, static_cast<const T*>(omega), ws, cache);
    TKBN_LAUNCH_CHECK("bin_scatter_kernel");
  }
  const unsigned ychunks = (unsigned)ceil_div(nrows, tg.CC);
  const dim3 grid3((unsigned)tg.maxwork, ychunks, (unsigned)zdim);
  const auto* kd = static_cast<const cplx<T>*>(kdata);
  const auto* om = static_cast<const T*>(omega);
  auto* gr = static_cast<cplx<T>*>(grid);
  if (det || std::is_same<T, float>::value) {
    // fixed point; the float pass only runs if kdata or omega is not finite.  The
    // slot starts at zero: cleared by the plan-cache check, or here without one
    if (!cache) {
      const int st = launch_zero_fill<unsigned long long>(static_cast<unsigned long long*>(maxabs_slot), 1, s);
      if (st != TKBN_OK) return st;
    }
    const int64_t n = g.B * g.C * g.M * 2;
    const int64_t nom = (g.batched ? g.B : 1) * D * g.M;
    const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>(ceil_div(std::max(n, nom), 1024), 256));
    if (!det) {
      const int64_t nzero = (int64_t)tg.NB * ychunks * zdim;
      TKBN_REQUIRE(nzero + blocks < (1LL << 31), TKBN_ERR_UNSUPPORTED, "too many tiles x row chunks");
      zero_hot_maxabs_kernel<T, D><<<dim3((unsigned)(nzero + blocks)), dim3(256), 0, s>>>(
          g, tg, ws, gr, (int64_t)ychunks, static_cast<const T*>(kdata), n, om, nom, maxabs_slot, blocks);
      TKBN_LAUNCH_CHECK("zero_hot_maxabs_kernel");
    } else {
      maxabs_kernel<T><<<dim3((unsigned)blocks), dim3(256), 0, s>>>(static_cast<const T*>(kdata), n, om, nom,
                                                                     maxabs_slot);
      TKBN_LAUNCH_CHECK("maxabs_kernel");
    }
    spread_tiles_either_kernel<T, D, JM><<<grid3, dim3(spread_tiles_threads(D)), lds, s>>>(g, tg, kd, om, ws,
                                                                                          maxabs_slot, gr);
    TKBN_LAUNCH_CHECK("spread_tiles_either_kernel");
    note_kernel(det ? "spread_tiles_kernel<fixed,deterministic>" : "spread_tiles_kernel<fixed>");
  } else {
    zero_hot_tiles_kernel<T, D><<<dim3((unsigned)tg.NB, ychunks, (unsigned)zdim), dim3(256), 0, s>>>(
        g, tg, ws, static_cast<cplx<T>*>(grid));
    TKBN_LAUNCH_CHECK("zero_hot_tiles_kernel");
    spread_tiles_kernel<T, false, D, JM><<<grid3, dim3(spread_tiles_threads(D)), lds, s>>>(g, tg, kd, om, ws, maxabs_slot, gr, 0);
    TKBN_LAUNCH_CHECK("spread_tiles_kernel");
    note_kernel("spread_tiles_kernel<float>");
  }
  return TKBN_OK;
}

// ---- separable variant ----------------------------------------------------------
static int64_t plans_of(const tkbn_interp_desc* d) { return d->omega_batched ? d->batch : 1; }
static int64_t rows_of(const tkbn_interp_desc* d) { return d->omega_batched ? d->coils : d->batch * d->coils; }
// Form of the spread (see spread_sep_item): the outer form up to four rows (two products per
// row and four entries; the rows form takes about eight per eight rows), else 8 rows at once;
// 16, in float32 (the weights of four entries then serve twice the rows), from 32 rows on one
// trajectory on, whose sums have always been float32.
static bool sep_many_rows(const tkbn_interp_desc* d) { return !d->omega_batched && d->batch * d->coils >= 32; }
static int mm_form(const tkbn_interp_desc* d) {
  const int64_t nrows = rows_of(d);
  return sep_many_rows(d) ? 16 : nrows > 4 ? 8 : nrows > 2 ? 4 : nrows > 1 ? 2 : 1;
}

// (sample, tile) entries of all trajectories, about: (21/16)^2 a sample
static int64_t sep_entries(const tkbn_interp_desc* d) { return plans_of(d) * (d->klength * 7 / 4); }
// Waves that share a tile's entries: the whole group where the tiles x chunks alone do not
// fill the chip (4096 waves) and hold at least a batch of entries each (39 rows, 434 x 362:
// 142 -> 77 us, 12 rows, 512^2: 75 -> 51 us; 64 rows, 640^2, the other way: 216 -> 273 us).
// `items`: tiles x chunks.  A launch's own choice: the pieces of a plan do not depend on it.
static int mm_waves_per_item(int64_t entries, int64_t tiles, int64_t items) {
  return items < 4096 && entries >= kMmBatch * tiles ? kMmWaves : 1;
}

static TileGeom make_coil_tile_geom(const tkbn_interp_desc* d) {
  TileGeom tg{};
  const int TT[2] = {kRegT0, kRegT1};
  for (int i = 0; i < 2; ++i) {
    tg.K[i] = (int)d->grid_size[i];
    tg.J[i] = (int)d->numpoints[i];
    tg.T[i] = TT[i];
    tg.nb[i] = (int)ceil_div(d->grid_size[i], TT[i]);
  }
  tg.K[2] = tg.J[2] = tg.nb[2] = 1;
  tg.bstride[1] = 1;
  tg.bstride[0] = tg.nb[1];
  tg.NB = tg.nb[0] * tg.nb[1];
  // Entries per piece: a multiple of the mean tile's, so that few tiles are cut (pieces add
  // with atomics) and none is a long serial chain.  The rows have no say in it (a plan serves
  // calls of any number of rows, see sep_many_rows), nor has the number of waves that a launch
  // gives a piece, so it holds for both.  Adjoint interpolation of 8 rows, us, pieces of 128 /
  // 256 / 512 / 768 / 1024 / 2048: 256^2, 206 k radial samples (352 entries a tile) 153 / 88 /
  // 69 / 65 / 64 / 84; 96^2, 12 k (140) 20 / 21 / 28 / 35 / 42 / 44; 512^2, 307 k (131) 142 /
  // 91 / 92 / 116 / 142 / 239.  64 rows, 320^2, 256 k (280), 512 / 704 / 896 / 1024: 255 / 230 /
  // 218 / 214; 32 rows, 96^2, 512 / 704 / 1024: 33 / 38 / 47; float32 chains of more than 768
  // entries would be further from 64-bit sums than they have been (one-sign data, 1000 entries
  // in a tile: 4.8e-7 at 1024, 3.1e-7 at 768).
  {
    const int64_t mean = sep_entries(d) / ((int64_t)tg.NB * std::max<int64_t>(plans_of(d), 1));
    const bool many = sep_many_rows(d);
    const int64_t t = ceil_div(many ? 4 * mean : mean * 5 / 2, kMmBatch) * kMmBatch;
    tg.target = (int)std::min<int64_t>(std::max<int64_t>(t, many ? 512 : 256), many ? 768 : 1024);
  }
  // tiles a footprint can meet per dimension: 2, or 3 when the last tile is shorter
  // than J - 1 (the footprint then crosses it into the first tile)
  int64_t per_sample = 1;
  for (int i = 0; i < 2; ++i) {
    const int last = tg.K[i] - (tg.nb[i] - 1) * tg.T[i];
    per_sample *= last >= tg.J[i] - 1 ? 2 : 3;
  }
  tg.maxent = per_sample * d->klength;
  tg.maxwork = tg.NB + tg.maxent / tg.target + 1;  // sum of ceil(V / target)
  tg.ftarget = make_fastdiv((uint32_t)tg.target);
  return tg;
}

// The separable kernels take complex64, 2-D, J <= 6.  From 32 coil rows on one trajectory
// they are the only 2-D path (their tuning fields are ignored); below, a caller's tile or
// work target asks for the sample-lane kernels, whose fields they are, and so does a
// problem one of whose separable workspaces (72 bytes a sample in the forward, 88 to 108 in
// the adjoint, tables and tile lists beside) would pass 1 GiB.  Below 32 rows,
// sample-lane against separable: spread 31 -> 21 us, gather 25 -> 17 us (one row, 512^2 grid,
// 206 000 samples); call pair 371 -> 207 us (8 trajectories x 8 rows, 384^2).
constexpr int64_t kSepMaxBytes = 1LL << 30;
static int64_t sep_fwd_bytes(const tkbn_interp_desc* d);
static int64_t sep_adj_bytes(const tkbn_interp_desc* d);

// (the spread needs grids of at least tile + J - 1 cells per dimension)
static bool sep_spread_grid(const tkbn_interp_desc* d) {
  return d->grid_size[0] >= kRegT0 + 5 && d->grid_size[1] >= kRegT1 + 5;
}
static bool sep_form(const tkbn_interp_desc* d) {
  return d->dtype == TKBN_F32 && d->ndim == 2 && d->numpoints[0] <= 6 && d->numpoints[1] <= 6;
}
static bool sep_eligible(const tkbn_interp_desc* d) {
  if (!sep_form(d)) return false;
  if (sep_many_rows(d)) return true;
  if (d->tile[0] > 0 || d->tile[1] > 0 || d->work_target > 0) return false;
  return std::max(sep_fwd_bytes(d), sep_spread_grid(d) ? sep_adj_bytes(d) : 0) <= kSepMaxBytes;
}
static bool coil_variant_eligible(const tkbn_interp_desc* d) { return sep_eligible(d) && sep_spread_grid(d); }

// One-shot timing hook: events the caller asked to have recorded around the next
// main interpolation kernel (tkbn_profile_next_kernel).
struct ProfileHook {
  hipEvent_t start = nullptr, stop = nullptr;
};
static thread_local ProfileHook g_profile;

static void profile_before(hipStream_t s) {
  if (g_profile.start) (void)hipEventRecord(g_profile.start, s);
}
static void profile_after(hipStream_t s) {
  if (g_profile.stop) (void)hipEventRecord(g_profile.stop, s);
  g_profile = ProfileHook{};
}

static TileGeom make_gather_geom(const tkbn_interp_desc* d);

// ---- separable multi-coil kernels: plans and launches ----------------------------------
constexpr int kPlanSepGather = 6;
constexpr int kPlanSepSpread = 7;

// Records 64-byte aligned after a plan's int arrays; after all trajectories' plans what they
// share: N - 1, the flag, cell phases and real tables.
static void sep_finish_layout(TileGeom& tg, SepGeom& sg, int64_t o, const tkbn_interp_desc* d) {
  o = (o + 15) & ~15LL;
  tg.plan_ints = o;
  tg.o_rec_bytes = o * 4;
  tg.plan_stride = o + (tg.rec_entry ? tg.maxent : d->klength) * (int64_t)(sizeof(SepRec) / 4);
  o = plans_of(d) * tg.plan_stride;
  sg.o_nm1 = o;
  sg.o_flag = o + 2;
  o += 4;
  for (int i = 0; i < 2; ++i) {
    sg.o_ptab[i] = o;
    o += 4 * d->grid_size[i];
  }
  for (int i = 0; i < 2; ++i) {
    sg.o_rtab[i] = o;
    o += d->numpoints[i] * d->table_oversamp[i] + 1;
  }
  sg.end = o;
}

static SepGeom sep_phase_of(const tkbn_interp_desc* d) {
  SepGeom sg{};
  for (int i = 0; i < 2; ++i) sg.L[i] = (int)d->table_oversamp[i];
  return sg;
}

static TileGeom make_sep_gather_geom(const tkbn_interp_desc* d, SepGeom* sg) {
  TileGeom tg = make_gather_geom(d);
  *sg = sep_phase_of(d);
  int64_t o = 0;
  tg.o_key = o;
  tg.o_perm = o;  // unused: the records carry the sample index
  tg.o_count = o; o += tg.NB + 1;  // + finished count blocks
  tg.o_start = o; o += tg.NB + 1;
  tg.o_cursor = o; o += tg.NB;
  tg.o_wstart = o; o += tg.NB + 1;
  tg.o_work = o; o += (tg.maxwork > tg.NB ? tg.maxwork : tg.NB);
  tg.o_nwork = o; o += 1;
  sep_finish_layout(tg, *sg, o, d);
  return tg;
}

static TileGeom make_sep_spread_geom(const tkbn_interp_desc* d, SepGeom* sg) {
  TileGeom tg = make_coil_tile_geom(d);
  // 16 rows a chunk: a record per entry is read in order (16 coils x 4, 320^2 radial: 225 us;
  // through the sample index: 245); fewer rows, where the plan weighs more against the data,
  // a record per sample (one row, 205 824 samples: 16 instead of 56 MB, 17.8 us both)
  tg.rec_entry = mm_form(d) == 16;
  tg.T[2] = 2 * tg.target + tg.rec_entry;  // part of the plan's key
  *sg = sep_phase_of(d);
  int64_t o = 0;
  tg.o_key = o;
  tg.o_perm = o; o += tg.maxent;
  tg.o_count = o; o += tg.NB + 1;  // + finished count blocks
  tg.o_start = o; o += tg.NB + 1;
  tg.o_cursor = o; o += tg.NB;
  tg.o_wstart = o; o += tg.NB + 1;
  tg.o_work = o; o += (tg.maxwork > tg.NB ? tg.maxwork : tg.NB);
  tg.o_nwork = o; o += 1;
  sep_finish_layout(tg, *sg, o, d);
  return tg;
}

static int64_t sep_adj_bytes(const tkbn_interp_desc* d) {
  SepGeom sg;
  make_sep_spread_geom(d, &sg);
  return plan_cache_bytes(d) + sg.end * 4;
}

// The plan kernels of the separable gather (grid = nullptr) or spread, one plan per
// trajectory; the spread's last one also clears what is added into in `grid`.
static int sep_plan_launch(const tkbn_interp_desc* d, float2* grid, const Geom<float>& g, const TileGeom& tg,
                           const SepGeom& sg, const float* om, void* ws, int* wsi, hipStream_t s) {
  const bool spread = grid != nullptr;
  const int kind = spread ? kPlanSepSpread : kPlanSepGather;
  const int64_t np = plans_of(d);
  TKBN_REQUIRE(np < 65536, TKBN_ERR_UNSUPPORTED, "too many trajectories in one call");
  const int64_t zero_blocks = spread ? tg.NB * ceil_div(rows_of(d), 64) : 0;
  const bool reused = plan_reused(d);
  const int nscatter = reused ? 0 : (int)bin_grid(g.M);
  TKBN_REQUIRE(zero_blocks + nscatter < (1LL << 31), TKBN_ERR_UNSUPPORTED,
               "too many coil rows x work items for one launch");
  CacheHdr* cache = nullptr;
  const dim3 gc((unsigned)nscatter, (unsigned)np);
  hipError_t e1 = hipSuccess;
  if (reused) {
    const int st = plan_registry_require(d, kind, tg.T, ws);
    if (st != TKBN_OK || !spread) return st;
  } else {
    CacheZero z;
    z.p = wsi + tg.o_count;
    z.n = tg.NB + 1;
    z.stride = tg.plan_stride;
    z.copies = np;
    z.p2 = wsi + sg.o_flag;
    z.n2 = 1;
    const int st = plan_cache_begin(d, kind, tg.T, om, ws, s, &cache, z);
    if (st != TKBN_OK) return st;
    if (spread)
      sep_spr_count_kernel<<<gc, dim3(256), 0, s>>>(g, tg, sg, om, wsi, cache);
    else
      sep_gat_count_kernel<<<gc, dim3(256), 0, s>>>(g, tg, sg, om, wsi, cache);
    e1 = hipGetLastError();
  }
  if (spread)
    sep_spr_scatter_kernel<<<dim3((unsigned)(nscatter + zero_blocks), (unsigned)np), dim3(256), 0, s>>>(
        g, tg, sg, om, wsi, cache, nscatter, grid);
  else
    sep_gat_scatter_kernel<<<gc, dim3(256), 0, s>>>(g, tg, sg, om, wsi, cache);
  const hipError_t e2 = hipGetLastError();
  if (e1 != hipSuccess || e2 != hipSuccess) {
    if (!reused) plan_cache_invalidate(ws, s);
    set_error("launch of the separable plan failed: %s", hipGetErrorString(e1 != hipSuccess ? e1 : e2));
    return TKBN_ERR_HIP;
  }
  return TKBN_OK;
}

// coil rows per work item of the gather (see gather_sep_kernel)
static int gat_rows(int64_t nrows) { return nrows > 8 ? 16 : nrows > 4 ? 8 : nrows > 2 ? 4 : nrows > 1 ? 2 : 1; }

template <int ROWS>
static void gather_sep_start(const Geom<float>& g, const TileGeom& tg, const SepGeom& sg, const float2* grid,
                             const float* om, const int* wsi, float2* kdata, int nchunk, dim3 grd, hipStream_t s) {
  if (g.J[0] == 6 && g.J[1] == 6)
    gather_sep_kernel<6, ROWS><<<grd, dim3(GatShape<ROWS>::kThreads), 0, s>>>(g, tg, sg, grid, om, wsi, kdata, nchunk);
  else
    gather_sep_kernel<0, ROWS><<<grd, dim3(GatShape<ROWS>::kThreads), 0, s>>>(g, tg, sg, grid, om, wsi, kdata, nchunk);
}

static int gather_sep_launch(const tkbn_interp_desc* d, const void* grid, const void* omega, void* kdata, void* ws,
                             hipStream_t s) {
  const Geom<float> g = make_geom<float>(d);
  SepGeom sg;
  const TileGeom tg = make_sep_gather_geom(d, &sg);
  int* wsi = reinterpret_cast<int*>(static_cast<char*>(ws) + plan_cache_bytes(d));
  const float* om = static_cast<const float*>(omega);
  const int st = sep_plan_launch(d, nullptr, g, tg, sg, om, ws, wsi, s);
  if (st != TKBN_OK) return st;
  const int rows = gat_rows(rows_of(d));
  const int nchunk = (int)ceil_div(rows_of(d), rows);
  const int64_t run = (int64_t)kXcdTiles * nchunk;  // see xcd_work_item
  const int64_t groups = ceil_div(tg.maxwork * nchunk, 8 * run) * 8 * run;
  TKBN_REQUIRE(groups < (1LL << 31), TKBN_ERR_UNSUPPORTED, "too many coil rows x work items for one launch");
  const dim3 grd((unsigned)groups, (unsigned)plans_of(d));
  const float2* gr = static_cast<const float2*>(grid);
  float2* kd = static_cast<float2*>(kdata);
  profile_before(s);
  switch (rows) {
    case 16: gather_sep_start<16>(g, tg, sg, gr, om, wsi, kd, nchunk, grd, s); break;
    case 8: gather_sep_start<8>(g, tg, sg, gr, om, wsi, kd, nchunk, grd, s); break;
    case 4: gather_sep_start<4>(g, tg, sg, gr, om, wsi, kd, nchunk, grd, s); break;
    case 2: gather_sep_start<2>(g, tg, sg, gr, om, wsi, kd, nchunk, grd, s); break;
    default: gather_sep_start<1>(g, tg, sg, gr, om, wsi, kd, nchunk, grd, s); break;
  }
  profile_after(s);
  TKBN_LAUNCH_CHECK("gather_sep_kernel");
  note_kernel("gather_sep_kernel");
  return TKBN_OK;
}

static int spread_sep_launch(const tkbn_interp_desc* d, const void* kdata, const void* omega, void* ws, void* grid,
                             hipStream_t s) {
  const Geom<float> g = make_geom<float>(d);
  SepGeom sg;
  const TileGeom tg = make_sep_spread_geom(d, &sg);
  int* wsi = reinterpret_cast<int*>(static_cast<char*>(ws) + plan_cache_bytes(d));
  const float* om = static_cast<const float*>(omega);
  const int st = sep_plan_launch(d, static_cast<float2*>(grid), g, tg, sg, om, ws, wsi, s);
  if (st != TKBN_OK) return st;
  const int64_t nrows = rows_of(d), np = plans_of(d);
  const int form = mm_form(d);
  const int nchunk = (int)ceil_div(nrows, mm_rows(form));
  const int ks = mm_waves_per_item(sep_entries(d), tg.NB * np, tg.NB * np * nchunk);
  const int64_t groups = ceil_div(tg.maxwork * nchunk, kMmWaves / ks);
  TKBN_REQUIRE(groups < (1LL << 31), TKBN_ERR_UNSUPPORTED, "too many coil rows x work items for one launch");
  const dim3 grd((unsigned)groups, (unsigned)np), blk(64 * kMmWaves);
  const float2* kd = static_cast<const float2*>(kdata);
  float2* gr = static_cast<float2*>(grid);
  profile_before(s);
  switch (form) {
    case 1: spread_sep_kernel<1><<<grd, blk, 0, s>>>(g, tg, sg, kd, om, wsi, gr, nchunk, ks); break;
    case 2: spread_sep_kernel<2><<<grd, blk, 0, s>>>(g, tg, sg, kd, om, wsi, gr, nchunk, ks); break;
    case 4: spread_sep_kernel<4><<<grd, blk, 0, s>>>(g, tg, sg, kd, om, wsi, gr, nchunk, ks); break;
    case 8: spread_sep_kernel<8><<<grd, blk, 0, s>>>(g, tg, sg, kd, om, wsi, gr, nchunk, ks); break;
    default: spread_sep_kernel<16><<<grd, blk, 0, s>>>(g, tg, sg, kd, om, wsi, gr, nchunk, ks); break;
  }
  profile_after(s);
  TKBN_LAUNCH_CHECK("spread_sep_kernel");
  note_kernel("spread_sep_kernel");
  return TKBN_OK;
}

// ---------------------------------------------------------------------------
// 3-D register-tile spread (complex64, J <= 6, at least kR3MinRows coil rows, one
// trajectory for all rows, grids of at least tile + J - 1 cells per dimension)
//   One group (8 waves) per (8 x 8 x 16 tile, piece, chunk of 8 coil rows): wave w owns
//   the tile's plane x = w; lane (y, row) owns the 16 cells along z of column (w, y) of
//   its coil row as float2 registers.  Every cell has one writer, so no atomics.
//   Entries (sample, tile) are staged 64 at a time: each sample's three rows of tap
//   weights (conjugated), the footprint's offsets inside the tile, and per (entry, y,
//   row) the sample's data times its y weight.  Each wave then walks the staged entries
//   that reach its plane, grouped by z offset so that every accumulator index is a
//   compile-time constant.
//   A tile with more than P entries is cut into pieces of P entries.  A piece stores its
//   partial tile into a pool slot and reg3_combine_kernel adds a tile's pieces in piece
//   order.  The plan raises P until the pieces fit the pool.
//   Deterministic mode sorts every tile's entries by sample index when the plan is
//   built, so the pieces, the batches and every float sum have a fixed order: the result
//   is bitwise repeatable without fixed point.
// ---------------------------------------------------------------------------
constexpr int kR3T0 = 8, kR3T1 = 8, kR3T2 = 16;
constexpr int kR3Rows = 8;                  // coil rows per work item (lanes = y x row)
constexpr int kR3Threads = 64 * kR3T0;      // one wave per x plane
constexpr int kR3Batch = 64;                // staged entries
constexpr int kR3Cells = kR3T0 * kR3T1 * kR3T2;
constexpr int kR3Target = 1024;             // entries per piece before the pool fit
constexpr int kR3SortChunk = 2048;          // entries sorted in LDS at once
constexpr int64_t kR3PoolCap = 128ll << 20;  // bytes of piece partials at most
constexpr int kR3MinRows = 4;
constexpr int kR3MinZ = -5;                 // first z offset of a footprint in a tile (J <= 6)
constexpr int64_t kR3SlotFloats2 = (int64_t)kR3Cells * kR3Rows;
constexpr int kR3FlushPitch = kR3T2 + 1;  // float2 per transposed column (odd: fewer bank conflicts)
constexpr int kR3LdsBytes = kR3T0 * 64 * kR3FlushPitch * 8;  // >= the staged batch (46848 bytes)
static_assert(kR3LdsBytes >= 46848, "flush buffer covers the staging layout");
// plan meta ints: piece size P, hot pieces, hot tiles, sort chunks, merge passes, entries
enum { kR3MetaP = 0, kR3MetaHotPieces, kR3MetaHotTiles, kR3MetaSort, kR3MetaPasses, kR3MetaEntries, kR3MetaInts = 8 };

static bool reg3_eligible(const tkbn_interp_desc* d) {
  if (d->dtype != TKBN_F32 || d->ndim != 3 || d->omega_batched) return false;
  const int T[3] = {kR3T0, kR3T1, kR3T2};
  for (int i = 0; i < 3; ++i)
    if (d->numpoints[i] > 6 || d->grid_size[i] < T[i] + d->numpoints[i] - 1) return false;
  return d->batch * d->coils >= kR3MinRows;
}

static TileGeom make_reg3_geom(const tkbn_interp_desc* d, bool det) {
  TileGeom tg{};
  const int TT[3] = {kR3T0, kR3T1, kR3T2};
  for (int i = 0; i < 3; ++i) {
    tg.K[i] = (int)d->grid_size[i];
    tg.J[i] = (int)d->numpoints[i];
    tg.T[i] = TT[i];
    tg.nb[i] = (int)ceil_div(d->grid_size[i], TT[i]);
    tg.lstride[i] = 1;
  }
  tg.bstride[2] = 1;
  tg.bstride[1] = tg.nb[2];
  tg.bstride[0] = tg.nb[1] * tg.nb[2];
  tg.NB = tg.nb[0] * tg.nb[1] * tg.nb[2];
  tg.tcells = kR3Cells;
  tg.own_only = 0;
  tg.CC = kR3Rows;
  tg.target = kR3Target;
  // tiles a sample reaches per dimension: 2, or 3 when the last tile is shorter than J - 1
  int64_t per_sample = 1;
  for (int i = 0; i < 3; ++i) {
    int mt = 1;
    if (tg.nb[i] > 1) {
      const int last = tg.K[i] - (tg.nb[i] - 1) * tg.T[i];
      mt = last >= tg.J[i] - 1 ? 2 : 3;
    }
    per_sample *= mt;
  }
  tg.maxent = per_sample * d->klength;
  tg.maxwork = tg.NB + tg.maxent / tg.target + 1;
  int64_t o = 0;
  tg.o_key = o;
  tg.o_perm = o; o += tg.maxent;
  tg.o_count = o; o += tg.NB;
  tg.o_start = o; o += tg.NB + 1;
  tg.o_cursor = o; o += tg.NB;
  tg.o_wstart = o; o += tg.NB + 1;
  tg.o_work = o; o += tg.maxwork;
  tg.o_nwork = o; o += 1;
  tg.o_hot = o; o += tg.NB;
  tg.o_meta = o; o += kR3MetaInts;
  tg.o_tmp = o; o += 3 * (tg.NB + 1);
  const int64_t nsort = det ? tg.NB + tg.maxent / kR3SortChunk + 1 : 0;
  tg.o_sort = o; o += 2 * nsort;
  tg.o_scratch = o; o += det ? tg.maxent : 0;
  o = (o + 3) & ~3LL;
  tg.o_sw = o; o += 3 * d->klength * 12;  // float2 [3][M][6]
  tg.o_sb = o; o += 3 * d->klength;       // int [3][M]
  o = (o + 63) & ~63LL;  // the pool starts 256-byte aligned
  tg.plan_ints = o;
  tg.nchunk = (int)ceil_div(d->batch * d->coils, kR3Rows);
  // a tile of V > P entries gives ceil(V / P) < 2 V / P pieces
  const int64_t bound = (2 * tg.maxent / tg.target + 1) * tg.nchunk;
  const int64_t cap = kR3PoolCap / (kR3SlotFloats2 * 8);
  tg.pool_slots = std::max<int64_t>(tg.nchunk, std::min<int64_t>(bound, cap));
  tg.pool_off_bytes = o * 4;
  return tg;
}

static int64_t reg3_workspace_bytes(const TileGeom& tg) {
  return tg.pool_off_bytes + tg.pool_slots * kR3SlotFloats2 * 8;
}

// block-wide sum or max of one int per thread (every thread gets the result)
__device__ __forceinline__ int block_reduce_int(int v, bool is_max, int* sb) {
  for (int o = 32; o > 0; o >>= 1) {
    const int u = __shfl_down(v, o, 64);
    v = is_max ? max(v, u) : v + u;
  }
  __syncthreads();  // sb may still be read by an earlier reduction
  if ((threadIdx.x & 63) == 0) sb[threadIdx.x >> 6] = v;
  __syncthreads();
  int r = sb[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = is_max ? max(r, sb[w]) : r + sb[w];
  return r;
}

// Tile starts, the piece size, the work list (hot tiles' pieces first, then one item per
// other tile, empty tiles included: they store zeros), the hot tile list and, in
// deterministic mode, the list of sort chunks and the number of merge passes.
__global__ void __launch_bounds__(1024) reg3_plan_scan_kernel(const TileGeom tg, int* __restrict__ plan,
                                                             const CacheHdr* cache, int det) {
  if (cache_hit(cache)) return;  // cached plan reused
  __shared__ int sbuf[1024];
  const int NB = tg.NB;
  const int* count = plan + tg.o_count;
  int* start = plan + tg.o_start;
  int* cursor = plan + tg.o_cursor;
  int* wstart = plan + tg.o_wstart;
  int* work = plan + tg.o_work;
  int* hot = plan + tg.o_hot;
  int* meta = plan + tg.o_meta;
  int* ta = plan + tg.o_tmp;
  int* tb = ta + (NB + 1);
  int* tc = tb + (NB + 1);
  block_exclusive_scan(count, start, NB, sbuf);
  int vmax = 0;
  for (int t = threadIdx.x; t < NB; t += blockDim.x) {
    cursor[t] = start[t];
    vmax = max(vmax, count[t]);
  }
  vmax = block_reduce_int(vmax, true, sbuf);
  // smallest P = target * 2^k whose hot pieces fit the pool (P >= vmax: no hot tiles)
  int P = tg.target;
  for (;;) {
    int pieces = 0;
    for (int t = threadIdx.x; t < NB; t += blockDim.x) {
      const int v = count[t];
      if (v > P) pieces += (v + P - 1) / P;
    }
    pieces = block_reduce_int(pieces, false, sbuf);
    if ((int64_t)pieces * tg.nchunk <= tg.pool_slots || P >= vmax) break;
    P *= 2;
  }
  for (int t = threadIdx.x; t < NB; t += blockDim.x) {
    const int v = count[t];
    ta[t] = v > P ? (v + P - 1) / P : 0;
  }
  __syncthreads();
  block_exclusive_scan(ta, tb, NB, sbuf);  // hot pieces before tile t
  for (int t = threadIdx.x; t < NB; t += blockDim.x) ta[t] = count[t] > P ? 0 : 1;
  __syncthreads();
  block_exclusive_scan(ta, tc, NB, sbuf);  // other tiles before tile t
  const int nhotp = tb[NB];
  const int cap = (int)tg.maxwork;
  for (int t = threadIdx.x; t < NB; t += blockDim.x) {
    const int v = count[t];
    const bool h = v > P;
    const int w0 = h ? tb[t] : nhotp + tc[t];
    const int n = h ? (v + P - 1) / P : 1;
    wstart[t] = w0;
    for (int w = w0; w < min(w0 + n, cap); ++w) work[w] = t;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < NB; t += blockDim.x) ta[t] = count[t] > P ? 1 : 0;
  __syncthreads();
  block_exclusive_scan(ta, tc, NB, sbuf);  // hot tiles before tile t
  for (int t = threadIdx.x; t < NB; t += blockDim.x)
    if (count[t] > P) hot[tc[t]] = t;
  int nsort = 0;
  if (det) {
    __syncthreads();
    for (int t = threadIdx.x; t < NB; t += blockDim.x) {
      const int v = count[t];
      ta[t] = v > 1 ? (v + kR3SortChunk - 1) / kR3SortChunk : 0;
    }
    __syncthreads();
    block_exclusive_scan(ta, tb, NB, sbuf);  // sort chunks before tile t
    int* sortl = plan + tg.o_sort;
    for (int t = threadIdx.x; t < NB; t += blockDim.x) {
      const int v = count[t];
      if (v <= 1) continue;
      for (int c = 0; c * kR3SortChunk < v; ++c) {
        sortl[2 * (tb[t] + c)] = start[t] + c * kR3SortChunk;
        sortl[2 * (tb[t] + c) + 1] = min(kR3SortChunk, v - c * kR3SortChunk);
      }
    }
    nsort = tb[NB];
  }
  if (threadIdx.x == 0) {
    int passes = 0;
    if (det)
      while (((int64_t)kR3SortChunk << passes) < vmax) ++passes;
    meta[kR3MetaP] = P;
    meta[kR3MetaHotPieces] = nhotp;
    meta[kR3MetaHotTiles] = tc[NB];
    meta[kR3MetaSort] = nsort;
    meta[kR3MetaPasses] = passes;
    meta[kR3MetaEntries] = start[NB];
    wstart[NB] = nhotp + (NB - tc[NB]);
    plan[tg.o_nwork] = min(nhotp + (NB - tc[NB]), cap);
  }
}

// Sorts each chunk of at most kR3SortChunk entries of a tile by sample index (bitonic,
// in LDS; padding sorts last).
__global__ void __launch_bounds__(1024) reg3_sort_chunks_kernel(const TileGeom tg, int* __restrict__ plan,
                                                               const CacheHdr* cache) {
  if (cache_hit(cache)) return;
  const int nsort = plan[tg.o_meta + kR3MetaSort];
  __shared__ int buf[kR3SortChunk];
  int* perm = plan + tg.o_perm;
  for (int c = blockIdx.x; c < nsort; c += gridDim.x) {
    const int pos = plan[tg.o_sort + 2 * c], len = plan[tg.o_sort + 2 * c + 1];
    for (int i = threadIdx.x; i < kR3SortChunk; i += blockDim.x) buf[i] = i < len ? perm[pos + i] : 0x7fffffff;
    __syncthreads();
    const int tid = threadIdx.x;  // 1024 threads: one compare-exchange pair each
    for (int k = 2; k <= kR3SortChunk; k <<= 1) {
      for (int j = k >> 1; j > 0; j >>= 1) {
        const int i = 2 * tid - (tid & (j - 1));
        const int p = i + j;
        const bool up = (i & k) == 0;
        const int a = buf[i], b = buf[p];
        if ((a > b) == up) {
          buf[i] = b;
          buf[p] = a;
        }
        __syncthreads();
      }
    }
    for (int i = threadIdx.x; i < len; i += blockDim.x) perm[pos + i] = buf[i];
    __syncthreads();  // buf is refilled by the next chunk
  }
}

// elements of the sorted run a[lo .. hi) smaller than key
__device__ __forceinline__ int count_less(const int* a, int lo, int hi, int key) {
  const int base = lo;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo - base;
}

// Merge pass `pass`: inside every tile longer than R = kR3SortChunk << pass, sorted runs
// [2kR, (2k+1)R) and [(2k+1)R, (2k+2)R) (tile-relative) become one sorted run.  Keys
// are distinct, so each element's place is its run offset plus its rank in the partner
// run.  Passes alternate between the permutation and the scratch array; passes past
// the plan's count do nothing.
__global__ void __launch_bounds__(256) reg3_merge_kernel(const TileGeom tg, int* __restrict__ plan,
                                                        const CacheHdr* cache, int pass) {
  if (cache_hit(cache)) return;
  const int* meta = plan + tg.o_meta;
  if (pass >= meta[kR3MetaPasses]) return;
  const int total = meta[kR3MetaEntries];
  const int* src = plan + ((pass & 1) ? tg.o_scratch : tg.o_perm);
  int* dst = plan + ((pass & 1) ? tg.o_perm : tg.o_scratch);
  const int* start = plan + tg.o_start;
  const int R = kR3SortChunk << pass;
  for (int64_t p64 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p64 < total;
       p64 += (int64_t)gridDim.x * blockDim.x) {
    const int p = (int)p64;
    int lo = 0, hi = tg.NB;  // last tile t with start[t] <= p
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (start[mid] <= p) lo = mid;
      else hi = mid;
    }
    const int s0 = start[lo], V = start[lo + 1] - s0, o = p - s0;
    const int key = src[p];
    if (V <= R) {
      dst[p] = key;
      continue;
    }
    const int r = o / R, base = (r & ~1) * R;
    int no;
    if ((r & 1) == 0) no = o + count_less(src + s0, min(base + R, V), min(base + 2 * R, V), key);
    else no = base + (o - base - R) + count_less(src + s0, base, base + R, key);
    dst[s0 + no] = key;
  }
}

// acc[C + j] += u * w[j] for the taps that land in the tile (C = the footprint's z offset)
template <int C>
__device__ __forceinline__ void r3_add_z(float2 (&acc)[kR3T2], const float2 u, const float2* w) {
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    if (C + j >= 0 && C + j < kR3T2) {
      const float2 t = w[j];
      acc[C + j].x = fmaf(u.x, t.x, acc[C + j].x);
      acc[C + j].x = fmaf(-u.y, t.y, acc[C + j].x);
      acc[C + j].y = fmaf(u.x, t.y, acc[C + j].y);
      acc[C + j].y = fmaf(u.y, t.x, acc[C + j].y);
    }
  }
}

// Per-sample tap rows of the plan: for every sample and dimension the conjugated table
// weights of its J taps (zero past J; dimension 0 also times the conjugated phase
// exp(-i theta)) and the wrapped base cell of its footprint.
__global__ void __launch_bounds__(256) reg3_sample_rows_kernel(const Geom<float> g, const TileGeom tg,
                                                              const float* __restrict__ omega, int* __restrict__ plan,
                                                              const CacheHdr* cache) {
  if (cache_hit(cache)) return;
  float2* sw = reinterpret_cast<float2*>(plan + tg.o_sw);
  int* sb = plan + tg.o_sb;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < 3 * g.M; i += (int64_t)gridDim.x * blockDim.x) {
    const int d = (int)(i / g.M);
    const int64_t m = i - d * g.M;
    float2 w[6];
    int mdx[6];
    sample_taps_md<float, 6>(g, d, omega[d * g.M + m], w, mdx);
    float2 ph = make_float2(1.f, 0.f);
    if (d == 0) {
      const float theta = sample_theta<float, 3>(g, omega, m);
      ph = make_float2(cosf(theta), sinf(theta));
    }
    float2* row = sw + (d * g.M + m) * 6;
#pragma unroll
    for (int j = 0; j < 6; ++j) row[j] = cmul_conj(make_float2(w[j].x, -w[j].y), ph);
    sb[d * g.M + m] = mdx[0];
  }
}

__global__ void __launch_bounds__(kR3Threads)
    spread_reg3_kernel(const Geom<float> g, const TileGeom tg, const float2* __restrict__ kdata,
                       const float* __restrict__ omega, const int* __restrict__ plan, float2* __restrict__ grid,
                       float2* __restrict__ pool) {
  // LDS: the staged batch, and afterwards (same bytes) each wave's flush transpose
  __shared__ __attribute__((aligned(16))) unsigned char smem[kR3LdsBytes];
  float2(&W0)[kR3Batch][6] = *reinterpret_cast<float2(*)[kR3Batch][6]>(smem);
  float2(&W1)[kR3Batch][6] = *reinterpret_cast<float2(*)[kR3Batch][6]>(smem + 3072);
  float2(&W2)[kR3Batch][6] = *reinterpret_cast<float2(*)[kR3Batch][6]>(smem + 6144);
  float2(&S)[kR3Batch][kR3Rows] = *reinterpret_cast<float2(*)[kR3Batch][kR3Rows]>(smem + 9216);
  float2(&Vy)[kR3Batch][64] = *reinterpret_cast<float2(*)[kR3Batch][64]>(smem + 13312);
  int* R0 = reinterpret_cast<int*>(smem + 46080);
  int* R1 = R0 + kR3Batch;
  int* R2 = R1 + kR3Batch;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int nchunk = tg.nchunk;
  const int64_t wi = blockIdx.x / nchunk;
  const int chunk = (int)(blockIdx.x - wi * nchunk);
  if (wi >= plan[tg.o_nwork]) return;
  const int* meta = plan + tg.o_meta;
  const int P = meta[kR3MetaP];
  const int t = plan[tg.o_work + wi];
  const int piece = (int)(wi - plan[tg.o_wstart + t]);
  const int s0 = plan[tg.o_start + t];
  const int V = plan[tg.o_start + t + 1] - s0;
  const bool split = V > P;
  const int i0 = split ? piece * P : 0;
  const int i1 = split ? min(i0 + P, V) : V;
  const int* perm = plan + ((meta[kR3MetaPasses] & 1) ? tg.o_scratch : tg.o_perm) + s0;
  const int64_t nrows = g.B * g.C;
  const int64_t rbase = (int64_t)chunk * kR3Rows;
  const int ncc = (int)(rbase + kR3Rows < nrows ? kR3Rows : nrows - rbase);
  int org[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) org[d] = ((t / tg.bstride[d]) % tg.nb[d]) * tg.T[d];

  float2 acc[kR3T2];
#pragma unroll
  for (int z = 0; z < kR3T2; ++z) acc[z] = make_float2(0.f, 0.f);

  // Staging reads are prefetched into registers: the sample indices two batches ahead,
  // the plan's tap rows and the data one batch ahead, so that a batch's global loads are
  // in flight while the previous batch is walked.  Thread (part, e) stages entry e:
  // parts 0..2 the tap row of dimension `part`, every part the data of coil row `part`.
  const int e_s = threadIdx.x & 63, part = threadIdx.x >> 6;
  const float4* sw4 = reinterpret_cast<const float4*>(plan + tg.o_sw);
  const int* sb = plan + tg.o_sb;
  auto load_m = [&](int b) { return b + e_s < i1 ? perm[b + e_s] : -1; };
  float4 wv[3];
  int bmv = 0;
  float2 kdv = make_float2(0.f, 0.f);
  auto load_vals = [&](int m) {
    if (m < 0) return;
    if (part < 3) {
      const float4* row = sw4 + ((int64_t)part * g.M + m) * 3;
#pragma unroll
      for (int k = 0; k < 3; ++k) wv[k] = row[k];
      bmv = sb[part * g.M + m];
    }
    if (part < ncc) kdv = kdata[(rbase + part) * g.M + m];
  };
  int m_cur = load_m(i0);
  int m_nxt = load_m(i0 + kR3Batch);
  load_vals(m_cur);

  for (int base = i0; base < i1; base += kR3Batch) {
    {
      const int e = e_s;
      const bool live = m_cur >= 0;
      if (part < 3) {
        float4(*Wd)[3] = reinterpret_cast<float4(*)[3]>(part == 0 ? W0 : (part == 1 ? W1 : W2));
        int* Rd = part == 0 ? R0 : (part == 1 ? R1 : R2);
        // footprint offset in the tile: taps run from the base cell, or from its wrap
        // below the grid start when the tile lies past the grid's end
        int r = -100;  // no tap of a dead lane lands in the tile
        if (live) {
          r = bmv - org[part];
          if (r >= tg.T[part]) r -= tg.K[part];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) Wd[e][k] = live ? wv[k] : make_float4(0.f, 0.f, 0.f, 0.f);
        Rd[e] = r;
      }
      S[e][part] = (live && part < ncc) ? kdv : make_float2(0.f, 0.f);
    }
    // next batch's loads, in flight during this batch's walk
    const int m_nn = base + 2 * kR3Batch < i1 ? load_m(base + 2 * kR3Batch) : -1;
    kdv = make_float2(0.f, 0.f);
    load_vals(m_nxt);
    m_cur = m_nxt;
    m_nxt = m_nn;
    lds_barrier();  // LDS only: the prefetch loads stay in flight
    // data times the y weight for every (entry, y, row)
#pragma unroll
    for (int k = 0; k < (kR3Batch * 64) / kR3Threads; ++k) {
      const int idx = (int)threadIdx.x + k * kR3Threads;
      const int e = idx >> 6, l = idx & 63, y = l >> 3, q = l & 7;
      const int j1 = y - R1[e];
      float2 v = make_float2(0.f, 0.f);
      if (j1 >= 0 && j1 < 6) v = cmul(S[e][q], W1[e][j1]);
      Vy[e][l] = v;
    }
    lds_barrier();  // LDS only: the prefetch loads stay in flight
    // walk: entries that reach this wave's plane, by z offset
    const int r0l = R0[lane], r2l = R2[lane];
    const int jxl = wave - r0l;
    const unsigned long long hits = __ballot(jxl >= 0 && jxl < g.J[0]);
#define TKBN_R3_GROUP(C)                                                     \
  {                                                                          \
    unsigned long long mk = __ballot(r2l == (C)) & hits;                     \
    while (mk) {                                                             \
      const int e = __ffsll(mk) - 1;                                         \
      mk &= mk - 1;                                                          \
      const int jx = wave - __builtin_amdgcn_readlane(r0l, e);               \
      const float2 u = cmul(Vy[e][lane], W0[e][jx]);                         \
      r3_add_z<C>(acc, u, W2[e]);                                            \
    }                                                                        \
  }
    TKBN_R3_GROUP(-5) TKBN_R3_GROUP(-4) TKBN_R3_GROUP(-3) TKBN_R3_GROUP(-2) TKBN_R3_GROUP(-1)
    TKBN_R3_GROUP(0) TKBN_R3_GROUP(1) TKBN_R3_GROUP(2) TKBN_R3_GROUP(3) TKBN_R3_GROUP(4)
    TKBN_R3_GROUP(5) TKBN_R3_GROUP(6) TKBN_R3_GROUP(7) TKBN_R3_GROUP(8) TKBN_R3_GROUP(9)
    TKBN_R3_GROUP(10) TKBN_R3_GROUP(11) TKBN_R3_GROUP(12) TKBN_R3_GROUP(13) TKBN_R3_GROUP(14)
    TKBN_R3_GROUP(15)
#undef TKBN_R3_GROUP
    lds_barrier();  // LDS only: the prefetch loads stay in flight
  }

  // Flush through LDS (each wave its own region, after the loop's last barrier): lane
  // c's z column goes out as 16 consecutive cells, four columns per store instruction.
  float2* fl = reinterpret_cast<float2*>(smem) + wave * (64 * kR3FlushPitch);
#pragma unroll
  for (int z = 0; z < kR3T2; ++z) fl[lane * kR3FlushPitch + z] = acc[z];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int z = lane & (kR3T2 - 1);
  const int k0 = org[0] + wave, k2 = org[2] + z;
  // partial tile of a piece: slot (wi, chunk), element ((x * 8 + y) * 8 + row) * 16 + z
  float2* slot = pool + ((int64_t)wi * nchunk + chunk) * kR3SlotFloats2 + wave * 64 * kR3T2;
#pragma unroll
  for (int i = 0; i < 64 / 4; ++i) {
    const int c = 4 * i + (lane >> 4);  // source lane: y = c / 8, row = c % 8
    const float2 v = fl[c * kR3FlushPitch + z];
    if (split) {
      slot[c * kR3T2 + z] = v;
    } else {
      const int yc = c >> 3, qc = c & 7, k1 = org[1] + yc;
      if (qc < ncc && k0 < g.K[0] && k1 < g.K[1] && k2 < g.K[2])
        grid[(rbase + qc) * g.G + (int64_t)k0 * g.stride[0] + (int64_t)k1 * g.stride[1] + k2] = v;
    }
  }
}

// element idx of a hot tile's chunk: the sum of its pieces' values, in piece order
__device__ __forceinline__ void combine_unit(const Geom<float>& g, const float2* __restrict__ pool,
                                             float2* __restrict__ grid, int w0, int np, int nchunk, int chunk,
                                             int64_t rbase, int ncc, const int (&org)[3], int idx) {
  {
    // slot element ((x * 8 + y) * 8 + row) * 16 + z
    const int z = idx & (kR3T2 - 1), q = (idx / kR3T2) & (kR3Rows - 1), y = (idx / (kR3T2 * kR3Rows)) & (kR3T1 - 1);
    const int x = idx / (kR3T2 * kR3Rows * kR3T1);
    const int k0 = org[0] + x, k1 = org[1] + y, k2 = org[2] + z;
    if (q >= ncc || k0 >= g.K[0] || k1 >= g.K[1] || k2 >= g.K[2]) return;
    float2 s = pool[((int64_t)w0 * nchunk + chunk) * kR3SlotFloats2 + idx];
    for (int k = 1; k < np; ++k) {
      const float2 v = pool[((int64_t)(w0 + k) * nchunk + chunk) * kR3SlotFloats2 + idx];
      s.x = s.x + v.x;
      s.y = s.y + v.y;
    }
    grid[(rbase + q) * g.G + (int64_t)k0 * g.stride[0] + (int64_t)k1 * g.stride[1] + k2] = s;
  }
}

// Every hot tile's coil chunks, 256 elements per unit: the sum of the tile's pieces.
__global__ void __launch_bounds__(256) reg3_combine_kernel(const Geom<float> g, const TileGeom tg,
                                                          const int* __restrict__ plan,
                                                          const float2* __restrict__ pool, float2* __restrict__ grid) {
  const int* meta = plan + tg.o_meta;
  const int nhot = meta[kR3MetaHotTiles];
  const int nchunk = tg.nchunk;
  const int P = meta[kR3MetaP];
  const int64_t nrows = g.B * g.C;
  constexpr int kSlices = (int)(kR3SlotFloats2 / 256);  // 256 elements per unit
  for (int64_t unit = blockIdx.x; unit < (int64_t)nhot * nchunk * kSlices; unit += gridDim.x) {
    const int slice = (int)(unit % kSlices);
    const int chunk = (int)((unit / kSlices) % nchunk);
    const int h = (int)(unit / ((int64_t)kSlices * nchunk));
    const int t = plan[tg.o_hot + h];
    const int w0 = plan[tg.o_wstart + t];
    const int V = plan[tg.o_start + t + 1] - plan[tg.o_start + t];
    const int np = (V + P - 1) / P;
    const int64_t rbase = (int64_t)chunk * kR3Rows;
    const int ncc = (int)(rbase + kR3Rows < nrows ? kR3Rows : nrows - rbase);
    int org[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) org[d] = ((t / tg.bstride[d]) % tg.nb[d]) * tg.T[d];
    combine_unit(g, pool, grid, w0, np, nchunk, chunk, rbase, ncc, org, slice * 256 + (int)threadIdx.x);
  }
}

constexpr int kPlanReg3 = 8;  // + 1 for deterministic mode (sorted entries)

static int reg3_spread_launch(const tkbn_interp_desc* d, bool det, const void* kdata, const void* omega, void* ws,
                              void* grid, hipStream_t s) {
  const Geom<float> g = make_geom<float>(d);
  const TileGeom tg = make_reg3_geom(d, det);
  TKBN_REQUIRE(tg.maxent + tg.maxwork < (1LL << 31) && tg.plan_ints < (1LL << 31), TKBN_ERR_UNSUPPORTED,
               "3-D spread plan too large (%lld entries)", (long long)tg.maxent);
  const int kind = kPlanReg3 + (det ? 1 : 0);
  const bool reuse = plan_reused(d);
  CacheHdr* cache = nullptr;
  int st = TKBN_OK;
  int* plan = reinterpret_cast<int*>(static_cast<char*>(ws) + plan_cache_bytes(d));
  float2* pool = reinterpret_cast<float2*>(reinterpret_cast<char*>(plan) + tg.pool_off_bytes);
  if (!reuse) {
    CacheZero z;  // the tile counts
    z.p = plan + tg.o_count;
    z.n = tg.NB;
    z.stride = tg.plan_ints;
    z.copies = 1;
    st = plan_cache_begin(d, kind, tg.T, omega, ws, s, &cache, z);
    if (st != TKBN_OK) return st;
  } else {
    st = plan_registry_require(d, kind, tg.T, ws);
    if (st != TKBN_OK) return st;
  }
  const float* om = static_cast<const float*>(omega);
  if (cache) {
    const dim3 gc(bin_grid(g.M));
    if (g.M > 0) {
      reg3_sample_rows_kernel<<<dim3(bin_grid(3 * g.M)), dim3(256), 0, s>>>(g, tg, om, plan, cache);
      TKBN_LAUNCH_CHECK("reg3_sample_rows_kernel");
      bin_count_kernel<float, 3><<<gc, dim3(256), 0, s>>>(g, tg, om, plan, cache);
      TKBN_LAUNCH_CHECK("bin_count_kernel<reg3>");
    }
    reg3_plan_scan_kernel<<<dim3(1), dim3(1024), 0, s>>>(tg, plan, cache, det ? 1 : 0);
    TKBN_LAUNCH_CHECK("reg3_plan_scan_kernel");
    if (g.M > 0) {
      bin_scatter_kernel<float, 3><<<gc, dim3(256), 0, s>>>(g, tg, om, plan, cache);
      TKBN_LAUNCH_CHECK("bin_scatter_kernel<reg3>");
    }
    if (det && g.M > 0) {
      const int64_t nsort = tg.NB + tg.maxent / kR3SortChunk + 1;
      reg3_sort_chunks_kernel<<<dim3((unsigned)std::min<int64_t>(nsort, 1024)), dim3(1024), 0, s>>>(tg, plan, cache);
      TKBN_LAUNCH_CHECK("reg3_sort_chunks_kernel");
      const dim3 gm(bin_grid(tg.maxent));
      // a tile holds at most M entries (one per sample)
      const int64_t vbound = std::min<int64_t>(tg.maxent, g.M);
      for (int pass = 0; ((int64_t)kR3SortChunk << pass) < vbound; ++pass) {
        reg3_merge_kernel<<<gm, dim3(256), 0, s>>>(tg, plan, cache, pass);
        TKBN_LAUNCH_CHECK("reg3_merge_kernel");
      }
    }
  }
  profile_before(s);
  spread_reg3_kernel<<<dim3((unsigned)(tg.maxwork * tg.nchunk)), dim3(kR3Threads), 0, s>>>(
      g, tg, static_cast<const float2*>(kdata), om, plan, static_cast<float2*>(grid), pool);
  profile_after(s);
  TKBN_LAUNCH_CHECK("spread_reg3_kernel");
  reg3_combine_kernel<<<dim3(2048), dim3(256), 0, s>>>(g, tg, plan, pool, static_cast<float2*>(grid));
  TKBN_LAUNCH_CHECK("reg3_combine_kernel");
  note_kernel(det ? "spread_reg3_kernel<deterministic>" : "spread_reg3_kernel");
  return TKBN_OK;
}

constexpr int kPlanSpreadTiles = 3;  // + 1 for the deterministic tile geometry
constexpr int kPlanFwdTiles = 5;

template <typename T>
static int spread_dispatch(const Geom<T>& g, const TileGeom& tg, bool det, const void* kdata, const void* omega,
                           int* wsi, void* slot, void* grid, size_t lds, hipStream_t s, const CacheHdr* cache,
                           int ndim, int jm) {
  TKBN_DISPATCH_DJ(ndim, jm, spread_launch, g, tg, det, kdata, omega, wsi, slot, grid, lds, s, cache);
}

template <typename T>
int interp_adj_t(const tkbn_interp_desc* d, bool det, const void* kdata, const void* omega, void* grid, void* ws,
                 hipStream_t s, bool sep = true) {
  if (std::is_same<T, float>::value && reg3_eligible(d)) return reg3_spread_launch(d, det, kdata, omega, ws, grid, s);
  if (std::is_same<T, float>::value && sep && !det && coil_variant_eligible(d))
    return spread_sep_launch(d, kdata, omega, ws, grid, s);
  const Geom<T> g = make_geom<T>(d);
  const TileGeom tg = make_tile_geom(d, det);
  const size_t lds = spread_lds_bytes(d, tg, det);
  const int64_t nplans = d->omega_batched ? d->batch : 1;
  const int kind = kPlanSpreadTiles + (det ? 1 : 0);
  const bool reuse = plan_reused(d);
  CacheHdr* cache = nullptr;
  int st = TKBN_OK;
  int* wsi = reinterpret_cast<int*>(static_cast<char*>(ws) + plan_cache_bytes(d));
  void* slot = reinterpret_cast<char*>(wsi) + nplans * tg.plan_ints * 4;
  if (!reuse) {
    // the check kernel clears every plan's counts and the max|kdata| slot
    CacheZero z;
    z.p = wsi + tg.o_count;
    z.n = tg.NB;
    z.stride = tg.plan_ints;
    z.copies = nplans;
    z.p2 = static_cast<int*>(slot);
    z.n2 = 2;
    st = plan_cache_begin(d, kind, tg.T, omega, ws, s, &cache, z);
    if (st != TKBN_OK) return st;
  } else {
    st = plan_registry_require(d, kind, tg.T, ws);
    if (st != TKBN_OK) return st;
  }
  st = spread_dispatch<T>(g, tg, det, kdata, omega, wsi, slot, grid, lds, s, cache, d->ndim, max_numpoints(d));
  if (st != TKBN_OK && !reuse) plan_cache_invalidate(ws, s);
  return st;
}

template <typename T, int D, int JM>
int fwd_tiled_launch(const Geom<T>& g, const TileGeom& tg, const void* grid, const void* omega, int* ws, void* kdata,
                     hipStream_t s, const CacheHdr* cache) {
  const int64_t nrows = g.batched ? g.C : g.B * g.C;
  const int64_t zdim = g.batched ? g.B : 1;
  if (cache) {  // no header: the caller reuses the plan
    dim3 gc(bin_grid(g.M), 1, (unsigned)zdim);
    bin_count_kernel<T, D><<<gc, dim3(256), 0, s>>>(g, tg, static_cast<const T*>(omega), ws, cache);
    TKBN_LAUNCH_CHECK("bin_count_kernel<own>");
    plan_scan_kernel<<<dim3((unsigned)zdim), dim3(1024), 0, s>>>(tg, ws, cache);
    TKBN_LAUNCH_CHECK("plan_scan_kernel<own>");
    bin_scatter_kernel<T, D><<<gc, dim3(256), 0, s>>>(g, tg, static_cast<const T*>(omega), ws, cache);
    TKBN_LAUNCH_CHECK("bin_scatter_kernel<own>");
  }
  const size_t lds = (size_t)tg.CC * tg.rcells * sizeof(cplx<T>);
  interp_fwd_tiled_kernel<T, D, JM>
      <<<dim3((unsigned)tg.maxwork, (unsigned)ceil_div(nrows, tg.CC), (unsigned)zdim), dim3(fwd_tiled_threads<T, JM, D>()),
         lds, s>>>(g, tg, static_cast<const cplx<T>*>(grid), static_cast<const T*>(omega), ws,
                   static_cast<cplx<T>*>(kdata));
  TKBN_LAUNCH_CHECK("interp_fwd_tiled_kernel");
  note_kernel("interp_fwd_tiled_kernel");
  return TKBN_OK;
}

template <typename T>
static int fwd_tiled_dispatch(const Geom<T>& g, const TileGeom& tg, const void* grid, const void* omega, int* wsi,
                              void* kdata, hipStream_t s, const CacheHdr* cache, int ndim, int jm) {
  TKBN_DISPATCH_DJ(ndim, jm, fwd_tiled_launch, g, tg, grid, omega, wsi, kdata, s, cache);
}

template <typename T>
int interp_fwd_tiled_t(const tkbn_interp_desc* d, const void* grid, const void* omega, void* kdata, void* ws,
                       hipStream_t s) {
  const Geom<T> g = make_geom<T>(d);
  const TileGeom tg = make_tile_geom(d, false, true);
  const int64_t nplans = d->omega_batched ? d->batch : 1;
  const bool reuse = plan_reused(d);
  CacheHdr* cache = nullptr;
  int st = TKBN_OK;
  int* wsi = reinterpret_cast<int*>(static_cast<char*>(ws) + plan_cache_bytes(d));
  if (!reuse) {
    CacheZero z;  // every plan's counts
    z.p = wsi + tg.o_count;
    z.n = tg.NB;
    z.stride = tg.plan_ints;
    z.copies = nplans;
    st = plan_cache_begin(d, kPlanFwdTiles, tg.T, omega, ws, s, &cache, z);
    if (st != TKBN_OK) return st;
  } else {
    st = plan_registry_require(d, kPlanFwdTiles, tg.T, ws);
    if (st != TKBN_OK) return st;
  }
  st = fwd_tiled_dispatch<T>(g, tg, grid, omega, wsi, kdata, s, cache, d->ndim, max_numpoints(d));
  if (st != TKBN_OK && !reuse) plan_cache_invalidate(ws, s);
  return st;
}

// ---- separable forward gather ----------------------------------------------------
static TileGeom make_gather_geom(const tkbn_interp_desc* d) {
  TileGeom tg{};
  const int TT[2] = {kGatT0, kGatT1};
  for (int i = 0; i < 2; ++i) {
    tg.K[i] = (int)d->grid_size[i];
    tg.J[i] = (int)d->numpoints[i];
    tg.T[i] = TT[i];
    tg.nb[i] = (int)ceil_div(d->grid_size[i], TT[i]);
  }
  tg.K[2] = tg.J[2] = tg.T[2] = tg.nb[2] = 1;
  tg.bstride[1] = 1;
  tg.bstride[0] = tg.nb[1];
  tg.bstride[2] = 0;
  tg.NB = tg.nb[0] * tg.nb[1];
  tg.own_only = 1;
  tg.target = kGatTarget;
  const int64_t M = d->klength;
  tg.maxent = M;
  tg.maxwork = tg.NB + M / tg.target + 1;
  tg.ftarget = make_fastdiv((uint32_t)tg.target);
  return tg;
}

static int64_t sep_fwd_bytes(const tkbn_interp_desc* d) {
  SepGeom sg;
  make_sep_gather_geom(d, &sg);
  return plan_cache_bytes(d) + sg.end * 4;
}

int64_t interp_fwd_workspace_bytes(const tkbn_interp_desc* d) {
  if (sep_eligible(d)) return sep_fwd_bytes(d);
  const TileGeom tg = make_tile_geom(d, false, true);
  const size_t lds = (size_t)tg.CC * tg.rcells * (d->dtype == TKBN_F32 ? 8 : 16);
  if (lds > (size_t)kLdsBudget) return 0;  // region too large for LDS: plain kernel
  return plan_cache_bytes(d) + spread_workspace_bytes(d, tg);
}

int interp_fwd_tiled(const tkbn_interp_desc* d, const void* grid, const void* omega, void* kdata, void* ws,
                     hipStream_t s) {
  if (sep_eligible(d)) return gather_sep_launch(d, grid, omega, kdata, ws, s);
  if (d->dtype == TKBN_F32) return interp_fwd_tiled_t<float>(d, grid, omega, kdata, ws, s);
  return interp_fwd_tiled_t<double>(d, grid, omega, kdata, ws, s);
}


// ---------------------------------------------------------------------------
// batches of uneven problems (complex64, separable and sample-lane paths): one launch per stage
//   The caller builds every problem's plans with ordinary tkbn_interp_fwd / _adj calls
//   (the same workspaces), then describes the problems once (tkbn_batch_create); the
//   library writes a table of per-problem records (geometry, tile plans, pointers) that
//   the caller copies to device memory.  Each batched call then computes the work-item
//   offsets of all problems on the device (their plans' work counts) and runs one launch
//   per stage: block -> (problem, work item) by a binary search over the offsets, and
//   the same per-item code as the single-problem kernels.
// ---------------------------------------------------------------------------
struct BatchProb {
  Geom<float> g;
  TileGeom tf, ta;         // forward / adjoint tile plans (of either kind)
  const float2* grid_in;   // forward input grid
  float2* kdata_out;       // forward output
  const float2* kdata_in;  // adjoint input
  float2* grid_out;        // adjoint output grid (fully overwritten)
  const float* omega;
  SepGeom sf, sa;          // separable plans (sep_f, sep_a: which kind the plan above is)
  int sep_f, sep_a;
  const int* wf;           // forward plan (past the workspace's cache header)
  const int* wa;           // adjoint plan
  void* slot;              // adjoint max|re|,|im| slot (8 bytes, cleared each call)
  int64_t yf, ya;          // coil-row chunks per work item, forward / adjoint
  int64_t zoff;            // first zero-hot block of this problem (host prefix of NB * ya)
  int64_t nom;             // trajectory values (ndim * klength)
};

// Offsets of the problems' work items: off_f[p] = sum_{q < p} nwork_f(q) * yf(q) (and
// off_a the same for the adjoint), off[nprob] the totals; clears every adjoint slot.  Both
// kinds of problem (separable, sample-lane) are counted; each kind's launch passes over
// the other's items.
__global__ void __launch_bounds__(1024) batch_offsets_kernel(const BatchProb* __restrict__ probs, int nprob,
                                                             int* __restrict__ off_f, int* __restrict__ off_a,
                                                             int clear_slots) {
  __shared__ int sbuf[1024];
  __shared__ int cf[1024], ca[1024];
  __shared__ int base[2];
  if (threadIdx.x == 0) base[0] = base[1] = 0;
  for (int p0 = 0; p0 < nprob; p0 += 1024) {
    const int n = min(1024, nprob - p0);
    if ((int)threadIdx.x < n) {
      const BatchProb& q = probs[p0 + threadIdx.x];
      cf[threadIdx.x] = q.wf[q.tf.o_nwork] * (int)q.yf;
      ca[threadIdx.x] = q.wa[q.ta.o_nwork] * (int)q.ya;
      if (clear_slots && !q.sep_a) *static_cast<unsigned long long*>(q.slot) = 0ull;
    }
    __syncthreads();
    block_exclusive_scan(cf, off_f + p0, n, sbuf);  // off_f[p0 .. p0 + n]
    block_exclusive_scan(ca, off_a + p0, n, sbuf);
    for (int i = threadIdx.x; i <= n; i += blockDim.x) {
      off_f[p0 + i] += base[0];
      off_a[p0 + i] += base[1];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      base[0] = off_f[p0 + n];
      base[1] = off_a[p0 + n];
    }
    __syncthreads();
  }
}

// largest p with off[p] <= item (off[0] = 0 <= item < off[nprob])
__device__ __forceinline__ int batch_find(const int* off, int nprob, int item) {
  int lo = 0, hi = nprob;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= item) lo = mid;
    else hi = mid;
  }
  return lo;
}

template <int D, int JM>
__global__ void __launch_bounds__((fwd_tiled_threads<float, JM, D>()))
    batch_fwd_kernel(const BatchProb* __restrict__ probs, int nprob, const int* __restrict__ off) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int item = blockIdx.x;
  if (item >= off[nprob]) return;
  const int p = batch_find(off, nprob, item);
  const BatchProb& q = probs[p];
  if (q.sep_f) return;
  const int li = item - off[p];
  const int64_t wi = li / q.yf, yc = li - wi * q.yf;
  fwd_tiled_item<float, D, JM>(q.g, q.tf, q.grid_in, q.omega, q.wf, q.kdata_out, wi, yc, 0, smem_raw);
}

template <int D>
__global__ void __launch_bounds__(256) batch_zero_hot_kernel(const BatchProb* __restrict__ probs, int nprob) {
  const int64_t blk = blockIdx.x;
  int lo = 0, hi = nprob;  // largest p with zoff(p) <= blk
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (probs[mid].zoff <= blk) lo = mid;
    else hi = mid;
  }
  const BatchProb& q = probs[lo];
  const int64_t li = blk - q.zoff;
  const int64_t t = li / q.ya, yc = li - t * q.ya;
  if (t >= q.ta.NB) return;
  if constexpr (D == 2) {
    if (q.sep_a) {  // the first chunk's block clears all rows (fewer than 32)
      if (yc == 0) sep_zero_hot_item(q.g, q.ta, q.wa, q.grid_out, (int)t, 0, q.g.B * q.g.C);
      return;
    }
  }
  zero_hot_tiles_item<float, D>(q.g, q.ta, q.wa, q.grid_out, (int)t, yc, 0);
}

// max |re|, |im| of each problem's samples (blockIdx.y = problem), +inf for a non-finite
// sample or trajectory value, into the problem's slot
__global__ void __launch_bounds__(256) batch_maxabs_kernel(const BatchProb* __restrict__ probs) {
  const BatchProb& q = probs[blockIdx.y];
  if (q.sep_a) return;  // the separable spread needs no bound
  const float* x = reinterpret_cast<const float*>(q.kdata_in);
  const int64_t n = q.g.B * q.g.C * q.g.M * 2;
  float mx = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float v = fabsf(x[i]);
    mx = isfinite(v) ? (v > mx ? v : mx) : INFINITY;
  }
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < q.nom; i += (int64_t)gridDim.x * blockDim.x)
    if (!isfinite(q.omega[i])) mx = INFINITY;
  for (int o = 32; o > 0; o >>= 1) {
    const float v = __shfl_down(mx, o, 64);
    mx = v > mx ? v : mx;
  }
  __shared__ float wmax[4];
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) mx = wmax[w] > mx ? wmax[w] : mx;
    unsigned int bits;
    memcpy(&bits, &mx, sizeof(bits));
    atomicMax(static_cast<unsigned int*>(q.slot), bits);
  }
}

template <bool FIXED, int D, int JM>
__global__ void __launch_bounds__(spread_tiles_threads(D))
    batch_spread_kernel(const BatchProb* __restrict__ probs, int nprob, const int* __restrict__ off, int fallback) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int item = blockIdx.x;
  if (item >= off[nprob]) return;
  const int p = batch_find(off, nprob, item);
  const BatchProb& q = probs[p];
  if (q.sep_a) return;
  const int li = item - off[p];
  const int64_t wi = li / q.ya, yc = li - wi * q.ya;
  spread_tiles_item<float, FIXED, D, JM>(q.g, q.ta, q.kdata_in, q.omega, q.wa, q.slot, q.grid_out, fallback, wi, yc, 0,
                                         smem_raw);
}

// the separable problems of a batch: a group (gather) or a wave (spread) per item
template <int ROWS>
__global__ void __launch_bounds__(GatShape<ROWS>::kThreads)
    batch_gather_sep_kernel(const BatchProb* __restrict__ probs, int nprob, const int* __restrict__ off) {
  __shared__ __attribute__((aligned(16))) float2 region[kGatCells * GatShape<ROWS>::kPitch];
  __shared__ float2 ph[kGatR0 + kGatR1];
  const int item = blockIdx.x;
  if (item >= off[nprob]) return;
  const int p = batch_find(off, nprob, item);
  const BatchProb& q = probs[p];
  if (!q.sep_f) return;
  const int li = item - off[p];
  const int64_t wi = li / q.yf;
  const int yc = (int)(li - wi * q.yf);
  if (q.g.J[0] == 6 && q.g.J[1] == 6)
    gather_sep_item<6, ROWS>(q.g, q.tf, q.sf, q.grid_in, q.omega, q.wf, q.wf, q.kdata_out, 0, q.g.B * q.g.C, wi, yc, region,
                             ph);
  else
    gather_sep_item<0, ROWS>(q.g, q.tf, q.sf, q.grid_in, q.omega, q.wf, q.wf, q.kdata_out, 0, q.g.B * q.g.C, wi, yc, region,
                             ph);
}

template <int G>
__global__ void __launch_bounds__(64 * kMmWaves) __attribute__((amdgpu_waves_per_eu(mm_waves(G))))
    batch_spread_sep_kernel(const BatchProb* __restrict__ probs, int nprob, const int* __restrict__ off, int ks) {
  __shared__ MmLds<G> lds[kMmWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = ks == 1 ? blockIdx.x * kMmWaves + wave : blockIdx.x;
  if (item >= off[nprob]) return;
  const int p = __builtin_amdgcn_readfirstlane(batch_find(off, nprob, item));
  const BatchProb& q = probs[p];
  if (!q.sep_a) return;
  const int li = item - off[p];
  const int64_t wi = li / q.ya;
  spread_sep_item<G>(q.g, q.ta, q.sa, q.kdata_in, q.omega, q.wa, q.wa, q.grid_out, 0, q.g.B * q.g.C, wi,
                     (int)(li - wi * q.ya), ks, wave, lds, lds[wave]);
}

}  // namespace tkbn

struct tkbn_batch {
  int nprob = 0, ndim = 0, jm = 6, det = 0;
  int gat_rows = 1, form = 1, ks = 1;              // shapes of the separable launches (the largest problem's rows)
  int nsep_f = 0, nsep_a = 0;              // separable problems
  std::vector<tkbn::BatchProb> probs;
  std::vector<int64_t> rows;
  std::vector<tkbn_interp_desc> descs_f, descs_a;
  std::vector<const void*> wsf, wsa;
  size_t lds_f = 0, lds_a = 0;
  int64_t bound_f = 0, bound_a = 0, zblocks = 0, maxabs_blocks = 1;
};

namespace tkbn {

// the batch's plans must be the ones its workspaces hold (same check as TKBN_PLAN_REUSE)
static int batch_plans_current(const tkbn_batch* b) {
  for (int p = 0; p < b->nprob; ++p) {
    const BatchProb& q = b->probs[p];
    int st = plan_registry_require(&b->descs_f[p], q.sep_f ? kPlanSepGather : kPlanFwdTiles, q.tf.T, b->wsf[p]);
    if (st != TKBN_OK) return st;
    st = plan_registry_require(&b->descs_a[p], q.sep_a ? kPlanSepSpread : kPlanSpreadTiles + b->det, q.ta.T, b->wsa[p]);
    if (st != TKBN_OK) return st;
  }
  return TKBN_OK;
}

// the two descriptors of a problem agree on everything but the tuning fields
static bool same_geometry(const tkbn_interp_desc* a, const tkbn_interp_desc* b) {
  if (a->dtype != b->dtype || a->ndim != b->ndim || a->batch != b->batch || a->coils != b->coils ||
      a->klength != b->klength || a->omega_batched != b->omega_batched)
    return false;
  for (int i = 0; i < a->ndim; ++i)
    if (a->grid_size[i] != b->grid_size[i] || a->numpoints[i] != b->numpoints[i] ||
        a->table_oversamp[i] != b->table_oversamp[i] || a->n_shift[i] != b->n_shift[i] || a->tables[i] != b->tables[i])
      return false;
  return true;
}

}  // namespace tkbn

extern "C" {

int tkbn_batch_create(const tkbn_interp_desc* descs, const tkbn_interp_desc* adj_descs, int32_t nprob, int32_t mode,
                      const void* const* grids_in,
                      void* const* kdatas_out, const void* const* kdatas_in, void* const* grids_out,
                      const void* const* omegas, void* const* fwd_workspaces, void* const* adj_workspaces,
                      tkbn_batch** out) {
  using namespace tkbn;
  TKBN_REQUIRE(out != nullptr && descs != nullptr && nprob >= 1, TKBN_ERR_INVALID, "tkbn_batch_create: no problems");
  TKBN_REQUIRE(mode == TKBN_ADJ_ATOMIC || mode == TKBN_ADJ_DETERMINISTIC, TKBN_ERR_INVALID, "bad adjoint mode %d", mode);
  *out = nullptr;
  tkbn_batch* b = new tkbn_batch();
  b->nprob = nprob;
  b->det = mode == TKBN_ADJ_DETERMINISTIC ? 1 : 0;
  b->ndim = descs[0].ndim;
  b->jm = max_numpoints(&descs[0]) <= 6 ? 6 : 16;
  int64_t zoff = 0, entries = 0, tiles = 0, items = 0;
  for (int p = 0; p < nprob; ++p) {
    const tkbn_interp_desc* d = &descs[p];
    const tkbn_interp_desc* da = adj_descs ? &adj_descs[p] : d;
    int st = validate_desc(d);
    if (st == TKBN_OK) st = validate_desc(da);
    if (st == TKBN_OK && !same_geometry(d, da)) {
      set_error("tkbn_batch_create: problem %d: forward and adjoint descriptors differ in more than tuning", p);
      st = TKBN_ERR_INVALID;
    }
    if (st == TKBN_OK && (d->dtype != TKBN_F32 || d->ndim != b->ndim || d->omega_batched ||
                          (max_numpoints(d) <= 6 ? 6 : 16) != b->jm)) {
      set_error("tkbn_batch_create: problem %d: batches take complex64 problems of one dimension and numpoints "
                "class with unbatched trajectories", p);
      st = TKBN_ERR_UNSUPPORTED;
    }
    if (st == TKBN_OK && ((d->ndim == 2 && d->numpoints[0] <= 6 && d->numpoints[1] <= 6 && d->batch * d->coils >= 32) ||
                          interp_fwd_workspace_bytes(d) <= 0 || reg3_eligible(da))) {
      set_error("tkbn_batch_create: problem %d takes a path of its own or is unbinned; batches take problems of "
                "fewer than 32 coil rows (2-D) or 4 (3-D)", p);
      st = TKBN_ERR_UNSUPPORTED;
    }
    if (st == TKBN_OK && !(grids_in && grids_in[p] && kdatas_out && kdatas_out[p] && kdatas_in && kdatas_in[p] &&
                           grids_out && grids_out[p] && omegas && omegas[p] && fwd_workspaces &&
                           fwd_workspaces[p] && adj_workspaces && adj_workspaces[p])) {
      set_error("tkbn_batch_create: problem %d: NULL pointer", p);
      st = TKBN_ERR_INVALID;
    }
    if (st != TKBN_OK) {
      delete b;
      return st;
    }
    BatchProb q{};
    q.g = make_geom<float>(d);
    q.sep_f = sep_eligible(d) ? 1 : 0;
    q.sep_a = !b->det && coil_variant_eligible(da) ? 1 : 0;
    q.tf = q.sep_f ? make_sep_gather_geom(d, &q.sf) : make_tile_geom(d, false, true);
    q.ta = q.sep_a ? make_sep_spread_geom(da, &q.sa) : make_tile_geom(da, b->det != 0);
    b->nsep_f += q.sep_f;
    b->nsep_a += q.sep_a;
    q.grid_in = static_cast<const float2*>(grids_in[p]);
    q.kdata_out = static_cast<float2*>(kdatas_out[p]);
    q.kdata_in = static_cast<const float2*>(kdatas_in[p]);
    q.grid_out = static_cast<float2*>(grids_out[p]);
    q.omega = static_cast<const float*>(omegas[p]);
    const int64_t hdr = plan_cache_bytes(d);
    q.wf = reinterpret_cast<const int*>(static_cast<const char*>(fwd_workspaces[p]) + hdr);
    q.wa = reinterpret_cast<const int*>(static_cast<const char*>(adj_workspaces[p]) + hdr);
    q.slot = q.sep_a ? nullptr : static_cast<char*>(adj_workspaces[p]) + hdr + q.ta.plan_ints * 4;
    const int64_t nrows = d->batch * d->coils;
    if (q.sep_f) b->gat_rows = std::max(b->gat_rows, gat_rows(nrows));
    if (q.sep_a) {
      b->form = std::max(b->form, mm_form(da));
      entries += sep_entries(da);
      tiles += q.ta.NB;
    }
    b->rows.push_back(nrows);
    q.nom = (int64_t)d->ndim * d->klength;
    b->maxabs_blocks = std::max<int64_t>(b->maxabs_blocks, std::min<int64_t>(ceil_div(nrows * d->klength * 2, 4096), 64));
    b->probs.push_back(q);
    b->descs_f.push_back(*d);
    b->descs_f.back().flags = 0;
    b->descs_a.push_back(*da);
    b->descs_a.back().flags = 0;
    b->wsf.push_back(fwd_workspaces[p]);
    b->wsa.push_back(adj_workspaces[p]);
  }
  // row chunks per work item: one shape for all separable problems of a launch
  for (int p = 0; p < nprob; ++p) {
    BatchProb& q = b->probs[p];
    q.yf = ceil_div(b->rows[p], q.sep_f ? b->gat_rows : q.tf.CC);
    q.ya = ceil_div(b->rows[p], q.sep_a ? mm_rows(b->form) : q.ta.CC);
    if (q.sep_a) items += q.ta.NB * q.ya;
    q.zoff = zoff;
    zoff += (int64_t)q.ta.NB * q.ya;
    if (!q.sep_f) b->lds_f = std::max(b->lds_f, (size_t)q.tf.CC * q.tf.rcells * sizeof(float2));
    if (!q.sep_a) b->lds_a = std::max(b->lds_a, spread_lds_bytes(&b->descs_a[p], q.ta, b->det != 0));
    b->bound_f += q.tf.maxwork * q.yf;
    b->bound_a += q.ta.maxwork * q.ya;
  }
  b->zblocks = zoff;
  b->ks = mm_waves_per_item(entries, tiles, items);  // of all problems: together they fill the chip
  if (b->bound_f >= (1LL << 31) || b->bound_a >= (1LL << 31) || b->zblocks >= (1LL << 31)) {
    set_error("tkbn_batch_create: too many work items for one launch");
    delete b;
    return TKBN_ERR_UNSUPPORTED;
  }
  *out = b;
  return TKBN_OK;
}

int tkbn_batch_destroy(tkbn_batch* b) {
  delete b;
  return TKBN_OK;
}

int64_t tkbn_batch_table_bytes(const tkbn_batch* b) {
  return b ? (int64_t)(b->probs.size() * sizeof(tkbn::BatchProb)) : -1;
}

int tkbn_batch_write_table(const tkbn_batch* b, void* host_dst) {
  TKBN_REQUIRE(b != nullptr && host_dst != nullptr, TKBN_ERR_INVALID, "tkbn_batch_write_table: NULL argument");
  memcpy(host_dst, b->probs.data(), b->probs.size() * sizeof(tkbn::BatchProb));
  return TKBN_OK;
}

int64_t tkbn_batch_workspace_bytes(const tkbn_batch* b) {
  return b ? (int64_t)(2 * (b->nprob + 1) * sizeof(int)) : -1;
}

int tkbn_batch_interp_fwd(const tkbn_batch* b, const void* table, void* workspace, int64_t workspace_bytes,
                          void* stream) {
  using namespace tkbn;
  TKBN_REQUIRE(b != nullptr && table != nullptr && workspace != nullptr, TKBN_ERR_INVALID, "tkbn_batch_interp_fwd: NULL argument");
  TKBN_REQUIRE(workspace_bytes >= tkbn_batch_workspace_bytes(b), TKBN_ERR_WORKSPACE, "batch workspace too small");
  int st = batch_plans_current(b);
  if (st != TKBN_OK) return st;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto* probs = static_cast<const BatchProb*>(table);
  int* off_f = static_cast<int*>(workspace);
  int* off_a = off_f + b->nprob + 1;
  batch_offsets_kernel<<<dim3(1), dim3(1024), 0, s>>>(probs, b->nprob, off_f, off_a, 0);
  TKBN_LAUNCH_CHECK("batch_offsets_kernel");
  if (b->bound_f == 0) return TKBN_OK;
  const dim3 grd((unsigned)b->bound_f);
#define TKBN_BATCH_FWD(DD, JJ) \
  batch_fwd_kernel<DD, JJ><<<grd, dim3(fwd_tiled_threads<float, JJ, DD>()), b->lds_f, s>>>(probs, b->nprob, off_f)
  if (b->nsep_f > 0) {
    switch (b->gat_rows) {
#define TKBN_BATCH_GAT(R) \
  batch_gather_sep_kernel<R><<<grd, dim3(GatShape<R>::kThreads), 0, s>>>(probs, b->nprob, off_f)
      case 16: TKBN_BATCH_GAT(16); break;
      case 8: TKBN_BATCH_GAT(8); break;
      case 4: TKBN_BATCH_GAT(4); break;
      case 2: TKBN_BATCH_GAT(2); break;
      default: TKBN_BATCH_GAT(1); break;
#undef TKBN_BATCH_GAT
    }
    TKBN_LAUNCH_CHECK("batch_gather_sep_kernel");
  }
  if (b->nsep_f == b->nprob) {
    note_kernel("batch_fwd_kernel");
    return TKBN_OK;
  }
  if (b->jm == 6) {
    if (b->ndim == 1) TKBN_BATCH_FWD(1, 6);
    else if (b->ndim == 2) TKBN_BATCH_FWD(2, 6);
    else TKBN_BATCH_FWD(3, 6);
  } else {
    if (b->ndim == 1) TKBN_BATCH_FWD(1, 16);
    else if (b->ndim == 2) TKBN_BATCH_FWD(2, 16);
    else TKBN_BATCH_FWD(3, 16);
  }
#undef TKBN_BATCH_FWD
  TKBN_LAUNCH_CHECK("batch_fwd_kernel");
  note_kernel("batch_fwd_kernel");
  return TKBN_OK;
}

int tkbn_batch_interp_adj(const tkbn_batch* b, const void* table, void* workspace, int64_t workspace_bytes,
                          void* stream) {
  using namespace tkbn;
  TKBN_REQUIRE(b != nullptr && table != nullptr && workspace != nullptr, TKBN_ERR_INVALID, "tkbn_batch_interp_adj: NULL argument");
  TKBN_REQUIRE(workspace_bytes >= tkbn_batch_workspace_bytes(b), TKBN_ERR_WORKSPACE, "batch workspace too small");
  int st = batch_plans_current(b);
  if (st != TKBN_OK) return st;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto* probs = static_cast<const BatchProb*>(table);
  int* off_f = static_cast<int*>(workspace);
  int* off_a = off_f + b->nprob + 1;
  batch_offsets_kernel<<<dim3(1), dim3(1024), 0, s>>>(probs, b->nprob, off_f, off_a, 1);
  TKBN_LAUNCH_CHECK("batch_offsets_kernel");
  if (!b->det && b->zblocks > 0) {
    if (b->ndim == 1) batch_zero_hot_kernel<1><<<dim3((unsigned)b->zblocks), dim3(256), 0, s>>>(probs, b->nprob);
    else if (b->ndim == 2) batch_zero_hot_kernel<2><<<dim3((unsigned)b->zblocks), dim3(256), 0, s>>>(probs, b->nprob);
    else batch_zero_hot_kernel<3><<<dim3((unsigned)b->zblocks), dim3(256), 0, s>>>(probs, b->nprob);
    TKBN_LAUNCH_CHECK("batch_zero_hot_kernel");
  }
  if (b->nsep_a < b->nprob) {
    batch_maxabs_kernel<<<dim3((unsigned)b->maxabs_blocks, (unsigned)b->nprob), dim3(256), 0, s>>>(probs);
    TKBN_LAUNCH_CHECK("batch_maxabs_kernel");
  }
  if (b->bound_a == 0) return TKBN_OK;
  const dim3 grd((unsigned)b->bound_a);
  if (b->nsep_a > 0) {
    const dim3 gs((unsigned)ceil_div(b->bound_a, kMmWaves / b->ks)), blk(64 * kMmWaves);
    switch (b->form) {
      case 1: batch_spread_sep_kernel<1><<<gs, blk, 0, s>>>(probs, b->nprob, off_a, b->ks); break;
      case 2: batch_spread_sep_kernel<2><<<gs, blk, 0, s>>>(probs, b->nprob, off_a, b->ks); break;
      case 4: batch_spread_sep_kernel<4><<<gs, blk, 0, s>>>(probs, b->nprob, off_a, b->ks); break;
      default: batch_spread_sep_kernel<8><<<gs, blk, 0, s>>>(probs, b->nprob, off_a, b->ks); break;
    }
    TKBN_LAUNCH_CHECK("batch_spread_sep_kernel");
  }
  if (b->nsep_a == b->nprob) {
    note_kernel("batch_spread_kernel<sep>");
    return TKBN_OK;
  }
#define TKBN_BATCH_ADJ(FX, DD, JJ, FB) \
  batch_spread_kernel<FX, DD, JJ><<<grd, dim3(spread_tiles_threads(DD)), b->lds_a, s>>>(probs, b->nprob, off_a, FB)
#define TKBN_BATCH_ADJ_PAIR(DD, JJ)      \
  do {                                   \
    TKBN_BATCH_ADJ(true, DD, JJ, 0);     \
    TKBN_BATCH_ADJ(false, DD, JJ, 1);    \
  } while (0)
  if (b->jm == 6) {
    if (b->ndim == 1) TKBN_BATCH_ADJ_PAIR(1, 6);
    else if (b->ndim == 2) TKBN_BATCH_ADJ_PAIR(2, 6);
    else TKBN_BATCH_ADJ_PAIR(3, 6);
  } else {
    if (b->ndim == 1) TKBN_BATCH_ADJ_PAIR(1, 16);
    else if (b->ndim == 2) TKBN_BATCH_ADJ_PAIR(2, 16);
    else TKBN_BATCH_ADJ_PAIR(3, 16);
  }
#undef TKBN_BATCH_ADJ_PAIR
#undef TKBN_BATCH_ADJ
  TKBN_LAUNCH_CHECK("batch_spread_kernel");
  note_kernel(b->det ? "batch_spread_kernel<fixed,deterministic>" : "batch_spread_kernel<fixed>");
  return TKBN_OK;
}

}  // extern "C"

// ---- adjoint without device allocation -------------------------------------------
// tkbn_interp_adj_noalloc keeps its workspace (plan-cache header, trajectory copy,
// plan) in `scratch`, a static device array that every GPU the library runs on holds
// from code-object load until the process ends.  In host code `scratch` names a
// host-side stand-in, never the device memory: the device address comes from
// hipGetSymbolAddress, once per device with that device current, and only that
// address is passed to kernels.
namespace tkbn {
constexpr int64_t kNoAllocScratchBytes = 128ll << 20;
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace tkbn

static __device__ __align__(256) unsigned char scratch[tkbn::kNoAllocScratchBytes];

namespace tkbn {
// Device address of the current device's `scratch`; the first call on a device zeroes
// its plan-cache header (a zero header never matches, so the first call builds).
static int noalloc_scratch(hipStream_t s, void** out) {
  int dev = -1;
  TKBN_HIP_CHECK(hipGetDevice(&dev));
  TKBN_REQUIRE(dev >= 0 && dev < kMaxDevices, TKBN_ERR_UNSUPPORTED, "device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    TKBN_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    TKBN_REQUIRE(p != nullptr, TKBN_ERR_HIP, "hipGetSymbolAddress returned NULL for the scratch array");
    const int st = launch_zero_fill(static_cast<uint32_t*>(p), kCacheHdrBytes / 4, s);
    if (st != TKBN_OK) return st;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return TKBN_OK;
}
}  // namespace tkbn

using namespace tkbn;

extern "C" {

int64_t tkbn_interp_adj_noalloc_max_bytes(void) { return kNoAllocScratchBytes; }

int tkbn_interp_adj_noalloc(const tkbn_interp_desc* desc, const void* kdata, const void* omega, void* grid,
                            int32_t mode, void* stream) {
  int st = validate_desc(desc);
  if (st != TKBN_OK) return st;
  TKBN_REQUIRE(mode == TKBN_ADJ_ATOMIC || mode == TKBN_ADJ_DETERMINISTIC, TKBN_ERR_INVALID, "bad adjoint mode %d", mode);
  TKBN_REQUIRE(desc->flags == 0, TKBN_ERR_INVALID,
               "tkbn_interp_adj_noalloc takes no flags (its scratch may hold another call's plan)");
  if (desc->batch == 0 || desc->coils == 0) return TKBN_OK;
  // The scratch holds one path's plan at a time.  Fewer than 32 coil rows fall back to the
  // sample-lane kernels, whose plan is smaller, where the separable plan does not fit.
  const bool det = mode == TKBN_ADJ_DETERMINISTIC;
  int64_t need = tkbn_interp_adj_workspace_bytes(desc, mode);
  bool sep = true;
  if (!det && coil_variant_eligible(desc)) {
    need = sep_adj_bytes(desc);
    if (need > kNoAllocScratchBytes && (desc->omega_batched || desc->batch * desc->coils < 32)) {
      sep = false;
      need = adj_lane_bytes(desc, det);
    }
  } else if (!det && desc->dtype == TKBN_F32 && desc->ndim == 2) {
    need = adj_lane_bytes(desc, det);
  }
  TKBN_REQUIRE(need >= 0 && need <= kNoAllocScratchBytes, TKBN_ERR_WORKSPACE,
               "tkbn_interp_adj_noalloc: this problem needs %lld bytes of workspace, more than the %lld-byte "
               "static scratch; use tkbn_interp_adj with a caller workspace",
               (long long)need, (long long)kNoAllocScratchBytes);
  hipStream_t s = static_cast<hipStream_t>(stream);
  void* ws = nullptr;
  st = noalloc_scratch(s, &ws);
  if (st != TKBN_OK) return st;
  TKBN_REQUIRE(grid != nullptr, TKBN_ERR_INVALID, "NULL grid pointer");
  TKBN_REQUIRE(desc->klength == 0 || (kdata && omega), TKBN_ERR_INVALID, "NULL data pointer");
  TKBN_REQUIRE(desc->klength < (1LL << 31), TKBN_ERR_INVALID, "klength must be < 2^31");
  if (desc->dtype == TKBN_F32) return interp_adj_t<float>(desc, det, kdata, omega, grid, ws, s, sep);
  return interp_adj_t<double>(desc, det, kdata, omega, grid, ws, s);
}

int tkbn_profile_next_kernel(void* start_event, void* stop_event) {
  g_profile.start = static_cast<hipEvent_t>(start_event);
  g_profile.stop = static_cast<hipEvent_t>(stop_event);
  return TKBN_OK;
}

int64_t tkbn_interp_adj_workspace_bytes(const tkbn_interp_desc* desc, int32_t mode) {
  if (validate_desc(desc) != TKBN_OK) return -1;
  if (mode != TKBN_ADJ_ATOMIC && mode != TKBN_ADJ_DETERMINISTIC) return -1;
  const bool det = mode == TKBN_ADJ_DETERMINISTIC;
  int64_t n = adj_lane_bytes(desc, det);
  // Room for either path's plan, also where tuning fields ask for the sample-lane kernels: a
  // caller that tunes one problem keeps one buffer (it holds one plan at a time).
  tkbn_interp_desc plain = *desc;
  for (int i = 0; i < 3; ++i) plain.tile[i] = 0;
  plain.work_target = 0;
  if (!det && coil_variant_eligible(&plain)) {
    // (a tuning that lists more tiles or pieces shows in the size, whichever plan is larger)
    const int64_t untuned = adj_lane_bytes(&plain, det);
    n = std::max(untuned, sep_adj_bytes(desc)) + std::max<int64_t>(0, n - untuned);
  }
  if (reg3_eligible(desc)) {
    const int64_t nr = plan_cache_bytes(desc) + reg3_workspace_bytes(make_reg3_geom(desc, det));
    n = nr > n ? nr : n;
  }
  return n;
}

int tkbn_interp_adj(const tkbn_interp_desc* desc, const void* kdata, const void* omega, void* grid, int32_t mode,
                    void* workspace, int64_t workspace_bytes, void* stream) {
  int st = validate_desc(desc);
  if (st != TKBN_OK) return st;
  TKBN_REQUIRE(mode == TKBN_ADJ_ATOMIC || mode == TKBN_ADJ_DETERMINISTIC, TKBN_ERR_INVALID, "bad adjoint mode %d", mode);
  if (desc->batch == 0 || desc->coils == 0) return TKBN_OK;
  TKBN_REQUIRE(grid != nullptr, TKBN_ERR_INVALID, "NULL grid pointer");
  TKBN_REQUIRE(desc->klength == 0 || (kdata && omega), TKBN_ERR_INVALID, "NULL data pointer");
  TKBN_REQUIRE(desc->klength < (1LL << 31), TKBN_ERR_INVALID, "klength must be < 2^31");
  const bool det = mode == TKBN_ADJ_DETERMINISTIC;
  const int64_t need = tkbn_interp_adj_workspace_bytes(desc, mode);
  TKBN_REQUIRE(workspace != nullptr && workspace_bytes >= need, TKBN_ERR_WORKSPACE,
               "workspace of %lld bytes needed, %lld given", (long long)need, (long long)workspace_bytes);
  TKBN_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, TKBN_ERR_INVALID, "workspace must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (desc->dtype == TKBN_F32) return interp_adj_t<float>(desc, det, kdata, omega, grid, workspace, s);
  return interp_adj_t<double>(desc, det, kdata, omega, grid, workspace, s);
}

}  // extern "C"
