// kernels.hip -- gfx950 kernels of the density build and their launchers.
//
// Batched pipeline (one call):
//   count_kernel    particles -> (grid, tile) membership counts     [reads x,y,z,m]
//   scan_*          exclusive scan of the counts -> entry offsets
//   scatter_kernel  particles -> 16-byte entries grouped by tile    [reads x,y,z,m]
//   plan_items      tiles -> work items (chunks of <= chunk entries)
//   deposit_kernel  ONE persistent launch over the item queue: LDS tile
//                   accumulation, the tile and its one-cell halo to the
//                   exchange buffer
//   combine_tiles   a tile's cells plus its neighbours' halo sums: normalised
//                   coalesced stores, FP64-exact tile mass partials
//   grid_sums       fixed-order per-grid mass sums
// Plain form: one launch per grid with global FP32 atomics (plain_*).
#include <hip/hip_runtime.h>

#include "dev.h"
#include "launch.h"

namespace asohf {

// ---------------------------------------------------------------------------
// fills (used instead of hipMemsetAsync so every step can live in a graph)
// ---------------------------------------------------------------------------
__global__ void fill_u32_kernel(unsigned* p, unsigned v, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---------------------------------------------------------------------------
// count / scatter
// ---------------------------------------------------------------------------
// Block-local aggregation of (tile) keys.  A workgroup takes a contiguous
// run of particles (consecutive particles of one halo share tiles) and counts
// its emissions per key in an LDS open-addressing table; only one global
// atomic per distinct key leaves the workgroup.  A key whose probe path is
// full is never inserted later (the table only fills), so every emission of
// that key takes the direct global path consistently in all phases.
constexpr int kBinThreads = 256;
constexpr int kBinPer = 2;                       // particles per thread per block
constexpr int kBinChunk = kBinThreads * kBinPer;
constexpr int kBinCap = 1024;                    // LDS table slots (power of two)
constexpr int kBinProbe = 32;

// tile keys are < 2^24 (2 * tiles); 24-bit multiplies are full rate
__device__ __forceinline__ unsigned key_hash(unsigned k) {
  k ^= k >> 13;
  k = __umul24(k, 0x9E3779u) ^ (k >> 11);
  k ^= k >> 7;
  return k & (kBinCap - 1);
}
// slot of key k, inserting it when absent; -1 when its probe path is full.
// A plain read first: most emissions find their key already present, and a
// read costs less than a compare-and-swap.
__device__ __forceinline__ int lds_insert(int* keys, int k) {
  unsigned h = key_hash((unsigned)k);
#pragma unroll 1
  for (int p = 0; p < kBinProbe; ++p) {
    const int cur = keys[h];
    if (cur == k) return (int)h;
    if (cur == -1) {
      const int old = atomicCAS(&keys[h], -1, k);
      if (old == -1 || old == k) return (int)h;
    }
    h = (h + 1) & (kBinCap - 1);
  }
  return -1;
}
__device__ __forceinline__ int lds_find(const int* keys, int k) {
  unsigned h = key_hash((unsigned)k);
  for (int p = 0; p < kBinProbe; ++p) {
    const int v = keys[h];
    if (v == k) return (int)h;
    if (v == -1) return -1;
    h = (h + 1) & (kBinCap - 1);
  }
  return -1;
}

// one particle of lookahead: the next particle's loads are in flight while
// the current one is enumerated
struct Prefetch {
  float x, y, z, m;
  __device__ Prefetch(const Parts& A, long long i) : x(0.f), y(0.f), z(0.f), m(0.f) {
    if (i < A.n) { x = A.x[i]; y = A.y[i]; z = A.z[i]; m = A.m[i]; }
  }
  __device__ __forceinline__ void next(const Parts& A, long long inext, bool more, float& cx, float& cy,
                                       float& cz, float& cm) {
    cx = x; cy = y; cz = z; cm = m;
    if (more && inext < A.n) { x = A.x[inext]; y = A.y[inext]; z = A.z[inext]; m = A.m[inext]; }
  }
};

// emission lists: (key << 9) | particle index within the block
constexpr int kEmitCap = 4096;
static_assert(kBinChunk <= 512, "the emission list keeps 9 bits of particle index");

template <int MODE>
__global__ void __launch_bounds__(kBinThreads) count_kernel(Plan P, Parts A, unsigned* cnt, Counters* C,
                                                            BlockTables BT) {
  __shared__ int keys[kBinCap];
  __shared__ unsigned vals[kBinCap];
  __shared__ unsigned elist_s[kEmitCap];
  __shared__ int s_ne;
  for (int k = threadIdx.x; k < kBinCap; k += kBinThreads) { keys[k] = -1; vals[k] = 0u; }
  if (threadIdx.x == 0) s_ne = 0;
  __syncthreads();
  const bool list = BT.use_elist;
  unsigned err = 0;
  unsigned long long pairs = 0;
  float mmax = 0.f;
  const long long c0 = (long long)blockIdx.x * kBinChunk;
  Prefetch pf(A, c0 + threadIdx.x);
  for (int r = 0; r < kBinPer; ++r) {
    const long long i = c0 + (long long)r * kBinThreads + threadIdx.x;
    if (i >= A.n) break;
    float x, y, z, m;
    pf.next(A, i + kBinThreads, r + 1 < kBinPer, x, y, z, m);
    if (!(isfinite(x) && isfinite(y) && isfinite(z) && isfinite(m))) { err |= kErrNonFinite; continue; }
    if (m < 0.f) { err |= kErrNegMass; continue; }
    mmax = fmaxf(mmax, m);
    const int s = MODE == 1 ? species_of(A, i) : 0;
    enumerate_particle<MODE>(
        P, i, x, y, z, m, s,
        [&](int, int t, int wide, int4) {
          const int key = 2 * t + wide;
          const int h = lds_insert(keys, key);
          if (h >= 0) atomicAdd(&vals[h], 1u);
          else atomicAdd(&cnt[key], 1u);
          if (list) {
            const int pos = atomicAdd(&s_ne, 1);
            if (pos < kEmitCap) elist_s[pos] = ((unsigned)key << 9) | (unsigned)(i - c0);
          }
        },
        [&](int, int, int, int) { ++pairs; }, err);
  }
  __syncthreads();
  // the emission list, when it fits, for the scatter pass
  if (list) {
    __shared__ long long s_eoff;
    const int ne = s_ne;
    if (threadIdx.x == 0) {
      long long eo = -1;
      if (ne == 0) {
        eo = 0;
      } else if (ne <= kEmitCap) {
        const int sub = blockIdx.x & (kPoolSubs - 1);
        const long long subcap = BT.ecap / kPoolSubs;
        const long long off = (long long)atomicAdd(&C->epool_fill[sub * (kLine / 2)], (unsigned long long)ne);
        eo = off + ne <= subcap ? sub * subcap + off : -1;
      }
      s_eoff = eo;
      BT.eoff[blockIdx.x] = eo;
      BT.ecount[blockIdx.x] = ne;
    }
    __syncthreads();
    const long long eo = s_eoff;
    if (eo >= 0)
      for (int j = threadIdx.x; j < ne; j += kBinThreads) BT.elist[eo + j] = elist_s[j];
  }
  // flush the counts, and save the table (compacted) for the scatter pass
  __shared__ int s_n;
  __shared__ long long s_off;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  for (int k = threadIdx.x; k < kBinCap; k += kBinThreads)
    if (keys[k] >= 0) {
      atomicAdd(&cnt[keys[k]], vals[k]);
      atomicAdd(&s_n, 1);
    }
  __syncthreads();
  if (threadIdx.x == 0) {
    // sub-pool of this block: 1/kPoolSubs of the pool, its own counter line
    const int sub = blockIdx.x & (kPoolSubs - 1);
    const long long subcap = BT.cap / kPoolSubs;
    const long long off = (long long)atomicAdd(&C->pool_fill[sub * (kLine / 2)], (unsigned long long)s_n);
    s_off = off + s_n <= subcap ? sub * subcap + off : -1;
    BT.off[blockIdx.x] = s_off;
    BT.nkeys[blockIdx.x] = s_n;
    s_n = 0;
  }
  __syncthreads();
  if (s_off >= 0)
    for (int k = threadIdx.x; k < kBinCap; k += kBinThreads)
      if (keys[k] >= 0) BT.pool[s_off + atomicAdd(&s_n, 1)] = make_int2(keys[k], (int)vals[k]);
  // per-block partials (no contended global atomics); reduce_blocks folds them
  __shared__ unsigned long long s_pairs[kBinThreads / 64];
  __shared__ float s_mmax[kBinThreads / 64];
  pairs = wave_sum(pairs);
  mmax = wave_max(mmax);
  err = wave_or(err);
  if ((threadIdx.x & 63) == 0) {
    s_pairs[threadIdx.x >> 6] = pairs;
    s_mmax[threadIdx.x >> 6] = mmax;
    if (err) atomicOr(&C->err, err);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long p = 0;
    float mm = 0.f;
    for (int w = 0; w < kBinThreads / 64; ++w) { p += s_pairs[w]; mm = fmaxf(mm, s_mmax[w]); }
    BT.pairs[blockIdx.x] = p;
    BT.mmax[blockIdx.x] = __float_as_uint(mm);
  }
}

// The call's base members and largest mass from the per-block partials:
// every workgroup folds a grid-stride slice and adds its part to the
// counters (cleared at the start of the call); integer sums and the maximum
// do not depend on the order.  The mass maximum compares FP32 bit patterns,
// which order like the values for masses >= 0; the sign bit is cleared so a
// -0 mass counts as 0.
__global__ void __launch_bounds__(256) reduce_blocks(BlockTables BT, long long nblk, Counters* C) {
  __shared__ unsigned long long sp[4];
  __shared__ float sm[4];
  unsigned long long p = 0;
  float mm = 0.f;
  for (long long b = blockIdx.x * (long long)blockDim.x + threadIdx.x; b < nblk;
       b += (long long)gridDim.x * blockDim.x) {
    p += BT.pairs[b];
    mm = fmaxf(mm, __uint_as_float(BT.mmax[b]));
  }
  p = wave_sum(p);
  mm = wave_max(mm);
  if ((threadIdx.x & 63) == 0) { sp[threadIdx.x >> 6] = p; sm[threadIdx.x >> 6] = mm; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) { p = sp[0] + sp[w]; sp[0] = p; sm[0] = fmaxf(sm[0], sm[w]); }
    if (sp[0]) atomicAdd(&C->n_pairs, sp[0]);
    atomicMax(&C->mmax_bits, __float_as_uint(sm[0]) & 0x7fffffffu);
  }
}

template <int MODE>
__global__ void __launch_bounds__(kBinThreads) scatter_kernel(Plan P, Parts A, unsigned long long* cursor,
                                                              int4* entries, unsigned long long cap,
                                                              BlockTables BT, const Counters* C) {
  __shared__ int keys[kBinCap];
  __shared__ unsigned vals[kBinCap];
  __shared__ unsigned long long base[kBinCap];
  __shared__ int4 parts_s[kBinChunk];
  if (C->overflow) return;   // the entry buffer is too small: the host rebuilds exactly
  for (int k = threadIdx.x; k < kBinCap; k += kBinThreads) { keys[k] = -1; vals[k] = 0u; }
  __syncthreads();
  unsigned err = 0;
  const long long c0 = (long long)blockIdx.x * kBinChunk;
  const long long saved = BT.off[blockIdx.x];
  if (saved >= 0) {
    // the count pass's table of this block: reinsert its keys
    const int nk = BT.nkeys[blockIdx.x];
    for (int j = threadIdx.x; j < nk; j += kBinThreads) {
      const int2 kv = BT.pool[saved + j];
      const int h = lds_insert(keys, kv.x);
      if (h >= 0) vals[h] = (unsigned)kv.y;
    }
  } else {
    // phase A: count this block's emissions per key
    Prefetch pf(A, c0 + threadIdx.x);
    for (int r = 0; r < kBinPer; ++r) {
      const long long i = c0 + (long long)r * kBinThreads + threadIdx.x;
      if (i >= A.n) break;
      float x, y, z, m;
      pf.next(A, i + kBinThreads, r + 1 < kBinPer, x, y, z, m);
      if (!(isfinite(x) && isfinite(y) && isfinite(z) && isfinite(m)) || m < 0.f) continue;
      const int s = MODE == 1 ? species_of(A, i) : 0;
      enumerate_particle<MODE>(
          P, i, x, y, z, m, s,
          [&](int, int t, int wide, int4) {
            const int h = lds_insert(keys, 2 * t + wide);
            if (h >= 0) atomicAdd(&vals[h], 1u);
          },
          [&](int, int, int, int) {}, err);
    }
  }
  __syncthreads();
  // phase B: one global reservation per key
  for (int k = threadIdx.x; k < kBinCap; k += kBinThreads) {
    if (keys[k] >= 0) base[k] = atomicAdd(&cursor[keys[k]], (unsigned long long)vals[k]);
    vals[k] = 0u;
  }
  __syncthreads();
  // phase C, from the count pass's emission list: the block's particles staged
  // in LDS, each listed emission written to its reserved slot
  const long long eo = BT.use_elist ? BT.eoff[blockIdx.x] : -1;
  if (eo >= 0) {
    for (int j = threadIdx.x; j < kBinChunk; j += kBinThreads) {
      const long long i = c0 + j;
      if (i < A.n)
        parts_s[j] = make_int4(__float_as_int(A.x[i]), __float_as_int(A.y[i]), __float_as_int(A.z[i]),
                               __float_as_int(A.m[i]));
    }
    __syncthreads();
    const int ne = BT.ecount[blockIdx.x];
    for (int j = threadIdx.x; j < ne; j += kBinThreads) {
      const unsigned v = BT.elist[eo + j];
      const int key = (int)(v >> 9);
      const int h = lds_find(keys, key);
      const unsigned long long slot =
          h >= 0 ? base[h] + atomicAdd(&vals[h], 1u) : atomicAdd(&cursor[key], 1ull);
      const int li = (int)(v & 511u);
      int4 e = parts_s[li];
      if (MODE == 1) {
        // the table-mode entry: cell indices in the tile's grid
        const float x = __int_as_float(e.x), y = __int_as_float(e.y), z = __int_as_float(e.z),
                    m = __int_as_float(e.w);
        const int g = P.tile_grid[key >> 1];
        e = g == 0 ? table_base_entry(P, x, y, z, m)
                   : table_patch_entry(P.grids[g], x, y, z, m, species_of(A, c0 + li));
      }
      if (slot < cap) entries[slot] = e;
    }
    return;
  }
  // phase C: the same emissions again, written to their reserved slots
  Prefetch pc(A, c0 + threadIdx.x);
  for (int r = 0; r < kBinPer; ++r) {
    const long long i = c0 + (long long)r * kBinThreads + threadIdx.x;
    if (i >= A.n) break;
    float x, y, z, m;
    pc.next(A, i + kBinThreads, r + 1 < kBinPer, x, y, z, m);
    if (!(isfinite(x) && isfinite(y) && isfinite(z) && isfinite(m)) || m < 0.f) continue;
    const int s = MODE == 1 ? species_of(A, i) : 0;
    enumerate_particle<MODE>(
        P, i, x, y, z, m, s,
        [&](int, int t, int wide, int4 e) {
          const int key = 2 * t + wide;
          const int h = lds_find(keys, key);
          const unsigned long long slot =
              h >= 0 ? base[h] + atomicAdd(&vals[h], 1u) : atomicAdd(&cursor[key], 1ull);
          if (slot < cap) entries[slot] = e;   // the gate checked the buffer against the count pass
        },
        [&](int, int, int, int) {}, err);
  }
}

// membership records {grid, particle, ix, jy, kz}
template <int MODE>
__global__ void __launch_bounds__(256) membership_kernel(Plan P, Parts A, int* out, long long cap,
                                                         unsigned long long* count) {
  unsigned err = 0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < A.n;
       i += (long long)gridDim.x * blockDim.x) {
    const float x = A.x[i], y = A.y[i], z = A.z[i], m = A.m[i];
    if (!(isfinite(x) && isfinite(y) && isfinite(z))) continue;
    const int s = MODE == 1 ? species_of(A, i) : 0;
    enumerate_particle<MODE>(
        P, i, x, y, z, m, s, [&](int, int, int, int4) {},
        [&](int g, int ix, int jy, int kz) {
          const unsigned long long slot = atomicAdd(count, 1ull);
          if ((long long)slot < cap) {
            int* r = out + 5 * slot;
            r[0] = g; r[1] = (int)i; r[2] = ix; r[3] = jy; r[4] = kz;
          }
        },
        err);
  }
  // validation flags of the enumeration in count[1]
  err = wave_or(err);
  if ((threadIdx.x & 63) == 0 && err) atomicOr(count + 1, (unsigned long long)err);
}

// ---------------------------------------------------------------------------
// exclusive scan of u32 counts into u64 offsets (3 kernels)
// ---------------------------------------------------------------------------
constexpr int kScanThreads = 1024;
constexpr int kScanPer = 4;
constexpr int kScanTile = kScanThreads * kScanPer;

__device__ unsigned long long block_exclusive_scan(unsigned long long v, unsigned long long* sh,
                                                   unsigned long long* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  unsigned long long inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    unsigned long long t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) sh[w] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long run = 0;
    for (int k = 0; k < nw; ++k) { unsigned long long t = sh[k]; sh[k] = run; run += t; }
    sh[nw] = run;
  }
  __syncthreads();
  const unsigned long long r = sh[w] + inc - v;
  *total = sh[nw];
  __syncthreads();
  return r;
}

__global__ void __launch_bounds__(kScanThreads) scan_reduce(const unsigned* in, long long n,
                                                           unsigned long long* bsum) {
  __shared__ unsigned long long sh[kScanThreads / 64 + 1];
  const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanPer;
  unsigned long long s = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k)
    if (base + k < n) s += in[base + k];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) bsum[blockIdx.x] = s;
}

__global__ void __launch_bounds__(kScanThreads) scan_bsums(unsigned long long* bsum, int nb,
                                                          unsigned long long* total_out) {
  __shared__ unsigned long long sh[kScanThreads / 64 + 1];
  unsigned long long carry = 0;
  for (int b0 = 0; b0 < nb; b0 += kScanThreads) {
    const int b = b0 + threadIdx.x;
    const unsigned long long v = b < nb ? bsum[b] : 0ull;
    unsigned long long tot;
    const unsigned long long ex = block_exclusive_scan(v, sh, &tot);
    if (b < nb) bsum[b] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) *total_out = carry;
}

__global__ void __launch_bounds__(kScanThreads) scan_apply(const unsigned* in, long long n,
                                                          const unsigned long long* bsum,
                                                          unsigned long long* start,
                                                          unsigned long long* cursor) {
  __shared__ unsigned long long sh[kScanThreads / 64 + 1];
  const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanPer;
  unsigned v[kScanPer];
  unsigned long long s = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    v[k] = base + k < n ? in[base + k] : 0u;
    s += v[k];
  }
  unsigned long long tot;
  unsigned long long ex = block_exclusive_scan(s, sh, &tot) + bsum[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    if (base + k < n) {
      start[base + k] = ex;
      if (cursor) cursor[base + k] = ex;
    }
    ex += v[k];
  }
}

// ---------------------------------------------------------------------------
// work items
// ---------------------------------------------------------------------------
// Work items.  plan_count: items per tile, narrow ones in cnt[t], wide ones in
// cnt[ntiles + t]; after one exclusive scan over both halves, plan_write places
// every tile's items (no atomics): all narrow items in tile order, then all
// wide items.  With chunk_wide = 0 the tile's whole range
// [start[2t], start[2t+2]) is chunked as narrow entries (the TSC hierarchy
// binning, which uses the keys 2t only).
__device__ __forceinline__ void tile_chunks(const unsigned long long* start, int t, int chunk, int chunk_wide,
                                            long long& s0, long long& s1, long long& s2, int& cn, int& cw) {
  s0 = start[2 * t]; s1 = start[2 * t + 1]; s2 = start[2 * t + 2];
  if (chunk_wide == 0) {
    s1 = s2;
    cn = (int)((s2 - s0 + chunk - 1) / chunk);
    cw = 0;
    return;
  }
  cn = (int)((s1 - s0 + chunk - 1) / chunk);
  cw = (int)((s2 - s1 + chunk_wide - 1) / chunk_wide);
}

__global__ void plan_count(const unsigned long long* start, int ntiles, int chunk, int chunk_wide,
                           unsigned* cnt, unsigned* nitems_tile) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  long long s0, s1, s2;
  int cn, cw;
  tile_chunks(start, t, chunk, chunk_wide, s0, s1, s2, cn, cw);
  cnt[t] = (unsigned)cn;
  cnt[ntiles + t] = (unsigned)cw;
  nitems_tile[t] = (unsigned)(cn + cw);   // none for a tile without entries
}

__global__ void plan_write(const unsigned long long* start, int ntiles, int chunk, int chunk_wide,
                           const unsigned long long* item_off, Item* items, int* split_tiles, unsigned* n_split,
                           const Counters* C) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles || C->overflow) return;
  long long s0, s1, s2;
  int cn, cw;
  tile_chunks(start, t, chunk, chunk_wide, s0, s1, s2, cn, cw);
  if (split_tiles && cn + cw > 1) split_tiles[atomicAdd(n_split, 1u)] = t;   // in any order
  long long k = (long long)item_off[t];
  for (int c = 0; c < cn; ++c, ++k) {
    const long long b = s0 + (long long)c * chunk;
    items[k] = Item{t, 0, b, min(b + (long long)chunk, s1)};
  }
  // bit 1: the item holds every wide entry of its tile (the histogram form
  // is used only then, so its one rounding per cell does not depend on how
  // the entries fall into items)
  k = (long long)item_off[ntiles + t];
  for (int c = 0; c < cw; ++c, ++k) {
    const long long b = s1 + (long long)c * chunk_wide;
    items[k] = Item{t, 1 | (cw == 1 ? 2 : 0), b, min(b + (long long)chunk_wide, s2)};
  }
}

// The narrow items once more, long ones first (by half powers of two of their
// length, in any order within one): a workgroup that takes a long item last
// keeps the deposit waiting for it.  The classes' counts and then their fill
// lie in the emission's queue words, which are 0 here.  Atomic TSC deposit of
// 2.1M particles, whose CUs worked 496 us of it on average: 789 -> 623 us; the
// shorter items of deterministic sums gain 1 to 4 percent.
constexpr int kItemClasses = 64;
__device__ __forceinline__ int item_class(const Item& it) {   // 0: longest
  const unsigned long long len = (unsigned long long)max(it.end - it.begin, 1ll);
  const int e = 63 - __clzll((long long)len);
  const int c = 2 * e + (e > 0 ? (int)((len >> (e - 1)) & 1ull) : 0);
  return kItemClasses - 1 - min(c, kItemClasses - 1);
}
__global__ void __launch_bounds__(256) order_items(const Item* items, Item* work, long long n_given, Counters* C,
                                                   int pass) {
  __shared__ unsigned cnt[kItemClasses], base[kItemClasses];
  unsigned* const total = C->equeue;
  unsigned* const fill = C->equeue + kItemClasses;
  const unsigned n = n_given >= 0 ? (unsigned)n_given : C->n_items_eff;   // narrow items
  // a contiguous part of the items per workgroup
  const unsigned per = (n + gridDim.x - 1) / gridDim.x;
  const unsigned i0 = min(blockIdx.x * per, n), i1 = min(i0 + per, n);
  if (threadIdx.x < kItemClasses) cnt[threadIdx.x] = 0u;
  __syncthreads();
  for (unsigned i = i0 + threadIdx.x; i < i1; i += blockDim.x) atomicAdd(&cnt[item_class(items[i])], 1u);
  __syncthreads();
  if (threadIdx.x < kItemClasses) {
    const unsigned c = cnt[threadIdx.x];
    if (pass == 0) {
      if (c) atomicAdd(&total[threadIdx.x], c);
    } else {
      unsigned b = 0;
      for (int k = 0; k < (int)threadIdx.x; ++k) b += total[k];
      base[threadIdx.x] = b + (c ? atomicAdd(&fill[threadIdx.x], c) : 0u);
    }
  }
  if (pass == 0) return;
  __syncthreads();
  for (unsigned i = i0 + threadIdx.x; i < i1; i += blockDim.x) {
    const Item it = items[i];
    const unsigned at = atomicAdd(&base[item_class(it)], 1u);
    if (at < n) work[at] = it;
  }
}

// The totals of the planning scans against the workspaces of this call.  A
// call whose buffers were sized by an earlier call finds out here, on the
// device, whether they still suffice; if not, every later kernel of the call
// does nothing and the host rebuilds with exact sizes.
__global__ void gate_kernel(const unsigned long long* tot_entries, const unsigned long long* item_off, int ntiles,
                            unsigned long long cap_entries, unsigned long long cap_items, Counters* C) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  const unsigned long long ne = *tot_entries, nn = item_off[ntiles], ni = item_off[2 * ntiles];
  C->n_entries = ne;
  C->n_items = ni;
  const bool over = ne > cap_entries || ni > cap_items || ni >= (1ull << 31);
  C->overflow = over ? 1u : 0u;
  C->n_items_eff = over ? 0u : (unsigned)nn;
  C->n_wide_eff = over ? 0u : (unsigned)(ni - nn);
}

// Fixed-point scale of the deterministic reduction: the power of two with
// max(m) * scale in [2^29, 2^30), so every quantised term is below 2^30,
// eight non-centre terms (each below half of it) sum below 2^32, and a sum
// over <= 2^32 particles fits an int64.  The unit is at most max(m) * 2^-29.
__device__ __forceinline__ double fixed_scale(unsigned mmax_bits) {
  const float mm = __uint_as_float(mmax_bits);
  int e = 0;
  if (mm > 0.f) (void)frexpf(mm, &e);
  return ldexp(1.0, 30 - e);
}

// ---------------------------------------------------------------------------
// the persistent deposit
// ---------------------------------------------------------------------------
template <int RED> struct AccT;
template <> struct AccT<0> { using T = long long; };
template <> struct AccT<1> { using T = float; };

__device__ __forceinline__ void lds_add(long long* a, long long v) {
  atomicAdd(reinterpret_cast<unsigned long long*>(a), (unsigned long long)v);
}
__device__ __forceinline__ void lds_add(float* a, float v) { atomicAdd(a, v); }
__device__ __forceinline__ void glb_add(long long* a, long long v) {
  atomicAdd(reinterpret_cast<unsigned long long*>(a), (unsigned long long)v);
}
__device__ __forceinline__ void glb_add(float* a, float v) { atomicAdd(a, v); }
__device__ __forceinline__ long long glb_load(long long* a) {
  return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float glb_load(float* a) {
  return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A deterministic term: ((m*scale*wx)*wy)*wz rounded to the nearest integer
// (halves up) as one fused multiply-add of 1/2 and a truncating conversion.
// The terms are >= 0 and below 2^30; a term of 2^23 or more comes out within
// one unit of the exact product's rounding.  Every term is a function of its
// particle alone, so the sums stay independent of the order of the adds.
__device__ __forceinline__ unsigned term_u32(float mxy, float wz) {
  return (unsigned)__fmaf_rn(mxy, wz, 0.5f);
}

// 27-cell deposit of one particle into the LDS tile, which carries a 2-cell
// halo on every side: the particle's centre cell lies within one cell of the
// tile (it was binned to the tile because one of its 27 cells is inside), so
// all 27 cells are in the array and the deposit needs no per-cell test, one
// base address and 27 constant offsets.  The terms are the reference's FP32
// products ((m*wx)*wy)*wz.  Deterministic mode scales the mass by the
// power-of-two fixed-point scale first (exact), rounds every term to an
// integer and gives the centre cell the remainder Q(m) - (sum of the other
// 26), so each particle deposits exactly Q(m) over its stencil.
template <int RED, int HX, int HY>
__device__ __forceinline__ void deposit27(typename AccT<RED>::T* base, float m, const float wx[3],
                                          const float wy[3], const float wz[3], float scale) {
  const float ms = RED == 0 ? m * scale : m;
  float mx[3], mxy[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a) mx[a] = ms * wx[a];
#pragma unroll
  for (int b = 0; b < 3; ++b)
#pragma unroll
    for (int a = 0; a < 3; ++a) mxy[b][a] = mx[a] * wy[b];
  if (RED == 1) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int a = 0; a < 3; ++a)
          lds_add(reinterpret_cast<float*>(base) + (a + HX * (b + HY * c)), mxy[b][a] * wz[c]);
  } else {
    // every term is >= 0 (masses >= 0, TSC and kernel weights >= 0) and
    // below 2^30, so it converts to an unsigned word whose 64-bit form needs
    // no sign extension
    unsigned rest = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          if (a == 1 && b == 1 && c == 1) continue;
          const unsigned q = term_u32(mxy[b][a], wz[c]);
          rest += q;
          lds_add(reinterpret_cast<long long*>(base) + (a + HX * (b + HY * c)), (long long)(unsigned long long)q);
        }
    lds_add(reinterpret_cast<long long*>(base) + (1 + HX * (1 + HY * 1)),
            (long long)__float2uint_rn(ms) - (long long)rest);
  }
}

// a wave-uniform 64-bit value, moved to scalar registers
__device__ __forceinline__ long long uniform64(long long v) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)((unsigned long long)v >> 32));
  return (long long)(((unsigned long long)hi << 32) | lo);
}

// the value of lane l^1 (l^2) of the wave, through a quad permutation
__device__ __forceinline__ unsigned from_xor1(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
}
__device__ __forceinline__ unsigned from_xor2(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
}
// the value of lane l+4 (l-4) of the same row of 16 lanes; a lane whose
// source lies outside its row gets 0 (the DPP default)
__device__ __forceinline__ unsigned from_plus4(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x104, 0xF, 0xF, false);   // row_shl:4
}
__device__ __forceinline__ unsigned from_minus4(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);   // row_shr:4
}
__device__ __forceinline__ long long from_plus4(long long v) {
  const unsigned lo = from_plus4((unsigned)v), hi = from_plus4((unsigned)((unsigned long long)v >> 32));
  return (long long)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ float from_xor1(float v) { return __uint_as_float(from_xor1(__float_as_uint(v))); }
__device__ __forceinline__ float from_xor2(float v) { return __uint_as_float(from_xor2(__float_as_uint(v))); }
__device__ __forceinline__ float from_plus4(float v) { return __uint_as_float(from_plus4(__float_as_uint(v))); }
__device__ __forceinline__ long long from_xor1(long long v) {
  const unsigned lo = from_xor1((unsigned)v), hi = from_xor1((unsigned)((unsigned long long)v >> 32));
  return (long long)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ long long from_xor2(long long v) {
  const unsigned lo = from_xor2((unsigned)v), hi = from_xor2((unsigned)((unsigned long long)v >> 32));
  return (long long)(((unsigned long long)hi << 32) | lo);
}

// Lanes of a merge step needed before it pays (each merged pair saves one
// lane's 27 LDS adds and costs every lane two instructions per term).
constexpr int kMergeMin = 4;

// The 27-cell deposit (TSC, or a table-mode narrow entry) with lanes merged
// first.  Clustered particles put many lanes of a wave on the same stencil,
// and the LDS serialises adds to one address; the terms can be summed in
// registers instead.  Deterministic mode: the terms are exact integers, so
// the result is the same.  Atomic mode: an FP32 sum in another order, as any
// order of its LDS atomics is.
// Three butterfly steps: lane l takes lane l^1's terms when both stencils
// start at the same cell (l even), then lane l^2's (bit 1 of l clear), then
// lane l^4's (bit 2 clear).  Every non-centre TSC term is below half of
// Q(m) < 2^30 (one factor is an outer weight: at most 0.5 * 0.75 * 0.75 with
// exact centres, below 0.48 with the centre rounding the plan admits;
// table mode merges only when the plan found every non-centre product of its
// row-0 weights at most 0.45), so eight of them sum below 2^32 and all three
// steps add in 32 bits; the centre remainder, negative for a light enough
// particle, merges as int64.
// Every lane of the wave must be active (the steps read other lanes); ok =
// the lane holds an entry, corner = its stencil's first cell in the tile.
template <int RED, int HX, int HY>
__device__ __forceinline__ void deposit27_merged(typename AccT<RED>::T* acc, int corner, bool ok, float m,
                                                 const float wx[3], const float wy[3], const float wz[3],
                                                 float scale) {
  const unsigned lane = __lane_id();
  // lanes without an entry get keys that match no other lane
  const unsigned key0 = ok ? (unsigned)corner : (0x80000000u | lane);
  const bool m1 = from_xor1(key0) == key0;
  if (__popcll(__ballot(m1)) < kMergeMin) {
    if (ok) deposit27<RED, HX, HY>(acc + corner, m, wx, wy, wz, scale);
    return;
  }
  // a lane absorbed by a step sends its value and every lane adds what it
  // receives: keepers receive their partner's, everyone else receives 0
  const bool send1 = m1 && (lane & 1u);
  const bool alive1 = ok && !send1;
  const unsigned key1 = alive1 ? (unsigned)corner : (0x80000000u | lane);
  const bool m2 = from_xor2(key1) == key1;
  const bool step2 = __popcll(__ballot(m2)) >= kMergeMin;
  const bool send2 = step2 && m2 && (lane & 2u);
  const bool alive2 = alive1 && !send2;
  // lane l^4 stays in the row of 16 lanes, so one row shift reaches it.  Both
  // shifts run on every lane and the lane picks its value afterwards: under a
  // branch, half the lanes would be inactive and their values unreadable.
  const unsigned key2 = alive2 ? (unsigned)corner : (0x80000000u | lane);
  const unsigned k_minus = from_minus4(key2), k_plus = from_plus4(key2);
  const unsigned pk = (lane & 4u) ? k_minus : k_plus;
  const bool m3 = pk == key2;
  const bool step3 = __popcll(__ballot(m3)) >= kMergeMin;
  const bool send3 = step3 && m3 && (lane & 4u);
  const bool alive = alive2 && !send3;

  const float ms = RED == 0 ? m * scale : m;
  float mx[3], mxy[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a) mx[a] = ms * wx[a];
#pragma unroll
  for (int b = 0; b < 3; ++b)
#pragma unroll
    for (int a = 0; a < 3; ++a) mxy[b][a] = mx[a] * wy[b];
  if (RED == 1) {
    float* fbase = reinterpret_cast<float*>(acc) + corner;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          float t = mxy[b][a] * wz[c];
          t += from_xor1(send1 ? t : 0.f);
          if (step2) t += from_xor2(send2 ? t : 0.f);
          if (step3) t += from_plus4(send3 ? t : 0.f);
          if (alive) lds_add(fbase + (a + HX * (b + HY * c)), t);
        }
    return;
  }
  long long* base = reinterpret_cast<long long*>(acc) + corner;
  unsigned rest = 0;
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        if (a == 1 && b == 1 && c == 1) continue;
        unsigned q = term_u32(mxy[b][a], wz[c]);
        rest += q;
        q += from_xor1(send1 ? q : 0u);
        if (step2) q += from_xor2(send2 ? q : 0u);
        if (step3) q += from_plus4(send3 ? q : 0u);
        if (alive) lds_add(base + (a + HX * (b + HY * c)), (long long)(unsigned long long)q);
      }
  long long cen = (long long)__float2uint_rn(ms) - (long long)rest;
  cen += from_xor1(send1 ? cen : 0ll);
  if (step2) cen += from_xor2(send2 ? cen : 0ll);
  if (step3) cen += from_plus4(send3 ? cen : 0ll);
  if (alive) lds_add(base + (1 + HX * (1 + HY * 1)), cen);
}

// base-grid cell centre RAD(i), i = 0..n+1: MALLA's own FP32 recurrence
// (RAD(i) = RAD(1)+(i-1)*C, ghost RAD(n+1) = RAD(n)+C) when the plan found the
// table to be exactly that, a table read otherwise
__device__ __forceinline__ float base_centre(const Plan& P, int a, int i, int n) {
  if (P.rad_malla) {
    if (i <= n) return P.rad1[a] + (float)(i - 1) * P.radc[a];
    return (P.rad1[a] + (float)(n - 1) * P.radc[a]) + P.radc[a];
  }
  const float* r = a == 0 ? P.radx : (a == 1 ? P.rady : P.radz);
  return r[i];
}

// tile-local coordinate of the centre cell of an entry in one of several tiles
// its stencil touches: on the periodic base grid the image of the (wrapped)
// centre that lies next to the tile
__device__ __forceinline__ int centre_local(int c, int org, int ext, int n, bool periodic) {
  if (!periodic) return c - org;
  int l = wrap1(c, n) - org;
  if (l > ext) l -= n;
  if (l < -1) l += n;
  return l;
}

// LDS layout of a deposit tile: cell (x, y, z), local coordinates from -1 (the
// tile's halo) to T, at kTileFront + (x + 1) + HX * ((y + 1) + HY * (z + 2)).
// Every entry's centre cell, clamped into its grid, lies in the tile, so a
// stencil reaches at most one cell past the tile, or two where the centre
// itself lies one cell outside a patch; that second cell is outside the patch
// and never read.  It falls into the pad column, the pad row or the outer
// planes (and, below row 0 of the first plane, into the front pad), so the
// deposit needs no per-cell test.
template <int TX, int TY, int TZ>
struct TileLds {
  static constexpr int HX = TX + 3, HY = TY + 3, HZ = TZ + 4;
  static constexpr int kFront = HX + 1;
  static constexpr int H = kFront + HX * HY * HZ;
  // the tile with its one-cell halo, as written to the exchange buffer.  The
  // odd row pitch spreads a stencil's adds over the LDS banks.
  static constexpr int EX = TX + 2, EY = TY + 2, EZ = TZ + 2, E = EX * EY * EZ;
  __device__ __forceinline__ static int at(int x, int y, int z) {
    return kFront + (x + 1) + HX * ((y + 1) + HY * (z + 2));
  }
  // exchange cell c (x fastest) in the LDS tile
  __device__ __forceinline__ static int of_exchange(int c) {
    return kFront + c % EX + HX * ((c / EX) % EY + HY * (c / (EX * EY) + 1));
  }
};

// Whether tile t received entries in this call (its exchange cells are then
// written): the binning through the base grid fills capacity ranges up to the
// cursors, the count pass fills [start[2t], start[2t+2]) exactly.
__device__ __forceinline__ bool tile_filled(const DepArgs& D, int t) {
  if (!D.cursor) return D.start[2 * t + 2] > D.start[2 * t];
  return D.cursor[2 * t] > D.start[2 * t] || D.cursor[2 * t + 1] > D.start[2 * t + 1];
}

template <int MODE, int RED, int TX, int TY, int TZ>
__global__ void __launch_bounds__(1024) deposit_kernel(Plan P, DepArgs D) {
  using Acc = typename AccT<RED>::T;
  using L = TileLds<TX, TY, TZ>;
  constexpr int HX = L::HX, HY = L::HY, H = L::H;
  __shared__ Acc acc[H];
  __shared__ unsigned s_item;
  const int tid = threadIdx.x, nthr = blockDim.x;
  stamp(D.C, kClkDeposit);
  const float scale = (float)fixed_scale(D.C->mmax_bits);
  const unsigned n_items = D.C->n_items_eff;
  const float k0[3] = {P.ktab[P.kmax - 1], P.ktab[P.kmax], P.ktab[P.kmax + 1]};
  auto at = [](int a, int b, int c) { return L::at(a, b, c); };

  // workgroup w serves queue w mod n_queues, which hands out items
  // q, q + n_queues, ...; consecutive workgroups land on different XCDs, so
  // each queue counter lives in one XCD's L2
  const int q = blockIdx.x % D.n_queues;
  for (;;) {
    if (tid == 0) s_item = atomicAdd(&D.C->queue[q * kLine], 1u) * D.n_queues + q;
    __syncthreads();
    const unsigned idx = __builtin_amdgcn_readfirstlane(s_item);
    if (idx >= n_items) break;
    const Item it = D.work[idx];
    const int t = __builtin_amdgcn_readfirstlane(it.tile);
    const int g = __builtin_amdgcn_readfirstlane(P.tile_grid[t]);
    const GridDesc G = P.grids[g];
    const int local = t - G.tile0;
    const int tx = local % G.nt[0], ty = (local / G.nt[0]) % G.nt[1], tz = local / (G.nt[0] * G.nt[1]);
    const int i0 = tx * TX + 1, j0 = ty * TY + 1, k0c = tz * TZ + 1;
    const bool periodic = g == 0;
    // two tiles on a periodic axis, the last one cell wide
    const bool images = periodic && ((G.nt[0] == 2 && G.n[0] == TX + 1) || (G.nt[1] == 2 && G.n[1] == TY + 1) ||
                                     (G.nt[2] == 2 && G.n[2] == TZ + 1));

    // the item's filled entries
    long long len = it.end - it.begin;
    if (D.cursor) len = min(it.end, (long long)D.cursor[2 * t]) - it.begin;
    len = uniform64(len);   // wave-uniform: kept in scalar registers
    if (len <= 0) {
      __syncthreads();   // every wave has read s_item before thread 0 takes the next item
      continue;
    }
    for (int c = tid; c < H; c += nthr) acc[c] = 0;
    __syncthreads();

    // ---- narrow entries: one lane per entry, 27 cells.  Lane j of the
    // workgroup takes entries j, j + nthr, ... of the item, so a wave reads
    // 64 consecutive entries (1 KB, every entry fetched once).  Two entries
    // per pass, in two registers refilled right after use (register copies
    // would wait on the loads); the prefetch indices are clamped into the
    // item instead of tested, so every pass issues the same loads, and the
    // loop runs the same number of passes on every lane (ok = the lane holds
    // an entry), which the lane merging of the TSC deposit needs.
    const int4* const eb = D.entries + uniform64(it.begin);
    auto narrow = [&](const int4 v, const bool ok) {
      int ci[3];
      float wx[3], wy[3], wz[3], m;
      if (MODE == 2) {
        const float p[3] = {__int_as_float(v.x), __int_as_float(v.y), __int_as_float(v.z)};
        m = __int_as_float(v.w);
        float* w[3] = {wx, wy, wz};
        // weights from the three centres RAD(I-1..I+1) on the base grid,
        // MINIRADX(I-1..I+1) on a patch; the indices are the reference's
        if (g == 0) {
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            ci[a] = tsc_base_index(p[a], P.xl, G.d[a], G.inv_d[a], G.n[a]);
            tsc_weights_f64(p[a], base_centre(P, a, ci[a] - 1, G.n[a]), base_centre(P, a, ci[a], G.n[a]),
                            base_centre(P, a, ci[a] + 1, G.n[a]), G.inv_dd[a], w[a]);
          }
        } else {
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            ci[a] = (int)index_quotient(p[a] - G.org[a], G.d[a], G.inv_d[a]);
            tsc_weights_f64(p[a], minirad(G.pr[a], ci[a] - 1, G.d[a]), minirad(G.pr[a], ci[a], G.d[a]),
                            minirad(G.pr[a], ci[a] + 1, G.d[a]), G.inv_dd[a], w[a]);
          }
        }
      } else {
        int irk;
        unpack_table(v, ci[0], ci[1], ci[2], irk, m);
#pragma unroll
        for (int k = 0; k < 3; ++k) { wx[k] = k0[k]; wy[k] = k0[k]; wz[k] = k0[k]; }
      }
      // in [-1, ext] by construction of the binning; clamped so the array
      // bounds never depend on that
      const int ext[3] = {min(TX, G.n[0] - i0 + 1), min(TY, G.n[1] - j0 + 1), min(TZ, G.n[2] - k0c + 1)};
      const int org[3] = {i0, j0, k0c};
      int lc[3];
#pragma unroll
      for (int a = 0; a < 3; ++a)
        lc[a] = MODE == 1 && RED == 1 ? centre_local(ci[a], org[a], ext[a], G.n[a], periodic)
                                      : (periodic ? wrap1(ci[a], G.n[a]) : ci[a]) - org[a];
      if (MODE == 1 && RED == 1 && images && ok) {
        // a centre next to the wrap reaches the first tile on both sides,
        // through two images
        for (int k = 1; k < 8; ++k) {
          int li[3];
          bool img = true;
          for (int a = 0; a < 3; ++a) {
            li[a] = lc[a];
            if (!((k >> a) & 1)) continue;
            const bool below = lc[a] - G.n[a] >= -1;
            li[a] += below ? -G.n[a] : G.n[a];
            img = img && G.nt[a] > 1 && (below || li[a] <= ext[a]);
          }
          if (img) deposit27<RED, HX, HY>(acc + at(li[0] - 1, li[1] - 1, li[2] - 1), m, wx, wy, wz, scale);
        }
      }
      const int lx = clampi(lc[0], -1, TX), ly = clampi(lc[1], -1, TY), lz = clampi(lc[2], -1, TZ);
      const int corner = at(lx - 1, ly - 1, lz - 1);
      if (MODE == 2 || P.merge_narrow)
        deposit27_merged<RED, HX, HY>(acc, corner, ok, m, wx, wy, wz, scale);
      else if (ok)
        deposit27<RED, HX, HY>(acc + corner, m, wx, wy, wz, scale);
    };
    // entry j of the item (j clamped to the last one)
    auto at_j = [&](long long j) { return eb[min(j, len - 1)]; };
    int4 va = at_j(tid), vb = at_j(tid + nthr);
    for (long long o = 0; o < len; o += 2 * nthr) {
      narrow(va, o + tid < len);
      va = at_j(o + 2 * nthr + tid);
      narrow(vb, o + nthr + tid < len);
      vb = at_j(o + 3 * nthr + tid);
    }
    __syncthreads();

    // ---- entries in every tile they touch (P.per_tile): the halo is the other
    // tiles' business, once a tile spanning a whole periodic axis has folded it
    // into its own cells (the reference's wrap) ----
    const int ex = min(TX, G.n[0] - i0 + 1), ey = min(TY, G.n[1] - j0 + 1), ez = min(TZ, G.n[2] - k0c + 1);
    auto inside = [&](int c) {
      const int a = c % L::EX - 1, b = (c / L::EX) % L::EY - 1, cz = c / (L::EX * L::EY) - 1;
      return a >= 0 && a < ex && b >= 0 && b < ey && cz >= 0 && cz < ez;
    };
    if (MODE == 1 && RED == 1 && periodic && (G.nt[0] == 1 || G.nt[1] == 1 || G.nt[2] == 1)) {
      for (int c = tid; c < L::E; c += nthr) {
        if (inside(c)) continue;
        const int a = c % L::EX - 1, b = (c / L::EX) % L::EY - 1, cz = c / (L::EX * L::EY) - 1;
        const int ga = wrap1(i0 + a, G.n[0]) - i0, gb = wrap1(j0 + b, G.n[1]) - j0, gc = wrap1(k0c + cz, G.n[2]) - k0c;
        if (ga >= 0 && ga < ex && gb >= 0 && gb < ey && gc >= 0 && gc < ez && acc[at(a, b, cz)] != 0)
          lds_add(acc + at(ga, gb, gc), acc[at(a, b, cz)]);
      }
      __syncthreads();
    }

    // ---- the tile and its halo to the exchange buffer: stored when the tile
    // has one item, added where several items share it (exact int64 adds, so
    // the sum does not depend on their order; the cells were cleared) ----
    Acc* dst = reinterpret_cast<Acc*>(D.scratch) + (long long)t * L::E;
    auto cell = [&](int c) -> Acc { return MODE == 1 && RED == 1 && !inside(c) ? (Acc)0 : acc[L::of_exchange(c)]; };
    if (D.nitems_tile[t] == 1) {
      for (int c = tid; c < L::E; c += nthr) dst[c] = cell(c);
    } else {
      for (int c = tid; c < L::E; c += nthr) {
        const Acc v = cell(c);
        if (v != 0) glb_add(dst + c, v);
      }
    }
    __syncthreads();
  }
}

// Deterministic table mode's narrow entries (N = 1).  Every entry's 27 terms
// are the kernel row's weights times its mass, rounded to the fixed-point unit,
// and most snapshots hold one mass: the entries of the item's first mass are
// counted at their centre cells, one LDS add per entry instead of 27, and the
// cells' sums are counts times the 8 distinct terms (per axis an outer or the
// centre weight; the centre keeps Q(m) minus the other 26).  Entries of another
// mass deposit their 27 terms one by one.  Both are the sums of the same
// integers, so the result depends on neither the item's first entry nor how
// entries fall into items.
// Bound by reading the entries and the 27 counts per cell.  Against 27 LDS adds
// per entry with neighbouring lanes merged: 16.8M particles, 4 levels 762 ->
// 371 us; 134M particles, 6 levels 6.2 -> 1.9 ms; 2.1M, 3 levels 111 -> 45 us.
template <int TX, int TY, int TZ>
__global__ void __launch_bounds__(1024) deposit_counts(Plan P, DepArgs D) {
  using L = TileLds<TX, TY, TZ>;
  // counts at local cells -1..T of the tile, with a ring of zeros around them
  constexpr int CX = TX + 4, CY = TY + 4, CZ = TZ + 4;
  __shared__ long long acc[L::H];
  __shared__ unsigned cnt[CX * CY * CZ];
  __shared__ unsigned s_item;
  const int tid = threadIdx.x, nthr = blockDim.x;
  stamp(D.C, kClkDeposit);
  const float scale = (float)fixed_scale(D.C->mmax_bits);
  const unsigned n_items = D.C->n_items_eff;
  const float k0[3] = {P.ktab[P.kmax - 1], P.ktab[P.kmax], P.ktab[P.kmax + 1]};
  const int q = blockIdx.x % D.n_queues;
  for (;;) {
    if (tid == 0) s_item = atomicAdd(&D.C->queue[q * kLine], 1u) * D.n_queues + q;
    __syncthreads();
    const unsigned idx = __builtin_amdgcn_readfirstlane(s_item);
    if (idx >= n_items) break;
    const Item it = D.work[idx];
    const int t = __builtin_amdgcn_readfirstlane(it.tile);
    const int g = __builtin_amdgcn_readfirstlane(P.tile_grid[t]);
    const GridDesc& G = P.grids[g];
    const int n[3] = {G.n[0], G.n[1], G.n[2]}, nt0 = G.nt[0], nt1 = G.nt[1];
    const int local = t - G.tile0;
    const int org[3] = {(local % nt0) * TX + 1, ((local / nt0) % nt1) * TY + 1, (local / (nt0 * nt1)) * TZ + 1};
    long long len = it.end - it.begin;
    if (D.cursor) len = min(it.end, (long long)D.cursor[2 * t]) - it.begin;
    len = uniform64(len);
    if (len <= 0) {
      __syncthreads();   // every wave has read s_item before thread 0 takes the next item
      continue;
    }
    const int4* const eb = D.entries + uniform64(it.begin);
    const bool positions = D.cursor && g == 0;
    const int m_bits = __builtin_amdgcn_readfirstlane(positions ? eb[0].w : eb[0].z);   // the item's first mass
    for (int c = tid; c < L::H; c += nthr) acc[c] = 0;
    for (int c = tid; c < CX * CY * CZ; c += nthr) cnt[c] = 0u;
    __syncthreads();
    bool others = false;   // the wave met another mass
    for (long long o = 0; o < len; o += 4 * nthr) {   // four loads in flight
      int4 v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = eb[min(o + r * nthr + tid, len - 1)];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = o + r * nthr + tid < len;
        int ci[3], irk;
        float m;
        const int4 e = positions ? table_base_entry(P, __int_as_float(v[r].x), __int_as_float(v[r].y),
                                                    __int_as_float(v[r].z), __int_as_float(v[r].w))
                                 : v[r];
        unpack_table(e, ci[0], ci[1], ci[2], irk, m);
        int lc[3];
        constexpr int T[3] = {TX, TY, TZ};
#pragma unroll
        for (int a = 0; a < 3; ++a) lc[a] = clampi((g == 0 ? wrap1(ci[a], n[a]) : ci[a]) - org[a], -1, T[a]);
        const bool same = __float_as_int(m) == m_bits;
        if (ok && same) {
          atomicAdd(&cnt[(lc[0] + 2) + CX * ((lc[1] + 2) + CY * (lc[2] + 2))], 1u);
        } else if (ok) {
          others = true;
          deposit27<0, L::HX, L::HY>(acc + L::at(lc[0] - 1, lc[1] - 1, lc[2] - 1), m, k0, k0, k0, scale);
        }
      }
    }
    const bool any_other = __syncthreads_or(others);
    // the terms of the first mass, as deposit27 forms them: index bit a set
    // where the cell is the centre's neighbour along axis a
    unsigned term[8];
    {
      const float ms = __int_as_float(m_bits) * scale;
      unsigned rest = 0;
#pragma unroll
      for (int k = 1; k < 8; ++k) {
        term[k] = term_u32((ms * k0[k & 1 ? 0 : 1]) * k0[k & 2 ? 0 : 1], k0[k & 4 ? 0 : 1]);
        rest += term[k] << __popc(k);   // 2, 4 or 8 cells
      }
      term[0] = rest;   // what the centre gives away
    }
    const unsigned whole = __float2uint_rn(__int_as_float(m_bits) * scale);
    const long long centre = (long long)whole - (long long)term[0];
    long long* dst = reinterpret_cast<long long*>(D.scratch) + (long long)t * L::E;
    const bool alone = D.nitems_tile[t] == 1;
    for (int c = tid; c < L::E; c += nthr) {
      // counts around exchange cell c, from the corner (-1, -1, -1)
      const unsigned* N = cnt + c % L::EX + CX * ((c / L::EX) % L::EY + CY * (c / (L::EX * L::EY)));
      unsigned sum[8] = {};
#pragma unroll
      for (int z = 0; z < 3; ++z)
#pragma unroll
        for (int y = 0; y < 3; ++y)
#pragma unroll
          for (int x = 0; x < 3; ++x)
            sum[(x != 1 ? 1 : 0) + (y != 1 ? 2 : 0) + (z != 1 ? 4 : 0)] += N[x + CX * (y + CY * z)];
      long long v = any_other ? acc[L::of_exchange(c)] : 0ll;
      v += (long long)sum[0] * centre;
#pragma unroll
      for (int k = 1; k < 8; ++k) v += (long long)((unsigned long long)sum[k] * term[k]);
      if (alone) dst[c] = v;
      else if (v != 0) glb_add(dst + c, v);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// wide table-mode entries (kernel level irk >= 1, half-width N = 2^irk)
// ---------------------------------------------------------------------------
constexpr int kWideThreads = 512;
constexpr int kWideCells = 8192;   // histogram cells (64 KB: two workgroups per CU)
constexpr int kWideK = 2 * 64 + 1;  // longest kernel row of a histogram form (form 2 fits up to N = 32)

// How a class's histogram is laid out for a block of BX x BY x BZ cells.  The
// field of the class is the masses summed at their cells, convolved with the
// kernel row along x, y and z (the histogram form of grids.f:888-951).  The
// more of the convolution an entry does itself, the smaller the histogram:
//   0  the mass at its cell: (BX+2N)(BY+2N)(BZ+2N) cells, one add per entry
//   1  the mass times its kernel column: (BX+2N)(BY+2N) BZ cells, BZ adds
//   2  the mass times its kernel plane: (BX+2N) BY BZ cells, BY BZ adds
// 0 is taken while it fits, then 1, then 2; -1: none fits.  Row and plane
// pitches keep the lanes of a pass on different LDS banks.
struct WideShape {
  int form, ny, nz, px, pz, cells;
};
template <int BX, int BY, int BZ>
__host__ __device__ __forceinline__ WideShape wide_shape(int nk) {
  WideShape w;
  for (int f = 0; f < 3; ++f) {
    w.form = f;
    w.ny = f < 2 ? BY + 2 * nk : BY;
    w.nz = f < 1 ? BZ + 2 * nk : BZ;
    w.px = (BX + 2 * nk) | 1;
    w.pz = w.px * w.ny;
    w.cells = w.pz * w.nz;
    // the x pass holds at most two groups of four outputs per thread
    if (w.cells <= kWideCells && w.ny * w.nz * (BX / 4) <= 2 * kWideThreads) return w;
  }
  w.form = -1;
  return w;
}

// Four outputs o..o+3 of a kernel row of half-width nk applied to a line of
// stride st: s[i] = sum_j line[i + j] K[j - nk], j from 2 nk down to 0.
__device__ __forceinline__ void conv4(const double* line, int st, int nk, const double* K, double s[4]) {
  const double* p = line + 2 * nk * st;
  double a = p[0], b = p[st], c = p[2 * st], d = p[3 * st];
  s[0] = s[1] = s[2] = s[3] = 0.0;
  auto tap = [&](double k, double w, double x, double y, double z) {
    s[0] += w * k;
    s[1] += x * k;
    s[2] += y * k;
    s[3] += z * k;
  };
  // 2 nk + 1 taps, nk even: four at a time, the window's registers in rotation
#pragma unroll 1
  for (int j = 2 * nk; j > 0; j -= 4) {
    tap(K[j], a, b, c, d);
    d = p[-st];
    tap(K[j - 1], d, a, b, c);
    c = p[-2 * st];
    tap(K[j - 2], c, d, a, b);
    b = p[-3 * st];
    tap(K[j - 3], b, c, d, a);
    a = p[-4 * st];
    p -= 4 * st;
  }
  tap(K[0], a, b, c, d);
}

// The wide items, persistent over 8 queues like the deposit.  A tile is taken
// in blocks of at most 16 x 8 x 8 cells, a block class by class: the class's
// masses (or masses times kernel values, see wide_shape) summed as exact
// int64 fixed point on the histogram, then the remaining axes of the
// convolution in FP64, each cell rounded once to the fixed-point unit.  The
// histogram form is used when the item holds all of the tile's wide entries
// (its rounding must not depend on how entries fall into items) and costs
// fewer operations than adding every entry's clipped box cell by cell (an LDS
// add counted as four FP64 multiply-adds).
// Bound by reading the entries once per class and by the LDS reads of the
// convolution.  As part of the narrow kernel the histogram had one layout, so
// N = 8 and more walked every entry's box (29 G adds at 512^3, 6 levels), and
// its LDS left one narrow workgroup per CU: 113 ms, now 12.2 here and 1.9 ms
// in the narrow kernel; 256^3, 4 levels 1,094 -> 85 + 371 us.  256 threads or
// a 41 KB histogram (three workgroups per CU) were slower: 19.2 and 17.5 ms
// when this took 14.7.
template <int RED, int TX, int TY, int TZ>
__global__ void __launch_bounds__(kWideThreads, 4) deposit_wide(Plan P, DepArgs D) {
  using Acc = typename AccT<RED>::T;
  using L = TileLds<TX, TY, TZ>;
  constexpr int BX = TX, BY = TY < 8 ? TY : 8, BZ = TZ < 8 ? TZ : 8, B = BX * BY * BZ;
  constexpr int nthr = kWideThreads;
  static_assert(BX % 4 == 0 && BY % 4 == 0 && BZ % 4 == 0 && B / 4 <= nthr, "four outputs per thread and pass");
  __shared__ long long hist[kWideCells];
  __shared__ Acc acc[B];
  __shared__ double s_k[kWideK];
  __shared__ unsigned s_item;
  __shared__ unsigned s_ccnt[kNLevels + 1];
  double* hd = reinterpret_cast<double*>(hist);
  const int tid = threadIdx.x;
  const double dscale = fixed_scale(D.C->mmax_bits);
  const float scale = (float)dscale;
  const double inv_scale = 1.0 / dscale;   // a power of two: exact
  const unsigned n_narrow = D.C->n_items_eff, n_wide = D.C->n_wide_eff;
  // a cell's FP64 sum into the block's accumulator (one thread per cell)
  auto put = [&](int c, double v) {
    if (RED == 0) acc[c] += (Acc)__double2ll_rn(v);
    else acc[c] += (Acc)(v * inv_scale);
  };
  const int q = blockIdx.x % D.n_queues;
  for (;;) {
    if (tid == 0) s_item = atomicAdd(&D.C->wqueue[q * kLine], 1u) * D.n_queues + q;
    if (tid <= kNLevels) s_ccnt[tid] = 0u;
    __syncthreads();
    const unsigned idx = __builtin_amdgcn_readfirstlane(s_item);
    if (idx >= n_wide) break;
    Item it = D.items[n_narrow + idx];
    const int t = __builtin_amdgcn_readfirstlane(it.tile);
    if (D.cursor) it.end = min(it.end, (long long)D.cursor[2 * t + 1]);
    if (it.end <= it.begin) {
      __syncthreads();   // every wave has read s_item before thread 0 takes the next item
      continue;
    }
    const int g = __builtin_amdgcn_readfirstlane(P.tile_grid[t]);
    const GridDesc& G = P.grids[g];
    const int local = t - G.tile0;
    const int i0 = (local % G.nt[0]) * TX + 1, j0t = ((local / G.nt[0]) % G.nt[1]) * TY + 1,
              k0t = (local / (G.nt[0] * G.nt[1])) * TZ + 1;
    // entries per class (wave ballots, one LDS add per wave and class)
    {
      unsigned cnt[kNLevels + 1] = {};
      for (long long b0 = it.begin; b0 < it.end; b0 += 4 * nthr) {   // four loads in flight
        int irk_e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const long long e = b0 + r * nthr + tid;
          irk_e[r] = e < it.end ? (D.entries[e].y >> 16) : 0;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
          for (int k = 1; k <= kNLevels; ++k) cnt[k] += (unsigned)__popcll(__ballot(irk_e[r] == k));
        }
      }
      if ((tid & 63) == 0)
        for (int k = 1; k <= kNLevels; ++k)
          if (cnt[k]) atomicAdd(&s_ccnt[k], cnt[k]);
    }
    Acc* dst = reinterpret_cast<Acc*>(D.scratch) + (long long)t * L::E;
    const bool alone = D.nitems_tile[t] == 1;
    for (int sub = 0; sub < (TY / BY) * (TZ / BZ); ++sub) {
      const int oy = (sub % (TY / BY)) * BY, oz = (sub / (TY / BY)) * BZ;
      const int j0 = j0t + oy, k0 = k0t + oz;   // the block's first cell
      if (j0 > G.n[1] || k0 > G.n[2]) continue;  // past the grid: never read
      for (int c = tid; c < B; c += nthr) acc[c] = 0;
      __syncthreads();
      for (int irk = 1; irk <= P.nl; ++irk) {
        const unsigned ncls = s_ccnt[irk];
        if (ncls == 0u) continue;
        const int nk = 1 << irk;
        const float* K = P.ktab + irk * P.kw + P.kmax;   // K[d], d in [-N, N]
        const WideShape w = wide_shape<BX, BY, BZ>(nk);
        const long long taps = 2 * nk + 1;
        // The histogram of masses (form 0) when its passes cost less than the
        // entries' direct adds.  The other forms trade the direct adds for 8 or
        // 64 of their own and give the cells another rounding, so a class takes
        // them from four times its passes' cost on (N = 8: 69 entries of a
        // 16 x 8 x 8 tile; with one, two, four and eight times this kernel takes
        // 10.8, 11.4, 12.2 and 15.2 ms at 512^3, 6 levels, and 113 without
        // these forms, the narrow entries included).
        bool use = false;
        if (w.form == 0) {
          const long long bx = TX + 2 * nk, by = TY + 2 * nk, bz = TZ + 2 * nk;
          use = 4 * (long long)ncls * taps * taps * taps > taps * (bx * by * TX + TX * bz * TY + TX * TY * TZ);
        } else if (w.form > 0 && RED == 0) {   // (atomic mode keeps its direct FP32 adds)
          const long long box = (long long)min((int)taps, BX) * min((int)taps, BY) * min((int)taps, BZ);
          const long long adds = w.form == 1 ? BZ : BY * BZ;
          const long long passes = taps * ((long long)BX * w.ny * w.nz + (w.form < 2 ? (long long)BX * BY * w.nz : 0));
          use = 4 * (long long)ncls * (box - adds) > 4 * passes;
        }
        if ((it.flags & 2) && use) {
          // ---- the histogram
          if (tid < taps) s_k[tid] = (double)K[tid - nk];
          for (int c = tid; c < w.cells; c += nthr) hist[c] = 0;
          __syncthreads();
          const double* Kd = s_k + nk;
          int4 nxt = it.begin + tid < it.end ? D.entries[it.begin + tid] : make_int4(0, 0, 0, 0);
          for (long long e = it.begin + tid; e < it.end; e += nthr) {
            const int4 cur = nxt;
            if (e + nthr < it.end) nxt = D.entries[e + nthr];
            int ci[3], irk_e;
            float m;
            unpack_table(cur, ci[0], ci[1], ci[2], irk_e, m);
            if (irk_e != irk) continue;
            const int cx = ci[0] - i0, cy = ci[1] - j0, cz = ci[2] - k0;
            if (cx < -nk || cx >= BX + nk || cy < -nk || cy >= BY + nk || cz < -nk || cz >= BZ + nk) continue;
            const double ms = (double)(m * scale);   // below 2^30 units
            if (w.form == 0) {
              lds_add(hist + (cx + nk) + w.px * (cy + nk) + w.pz * (cz + nk), (long long)__double2int_rn(ms));
              continue;
            }
            const int z0 = max(0, cz - nk), z1 = min(BZ - 1, cz + nk);
            const int y0 = max(0, cy - nk), y1 = min(BY - 1, cy + nk);
            for (int z = z0; z <= z1; ++z) {
              const double mz = ms * Kd[z - cz];
              if (w.form == 1) {
                lds_add(hist + (cx + nk) + w.px * (cy + nk) + w.pz * z, (long long)__double2int_rn(mz));
                continue;
              }
              for (int y = y0; y <= y1; ++y)
                lds_add(hist + (cx + nk) + w.px * y + w.pz * z, (long long)__double2int_rn(mz * Kd[y - cy]));
            }
          }
          __syncthreads();
          for (int c = tid; c < w.cells; c += nthr) hd[c] = (double)hist[c];
          __syncthreads();
          // ---- x: lanes on consecutive rows (odd pitch), four outputs each
          const int rows = w.ny * w.nz, ux = rows * (BX / 4);
          double s[2][4];
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            const int u = tid + r * nthr;
            if (u < ux) conv4(hd + w.px * (u % rows) + 4 * (u / rows), 1, nk, s_k, s[r]);
          }
          if (w.form == 2) {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
              const int u = tid + r * nthr;
              if (u < ux)
                for (int i = 0; i < 4; ++i) put(4 * (u / rows) + i + BX * (u % rows), s[r][i]);
            }
            __syncthreads();
            continue;
          }
          const int pz = BX * w.ny + 16;   // plane pitch of the x pass's output
          __syncthreads();
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            const int u = tid + r * nthr;
            if (u < ux) {
              const int row = u % rows;
              double* o = hd + 4 * (u / rows) + BX * (row % w.ny) + pz * (row / w.ny);
              for (int i = 0; i < 4; ++i) o[i] = s[r][i];
            }
          }
          __syncthreads();
          // ---- y: lanes along x, then z
          const int uy = BX * w.nz * (BY / 4);
          const int ax = tid % BX, az = (tid / BX) % w.nz, ay = 4 * (tid / (BX * w.nz));
          if (tid < uy) conv4(hd + ax + pz * az + BX * ay, BX, nk, s_k, s[0]);
          if (w.form == 1) {
            if (tid < uy)
              for (int i = 0; i < 4; ++i) put(ax + BX * (ay + i + BY * az), s[0][i]);
            __syncthreads();
            continue;
          }
          __syncthreads();
          if (tid < uy)
            for (int i = 0; i < 4; ++i) hd[ax + BX * (ay + i + BY * az)] = s[0][i];
          __syncthreads();
          // ---- z: lanes along x and y
          if (tid < B / 4) {
            const int xy = tid % (BX * BY), zo = 4 * (tid / (BX * BY));
            conv4(hd + xy + BX * BY * zo, BX * BY, nk, s_k, s[0]);
            for (int i = 0; i < 4; ++i) put(xy + BX * BY * (zo + i), s[0][i]);
          }
          __syncthreads();
          continue;
        }
        // ---- direct: a wave reads 64 entries and takes those of the class one
        // by one (short lists: every wave reads them all and takes every
        // eighth, so no wave is left without work).  The entry's box clipped to the block (bx x by x bz cells) is
        // walked as one flat range, lane l taking cells l, l + 64, ...; its
        // (x, y, z) counters advance by constant steps, so the loop has no
        // divisions.  Terms are ((m*Kx)*Ky)*Kz as in the reference's loop.
        const int ex = min(BX, G.n[0] - i0 + 1), ey = min(BY, G.n[1] - j0 + 1), ez = min(BZ, G.n[2] - k0 + 1);
        const int wave = tid >> 6, lane = tid & 63, nwaves = nthr >> 6;
        const int4 none = make_int4(0, 0, 0, 0);   // class 0
        static_assert(nthr / 64 == 8, "every eighth lane");
        const bool shared = it.end - it.begin <= 4 * nthr;
        const unsigned long long share = shared ? 0x0101010101010101ull << wave : ~0ull;
        const int step = shared ? 64 : 64 * nwaves;
        long long e = it.begin + (shared ? 0 : 64 * wave);
        int4 nxt = e + lane < it.end ? D.entries[e + lane] : none;
        unsigned long long todo = 0;
        int4 mine = none;
        for (;;) {
          if (!todo) {
            if (e >= it.end) break;
            mine = nxt;
            e += step;
            nxt = e + lane < it.end ? D.entries[e + lane] : none;
            todo = __ballot((mine.y >> 16) == irk) & share;
            continue;
          }
          const int src = __ffsll((long long)todo) - 1;
          todo &= todo - 1;
          int ci[3], irk_e;
          float m;
          unpack_table(make_int4(__builtin_amdgcn_readlane(mine.x, src), __builtin_amdgcn_readlane(mine.y, src),
                                 __builtin_amdgcn_readlane(mine.z, src), 0),
                       ci[0], ci[1], ci[2], irk_e, m);
          const int xa = max(ci[0] - nk, i0), xb = min(ci[0] + nk, i0 + ex - 1);
          const int ya = max(ci[1] - nk, j0), yb = min(ci[1] + nk, j0 + ey - 1);
          const int za = max(ci[2] - nk, k0), zb = min(ci[2] + nk, k0 + ez - 1);
          if (xb < xa || yb < ya || zb < za) continue;
          const int cx = xb - xa + 1, cy = yb - ya + 1, total = cx * cy * (zb - za + 1);
          // q / n for q <= 64 * 16 and n <= 16: (q + 1/2) / n is at least 1/32
          // away from an integer, far beyond the FP32 error of the product
          const float rbx = 1.0f / (float)cx, rby = 1.0f / (float)cy;
          auto divn = [](int v, float rn) { return (int)(((float)v + 0.5f) * rn); };
          const int r0 = divn(lane, rbx);
          int a = lane - r0 * cx;
          int c = divn(r0, rby);
          int b = r0 - c * cy;
          const int dr = divn(64, rbx), da = 64 - dr * cx;
          const int dc0 = divn(dr, rby), db0 = dr - dc0 * cy;
          const int dc1 = divn(dr + 1, rby), db1 = dr + 1 - dc1 * cy;
          const float ms = RED == 0 ? m * scale : m;
          const float* Kx = K + (xa - ci[0]);
          const float* Ky = K + (ya - ci[1]);
          const float* Kz = K + (za - ci[2]);
          Acc* base = acc + (xa - i0) + BX * ((ya - j0) + BY * (za - k0));
          for (int q2 = lane; q2 < total; q2 += 64) {
            const float term = ((ms * Kx[a]) * Ky[b]) * Kz[c];
            Acc* cell = base + (a + BX * (b + BY * c));
            if (RED == 0) lds_add(reinterpret_cast<long long*>(cell), (long long)__float2int_rn(term));
            else lds_add(reinterpret_cast<float*>(cell), term);
            a += da;
            const bool carry = a >= cx;
            if (carry) a -= cx;
            b += carry ? db1 : db0;
            c += carry ? dc1 : dc0;
            if (b >= cy) {
              b -= cy;
              ++c;
            }
          }
        }
        __syncthreads();
      }
      // the block's cells to the tile's exchange cells, as the deposit's
      for (int c = tid; c < B; c += nthr) {
        Acc* cell = dst + (c % BX + 1) + L::EX * (((c / BX) % BY + oy + 1) + L::EY * (c / (BX * BY) + oz + 1));
        const Acc v = acc[c];
        if (alone) *cell = v;
        else if (v != 0) glb_add(cell, v);
      }
      __syncthreads();
    }
    // wide boxes are clipped to their tile: nothing in the halo
    if (alone)
      for (int c = tid; c < L::E; c += nthr) {
        const int x = c % L::EX, y = (c / L::EX) % L::EY, z = c / (L::EX * L::EY);
        if (x == 0 || x == L::EX - 1 || y == 0 || y == L::EY - 1 || z == 0 || z == L::EZ - 1) dst[c] = 0;
      }
    __syncthreads();   // the item's class counts are read above
  }
}

// The output cells from the tiles' exchange cells.  A workgroup takes a tile
// at a time: a cell is the tile's own sum plus what the stencils of the up to
// 26 neighbouring tiles spilled over it (their halo cells; on the base grid
// the neighbours wrap, and a tile spanning an axis is its own neighbour),
// divided by DENBAS then FDM (FP32, the reference's two divisions) and stored
// row by row.  The exact int64 (FP64 in atomic mode) tile mass is the sum of
// the cells before the divisions.
// Exchanging halo sums costs 14 B written and read per cell of a 16x8x8 tile,
// less than the entries it saves: a stencil crossing tile borders used to be
// binned, emitted and deposited once per tile it touched, 1.5 to 1.8 entries
// per member (the whole build on 256^3 particles and 4 levels 4.01 -> 2.22 ms,
// 512^3 and 6 levels 28.9 -> 18.0 ms).
// Bound by latency in small builds and by the strided halo reads in large ones.
// A thread's four cells are loaded together, their neighbours' terms too: one
// after the other they took 13 us on 38,000 cells (now 6.4), 180 on 18.1M (157)
// and 1,184 on 93.9M (1,016).
template <int RED, int TX, int TY, int TZ>
__global__ void __launch_bounds__(256) combine_tiles(Plan P, DepArgs D) {
  using Acc = typename AccT<RED>::T;
  using L = TileLds<TX, TY, TZ>;
  constexpr int T = TX * TY * TZ;
  __shared__ long long s_nb[27];   // first exchange cell of each neighbour, -1: none or empty
  __shared__ long long s_redi[4];
  __shared__ double s_redd[4];
  stamp(D.C, kClkCombine);
  if (D.C->overflow) return;
  const double inv_scale = 1.0 / fixed_scale(D.C->mmax_bits);   // a power of two: exact
  const int tid = threadIdx.x;
  for (int t = blockIdx.x; t < P.ntiles; t += gridDim.x) {
    const int g = P.tile_grid[t];
    const GridDesc& G = P.grids[g];
    const bool periodic = g == 0;
    const int local = t - G.tile0;
    const int tc[3] = {local % G.nt[0], (local / G.nt[0]) % G.nt[1], local / (G.nt[0] * G.nt[1])};
    const int sh[3] = {TX, TY, TZ};
    int o[3], ext[3], prev[3];   // first cell, cells, and the cell past the last one of the tile before
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      o[a] = tc[a] * sh[a];
      ext[a] = min(sh[a], G.n[a] - o[a]);
      prev[a] = tc[a] > 0 ? sh[a] : G.n[a] - (G.nt[a] - 1) * sh[a];
    }
    if (tid < 27) {
      const int d[3] = {tid % 3 - 1, (tid / 3) % 3 - 1, tid / 9 - 1};
      int c[3];
      bool in = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        c[a] = tc[a] + d[a];
        if (periodic) c[a] = c[a] < 0 ? G.nt[a] - 1 : (c[a] >= G.nt[a] ? 0 : c[a]);
        else in = in && c[a] >= 0 && c[a] < G.nt[a];
      }
      const int tn = G.tile0 + (c[2] * G.nt[1] + c[1]) * G.nt[0] + c[0];
      s_nb[tid] = in && tile_filled(D, tn) ? (long long)tn * L::E : -1ll;
    }
    __syncthreads();
    const Acc* S = reinterpret_cast<const Acc*>(D.scratch);
    float* out = (g == 0 ? D.u1 : D.u11) + G.off;
    long long msi = 0;
    double msd = 0.0;
    const long long own = s_nb[13];
    const bool thin = ext[0] == 1 || ext[1] == 1 || ext[2] == 1;
    constexpr int U = T / 256 < 4 ? T / 256 : 4;   // cells of a thread in flight
    for (int c0 = tid; c0 < T; c0 += 256 * U) {
      Acc v[U];
      if (!thin) {
        // a cell has a neighbour on at most one side per axis: up to 7 terms,
        // all loads issued before the first is used
        Acc term[U][8];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int c = c0 + 256 * u;
          const int l[3] = {c % TX, (c / TX) % TY, c / (TX * TY)};
          const bool on = l[0] < ext[0] && l[1] < ext[1] && l[2] < ext[2];
          constexpr int pitch[3] = {1, L::EX, L::EX * L::EY}, step[3] = {1, 3, 9};
          int self[3], side[3], nbr[3];   // the cell's offset, as seen from its side's tile, and that tile's slot
          bool has[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const bool low = l[a] == 0, high = l[a] == ext[a] - 1;
            has[a] = on && (low || high);
            self[a] = (l[a] + 1) * pitch[a];
            side[a] = (low ? prev[a] + 1 : 0) * pitch[a];
            nbr[a] = low ? -step[a] : step[a];
          }
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            term[u][k] = 0;
            const bool need = k == 0 ? on && own >= 0
                                     : (!(k & 1) || has[0]) && (!(k & 2) || has[1]) && (!(k & 4) || has[2]);
            if (need) {
              const long long nb =
                  k == 0 ? own : s_nb[13 + (k & 1 ? nbr[0] : 0) + (k & 2 ? nbr[1] : 0) + (k & 4 ? nbr[2] : 0)];
              if (nb >= 0)
                term[u][k] = S[nb + (k & 1 ? side[0] : self[0]) + (k & 2 ? side[1] : self[1]) +
                               (k & 4 ? side[2] : self[2])];
            }
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          v[u] = term[u][0];
#pragma unroll
          for (int k = 1; k < 8; ++k) v[u] += term[u][k];
        }
      } else {
        // a tile one cell wide: neighbours on both sides of a cell
#pragma unroll 1
        for (int u = 0; u < U; ++u) {
          const int c = c0 + 256 * u;
          const int l[3] = {c % TX, (c / TX) % TY, c / (TX * TY)};
          Acc w = 0;
          if (l[0] < ext[0] && l[1] < ext[1] && l[2] < ext[2]) {
            int lo[3], hi[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
              lo[a] = l[a] == 0 ? -1 : 0;
              hi[a] = l[a] == ext[a] - 1 ? 1 : 0;
            }
            for (int dz = lo[2]; dz <= hi[2]; ++dz)
              for (int dy = lo[1]; dy <= hi[1]; ++dy)
                for (int dx = lo[0]; dx <= hi[0]; ++dx) {
                  const long long nb = s_nb[(dx + 1) + 3 * ((dy + 1) + 3 * (dz + 1))];
                  if (nb < 0) continue;
                  // this cell in the neighbour's coordinates: past the last cell
                  // of the tile before, or the halo below the tile after
                  const int x = dx == 0 ? l[0] : (dx < 0 ? prev[0] : -1);
                  const int y = dy == 0 ? l[1] : (dy < 0 ? prev[1] : -1);
                  const int z = dz == 0 ? l[2] : (dz < 0 ? prev[2] : -1);
                  w += S[nb + (x + 1) + L::EX * ((y + 1) + L::EY * (z + 1))];
                }
          }
#pragma unroll
          for (int q = 0; q < U; ++q)
            if (q == u) v[q] = w;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + 256 * u;
        const int l[3] = {c % TX, (c / TX) % TY, c / (TX * TY)};
        if (l[0] >= ext[0] || l[1] >= ext[1] || l[2] >= ext[2]) continue;
        if (RED == 0) msi += (long long)v[u];
        else msd += (double)v[u];
        float f = RED == 0 ? (float)((double)v[u] * inv_scale) : (float)v[u];
        f = f / G.den;
        f = f / P.fdm;
        out[(long long)(o[0] + l[0]) + (long long)G.ld1 * (o[1] + l[1]) + (long long)G.ld2 * (o[2] + l[2])] = f;
      }
    }
    if (RED == 0) {
      msi = block_sum(msi, s_redi);
      if (tid == 0) D.tile_mass_i[t] = msi;
    } else {
      msd = block_sum(msd, s_redd);
      if (tid == 0) D.tile_mass_d[t] = msd;
    }
  }
}

// Clears the exchange cells of the tiles that several work items add to; a
// kernel, not a memset, so the build can be captured.
__global__ void __launch_bounds__(256) zero_split(DepArgs D, int ntiles, int words) {
  if (D.C->overflow) return;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    if (D.nitems_tile[t] <= 1) continue;
    unsigned* p = reinterpret_cast<unsigned*>(D.scratch) + (long long)t * words;
    for (int i = threadIdx.x; i < words; i += blockDim.x) p[i] = 0u;
  }
}

// per-grid mass in a fixed order; FP64 (int64-exact in deterministic mode)
template <int RED>
__global__ void __launch_bounds__(256) grid_sums(Plan P, DepArgs D, double* grid_mass) {
  __shared__ long long shi[16];
  __shared__ double shd[16];
  const int g = blockIdx.x;
  const GridDesc& G = P.grids[g];
  const int nt = G.level == 0 && g != 0 ? 0 : G.nt[0] * G.nt[1] * G.nt[2];
  if (RED == 0) {
    long long s = 0;
    for (int k = threadIdx.x; k < nt; k += blockDim.x) s += D.tile_mass_i[G.tile0 + k];
    s = block_sum(s, shi);
    if (threadIdx.x == 0) grid_mass[g] = (double)s / fixed_scale(D.C->mmax_bits);
  } else {
    double s = 0;
    for (int k = threadIdx.x; k < nt; k += blockDim.x) s += D.tile_mass_d[G.tile0 + k];
    s = block_sum(s, shd);
    if (threadIdx.x == 0) grid_mass[g] = s;
  }
}

// The first kernel of a call binned through the base grid: clears the
// counters (the queue lengths to n_narrow and n_wide), the items' member
// counts and the exchange cells of the tiles that several items add to, and
// starts every tile's range empty.
// One launch for what took six, and no events, memory copy or sums of their
// own at the call's end (finish_call): a small call is bound by its launches
// and the gaps between them.  13,824 particles 245 -> 189 us, 250,047 (kernel
// table, graph) 247 -> 225, 2.1M (kernel table) 409 -> 352.
__global__ void __launch_bounds__(256) begin_call(DepArgs D, unsigned n_narrow, unsigned n_wide, unsigned* item_pairs,
                                                  long long n_items, unsigned long long* cursor, long long nkeys,
                                                  const int* split_tiles, const unsigned* n_split, int words) {
  const long long i0 = blockIdx.x * (long long)blockDim.x + threadIdx.x, di = (long long)gridDim.x * blockDim.x;
  Counters* C = D.C;
  unsigned* c = reinterpret_cast<unsigned*>(C);
  const long long eff = &C->n_items_eff - c, wide = &C->n_wide_eff - c;
  const long long clk0 = reinterpret_cast<unsigned*>(C->clk) - c, clk1 = clk0 + kLine;
  for (long long k = i0; k < (long long)(sizeof(Counters) / 4); k += di)
    if (k < clk0 || k >= clk1) c[k] = k == eff ? n_narrow : (k == wide ? n_wide : 0u);
  stamp(C, kClkBegin);
  for (long long k = i0; k < n_items; k += di) item_pairs[k] = 0u;
  for (long long k = i0; k < nkeys; k += di) cursor[k] = D.start[k];
  const unsigned ns = *n_split;
  for (unsigned k = blockIdx.x; k < ns; k += gridDim.x) {
    unsigned* p = reinterpret_cast<unsigned*>(D.scratch) + (long long)split_tiles[k] * words;
    for (int w = threadIdx.x; w < words; w += 256) p[w] = 0u;
  }
}

// The last kernel of such a call: every grid's mass in a fixed order (a wave
// per grid; a workgroup where the grid has many tiles), the call's members
// (what the emission's items found; base members are in the counters already)
// and entries (the filled part of every tile's range), and, by the last
// workgroup to end, the counters written to the host.
template <int RED>
__global__ void __launch_bounds__(256) finish_call(Plan P, DepArgs D, double* grid_mass, const unsigned* item_pairs,
                                                   long long n_items, long long nkeys, unsigned* host) {
  __shared__ long long shi[4];
  __shared__ double shd[4];
  __shared__ unsigned long long sp[4], se[4];
  __shared__ unsigned s_last;
  constexpr int kWaveTiles = 1024;   // tiles up to which a wave sums a grid
  Counters* C = D.C;
  stamp(C, kClkSums);
  const int tid = threadIdx.x, lane = tid & 63;
  const double scale = fixed_scale(C->mmax_bits);
  auto tiles = [&](int g) {
    const GridDesc& G = P.grids[g];
    return G.level == 0 && g != 0 ? 0 : G.nt[0] * G.nt[1] * G.nt[2];
  };
  if (grid_mass) {
    for (int g = blockIdx.x * 4 + (tid >> 6); g < P.ngrids; g += gridDim.x * 4) {
      const int nt = tiles(g), t0 = P.grids[g].tile0;
      if (nt > kWaveTiles) continue;
      if (RED == 0) {
        long long s = 0;
        for (int k = lane; k < nt; k += 64) s += D.tile_mass_i[t0 + k];
        s = wave_sum(s);
        if (lane == 0) grid_mass[g] = (double)s / scale;
      } else {
        double s = 0;
        for (int k = lane; k < nt; k += 64) s += D.tile_mass_d[t0 + k];
        s = wave_sum(s);
        if (lane == 0) grid_mass[g] = s;
      }
    }
    for (int g = blockIdx.x; g < P.ngrids; g += gridDim.x) {
      const int nt = tiles(g), t0 = P.grids[g].tile0;
      if (nt <= kWaveTiles) continue;
      long long si[8] = {};
      double sd[8] = {};
      for (int k0 = tid; k0 < nt; k0 += 8 * 256) {   // eight loads in flight
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const int k = k0 + r * 256;
          if (k < nt) {
            if (RED == 0) si[r] += D.tile_mass_i[t0 + k];
            else sd[r] += D.tile_mass_d[t0 + k];
          }
        }
      }
#pragma unroll
      for (int r = 1; r < 8; ++r) { si[0] += si[r]; sd[0] += sd[r]; }
      if (RED == 0) {
        const long long s = block_sum(si[0], shi);
        if (tid == 0) grid_mass[g] = (double)s / scale;
      } else {
        const double s = block_sum(sd[0], shd);
        if (tid == 0) grid_mass[g] = s;
      }
    }
  }
  unsigned long long p = 0, e = 0;
  const long long i0 = blockIdx.x * (long long)blockDim.x + tid, di = (long long)gridDim.x * blockDim.x;
  for (long long i = i0; i < n_items; i += di) p += item_pairs[i];
  for (long long k = i0; k < nkeys; k += di) e += D.cursor[k] - D.start[k];
  p = wave_sum(p);
  e = wave_sum(e);
  if (lane == 0) { sp[tid >> 6] = p; se[tid >> 6] = e; }
  __syncthreads();
  if (tid == 0) {
    p = sp[0] + sp[1] + sp[2] + sp[3];
    e = se[0] + se[1] + se[2] + se[3];
    if (p) atomicAdd(&C->n_pairs, p);
    if (e) atomicAdd(&C->n_entries, e);
    __threadfence();
    s_last = atomicAdd(&C->ticket, 1u) == gridDim.x - 1 ? 1u : 0u;
  }
  __syncthreads();
  if (!s_last) return;
  if (tid == 0) C->clk[kClkEnd] = wall_clock64();
  __syncthreads();
  __threadfence();
  if (tid < kHostWords)
    host[tid] = __hip_atomic_load(reinterpret_cast<unsigned*>(C) + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __threadfence_system();
}

// ---------------------------------------------------------------------------
// adjoint of the TSC mode: one thread per particle, gathers the upstream
// gradient at every stencil cell of every grid the particle belongs to
// ---------------------------------------------------------------------------
// three consecutive cells of a row in one load (dword alignment suffices)
struct __attribute__((aligned(4))) Row3 {
  float v[3];
};
__device__ __forceinline__ void load_row3(const float* p, float out[3]) {
  const Row3 r = *reinterpret_cast<const Row3*>(p);
  out[0] = r.v[0];
  out[1] = r.v[1];
  out[2] = r.v[2];
}

// Gather key of every particle for the adjoint: the bits of its position in
// base cells of 2^-sub, interleaved, so that neighbours in the order are
// neighbours in space and their gradient rows are cached together.  The pass
// also packs the particles, (x, y, z, m) in one 16-byte record each (rec NULL:
// not), and makes the TSC input checks (non-finite values, negative masses,
// positions outside the base range: the flags of the forward's validation), as
// it reads the positions anyway.
__global__ void __launch_bounds__(256) cell_keys(Plan P, Parts A, KeyBits B, unsigned* key, unsigned* idx,
                                                 float4* rec, Counters* C) {
  const GridDesc& G = P.grids[0];
  unsigned err = 0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < A.n;
       i += (long long)gridDim.x * blockDim.x) {
    const float p[3] = {A.x[i], A.y[i], A.z[i]};
    const float m = A.m[i];
    if (!(isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]) && isfinite(m))) {
      err |= kErrNonFinite;
    } else {
      if (m < 0.f) err |= kErrNegMass;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        if (!tsc_base_in_range(p[a], P.xl, G.inv_d[a], G.n[a])) err |= kErrWrap;
    }
    unsigned c[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float t = (p[a] - P.xl) * G.inv_d[a] * B.scale;
      c[a] = t > 0.f ? min((unsigned)fminf(t, 2.0e9f), (1u << B.b[a]) - 1u) : 0u;
    }
    // highest bits first; an axis out of bits drops out
    unsigned k = 0u;
    for (int b = max(max(B.b[0], B.b[1]), B.b[2]); b-- > 0;)
#pragma unroll
      for (int a = 2; a >= 0; --a)
        if (b < B.b[a]) k = (k << 1) | ((c[a] >> b) & 1u);
    key[i] = k;
    if (rec) rec[i] = make_float4(p[0], p[1], p[2], m);
    idx[i] = (unsigned)i;
  }
  err = wave_or(err);
  if ((threadIdx.x & 63) == 0 && err) atomicOr(&C->err, err);
}

// One (particle, grid) term of the adjoint: the nine rows of three gradient
// values around the centre cell, weighted.  Per row (b, c):
// sx = sum_a wx_a g, sdx = sum_a wx'_a g; then am += wy wz sx,
// ax += wy wz sdx, ay += wy' wz sx, az += wy dwz sx.
struct AdjAcc {
  float am = 0.f, ax = 0.f, ay = 0.f, az = 0.f;
  __device__ __forceinline__ void row(const float gv[3], const float w[3][3], const float dw[3][3], int b, int c,
                                      float sc) {
    const float sx = (w[0][0] * gv[0] + w[0][1] * gv[1] + w[0][2] * gv[2]) * sc;
    const float sdx = (dw[0][0] * gv[0] + dw[0][1] * gv[1] + dw[0][2] * gv[2]) * sc;
    const float yz = w[1][b] * w[2][c];
    am += yz * sx;
    ax += yz * sdx;
    ay += dw[1][b] * w[2][c] * sx;
    az += w[1][b] * dw[2][c] * sx;
  }
};

// One thread per particle, in the given order (NULL: index order).  The
// result of a particle does not depend on the order.  With packed records the
// particle is read from its record and its results replace it there (dm, dx,
// dy, dz; adjoint_unpack moves them to their arrays): in another order than the
// arrays', every access to one costs a 64-byte sector, and a record is one
// sector instead of four in and four out.  Eight workgroups per CU (at most 64
// VGPRs, a few of them spilled): the gather waits on memory, and the extra waves
// in flight gain more than the spills cost.
// 16.8M particles, 4 levels: 2,909 us in x-fastest order of the cells without
// records; with both 1,720 and 89 to unpack, the whole adjoint 3,290 -> 2,440
// us; 2.1M 370 -> 354 us.  A contiguous part of the order per XCD was slower by
// 1 to 5 percent (the parts' costs differ).
__global__ void __launch_bounds__(256, 8) adjoint_gather(Plan P, Parts A, const float* g1, const float* g11,
                                                      float* dm, float* dxo, float* dyo, float* dzo,
                                                      const unsigned* order, float4* rec) {
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < A.n;
       t += (long long)gridDim.x * blockDim.x) {
    const long long i = order ? (long long)order[t] : t;
    if (i >= A.n) continue;   // the order is a permutation of [0, n); checked so a bad one cannot read out of range
    const float4 r = rec ? rec[i] : make_float4(A.x[i], A.y[i], A.z[i], A.m[i]);
    const float p[3] = {r.x, r.y, r.z};
    const float m = r.w;
    AdjAcc acc;
    // the first level's hash slot is loaded while the base grid is handled
    Probe nxt;
    if (P.nl >= 1) nxt = probe_start(P, 1, p[0], p[1], p[2]);
    // base grid
    {
      const GridDesc& G = P.grids[0];
      int ci[3];
      float w[3][3], dw[3][3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        ci[a] = tsc_base_index(p[a], P.xl, G.d[a], G.inv_d[a], G.n[a]);
        tsc_weights_dc(p[a], base_centre(P, a, ci[a] - 1, G.n[a]), base_centre(P, a, ci[a], G.n[a]),
                       base_centre(P, a, ci[a] + 1, G.n[a]), G.inv_d[a], w[a], dw[a]);
      }
      const float sc = 1.0f / (G.den * P.fdm);
      // the three x cells of a row are contiguous unless the row wraps
      const bool xin = ci[0] >= 2 && ci[0] <= G.n[0] - 1;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const long long kz = wrap1(ci[2] - 1 + c, G.n[2]) - 1;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          const long long jy = wrap1(ci[1] - 1 + b, G.n[1]) - 1;
          const float* row = g1 + G.off + G.ld1 * jy + G.ld2 * kz;
          float gv[3];
          if (xin) {
            load_row3(row + (ci[0] - 2), gv);
          } else {
#pragma unroll
            for (int a = 0; a < 3; ++a) gv[a] = row[wrap1(ci[0] - 1 + a, G.n[0]) - 1];
          }
          acc.row(gv, w, dw, b, c, sc);
        }
      }
    }
    // the descent stops where the forward enumeration stops (nested boxes)
    for (int l = 1; l <= P.nl; ++l) {
      const int2 se = probe_finish(P, nxt);
      if (l < P.nl) nxt = probe_start(P, l + 1, p[0], p[1], p[2]);
      bool any = false;
      for (int q = 0; q < se.y; ++q) {
        const BoxRec& G = P.hrec[se.x + q];   // the grid's fields travel in its candidate record
        if (!in_box(G, p[0], p[1], p[2])) continue;
        any = true;
        int ci[3];
        float w[3][3], dw[3][3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          ci[a] = (int)index_quotient(p[a] - G.org[a], G.d[a], G.inv_d[a]);
          tsc_weights_dc(p[a], minirad(G.pr[a], ci[a] - 1, G.d[a]), minirad(G.pr[a], ci[a], G.d[a]),
                         minirad(G.pr[a], ci[a] + 1, G.d[a]), G.inv_d[a], w[a], dw[a]);
        }
        const float sc = 1.0f / (G.den * P.fdm);
        const float* gp = g11 + G.off;
        const bool xin = ci[0] >= 2 && ci[0] <= G.n[0] - 1;
        const long long ld1 = G.ld1, ld2 = G.ld2;
        const int gn0 = G.n[0], gn1 = G.n[1], gn2 = G.n[2];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const int kz = ci[2] - 1 + c;
          if (kz < 1 || kz > gn2) continue;
#pragma unroll
          for (int b = 0; b < 3; ++b) {
            const int jy = ci[1] - 1 + b;
            if (jy < 1 || jy > gn1) continue;
            const float* row = gp + ld1 * (jy - 1) + ld2 * (kz - 1);
            float gv[3];
            if (xin) {
              load_row3(row + (ci[0] - 2), gv);
            } else {
#pragma unroll
              for (int a = 0; a < 3; ++a) {
                const int ix = ci[0] - 1 + a;
                gv[a] = (ix >= 1 && ix <= gn0) ? row[ix - 1] : 0.f;
              }
            }
            acc.row(gv, w, dw, b, c, sc);
          }
        }
      }
      if (!any && P.nested) break;
    }
    if (rec) {
      rec[i] = make_float4(acc.am, m * acc.ax, m * acc.ay, m * acc.az);
    } else {
      dm[i] = acc.am;
      dxo[i] = m * acc.ax;
      dyo[i] = m * acc.ay;
      dzo[i] = m * acc.az;
    }
  }
}

// the adjoint's results from their records to the caller's arrays
__global__ void __launch_bounds__(256) adjoint_unpack(long long n, const float4* rec, float* dm, float* dx, float* dy,
                                                      float* dz) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const float4 r = rec[i];
    dm[i] = r.x;
    dx[i] = r.y;
    dy[i] = r.z;
    dz[i] = r.w;
  }
}

// ---------------------------------------------------------------------------
// plain form: one launch per grid, global FP32 atomics into the outputs
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) plain_zero(Plan P, float* u1, float* u11) {
  const GridDesc& G = P.grids[blockIdx.x];
  if (G.level == 0 && blockIdx.x != 0) return;
  float* out = (blockIdx.x == 0 ? u1 : u11) + G.off;
  const long long nc = (long long)G.n[0] * G.n[1] * G.n[2];
  for (long long c = threadIdx.x; c < nc; c += blockDim.x) {
    const long long a = c % G.n[0], r = c / G.n[0], b = r % G.n[1], cz = r / G.n[1];
    out[a + G.ld1 * b + G.ld2 * cz] = 0.f;
  }
}

template <int MODE>
__global__ void __launch_bounds__(256) plain_base(Plan P, Parts A, float* u1) {
  const GridDesc& G = P.grids[0];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < A.n;
       i += (long long)gridDim.x * blockDim.x) {
    const float p[3] = {A.x[i], A.y[i], A.z[i]};
    const float m = A.m[i];
    int ci[3];
    float w[3][3];
    if (MODE == 2) {
      const float* rad[3] = {P.radx, P.rady, P.radz};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        ci[a] = tsc_base_index(p[a], P.xl, G.d[a], G.inv_d[a], G.n[a]);
        tsc_weights(p[a], rad[a][ci[a] - 1], rad[a][ci[a]], rad[a][ci[a] + 1], G.d[a], w[a]);
      }
    } else {
      bool ok = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float t = (p[a] - P.xl) / G.d[a];
        ok = ok && t > -1.0e9f && t < 1.0e9f;
        ci[a] = ok ? (int)t + 1 : 1;
        ok = ok && ci[a] >= 2 - G.n[a] && ci[a] <= 2 * G.n[a] - 1;
        w[a][0] = P.ktab[P.kmax - 1]; w[a][1] = P.ktab[P.kmax]; w[a][2] = P.ktab[P.kmax + 1];
      }
      if (!ok) continue;   // rejected by the count pass of the same call
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const long long kz = wrap1(ci[2] - 1 + c, G.n[2]) - 1;
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        const long long jy = wrap1(ci[1] - 1 + b, G.n[1]) - 1;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const long long ix = wrap1(ci[0] - 1 + a, G.n[0]) - 1;
          atomicAdd(u1 + G.off + ix + G.ld1 * jy + G.ld2 * kz, m * w[0][a] * w[1][b] * w[2][c]);
        }
      }
    }
  }
}

// input validation of the plain form (same flags as the count pass)
template <int MODE>
__global__ void __launch_bounds__(256) plain_validate(Plan P, Parts A, Counters* C) {
  unsigned err = 0;
  const GridDesc& B = P.grids[0];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < A.n;
       i += (long long)gridDim.x * blockDim.x) {
    const float p[3] = {A.x[i], A.y[i], A.z[i]};
    const float m = A.m[i];
    if (!(isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]) && isfinite(m))) { err |= kErrNonFinite; continue; }
    if (m < 0.f) err |= kErrNegMass;
    if (MODE == 2) {
#pragma unroll
      for (int a = 0; a < 3; ++a)
        if (!tsc_base_in_range(p[a], P.xl, B.inv_d[a], B.n[a])) err |= kErrWrap;
    }
    if (MODE == 1) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float t = (p[a] - P.xl) / B.d[a];
        if (!(t > -1.0e9f && t < 1.0e9f)) { err |= kErrWrap; break; }
        const int c = (int)t + 1;
        if (c < 2 - B.n[a] || c > 2 * B.n[a] - 1) err |= kErrWrap;
      }
    }
  }
  err = wave_or(err);
  if ((threadIdx.x & 63) == 0 && err) atomicOr(&C->err, err);
}

// level membership flags for the plain form's per-level compaction: flag = 1
// when the particle lies in some level-l box (TSC: the PLEV rule of
// grids.f:1114-1157; table mode: the DX-extended boxes of grids.f:871-909)
__global__ void __launch_bounds__(256) plain_level_flags(Plan P, Parts A, int l, unsigned* flag) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < A.n;
       i += (long long)gridDim.x * blockDim.x) {
    const float x = A.x[i], y = A.y[i], z = A.z[i];
    unsigned f = 0;
    const int2 se = bucket_lookup(P, l, x, y, z);
    for (int q = 0; q < se.y && !f; ++q)
      if (in_box(P.hrec[se.x + q], x, y, z)) f = 1;
    flag[i] = f;
  }
}

__global__ void plain_compact(const unsigned* flag, const unsigned long long* start, long long n,
                              long long* idx) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    if (flag[i]) idx[start[i]] = i;
}

template <int MODE>
__global__ void __launch_bounds__(256) plain_patch(Plan P, Parts A, int g, const long long* idx,
                                                   const unsigned long long* nidx_p, float* u11) {
  const GridDesc& G = P.grids[g];
  const long long nidx = (long long)*nidx_p;
  float* out = u11 + G.off;
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < nidx;
       k += (long long)gridDim.x * blockDim.x) {
    const long long i = idx[k];
    const float p[3] = {A.x[i], A.y[i], A.z[i]};
    if (!(G.lo[0] < p[0] && p[0] < G.hi[0] && G.lo[1] < p[1] && p[1] < G.hi[1] && G.lo[2] < p[2] && p[2] < G.hi[2]))
      continue;
    const float m = A.m[i];
    if (MODE == 2) {
      int ci[3];
      float w[3][3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        ci[a] = (int)((p[a] - G.org[a]) / G.d[a]);
        tsc_weights(p[a], minirad(G.pr[a], ci[a] - 1, G.d[a]), minirad(G.pr[a], ci[a], G.d[a]),
                    minirad(G.pr[a], ci[a] + 1, G.d[a]), G.d[a], w[a]);
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int kz = ci[2] - 1 + c;
        if (kz < 1 || kz > G.n[2]) continue;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          const int jy = ci[1] - 1 + b;
          if (jy < 1 || jy > G.n[1]) continue;
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const int ix = ci[0] - 1 + a;
            if (ix < 1 || ix > G.n[0]) continue;
            atomicAdd(out + (ix - 1) + (long long)G.ld1 * (jy - 1) + (long long)G.ld2 * (kz - 1),
                      m * w[0][a] * w[1][b] * w[2][c]);
          }
        }
      }
    } else {
      const int s = species_of(A, i);
      const int irk = max(G.level - s, 0), nk = 1 << irk;
      const float* K = P.ktab + irk * P.kw + P.kmax;
      int ci[3], lo[3], hi[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        ci[a] = (int)floorf((p[a] - G.org[a]) / G.d[a]) + 1;
        lo[a] = max(ci[a] - nk, 1);
        hi[a] = min(ci[a] + nk, G.n[a]);
      }
      for (int kk = lo[2]; kk <= hi[2]; ++kk)
        for (int jj = lo[1]; jj <= hi[1]; ++jj)
          for (int ii = lo[0]; ii <= hi[0]; ++ii)
            atomicAdd(out + (ii - 1) + (long long)G.ld1 * (jj - 1) + (long long)G.ld2 * (kk - 1),
                      m * K[ii - ci[0]] * K[jj - ci[1]] * K[kk - ci[2]]);
    }
  }
}

// normalise every grid (/DENBAS, then /FDM) and sum its mass in FP64
__global__ void __launch_bounds__(256) plain_finish(Plan P, float* u1, float* u11, double* grid_mass) {
  __shared__ double sh[16];
  const int g = blockIdx.x;
  const GridDesc& G = P.grids[g];
  if (G.level == 0 && g != 0) {
    if (threadIdx.x == 0 && grid_mass) grid_mass[g] = 0.0;
    return;
  }
  float* out = (g == 0 ? u1 : u11) + G.off;
  const long long nc = (long long)G.n[0] * G.n[1] * G.n[2];
  double s = 0.0;
  for (long long c = threadIdx.x; c < nc; c += blockDim.x) {
    const long long a = c % G.n[0], r = c / G.n[0], b = r % G.n[1], cz = r / G.n[1];
    float* q = out + a + G.ld1 * b + G.ld2 * cz;
    const float v = *q;
    s += v;
    *q = (v / G.den) / P.fdm;
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0 && grid_mass) grid_mass[g] = s;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static int grid_for(long long n, int block, int cap) {
  long long b = (n + block - 1) / block;
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return (int)b;
}

hipError_t launch_fill_u32(unsigned* p, unsigned v, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  fill_u32_kernel<<<grid_for(n, 256, 65536), 256, 0, s>>>(p, v, n);
  return hipGetLastError();
}

long long bin_blocks(long long n) { return (n + kBinChunk - 1) / kBinChunk; }

hipError_t launch_count(const Plan& P, const Parts& A, unsigned* cnt, Counters* C, const BlockTables& BT,
                        int cus, hipStream_t s) {
  (void)cus;
  if (A.n <= 0) return hipSuccess;
  const int grid = (int)bin_blocks(A.n);
  if (P.mode == 2) count_kernel<2><<<grid, 256, 0, s>>>(P, A, cnt, C, BT);
  else count_kernel<1><<<grid, 256, 0, s>>>(P, A, cnt, C, BT);
  return hipGetLastError();
}

hipError_t launch_scatter(const Plan& P, const Parts& A, unsigned long long* cursor, int4* entries,
                          unsigned long long cap, const BlockTables& BT, const Counters* C, int cus,
                          hipStream_t s) {
  (void)cus;
  if (A.n <= 0) return hipSuccess;
  const int grid = (int)bin_blocks(A.n);
  if (P.mode == 2) scatter_kernel<2><<<grid, 256, 0, s>>>(P, A, cursor, entries, cap, BT, C);
  else scatter_kernel<1><<<grid, 256, 0, s>>>(P, A, cursor, entries, cap, BT, C);
  return hipGetLastError();
}

hipError_t launch_membership(const Plan& P, const Parts& A, int* out, long long cap,
                             unsigned long long* count, int cus, hipStream_t s) {
  const int grid = grid_for(A.n, 256, cus * 16);
  if (P.mode == 2) membership_kernel<2><<<grid, 256, 0, s>>>(P, A, out, cap, count);
  else membership_kernel<1><<<grid, 256, 0, s>>>(P, A, out, cap, count);
  return hipGetLastError();
}

long long scan_scratch_elems(long long n) { return (n + kScanTile - 1) / kScanTile + 1; }

hipError_t launch_scan(const unsigned* in, long long n, unsigned long long* bsum, unsigned long long* start,
                       unsigned long long* cursor, hipStream_t s) {
  const int nb = (int)((n + kScanTile - 1) / kScanTile);
  if (nb > 0) scan_reduce<<<nb, kScanThreads, 0, s>>>(in, n, bsum);
  scan_bsums<<<1, kScanThreads, 0, s>>>(bsum, nb, start + n);
  if (nb > 0) scan_apply<<<nb, kScanThreads, 0, s>>>(in, n, bsum, start, cursor);
  return hipGetLastError();
}

hipError_t launch_reduce_blocks(const BlockTables& BT, long long nblk, Counters* C, int cus, hipStream_t s) {
  if (nblk <= 0) return hipSuccess;
  const long long want = (nblk + 255) / 256;
  reduce_blocks<<<(int)std::min<long long>(want, (long long)std::max(cus, 1) * 4), 256, 0, s>>>(BT, nblk, C);
  return hipGetLastError();
}

hipError_t launch_plan_count(const unsigned long long* start, int ntiles, int chunk, int chunk_wide,
                             unsigned* cnt, unsigned* nitems_tile, hipStream_t s) {
  plan_count<<<grid_for(ntiles, 256, 1 << 30), 256, 0, s>>>(start, ntiles, chunk, chunk_wide, cnt, nitems_tile);
  return hipGetLastError();
}

hipError_t launch_plan_write(const unsigned long long* start, int ntiles, int chunk, int chunk_wide,
                             const unsigned long long* item_off, Item* items, int* split_tiles, unsigned* n_split,
                             const Counters* C, hipStream_t s) {
  plan_write<<<grid_for(ntiles, 256, 1 << 30), 256, 0, s>>>(start, ntiles, chunk, chunk_wide, item_off, items,
                                                           split_tiles, n_split, C);
  return hipGetLastError();
}

// n < 0: the items that the gate admitted, at most n_max
hipError_t launch_order_items(const Item* items, Item* work, long long n, long long n_max, Counters* C, int cus,
                              hipStream_t s) {
  const int grid = grid_for(std::max(n_max, 1ll), 1024, cus);
  order_items<<<grid, 256, 0, s>>>(items, work, n, C, 0);
  order_items<<<grid, 256, 0, s>>>(items, work, n, C, 1);
  return hipGetLastError();
}

hipError_t launch_gate(const unsigned long long* tot_entries, const unsigned long long* item_off, int ntiles,
                       unsigned long long cap_entries, unsigned long long cap_items, Counters* C, hipStream_t s) {
  gate_kernel<<<1, 64, 0, s>>>(tot_entries, item_off, ntiles, cap_entries, cap_items, C);
  return hipGetLastError();
}

// the narrow items' kernel on tiles of TX x TY x TZ cells
template <int TX, int TY, int TZ>
static void narrow_tile(const Plan& P, const DepArgs& D, int red, int grid, int block, hipStream_t s) {
  if (P.mode == 1 && red == 0) deposit_counts<TX, TY, TZ><<<grid, block, 0, s>>>(P, D);
  else if (P.mode == 1) deposit_kernel<1, 1, TX, TY, TZ><<<grid, block, 0, s>>>(P, D);
  else if (red == 0) deposit_kernel<2, 0, TX, TY, TZ><<<grid, block, 0, s>>>(P, D);
  else deposit_kernel<2, 1, TX, TY, TZ><<<grid, block, 0, s>>>(P, D);
}

template <int RED>
static hipError_t wide_shape_launch(const Plan& P, const DepArgs& D, int grid, hipStream_t s) {
  const int* t = P.tile;
  if (t[0] == 8 && t[1] == 8 && t[2] == 8) deposit_wide<RED, 8, 8, 8><<<grid, kWideThreads, 0, s>>>(P, D);
  else if (t[0] == 16 && t[1] == 8 && t[2] == 8) deposit_wide<RED, 16, 8, 8><<<grid, kWideThreads, 0, s>>>(P, D);
  else if (t[0] == 16 && t[1] == 16 && t[2] == 8) deposit_wide<RED, 16, 16, 8><<<grid, kWideThreads, 0, s>>>(P, D);
  else if (t[0] == 16 && t[1] == 16 && t[2] == 16) deposit_wide<RED, 16, 16, 16><<<grid, kWideThreads, 0, s>>>(P, D);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

// the wide table-mode items: two workgroups per CU fit (LDS)
hipError_t launch_deposit_wide(const Plan& P, const DepArgs& D, int reduction, int cus, hipStream_t s) {
  DepArgs d2 = D;
  const int grid = std::max(cus, 1) * 2;
  d2.n_queues = std::min(kQueues, grid);
  return reduction == 0 ? wide_shape_launch<0>(P, d2, grid, s) : wide_shape_launch<1>(P, d2, grid, s);
}

bool tile_shape_supported(const int t[3]) {
  return (t[0] == 8 && t[1] == 8 && t[2] == 8) || (t[0] == 16 && t[1] == 8 && t[2] == 8) ||
         (t[0] == 16 && t[1] == 16 && t[2] == 8) || (t[0] == 16 && t[1] == 16 && t[2] == 16);
}

template <int RED>
static hipError_t combine_shape(const Plan& P, const DepArgs& D, int grid, hipStream_t s) {
  const int* t = P.tile;
  if (t[0] == 8 && t[1] == 8 && t[2] == 8) combine_tiles<RED, 8, 8, 8><<<grid, 256, 0, s>>>(P, D);
  else if (t[0] == 16 && t[1] == 8 && t[2] == 8) combine_tiles<RED, 16, 8, 8><<<grid, 256, 0, s>>>(P, D);
  else if (t[0] == 16 && t[1] == 16 && t[2] == 8) combine_tiles<RED, 16, 16, 8><<<grid, 256, 0, s>>>(P, D);
  else if (t[0] == 16 && t[1] == 16 && t[2] == 16) combine_tiles<RED, 16, 16, 16><<<grid, 256, 0, s>>>(P, D);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

long long exchange_cells(const int t[3]) { return (long long)(t[0] + 2) * (t[1] + 2) * (t[2] + 2); }

hipError_t launch_zero_split(const Plan& P, const DepArgs& D, int reduction, int cus, hipStream_t s) {
  const int words = (int)exchange_cells(P.tile) * (reduction == 0 ? 2 : 1);
  zero_split<<<std::max(1, std::min(P.ntiles, cus * 8)), 256, 0, s>>>(D, P.ntiles, words);
  return hipGetLastError();
}

hipError_t launch_combine(const Plan& P, const DepArgs& D, int reduction, int cus, hipStream_t s) {
  const int grid = std::max(1, std::min(P.ntiles, cus * 8));
  return reduction == 0 ? combine_shape<0>(P, D, grid, s) : combine_shape<1>(P, D, grid, s);
}

hipError_t launch_deposit(const Plan& P, const DepArgs& D, int reduction, int grid, int block, hipStream_t s) {
  const int* t = P.tile;
  if (t[0] == 8 && t[1] == 8 && t[2] == 8) narrow_tile<8, 8, 8>(P, D, reduction, grid, block, s);
  else if (t[0] == 16 && t[1] == 8 && t[2] == 8) narrow_tile<16, 8, 8>(P, D, reduction, grid, block, s);
  else if (t[0] == 16 && t[1] == 16 && t[2] == 8) narrow_tile<16, 16, 8>(P, D, reduction, grid, block, s);
  else if (t[0] == 16 && t[1] == 16 && t[2] == 16) narrow_tile<16, 16, 16>(P, D, reduction, grid, block, s);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_grid_sums(const Plan& P, const DepArgs& D, int reduction, double* grid_mass, hipStream_t s) {
  if (P.ngrids <= 0) return hipSuccess;
  if (reduction == 0) grid_sums<0><<<P.ngrids, 256, 0, s>>>(P, D, grid_mass);
  else grid_sums<1><<<P.ngrids, 256, 0, s>>>(P, D, grid_mass);
  return hipGetLastError();
}

hipError_t launch_begin_call(const DepArgs& D, const int tile[3], int reduction, long long n_narrow, long long n_wide,
                             unsigned* item_pairs, long long n_items, unsigned long long* cursor, long long nkeys,
                             const int* split_tiles, const unsigned* n_split, int cus, hipStream_t s) {
  const int words = (int)exchange_cells(tile) * (reduction == 0 ? 2 : 1);
  const long long want = (std::max(std::max(n_items, nkeys), (long long)(sizeof(Counters) / 4)) + 255) / 256;
  begin_call<<<(int)std::min<long long>(std::max<long long>(want, 64), (long long)std::max(cus, 1) * 8), 256, 0, s>>>(
      D, (unsigned)n_narrow, (unsigned)n_wide, item_pairs, n_items, cursor, nkeys, split_tiles, n_split, words);
  return hipGetLastError();
}

hipError_t launch_finish_call(const Plan& P, const DepArgs& D, int reduction, double* grid_mass,
                              const unsigned* item_pairs, long long n_items, long long nkeys, unsigned* host, int cus,
                              hipStream_t s) {
  const long long want = std::max((std::max(n_items, nkeys) + 1023) / 1024, grid_mass ? (P.ngrids + 3ll) / 4 : 1ll);
  const int grid = (int)std::min<long long>(std::max<long long>(want, 1), (long long)std::max(cus, 1) * 4);
  if (reduction == 0) finish_call<0><<<grid, 256, 0, s>>>(P, D, grid_mass, item_pairs, n_items, nkeys, host);
  else finish_call<1><<<grid, 256, 0, s>>>(P, D, grid_mass, item_pairs, n_items, nkeys, host);
  return hipGetLastError();
}

hipError_t launch_cell_keys(const Plan& P, const Parts& A, const KeyBits& B, unsigned* key, unsigned* idx,
                            float4* rec, Counters* C, int cus, hipStream_t s) {
  cell_keys<<<grid_for(A.n, 256, cus * 16), 256, 0, s>>>(P, A, B, key, idx, rec, C);
  return hipGetLastError();
}

hipError_t launch_adjoint(const Plan& P, const Parts& A, const float* g1, const float* g11, float* dm,
                          float* dx, float* dy, float* dz, const unsigned* order, float4* rec, int cus, hipStream_t s) {
  adjoint_gather<<<grid_for(A.n, 256, cus * 16), 256, 0, s>>>(P, A, g1, g11, dm, dx, dy, dz, order, rec);
  if (rec) adjoint_unpack<<<grid_for(A.n, 256, cus * 16), 256, 0, s>>>(A.n, rec, dm, dx, dy, dz);
  return hipGetLastError();
}

hipError_t launch_plain_zero(const Plan& P, float* u1, float* u11, hipStream_t s) {
  plain_zero<<<P.ngrids, 256, 0, s>>>(P, u1, u11);
  return hipGetLastError();
}
hipError_t launch_plain_base(const Plan& P, const Parts& A, float* u1, int cus, hipStream_t s) {
  const int grid = grid_for(A.n, 256, cus * 16);
  if (P.mode == 2) plain_base<2><<<grid, 256, 0, s>>>(P, A, u1);
  else plain_base<1><<<grid, 256, 0, s>>>(P, A, u1);
  return hipGetLastError();
}
hipError_t launch_plain_validate(const Plan& P, const Parts& A, Counters* C, int cus, hipStream_t s) {
  const int grid = grid_for(A.n, 256, cus * 16);
  if (P.mode == 2) plain_validate<2><<<grid, 256, 0, s>>>(P, A, C);
  else plain_validate<1><<<grid, 256, 0, s>>>(P, A, C);
  return hipGetLastError();
}
hipError_t launch_plain_flags(const Plan& P, const Parts& A, int l, unsigned* flag, int cus, hipStream_t s) {
  plain_level_flags<<<grid_for(A.n, 256, cus * 16), 256, 0, s>>>(P, A, l, flag);
  return hipGetLastError();
}
hipError_t launch_plain_compact(const unsigned* flag, const unsigned long long* start, long long n,
                                long long* idx, int cus, hipStream_t s) {
  plain_compact<<<grid_for(n, 256, cus * 16), 256, 0, s>>>(flag, start, n, idx);
  return hipGetLastError();
}
hipError_t launch_plain_patch(const Plan& P, const Parts& A, int g, const long long* idx,
                              const unsigned long long* nidx, long long nmax, float* u11, int cus,
                              hipStream_t s) {
  if (nmax <= 0) return hipSuccess;
  const int grid = grid_for(nmax, 256, cus * 8);
  if (P.mode == 2) plain_patch<2><<<grid, 256, 0, s>>>(P, A, g, idx, nidx, u11);
  else plain_patch<1><<<grid, 256, 0, s>>>(P, A, g, idx, nidx, u11);
  return hipGetLastError();
}
hipError_t launch_plain_finish(const Plan& P, float* u1, float* u11, double* grid_mass, hipStream_t s) {
  plain_finish<<<P.ngrids, 256, 0, s>>>(P, u1, u11, grid_mass);
  return hipGetLastError();
}

}  // namespace asohf
