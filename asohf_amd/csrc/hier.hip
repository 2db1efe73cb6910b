// hier.hip -- binning through the base grid and along the patch hierarchy
// (gfx950).
//
// The batched build bins each 27-cell (particle, grid) member into the tile
// that holds its centre cell (clamped into the grid); what its stencil spills
// over the tile's border is exchanged between tiles after the deposit.
// Instead of testing every particle against a hash of every level's patch
// boxes, the binning starts from the base-grid tiles:
//
//   bin_base      particles -> base-grid tile entries (16 B: x, y, z, m);
//                 every particle is a member of the base grid
//                 (grids.f:761-835, 1159-1246)
//   emit_tsc      TSC, one level at a time: the entries of a level-l tile are
//                 tested against the patch boxes of the tile's target
//                 list: the patches whose membership box lies inside this
//                 grid's box (found on the host in FP32, the values the
//                 device compares), so every member of such a patch is a
//                 member of this grid and has exactly one entry here.
//                 A member gets its entry in that patch, exactly as the
//                 reference's strict box test and index expressions give it
//                 (grids.f:1294-1323).
//   emit_table    kernel table: the base entries are tested against every
//                 patch whose membership box can hold a particle of the tile
//                 (grids.f:871-909); members whose box of 2N+1 cells meets the
//                 patch get their entries there.  (The boxes reach a base cell
//                 past the patch, so following the hierarchy would need
//                 entries for five times as many members as deposit.)
//
// Entries go to per-tile ranges whose capacities come from an exact count
// pass (the first call on a geometry, or after an overflow): every workgroup
// counts its emissions per tile in LDS, reserves each tile's range with one
// atomic add, and writes.  An emission that finds the LDS table or list full
// reserves its own slot directly.  A reservation past a tile's capacity sets
// the overflow flag (nothing is written past it) and the host rebuilds the
// capacities exactly.
#include <type_traits>

#include "dev.h"
#include "launch.h"

namespace asohf {

namespace {

constexpr int kHbThreads = 256;
constexpr int kHbPer = 2;                        // particles per thread
constexpr int kHbChunk = kHbThreads * kHbPer;    // particles per bin_base workgroup (< 2^16)
constexpr int kHbCap = 1024;                     // LDS key slots (power of two, < 2^16)
constexpr int kHbProbe = 32;
constexpr int kEmThreads = 256;
constexpr int kEmPer = 2;                        // entries per thread and round
constexpr int kEmRound = kEmPer * kEmThreads;    // entries per round
constexpr int kEmCap = 512;                      // LDS key slots of an item
constexpr int kEmWList = 384;                    // list words per wave and round
constexpr unsigned kEmSkip = ~0u;                // list word of an emission written directly
// a list word: the key's slot | position in the key's range of the round << 9 |
// entry of the round << 19 (an entry is in a patch's tile at most once, so a
// position is below kEmRound)
static_assert(kEmPer == 2 && kEmRound <= 512 && kEmCap <= 512, "the fields of a list word");
constexpr int kEmTargets = 32;                   // target records staged in LDS at once

__device__ __forceinline__ unsigned slot_hash(unsigned k, unsigned mask) {
  k ^= k >> 15;
  k *= 0x2c1b3c6du;
  k ^= k >> 12;
  k *= 0x297a2d39u;
  k ^= k >> 15;
  return k & mask;
}
// slot of key k in an LDS open-addressing table of CAP slots, inserting it
// when absent; -1 when the probe path is full
template <int CAP>
__device__ __forceinline__ int slot_insert(int* keys, int k) {
  unsigned h = slot_hash((unsigned)k, CAP - 1);
#pragma unroll 1
  for (int p = 0; p < kHbProbe; ++p) {
    const int cur = keys[h];
    if (cur == k) return (int)h;
    if (cur == -1) {
      const int old = atomicCAS(&keys[h], -1, k);
      if (old == -1 || old == k) return (int)h;
    }
    h = (h + 1) & (CAP - 1);
  }
  return -1;
}

__device__ __forceinline__ void set_overflow(Counters* C) {
  C->overflow = 1u;
  C->n_items_eff = 0u;   // the deposits of this call then do nothing
  C->n_wide_eff = 0u;
}

// one entry written at its own reserved slot (the path of an emission that
// found the LDS table or list full)
__device__ __forceinline__ void emit_direct(unsigned long long* cursor, const unsigned long long* start,
                                            int4* entries, Counters* C, int key, int4 e) {
  const unsigned long long p = atomicAdd(&cursor[key], 1ull);
  if (p < start[key + 1]) entries[p] = e;
  else set_overflow(C);
}

}  // namespace

// per-key capacity from an exact count: the count plus an eighth plus 32
// entries, so a later snapshot with a similar distribution fits
__global__ void __launch_bounds__(256) count_to_capacity(unsigned* cnt, long long nkeys) {
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < nkeys;
       k += (long long)gridDim.x * blockDim.x) {
    const unsigned c = cnt[k];
    cnt[k] = c == 0u ? 0u : c + (c >> 3) + 32u;
  }
}

// The position of an emission (key = destination tile key) in its key's range
// of the workgroup's round: the lane finds the key's table slot h and adds 1
// to its count, whose old value is the position.  Lanes of a wave with the
// same key meet at one LDS address, which the LDS serialises at less cost
// than grouping the lanes first (ballots and lane reads per group, measured
// slower with 1 to 8 groups).  h = -1 when the table is full (the emission is
// then not counted).
template <int CAP>
__device__ __forceinline__ int count_key(int* keys, unsigned* vals, int key, unsigned& at) {
  const int h = slot_insert<CAP>(keys, key);
  at = h >= 0 ? atomicAdd(&vals[h], 1u) : 0u;
  return h;
}

// a reserved range in one word: its first slot (below 2^40; the host rejects
// larger entry buffers) and, above it, how many of its slots lie within the
// key's capacity (all of them unless the reservation overflowed)
constexpr int kSlotBits = 40;
constexpr unsigned long long kSlotMask = (1ull << kSlotBits) - 1ull;

// one reservation per tile key of the round: base[k] = the key's first slot
// and its room
template <int CAP, int NTHR>
__device__ __forceinline__ void reserve_round(const int* keys, unsigned* vals, unsigned long long* base,
                                              unsigned long long* cursor, const unsigned long long* start,
                                              Counters* C) {
  for (int k = threadIdx.x; k < CAP; k += NTHR) {
    const int key = keys[k];
    const unsigned v = vals[k];
    if (key >= 0 && v) {
      const unsigned long long b0 = atomicAdd(&cursor[key], (unsigned long long)v);
      const unsigned long long lim = start[key + 1];
      const unsigned long long room = b0 >= lim ? 0ull : (lim - b0 < v ? lim - b0 : (unsigned long long)v);
      base[k] = (b0 & kSlotMask) | (room << kSlotBits);   // room 0 when b0 is past the capacity
      if (b0 + v > lim) set_overflow(C);
    }
    vals[k] = 0u;
  }
}

// the slot of position `at` of a reserved range, or -1 past the key's capacity
__device__ __forceinline__ long long reserved_slot(unsigned long long b, unsigned at) {
  return at < (unsigned)(b >> kSlotBits) ? (long long)((b & kSlotMask) + at) : -1ll;
}

// Base-grid binning, persistent: each workgroup takes chunks of kHbChunk
// particles (kHbPer per thread) in turn and loads its next chunk while it
// bins this one.  Each valid particle (finite, mass >= 0, within the range the
// mode accepts) has one entry, in the tile of its clamped (TSC) or wrapped
// (table) cell.  Every lane counts its particles' keys in the workgroup's LDS
// table (a position in the key's range of the workgroup), one global add per
// key reserves the ranges, and every lane writes its particles from registers.
// Table mode also writes each entry's species; a particle outside the box,
// whose tile is a periodic image, gets kSpOutside and goes to the outside
// list.  Per-chunk partials: base members and the largest mass.
// Bound by latency (LDS counting, then one round of global reservations per
// chunk).  One entry per particle instead of one per tile its stencil touches
// needs no emission list, so twice the workgroups fit a CU and a third fewer
// entries are written: 16.8M particles on 256^3 cells (16x8x8 tiles) 1,431 ->
// 356 us, 134M particles 6.57 -> 2.11 ms.
template <int MODE>
__global__ void __launch_bounds__(kHbThreads, 7) bin_base(Plan P, Parts A, unsigned long long* cursor,
                                                       const unsigned long long* start, int4* entries,
                                                       Counters* C, BlockTables BT, TableBin TB) {
  __shared__ int keys[kHbCap];
  __shared__ unsigned vals[kHbCap];
  __shared__ unsigned long long base[kHbCap];
  __shared__ unsigned long long s_valid[kHbThreads / 64];
  __shared__ float s_mmax[kHbThreads / 64];
  const int tid = threadIdx.x;
  const GridDesc& B = P.grids[0];
  const int bn[3] = {B.n[0], B.n[1], B.n[2]};
  const float bd[3] = {B.d[0], B.d[1], B.d[2]};
  const float bid[3] = {B.inv_d[0], B.inv_d[1], B.inv_d[2]};
  const int bnt0 = B.nt[0], bnt1 = B.nt[1];
  const long long nchunks = (A.n + kHbChunk - 1) / kHbChunk;
  // the workgroup's next chunk of particles, loaded while this one is binned
  float fx[kHbPer], fy[kHbPer], fz[kHbPer], fm[kHbPer];
  auto fetch = [&](long long cc) {
#pragma unroll
    for (int r = 0; r < kHbPer; ++r) {
      const long long i = cc * kHbChunk + r * kHbThreads + tid;
      fx[r] = fy[r] = fz[r] = fm[r] = 0.f;
      if (cc < nchunks && i < A.n) { fx[r] = A.x[i]; fy[r] = A.y[i]; fz[r] = A.z[i]; fm[r] = A.m[i]; }
    }
  };
  fetch(blockIdx.x);
  for (long long chunk = blockIdx.x; chunk < nchunks; chunk += gridDim.x) {
    const long long c0 = chunk * kHbChunk;
    float px[kHbPer], py[kHbPer], pz[kHbPer], pm[kHbPer];
    int slot[kHbPer];       // the key's table slot, -1: no entry to write
    unsigned at[kHbPer];    // the position in the key's range
    int sp[kHbPer];         // table mode: the particle's species
#pragma unroll
    for (int r = 0; r < kHbPer; ++r) { px[r] = fx[r]; py[r] = fy[r]; pz[r] = fz[r]; pm[r] = fm[r]; }
    fetch(chunk + gridDim.x);
    for (int k = tid; k < kHbCap; k += kHbThreads) { keys[k] = -1; vals[k] = 0u; }
    __syncthreads();
    unsigned err = 0;
    unsigned long long valid = 0;
    float mmax = 0.f;
    // the particles are ordered by species: most chunks hold one
    const int sp_lo = MODE == 1 ? species_of(A, c0) : 0;
    const int sp_hi = MODE == 1 ? species_of(A, min(c0 + kHbChunk, A.n) - 1) : 0;
#pragma unroll
    for (int r = 0; r < kHbPer; ++r) {
      const int k = r * kHbThreads + tid;
      bool ok = c0 + k < A.n;
      const float x = px[r], y = py[r], z = pz[r], m = pm[r];
      if (ok && !(isfinite(x) && isfinite(y) && isfinite(z) && isfinite(m))) { err |= kErrNonFinite; ok = false; }
      if (ok && m < 0.f) { err |= kErrNegMass; ok = false; }
      slot[r] = -1;
      at[r] = 0u;
      sp[r] = 0;
      int c[3];   // the cell whose tile takes the entry
      if (MODE == 2) {
        if (ok && !(tsc_base_in_range(x, P.xl, bid[0], bn[0]) && tsc_base_in_range(y, P.xl, bid[1], bn[1]) &&
                    tsc_base_in_range(z, P.xl, bid[2], bn[2]))) {
          err |= kErrWrap;
          ok = false;
        }
        if (ok) {
          c[0] = tsc_base_index(x, P.xl, bd[0], bid[0], bn[0]);
          c[1] = tsc_base_index(y, P.xl, bd[1], bid[1], bn[1]);
          c[2] = tsc_base_index(z, P.xl, bd[2], bid[2], bn[2]);
        }
      } else if (ok) {
        const float t[3] = {index_quotient(x - P.xl, bd[0], bid[0]), index_quotient(y - P.xl, bd[1], bid[1]),
                            index_quotient(z - P.xl, bd[2], bid[2])};
        sp[r] = sp_lo == sp_hi ? sp_lo : species_of(A, c0 + k);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          ok = ok && t[a] > -1.0e9f && t[a] < 1.0e9f;
          const int i = ok ? (int)t[a] + 1 : 1;
          ok = ok && i >= 2 - bn[a] && i <= 2 * bn[a] - 1;   // the single wrap must land in 1..N
          if (t[a] < 0.f || i > bn[a]) sp[r] = kSpOutside;
          c[a] = wrap1(i, bn[a]);
        }
        if (!ok) err |= kErrWrap;
        else if (sp[r] == kSpOutside) {
          const unsigned o = atomicAdd(&C->n_outside, 1u);
          if (o < TB.outside_cap) TB.outside[o] = (unsigned)(c0 + k);
          else set_overflow(C);
        }
      }
      if (ok) {
        ++valid;
        mmax = fmaxf(mmax, m);
        const int tx = (c[0] - 1) >> P.tshift[0], ty = (c[1] - 1) >> P.tshift[1], tz = (c[2] - 1) >> P.tshift[2];
        const int key = 2 * ((tz * bnt1 + ty) * bnt0 + tx);
        slot[r] = count_key<kHbCap>(keys, vals, key, at[r]);
        if (slot[r] < 0) {
          const unsigned long long p = atomicAdd(&cursor[key], 1ull);
          if (p < start[key + 1]) {
            entries[p] = make_int4(__float_as_int(x), __float_as_int(y), __float_as_int(z), __float_as_int(m));
            if (MODE == 1) TB.species[p] = (unsigned char)sp[r];
          } else {
            set_overflow(C);
          }
        }
      }
    }
    __syncthreads();
    reserve_round<kHbCap, kHbThreads>(keys, vals, base, cursor, start, C);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kHbPer; ++r) {
      if (slot[r] < 0) continue;
      const long long pos = reserved_slot(base[slot[r]], at[r]);
      if (pos >= 0) {
        entries[pos] = make_int4(__float_as_int(px[r]), __float_as_int(py[r]), __float_as_int(pz[r]),
                                 __float_as_int(pm[r]));
        if (MODE == 1) TB.species[pos] = (unsigned char)sp[r];
      }
    }
    // per-workgroup partials (members of the base grid, largest mass)
    valid = wave_sum(valid);
    mmax = wave_max(mmax);
    err = wave_or(err);
    if ((tid & 63) == 0) {
      s_valid[tid >> 6] = valid;
      s_mmax[tid >> 6] = mmax;
      if (err) atomicOr(&C->err, err);
    }
    __syncthreads();
    if (tid == 0) {
      unsigned long long p = 0;
      float mm = 0.f;
      for (int w = 0; w < kHbThreads / 64; ++w) { p += s_valid[w]; mm = fmaxf(mm, s_mmax[w]); }
      BT.pairs[chunk] = p;
      BT.mmax[chunk] = __float_as_uint(mm);
    }
    __syncthreads();   // the chunk's writes read base; its partials s_valid
  }
}

// The emission pass of one level: items [item_lo, item_hi) are the work items
// (chunks of one tile's entry range) of the level's tiles, each in `pieces`
// pieces of plen entries where there are fewer items than workgroups fit.  A
// workgroup takes `batch` consecutive pieces at a time from the level's queue
// counter and works through those whose tile has targets (the others' member
// counts stay 0).  Per piece the target records are staged in LDS (kEmTargets
// at a time); the piece's entries are taken kEmPer per thread per round (one
// per round where overlapping patches make the lists long), loaded a round
// ahead and kept in LDS.  In a round every wave tests its entries against the
// targets and collects the members; 64 of them at a time, one per lane, get
// their tile in the patch, a position in the tile key's range of the round and
// a word in the wave's list; one global add per key reserves the round's ranges
// and every wave writes its listed entries from LDS.
// Bound by latency (the waves wait 80 percent of their time, VALU 35 percent
// busy): the reservation's round trip and the barriers of a round.  With one
// entry per member instead of one per tile, rounds loaded ahead, and entries
// written from LDS instead of read again: 256^3 particles, 4 levels 1,111 ->
// 762 -> 704 us; 512^3, 6 levels 9.23 -> 6.06 -> 5.52 ms.  Six workgroups per CU
// (48 bytes a lane spilled) take 705 us and 5.30 ms, but 158 instead of 138 us
// on 2.1M particles.  Pieces: 13,824 particles, 3 levels 75 -> 25 us.
__global__ void __launch_bounds__(kEmThreads, 5) emit_tsc(Plan P, const Item* items, long long item_lo,
                                                       long long n_pieces, int pieces, int plen, int level,
                                                       int batch, unsigned long long* cursor,
                                                       const unsigned long long* start, int4* entries,
                                                       unsigned* item_pairs, Counters* C) {
  __shared__ int keys[kEmCap];
  __shared__ unsigned vals[kEmCap];
  __shared__ unsigned long long base[kEmCap];
  __shared__ unsigned wlist_all[(kEmThreads / 64) * kEmWList];
  __shared__ int4 stage[kEmRound];   // the round's entries; a wave reads its own
  __shared__ unsigned mlist_all[(kEmThreads / 64) * 128];
  __shared__ BoxRec recs[kEmTargets];
  __shared__ long long s_i0;
  __shared__ unsigned s_red[kEmThreads / 64];
  __shared__ int s_nwmax[2];   // the waves' longest list of a round, by round parity
  const int tid = threadIdx.x, lane = (int)__lane_id();
  unsigned* wl = wlist_all + (tid >> 6) * kEmWList;
  // wave-steps per round: kEmPer, or 1 after a round whose lists would have
  // overflowed with kEmPer (members of overlapping patches emit several
  // entries each); kept from one item to the next
  int steps = kEmPer;
  unsigned* ml = mlist_all + (tid >> 6) * 128;
  unsigned* queue = &C->equeue[level * kLine];
  for (;;) {
    if (tid == 0) s_i0 = (long long)atomicAdd(queue, (unsigned)batch);
    __syncthreads();
    const long long i0 = s_i0;
    __syncthreads();   // every wave has read s_i0 before thread 0 takes the next batch
    if (i0 >= n_pieces) break;
    const int nb = (int)min((long long)batch, n_pieces - i0);
    for (int bi = 0; bi < nb; ++bi) {
      const long long ii = item_lo + (i0 + bi) / pieces;
      const Item it = items[ii];
      const int t = it.tile;
      const unsigned q0 = P.tgt_off[t], q1 = P.tgt_off[t + 1];
      if (q0 == q1) continue;
      // the piece's filled entries
      const long long e0 = it.begin + (i0 + bi) % pieces * plen;
      const long long e1 = min(min(it.end, e0 + plen), (long long)cursor[2 * t]);
      if (e1 <= e0) continue;
      for (int k = tid; k < kEmCap; k += kEmThreads) { keys[k] = -1; vals[k] = 0u; }
      if (tid < 2) s_nwmax[tid] = 0;
      int par = 0;
      unsigned pairs = 0;
      for (unsigned q = q0; q < q1; q += kEmTargets) {
        const int nq = (int)min((unsigned)kEmTargets, q1 - q);
        for (int k = tid; k < nq * 8; k += kEmThreads)
          reinterpret_cast<int4*>(recs)[k] = reinterpret_cast<const int4*>(P.grec + P.tgt[q + (k >> 3)])[k & 7];
        __syncthreads();
        // the next round's entries, on their way while this one is worked through
        int4 nxt0, nxt1;
        auto fetch = [&](long long r) {
          nxt0 = entries[min(r + tid, e1 - 1)];
          nxt1 = entries[min(r + kEmThreads + tid, e1 - 1)];
        };
        fetch(e0);
        for (long long r0 = e0, rn = 0; r0 < e1; r0 += rn) {
          const int nsteps = steps;
          rn = (long long)nsteps * kEmThreads;
          const int4 cur0 = nxt0, cur1 = nxt1;
          fetch(r0 + rn);
          // ---- list the wave's member emissions
          int nw = 0;   // the wave's list length (uniform)
#pragma unroll 1
          for (int i = 0; i < nsteps; ++i) {
            const int k = i * kEmThreads + tid;
            const bool ok = r0 + k < e1;
            const int4 v = i == 0 ? cur0 : cur1;
            stage[k] = v;
            const float p[3] = {__int_as_float(v.x), __int_as_float(v.y), __int_as_float(v.z)};
            // the item's targets, one per pass: the box tests, with the
            // members listed (lane, target) in the wave's member list; every
            // 64 listed members, and at the end, the wave works through them
            // one per lane
            int nm = 0;   // the member list's length (uniform)
            auto members = [&](int n) {
              const int src = (int)(ml[lane < n ? lane : 0] & 63u);
              const int j = (int)(ml[lane < n ? lane : 0] >> 8);
              const int4 u = make_int4(__shfl(v.x, src), __shfl(v.y, src), __shfl(v.z, src), __shfl(v.w, src));
              const float q[3] = {__int_as_float(u.x), __int_as_float(u.y), __int_as_float(u.z)};
              const BoxRec& R = recs[j];
              bool mem = lane < n;
              int tc[3] = {0, 0, 0};
              if (mem) {
                ++pairs;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                  const int ci = (int)index_quotient(q[a] - R.org[a], R.d[a], R.inv_d[a]);
                  // a member whose quotient rounds onto the far face of the
                  // box (ci = N + 2) has no stencil cell in the patch
                  mem = mem && ci <= R.n[a] + 1;
                  tc[a] = (clampi(ci, 1, R.n[a]) - 1) >> P.tshift[a];
                }
              }
              const unsigned long long mb = __ballot(mem);
              const int off = nw + __popcll(mb & ((1ull << lane) - 1ull));
              if (mem) {
                const int ks = i * kEmThreads + (tid & ~63) + src;
                const int key = 2 * (R.tile0 + (tc[2] * R.nt1 + tc[1]) * R.nt0 + tc[0]);
                unsigned at = 0;
                const int h = off < kEmWList ? count_key<kEmCap>(keys, vals, key, at) : -1;
                if (h < 0) emit_direct(cursor, start, entries, C, key, u);
                if (off < kEmWList)
                  wl[off] = h < 0 ? kEmSkip : ((unsigned)ks << 19) | (at << 9) | (unsigned)h;
              }
              nw = min(nw + __popcll(mb), kEmWList);
            };
            for (int j = 0; j < nq; ++j) {
              const bool mem = ok && in_box(recs[j], p[0], p[1], p[2]);
              const unsigned long long mb = __ballot(mem);
              if (mem) ml[nm + __popcll(mb & ((1ull << lane) - 1ull))] = (unsigned)lane | ((unsigned)j << 8);
              nm += __popcll(mb);
              if (nm >= 64) {
                members(64);
                nm -= 64;
                if (lane < nm) ml[lane] = ml[64 + lane];
              }
            }
            if (nm > 0) members(nm);
          }
          if (lane == 0) atomicMax(&s_nwmax[par], nw);
          if (tid == 0) s_nwmax[par ^ 1] = 0;   // the next round's, before this barrier
          __syncthreads();
          {
            const int mx = s_nwmax[par];
            steps = (mx * kEmPer > nsteps * (kEmWList * 3 / 4)) ? 1 : kEmPer;
            par ^= 1;
          }
          reserve_round<kEmCap, kEmThreads>(keys, vals, base, cursor, start, C);
          __syncthreads();
          // ---- write the listed entries
          for (int idx = lane; idx < nw; idx += 64) {
            const unsigned w = wl[idx];
            if (w == kEmSkip) continue;
            const long long pos = reserved_slot(base[w & 0x1ffu], (w >> 9) & 0x3ffu);
            if (pos >= 0) entries[pos] = stage[w >> 19];
          }
        }
      }
      // members found in this piece
      const unsigned sw = wave_sum(pairs);
      if ((tid & 63) == 0) s_red[tid >> 6] = sw;
      __syncthreads();
      if (tid == 0) {
        unsigned tot = 0;
        for (int w = 0; w < kEmThreads / 64; ++w) tot += s_red[w];
        if (tot) atomicAdd(&item_pairs[ii], tot);
      }
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
// kernel-table emission
// ---------------------------------------------------------------------------
constexpr int kEtThreads = 256;
constexpr int kEtPiece = 1024;     // entries of a work unit (a collected member keeps 10 bits of it)
constexpr int kEtRows = kEtPiece / kEtThreads;   // rows of 64 entries per wave
constexpr int kEtTargets = 32;     // target records staged in LDS at once
constexpr int kEtCap = 1024;       // LDS key slots
constexpr int kEtWList = 128;      // emissions a wave lists before it works through them
constexpr int kEtPend = 128;       // members a wave collects before it works through them
constexpr unsigned long long kEtFull = ~0ull;   // a key's reservation past its capacity

// A target patch in LDS, for its members: the cell and tile fields (padded so
// that the records of several targets start in different banks).
struct EtTarget {
  float org[3], d[3], inv_d[3];
  int n[3], level, tile0, nt0, nt1, pad[4];
};
static_assert(sizeof(EtTarget) == 80, "16-byte LDS reads");

// slot of key k in the table, -1 when it is not there (slot_insert found its
// probe path full)
template <int CAP>
__device__ __forceinline__ int slot_find(const int* keys, int k) {
  unsigned h = slot_hash((unsigned)k, CAP - 1);
#pragma unroll 1
  for (int p = 0; p < kHbProbe; ++p) {
    const int cur = keys[h];
    if (cur == k) return (int)h;
    if (cur == -1) return -1;
    h = (h + 1) & (CAP - 1);
  }
  return -1;
}

__device__ __forceinline__ float readlanef(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ unsigned long long readlane64(unsigned long long v, int lane) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), lane);
  return ((unsigned long long)hi << 32) | lo;
}

// exclusive prefix over the wave's lanes of v >= 0, and the total
__device__ __forceinline__ int wave_exclusive(int v, int& total) {
  int s = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(s, o, 64);
    if ((int)__lane_id() >= o) s += t;
  }
  total = __shfl(s, 63, 64);
  return s - v;
}

// The kernel-table members of every patch from the base-grid entries.  A work
// unit is kEtPiece entries of a base tile's work item; workgroups take units
// from the list in turn, the next one's number on its way while this one is
// worked through; up to kEtTargets target patches at a time are worked through
// in three steps over the unit's entries:
//   test   every wave holds its kEtRows rows of entries in registers, and the
//          targets' boxes one per lane: a target's box is read from its lane
//          into scalars once for all rows.  Members are counted (the
//          reference's strict box); those whose 2N+1 cells can meet the patch
//          (the distance to the patch against N cells) are kept as a bit mask
//   count  the emissions of the masks' members are added up per tile key in the
//          LDS table: one for the tile of the centre cell where N = 1, one per
//          tile the clipped box touches otherwise
//   write  after one global add per key reserved the unit's ranges, the same
//          members again, every emission written at the next slot of its key's
//          range
// The last two collect members over the wave's entries and work through 64 at
// a time, one per lane (their entries read again), and spread the emissions of
// wide members densely over the lanes.
// Bound by VALU work (54 targets per entry at 512^3, 4.1 members, 1.8 tiles
// each).  With the boxes read from LDS for every row, and the tests inside the
// count: 512^3, 6 levels 20.7 -> 16.7 ms (2.2 of them the box tests); 256^3, 4
// levels 788 -> 640 us; 128^3, 3 levels 69 us either way.  Five workgroups per
// CU spill 48 bytes a lane; with four and no spill 18.8 ms, 684 and 78 us, with
// six 16.0 ms, 676 and 78 us.  The count and scatter passes over the patch hash
// that this replaced, against this and bin_base<1>: 70.1 -> 19.2 ms; 2,235 ->
// 1,040 us; 175 -> 127 us.  A slot per tile of the staged targets instead of
// the hash table took 36 ms: the tiles of a few targets fill the slots.  One pass that listed the emissions for a reservation per
// round of 256 entries took 35.6 ms, and 97 ms with lists short enough for six
// workgroups per CU: what overflowed them reserved one by one.
__global__ void __launch_bounds__(kEtThreads, 5) emit_table(Plan P, const Item* items, const unsigned long long* units,
                                                         unsigned long long* cursor, const unsigned long long* start,
                                                         int4* entries, unsigned* item_pairs, Counters* C,
                                                         TableBin TB) {
  __shared__ int keys[kEtCap];
  __shared__ unsigned long long slots[kEtCap];   // emissions of a key, then its next slot
  __shared__ unsigned long long mask[kEtPiece / 64][kEtTargets];
  __shared__ unsigned long long wlist_all[(kEtThreads / 64) * kEtWList];   // key | member's lane << 32
  __shared__ unsigned pend_all[(kEtThreads / 64) * kEtPend];               // entry of the unit | target << 10
  __shared__ EtTarget targets[kEtTargets];
  __shared__ unsigned s_next;
  const int tid = threadIdx.x, lane = (int)__lane_id();
  unsigned long long* wl = wlist_all + (tid >> 6) * kEtWList;
  unsigned* pd = pend_all + (tid >> 6) * kEtPend;
  const float dx = P.grids[0].d[0];
  const unsigned n_units = C->n_units;
  unsigned unit = blockIdx.x;
  while (unit < n_units) {
    // the next unit's number, read at the end of this one
    unsigned next = 0;
    if (tid == 0) next = gridDim.x + atomicAdd(&C->equeue[0], 1u);
    const unsigned long long u = units[unit];
    const long long ii = (long long)(u >> 32);
    const Item it = items[ii];
    const int t = it.tile;
    const unsigned q0 = P.tgt_off[t], q1 = P.tgt_off[t + 1];
    const long long e0 = it.begin + (long long)(unsigned)u * kEtPiece;
    const int ne = (int)(min(min(it.end, e0 + kEtPiece), (long long)cursor[2 * t]) - e0);
    const int4* const ent = entries + e0;
    const unsigned char* const spc = TB.species + e0;
    unsigned pairs = 0;   // the wave's members (uniform)
    for (unsigned q = q0; q < q1; q += kEtTargets) {
      const int nq = (int)min((unsigned)kEtTargets, q1 - q);
      for (int k = tid; k < kEtCap; k += kEtThreads) { keys[k] = -1; slots[k] = 0ull; }
      {
        // every wave holds the targets' boxes, one per lane, and tests its rows
        // of entries against one target at a time
        const BoxRec& R = P.grec[P.tgt[q + min(lane, nq - 1)]];
        const float dm = fmaxf(R.d[0], fmaxf(R.d[1], R.d[2]));
        float blo[3], bhi[3], borg[3], bnd[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          blo[a] = R.lo[a];
          bhi[a] = R.hi[a];
          borg[a] = R.org[a];
          bnd[a] = (float)R.n[a] * R.d[a];
        }
        const float bdl = 1.015625f * dm, bratio = dm / R.d[0];
        if (tid < nq) {
          EtTarget& T = targets[tid];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            T.org[a] = R.org[a];
            T.d[a] = R.d[a];
            T.inv_d[a] = R.inv_d[a];
            T.n[a] = R.n[a];
          }
          T.level = R.level;
          T.tile0 = R.tile0;
          T.nt0 = R.nt0;
          T.nt1 = R.nt1;
        }
        float p[kEtRows][3], reach[kEtRows];
#pragma unroll
        for (int i = 0; i < kEtRows; ++i) {
          const int k = 64 * (i * (kEtThreads / 64) + (tid >> 6)) + lane;
          const int4 v = ent[min(k, ne - 1)];
          const int sp = k < ne ? (int)spc[k] : kSpOutside;
          // NaN is in no box: past the end, and a particle outside the box,
          // which is enumerated by itself
          p[i][0] = sp != kSpOutside ? __int_as_float(v.x) : __int_as_float(0x7fc00000);
          p[i][1] = __int_as_float(v.y);
          p[i][2] = __int_as_float(v.z);
          reach[i] = ldexpf(dx, -sp);   // N cells of any level >= the species
          if (lane < nq) mask[i * (kEtThreads / 64) + (tid >> 6)][lane] = 0ull;
        }
#pragma unroll 1
        for (int j = 0; j < nq; ++j) {
          const float l0 = readlanef(blo[0], j), l1 = readlanef(blo[1], j), l2 = readlanef(blo[2], j);
          const float h0 = readlanef(bhi[0], j), h1 = readlanef(bhi[1], j), h2 = readlanef(bhi[2], j);
          unsigned long long mb[kEtRows], any = 0;
#pragma unroll
          for (int i = 0; i < kEtRows; ++i) {
            mb[i] = __ballot(l0 < p[i][0]) & __ballot(p[i][0] < h0) & __ballot(l1 < p[i][1]) &
                    __ballot(p[i][1] < h1) & __ballot(l2 < p[i][2]) & __ballot(p[i][2] < h2);
            any |= mb[i];
          }
          if (!any) continue;
          // distance past the patch's cells [org, org + n d] against N cells
          // (at least one); 1/64 of a cell of slack covers the rounding of the
          // cell index (16,512 cells of 2^-22) and of this test
          const float o0 = readlanef(borg[0], j), o1 = readlanef(borg[1], j), o2 = readlanef(borg[2], j);
          const float n0 = readlanef(bnd[0], j), n1 = readlanef(bnd[1], j), n2 = readlanef(bnd[2], j);
          const float dl = readlanef(bdl, j), ratio = readlanef(bratio, j);
#pragma unroll
          for (int i = 0; i < kEtRows; ++i) {
            if (!mb[i]) continue;
            pairs += (unsigned)__popcll(mb[i]);
            const float lim = fmaxf(reach[i] * ratio + dl * 0.015625f, dl);
            const float f0 = p[i][0] - o0, f1 = p[i][1] - o1, f2 = p[i][2] - o2;
            const float far = fmaxf(fmaxf(fmaxf(-f0, f0 - n0), fmaxf(-f1, f1 - n1)), fmaxf(-f2, f2 - n2));
            const unsigned long long tb = mb[i] & __ballot(far <= lim);
            if (lane == j) mask[i * (kEtThreads / 64) + (tid >> 6)][j] = tb;
          }
        }
      }
      __syncthreads();
      auto work = [&](auto pass_c) {
        constexpr int pass = decltype(pass_c)::value;
        int np = 0;
        // the first n collected members, one per lane
        auto members = [&](int n) {
          const unsigned w = pd[lane < n ? lane : 0];
          const int src = (int)(w & (kEtPiece - 1));
          const EtTarget& R = targets[w >> 10];
          const int4 u = ent[src];
          const int su = (int)spc[src];
          const float x[3] = {__int_as_float(u.x), __int_as_float(u.y), __int_as_float(u.z)};
          bool mem = lane < n;
          const int irk = max(R.level - su, 0), nk = 1 << irk;
          int ci[3], lo[3], ext[3] = {1, 1, 1};
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            ci[a] = (int)floorf(index_quotient(x[a] - R.org[a], R.d[a], R.inv_d[a])) + 1;
            const int c0 = max(ci[a] - nk, 1), c1 = min(ci[a] + nk, R.n[a]);
            mem = mem && c0 <= c1;
            if (irk == 0) {
              lo[a] = (clampi(ci[a], 1, R.n[a]) - 1) >> P.tshift[a];
            } else {
              lo[a] = (c0 - 1) >> P.tshift[a];
              ext[a] = ((c1 - 1) >> P.tshift[a]) - lo[a] + 1;
            }
          }
          const int4 pe = pack_table(ci[0], ci[1], ci[2], irk, __int_as_float(u.w));
          auto emit = [&](bool want, int key, const int4& q4) {
            if (!want) return;
            if (pass == 0) {
              const int h = slot_insert<kEtCap>(keys, key);
              if (h >= 0) atomicAdd(&slots[h], 1ull);
            } else {
              const int h = slot_find<kEtCap>(keys, key);
              if (h < 0) {
                emit_direct(cursor, start, entries, C, key, q4);
              } else if (slots[h] != kEtFull) {   // (a full key's slots never change in this pass)
                entries[atomicAdd(&slots[h], 1ull)] = q4;
              }
            }
          };
          const int nt = mem ? ext[0] * ext[1] * ext[2] : 0;
          int key = 2 * (R.tile0 + (lo[2] * R.nt1 + lo[1]) * R.nt0 + lo[0]) + (irk > 0 ? 1 : 0);
          if (!__ballot(nt > 1)) {
            emit(nt > 0, key, pe);
            return;
          }
          int tot;
          const int off = wave_exclusive(nt, tot);
          int c = 0, cx = 0, cy = 0, row = key, plane = key;
          for (int w0 = 0; w0 < tot; w0 += kEtWList) {
            for (; c < nt && off + c < w0 + kEtWList; ++c) {
              wl[off + c - w0] = (unsigned long long)(unsigned)key | ((unsigned long long)lane << 32);
              key += 2;
              if (++cx == ext[0]) {
                cx = 0;
                row += 2 * R.nt0;
                if (++cy == ext[1]) {
                  cy = 0;
                  plane += 2 * R.nt0 * R.nt1;
                  row = plane;
                }
                key = row;
              }
            }
            const int len = min(tot - w0, kEtWList);
            for (int b0 = 0; b0 < len; b0 += 64) {
              const bool want = b0 + lane < len;
              const unsigned long long word = wl[want ? b0 + lane : 0];
              const int from = (int)(word >> 32);
              int4 q4 = make_int4(0, 0, 0, 0);
              if (pass == 1) q4 = make_int4(__shfl(pe.x, from), __shfl(pe.y, from), __shfl(pe.z, from), 0);
              emit(want, (int)(unsigned)word, q4);
            }
          }
        };
#pragma unroll 1
        for (int r = tid >> 6; 64 * r < ne; r += kEtThreads / 64) {
          const unsigned long long mine = lane < nq ? mask[r][lane] : 0ull;
          for (unsigned long long js = __ballot(mine != 0ull); js; js &= js - 1) {
            const int j = __ffsll((long long)js) - 1;
            const unsigned long long tb = readlane64(mine, j);
            if ((tb >> lane) & 1ull)
              pd[np + __popcll(tb & ((1ull << lane) - 1ull))] = (unsigned)(64 * r + lane) | ((unsigned)j << 10);
            np += __popcll(tb);
            if (np >= 64) {
              members(64);
              np -= 64;
              if (lane < np) pd[lane] = pd[64 + lane];
            }
          }
        }
        if (np > 0) members(np);
      };
      work(std::integral_constant<int, 0>());
      __syncthreads();
      for (int k = tid; k < kEtCap; k += kEtThreads) {
        const int key = keys[k];
        const unsigned long long v = slots[k];
        if (key >= 0 && v) {
          const unsigned long long b0 = atomicAdd(&cursor[key], v);
          slots[k] = b0;
          if (b0 + v > start[key + 1]) {   // past the capacity: nothing is written, the call is redone
            slots[k] = kEtFull;
            set_overflow(C);
          }
        }
      }
      __syncthreads();
      work(std::integral_constant<int, 1>());
      __syncthreads();   // the next batch stages its targets and clears the table
    }
    if (lane == 0 && pairs) atomicAdd(&item_pairs[ii], pairs);
    if (tid == 0) s_next = next;
    __syncthreads();
    unit = s_next;
    __syncthreads();   // every wave has read s_next
  }
}

// Between the base binning and the emission: the call's base members and
// largest mass from the per-chunk partials (as reduce_blocks folds them), and
// in table mode the emission's work units, (item << 32 | piece) for every piece
// of kEtPiece filled entries of the items of tiles with targets, and the
// particles outside the box [-L/2, L/2), whose base tile is a periodic image, so
// that its target list says nothing about them: one thread each walks the patch
// hash and reserves its entries one by one.
template <int MODE>
__global__ void __launch_bounds__(256) after_bin(Plan P, Parts A, BlockTables BT, long long nblk, const Item* items,
                                                 long long n_items, unsigned long long* cursor,
                                                 const unsigned long long* start, int4* entries, Counters* C,
                                                 TableBin TB) {
  __shared__ unsigned long long sp[4];
  __shared__ float sm[4];
  stamp(C, kClkBinned);
  const long long i0 = blockIdx.x * (long long)blockDim.x + threadIdx.x, di = (long long)gridDim.x * blockDim.x;
  unsigned long long p = 0;
  float mm = 0.f;
  for (long long b = i0; b < nblk; b += di) {
    p += BT.pairs[b];
    mm = fmaxf(mm, __uint_as_float(BT.mmax[b]));
  }
  if (MODE == 1 && P.nl > 0) {
    for (long long k0 = i0 - __lane_id(); k0 < n_items; k0 += di) {
      const long long ii = k0 + __lane_id();
      int n = 0;
      if (ii < n_items) {
        const Item it = items[ii];
        if (P.tgt_off[it.tile] < P.tgt_off[it.tile + 1]) {
          const long long len = min(it.end, (long long)cursor[2 * it.tile]) - it.begin;
          n = len > 0 ? (int)((len + kEtPiece - 1) / kEtPiece) : 0;
        }
      }
      int tot;
      const int off = wave_exclusive(n, tot);
      unsigned b0 = 0;
      if (__lane_id() == 0 && tot) b0 = atomicAdd(&C->n_units, (unsigned)tot);
      b0 = __builtin_amdgcn_readfirstlane(b0);
      for (int k = 0; k < n; ++k) TB.units[b0 + off + k] = ((unsigned long long)ii << 32) | (unsigned)k;
    }
    const unsigned n = min(C->n_outside, TB.outside_cap);
    unsigned err = 0;
    for (long long k = i0; k < n; k += di) {
      const long long i = (long long)TB.outside[k];
      enumerate_particle<1>(
          P, i, A.x[i], A.y[i], A.z[i], A.m[i], species_of(A, i),
          [&](int g, int t, int wide, int4 e) {
            if (g > 0) emit_direct(cursor, start, entries, C, 2 * t + wide, e);   // the base entry is binned
          },
          [&](int g, int, int, int) { p += g > 0 ? 1 : 0; }, err);
    }
  }
  p = wave_sum(p);
  mm = wave_max(mm);
  if ((threadIdx.x & 63) == 0) { sp[threadIdx.x >> 6] = p; sm[threadIdx.x >> 6] = mm; }
  __syncthreads();
  if (threadIdx.x == 0) {
    p = sp[0] + sp[1] + sp[2] + sp[3];
    mm = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]));
    if (p) atomicAdd(&C->n_pairs, p);
    atomicMax(&C->mmax_bits, __float_as_uint(mm) & 0x7fffffffu);   // the sign bit cleared: a -0 mass counts as 0
  }
}

long long hier_bin_blocks(long long n) { return (n + kHbChunk - 1) / kHbChunk; }

hipError_t launch_count_to_capacity(unsigned* cnt, long long nkeys, int cus, hipStream_t s) {
  if (nkeys <= 0) return hipSuccess;
  const long long want = (nkeys + 255) / 256;
  count_to_capacity<<<(int)std::min<long long>(want, (long long)cus * 16), 256, 0, s>>>(cnt, nkeys);
  return hipGetLastError();
}

template <int MODE>
static hipError_t bin_base_mode(const Plan& P, const Parts& A, unsigned long long* cursor,
                                const unsigned long long* start, int4* entries, Counters* C, const BlockTables& BT,
                                const TableBin& TB, int cus, hipStream_t s) {
  const long long nb = hier_bin_blocks(A.n);
  if (nb == 0) return hipSuccess;
  static int per_cu = 0;
  if (per_cu <= 0) {
    int k = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&k, bin_base<MODE>, kHbThreads, 0) != hipSuccess || k <= 0) k = 4;
    per_cu = k;
  }
  // the workgroups that fit the chip at once, each taking chunks in turn
  const long long grid = std::min<long long>(nb, (long long)cus * per_cu);
  bin_base<MODE><<<(unsigned)grid, kHbThreads, 0, s>>>(P, A, cursor, start, entries, C, BT, TB);
  return hipGetLastError();
}

hipError_t launch_bin_base(const Plan& P, const Parts& A, unsigned long long* cursor,
                           const unsigned long long* start, int4* entries, Counters* C, const BlockTables& BT,
                           const TableBin& TB, int cus, hipStream_t s) {
  return P.mode == 2 ? bin_base_mode<2>(P, A, cursor, start, entries, C, BT, TB, cus, s)
                     : bin_base_mode<1>(P, A, cursor, start, entries, C, BT, TB, cus, s);
}

long long emit_pieces(int chunk) { return (chunk + kEtPiece - 1) / kEtPiece; }

hipError_t launch_after_bin(const Plan& P, const Parts& A, const BlockTables& BT, const Item* items,
                            long long n_items, unsigned long long* cursor, const unsigned long long* start,
                            int4* entries, Counters* C, const TableBin& TB, int cus, hipStream_t s) {
  const long long nblk = hier_bin_blocks(A.n);
  const long long want = (std::max(nblk, P.mode == 1 && P.nl > 0 ? n_items : 0ll) + 255) / 256;
  const int grid = (int)std::min<long long>(std::max<long long>(want, 1), (long long)std::max(cus, 1) * 4);
  if (P.mode == 2) after_bin<2><<<grid, 256, 0, s>>>(P, A, BT, nblk, items, n_items, cursor, start, entries, C, TB);
  else after_bin<1><<<grid, 256, 0, s>>>(P, A, BT, nblk, items, n_items, cursor, start, entries, C, TB);
  return hipGetLastError();
}

hipError_t launch_emit_table(const Plan& P, const Item* items, long long n_items, int chunk,
                             unsigned long long* cursor, const unsigned long long* start, int4* entries,
                             unsigned* item_pairs, Counters* C, const TableBin& TB, int cus, hipStream_t s) {
  if (n_items <= 0) return hipSuccess;
  static int per_cu = 0;
  if (per_cu <= 0) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, emit_table, kEtThreads, 0) != hipSuccess || nb <= 0) nb = 4;
    per_cu = nb;
  }
  const long long most = n_items * emit_pieces(chunk);
  emit_table<<<(int)std::min<long long>(most, (long long)cus * per_cu), kEtThreads, 0, s>>>(
      P, items, TB.units, cursor, start, entries, item_pairs, C, TB);
  return hipGetLastError();
}

hipError_t launch_emit_tsc(const Plan& P, const Item* items, long long item_lo, long long item_hi, int chunk, int level,
                           unsigned long long* cursor, const unsigned long long* start, int4* entries,
                           unsigned* item_pairs, Counters* C, int cus, hipStream_t s) {
  if (item_hi <= item_lo) return hipSuccess;
  if (level < 0 || level >= kNLevels) return hipErrorInvalidValue;
  // the workgroups that fit the chip at once; the queue balances the items,
  // taken up to 8 at a time while there are many per workgroup
  static int per_cu = 0;
  if (per_cu <= 0) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, emit_tsc, kEmThreads, 0) != hipSuccess || nb <= 0) nb = 4;
    per_cu = nb;
  }
  const long long items_n = item_hi - item_lo, room = (long long)cus * per_cu;
  // pieces of at least one round, as many as workgroups fit
  const int rounds = (chunk + kEmRound - 1) / kEmRound;
  const int pieces = (int)std::max<long long>(1, std::min<long long>(rounds, room / items_n));
  const int plen = (rounds + pieces - 1) / pieces * kEmRound;
  const long long n = items_n * pieces;
  const int grid = (int)std::min<long long>(n, room);
  const int batch = (int)std::max<long long>(1, std::min<long long>(8, n / ((long long)grid * 16)));
  emit_tsc<<<grid, kEmThreads, 0, s>>>(P, items, item_lo, n, pieces, plen, level, batch, cursor, start, entries,
                                       item_pairs, C);
  return hipGetLastError();
}

}  // namespace asohf
