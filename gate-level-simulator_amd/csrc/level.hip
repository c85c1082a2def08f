// Fused per-level gate evaluation (gfx950): walk, join, compact.
//
// Work unit: a tile = a run of consecutive words of a gate's longest input
// (the "leader") and the other inputs' words of the same time span, so tile
// boundaries are exact event times.
//
// k_level (walk), one tile at a time per wavefront, tiles independent:
//   1. the tile's input ranges (one event before the tile for the starting
//      values, a D_max look-ahead halo after it) and the gate's two tables
//      are copied into LDS with direct-to-LDS loads, each range followed by an
//      INF sentinel (tiles too long for LDS keep their stacks in the overflow
//      buffer and, where even their inputs do not fit, read HBM instead);
//   2. the tile's words are cut into equal shares, one per lane (lane_bounds);
//      every lane merges its share in time order and looks every event up:
//      a truth byte by the input values, then a delay word by the gate's old
//      and new value and the inputs with an event (lane_walk);
//   3. the preemption rule is applied backwards over each lane's candidates,
//      with one suffix minimum over the wavefront for the lanes after it
//      (keep_entries);
//   4. the lanes' lists are joined (a list that starts with the value before
//      it drops that entry) and stored into the level scratch, and lane 0
//      writes the tile summary (count, first and last entry, gate events)
//      (emit_tile).
//   The next tile's loads are issued when the walk no longer reads its inputs.
//
// What bounds the walk: VALU issue (61% of the SIMDs' cycles) and, with two
// wavefronts per SIMD (LDS-limited), the latency of LDS reads (bank conflicts take
// 38% of the LDS's cycles: lanes read their inputs at unrelated places).  On the
// 200k-cell configuration (gap 500 ps) it issues 0.97 VALU and 0.29 scalar
// wave-instructions per gate event, and a tile of 1,940 events takes 24,000 cycles
// of a wavefront: 4,700 to the lanes' bounds, 10,800 in the steps (41 of 22 to 34
// VALU instructions, where 31 would do if the lanes' shares were exact), 3,800
// for preemption, 2,000 to issue the next tile's loads, 900 waiting for them, 1,800
// to store.  Per run over 10 Mps (2M cells over 2 Mps):
//   154 ms (615)  delays by edge class and event bits each step, a halo walked by
//                 every lane, a wavefront scan of 3-word aggregates
//    99 ms (405)  table lookups, equal lane shares, one lane's halo
//    96 ms (395)  lane starts from exact ranks, lighter level ends
//    87 ms        descriptor fields as scalars
//    79 ms (323)  preemption without branches, SAIF durations left to the copy
//    76 ms (310)  no wait for a tile's stores, a ticket counter of its own
// Tried and slower: tiles of 16, 24 or 28 words a lane at the more workgroups a CU
// that they allow, less LDS around a tile's words (tiles in HBM cost 40 us each),
// searches that start in a window around the even split.
// k_join: per gate, joins its tiles in order (a tile whose first entry repeats
//   the value before it drops that entry), places them, and adds the SAIF
//   durations between them.
// k_compact: copies each tile's joined entries into the gate's dense waveform
//   in the pool (coalesced), so the pool holds exactly the outputs, and sums the
//   SAIF durations (and toggles when asked) inside tiles.
//
// Event rules: src/simulate.cpp:919-1201 (Calculate, AddDelay, CheckDelay),
// src/simulate.cpp:1365-1506 (Process, GetValueAt).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include <type_traits>

#include "device.h"

namespace gls {

constexpr int kLanes = 64;

// ERR_ORDER: a bound that holds for time-ordered inputs was hit (a lane's
// stack region or a tile's output region would have been overrun); the
// write was dropped.
enum : unsigned { ERR_OVERFLOW = 2u, ERR_RANGE = 4u, ERR_CAPACITY = 8u, ERR_POOL = 16u,
                  ERR_ORDER = 32u };

__device__ __forceinline__ uint32_t edge_cls(uint32_t pre, uint32_t cur) {
  // CheckDelay (src/simulate.cpp:1178-1201); codes 0=0 1=X 2=Z 3=1
  const uint64_t T = 0x0222ull << 48 | 0x1042ull << 32 | 0x1302ull << 16 | 0x1110ull;
  return (uint32_t)(T >> ((pre * 4 + cur) * 4)) & 0xF;
}

// Cross-lane moves with DPP (no LDS round trip).  Lanes without a source
// lane (outside the row, or rows left out by ROW_MASK) receive OLD.
// Control codes: row_shr:d 0x110+d, row_shl:d 0x100+d, wave_shl:1 0x130,
// wave_shr:1 0x138, row_bcast:15 0x142, row_bcast:31 0x143.
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ uint32_t dpp(uint32_t x, uint32_t old = 0) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)x, CTRL, ROW_MASK, 0xF, false);
}

// Inclusive prefix sum over the wavefront: within rows of 16 by row shifts,
// then row 0's total into row 1 and row 2's into row 3 (row_bcast:15), then
// lane 31's prefix into rows 2 and 3 (row_bcast:31).
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
  x += dpp<0x111>(x);
  x += dpp<0x112>(x);
  x += dpp<0x114>(x);
  x += dpp<0x118>(x);
  x += dpp<0x142, 0xA>(x);
  x += dpp<0x143, 0xC>(x);
  return x;
}

// Sum over the wavefront (uniform result).
__device__ __forceinline__ uint32_t wave_sum(uint32_t x) {
  return __builtin_amdgcn_readlane(wave_scan(x), 63);
}

// Minimum over the lanes after this one (all ones for lane 63): within rows
// by row shifts, the later rows' minima from their first lanes.
__device__ __forceinline__ uint32_t wave_min_after(uint32_t x) {
  x = min(x, dpp<0x101>(x, 0xFFFFFFFFu));
  x = min(x, dpp<0x102>(x, 0xFFFFFFFFu));
  x = min(x, dpp<0x104>(x, 0xFFFFFFFFu));
  x = min(x, dpp<0x108>(x, 0xFFFFFFFFu));
  const uint32_t r3 = __builtin_amdgcn_readlane(x, 48);
  const uint32_t r2 = min((uint32_t)__builtin_amdgcn_readlane(x, 32), r3);
  const uint32_t r1 = min((uint32_t)__builtin_amdgcn_readlane(x, 16), r2);
  const uint32_t lane = threadIdx.x;
  const uint32_t later = lane < 16 ? r1 : (lane < 32 ? r2 : (lane < 48 ? r3 : 0xFFFFFFFFu));
  return dpp<0x130>(min(x, later), 0xFFFFFFFFu);
}

__device__ __forceinline__ void saif_acc(unsigned long long* acc, uint32_t v, unsigned long long a,
                                         unsigned long long b, unsigned long long start,
                                         unsigned long long end) {
  unsigned long long lo = a > start ? a : start, hi = b < end ? b : end;
  const unsigned long long len = hi > lo ? hi - lo : 0ull;
  acc[0] += v == 0 ? len : 0ull;
  acc[1] += v == 3 ? len : 0ull;
  acc[2] += (v == 1 || v == 2) ? len : 0ull;
}

template <typename P>
__device__ __forceinline__ uint32_t lb_words(P a, uint32_t n, uint32_t key) {
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    uint32_t mid = (lo + hi) >> 1;
    if (a[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(3))) uint8_t lds_u8;
// Global memory behind an address that travelled as a number: without the
// address space its accesses would be flat ones, which also count as LDS
// accesses and hold up the waits for them.
typedef __attribute__((address_space(1))) uint32_t glb_u32;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef __attribute__((address_space(1))) u32x4 glb_u32x4;

// LDS by byte address (32-bit local pointers: the reads are ds_read with the
// constant part of the address in the instruction).
__device__ __forceinline__ uint32_t lds32(uint32_t a) { return *(const lds_u32*)a; }
__device__ __forceinline__ uint32_t lds16(uint32_t a) { return *(const lds_u16*)a; }
__device__ __forceinline__ uint32_t lds8(uint32_t a) { return *(const lds_u8*)a; }

// One 4-byte direct-to-LDS load per lane: lane i's word lands at l + i.
__device__ __forceinline__ void dma_word(const uint32_t* g, uint32_t* l) {
  __builtin_amdgcn_global_load_lds(g, (lds_void*)l, 4, 0, 0);
}

// One 16-byte direct-to-LDS load per lane (gfx950): lane i's four words
// land at l + 4 i.  g is 16-byte aligned.
__device__ __forceinline__ void dma_x4(const uint32_t* g, uint32_t* l) {
  __builtin_amdgcn_global_load_lds(g, (lds_void*)l, 16, 0, 0);
}

// Wait until this wavefront has no vector-memory access in flight (direct-to-
// LDS loads included): s_waitcnt vmcnt(0).  A workgroup is one wavefront, whose
// LDS accesses stay in order: beside this wait only the compiler needs fences
// (a barrier's would also wait for the stores in flight).
__device__ __forceinline__ void lds_fence() { asm volatile("" ::: "memory"); }
__device__ __forceinline__ void wait_vm() {
  lds_fence();
  __builtin_amdgcn_s_waitcnt(0x0F70);
  lds_fence();
}

// A tile's descriptor in scalar registers.
struct Tile {
  uint32_t in_lo[6], n[6], in_hi[2];
  uint64_t scr;
  uint32_t own, xend, meta, dt_off, tt_off, dmax, job, out_cap, g, at2[3], words, tab;

  __device__ __forceinline__ uint32_t id() const { return meta & 15u; }
  __device__ __forceinline__ uint32_t k() const { return (meta >> 4) & 15u; }
  __device__ __forceinline__ uint32_t lead() const { return (meta >> 8) & 15u; }
  __device__ __forceinline__ bool starts_gate() const { return (meta >> 12) & 1u; }
  __device__ __forceinline__ uint32_t edge_in() const { return (meta >> 16) & 15u; }
  __device__ __forceinline__ uint64_t src(int j) const {
    return ((uint64_t)((in_hi[j >> 2] >> (8 * (j & 3))) & 0xFFu) << 32) | in_lo[j];
  }
  __device__ __forceinline__ uint32_t dt_words() const { return tab & 0xFFFFu; }
  __device__ __forceinline__ uint32_t tt_words() const { return tab >> 16; }
  // LDS word of input j's range (range_at)
  __device__ __forceinline__ uint32_t at(int j) const { return (at2[j >> 1] >> (16 * (j & 1))) & 0xFFFFu; }
};

// A tile descriptor is read with one coalesced load (lane i < 32 holds
// dword i), a tile ahead, and broadcast with readlane: its fields are scalars
// and no load of theirs waits behind the staging loads in flight.  The loaded
// word is what a loop carries, not the scalars: uniform for a reader, they are
// divergent for the compiler wherever a branch of single lanes meets the loop's,
// and it then keeps them in vector registers and walks every branch on them with
// the execution mask (a quarter of the instructions of a tile's fixed part).
__device__ __forceinline__ uint32_t desc_word(const TileDesc* p) {
  return threadIdx.x < 32 ? ((const uint32_t*)p)[threadIdx.x] : 0u;
}

__device__ __forceinline__ Tile tile_of(uint32_t dw) {
  uint32_t w[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) w[i] = __builtin_amdgcn_readlane(dw, i);
  Tile D;
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    D.in_lo[j] = w[j];
    D.n[j] = w[6 + j];
  }
  D.in_hi[0] = w[12];
  D.in_hi[1] = w[13];
  D.scr = ((uint64_t)w[15] << 32) | w[14];
  D.own = w[16];
  D.xend = w[17];
  D.meta = w[18];
  D.dt_off = w[19];
  D.tt_off = w[20];
  D.dmax = w[21];
  D.job = w[22];
  D.out_cap = w[23];
  D.g = w[24];
  D.at2[0] = w[27];
  D.at2[1] = w[28];
  D.at2[2] = w[29];
  D.words = w[30];
  D.tab = w[31];
  return D;
}

// A value that is the same in every lane, for the compiler too.
__device__ __forceinline__ uint32_t uni(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint64_t uni(uint64_t x) {
  return ((uint64_t)uni((uint32_t)(x >> 32)) << 32) | uni((uint32_t)x);
}

__device__ __forceinline__ bool tile_fits(const LevelArgs& A, const Tile& D) {
  return D.id() < W_COUNT &&
         D.dt_words() + D.tt_words() + 2 * D.words + 8 * D.k() + kStackSlack <= A.lds_words;
}
// A tile whose inputs fit, but not its stacks beside them.
__device__ __forceinline__ bool inputs_fit(const LevelArgs& A, const Tile& D) {
  return D.id() < W_COUNT && D.dt_words() + D.tt_words() + D.words + 8 * D.k() <= A.lds_words;
}
// First word behind the tile's input ranges.
__device__ __forceinline__ uint32_t in_end(const Tile& D) {
  return D.dt_words() + D.tt_words() + D.words + 8 * D.k();
}
// First word of the tile's stacks: they end with the workgroup's LDS, so the
// next tile's inputs can be staged at the front while they are read.
__device__ __forceinline__ uint32_t stack_at(const LevelArgs& A, const Tile& D) {
  return A.lds_words - D.words - kStackSlack;
}

// Issue the loads of a tile into LDS: its gate's tables (unless the tile
// before was of the same gate) and its input ranges (the 16-byte copies may also
// bring up to 3 words before and after a range, inside its slot).  Completion:
// wait_vm().
__device__ __forceinline__ void stage_tile(const LevelArgs& A, const Tile& D, bool tables,
                                           uint32_t* lds) {
  const uint32_t lane = threadIdx.x;
  if (tables) {
    const uint32_t dw = D.dt_words(), tw = D.tt_words();
    const uint32_t* dsrc = A.dtab + D.dt_off;
    const uint32_t* tsrc = A.ttab + D.tt_off;
#pragma unroll 1
    for (uint32_t i = 0; i < dw; i += 4 * kLanes)
      if (i + 4 * lane < dw) dma_x4(dsrc + i + 4 * lane, lds + i);
#pragma unroll 1
    for (uint32_t i = 0; i < tw; i += 4 * kLanes)
      if (i + 4 * lane < tw) dma_x4(tsrc + i + 4 * lane, lds + dw + i);
  }
#pragma unroll
  for (uint32_t j = 0; j < kWideK; ++j) {
    if (j >= D.k()) break;
    const uint32_t a = D.in_lo[j] & 3u;
    const uint32_t m = (a + D.n[j] + 3) & ~3u;  // words copied, a multiple of 4
    const uint32_t* src = A.pool + (D.src(j) - a);
    uint32_t* l = lds + (D.at(j) - a);
#pragma unroll 1
    for (uint32_t i = 0; i < m; i += 4 * kLanes)
      if (i + 4 * lane < m) dma_x4(src + i + 4 * lane, l + i);
  }
}

// INF after every input range of a staged tile (its loads have arrived).  Every
// lane writes the same word: a branch for one lane is dearer.
__device__ __forceinline__ void put_sentinels(const Tile& D) {
#pragma unroll
  for (uint32_t j = 0; j < kWideK; ++j) {
    if (j >= D.k()) break;
    *(lds_u32*)(4 * (D.at(j) + D.n[j])) = kWordInf;
  }
}

// What one lane's walk leaves: candidates (or, later, kept entries) at
// [lo, hi) in time order, and the gate events the lane owned.  SP: pointer
// into LDS or HBM.
template <typename SP>
struct Lane {
  SP lo, hi;
  uint32_t nown;
  bool look;  // (uniform) some lane's events lie before the chunk
};

// The lanes' segments.  The tile's own words, in the merged time order of
// its inputs, are cut into equal shares: lane l starts at the event time of
// word floor(l * own / M).  When another tile follows, M = 63 and the last
// lane takes the halo (the dmax window after the tile): its candidates only
// pre-empt.  A lane's candidates pre-empt those of the lanes before it through
// one suffix minimum over the wavefront, so no lane walks another's events.
//
// x[j]: index of the lane's first word in input j's range (times at or after
// the segment's start); t0 / t1: the segment's bounds as words (time << 2).
//   fan-in 1: the index itself.
//   fan-in 2: binary search on the merge path's diagonal (exact: 11 steps of
//     two LDS reads for 2,000 words).
//   fan-in 3+: a start is an event of the leader input: its index at the
//     leader's share of the rank, the other inputs' positions and with them the
//     exact rank by binary search, then interpolation between the two lanes
//     around the wanted rank and a short second search (the merged rank of
//     3..6 ranges has no direct search).  Of 32.5 words a lane on average the
//     longest lane has 41; corrected by its own rank error alone it had 48, and
//     a tile's walk lasts as long as its longest lane's.
template <int K>
__device__ __forceinline__ void lane_bounds(const uint32_t (&in)[K], const Tile& D, uint32_t k,
                                            uint32_t (&a)[K], uint32_t& t0, uint32_t& t1) {
  const uint32_t lane = threadIdx.x;
  const bool more = D.xend != 0;
  const uint32_t d = more ? lane * D.own / 63u : lane * D.own / 64u;
  if constexpr (K == 1) {
    a[0] = in[0] + 4 * (1 + d);
    t0 = lds32(a[0]) & ~3u;
  } else if constexpr (K == 2) {
    const uint32_t nA = D.n[0] - 1, nB = D.n[1] - 1;
    uint32_t lo = d > nB ? d - nB : 0u, hi = min(d, nA);
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      // the mid-th word of input 0 comes before the (d - 1 - mid)-th of input 1
      if (lds32(in[0] + 4 * mid + 4) <= lds32(in[1] + 4 * (d - mid))) lo = mid + 1;
      else hi = mid;
    }
    a[0] = in[0] + 4 * lo + 4;
    a[1] = in[1] + 4 * (d - lo) + 4;
    t0 = min(lds32(a[0]), lds32(a[1])) & ~3u;
    // a word of the same time on the other side of the cut belongs to it
    a[0] -= lds32(a[0] - 4) >= t0 ? 4u : 0u;
    a[1] -= lds32(a[1] - 4) >= t0 ? 4u : 0u;
  } else {
    uint32_t il = in[0], nl = D.n[0];
#pragma unroll
    for (int j = 1; j < K; ++j) {
      il = (uint32_t)j == D.lead() ? in[j] : il;
      nl = (uint32_t)j == D.lead() ? D.n[j] : nl;
    }
    const uint32_t last = more ? D.xend : nl;  // leader index of the tile's end
    const float r = (float)(last - 1) * __builtin_amdgcn_rcpf((float)max(D.own, 1u));
    const bool halo = more && lane == kLanes - 1;
    const int top = max((int)last - 1, 1);
    int x = halo ? (int)last : min(1 + (int)((float)d * r), top);
    // lane 0 starts with the tile, also where the leader starts later
    t0 = lane == 0 ? 4u : lds32(il + 4 * x) & ~3u;
    // p[j]: the last word before t0.  All inputs' searches descend together
    // (their reads overlap) in steps of powers of two; a step past the range
    // reads its sentinel.
    uint32_t p[K], nmax = 1;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      p[j] = in[j];
      nmax = max(nmax, (uint32_t)j < k ? D.n[j] : 0u);
    }
    auto descend = [&](uint32_t step) {
      for (; step; step >>= 1) {
        uint32_t v[K], c[K];
#pragma unroll
        for (int j = 0; j < K; ++j) {
          c[j] = p[j] + 4 * step;
          v[j] = lds32(min(c[j], in[j] + ((uint32_t)j < k ? 4 * D.n[j] : 0u)));
        }
#pragma unroll
        for (int j = 0; j < K; ++j) p[j] = v[j] < t0 && (uint32_t)j < k ? c[j] : p[j];
      }
    };
    const uint32_t full = 0x80000000u >> __builtin_clz(nmax);
    descend(full);
    uint32_t rank = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) rank += (uint32_t)j < k ? (p[j] - in[j]) / 4 : 0u;
    // the lanes' guesses are 64 knots of the exact rank over the leader: take
    // the knots around the wanted rank (i the last at or below it) and
    // interpolate; the positions follow knot i's
    const uint32_t knot = rank << 16 | (uint32_t)x, past = D.own << 16 | last;
    uint32_t i = 0;
#pragma unroll
    for (uint32_t s = 32; s; s >>= 1) i += (uint32_t)__shfl((int)knot, (int)(i + s)) >> 16 <= d ? s : 0u;
    const uint32_t ka = (uint32_t)__shfl((int)knot, (int)i), kn = (uint32_t)__shfl((int)knot, (int)(i + 1));
    const uint32_t kb = i < 63 ? kn : past;
    const int xa = (int)(ka & 0xFFFFu), xb = (int)(kb & 0xFFFFu);
    const float per = (float)(xb - xa) * __builtin_amdgcn_rcpf((float)max((kb >> 16) - (ka >> 16), 1u));
    const int dx = (int)((float)(d - (ka >> 16)) * per + 0.5f);
    const int xi = max(min(min(xa + dx, xb), top), 1);
#pragma unroll
    for (int j = 0; j < K; ++j) p[j] = (uint32_t)__shfl((int)p[j], (int)i);
    x = halo ? x : xi;
    t0 = lane == 0 ? 4u : lds32(il + 4 * x) & ~3u;
    // 31 words from knot i's positions, and everywhere when a lane's lies beyond
    uint32_t p0[K];
    bool miss = false;
#pragma unroll
    for (int j = 0; j < K; ++j) p0[j] = p[j];
    descend(16);
#pragma unroll
    for (int j = 0; j < K; ++j) miss |= (uint32_t)j < k && p[j] == p0[j] + 4 * 31;
    if (__ballot(miss)) {
#pragma unroll
      for (int j = 0; j < K; ++j) p[j] = in[j];
      descend(full);
    }
#pragma unroll
    for (int j = 0; j < K; ++j) a[j] = (uint32_t)j < k ? p[j] + 4 : in[j];
  }
  t1 = dpp<0x130>(t0, more ? t0 + 4 * D.dmax : 0xFFFFFFFCu);
}

// One lane's walk over its segment in LDS: merges the inputs in time order
// and evaluates every event without branches (4-state truth table, edge
// class and AddDelay folded into the gate's tables, WalkId); each change of
// the gate's value is appended as a candidate word o << 2 | f.
//
// A step takes every input event at the next event time (w: its smallest
// word): heads h, addresses a of the next words, last words taken pw (their
// low bits are the inputs' values), packed by alignbit into the top bits of x
// (the old values stay below the new ones).
//
// Index 0 of every range is the word before the tile, so the values before a
// segment are the low bits of the words before its first ones.
template <int ID, int K>
__device__ __forceinline__ Lane<lds_u32*> lane_walk(const LevelArgs& A, const Tile& D) {
  constexpr bool NE = ID <= W_NE6, EO = ID == W_EO3 || ID == W_EO4, GEN = ID == W_GEN;
  const uint32_t k = GEN ? D.k() : (uint32_t)K;
  const uint32_t lane = threadIdx.x;
  const uint32_t ttb = 4 * walk_dt_words(ID, K);  // truth bytes; the delay table is at 0
  uint32_t in[K], a[K];
#pragma unroll
  for (int j = 0; j < K; ++j) in[j] = 4 * D.at(j);
  if (GEN) {
    // unused inputs stand at input 0's sentinel
#pragma unroll
    for (int j = 0; j < K; ++j)
      if ((uint32_t)j >= k) in[j] = in[0] + 4 * D.n[0];
  }
  uint32_t t0, t1;
  lane_bounds<K>(in, D, k, a, t0, t1);
  uint32_t h[K], pw[K], x = 0, soff = lane + min(lane, 1u);
#pragma unroll
  for (int j = 0; j < K; ++j) {
    h[j] = lds32(a[j]);
    pw[j] = GEN && (uint32_t)j >= k ? 0u : lds32(a[j] - 4);
    soff += (a[j] - in[j]) / 4 - (GEN && (uint32_t)j >= k ? 0u : 1u);
    x = __builtin_amdgcn_alignbit(pw[j], x, 2);
  }
  Lane<lds_u32*> ln;
  uint32_t sp = 4 * (stack_at(A, D) + soff);
  ln.lo = (lds_u32*)sp;
  // the gate's value before the first event: X at t = 0 (src/simulate.cpp:933),
  // else the function of the values
  const bool init = D.starts_gate() && A.first && lane == 0;
  const uint32_t fsh = ne_shift(k);
  // NE, EO: the value before, at its place in the delay table's byte offset;
  // GEN: the value before
  uint32_t fp = 0;
  if (NE) {
    fp = lds8(ttb + (x >> (32 - 2 * K)));
    fp = init ? 1u << ne_shift(K) : fp;
    fp <<= K > 4 ? K - 2 : 2;
  } else if (EO) {
    fp = lds8(ttb + (x >> (32 - 2 * K))) >> (kEoShift + 1);
    fp = (init ? 1u : fp) << (K + 5);
  } else if (GEN) {
    fp = init ? 1u : lds8(ttb + (x >> 20)) >> fsh;
  }
  if (init) {  // every output starts with (0, X) (src/simulate.cpp:882-887); t = 0 is rel 1
    *(lds_u32*)sp = (1u << 2) | 1u;
    sp += 4;
  }
  uint32_t w = h[0];
#pragma unroll
  for (int j = 1; j < K; ++j) w = min(w, h[j]);
  // look-back events (t < lo_rel, chunks after the first) come first: they
  // make candidates but are not this chunk's gate events
  const uint32_t lo_w = A.lo_rel << 2;
  uint32_t bound = t1;
  bool look = __ballot(w < lo_w && w < t1) != 0;
  ln.look = look;
  if (look) bound = min(lo_w, t1);
  uint32_t nown = 0;
  // The two lookups of a step and its push are spread over the steps after it,
  // so that a step waits only for its heads: fa, ea, la are the truth byte
  // (being read), events and time of the step before; vb, lb, tb the delay
  // word (being read), time and truth byte of the one before that.  The first
  // values stand for a step without a change.
  uint32_t fa = 0, ea = 0, la = 0, vb = 0, lb = 0, tb = 0;
  if (NE) fa = fp >> (K > 4 ? K - 2 : 2);
  if (EO) fa = fp >> (K + 5 - kEoShift - 1);
  const uint32_t xs = 32 - 4 * K + 2 * D.edge_in();  // EO: the edge input's old value in x
  auto push = [&] {
    if constexpr (NE || EO) {
      uint32_t o;
      asm("v_mad_u32_u24 %0, %1, 1, %2" : "=v"(o) : "v"(vb), "v"(lb));
      *(lds_u32*)sp = o;
      sp += __builtin_amdgcn_ubfe(vb, 22, 3);
    } else {
      *(lds_u32*)sp = lb + vb + (tb & 3u);
      sp += (tb >> 7) << 2;
    }
  };
  auto look_up = [&] {
    if constexpr (NE) {
      vb = lds32(ea | (fa << (K > 4 ? K - 4 : 0)) | fp);
      fp = fa << (K > 4 ? K - 2 : 2);
    } else if constexpr (EO) {
      vb = lds32(ea | (fa << (K + 2 - kEoShift)) | fp);
      fp = (fa >> (kEoShift + 1)) << (K + 5);
    } else {
      vb = lds32((ea << (K + 2)) | (fa & (((4u << K) - 1u) << 2)));
      tb = fa;
    }
    lb = la;
  };
  for (;;) {
    while (w < bound) {
      const uint32_t lim = w | 3u;
      uint32_t e = 0;
      const uint32_t xo = x;
#pragma unroll
      for (int j = 0; j < K; ++j) {
        const bool take = K == 1 || h[j] <= lim;
        const uint32_t s4 = take ? 4u : 0u;
        pw[j] = take ? h[j] : pw[j];
        a[j] += s4;
        e |= s4 << j;
        x = __builtin_amdgcn_alignbit(pw[j], x, 2);
      }
#pragma unroll
      for (int j = 0; j < K; ++j) h[j] = lds32(a[j]);
      if constexpr (!GEN) {
        push();
        look_up();
        if constexpr (EO)
          fa = lds8(ttb + ((__builtin_amdgcn_ubfe(x, xs, 2) << (2 * K)) | (x >> (32 - 2 * K))));
        else
          fa = lds8(ttb + (x >> (NE ? 32 - 2 * K : 32 - 4 * K)));
        ea = e;
        la = lim;
      } else {
        const uint32_t f = lds8(ttb + (x >> 20)) >> fsh;
        const uint32_t sc = edge_cls(fp, f);
        // per input: bit 2j an event, bit 2j+1 it fell (CheckDelay == 2: to 0
        // from X/Z/1, or from 1 to X/Z)
        const uint32_t c = x >> 20, p = xo >> 20;
        const uint32_t cs = c << 1, ps = p << 1;
        const uint32_t fell = (~c & ~cs & (p | ps)) | ((p & ps) & (c ^ cs));
        uint32_t ev = 0;
#pragma unroll
        for (int j = 0; j < K; ++j) ev |= ((e >> (2 + j)) & 1u) << (2 * j);
        const uint32_t bits = (fell & 0xAAAu) | ev;
        const uint32_t b0 = bits & 63u, b1 = bits >> 6;
        const uint32_t s0 = ((sc - 1u) & 3u) << 6;
        const bool both = (b0 & 0x15u) && (b1 & 0x15u);
        const uint32_t bo = both ? 256u : 0u;
        const uint32_t d0 = lds16(2 * (bo + s0 + b0)), d1 = lds16(2 * (512u + bo + s0 + b1));
        uint32_t dd = both ? min(d0, d1) : ((b0 & 0x15u) ? d0 : d1);
        dd = both && dd == 0xFFFFu ? 1u : dd;
        *(lds_u32*)sp = lim + 4 * dd - 3 + f;
        sp += sc != 0u ? 4u : 0u;
        fp = f;
      }
      ++nown;
      w = h[0];
#pragma unroll
      for (int j = 1; j < K; ++j) w = min(w, h[j]);
    }
    if (!look) break;
    look = false;
    nown = 0;
    bound = t1;
  }
  if constexpr (!GEN) {
    push();
    look_up();
    push();
  }
  ln.hi = (lds_u32*)sp;
  ln.nown = nown;
  return ln;
}

// The same walk for a tile too long for LDS: stacks in the overflow buffer,
// tables read from HBM, inputs too unless they fit LDS by themselves (`lds`: where
// they are staged), lanes at equal shares of the leader's words.  Rare (a tile's
// words are kept to its LDS share), so it is one form for every gate, and what it
// reads may be either kind of memory.  A step that waited for HBM made such a tile
// last about 40 us, a quarter of a level of 200,000 quiet cells, of which one in
// three has one (its walks 6.39 -> 6.15 ms a run with the inputs in LDS).  Writes
// that would leave the lane's buffer (inputs out of order) land on its last word
// and set bad.
__device__ __forceinline__ void hbm_walk(const LevelArgs& A, const Tile& D, const uint32_t* lds,
                                         uint32_t* stk, uint32_t stk_words, Lane<uint32_t*>& ln,
                                         uint32_t& bad) {
  const uint32_t lane = threadIdx.x;
  const uint32_t k = D.k(), id = D.id();
  const bool more = D.xend != 0;
  const uint32_t* in[6];
  uint32_t r[6], h[6], pw[6];
  const uint32_t* lead = nullptr;
  uint32_t nl = 0;
#pragma unroll
  for (uint32_t j = 0; j < kWideK; ++j) {
    in[j] = lds ? lds + D.at(j) : A.pool + D.src(j);
    if (j == D.lead()) {
      lead = in[j];
      nl = D.n[j];
    }
  }
  const uint32_t last = more ? D.xend : nl;  // leader index of the tile's end
  const uint32_t M = more ? 63u : 64u;
  const uint32_t xl = 1u + (uint32_t)((uint64_t)(last - 1) * min(lane, M) / M);
  uint32_t t0 = xl < nl ? lead[xl] & ~3u : 0xFFFFFFFCu;
  t0 = lane == 0 ? 4u : t0;
  const uint32_t t1 = dpp<0x130>(t0, more ? t0 + 4 * D.dmax : 0xFFFFFFFCu);
  uint32_t soff = lane, idx = 0;
#pragma unroll
  for (uint32_t j = 0; j < kWideK; ++j) {
    r[j] = 0;
    h[j] = kWordInf;
    pw[j] = 0;
    if (j >= k) continue;
    r[j] = 1 + lb_words(in[j] + 1, D.n[j] - 1, t0);
    pw[j] = in[j][r[j] - 1];
    h[j] = r[j] < D.n[j] ? in[j][r[j]] : kWordInf;
    soff += r[j] - 1;
    idx |= (pw[j] & 3u) << (2 * j);
  }
  const uint32_t s0 = min(soff, stk_words - 1), lim_n = stk_words - s0;
  uint32_t* st = stk + s0;
  const uint8_t* tt = (const uint8_t*)(A.ttab + D.tt_off);
  const uint32_t* dt = A.dtab + D.dt_off;
  const bool ed = id == W_ED1 || id == W_ED2, eo = id == W_EO3 || id == W_EO4;
  const uint32_t fsh = ne_shift(k);
  const bool init = D.starts_gate() && A.first && lane == 0;
  uint32_t fp = 1u, nc = 0, nown = 0;
  if (init) st[nc++] = (1u << 2) | 1u;
  else fp = ed ? tt[(idx << (2 * k)) | idx] & 3u : (uint32_t)tt[idx] >> (eo ? kEoShift + 1 : fsh);
  for (;;) {
    uint32_t w = h[0];
#pragma unroll
    for (uint32_t j = 1; j < kWideK; ++j) w = min(w, h[j]);
    if (w >= t1) break;
    const uint32_t lim = w | 3u;
    uint32_t ev = 0, nidx = 0;
#pragma unroll
    for (uint32_t j = 0; j < kWideK; ++j) {
      if (h[j] <= lim) {
        ev |= 1u << j;
        pw[j] = h[j];
        ++r[j];
        h[j] = r[j] < D.n[j] ? in[j][r[j]] : kWordInf;
      }
      nidx |= (pw[j] & 3u) << (2 * j);
    }
    uint32_t o;
    bool cand;
    if (ed) {
      const uint32_t t = tt[(nidx << (2 * k)) | idx];
      o = lim + dt[(ev << (k + 2)) | ((t >> 2) & ((4u << k) - 1u))] + (t & 3u);
      cand = (t >> 7) != 0;
    } else if (eo) {
      const uint32_t old = (idx >> (2 * D.edge_in())) & 3u;
      const uint32_t t = (uint32_t)tt[(old << (2 * k)) | nidx] >> kEoShift;
      o = lim + (dt[(((fp << 3) | t) << k) | ev] & 0x3FFFFu);
      cand = (t >> 1) != fp;
      fp = t >> 1;
    } else {
      const uint32_t f = (uint32_t)tt[nidx] >> fsh;
      cand = f != fp;
      if (id != W_GEN) {
        o = lim + (dt[(((fp << 2) | f) << k) | ev] & 0x3FFFFu);
      } else {
        const uint32_t sc = edge_cls(fp, f);
        uint32_t bits = 0;
#pragma unroll
        for (uint32_t j = 0; j < kWideK; ++j) {
          const uint32_t p = (idx >> (2 * j)) & 3u, c = (nidx >> (2 * j)) & 3u;
          bits |= ((ev >> j) & 1u) << (2 * j);
          bits |= (edge_cls(p, c) == 2u ? 2u : 0u) << (2 * j);
        }
        const uint32_t b0 = bits & 63u, b1 = bits >> 6, s = ((sc - 1u) & 3u) << 6;
        const bool both = (b0 & 0x15u) && (b1 & 0x15u);
        const uint16_t* q = (const uint16_t*)dt;
        const uint32_t d0 = q[(both ? 256u : 0u) + s + b0], d1 = q[(both ? 768u : 512u) + s + b1];
        uint32_t dd = both ? min(d0, d1) : ((b0 & 0x15u) ? d0 : d1);
        dd = both && dd == 0xFFFFu ? 1u : dd;
        o = lim + 4 * dd - 3 + f;
      }
      fp = f;
    }
    if (cand) {
      const bool room = nc < lim_n;
      bad |= room ? 0u : 1u;
      st[room ? nc : lim_n - 1] = o;
      nc += room ? 1u : 0u;
    }
    nown += (w >> 2) >= A.lo_rel ? 1u : 0u;
    idx = nidx;
  }
  ln.lo = st;
  ln.hi = st + nc;
  ln.nown = nown;
  ln.look = true;
}

// The preemption rule of src/simulate.cpp:990-1009 in its closed form: a
// candidate is kept iff its output time is strictly below that of every
// later candidate.  Backwards over the lane's candidates with a running
// minimum, kept ones compacted (in time order) to the end of the region and
// an entry that repeats its predecessor's value dropped; then the later
// lanes' minimum (one suffix minimum over the wavefront) and the chunk's end
// (candidates at or above hi_rel belong to the next chunk) cut the list from
// the end.  Look-back candidates below lo_rel only pre-empt: a lane has some
// only where the tile has events before the chunk.
//
// Without them the step has no branch: the last kept entry `last` holds both
// the running minimum and the value to compare with, and a candidate that is
// not kept writes `last` once more where it stands.  Seven VALU instructions a
// candidate; with the two conditions as branches a tile's pass took 6,080 cycles
// of its 29,600 (200,000 cells at gap 500 ps).
template <typename SP>
__device__ __forceinline__ void keep_entries(const LevelArgs& A, Lane<SP>& ln, bool halo_lane) {
  SP q = ln.hi, jp = ln.hi;
  uint32_t rm = 0xFFFFFFFFu, left = (uint32_t)(ln.hi - ln.lo);
  // four reads in flight; `ahead`: the next four before this four's steps
  // (their words lie below those that the steps write)
  auto pass = [&](auto& take, auto ahead) {
    uint32_t e4[4];
    auto read4 = [&](uint32_t n) {
#pragma unroll
      for (int i = 0; i < 4; ++i) e4[i] = (uint32_t)i < n ? q[-1 - i] : kWordInf;
    };
    if (decltype(ahead)::value) read4(4);
    while (left >= 4) {
      if (!decltype(ahead)::value) read4(4);
      uint32_t t4[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) t4[i] = e4[i];
      q -= 4;
      left -= 4;
      if (decltype(ahead)::value) read4(4);
#pragma unroll
      for (int i = 0; i < 4; ++i) take(t4[i]);
    }
    if (left) {
      if (!decltype(ahead)::value) read4(left);
#pragma unroll
      for (int i = 0; i < 3; ++i) take((uint32_t)i < left ? e4[i] : kWordInf);
    }
  };
  // (reading ahead may read words below the lane's: inputs, in LDS)
  constexpr bool kLds = std::is_same<SP, lds_u32*>::value;
  if (!kLds || ln.look) {
    uint32_t lastv = 4u;
    const uint32_t lo_w = A.lo_rel << 2;
    auto take = [&](uint32_t e) {
      if (e < rm) {
        rm = e & ~3u;
        if (e >= lo_w) {
          const uint32_t v = e & 3u;
          jp -= v != lastv ? 1 : 0;
          *jp = e;
          lastv = v;
        }
      }
    };
    pass(take, std::false_type{});
  } else {
    // (the first candidate is below 0xFFFFFFFC, and its value is not that of the
    // initial `last`; a lane without candidates writes nothing)
    const bool some = left != 0;
    uint32_t last = ~q[-1] | 0xFFFFFFFCu;
    auto take = [&](uint32_t e) {
      const bool kept = e < (last & ~3u);
      const bool other = ((e ^ last) & 3u) != 0u;
      jp -= kept && other ? 1 : 0;
      last = kept ? e : last;
      *jp = last;
    };
    pass(take, std::true_type{});
    rm = some ? last & ~3u : 0xFFFFFFFFu;
  }
  const uint32_t hi_w = A.hi_rel == 0xFFFFFFFFu ? 0xFFFFFFFFu : A.hi_rel << 2;
  const uint32_t cut = min(wave_min_after(rm), hi_w);
  SP te = ln.hi;
  while (te > jp && te[-1] >= cut) --te;
  if (halo_lane) te = jp;
  ln.lo = jp;
  ln.hi = te;
}

// Join the lanes' lists (a list that starts with the value before it drops
// that entry), store the tile's entries at dst and write the tile summary.
// (The SAIF durations between them are summed where the entries are copied,
// one wavefront instruction for 64 of them: here it was one for as many as the
// lanes have at the same place of their lists.)  out_cap: words of the tile's
// output region (never reached for time-ordered inputs; entries beyond it are
// dropped, with ERR_ORDER).  `before_stores` runs just before the first store.
template <typename SP, typename F>
__device__ __forceinline__ void emit_tile(const LevelArgs& A, uint64_t tk, const Lane<SP>& ln,
                                          glb_u32* dst, uint32_t out_cap, F&& before_stores) {
  const int lane = threadIdx.x;
  const uint32_t n = (uint32_t)(ln.hi - ln.lo);
  const uint32_t e_first = n ? ln.lo[0] : 0u, e_last = n ? ln.hi[-1] : 0u;
  const uint64_t mask = __ballot(n > 0);
  const uint64_t below = mask & ((1ull << lane) - 1ull);
  const uint32_t prev = __shfl(e_last, below ? 63 - __clzll((long long)below) : 0);
  const uint32_t dup = (n && below && ((prev ^ e_first) & 3u) == 0u) ? 1u : 0u;
  const uint32_t mine = n - dup;
  const uint32_t incl = wave_scan(mine);
  const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
  uint32_t first = 0, last = 0;  // the tile's first and last entries
  const uint64_t with = __ballot(mine > 0);
  if (with) {
    first = __builtin_amdgcn_readlane(e_first, __ffsll((long long)with) - 1);
    last = __builtin_amdgcn_readlane(e_last, 63 - __clzll((long long)with));
  }
  const uint32_t ev = wave_sum(ln.nown);
  const uint32_t w = min(incl - mine, out_cap);
  before_stores();
  if (mine) {
    // (the tile's region is uniform: lanes add 32-bit offsets to it)
    auto to = [&](uint32_t q) { return (glb_u32*)((__attribute__((address_space(1))) char*)dst + q); };
    uint32_t dp = 4 * w;
    uint32_t left = min(mine, out_cap - w);  // entries that the region takes
    SP p = ln.lo + dup;
    // whole groups of four: four reads in flight, one store
    while (left >= 4) {
      *(glb_u32x4*)to(dp) = u32x4{p[0], p[1], p[2], p[3]};
      dp += 16;
      p += 4;
      left -= 4;
    }
    uint32_t e4[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) e4[q] = (uint32_t)q < left ? p[q] : 0u;
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if ((uint32_t)q < left) *to(dp + 4 * q) = e4[q];
  }
  if (lane == 0) {
    TileOut o;
    o.cnt = min(total, out_cap);
    if (total > out_cap) atomicOr((unsigned int*)(A.scal + S_ERR), ERR_ORDER);
    o.first = first;
    o.last = last;
    o.ev = ev;
    A.tout[tk] = o;
  }
}

// Persistent, software-pipelined walk kernel.  Tiles are independent (no
// tile waits for another): a workgroup walks a run of consecutive tiles and then
// draws batches by ticket.  The next tile's descriptor and ticket are on the
// way during the walk; its inputs are staged into LDS from the end of the
// walk on, behind the current tile's stacks, and waited for before the current
// tile's first store (a later wait would include the stores).  A static
// round-robin schedule left the workgroups that drew many tiles too long for
// LDS as a long tail (14% slower on the 200k-cell workload).  Whatever a tile
// leaves in flight on either path is waited for on that path: what may be in
// flight anywhere, the compiler waits for at the next tile's start, together with
// this one's stores.
__global__ __launch_bounds__(kLanes) void k_level(LevelArgs A) {
  // dynamic LDS, A.lds_words: tables, inputs, ..., stacks (walk_lds_need)
  extern __shared__ uint32_t s_dyn[];
  const int lane = threadIdx.x;
  unsigned long long wave_hbm = 0;  // of this wavefront's tiles
  if (A.scal[S_TRIP]) return;
  if (blockIdx.x == 0 && lane == 0) A.scal[S_CLOCK] = (uint64_t)wall_clock64();
  const uint64_t ntiles = A.scal[S_NTILES + A.slot];  // uniform: one scalar load
  glb_u32* const scratch = (glb_u32*)A.scal[S_SCRATCH + A.slot];
  unsigned int* const err = (unsigned int*)(A.scal + S_ERR);
  // Tiles are handed out in two parts.  The first half is split into
  // one run of consecutive tiles per workgroup (consecutive tiles of one gate
  // keep its tables in LDS).  The rest is drawn by ticket in batches of B, so
  // that workgroups with slow tiles take fewer and the level's tail stays
  // short.  One counter serves about 70 M tickets a second, which held levels of
  // short waveforms (one or two tiles a gate) to 70 M tiles a second: up to four
  // counters hand out every fourth batch each, to a quarter of the workgroups
  // each.  (A workgroup whose counter had run out went on to the other three,
  // one wait after the other and 6,000 tickets a level that found nothing: of
  // 200,000 quiet cells' 26,200 cycles a tile, 2,300.)
  const uint64_t n_run = max(1ull, (unsigned long long)(ntiles / 2 / gridDim.x));
  const uint64_t t_drawn = n_run * gridDim.x;  // first tile handed out by ticket
  const uint32_t B = (uint32_t)max(
      1ull, min(8ull, (unsigned long long)((ntiles - min(t_drawn, ntiles)) / (16ull * gridDim.x))));
  uint64_t tk = (uint64_t)blockIdx.x * n_run;
  if (tk >= ntiles) return;
  uint64_t bend = min(tk + n_run, ntiles);  // end of the current run or batch
  const uint32_t counters = min(kTickets, (gridDim.x + 7) / 8);  // every one has workgroups
  const uint32_t counter = (blockIdx.x >> 3) % counters;
  // lane 0: the ticket on its way; and the last one that has arrived.  It is
  // taken from `drawn` where the tile's loads are waited for: taken where it is
  // used, after the tile's stores, it would wait for those too.
  unsigned long long drawn = 0;
  uint64_t ticket = 0;
  auto draw = [&] {
    if (lane == 0 && t_drawn < ntiles) drawn = atomicAdd(A.ticket + counter * kTicketStride, 1ull);
  };
  auto drawn_batch = [&]() -> uint64_t {  // first tile of the drawn batch (at least ntiles: none left)
    return t_drawn + (counter + counters * ticket) * B;
  };
  if (tk + 1 >= bend) draw();
  uint32_t dw = desc_word(A.tiles + tk);
  uint32_t tab_g = 0xFFFFFFFFu;  // gate whose tables are in LDS
  {
    const Tile D = tile_of(dw);
    if (inputs_fit(A, D)) {
      stage_tile(A, D, true, s_dyn);
      tab_g = D.g;
      wait_vm();
      put_sentinels(D);
    }
  }
  ticket = uni((uint64_t)drawn);
  for (;;) {
    tk = uni(tk);
    tab_g = uni(tab_g);
    const Tile D = tile_of(dw);
    const bool fits = tile_fits(A, D);
    // the tile after this one: the next of its run, or the first of the batch
    // drawn a tile ago
    uint64_t tn = tk + 1;
    if (tn >= bend) {
      tn = drawn_batch();
      bend = tn + B < ntiles ? tn + B : ntiles;
    }
    tn = uni(tn);
    bend = uni(bend);
    const bool more_tiles = tn < ntiles;
    const uint32_t dwn = more_tiles ? desc_word(A.tiles + tn) : 0u;
    if (more_tiles && tn + 1 >= bend) draw();
    lds_fence();
    bool staged = false;  // the next tile's loads are on their way
    auto finish = [&](auto& ln) {
      // inputs and tables are no longer read
      lds_fence();
      const Tile Dn = tile_of(dwn);
      staged = more_tiles && A.prefetch && tile_fits(A, Dn) && !(fits && in_end(Dn) > stack_at(A, D));
      if (staged) stage_tile(A, Dn, Dn.g != tab_g, s_dyn);
      const bool halo = D.xend != 0 && lane == kLanes - 1;
      keep_entries(A, ln, halo);
      if (halo) ln.nown = 0;
      emit_tile(A, tk, ln, scratch + D.scr, D.out_cap, [&] {
        wait_vm();
        ticket = uni((uint64_t)drawn);
        if (staged) put_sentinels(Dn);
      });
    };
    if (fits) {
      Lane<lds_u32*> ln;
      switch (D.id()) {
        case W_NE1: ln = lane_walk<W_NE1, 1>(A, D); break;
        case W_NE2: ln = lane_walk<W_NE2, 2>(A, D); break;
        case W_NE3: ln = lane_walk<W_NE3, 3>(A, D); break;
        case W_NE4: ln = lane_walk<W_NE4, 4>(A, D); break;
        case W_NE5: ln = lane_walk<W_NE5, 5>(A, D); break;
        case W_NE6: ln = lane_walk<W_NE6, 6>(A, D); break;
        case W_EO3: ln = lane_walk<W_EO3, 3>(A, D); break;
        case W_EO4: ln = lane_walk<W_EO4, 4>(A, D); break;
        case W_ED1: ln = lane_walk<W_ED1, 1>(A, D); break;
        case W_ED2: ln = lane_walk<W_ED2, 2>(A, D); break;
        default: ln = lane_walk<W_GEN, 6>(A, D); break;
      }
      finish(ln);
    } else {
      Lane<uint32_t*> ln;
      ln.lo = ln.hi = A.ovf;
      ln.nown = 0;
      ln.look = true;
      if (D.id() < W_COUNT) {
        const unsigned long long need = (unsigned long long)D.words + kStackSlack;
        unsigned long long base = 0;
        if (lane == 0) base = atomicAdd((unsigned long long*)(A.scal + S_OVF_USED), need);
        base = uni((uint64_t)base);  // lane 0's value
        uint32_t bad = 0;
        if (base + need > A.ovf_cap) {
          // no room: the tile's output is left empty (so the level's waveforms
          // stay in time order) and the run reports the error
          if (lane == 0) atomicOr(err, ERR_OVERFLOW);
        } else {
          hbm_walk(A, D, inputs_fit(A, D) ? s_dyn : nullptr, A.ovf + base, (uint32_t)need, ln, bad);
        }
        if (bad) atomicOr(err, ERR_ORDER);
      }
      finish(ln);
      wait_vm();
    }
    lds_fence();
    wave_hbm += fits ? 0u : 1u;
    if (!more_tiles) break;
    const Tile Dn = tile_of(dwn);
    if (inputs_fit(A, Dn)) {
      if (!staged) {
        stage_tile(A, Dn, Dn.g != tab_g, s_dyn);
        wait_vm();
        put_sentinels(Dn);
      }
      tab_g = Dn.g;
    }
    lds_fence();
    tk = tn;
    dw = dwn;
  }
  if (lane == 0) {
    unsigned long long* n = (unsigned long long*)A.scal;
    if (wave_hbm) atomicAdd(n + S_TILES_HBM, wave_hbm);
  }
}

// Exclusive scan of one value per thread over a block of T threads.
template <int T>
__device__ __forceinline__ uint64_t block_scan(uint64_t v, uint64_t* sh, uint64_t& total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  uint64_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  __syncthreads();
  if (lane == 63) sh[wid] = x;
  __syncthreads();
  uint64_t before = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < T / 64; ++i) {
    if (i < wid) before += sh[i];
    tot += sh[i];
  }
  total = tot;
  return before + x - v;
}

// Scans over blocks in one launch: every block leaves its totals in `part`
// (agent-scope stores: the blocks run on XCDs with L2s of their own) and
// counts itself done; the last one turns the totals into prefixes.  No block
// waits for another.  The totals have left for memory before the block counts
// itself (the wait for its stores), and they are all that the last block reads
// of the others: a release fence here would write the XCD's whole L2 back, once
// per block.
__device__ __forceinline__ void put_part(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// `v`: a total small enough (40 bits) to travel with the count (24 bits): in,
// the block's; out, in the last block's first thread, the sum of all.
__device__ __forceinline__ bool last_block(uint64_t* done, uint32_t nb, uint64_t& v) {
  if (nb == 1) return true;
  __shared__ uint32_t s_last;
  if (threadIdx.x == 0) {  // the thread that stored the block's totals
    wait_vm();
    const unsigned long long n = __hip_atomic_fetch_add((unsigned long long*)done, v << 24 | 1ull,
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = (n & 0xFFFFFFull) + 1 == nb ? 1u : 0u;
    if (s_last) {
      v += n >> 24;
      *done = 0;  // for the next scan
    }
  }
  __syncthreads();
  return s_last != 0;
}
__device__ __forceinline__ bool last_block(uint64_t* done, uint32_t nb) {
  uint64_t none = 0;
  return last_block(done, nb, none);
}
// part[stride * b] for every block b: totals to exclusive prefixes; returns
// the sum (`own`: this block's total, all there is when it is the only one).
template <int T>
__device__ __forceinline__ uint64_t scan_parts(uint64_t* part, uint32_t stride, uint32_t nb,
                                               uint64_t own, uint64_t* sh) {
  if (nb == 1) {
    if (threadIdx.x == 0) *part = 0;
    return own;
  }
  uint64_t carry = 0;
  for (uint32_t b0 = 0; b0 < nb; b0 += T * 4) {
    uint64_t v[4], sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      const uint32_t b = b0 + threadIdx.x * 4 + i;
      v[i] = b < nb ? __hip_atomic_load(part + (uint64_t)stride * b, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT)
                           : 0;
      sum += v[i];
    }
    uint64_t tot, x = carry + block_scan<T>(sum, sh, tot);
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      const uint32_t b = b0 + threadIdx.x * 4 + i;
      if (b < nb) part[(uint64_t)stride * b] = x;
      x += v[i];
    }
    carry += tot;
  }
  return carry;
}

// Plan of a level, one gate per thread: per gate its leader (the input with
// the most words), words of the leader per tile, tiles and output bound, and
// their prefixes over the level; then, in the block that finishes last, whether
// the level has room, where its scratch lies, and the walk's counters.  A tile
// of a gate of fan-in 1..4 holds 64 times the leader's words of a lane share of
// about seg_target input words, spread evenly over the gate's tiles; a wide
// gate's tiles hold wide_words input words (its tables leave less LDS).
//
// One launch at most: with the plan, two three-kernel scans, the capacity check
// and the clears as launches of their own, a level of the 300-cell netlist spent
// 9 of its 18 launches (25 of 48 us) before its first descriptor.  Every level
// but a chunk's first is planned by blocks of the launch that copies the outputs
// of the level before it (the lengths it reads are final by then).
__device__ __forceinline__ void plan_block(const PlanArgs& A, uint32_t bi, uint32_t nb, uint64_t* sh) {
  if (A.scal[S_TRIP]) return;
  const uint32_t g = bi * kPlanGates + threadIdx.x;
  uint32_t nt = 0;
  uint64_t bound = 0;
  if (g < A.ng) {
    const GateRec& G = A.gates[g];
    const uint32_t tail = A.tail_len[G.out_net];
    uint32_t n6[6];
#pragma unroll
    for (uint32_t j = 0; j < kWideK; ++j) n6[j] = j < G.k ? A.wlen[G.in_net[j]] : 0u;
    uint64_t N = 0;
    uint32_t nl = 0, lead = 0;
#pragma unroll
    for (uint32_t j = 0; j < kWideK; ++j) {
      N += n6[j];
      if (n6[j] > nl) {
        nl = n6[j];
        lead = j;
      }
    }
    // a tile's offset inside its gate's waveform travels in 31 bits
    if (N + 1 >= (1ull << 30)) atomicOr((unsigned int*)(A.scal + S_ERR), ERR_RANGE);
    GatePlan P;
    const uint32_t seg =
        A.spread > 0 ? min(A.seg_target, max(kSpreadSeg, (uint32_t)((float)N * A.spread))) : A.seg_target;
    if (G.k > kTileK) {
      const uint32_t ww = (uint32_t)min<uint64_t>(A.wide_words, (uint64_t)seg * kLanes);
      const uint32_t nt0 = (uint32_t)max<uint64_t>(1, (N + ww - 1) / ww);
      P.lt = max(1u, (nl + nt0 - 1) / nt0);
    } else {
      // (64-bit divisions only where 32 bits do not hold the product)
      uint64_t s = 1;
      if (N > 0)
        s = N < (1ull << 31) && (uint64_t)seg * nl < (1ull << 32)
                ? (uint64_t)(seg * nl / (uint32_t)N)
                : (uint64_t)seg * nl / N;
      if (s < 1) s = 1;
      if (nl > 0) {
        if (s < (1u << 24) && nl < (1u << 31)) {
          const uint32_t t = (uint32_t)s, nt0 = ((nl + t - 1) / t + kLanes - 1) / kLanes;
          s = (nl + nt0 * kLanes - 1) / (nt0 * kLanes);
        } else {
          const uint64_t nt0 = ((nl + s - 1) / s + kLanes - 1) / kLanes;
          s = (nl + nt0 * kLanes - 1) / (nt0 * kLanes);
        }
      }
      P.lt = (uint32_t)min<uint64_t>(s * kLanes, 0xFFFFFFFFu);
    }
    P.lead = lead;
    A.plan[g] = P;
    nt = max(1u, nl / P.lt + (nl % P.lt ? 1u : 0u));
    A.ntile[g] = nt;
    // scratch words of the gate's tile outputs: every tile keeps at most its
    // own input events + 1 entries; the gate's tail is added so that the
    // level's waveforms (tails + joined entries) never exceed the scratch
    bound = N + nt + 1 + tail;
  }
  uint64_t nt_tot, bd_tot;
  const uint64_t t = block_scan<256>(nt, sh, nt_tot);
  const uint64_t b = block_scan<256>(bound, sh, bd_tot);
  if (g < A.ng) {
    A.tile_loc[g] = (uint32_t)t;
    A.scr_loc[g] = b;
  }
  if (threadIdx.x == 0) {
    put_part(A.part + 2 * bi, nt_tot);
    put_part(A.part + 2 * bi + 1, bd_tot);
  }
  if (!last_block(A.scal + S_DONE, nb)) return;
  const uint64_t tiles = scan_parts<256>(A.part, 2, nb, nt_tot, sh);
  const uint64_t scr = scan_parts<256>(A.part + 1, 2, nb, bd_tot, sh);
  if (threadIdx.x < kTickets) A.ticket[threadIdx.x * kTicketStride] = 0;
  if (threadIdx.x != 0) return;
  const uint64_t used = A.scal[S_BUMP], stim = A.scal[S_STIM];
  unsigned why = 0;
  if (A.stop && __hip_atomic_load(A.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)) why = TRIP_STOP;
  if (!why && A.proj_cap > 0 && used > stim) {
    const double proj = (double)(used - stim) * A.all_gates / A.done_gates;
    if (((double)stim + proj) * 1.35 > A.proj_cap) why = TRIP_PROJECTED;
  }
  // The level scratch lies in the unused top of the event pool when twice its
  // size is free above the bump (the level's outputs, at most the scratch size,
  // then land below it); otherwise in an allocation of its own.  (The scratch of
  // the level before, still being copied, is not written before this level's
  // walk.)
  uint32_t* scratch = nullptr;
  if (!why) {
    if (tiles > A.tiles_cap) {
      why = TRIP_ROOM;
    } else if (used <= A.pool_words && 2 * scr <= A.pool_words - used) {
      A.scal[S_LIMIT] = A.pool_words - scr;
      scratch = A.pool + (A.pool_words - scr);
    } else if (A.allow_apart && used + scr <= A.pool_words && scr <= A.apart_cap) {
      A.scal[S_LIMIT] = A.pool_words;
      scratch = A.apart;
    } else {
      why = TRIP_ROOM;
    }
  }
  A.scal[S_TOT_A] = tiles;
  A.scal[S_TOT_B] = scr;
  A.scal[S_NTILES + A.slot] = tiles;
  A.scal[S_SCRATCH + A.slot] = (uint64_t)scratch;
  A.scal[S_OVF_USED] = 0;
  if (why) {
    A.scal[S_WHY] = why;
    // (the copy of the level before goes on: it is below S_TRIP)
    __hip_atomic_store(A.scal + S_TRIP, (uint64_t)A.level, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__global__ __launch_bounds__(256) void k_plan(PlanArgs A) {
  __shared__ uint64_t sh[4];
  plan_block(A, blockIdx.x, gridDim.x, sh);
}

// Words below `key` among the (at most) 8 of a sorted range [p, n) from p on.
__device__ __forceinline__ uint32_t below8(const uint32_t* a, uint32_t p, uint32_t n, uint32_t key) {
  uint32_t v[8], c = 0;
  if (p + 8 <= n) {
    __builtin_memcpy(v, a + p, 32);  // two 16-byte loads
  } else {
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) v[i] = p + i < n ? a[p + i] : 0xFFFFFFFFu;
  }
#pragma unroll
  for (uint32_t i = 0; i < 8; ++i) c += v[i] < key ? 1u : 0u;
  return c;
}

// First index of a sorted word range [0, n) at or after `key` (n if none),
// looked for near `g` (< n): two probes corrected by the density `dens` (words per unit
// of word value), a window of 16 words, then doubling strides away from it and
// a search by halves inside the last one.
//
// The searches of a level's tile boundaries are bound by the cache lines that
// they fetch from HBM and, on small levels, by the chain of dependent loads.
// Event counts follow time closely, so the window is usually the end: about 4
// lines in 3 rounds, against 11 lines in 15 rounds by halves over 20,000 words
// (and 24 lines in 5 rounds with seven probes a round: 93 us a level against
// 72 by halves on the busy 200,000-cell netlist).
__device__ __forceinline__ uint32_t lb_near(const uint32_t* a, uint32_t n, uint32_t key, uint32_t g,
                                            float dens) {
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const uint32_t v = a[g];
    const float d = v < key ? (float)(key - v) : -(float)(v - key);
    const float x = (float)g + d * dens;
    g = (uint32_t)max(0.0f, min(x, (float)(n - 1)));
    g = min(g, n - 1);
  }
  uint32_t s = g > 8 ? g - 8 : 0u;
  const uint32_t c0 = below8(a, s, n, key), c1 = s + 8 < n ? below8(a, s + 8, n, key) : 0u;
  const uint32_t c = c0 + c1;
  if (c > 0 && c < 16) return s + c;
  uint32_t lo, hi;  // every word before lo is below key, a[hi] is not (or hi = n)
  if (c == 0) {
    if (s == 0) return 0;
    uint32_t d = 16;
    hi = s;
    for (;;) {
      lo = 0;
      if (d > hi) break;
      if (a[hi - d] < key) {
        lo = hi - d + 1;
        break;
      }
      hi -= d;
      d <<= 1;
    }
  } else {
    uint32_t d = 16;
    lo = s + 16;
    for (;;) {
      hi = n;
      if (n - lo < d) break;
      hi = lo + d - 1;
      if (a[hi] >= key) break;
      lo = hi + 1;
      d <<= 1;
    }
  }
  return lo + lb_words(a + lo, hi - lo, key);
}

// Per tile: its descriptor; thread j of the tile's four takes inputs j and
// j + 4.  Bound by the latency of a chain of dependent loads (gate, lengths,
// the boundary's time, the searches).  A block describes 63 tiles: the threads of the 64th only find where
// its inputs start, which is where the 63rd ends.
__global__ __launch_bounds__(256) void k_tile_desc(
    const GateRec* __restrict__ gates, uint32_t ng, const GatePlan* __restrict__ plan,
    const uint32_t* __restrict__ tile_loc, const uint64_t* __restrict__ scr_loc,
    const uint64_t* __restrict__ part, const uint64_t* __restrict__ woff,
    const uint32_t* __restrict__ wlen, const uint32_t* __restrict__ pool,
    TileDesc* __restrict__ tiles, const uint64_t* __restrict__ scal, uint32_t slot) {
  constexpr uint32_t kRow = kDescTiles;  // row that only marks the end
  // a tile's first own word of each input is the previous tile's end: the
  // block's tiles pass them on through LDS (each boundary searched once)
  __shared__ uint32_t s_first[2][256];
  __shared__ int32_t s_start[2 * kPlanGates];  // first tiles of the gates near, from t0
  __shared__ uint32_t s_n[4];
  if (scal[S_TRIP]) return;
  const uint64_t nt = scal[S_NTILES + slot];
  const uint32_t nb = (ng + kPlanGates - 1) / kPlanGates;
  const uint32_t row = threadIdx.x >> 2, wid = threadIdx.x >> 6;
  for (uint64_t t0 = (uint64_t)blockIdx.x * kDescTiles; t0 < nt; t0 += (uint64_t)gridDim.x * kDescTiles) {
    const uint64_t t = t0 + row;
    const int j0 = (int)(threadIdx.x & 3);
    const bool valid = t < nt;
    // the plan's block with tile t0: the whole block probes
    uint32_t b0 = 0, len = nb;
    while (len > 1) {
      const uint32_t st = (len + 255) / 256, at = threadIdx.x * st;
      const uint64_t le = __ballot(at < len && part[2 * (b0 + (at < len ? at : 0u))] <= t0);
      if ((threadIdx.x & 63) == 0) s_n[wid] = (uint32_t)__popcll(le);
      __syncthreads();
      const uint32_t c = max(s_n[0] + s_n[1] + s_n[2] + s_n[3], 1u) - 1;
      __syncthreads();
      b0 += c * st;
      len = min(st, len - c * st);
    }
    // the tiles here are of its gates and of the next block's (every gate has
    // at least one): the last gate that starts at or before the tile
    __syncthreads();  // the block's tiles before these are done with s_first, s_start
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) {
      const uint32_t g = (b0 + q) * kPlanGates + threadIdx.x;
      int32_t s = 0x7FFFFFFF;
      if (g < ng) {
        const int64_t rel = (int64_t)(part[2 * (b0 + q)] + tile_loc[g]) - (int64_t)t0;
        s = (int32_t)max((int64_t)-0x7FFFFFFF, min(rel, (int64_t)0x7FFFFFFF));
      }
      s_start[q * kPlanGates + threadIdx.x] = s;
    }
    __syncthreads();
    uint32_t gl = 0;
#pragma unroll
    for (uint32_t st = kPlanGates; st; st >>= 1)
      if (s_start[gl + st] <= (int32_t)row) gl += st;
    const uint32_t g = valid ? b0 * kPlanGates + gl : 0u;
    const uint32_t ti = (uint32_t)((int32_t)row - s_start[gl]);
    GateRec G;
    GatePlan P;
    uint32_t nl = 0, L[2] = {0, 0}, n2[2] = {0, 0}, tau_nx = 0;
    uint64_t off2[2] = {0, 0};
    const uint32_t* lw = nullptr;
    bool more = false;  // another tile of the gate follows
    if (valid) {
      G = gates[g];
      P = plan[g];
      lw = pool + woff[G.in_net[P.lead]];
      nl = wlen[G.in_net[P.lead]];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint32_t j = j0 + 4 * q;
        if (j >= G.k) continue;
        off2[q] = woff[G.in_net[j]];
        n2[q] = wlen[G.in_net[j]];
      }
      more = (ti + 1) * (uint64_t)P.lt < nl;
      const uint32_t tau_lo = ti > 0 ? lw[ti * P.lt] >> 2 : 0u;
      tau_nx = more ? lw[(ti + 1) * P.lt] >> 2 : 0u;
      if (ti > 0) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const uint32_t j = j0 + 4 * q;
          if (j >= G.k) continue;
          const uint32_t x = ti * P.lt, n = n2[q];
          const float at = (float)x * ((float)n / (float)nl);
          L[q] = j == P.lead ? x
                 : n == 0    ? 0u
                             : lb_near(pool + off2[q], n, tau_lo << 2, min((uint32_t)at, n - 1),
                                       at / (float)(tau_lo << 2));
        }
      }
    }
    s_first[0][threadIdx.x] = L[0];
    s_first[1][threadIdx.x] = L[1];
    __syncthreads();
    if (!valid || row == kRow) continue;
    TileDesc& D = tiles[t];
    const uint32_t dtw = walk_dt_words(G.walk, G.k), ttw = walk_tt_words(G.walk, G.k);
    uint32_t slot8[2] = {0, 0}, nq[2] = {0, 0}, in_lo8[2] = {0, 0};
    // own input words of the tile (up to the next tile's first words), summed
    // over the tile's threads: its output region in the level scratch holds
    // that many entries plus one
    uint32_t span = 0, own = 0, xend = 0, dead = 0, lsum = 0, hi8[2] = {0, 0};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint32_t j = j0 + 4 * q;
      if (j >= G.k) {
        if (j < kWideK) {
          D.in_lo[j] = 0;
          D.n[j] = 0;
        }
        continue;
      }
      const uint64_t off = off2[q];
      const uint32_t n = n2[q];
      const uint32_t* iw = pool + off;
      uint32_t E = n, Ln = n;
      if (more) {
        // the next tile is this gate's: its first words end this one
        Ln = s_first[q][threadIdx.x + 4];
        // halo end: the first word at or after tau_nx + dmax lies at or a few
        // words after Ln; eight at once, then doubling strides and a search
        // inside the last stride (every word before a is below the key)
        const uint32_t key = (tau_nx + G.dmax) << 2;
        const uint32_t c = below8(iw, Ln, n, key);
        E = Ln + c;
        if (c == 8) {
          uint32_t a = E - 1, d = 8, b = a + d;
          while (b < n && iw[b] < key) {
            a = b;
            d <<= 1;
            b = a + d;
          }
          if (b > n) b = n;
          E = a + 1 + lb_words(iw + a + 1, b - a - 1, key);
        }
        if (j == P.lead) xend = (ti + 1) * P.lt - (L[q] > 0 ? L[q] - 1 : 0u);
      }
      const uint32_t B = L[q] > 0 ? L[q] - 1 : 0u;
      D.in_lo[j] = in_lo8[q] = (uint32_t)(off + B);
      D.n[j] = nq[q] = E - B;
      slot8[q] = range_words(in_lo8[q], E - B);
      hi8[q] = (uint32_t)((off + B) >> 32) << (8 * j0);
      span += Ln - L[q];
      own += Ln - max(L[q], 1u);
      lsum += L[q];
      dead |= n == 0 ? 1u : 0u;
    }
#pragma unroll
    for (int d = 1; d < 4; d <<= 1) {
      span += __shfl_xor(span, d);
      own += __shfl_xor(own, d);
      xend |= __shfl_xor(xend, d);
      dead |= __shfl_xor(dead, d);
      lsum += __shfl_xor(lsum, d);
      hi8[0] |= __shfl_xor(hi8[0], d);
      hi8[1] |= __shfl_xor(hi8[1], d);
    }
    // where the ranges start in LDS: the slots before, and the words that the
    // first one's 16-byte copies bring before it
    uint32_t words = nq[0] + nq[1], at[2];
    words += __shfl_xor(words, 1);
    words += __shfl_xor(words, 2);
    const uint32_t b1 = __shfl_up(slot8[0], 1, 4), b2 = __shfl_up(slot8[0], 2, 4), b3 = __shfl_up(slot8[0], 3, 4);
    uint32_t all4 = slot8[0] + __shfl_xor(slot8[0], 1);
    all4 += __shfl_xor(all4, 2);
    at[0] = dtw + ttw + (j0 > 0 ? b1 : 0u) + (j0 > 1 ? b2 : 0u) + (j0 > 2 ? b3 : 0u) + (in_lo8[0] & 3u);
    const uint32_t c0 = __shfl(slot8[1], 0, 4);
    at[1] = dtw + ttw + all4 + (j0 > 0 ? c0 : 0u) + (in_lo8[1] & 3u);
    uint32_t pair[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) pair[q] = (at[q] & 0xFFFFu) | __shfl_down(at[q], 1, 4) << 16;
    if (j0 == 0 || j0 == 2) D.at2[j0 / 2] = pair[0];
    if (j0 == 0) {
      D.at2[2] = pair[1];
      D.words = words;
      D.tab = dtw | ttw << 16;
      D.in_hi[0] = hi8[0];
      D.in_hi[1] = hi8[1];
      // a gate's region, then the tile's first own event in the gate's merged
      // input order plus one slack word per earlier tile (a tile keeps at most
      // its own events + 1 entries)
      const uint64_t scr = part[2 * (g / kPlanGates) + 1] + scr_loc[g] + ti + lsum;
      D.scr_lo = (uint32_t)scr;
      D.scr_hi = (uint32_t)(scr >> 32);
      D.own = dead ? 0u : own;
      D.xend = xend;
      D.meta = (dead ? (uint32_t)W_DEAD : (uint32_t)G.walk) | ((uint32_t)G.k << 4) | (P.lead << 8) |
               ((ti == 0 ? 1u : 0u) << 12) | (G.edge_in << 16);
      D.dt_off = G.dt_off;
      D.tt_off = G.tt_off;
      D.dmax = G.dmax;
      D.job = G.job;
      D.out_cap = span + 1;
      D.g = g;
      D.ti = ti;
      D.out_net = G.out_net;
    }
  }
}

// Per gate, in tile order: join the tiles' outputs (a tile whose first
// entry repeats the last value before it drops that entry), place each
// tile's output (offset inside the gate, bit 31: first entry dropped), and
// add up the SAIF durations between tiles and from the last entry to the window
// end (the copy adds those inside tiles).  Eight lanes per gate, 8 tiles per step: each
// lane takes the last value and time of the nearest non-empty tile before
// it (a ballot of the non-empty lanes, then a shuffle; the step's first
// non-empty tile takes them from the previous step), the offsets are an
// exclusive scan of the joined counts, and the sums are reduced at the end.
// (A wavefront per gate left most lanes idle: gates have 2 to 40 tiles.)  In a
// batch (ev_job set) the gates' events are added to their instance's count
// for the chunk, one atomic per block of one instance (one per gate held the
// batching mix's joins to 88 us a level).
//
// The block that finishes last places the gates in the pool and closes the
// level: bump pointer, gate events, or a trip when the level ran out of
// overflow stacks.
__global__ __launch_bounds__(8 * kJoinGates) void k_join(JoinArgs A, TailArgs T) {
  constexpr int kThreads = 8 * kJoinGates;
  __shared__ uint64_t sh[kThreads / 64], s_all[kThreads / 64];
  __shared__ uint32_t s_job[kJoinGates];
  __shared__ unsigned long long s_ev[kJoinGates];
  if (A.scal[S_TRIP]) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    A.scal[S_EVAL] += (uint64_t)wall_clock64() - A.scal[S_CLOCK];
    A.scal[S_LEVELS] += 1;
    A.scal[S_TILES] += A.scal[S_NTILES + A.slot];
  }
  const uint32_t grp = threadIdx.x >> 3, l8 = threadIdx.x & 7u;
  const int sh8 = (int)(threadIdx.x & 56u);  // the group's first lane in its wavefront
  const uint32_t g = blockIdx.x * kJoinGates + grp;
  uint32_t words = 0;  // the gate's, in its first lane
  uint64_t ev = 0;     // events of the lane's tiles
  if (l8 == 0) {
    s_ev[grp] = 0;
    s_job[grp] = 0xFFFFFFFFu;
  }
  if (g < A.ng) {
    const GateRec& G = A.gates[g];
    const ChunkWin W = A.cwin[G.job];
    const unsigned long long start = W.lo, end = W.hi;
    const uint64_t t0 = A.plan_part[2 * (g / kPlanGates)] + A.tile_loc[g];
    const uint32_t n = A.ntile[g];
    // carried from the previous step: count so far, last value and time.  The
    // gate's waveform starts with its tail (state entry and look-back
    // entries); after chunk 0 the first new entry is compared with the tail's
    // last value, which holds from before the chunk (time 0 is clipped to
    // the chunk's SAIF start).
    const uint32_t tl = T.tail_len[G.out_net];
    uint32_t cnt = tl, lv = 0, lt = 0, has = 0, any = 0;
    if (!T.first && tl) {
      lv = T.tails[T.tail_off[G.out_net] + tl - 1] & 3u;
      has = 1;
    }
    unsigned long long acc[3] = {0, 0, 0}, tc = 0, gev = 0;
    for (uint32_t c = 0; c < n; c += 8) {
      const bool in = c + l8 < n;
      const uint64_t t = t0 + c + l8;
      TileOut S = {};
      if (in) S = A.tout[t];
      const bool ne = S.cnt != 0;
      const uint32_t mask = (uint32_t)(__ballot(ne) >> sh8) & 0xFFu;
      const uint32_t my_lv = S.last & 3u, my_lt = S.last >> 2, my_fv = S.first & 3u, my_ft = S.first >> 2;
      // nearest non-empty tile below this lane in the step, if any
      const uint32_t below = mask & ((1u << l8) - 1u);
      const int pl = below ? 31 - __clz((int)below) : 0;
      const uint32_t s_lv = __shfl(my_lv, pl, 8), s_lt = __shfl(my_lt, pl, 8);
      const uint32_t p_has = below ? 1u : has;
      const uint32_t p_lv = below ? s_lv : lv, p_lt = below ? s_lt : lt;
      uint32_t mine = 0, skip = 0;
      if (ne) {
        skip = (p_has && p_lv == my_fv) ? 1u : 0u;
        mine = S.cnt - skip;
        if (p_has) saif_acc(acc, p_lv, p_lt, my_ft, start, end);
        // the tile's first entry against the previous tile's last value
        tc += (p_has && is_toggle(p_lv, my_fv) && my_ft > W.tc_lo && my_ft <= W.tc_hi) ? 1u : 0u;
      }
      // an instance counts the events of its tiles with entries; the tiles of a
      // wide gate count as one
      gev += ne || G.k > kTileK ? S.ev : 0u;
      ev += S.ev;
      any |= mask;
      // inclusive scan of the joined counts over the step
      uint32_t incl = mine;
#pragma unroll
      for (int d = 1; d < 8; d <<= 1) {
        const uint32_t v = __shfl_up(incl, d, 8);
        if ((int)l8 >= d) incl += v;
      }
      if (in) A.tile_off[t] = (cnt + incl - mine) | (skip << 31);
      cnt += __shfl(incl, 7, 8);
      if (mask) {  // the step's last non-empty tile carries on
        const int ll = 31 - __clz((int)mask);
        lv = __shfl(my_lv, ll, 8);
        lt = __shfl(my_lt, ll, 8);
        has = 1;
      }
    }
    if (has && l8 == 0) saif_acc(acc, lv, lt, end > lt ? end : (unsigned long long)lt, start, end);
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) {
      acc[0] += __shfl_xor(acc[0], d, 8);
      acc[1] += __shfl_xor(acc[1], d, 8);
      acc[2] += __shfl_xor(acc[2], d, 8);
      tc += __shfl_xor(tc, d, 8);
      gev += __shfl_xor(gev, d, 8);
    }
    if (l8 == 0) {
      words = cnt;
      s_job[grp] = G.job;
      s_ev[grp] = any ? gev : 0ull;
      A.wlen[G.out_net] = cnt;
      unsigned long long* sa = A.saif + (uint64_t)kSaifWords * G.out_net;
      sa[0] = acc[0];
      sa[1] = acc[1];
      sa[2] = acc[2];
      sa[3] = tc;
    }
  }
  const unsigned int err = *(const unsigned int*)(A.scal + S_ERR);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) ev += __shfl_xor(ev, d);
  if ((threadIdx.x & 63) == 0) s_all[threadIdx.x >> 6] = ev;
  uint64_t own;  // the block's words
  const uint64_t x = block_scan<kThreads>(words, sh, own);  // (its barriers: s_all, s_ev, s_job)
  if (l8 == 0 && g < A.ng) A.out_loc[g] = x;
  uint64_t events = 0;
  if (threadIdx.x == 0) {
    put_part(A.part + blockIdx.x, own);
#pragma unroll
    for (int i = 0; i < kThreads / 64; ++i) events += s_all[i];
  }
  // a level whose tiles ran out of overflow stacks runs again: counted then
  if (A.ev_job && !(err & ERR_OVERFLOW) && threadIdx.x < 64) {
    const uint32_t i = threadIdx.x;
    const uint32_t job = i < kJoinGates ? s_job[i] : 0xFFFFFFFFu;
    unsigned long long e = i < kJoinGates ? s_ev[i] : 0ull;
    const uint32_t job0 = __shfl(job, 0, 64);
    if (__ballot(job != job0 && job != 0xFFFFFFFFu)) {
      if (job != 0xFFFFFFFFu && e) atomicAdd(A.ev_job + job, e);
    } else {
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) e += __shfl_xor(e, d);
      if (i == 0 && e) atomicAdd(A.ev_job + job0, e);
    }
  }
  if (!last_block(A.scal + S_DONE, gridDim.x, events)) return;
  const uint64_t total = scan_parts<kThreads>(A.part, 1, gridDim.x, own, sh);
  if (threadIdx.x != 0) return;
  if (A.ovf_trip && (err & ERR_OVERFLOW)) {
    A.scal[S_TRIP] = A.level;
    A.scal[S_WHY] = TRIP_OVERFLOW;
    return;
  }
  const uint64_t base = A.scal[S_BUMP];
  if (base + total > A.scal[S_LIMIT]) {  // (outputs never exceed the scratch's size)
    atomicOr((unsigned int*)(A.scal + S_ERR), ERR_CAPACITY | ERR_POOL);
    A.scal[S_TRIP] = A.level;
    A.scal[S_WHY] = TRIP_POOL;
    return;
  }
  A.scal[S_OUTBASE] = base;
  A.scal[S_BUMP] = base + total;
  A.scal[S_EVC] += events;
}

// Copy every tile's joined output from the scratch into the gate's dense
// waveform in the pool (one wavefront per tile, coalesced); the gate's first
// tile also copies the gate's tail (state and look-back entries, moved to
// this chunk's time base) to the front.  On its way every entry adds its SAIF
// durations (and toggles when asked) to its net's record: the copy waits for
// memory, and the walk that left the entries waits for its VALU.  The first nplan
// blocks plan the next level.
__global__ __launch_bounds__(256) void k_compact(CompactArgs A, TailArgs T, PlanArgs next,
                                                 uint32_t nplan) {
  __shared__ uint64_t sh[4];
  if (blockIdx.x < nplan) {
    plan_block(next, blockIdx.x, nplan, sh);
    return;
  }
  // a trip of this level or one before it; the next one's plan may trip now
  const uint64_t trip = __hip_atomic_load(A.scal + S_TRIP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (trip && trip <= A.level) return;
  const TileDesc* __restrict__ tiles = A.tiles;
  const TileOut* __restrict__ tout = A.tout;
  const uint32_t* __restrict__ tile_off = A.tile_off;
  uint32_t* __restrict__ pool = A.pool;
  const int lane = threadIdx.x & 63;
  const uint32_t bi = blockIdx.x - nplan;
  const uint64_t waves = (uint64_t)(gridDim.x - nplan) * (blockDim.x / 64);
  const uint64_t nt = A.scal[S_NTILES + A.slot], base = A.scal[S_OUTBASE];
  const glb_u32* scratch = (const glb_u32*)A.scal[S_SCRATCH + A.slot];
  for (uint64_t t = (uint64_t)bi * (blockDim.x / 64) + threadIdx.x / 64; t < nt; t += waves) {
    const TileDesc& D = tiles[t];
    const uint64_t gate = base + A.part[D.g / kJoinGates] + A.out_loc[D.g];
    if (D.ti == 0) {
      if (lane == 0) A.woff[D.out_net] = gate;
      const uint32_t tl = T.tail_len[D.out_net];
      const uint32_t* ts = T.tails + T.tail_off[D.out_net];
      uint32_t* td = pool + gate;
      for (uint32_t q = lane; q < tl; q += 64) {
        const uint32_t w = ts[q], tt = w >> 2;
        td[q] = ((tt > T.shift ? tt - T.shift : 0u) << 2) | (w & 3u);
      }
    }
    const TileOut S = tout[t];
    if (!S.cnt) continue;
    const uint32_t off = tile_off[t] & 0x7FFFFFFFu, skip = tile_off[t] >> 31;
    const uint32_t n = S.cnt - skip;
    const glb_u32* src = scratch + (((uint64_t)D.scr_hi << 32) | D.scr_lo) + skip;
    uint32_t* dst = pool + gate + off;
    const ChunkWin W = A.cwin[D.job];
    // SAIF durations between the tile's entries, in 32 bits (times < 2^30; a
    // lane's intervals are disjoint pieces of the tile's span): an entry ends the
    // interval of the one before it, which is the lane's below, and lane 0's is
    // the last of the 64 entries before
    const uint32_t s32 = (uint32_t)min(W.lo, 0x7FFFFFFFull);
    const uint32_t e32 = (uint32_t)min(W.hi, 0x7FFFFFFFull);
    uint32_t carry = S.first, a0 = 0, a3 = 0, tc = 0;
    auto add = [&](uint32_t p, uint32_t e) {
      const uint32_t len = max(min(e >> 2, e32), s32) - max(min(p >> 2, e32), s32), pv = p & 3u;
      a0 += pv == 0u ? len : 0u;
      a3 += pv == 3u ? len : 0u;
      // SAIF TC: 0<->1 changes (the first entry against the tile before is the join's)
      if (A.count_tc) {
        const unsigned long long tt = e >> 2;
        tc += (is_toggle(pv, e & 3u) && tt > W.tc_lo && tt <= W.tc_hi) ? 1u : 0u;
      }
    };
    // four entries a lane in one access, four accesses in flight: a tile of
    // 1,000 entries waits for memory once.  (The copy is bound by those waits: a
    // wavefront's chain is descriptor, place, entries.)
    const uint32_t n4 = n / 4;
    for (uint32_t b = 0; b < n4; b += 256) {
      const uint32_t left = n4 - b;
      u32x4 w[4];
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i)
        if (64 * i + lane < left) w[i] = ((const glb_u32x4*)src)[b + 64 * i + lane];
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        if (64 * i >= left) break;
        const bool in = 64 * i + lane < left;
        if (in) *(u32x4*)(dst + 4 * (b + 64 * i + lane)) = w[i];
        // (lanes behind the end repeat the entry before, which adds nothing)
        const uint32_t p = dpp<0x138>(w[i].w, carry);
        carry = __builtin_amdgcn_readlane(w[i].w, min(left - 64 * i, 64u) - 1);
        const uint32_t e0 = in ? w[i].x : p, e1 = in ? w[i].y : p, e2 = in ? w[i].z : p;
        add(p, e0);
        add(e0, e1);
        add(e1, e2);
        add(e2, in ? w[i].w : p);
      }
    }
    if (n & 3u) {
      const uint32_t e = 4 * n4 + lane < n ? src[4 * n4 + lane] : S.last;
      if (4 * n4 + lane < n) dst[4 * n4 + lane] = e;
      add(dpp<0x138>(e, carry), e);
    }
    const uint32_t t0 = wave_sum(a0), t1 = wave_sum(a3);
    // the intervals between the tile's entries add up to its span
    const uint32_t span = max(min(S.last >> 2, e32), s32) - max(min(S.first >> 2, e32), s32);
    if (A.count_tc) tc = wave_sum(tc);
    const uint32_t v = lane == 0 ? t0 : (lane == 1 ? t1 : (lane == 2 ? span - t0 - t1 : tc));
    if (lane < (int)kSaifWords && v)
      atomicAdd(A.saif + (uint64_t)kSaifWords * D.out_net + lane, (unsigned long long)v);
  }
}

// ------------------------------------------------------- stimulus and tails ---

// first index of a sorted 64-bit word range whose time (word >> 2) is at or
// after `t`
__device__ __forceinline__ uint32_t lb_time64(const uint64_t* a, uint32_t n, uint64_t t) {
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if ((a[mid] >> 2) < t) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Per stimulus signal: the range [lb, ub) of its resident waveform, the chunk
// words it needs (one state entry + the range) and their prefixes; the chunk
// trips when its stimulus does not leave the pool 1,024 words.
__global__ __launch_bounds__(256) void k_stim_plan(const uint64_t* __restrict__ store,
                                                   const uint64_t* __restrict__ soff,
                                                   const uint32_t* __restrict__ slen, uint32_t ns,
                                                   uint64_t lb, uint64_t ub, uint64_t* __restrict__ cnt,
                                                   uint32_t* __restrict__ first,
                                                   uint64_t* __restrict__ loc, uint64_t* __restrict__ part,
                                                   uint64_t pool_words, uint64_t* __restrict__ scal) {
  __shared__ uint64_t sh[4];
  if (scal[S_TRIP]) return;
  const uint32_t s = blockIdx.x * kStimSignals + threadIdx.x;
  uint64_t n = 0;
  if (s < ns) {
    const uint64_t* w = store + soff[s];
    const uint32_t len = slen[s];
    const uint32_t i = lb ? lb_time64(w, len, lb) : 0u;
    const uint32_t j = lb_time64(w, len, ub);
    first[s] = i;
    n = 1ull + (j - i);
    cnt[s] = n;
  }
  uint64_t tot;
  const uint64_t x = block_scan<256>(n, sh, tot);
  if (s < ns) loc[s] = x;
  if (threadIdx.x == 0) put_part(part + blockIdx.x, tot);
  if (!last_block(scal + S_DONE, gridDim.x)) return;
  const uint64_t total = scan_parts<256>(part, 1, gridDim.x, tot, sh);
  if (threadIdx.x != 0) return;
  scal[S_BUMP] = scal[S_STIM] = total;
  if (total + 1024 > pool_words) {
    scal[S_TRIP] = 1;  // before every level
    scal[S_WHY] = TRIP_STIM;
  }
}

// One block per stimulus signal: state entry at relative time 0, then the range
// in relative time (abs - lb + 1 >= 1); sets the net's waveform.
__global__ __launch_bounds__(256) void k_stim_copy(
    const uint64_t* __restrict__ store, const uint64_t* __restrict__ soff,
    const uint32_t* __restrict__ snet, uint64_t lb, const uint64_t* __restrict__ cnt,
    const uint32_t* __restrict__ first, const uint64_t* __restrict__ loc,
    const uint64_t* __restrict__ part, uint32_t* __restrict__ pool, uint64_t* __restrict__ woff,
    uint32_t* __restrict__ wlen, const uint64_t* __restrict__ scal) {
  if (scal[S_TRIP]) return;
  const uint32_t s = blockIdx.x;
  const uint64_t base = part[s / kStimSignals] + loc[s];
  const uint64_t* w = store + soff[s] + first[s];
  const uint32_t n = (uint32_t)(cnt[s] - 1);
  uint32_t* d = pool + base;
  if (threadIdx.x == 0) {
    d[0] = first[s] > 0 ? (uint32_t)(w[-1] & 3u) : 1u;  // X before the first entry
    woff[snet[s]] = base;
    wlen[snet[s]] = n + 1;
  }
#pragma unroll 4
  for (uint64_t q = threadIdx.x; q < n; q += 256) {
    const uint64_t e = w[q];
    d[1 + q] = (uint32_t)((((e >> 2) - lb + 1) << 2) | (e & 3u));
  }
}

// End of chunk k, per gate output: where its tail for chunk k+1 starts in
// its chunk waveform (relative time of chunk k): the last entry before
// `key` (lb_k+1 in chunk k's time; index 0, the state entry, is below it)
// and everything after it.  Tails are short, so the search gallops back
// from the end.  Their prefixes place them in the tail store.
__global__ __launch_bounds__(256) void k_tail_len(const GateRec* __restrict__ gates, uint32_t ng,
                                                  const uint64_t* __restrict__ woff,
                                                  const uint32_t* __restrict__ wlen,
                                                  const uint32_t* __restrict__ pool, uint32_t key,
                                                  uint64_t* __restrict__ len, uint64_t* __restrict__ src,
                                                  uint64_t* __restrict__ loc, uint64_t* __restrict__ part,
                                                  uint64_t* __restrict__ scal) {
  __shared__ uint64_t sh[4];
  if (scal[S_TRIP]) return;
  const uint32_t kw = key << 2;
  const uint32_t g = blockIdx.x * kPlanGates + threadIdx.x;
  uint64_t mine = 0;
  if (g < ng) {
    const uint32_t net = gates[g].out_net;
    const uint32_t* w = pool + woff[net];
    const uint32_t n = wlen[net];
    // w[lo] < kw; every index at or after hi is >= kw (hi = n: none checked)
    uint32_t lo = 0, hi = n, d = 1;
    while (hi > lo + 1) {
      const uint32_t p = hi - min(d, hi - lo - 1);
      if (w[p] < kw) {
        lo = p;
        break;
      }
      hi = p;
      d <<= 1;
    }
    while (hi > lo + 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (w[mid] < kw) lo = mid;
      else hi = mid;
    }
    mine = n - lo;
    len[g] = mine;
    src[g] = woff[net] + lo;
  }
  uint64_t tot;
  const uint64_t x = block_scan<256>(mine, sh, tot);
  if (g < ng) loc[g] = x;
  if (threadIdx.x == 0) put_part(part + blockIdx.x, tot);
  if (!last_block(scal + S_DONE, gridDim.x)) return;
  const uint64_t total = scan_parts<256>(part, 1, gridDim.x, tot, sh);
  if (threadIdx.x == 0) scal[S_TAILS] = total;
}

// Copies each gate output's tail into the tail store (kept in chunk k's
// relative time; k_compact moves it to chunk k+1's).  A store too small for
// the chunk (a replayed sequence that outgrew its first run) flags
// ERR_CAPACITY and copies nothing past its end.
__global__ void k_tail_copy(const GateRec* __restrict__ gates, uint32_t ng,
                            const uint64_t* __restrict__ len, const uint64_t* __restrict__ src,
                            const uint64_t* __restrict__ loc, const uint64_t* __restrict__ part,
                            const uint32_t* __restrict__ pool, uint32_t* __restrict__ tails,
                            uint64_t cap, uint32_t* __restrict__ tail_len,
                            uint64_t* __restrict__ tail_off, uint64_t* __restrict__ scal) {
  if (scal[S_TRIP]) return;
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ng) return;
  const uint32_t net = gates[g].out_net;
  const uint64_t n = len[g], o = part[g / kPlanGates] + loc[g];
  if (o + n > cap) {
    atomicOr((unsigned int*)(scal + S_ERR), ERR_CAPACITY);
    tail_len[net] = 0;
    tail_off[net] = 0;
    return;
  }
  const uint32_t* s = pool + src[g];
  for (uint64_t q = 0; q < n; ++q) tails[o + q] = s[q];
  tail_len[net] = (uint32_t)n;
  tail_off[net] = o;
}

// Start of a run: scalars, SAIF counters, waveform lengths and instance event
// counts to zero.
__global__ void k_run_begin(uint64_t* scal, unsigned long long* saif, uint64_t n_saif,
                            unsigned long long* wtot, uint64_t n_nets, unsigned long long* evjob,
                            uint64_t n_jobs) {
  const uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
  if (i0 < S_COUNT) scal[i0] = 0;
  for (uint64_t i = i0; i < n_saif; i += step) saif[i] = 0;
  for (uint64_t i = i0; i < n_nets; i += step) wtot[i] = 0;
  if (evjob)
    for (uint64_t i = i0; i < n_jobs; i += step) evjob[i] = 0;
}

// End of a run: waveform words read by the gates and written by them (wtot:
// whole-run waveform lengths of every net).
__global__ __launch_bounds__(256) void k_word_counts(const GateRec* __restrict__ gates, uint32_t ng,
                                                     const unsigned long long* __restrict__ wtot,
                                                     uint64_t* __restrict__ scal) {
  __shared__ uint64_t sh[4];
  if (scal[S_TRIP]) return;
  uint64_t in = 0, out = 0;
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < ng; g += gridDim.x * blockDim.x) {
    const GateRec& G = gates[g];
    for (int j = 0; j < G.k; ++j) in += wtot[G.in_net[j]];
    out += wtot[G.out_net];
  }
  uint64_t ti, to;
  block_scan<256>(in, sh, ti);
  block_scan<256>(out, sh, to);
  if (threadIdx.x == 0) {
    atomicAdd((unsigned long long*)(scal + S_IN_W), (unsigned long long)ti);
    atomicAdd((unsigned long long*)(scal + S_OUT_W), (unsigned long long)to);
  }
}

__global__ void k_fill_u64(unsigned long long* p, uint64_t n, unsigned long long v) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ------------------------------------------------------- launch helpers ----

static inline unsigned nblk(uint64_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

hipError_t launch_plan(const PlanArgs& a, hipStream_t st) {
  if (a.ng == 0) return hipSuccess;
  k_plan<<<nblk(a.ng, kPlanGates), 256, 0, st>>>(a);
  return hipGetLastError();
}

// `guess`: expected tiles, for the launch width alone
hipError_t launch_tile_desc(const GateRec* gates, uint32_t ng, const GatePlan* plan,
                            const uint32_t* tile_loc, const uint64_t* scr_loc, const uint64_t* part,
                            const uint64_t* woff, const uint32_t* wlen, const uint32_t* pool,
                            TileDesc* tiles, const uint64_t* scal, uint32_t slot, uint64_t guess,
                            hipStream_t st) {
  const unsigned nb = (unsigned)std::min<uint64_t>(guess / kDescTiles + 1, 8192);
  k_tile_desc<<<nb, 256, 0, st>>>(gates, ng, plan, tile_loc, scr_loc, part, woff, wlen, pool, tiles,
                                  scal, slot);
  return hipGetLastError();
}

hipError_t launch_fill_u64(unsigned long long* p, uint64_t n, unsigned long long v,
                           hipStream_t st) {
  if (n == 0) return hipSuccess;
  k_fill_u64<<<nblk(n, 256), 256, 0, st>>>(p, n, v);
  return hipGetLastError();
}

hipError_t launch_join(const JoinArgs& a, const TailArgs& T, hipStream_t st) {
  if (a.ng == 0) return hipSuccess;
  k_join<<<nblk(a.ng, kJoinGates), 8 * kJoinGates, 0, st>>>(a, T);
  return hipGetLastError();
}

// `next`: the plan of the level after it (null: none)
hipError_t launch_compact(const CompactArgs& a, const TailArgs& T, const PlanArgs* next, uint64_t guess,
                          hipStream_t st) {
  const unsigned nb = (unsigned)std::min<uint64_t>(guess / 4 + 1, 8192);  // 4 wavefronts each
  const unsigned np = next ? nblk(next->ng, kPlanGates) : 0;
  k_compact<<<nb + np, 256, 0, st>>>(a, T, next ? *next : PlanArgs{}, np);
  return hipGetLastError();
}

hipError_t launch_run_begin(uint64_t* scal, unsigned long long* saif, uint64_t n_saif,
                            unsigned long long* wtot, uint64_t n_nets, unsigned long long* evjob,
                            uint64_t n_jobs, hipStream_t st) {
  const unsigned nb = (unsigned)std::min<uint64_t>(nblk(std::max<uint64_t>(n_saif, S_COUNT), 256), 2048);
  k_run_begin<<<nb, 256, 0, st>>>(scal, saif, n_saif, wtot, n_nets, evjob, n_jobs);
  return hipGetLastError();
}

hipError_t launch_word_counts(const GateRec* gates, uint32_t ng, const unsigned long long* wtot,
                              uint64_t* scal, hipStream_t st) {
  if (ng == 0) return hipSuccess;
  k_word_counts<<<std::min(nblk(ng, 256), 1024u), 256, 0, st>>>(gates, ng, wtot, scal);
  return hipGetLastError();
}

hipError_t launch_stim_plan(const uint64_t* store, const uint64_t* soff, const uint32_t* slen,
                            uint32_t ns, uint64_t lb, uint64_t ub, uint64_t* cnt, uint32_t* first,
                            uint64_t* loc, uint64_t* part, uint64_t pool_words, uint64_t* scal,
                            hipStream_t st) {
  k_stim_plan<<<std::max(1u, nblk(ns, kStimSignals)), 256, 0, st>>>(store, soff, slen, ns, lb, ub, cnt,
                                                                    first, loc, part, pool_words, scal);
  return hipGetLastError();
}

hipError_t launch_stim_copy(const uint64_t* store, const uint64_t* soff, const uint32_t* snet,
                            uint32_t ns, uint64_t lb, const uint64_t* cnt, const uint32_t* first,
                            const uint64_t* loc, const uint64_t* part, uint32_t* pool, uint64_t* woff,
                            uint32_t* wlen, const uint64_t* scal, hipStream_t st) {
  if (ns == 0) return hipSuccess;
  k_stim_copy<<<ns, 256, 0, st>>>(store, soff, snet, lb, cnt, first, loc, part, pool, woff, wlen, scal);
  return hipGetLastError();
}

hipError_t launch_tail_len(const GateRec* gates, uint32_t ng, const uint64_t* woff,
                           const uint32_t* wlen, const uint32_t* pool, uint32_t key, uint64_t* len,
                           uint64_t* src, uint64_t* loc, uint64_t* part, uint64_t* scal,
                           hipStream_t st) {
  if (ng == 0) return hipSuccess;
  k_tail_len<<<nblk(ng, kPlanGates), 256, 0, st>>>(gates, ng, woff, wlen, pool, key, len, src, loc, part,
                                                   scal);
  return hipGetLastError();
}

hipError_t launch_tail_copy(const GateRec* gates, uint32_t ng, const uint64_t* len,
                            const uint64_t* src, const uint64_t* loc, const uint64_t* part,
                            const uint32_t* pool, uint32_t* tails, uint64_t cap, uint32_t* tail_len,
                            uint64_t* tail_off, uint64_t* scal, hipStream_t st) {
  if (ng == 0) return hipSuccess;
  k_tail_copy<<<nblk(ng, 256), 256, 0, st>>>(gates, ng, len, src, loc, part, pool, tails, cap, tail_len,
                                             tail_off, scal);
  return hipGetLastError();
}

hipError_t launch_level(const LevelArgs& a, unsigned nblocks, hipStream_t st) {
  if (nblocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_level, dim3(nblocks), dim3(kLanes), a.lds_words * 4, st, a);
  return hipGetLastError();
}

int level_max_blocks(uint32_t lds_words) {
  int per_cu = 0, dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 2048;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_level, kLanes, lds_words * 4) != hipSuccess)
    per_cu = 4;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    cus = 256;
  // LDS is handed out in pieces of 1,280 bytes, 160 KiB per CU (workgroups
  // that do not fit at once would start their fixed runs late)
  const uint32_t piece = (lds_words * 4 + 1279) / 1280;
  per_cu = std::min<int>(per_cu, (int)(128 / std::max(1u, piece)));
  return std::max(per_cu, 1) * cus;
}

}  // namespace gls
