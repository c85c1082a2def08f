// Records shared between the host packer and the HIP kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace gls {

// Event word: (time << 2) | value, time < 2^30 time units of the chunk's
// relative time (see ChunkWin).  Resident stimulus words are 64-bit:
// (absolute time << 2) | value.
constexpr uint32_t kTimeInf = 0x3FFFFFFFu;
constexpr uint32_t kWordInf = 0xFFFFFFFFu;
// Largest span of one chunk in relative time: every event and candidate
// time of a chunk stays below it (room is kept for one more delay).
constexpr uint64_t kRelSpan = (1ull << 30) - (1ull << 18);

// One simulated output ("gate"), 80 bytes.  Delays are integer time units;
// 0xFFFF marks a missing IOPATH of that kind.
struct alignas(16) GateDev {
  uint32_t in_net[4];     // distinct input nets (resolved)
  uint32_t out_net;
  uint16_t lut;           // truth-table id (256 bytes each, index = sum v_j << 2j)
  uint8_t k;              // number of distinct inputs (1..4)
  uint8_t pad0;
  uint16_t dly[4][3][2];  // [input][both,pos,neg][rise,fall]
  uint8_t nrec[4];        // IOPATH records per input for this output
  uint16_t dmax;          // largest delay (>= 1)
  uint16_t pad1;
};
static_assert(sizeof(GateDev) == 80, "GateDev layout");

// Gate record of the fused level path, 48 bytes.  The walk evaluates an event
// with two table lookups, a truth-table byte and a delay word; `walk` names
// the form of the two tables (WalkId) and dt_off / tt_off place them.
struct alignas(16) GateRec {
  uint32_t in_net[6];
  uint32_t out_net;
  uint32_t dt_off;  // first word of the delay table (DevProgram::d_dtab)
  uint16_t lut;     // first 256-byte truth-table block (two-pass path)
  uint8_t k;        // distinct inputs, 1..6 (the reference's MAX_IN_NUM, src/simulate.cu:25)
  uint8_t walk;     // WalkId
  uint16_t dmax;
  uint16_t job;     // instance of a batch (SAIF window)
  uint32_t tt_off;  // first word of the truth-table bytes (DevProgram::d_ttab)
  uint32_t edge_in; // W_EO: the input whose edge the delays depend on
};
static_assert(sizeof(GateRec) == 48, "GateRec layout");

// Largest fan-in of the two-pass path, and of the walk.
constexpr uint32_t kTileK = 4;
constexpr uint32_t kWideK = 6;

// How the walk evaluates an event.  f, p: the gate's value after and before
// the event; ev: bit j = input j has an event; fell: bit j = that event fell
// (CheckDelay == 2); sc: output edge class 1..4; idx: packed input values,
// 2 bits per input.
//   W_NE1..W_NE6 (fan-in 1..6, no delay depends on an input's edge)
//     truth byte [new idx]          f << ne_shift(k)
//     delay word [p][f][ev]         4 d - 3 + f in bits 0..17, bit 24: f != p
//   W_EO3, W_EO4 (fan-in 3 and 4, the delays depend on the edge of one input)
//     truth byte [old value of that input][new idx]
//                                   (f << 1 | fell) << kEoShift
//     delay word [p][f][fell][ev]   as W_NE
//   W_ED1, W_ED2 (fan-in 1 and 2, edge-dependent delays; f(X..X) = X, so that p
//   is the function of the old values from the start on)
//     truth byte [new idx][old idx] f | (sc - 1) << 2 | fell << 4 | (f != p) << 7
//     delay word [ev][fell][sc - 1] 4 d - 3
//   W_GEN (any other gate)
//     truth byte as W_NE; delay table of half-words [half][both][sc - 1][bits]:
//     half h covers inputs 3h..3h+2, bits = per input (has an event, fell);
//     both = 0: the delay when only this half has events (AddDelay's
//     single-input rule when it is one event), 1: the smallest delay of its
//     events (0xFFFF: none) when the other half has events too.
enum WalkId : uint8_t {
  W_NE1 = 0, W_NE2, W_NE3, W_NE4, W_NE5, W_NE6, W_EO3, W_EO4, W_ED1, W_ED2, W_GEN, W_COUNT,
  W_DEAD = 15  // tile of a gate whose inputs were not made (a level before it failed)
};
inline constexpr uint32_t ne_shift(uint32_t k) { return (k < 4 ? k : 4u) + 2; }
constexpr uint32_t kEoShift = 5;  // bits of the truth byte below f << 1 | fell
// words of the two tables
__host__ __device__ inline constexpr uint32_t walk_dt_words(uint32_t id, uint32_t k) {
  return id <= W_NE6 ? 16u << k : (id <= W_EO4 ? 32u << k : (id <= W_ED2 ? 4u << (2 * k) : 512u));
}
__host__ __device__ inline constexpr uint32_t walk_tt_words(uint32_t id, uint32_t k) {
  const uint32_t b = id == W_EO3 || id == W_EO4   ? 4u << (2 * k)
                     : id == W_ED1 || id == W_ED2 ? 1u << (4 * k)
                                                  : 1u << (2 * k);
  return (b + 15) / 16 * 4;  // whole 16-byte pieces
}
inline constexpr uint32_t gen_dt_index(uint32_t half, uint32_t both, uint32_t s, uint32_t bits) {
  return ((half * 2 + both) * 4 + (s - 1)) * 64 + bits;
}

// Stack words beside one per staged word: one per lane (a step without a
// candidate writes the slot after the lane's last one) and one for the first
// lane's initial entry.
constexpr uint32_t kStackSlack = 68;

// LDS of one walk workgroup, in words: the tables of the tile's gate, its
// input ranges (range_layout), and the stacks at the end.
__host__ __device__ inline constexpr uint32_t walk_lds_need(uint32_t id, uint32_t k, uint32_t words) {
  return walk_dt_words(id, k) + walk_tt_words(id, k) + (words + 8 * k) + (words + kStackSlack);
}

// LDS words of one input range's slot: n words from pool word lo.  The slots
// follow the tables; the range starts lo mod 4 words into its slot, so that it
// is copied with 16-byte loads from the aligned word before it, and the word
// behind it is its sentinel's.  At most n + 7 words.
__host__ __device__ inline constexpr uint32_t range_words(uint32_t lo, uint32_t n) {
  return ((lo & 3u) + n + 4) & ~3u;
}

// Per-gate tiling of one level: tile i covers the leader input's words
// [i * lt, (i + 1) * lt).
struct GatePlan {
  uint32_t lt, lead;
};

// Everything one tile of the walk needs, 128 bytes, written by k_tile_desc.
// Input j's staged range starts one word before the tile (its value before
// the tile; the state entry for the gate's first tile) and ends with the
// look-ahead halo, n[j] words from pool word in_hi[j] << 32 | in_lo[j]; the
// tile's own words start at index 1 of each range.
struct alignas(16) TileDesc {
  uint32_t in_lo[6], n[6];
  uint32_t in_hi[2];       // byte j: bits 32..39 of input j's pool word
  uint32_t scr_lo, scr_hi; // first word of the tile's output region in the level scratch
  uint32_t own;            // the tile's own words (without its halo)
  uint32_t xend;           // index in the leader's range of the tile's end (0: the gate's last tile)
  uint32_t meta;           // WalkId | k << 4 | leader input << 8 | first tile of its gate << 12 |
                           // edge input << 16
  uint32_t dt_off, tt_off;
  uint32_t dmax, job;
  uint32_t out_cap;        // words of the tile's output region in the level scratch
  uint32_t g, ti;          // gate (index in the level), tile of the gate
  uint32_t out_net;
  uint32_t at2[3];         // where the ranges are staged: LDS words, two inputs a word (range_words)
  uint32_t words;          // sum of n
  uint32_t tab;            // words of the gate's delay table | truth bytes << 16
};
static_assert(sizeof(TileDesc) == 128, "TileDesc layout");

// What the walk kernel leaves for one tile, 16 bytes: its output entries
// (deduplicated inside the tile) sit in the level scratch; the join places
// them behind the tiles before.
struct alignas(16) TileOut {
  uint32_t cnt;          // entries after dedup inside the tile
  uint32_t first, last;  // the first and the last of them
  uint32_t ev;           // gate events of the tile (input-event times from the chunk start on)
};
static_assert(sizeof(TileOut) == 16, "TileOut layout");

// SAIF counters per net: T0, T1, TX durations and TC, the number of direct
// 0<->1 transitions at times in (dumpon, dumpoff].
constexpr uint32_t kSaifWords = 4;

// A value change from p to v is a toggle when it is 0 -> 1 or 1 -> 0
// (codes 0 and 3; X <-> Z, codes 1 and 2, also differ by 3 and is excluded).
__host__ __device__ inline bool is_toggle(uint32_t p, uint32_t v) {
  return (p ^ v) == 3u && (v == 0u || v == 3u);
}

// Time chunks.  A simulation runs as a sequence of time chunks
// [F_k, F_k+1); every chunk runs all levels.  Inside chunk k, times are
// relative: rel = abs - (lb_k - 1) with lb_k = F_k - W (W = the largest gate
// delay; lb_0 = 0), so every net's chunk waveform starts with a state entry
// at rel 0 (its value before lb_k), followed by its entries at abs times in
// [lb_k, F_k+1).  Entries at abs times in [lb_k, F_k) are the look-back
// window: they were final after chunk k-1 and are walked again only so that
// the candidates they make with output times >= F_k are known.
//
// Per instance and chunk: SAIF bounds in the chunk's relative time.
// Durations are summed over [lo, hi) (the chunk's part of the SAIF window);
// toggles are counted at entry times in (tc_lo, tc_hi].
struct ChunkWin {
  unsigned long long lo, hi, tc_lo, tc_hi;
};

// Tails of the gate outputs, the first words of their chunk waveforms: per
// net, the state entry and the look-back entries, kept from the previous
// chunk (in its relative time; `shift` = this chunk's time base minus the
// previous one).  In chunk 0 every tail is one X state entry.
struct TailArgs {
  const uint32_t* tail_len;  // per net
  const uint64_t* tail_off;  // per net: first word in `tails`
  const uint32_t* tails;
  uint32_t shift;
  uint32_t first;            // 1 in chunk 0
};

// Run scalars in device memory (64-bit slots).  The levels of a chunk run with
// no host round trip: each level's kernels read its counts here, and the plan
// kernel trips the chunk (S_TRIP) when a level needs more room than it has (or
// the caller asked to stop); every later kernel then returns at once and the
// host reads why, makes room and goes on from that level.
enum ScalSlot {
  S_BUMP = 0,     // pool words used
  S_TOT_A = 1,    // tiles and scratch words that the last planned level asked for
  S_TOT_B = 2,
  S_TOT_OUT = 3,  // output words of the level (two-pass path)
  S_EVC = 4,      // gate events of the run
  S_OVF_USED = 6, // overflow stack words the level asked for
  S_ERR = 7,      // error flags
  S_TILES = 8, S_TILES_HBM = 9,  // tiles walked, of them on the HBM path
  S_TAILS = 10,   // words of the chunk's gate-output tails
  S_TRIP = 11,    // 0, or the tripped level + 1
  S_WHY = 12,     // TripWhy
  S_LIMIT = 14,   // pool word that the level's outputs must not reach
  S_OUTBASE = 15, // pool word of the level's first output
  S_STIM = 16,    // pool words of the chunk's stimulus
  S_DONE = 17,    // blocks of the running scan that are done
  S_CLOCK = 18,   // start of the level's walk
  S_EVAL = 19,    // ticks spent in walks
  S_LEVELS = 20,  // walks run
  S_IN_W = 21, S_OUT_W = 22,     // waveform words read by gates, written by gates
  // of the level in hand and the one planned while its outputs are copied
  // (LevelArgs::slot): tiles, address of the level scratch
  S_NTILES = 23, S_SCRATCH = 25,
  S_COUNT = 32
};
enum TripWhy : unsigned { TRIP_STOP = 1, TRIP_PROJECTED, TRIP_ROOM, TRIP_OVERFLOW, TRIP_STIM, TRIP_POOL };

// The walk's ticket counters, each on a cache line of its own.
constexpr uint32_t kTickets = 4, kTicketStride = 32;

// Gates per block of the plan's and the join's scans (a gate's prefix = its
// block's, in `part`, plus its own inside the block), and signals per block of
// the stimulus cut.
constexpr uint32_t kPlanGates = 256, kJoinGates = 32, kStimSignals = 256;

// Smallest lane share of a level too small for the chip (PlanArgs::spread).
constexpr uint32_t kSpreadSeg = 16;

// Tiles per block of the descriptors.
constexpr uint32_t kDescTiles = 63;

// Plan of one level.
struct PlanArgs {
  const GateRec* gates;
  uint32_t ng;
  const uint32_t* wlen;
  const uint32_t* tail_len;
  uint32_t seg_target, wide_words;
  float spread;         // 0, or: lane share of a small level per input word of the gate
  GatePlan* plan;
  uint32_t* ntile;      // tiles per gate
  uint32_t* tile_loc;   // tiles before the gate in its block
  uint64_t* scr_loc;    // scratch words before the gate in its block
  uint64_t* part;       // per block: tiles, scratch words before it
  uint64_t* scal;
  unsigned long long* ticket;
  // room: tile arrays, pool, a scratch apart from the pool (when allowed)
  uint64_t tiles_cap, pool_words, apart_cap;
  uint32_t* pool;
  uint32_t* apart;
  uint32_t allow_apart;
  uint32_t level;       // level + 1, for S_TRIP
  uint32_t slot;        // 0 or 1
  // automatic chunks: trip when the chunk's outputs so far, over `done_gates`
  // of `all_gates`, project to more than proj_cap words (0: not asked)
  double proj_cap, all_gates, done_gates;
  const uint32_t* stop; // host flag: nonzero trips the chunk (null: none)
};

// Compaction of one level's outputs.
struct CompactArgs {
  const TileDesc* tiles;
  const TileOut* tout;
  const uint32_t* tile_off;
  const uint64_t* out_loc;
  const uint64_t* part;
  uint32_t* pool;
  uint64_t* woff;
  const uint64_t* scal;
  unsigned long long* saif;
  const ChunkWin* cwin;
  uint32_t count_tc;
  uint32_t level;       // level + 1
  uint32_t slot;
};

// Join of one level's tiles.
struct JoinArgs {
  const GateRec* gates;
  uint32_t ng;
  const uint32_t* ntile;
  const uint32_t* tile_loc;
  const uint64_t* plan_part;
  const TileOut* tout;
  uint32_t* tile_off;
  uint64_t* out_loc;    // output words before the gate in its block
  uint64_t* part;       // per block: output words before it
  uint32_t* wlen;
  unsigned long long* saif;
  const ChunkWin* cwin;
  uint64_t* scal;
  unsigned long long* ev_job;  // batches: gate events per instance (null: none)
  uint32_t level;       // level + 1, for S_TRIP
  uint32_t slot;
  uint32_t ovf_trip;    // 1: a level that ran out of overflow stacks is run again
};

// Arguments of the fused level (walk) kernel.
struct LevelArgs {
  const TileDesc* tiles;      // per tile
  const uint32_t* pool;       // input waveforms
  const uint32_t* dtab;       // delay tables (GateRec::dt_off)
  const uint32_t* ttab;       // truth tables (GateRec::tt_off)
  uint64_t* scal;
  TileOut* tout;              // per tile
  uint32_t* ovf;              // stacks of tiles that do not fit LDS
  unsigned long long ovf_cap;
  unsigned long long* ticket;   // batches handed out by each counter (0 per level)
  const ChunkWin* cwin;        // SAIF bounds of this chunk per instance
  uint32_t lds_words;          // LDS of a workgroup
  uint32_t prefetch;           // 1: stage the next tile before storing this one
  uint32_t slot;
  uint32_t lo_rel;             // F_k in chunk time: candidates below it only pre-empt
  uint32_t hi_rel;             // F_k+1 in chunk time (0xFFFFFFFF: last chunk): candidates
                               // at or above it belong to the next chunk and are dropped
  uint32_t first;              // 1 in chunk 0: outputs start with (0, X), f before t = 0 is X
};

// Per time-segment summary written by the evaluation kernel.
struct SegSum {
  uint64_t scr_off;   // scratch offset of the segment's kept candidates
  uint32_t n_raw;     // kept candidates (after preemption, before dedup)
  uint32_t n_dd;      // after in-segment dedup (first entry always counted)
  uint32_t last_o;    // time of the last kept candidate
  uint8_t first_v, last_v, pad[2];
};

// Per-segment carry computed by the gate scan.
struct SegCarry {
  uint32_t pos;       // output index of the segment's first emitted entry
  uint32_t carry_t;   // time of the last kept candidate before the segment
  uint8_t carry_v;    // its value (4 = none: first entry always emitted)
  uint8_t pad[3];
};

}  // namespace gls
