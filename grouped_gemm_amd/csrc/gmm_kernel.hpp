// Grouped GEMM for gfx950 (MI355X): one persistent launch, scheduler on the device.
//
// Replaces the reference's CUTLASS grouped kernel and its argument builders
// (csrc/grouped_gemm.cu:38-81, 230-371; csrc/fill_arguments.cuh:34-131).
//
// Every workgroup first derives the same schedule from batch_sizes (prefix sums of
// rows and of tiles, kept in LDS), then walks tiles t = id, id + grid, ... .  A tile is
// up to BM x BN outputs of one group: a group's rows are split evenly over its tile rows,
// and a tile issues MFMAs only for the 32-row blocks that have rows.  Operand tiles go from
// HBM straight into LDS
// (buffer_load_dwordx4 ... lds, 16 bytes per lane), through a ring of STAGES buffers;
// rows past a group's end are cut off by the buffer descriptor's size, so they
// arrive as zeros and no lane ever touches memory outside its group.  Fragments are read
// from LDS with ds_read_b128 where the depth dimension is contiguous in memory and
// with the transposing ds_read_b64_tr_b16 where it is not, feed
// v_mfma_f32_16x16x32_bf16 with fp32 accumulators, and leave as bf16 through
// buffer stores that the descriptor clips at the group's last row (or are added to an fp32
// output, in the accumulating form of the weight-gradient layout).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

namespace gg {

constexpr int kMaxGroups = 512;
constexpr int kSchedCols = 14;

enum : int { kNN = 0, kNT = 1, kTN = 2 };
// Element types of a and b.  Two-byte types give a c of the same type; the one-byte (OCP fp8)
// types give a bf16 c.
enum : int { kBF16 = 0, kF16 = 1, kF8E4M3 = 2, kF8E5M2 = 3 };
constexpr bool is_f8(int dt) { return dt == kF8E4M3 || dt == kF8E5M2; }

using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using bf16x4 = __attribute__((ext_vector_type(4))) __bf16;
using f16x8 = __attribute__((ext_vector_type(8))) _Float16;
using f16x4 = __attribute__((ext_vector_type(4))) _Float16;
using f32x16 = __attribute__((ext_vector_type(16))) float;
using f32x4 = __attribute__((ext_vector_type(4))) float;
using u32x2 = __attribute__((ext_vector_type(2))) uint32_t;
using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
using i32x4 = __attribute__((ext_vector_type(4))) int;
using i32x8 = __attribute__((ext_vector_type(8))) int;

#define GG_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

struct GmmParams {
  const char* a;
  const char* b;
  char* c;
  const int64_t* sizes_dev;  // device-resident batch_sizes of ALL groups, or nullptr (then HostSizes)
  int64_t* sched_out;        // only read by the schedule dump kernel
  char* workspace;           // counters + fp32 partial tiles of depth pieces, or nullptr
  int64_t tokens;            // rows of a
  int64_t row_base;          // host-resident sizes: rows taken by the groups before first_group
  int32_t first_group;       // this launch schedules groups first_group .. first_group + num_groups - 1
  int32_t num_groups;        // at most kMaxGroups
  int32_t hidden_in;
  int32_t hidden_out;
  int32_t group_m;     // tile rows per band of the in-group tile order
  int32_t flags;       // kFlag* bits
  int32_t ws_slots;    // partial-tile slots the workspace holds (0: no depth pieces)
  int32_t b_cols;      // columns of one group's b in memory: hidden_out, or twice that for gate | up
  int32_t lda, ldb;    // elements from one row of a (of b) in memory to the next: more than a row has in copies
                       // that are padded to whole lines, with zeros where the rows run along the depth
  // the variants with row indices only:
  const int32_t* a_rows;   // row r of the left operand is row a_rows[r] of a, or nullptr (rows in place)
  const int32_t* c_rows;   // row r of the output goes to row c_rows[r] of c, or nullptr
  uint32_t a_bytes;        // bytes of a and of c in memory, below kOutOfRangeIndexed
  uint32_t c_bytes;
  uint32_t a_index_rows;   // rows of a and of c in memory: an index that names no row of them is a
  uint32_t c_index_rows;   // missing row (read as zeros, not stored)
  char* gate_up;           // kEpiSwiGLUKeep: (tokens, 2 hidden_out), rows like those of c
  int32_t* status;         // device word that collects kStatus* bits about the sizes, or nullptr
};

enum : int {
  kStatusNegativeSize = 1,   // a batch size was negative (taken as 0)
  kStatusRowsPastEnd = 2,    // the sizes sum past `tokens` (the rows past the end were dropped)
};

enum : int {
  kEpiStore = 0,    // c in the operands' element type, overwritten
  kEpiAccF32 = 1,   // c in fp32, added to (weight-gradient layout only)
  kEpiSwiGLU = 2,   // b holds gate | up columns; c = silu(a @ gate) * (a @ up), half as wide
  // kEpiAccF32 with atomic additions instead of read, add, write: faster while the launch is bound
  // by the matrix pipe (deep groups: 3.35 -> 3.16 ms at 8 x 4096 rows, 4096 x 14336), much slower
  // when it is bound by the traffic of c itself (256 x 256 rows, 2048 x 7168: 7.0 -> 11.7 ms)
  kEpiAccF32Atomic = 3,
  kEpiSwiGLUKeep = 4,   // kEpiSwiGLU that also stores gate | up, rounded, for the gradient
};

enum : int {   // debugging switches, for comparing the ways a call can be scheduled
  kFlagWholeTiles = 1,    // never cut the tiles of the last round into pieces
  kFlagOneClass = 2,      // hand out runt rows in place, not after all other tiles
  kFlagRowPieces = 4,     // ignore the workspace: cut along the rows only
  kFlagGroupOrder = 8,    // NN and NT layouts: never hand out the groups' tiles by tile rows
  kFlagByTileRows = 16,   // set by the host side (never by callers): hand them out by tile rows
  kFlagAnyRows = 64,      // set by the host side: rows of c on 2-byte boundaries, of any length
  kFlagPiecesByLength = 128,   // set by the host side: plan_pieces_by_length instead of plan_deep_tiles
  kFlagMergeStores = 32,  // set by the host side: kStoreMerging instead of kStoreStreaming (merge_stores in gmm_api.hip)
};

// Workspace layout: kWsCounterBytes of int32 arrival counters (one per tile of the last round; all
// zero before a launch and all zero again after it), then ws_slots partial tiles of BM x BN floats.
constexpr int kWsCounterBytes = 4096;
// Into how many depth pieces `tiles` tiles of `slices` depth slices, `rows` rows and BN columns are
// best cut, at most `most` (1: not at all), on `units` compute units.  In units of depth slices of the
// same tile: the slices left to a piece, half as slow again where two pieces share a compute unit, and
// the fix-up: a constant (the arrival counted, the tile loop left) and the partial tiles, written
// by their pieces and read back by the last of them to arrive, which go through memory and slow down
// when more than half the device does it at once.  Measured, at 0.6-0.7 us a slice: 64 tiles of 256 x
// 256, 2 pieces: 25 us of fix-up; 16 of them, 4 pieces: 26 us; 128 of 64 rows x 256, 4 pieces: 18 us;
// 16 rows x 256, 4 and 8 pieces: 7 and 9 us.
constexpr int kMaxDepthPieces = 16;
__host__ __device__ inline int best_depth_pieces(int slices, int rows, int bn, int tiles, int units, int most) {
  int best = 1, best_cost = slices;
  for (int pieces = 2; pieces <= most && pieces <= kMaxDepthPieces; pieces *= 2) {
    const int all = tiles * pieces;
    int each = (slices + pieces - 1) / pieces;
    if (all > units) each = each * (units + all) / (2 * units);
    const int cost = each + 10 + pieces * rows * bn / (2 * all > units ? 3500 : 8000);
    if (cost < best_cost) best = pieces, best_cost = cost;
  }
  return best;
}
// ... and for the tiles of a weight gradient that are so deep that they set the length of the launch:
// fewest slices per piece, most pieces.
constexpr int min_slices_per_piece(int tile_outputs) { return tile_outputs > 128 * 128 ? 48 : 16; }
constexpr int kMaxDeepPieces = 4;
// Tiles go out by descending depth, one workgroup each, so groups much deeper than the rest set the length of the launch.
// depth(q): depth slices (of bk rows) of the q-th deepest of E groups, which have `rows` rows in all and per_group tiles each.  Where
// the deepest tile is longer than a workgroup's even share of all slices, the tiles deeper than half of that share that leave every
// piece min_slices are cut, as long as there are workgroups and partial tiles (`slots`) for their pieces.  Into as many
// pieces as end the launch soonest: its longest piece, or the deepest tile that stays whole (84 tiles of 100 slices: in 4
// pieces each, 64 are cut and 20 set the length, whatever the groups behind them are: 9000, 30, 0 and 1400 rows, 1536 x
// 896: 95 us in four pieces, 51 in two).
struct DeepCut {
  int pieces, tiles;   // pieces per tile, tiles cut (0: none)
};
template <typename DEPTH>
__host__ __device__ inline DeepCut cut_deep_tiles(const DEPTH& depth, int E, int64_t rows, int per_group, int grid, int slots,
                                                  int min_slices, int bk) {
  DeepCut chosen{0, 0};
  const int deepest = depth(0);
  // (half a slice per group for the rounding)
  const int64_t share = (rows + (int64_t)E * (bk / 2)) / bk * per_group / grid;
  if (deepest <= share) return chosen;
  int best = deepest;
  for (int n = kMaxDeepPieces; n >= 2; n >>= 1) {
    int most = grid / n;
    most = most < slots / n ? most : slots / n;
    most = most < kWsCounterBytes / 4 ? most : kWsCounterBytes / 4;
    int cut = 0, whole = 0;   // tiles cut, depth of the deepest one that is not
    for (int q = 0; q < E; ++q) {
      const int mine = depth(q);
      const bool fits = cut < most && 2 * (int64_t)mine > share && mine >= n * min_slices;
      if (fits) cut += per_group;
      if (!fits || cut > most) {
        whole = mine;
        break;
      }
    }
    const int each = (deepest + n - 1) / n, length = each > whole ? each : whole;
    if (cut > 0 && length < best) best = length, chosen = DeepCut{n, cut < most ? cut : most};
  }
  return chosen;
}

// Pieces of one length instead (GG_FLAG_FEW_TILES): as many of a tile as it has such lengths, so that groups of all depths end
// together, also where there are few tiles and the deepest are many times as long as the rest (small hidden sizes and many
// rows).  The deepest groups are cut; those that are no more than half as long again as a piece stay whole.
// In depth slices of such a tile: a tile's turnover; a fix-up, constant and per piece; a partial tile's way through memory; the shortest
// piece.
template <int OUTPUTS>
struct PieceCosts {
  static constexpr int OUT = OUTPUTS;
  static constexpr bool FULL = OUTPUTS > 128 * 128;
  static constexpr float TILE = FULL ? 4 : 3, FIX = FULL ? 14 : 4, FIX_PIECE = FULL ? 3 : 1.5f, PARTIAL = FULL ? 6 : 3;
  static constexpr int SHORTEST = FULL ? 16 : 6;
};
// The lengths tried: the deepest tile's halves to sixteenths.  (No fifths of full tiles: 56 Zipf (1.2) groups, 19094 rows, 704 x 1376, 5
// and 3 pieces of the deepest two against 4 and 2: 93.5 us and 91.5.)
constexpr int kPieceLengths = 8;
template <int OUTPUTS>
__host__ __device__ constexpr int piece_count(int k) {
  return k < 5 ? k + 2 - (PieceCosts<OUTPUTS>::FULL && k == 3 ? 1 : 0) : 4 * (k - 3);
}
__host__ __device__ constexpr bool is_cut(uint32_t depth, uint32_t length) { return depth > length + length / 2; }
// The one with which the launch is expected to end soonest: the longest of the first round (a piece and its fix-up, or the deepest whole
// tile), and an even share of what is left.  More pieces than compute units: two of them share a unit and take twice as long (7
// groups of 6377 rows, 12 small tiles each: 3 pieces 31.0 us, 4 of them 36.0; 2 of 20000, 22 each: 5 pieces 44.5, 6 of them 48.3).  Where
// there are more tiles than that, whole ones share units too, and nothing sets the pieces apart.
// `depths` is the groups' depths, deepest first: at(q) that of position q (0 behind the last), first(n) the sum of n.
struct PieceLaunch {
  int tiles, per_group, grid, units, slots;
};
template <int OUTPUTS, typename DEPTHS>
__host__ __device__ inline float pieces_end(const DEPTHS& depths, const PieceLaunch& of, int n, int length, int cut, int pieces, float share) {
  using Costs = PieceCosts<OUTPUTS>;
  const uint32_t front = (uint32_t)pieces * (uint32_t)of.per_group;
  const int most = of.grid < of.slots ? of.grid : of.slots;
  const bool fits = (uint64_t)(uint32_t)pieces * of.per_group <= (uint64_t)most && (uint64_t)(uint32_t)cut * of.per_group <= kWsCounterBytes / 4;
  if (n > 1 && (length < Costs::SHORTEST || cut == 0 || !fits)) return 1e30f;
  const float whole = (float)depths.at(cut) + Costs::TILE;
  const bool shared = (int)front > of.units && of.tiles <= of.units;
  const float piece = cut > 0 ? (shared ? 2.0f : 1.0f) * length + Costs::FIX + Costs::FIX_PIECE * n : 0.0f;
  float end = piece > whole ? piece : whole;
  if (of.tiles - cut * of.per_group + (int)front > of.grid) {
    // what follows: the share of all, less that of the first round (the pieces and whole tiles for the workgroups left)
    const uint32_t to = (uint32_t)cut + (uint32_t)(of.grid - (int)front) / of.per_group;
    const float after = share - Costs::TILE + (Costs::PARTIAL * pieces - (float)depths.first(to)) * of.per_group / of.grid;
    end += after > 0 ? after : 0.0f;
  }
  return end;
}
// ... and of a launch as it is: whole tiles, or all of them in `tail` pieces.
template <int OUTPUTS, typename DEPTHS>
__host__ __device__ inline float uncut_end(const DEPTHS& depths, const PieceLaunch& of, int tail, float share) {
  using Costs = PieceCosts<OUTPUTS>;
  if (tail <= 1) return pieces_end<OUTPUTS>(depths, of, 1, 0, 0, 0, share);
  return (of.tiles * tail > of.units ? 2.0f : 1.0f) * (float)depths.at(0) / tail + Costs::FIX + Costs::FIX_PIECE * tail;
}
// (a change has to pay by a tenth: 6 groups of 6000 rows, 8 small tiles each, stay in 4 pieces: 25.7 us, in 5 26.7)
constexpr float kPiecesPay = 0.9f;
// Index t of the pieces of one group's tiles, the first of which is `first`: first all tiles' first pieces, then all their second ones
// (neighbours share rows of both operands).
struct PieceAt {
  int piece, tile, slot;   // which piece of which tile of the group; place of that tile's first partial tile, the others are per_group apart
};
__host__ __device__ inline PieceAt piece_at(int t, int first, int per_group) {
  const int piece = (t - first) / per_group, slot = t - piece * per_group;
  return PieceAt{piece, slot - first, slot};
}

// The last round of a persistent grid is filled only partly: `tiles % grid` workgroups have a
// tile, the others idle.  When that rest is at most half of the grid, each of its tiles is cut
// into pieces that go to different workgroups.  With a workspace (and a deep product) the cut
// runs along the depth:
// every piece accumulates its share of the depth slices into an fp32 partial tile in the
// workspace, and the piece that arrives last adds the partial tiles up in piece order (so the sum
// does not depend on which piece that is) and stores the result.  Without a workspace the cut
// runs along the rows (2 or 4 pieces of whole 32-row blocks; not in the weight-gradient layout).
// A launch with fewer tiles than workgroups is all "last round".
struct TailPlan {
  int main_tiles;   // tiles before the last round, handed out whole
  int pieces;       // pieces per tile of the last round
  int total;        // indices to hand out: main_tiles + rest * pieces
  bool by_depth;
};
template <int LAYOUT, int BM, int BN, int WGS_PER_CU, bool DEPTH_PIECES_ALLOWED = true>
__device__ __forceinline__ TailPlan plan_tail(int tiles, int grid, const GmmParams& p, int bk) {
  TailPlan t;
  const int rest = tiles % grid;
  t.pieces = 1;
  t.by_depth = false;
  if (rest > 0 && 2 * rest <= grid && !(p.flags & kFlagWholeTiles)) {
    if (DEPTH_PIECES_ALLOWED && p.ws_slots > 0 && !(p.flags & kFlagRowPieces)) {
      // The depth is the same for every tile, or, in the weight-gradient layout, the group's row
      // count: there the average over the groups stands for it, as it does for the rows of a tile
      // in the other layouts.
      const int average = (int)(p.tokens / (p.num_groups > 0 ? p.num_groups : 1));
      const int depth = LAYOUT != kTN ? p.hidden_in : average;
      const int rows = LAYOUT != kTN && average < BM ? (average + 31) / 32 * 32 : BM;
      t.pieces = best_depth_pieces((depth + bk - 1) / bk, rows, BN, rest, grid / WGS_PER_CU, min(grid, p.ws_slots) / rest);
      t.by_depth = t.pieces > 1;
    }
    // (a tile of two 32-row blocks is spread over both wave rows already)
    if (!t.by_depth && LAYOUT != kTN && BM > 64) t.pieces = 4 * rest <= grid ? 4 : 2;
  }
  t.main_tiles = t.pieces > 1 ? tiles - rest : tiles;
  t.total = t.main_tiles + (tiles - t.main_tiles) * t.pieces;
  return t;
}

// Host-resident batch_sizes travel in the kernel argument block: no copy, no staging.
struct HostSizes {
  int32_t v[kMaxGroups];
};

// What every workgroup keeps in LDS about the groups.  Tiles come in two classes: first all
// tiles except each group's last, much shorter tile row ("runt" row: at most half the 32-row
// blocks of the group's other tile rows), then the runt rows.  Tiles of one class take about the
// same time, so workgroups that walk the classes in this order stay in step, and the cheap tiles
// fill the end of the launch.
struct Sched {
  int32_t row_start[kMaxGroups + 1];   // exclusive prefix sum of rows, clipped to tokens
  int32_t rows[kMaxGroups];            // rows of `a` the group uses
  int32_t tile_start[kMaxGroups + 1];  // exclusive prefix sum of the first class's tiles
  int32_t runt_start[kMaxGroups + 1];  // exclusive prefix sum of the runt rows' tiles
  int32_t arrived;                     // broadcast slot for the arrival count of a depth piece
  int32_t fix_tile[24];                // the tile whose depth pieces this workgroup adds up after its last tile
  // Weight-gradient layout (plan_deep_tiles): the first front_tiles tiles, the deepest ones, are
  // cut along the depth into front_pieces pieces each; tile indices 0 .. front_tiles *
  // front_pieces - 1 name those pieces, the tiles behind follow whole, and the last round is not
  // cut.  (Kept here, not in registers: the tile loop has no scalar registers to spare.)
  // With plan_pieces_by_length front_pieces is 0, indices 0 .. front_tiles - 1 name the pieces of the first cut_groups
  // positions of `order`: position q's begin at tile_start[q], runt_start[q] of every tile (first all tiles' first
  // pieces, then all their second ones: neighbours share rows of both operands).
  int32_t front_tiles, front_pieces, cut_groups;
  int32_t group_tiles;                 // tiles per group
  int32_t most_rows;                   // rows of the largest group
  // order[q] is the group whose tiles are handed out q-th.  Weight-gradient layout: by descending
  // depth.  Every group has the same number of tiles there and a tile's cost is its group's depth,
  // so the deepest groups go first and the shallow ones fill the end of the launch: what the
  // reference's sort by k does for its scheduler (csrc/grouped_gemm.cu:193-207,
  // csrc/fill_arguments.cuh:80-81).  Other layouts, with kFlagByTileRows: by ascending number of
  // tile rows (tile_start and runt_start then count in that order); without: not used.  Results
  // do not depend on it.
  int16_t order[kMaxGroups];
};

constexpr uint32_t kOutOfRange = 0x80000000u;  // beyond the descriptor of one tile's rows
// ... and for the descriptors that may be larger: of a whole tensor (rows reached through an index), of gate | up
constexpr uint32_t kOutOfRangeIndexed = 0xfffffff0u;
constexpr uint32_t kRsrcFlags = 0x00020000u;   // raw buffer, 32-bit data format
// Cache policy of the output stores: non-temporal.  The output is written once and never read by
// this kernel, so it should not push operand lines that other tiles still share out of L2.
constexpr int kStoreStreaming = 2;
// ... and write-back, for rows of c that do not start on 64-byte boundaries: L2 then puts the parts of a 64-byte
// sector that different stores bring together.  A sector written past L2 in parts costs a read and two writes of
// memory: 1.4 TB/s against 4.1 for whole sectors (1 GiB, 8 rows x 128 bytes per instruction), 2.9 where L2 merges.
constexpr int kStoreMerging = 0;
// Cache policy of the partial tiles of depth pieces: device scope (sc1), i.e. written through to and
// read from where all XCDs see them.  Their hand-over then needs no fence, which would write back
// and invalidate whole L2s: 512 pieces of 16 depth slices took 100 us for theirs.
constexpr int kDeviceScope = 16;

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ const char* uniform_ptr(const char* p) {
  const uint64_t b = reinterpret_cast<uint64_t>(p);
  return reinterpret_cast<const char*>((uint64_t)(uint32_t)uniform((int)(uint32_t)b) | ((uint64_t)(uint32_t)uniform((int)(uint32_t)(b >> 32)) << 32));
}

// Buffer descriptor of `bytes` bytes at `base`, as the four dwords the hardware reads.
// Both inputs are the same in every lane; reading them through the first lane tells the
// compiler so and keeps the descriptor in scalar registers.
using rsrc_words = __attribute__((ext_vector_type(4))) int;

__device__ __forceinline__ rsrc_words make_rsrc_words(const void* base, uint32_t bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  rsrc_words r;
  r[0] = uniform((int)(uint32_t)b);
  r[1] = uniform((int)((uint32_t)(b >> 32) & 0xffffu));   // 48-bit base, stride 0
  r[2] = uniform((int)bytes);
  r[3] = (int)kRsrcFlags;
  return r;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  const uint64_t ub = (uint64_t)(uint32_t)uniform((int)(uint32_t)b) |
                      ((uint64_t)(uint32_t)uniform((int)(uint32_t)(b >> 32)) << 32);
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(ub), 0,
                                           (uint32_t)uniform((int)bytes), kRsrcFlags);
}

// 16 bytes per lane from global memory straight into LDS at lds_addr + OFFSET + lane * 16: the address, then
// the load, which needs an instruction between the two.  Nothing else writes m0 (a reserved register: the compiler uses
// it for nothing that occurs here).
// Written as assembly on purpose: the compiler then keeps no record of pending writes
// into LDS, and does not put a full wait for them in front of later LDS reads that touch
// other buffers of the ring.  The waits that are needed are the explicit wait_vmcnt calls.
template <int OFFSET>
__device__ __forceinline__ void aim_lds(uint32_t lds_addr) {
  asm volatile("s_add_u32 m0, %0, %1" : : "s"(lds_addr), "n"(OFFSET) : "memory", "m0", "scc");
}
// The hardware does not wait for a descriptor word that a vector instruction (v_readfirstlane, v_readlane) writes less
// than five instructions before the load that reads it, and the compiler does not look into assembly: settle
// puts the words where they stay, five instructions or more ahead of the first load that uses them (fetch_begin).  A test reads
// the built library for loads that come too soon.
template <int MORE = 0>   // instructions to wait here
__device__ __forceinline__ void settle(rsrc_words& rsrc) {
  if constexpr (MORE > 0) {
    asm volatile("s_nop %1" : "+s"(rsrc) : "n"(MORE - 1));
  } else {
    asm volatile("" : "+s"(rsrc));
  }
}
template <bool RIGHT_BEHIND>   // right behind aim_lds
__device__ __forceinline__ void load_to_lds_16(const rsrc_words& rsrc, uint32_t voffset) {
  if constexpr (RIGHT_BEHIND) {
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(voffset), "s"(rsrc) : "memory");
  } else {
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(voffset), "s"(rsrc) : "memory");
  }
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)reinterpret_cast<uintptr_t>(GG_LDS_PTR(p));
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit field");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ void block_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// One 32x32x16 matrix instruction on fragments of 8 two-byte elements per lane (carried as
// bf16x8 whatever the element type; the type only selects the instruction).
template <int DT>
__device__ __forceinline__ f32x16 mfma_32x32x16(bf16x8 x, bf16x8 y, f32x16 acc) {
  if constexpr (DT == kBF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, acc, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, x),
                                                  __builtin_bit_cast(f16x8, y), acc, 0, 0, 0);
  }
}

// One 16x16x32 matrix instruction on fragments of 8 two-byte elements per lane: what the streaming kernel
// multiplies two-byte elements with.  Per operation it moves half the accumulators of the 32x32x16 one in and out
// of the register file, and power is what bounds these products: on operands like real activations, in
// registers and nothing else running, 16x16x32 sustains 1930-1970 TFLOP/s (bf16; on zeros, at full clock, 2331-2352), 32x32x16
// 1635-1740 (the rate probe of the benchmark, each at its time).
template <int DT>
__device__ __forceinline__ f32x4 mfma_16x16x32(bf16x8 x, bf16x8 y, f32x4 acc) {
  if constexpr (DT == kBF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, acc, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x), __builtin_bit_cast(f16x8, y), acc, 0, 0, 0);
  }
}

// One 32x32x64 matrix instruction on fp8 fragments: 32 one-byte elements per lane and operand,
// handed over as the two 16-byte halves they are read from LDS in.
template <int DT>
__device__ __forceinline__ f32x16 mfma_32x32x64_f8(bf16x8 x_lo, bf16x8 x_hi, bf16x8 y_lo, bf16x8 y_hi, f32x16 acc) {
  const i32x8 x = __builtin_shufflevector(__builtin_bit_cast(i32x4, x_lo), __builtin_bit_cast(i32x4, x_hi), 0, 1, 2,
                                          3, 4, 5, 6, 7);
  const i32x8 y = __builtin_shufflevector(__builtin_bit_cast(i32x4, y_lo), __builtin_bit_cast(i32x4, y_hi), 0, 1, 2,
                                          3, 4, 5, 6, 7);
  constexpr int FORMAT = DT == kF8E5M2 ? 1 : 0;   // e4m3 : e5m2, for both operands; no block scales
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, y, acc, FORMAT, FORMAT, 0, 0, 0, 0);
}

// Four fp32 values rounded (to nearest even) to the element type, as 8 bytes.
template <int DT>
__device__ __forceinline__ u32x2 round4(float v0, float v1, float v2, float v3) {
  if constexpr (DT == kBF16) {
    bf16x4 o = {(__bf16)v0, (__bf16)v1, (__bf16)v2, (__bf16)v3};
    return __builtin_bit_cast(u32x2, o);
  } else {
    f16x4 o = {(_Float16)v0, (_Float16)v1, (_Float16)v2, (_Float16)v3};
    return __builtin_bit_cast(u32x2, o);
  }
}

// ---------------------------------------------------------------------- schedule

// How a group's output is cut into tiles.
struct GroupTiles {
  int tiles_m, tiles_n;
  int height;       // rows per tile row (the last tile row takes what is left)
  int main_rows;    // tile rows of the first class
  int runt;         // 1: the last tile row is a runt row (second class)
};

// The rows of a group are split evenly over its tile rows, in whole 32-row blocks: 300 rows make
// two tile rows of 160 (5 blocks each), not one of 256 and one of 44.  Tile rows of a group then
// take the same time, and blocks without rows cost nothing.  What is left for the last tile row
// of a tall group can still be much less than the others' (4122 rows: 16 tile rows of 256 and one
// of 26): such a row goes to the second class.
template <int LAYOUT, int BM, int BN>
__device__ __forceinline__ GroupTiles group_tiles(int rows, int hidden_in, int hidden_out, int flags) {
  GroupTiles g;
  g.tiles_n = (hidden_out + BN - 1) / BN;
  g.runt = 0;
  if (LAYOUT == kTN) {
    g.tiles_m = (hidden_in + BM - 1) / BM;
    g.height = BM;
  } else {
    g.tiles_m = (rows + BM - 1) / BM;
    g.height = BM;
    if (g.tiles_m > 0) {
      // rows / tiles_m rounded up to whole blocks: 1 .. BM / 32 of them, counted instead of divided out
      int blocks = 1;
#pragma unroll
      for (int h = 1; h < BM / 32; ++h) blocks += (uint32_t)(h * 32) * (uint32_t)g.tiles_m < (uint32_t)rows ? 1 : 0;
      g.height = blocks * 32;
      const int last_blocks = (rows - (g.tiles_m - 1) * g.height + 31) / 32;
      g.runt = g.tiles_m >= 2 && 2 * last_blocks <= g.height / 32 && !(flags & kFlagOneClass) ? 1 : 0;
    }
  }
  g.main_rows = g.tiles_m - g.runt;
  return g;
}

// Inclusive scan over the lanes of a wave by `op`, whose identity is 0: data-parallel moves, a few cycles
// each, where a shuffle goes through LDS.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROW_MASK, 0xf, false);
}
template <typename OP>
__device__ __forceinline__ uint32_t wave_scan(uint32_t x, OP op) {
  x = op(x, dpp_or_zero<0x111, 0xf>(x));   // row_shr:1, 2, 4, 8: inside rows of 16 lanes
  x = op(x, dpp_or_zero<0x112, 0xf>(x));
  x = op(x, dpp_or_zero<0x114, 0xf>(x));
  x = op(x, dpp_or_zero<0x118, 0xf>(x));
  x = op(x, dpp_or_zero<0x142, 0xa>(x));   // row_bcast:15 into rows 1 and 3, row_bcast:31 into rows 2 and 3
  return op(x, dpp_or_zero<0x143, 0xc>(x));
}

// Run by the first wave of a workgroup.  Each lane owns up to 8 consecutive groups; one wave-wide scan of row
// counts and one of each of the two tile counts.  Every size is clamped to [0, tokens] before it enters a
// sum, and sums of rows stay at 2^32 - 1 once they are there (tokens is below 2^31), so no size vector can make a
// sum overflow or a group start before row 0 or end past row `tokens`.
// Every launch starts with this: 2.4 us of the 7 of a small one, most of it in divisions, 1.3 without them
// and with data-parallel moves for the scans.
template <int LAYOUT, int BM, int BN>
__device__ __forceinline__ void build_schedule(Sched* s, const GmmParams& p, const HostSizes& hs, int w) {
  const int lane = threadIdx.x;
  if (lane >= 64) return;
  const int E = p.num_groups;
  const int per = (E + 63) >> 6;
  const int e0 = lane * per;
  const uint32_t tokens = (uint32_t)p.tokens;
  int bad = 0;   // kStatus* bits seen by this lane
  auto clamp = [&](int64_t v) {
    if (v < 0) bad |= kStatusNegativeSize;
    if (v > p.tokens) bad |= kStatusRowsPastEnd;
    return v < 0 ? 0u : (v > p.tokens ? tokens : (uint32_t)v);
  };
  auto add = [](uint32_t x, uint32_t y) { return x + y; };
  auto add_sat = [](uint32_t x, uint32_t y) { return __builtin_elementwise_add_sat(x, y); };
  auto larger = [](uint32_t x, uint32_t y) { return x > y ? x : y; };
  // rows taken by the groups before this launch's first one
  uint32_t base = (uint32_t)(p.row_base < (int64_t)0xffffffffll ? p.row_base : (int64_t)0xffffffffll);
  if (p.sizes_dev != nullptr && p.first_group > 0) {
    uint32_t part = 0;
    for (int i = lane; i < p.first_group; i += 64) part = add_sat(part, clamp(p.sizes_dev[i]));
    base = (uint32_t)__builtin_amdgcn_readlane((int)wave_scan(part, add_sat), 63);
  }
  uint32_t sz[8];
  uint32_t sum = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    sz[i] = 0;
    if (i < per) {   // (the same in every lane: groups that no lane has cost nothing)
      const int e = e0 + i;
      if (e < E) sz[i] = clamp(p.sizes_dev != nullptr ? p.sizes_dev[p.first_group + e] : (int64_t)hs.v[e]);
      sum = add_sat(sum, sz[i]);
    }
  }
  // (what the lanes before this one add up to, not this one's sum less: sums may be at their limit)
  uint32_t run = wave_scan(sum, add_sat);
  const uint32_t all = add_sat(base, (uint32_t)__builtin_amdgcn_readlane((int)run, 63));
  run = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)run, 0x138, 0xf, 0xf, false);   // wave_shr:1
  run = add_sat(base, run);
  uint32_t main_tiles[8], runt_tiles[8];
  uint32_t tsum = 0, rsum = 0, most = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    main_tiles[i] = runt_tiles[i] = 0;
    if (i < per) {
      const int e = e0 + i;
      const uint32_t start = run < tokens ? run : tokens, left = tokens - start;
      const uint32_t rows = sz[i] < left ? sz[i] : left;
      if (e < E) {
        s->row_start[e] = (int)start;
        s->rows[e] = (int)rows;
        const GroupTiles g = group_tiles<LAYOUT, BM, BN>((int)rows, p.hidden_in, p.hidden_out, p.flags);
        main_tiles[i] = (uint32_t)(g.main_rows * g.tiles_n);
        runt_tiles[i] = (uint32_t)(g.runt * g.tiles_n);
        most = larger(most, rows);
      }
      tsum += main_tiles[i];
      rsum += runt_tiles[i];
      run = add_sat(run, sz[i]);
    }
  }
  const uint32_t tincl = wave_scan(tsum, add), rincl = LAYOUT == kTN ? 0u : wave_scan(rsum, add);
  most = wave_scan(most, larger);
  uint32_t trun = tincl - tsum, rrun = rincl - rsum;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (i < per) {
      const int e = e0 + i;
      if (e < E) {
        s->tile_start[e] = (int)trun;
        s->runt_start[e] = (int)rrun;
      }
      trun += main_tiles[i];
      rrun += runt_tiles[i];
    }
  }
  if (lane == 0) s->group_tiles = (int)main_tiles[0];   // (weight-gradient layout: the same for every group)
  if (lane == 63) {
    s->front_tiles = 0;
    s->front_pieces = 1;
    s->cut_groups = 0;
    s->most_rows = (int)most;
    s->row_start[E] = (int)(all < tokens ? all : tokens);
    s->tile_start[E] = (int)tincl;
    s->runt_start[E] = (int)rincl;
    if (all > tokens) bad |= kStatusRowsPastEnd;
  }
  // What the host would have rejected in host-resident sizes is reported for device-resident
  // ones: one workgroup ORs what its first wave saw into the caller's status word.
  if (p.status != nullptr && w == 0) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) bad |= __shfl_xor(bad, d);
    if (lane == 0 && bad != 0) atomicOr(p.status, bad);
  }
}

// Weight-gradient layout: the groups by descending depth, groups of equal depth in their own order
// (what the reference's stable sort gives).  Run by every thread of the workgroup after
// build_schedule and a barrier; ends with a barrier.  `keys` is scratch for kMaxGroups 64-bit
// words (the tile buffers are not in use yet).
__device__ __forceinline__ void order_groups_by_depth(Sched* s, int num_groups, uint64_t* keys) {
  // Up to a few hundred groups it is quicker to count, per group, the groups that go before it
  // (measured equal at 256 groups, 12 us slower than the sort at 512): straight from
  // Sched::rows, nothing written to `keys` (with the row counts copied there first the compiler
  // built a different and 4-6 % slower depth loop for this layout).
  if (num_groups <= 256) {
    for (int e = threadIdx.x; e < num_groups; e += blockDim.x) {
      const int mine = s->rows[e];
      int before = 0;
      auto count = [&](int other, int j) { before += (other > mine || (other == mine && j < e)) ? 1 : 0; };
      int j = 0;
      for (; j + 8 <= num_groups; j += 8) {   // (eight reads in flight, the same addresses in every lane)
        int other[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) other[k] = s->rows[j + k];
#pragma unroll
        for (int k = 0; k < 8; ++k) count(other[k], j + k);
      }
      for (; j < num_groups; ++j) count(s->rows[j], j);
      s->order[before] = (int16_t)e;
    }
    __syncthreads();
    return;
  }
  // A bitonic sort in LDS of one 64-bit word per group, depth above and 0xffff - index below.
  int n = 2;
  while (n < num_groups) n <<= 1;
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    keys[i] = i < num_groups ? ((uint64_t)(uint32_t)s->rows[i] << 16) | (uint64_t)(0xffff - i) : 0;   // padding sorts last
  __syncthreads();
  for (int k = 2; k <= n; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int partner = i ^ j;
        if (partner > i) {
          const uint64_t x = keys[i], y = keys[partner];
          const bool descending = (i & k) == 0;
          if (descending ? x < y : x > y) {
            keys[i] = y;
            keys[partner] = x;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < num_groups; i += blockDim.x) s->order[i] = (int16_t)(0xffff - (int)(keys[i] & 0xffff));
  __syncthreads();
}

// Weight-gradient layout with a workspace, after order_groups_by_depth: the deepest tiles in depth pieces (cut_deep_tiles), which
// are handed out first, one per workgroup (Zipf depths: the deepest tile 227 slices, 144 slices of work per workgroup).  Run
// by every thread; the same answer in each.
template <int BM, int BN>
__device__ __forceinline__ void plan_deep_tiles(Sched* s, const GmmParams& p, int grid, int bk, TailPlan* plan) {
  const int E = p.num_groups;
  const int tiles = s->tile_start[E];
  if (E == 0 || tiles == 0 || p.ws_slots <= 0 || (p.flags & (kFlagWholeTiles | kFlagRowPieces))) return;
  const DeepCut cut = cut_deep_tiles([&](int q) { return (s->rows[s->order[q]] + bk - 1) / bk; }, E,
                                     (int64_t)s->row_start[E] - s->row_start[0], tiles / E, grid, p.ws_slots,
                                     min_slices_per_piece(BM * BN), bk);   // (every group has the same number of tiles here)
  const int pieces = cut.pieces, front = cut.tiles;
  if (front == 0) return;
  s->front_tiles = front;     // (every thread writes the same two values, and reads its own wave's)
  s->front_pieces = pieces;
  plan->pieces = 1;   // the last round stays whole: a workgroup has at most one tile to fix
  plan->by_depth = true;
  plan->main_tiles = plan->total = front * pieces + (tiles - front);
}

// x / y, rounded up, for small quotients
__device__ __forceinline__ uint32_t ceil_quotient(uint32_t x, uint32_t y) {
  uint32_t q = (uint32_t)((float)x * __builtin_amdgcn_rcpf((float)y));   // (one off at most)
  q += q * y < x ? 1 : 0;
  q += q * y < x ? 1 : 0;
  return q - (q > 0 && (q - 1) * y >= x ? 1 : 0);
}
__device__ __forceinline__ uint32_t wave_sums(uint32_t x) {
  return wave_scan(x, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ uint32_t lane_of(uint32_t x, int lane) { return (uint32_t)__builtin_amdgcn_readlane((int)x, lane); }

// What a launch's groups hold, in LDS: depth[q] of position q of the order, upto[q] the sum of those before it.
struct GroupDepths {
  const uint32_t *depth, *upto;
  uint32_t groups, sum;
  __device__ __forceinline__ uint32_t at(uint32_t q) const { return q < groups ? depth[q] : 0; }
  __device__ __forceinline__ uint32_t first(uint32_t n) const { return n < groups ? upto[n] : sum; }
};

// ... and with kFlagPiecesByLength: pieces of one length (pieces_end).  All lengths are looked at together, eight lanes each: one
// after the other, each with sums over the lanes that wait for those before, they were 3 us of every such launch.  A lane for each
// length and every group in a lane took 1 us, and so many scalar registers that others were spilled all over the pair kernels (1.2 us of
// launches that cut nothing).  us per launch, plan_deep_tiles / this one: 21 Zipf (1.2) groups, 51204 rows, 128 x 560: 46 / 32; 56, 19094
// rows, 704 x 1376: 124 / 90; 64, 49152 rows, 2048 x 1408: 331 / 310; 7 even groups, 44642 rows, 360 x 424: 38.0 / 30.7; 4 of 8483, 128 x
// 1384: 31.2 / 30.0; 2 of 20000, 256 x 1408: 49.6 / 44.3; 15, 40804, 416 x 136 (cut as the last round by both): 24.5 / 23.3.
// `scratch` is for 2 kMaxGroups words (the tile buffers are not in use yet); ends with a barrier.
template <int BM, int BN, int WGS_PER_CU>
__device__ __forceinline__ void plan_pieces_by_length(Sched* s, const GmmParams& p, int grid, int bk, uint32_t* scratch, TailPlan* plan) {
  const int E = p.num_groups, tiles = s->tile_start[E], per_group = s->group_tiles, lane = threadIdx.x & 63;
  if (E == 0 || tiles == 0 || p.ws_slots <= 0 || (p.flags & (kFlagWholeTiles | kFlagRowPieces))) return;
  // (every wave works out the same plan and writes the same words)
  uint32_t *depth = scratch, *upto = scratch + kMaxGroups;
  const int per = (E + 63) >> 6;
  auto depth_of = [&](int q) { return q < E ? (uint32_t)(s->rows[s->order[q]] + bk - 1) / bk : 0u; };
  const uint32_t deepest = (uint32_t)uniform((int)depth_of(0));
  if (deepest < 4 * PieceCosts<BM * BN>::SHORTEST) return;
  uint32_t sum = 0;
#pragma unroll 1
  for (int i = 0; i < per; ++i) {
    const int q = lane + 64 * i;
    const uint32_t d = depth_of(q), up = wave_sums(d);
    depth[q] = d;
    upto[q] = sum + up - d;
    sum += lane_of(up, 63);
  }
  __syncthreads();   // (all lanes' words are there, and tile_start has been read by every wave)
  // Eight lanes to each length, every eighth group for each of them.
  static_assert(kPieceLengths == 8, "");
  const int k = lane / 8, n = piece_count<BM * BN>(k);
  const uint32_t length = (deepest + n - 1) / n;
  uint32_t cut = 0, pieces = 0;
#pragma unroll 1
  for (int q = lane % 8;; q += 8) {
    const uint32_t d = q < E ? depth[q] : 0;
    const bool yes = is_cut(d, length);
    if (__ballot(yes) == 0) break;   // (nor any of the groups behind these)
    cut += yes ? 1 : 0;
    pieces += yes ? ceil_quotient(d, length) : 0;
  }
#pragma unroll
  for (int d = 1; d < 8; d *= 2) cut += (uint32_t)__shfl_xor((int)cut, d), pieces += (uint32_t)__shfl_xor((int)pieces, d);
  const GroupDepths depths{depth, upto, (uint32_t)E, sum};
  const PieceLaunch launch{tiles, per_group, grid, grid / WGS_PER_CU, p.ws_slots};
  const float share = ((float)sum * per_group + PieceCosts<BM * BN>::TILE * tiles) / grid;
  const float end = pieces_end<BM * BN>(depths, launch, n, (int)length, (int)cut, (int)pieces, share);
  const float uncut = uncut_end<BM * BN>(depths, launch, plan->by_depth && plan->main_tiles == 0 ? plan->pieces : 1, share);
  // the least, the first of equals: by its bits, the lowest three of which are its number
  const uint32_t mine = (__builtin_bit_cast(uint32_t, end) & ~7u) | (uint32_t)k;
  const uint32_t least = ~lane_of(wave_scan(~mine, [](uint32_t a, uint32_t b) { return a > b ? a : b; }), 63);
  const int chosen = uniform(__builtin_bit_cast(float, least & ~7u) < kPiecesPay * uncut ? (int)(least & 7u) * 8 : -1);
  if (chosen >= 0) {
    const int l = (int)lane_of(length, chosen), groups = (int)lane_of(cut, chosen), all = (int)lane_of(pieces, chosen);
    uint32_t start = 0;
#pragma unroll 1
    for (int i = 0; 64 * i < groups; ++i) {
      const int q = lane + 64 * i;
      const uint32_t of_tile = q < groups ? ceil_quotient(depth[q], l) : 0, up = wave_sums(of_tile);
      if (q < groups) {
        s->tile_start[q] = (int)(start + up - of_tile) * per_group;
        s->runt_start[q] = (int)of_tile;
      }
      start += lane_of(up, 63);
    }
    s->tile_start[groups] = all * per_group;
    s->front_tiles = all * per_group;
    s->front_pieces = 0;
    s->cut_groups = groups;
    plan->pieces = 1;   // the last round stays whole: a workgroup has at most one tile to fix
    plan->by_depth = true;
    plan->main_tiles = plan->total = all * per_group + (tiles - groups * per_group);
  }
  __syncthreads();   // (find_tile's lanes read what other lanes have written; the scratch is free again)
}

// NN and NT layouts with many short groups: the groups by ascending number of tile rows, groups
// of equal number in their own order.  Where group sizes straddle a multiple of the tile height,
// groups of k and of k + 1 tile rows alternate at random in group order; with equal groups side by
// side such launches measured 2-5 % faster (tile indices are dealt to the XCDs in runs of 32 and
// walk a group in bands of tile rows: runs and bands then cut every group the same way).  A
// launch with a group of more than kMaxTileRowsForOrder tile rows (Zipf-like sizes) keeps the
// group order: there it measured 1-2 % slower.  The tile prefix sums are counted again, in the
// new order (the first wave, as in build_schedule; the totals do not change).
constexpr int kMaxTileRowsForOrder = 8;

template <int LAYOUT, int BM, int BN>
__device__ __forceinline__ void order_groups_by_tile_rows(Sched* s, const GmmParams& p) {
  const int E = p.num_groups;
  // A counting sort with one bucket per number of tile rows, by the first wave: each lane owns up
  // to 8 consecutive groups, counts them by bucket, and one wave-wide scan per bucket gives every
  // group its place (about a microsecond, where ranking the groups one against the other took 12).
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const int per = (E + 63) >> 6;
    const int e0 = lane * per;
    if (s->most_rows > kMaxTileRowsForOrder * BM) {
      for (int i = 0; i < per; ++i)
        if (e0 + i < E) s->order[e0 + i] = (int16_t)(e0 + i);
    } else {
      constexpr int BUCKETS = kMaxTileRowsForOrder + 1;
      int key[8], count[BUCKETS];
#pragma unroll
      for (int b = 0; b < BUCKETS; ++b) count[b] = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        key[i] = (i < per && e0 + i < E) ? (s->rows[e0 + i] + BM - 1) / BM : -1;
#pragma unroll
        for (int b = 0; b < BUCKETS; ++b) count[b] += key[i] == b ? 1 : 0;
      }
      int next[BUCKETS];   // where this lane's next group of a bucket goes
      int base = 0;
#pragma unroll
      for (int b = 0; b < BUCKETS; ++b) {
        int incl = count[b];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const int o = __shfl_up(incl, d);
          if (lane >= d) incl += o;
        }
        next[b] = base + incl - count[b];
        base += __shfl(incl, 63);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        int at = -1;
#pragma unroll
        for (int b = 0; b < BUCKETS; ++b) {
          if (key[i] == b) {
            at = next[b];
            next[b] += 1;
          }
        }
        if (at >= 0) s->order[at] = (int16_t)(e0 + i);
      }
    }
  }
  __syncthreads();
  const int lane = threadIdx.x;
  if (lane < 64) {
    const int per = (E + 63) >> 6;
    const int q0 = lane * per;
    int tsum = 0, rsum = 0;
    for (int i = 0; i < per; ++i) {
      const int q = q0 + i;
      if (q < E) {
        const GroupTiles g = group_tiles<LAYOUT, BM, BN>(s->rows[s->order[q]], p.hidden_in, p.hidden_out, p.flags);
        tsum += g.main_rows * g.tiles_n;
        rsum += g.runt * g.tiles_n;
      }
    }
    int tincl = tsum, rincl = rsum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(tincl, d);
      const int o2 = __shfl_up(rincl, d);
      if (lane >= d) {
        tincl += o;
        rincl += o2;
      }
    }
    int trun = tincl - tsum, rrun = rincl - rsum;
    for (int i = 0; i < per; ++i) {
      const int q = q0 + i;
      if (q < E) {
        s->tile_start[q] = trun;
        s->runt_start[q] = rrun;
        const GroupTiles g = group_tiles<LAYOUT, BM, BN>(s->rows[s->order[q]], p.hidden_in, p.hidden_out, p.flags);
        trun += g.main_rows * g.tiles_n;
        rrun += g.runt * g.tiles_n;
      }
    }
  }
  __syncthreads();
}

// Element offsets of a group's A, B and C blocks, the quantities of the reference's
// problem table (csrc/fill_arguments.cuh:72-76) in int64.  The kernel addresses memory
// through these and the schedule dump prints these.
struct GroupGeom {
  int64_t a_off, b_off, c_off;
  int32_t m, n, k;
  int32_t row0;   // first row of the group in a (and in c, unless c is the weight gradient)
};

// `e` is the group's index among all groups of the call; `start` and `rows` are the group's
// entries of Sched::row_start and Sched::rows.
template <int LAYOUT>
__device__ __forceinline__ GroupGeom group_geometry(const GmmParams& p, int e, int64_t start,
                                                    int rows) {
  GroupGeom g;
  const int64_t hin = p.hidden_in, hout = p.hidden_out;
  g.row0 = (int32_t)start;
  if (LAYOUT == kTN) {
    g.m = p.hidden_in;
    g.n = p.hidden_out;
    g.k = rows;
    g.a_off = start * p.lda;
    g.b_off = start * p.ldb;
    g.c_off = (int64_t)e * hin * hout;
  } else {
    g.m = rows;
    g.n = p.hidden_out;
    g.k = p.hidden_in;
    g.a_off = start * p.lda;
    g.b_off = (int64_t)e * (LAYOUT == kNT ? (int64_t)p.b_cols : hin) * p.ldb;
    g.c_off = start * hout;
  }
  return g;
}

// In-group tile order: bands of `group_m` tile rows, tile rows fastest inside a band, so
// that tiles running at the same time share A rows and B columns in L2.
__device__ __forceinline__ void tile_coords(int u, int tiles_m, int tiles_n, int group_m,
                                            int* tm, int* tn) {
  const int per_band = group_m * tiles_n;
  const int band = u / per_band;
  const int first_m = band * group_m;
  const int left = tiles_m - first_m;
  const int gsz = left < group_m ? left : group_m;
  const int r = u - band * per_band;
  *tm = first_m + r % gsz;
  *tn = r / gsz;
}

template <int LAYOUT, int BM, int BN>
__global__ __launch_bounds__(64) void schedule_dump_kernel(GmmParams p, HostSizes hs) {
  __shared__ Sched s;
  __shared__ uint64_t sort_keys[kMaxGroups];
  build_schedule<LAYOUT, BM, BN>(&s, p, hs, (int)blockIdx.x);
  __syncthreads();
  const bool ordered = LAYOUT == kTN || (p.flags & kFlagByTileRows) != 0;
  if (LAYOUT == kTN) {
    order_groups_by_depth(&s, p.num_groups, sort_keys);
  } else if (ordered) {
    order_groups_by_tile_rows<LAYOUT, BM, BN>(&s, p);
  }
  for (int e = threadIdx.x; e < p.num_groups; e += 64) {
    const GroupGeom g = group_geometry<LAYOUT>(p, p.first_group + e, s.row_start[e], s.rows[e]);
    const GroupTiles gt = group_tiles<LAYOUT, BM, BN>(s.rows[e], p.hidden_in, p.hidden_out, p.flags);
    int64_t* row = p.sched_out + (int64_t)e * kSchedCols;
    row[0] = g.m;
    row[1] = g.n;
    row[2] = g.k;
    row[3] = LAYOUT == kTN ? g.m : g.k;  // lda: column-major A has ld = rows
    row[4] = LAYOUT == kNT ? g.k : g.n;  // ldb
    row[5] = g.n;                        // ldc
    row[6] = g.a_off;
    row[7] = g.b_off;
    row[8] = g.c_off;
    int position = e;   // where the group's tiles stand in the order they are handed out
    if (ordered) {
      for (int q = 0; q < p.num_groups; ++q)
        if (s.order[q] == e) position = q;
    }
    row[9] = s.tile_start[position];
    row[10] = gt.tiles_m * gt.tiles_n;
    row[11] = s.rows[e];
    row[12] = s.tile_start[p.num_groups] + s.runt_start[position];
    row[13] = gt.runt * gt.tiles_n;
  }
}

// ------------------------------------------------------------ operand tile movers
//
// Two kinds of operand tile, by which dimension is contiguous in memory.
//
// DepthMajor ("KC"): R rows (M or N index) of BK depth elements, depth contiguous.  LDS
// keeps row-major rows of BK*2 bytes; the 16-byte chunk c of row r sits at chunk slot
// c ^ ((r / RP) % CPR), which makes 16 consecutive rows at one depth hit 64 distinct
// banks for ds_read_b128.
//
// WidthMajor ("MC"): BK depth rows of W elements (M or N index contiguous).  LDS keeps
// row-major rows of W*2 bytes; 64-byte segment s of depth row k sits at segment slot
// s ^ (k & 3), and rows 8 .. 15 of every 16 start 32 bytes later (row_at), so the 8 depth rows (k .. k + 3 and
// 8 below them) of which half a wave reads 16 columns at a time land in distinct groups of 8 banks, and the second
// 16 columns of a block are 32 bytes behind the first ones in every lane.
//
// A lane's LDS slot is fixed by the hardware (wave base + lane * 16), so the swizzle is
// applied by choosing which global chunk each lane fetches.

// GATHER: rows come through an index (or in place) at byte offsets kept per load, relative to
// the start of the whole tensor.  GATE_UP (B of the NT layout with gate | up rows): the tile's R
// rows are 32-row blocks taken alternately from the gate rows and, `up_step` bytes further, the
// up rows of b, so that a wave finds the gate and the up value of an output column side by side.
template <int R, int BK, int NT, bool GATHER = false, bool GATE_UP = false>
struct DepthMajor {
  static constexpr int CPR = BK / 8;                                  // chunks per row
  static constexpr int RP = (BK * 2 >= 256) ? 1 : 256 / (BK * 2);     // rows per 256 B
  static constexpr int ROWS_PER_INSTR = NT / CPR;
  static constexpr int NI = R * CPR / NT;                             // loads per lane per tile
  static constexpr int BYTES = R * BK * 2;
  static_assert(NT % CPR == 0 && (R * CPR) % NT == 0, "tile does not split over the block");
  static_assert(ROWS_PER_INSTR % (RP * CPR) == 0, "swizzle must not depend on the load index");

  const char* base;   // first row of the tile, next depth slice
  int ld;             // elements between rows ( = depth extent )
  int span;           // elements from the tile's first row to its last existing row
  int depth;          // depth values ahead of the cursor (below 0: past the end)
  int my_chunk;       // depth chunk (of 8) this lane fetches
  uint32_t voff0;     // byte offset of this lane's chunk for load 0
  uint32_t vrow[GATHER ? NI : 1];   // GATHER: byte offset of this lane's chunk per load
  uint32_t total_bytes;             // GATHER: bytes of the whole tensor
  uint32_t up_step;                 // GATE_UP: bytes from a gate row to its up row

  __device__ __forceinline__ void setup(const char* tile_base, int ld_, int rows_valid_, int depth_) {
    base = tile_base;
    ld = ld_;
    span = rows_valid_ > 0 ? (rows_valid_ - 1) * ld_ : -(1 << 30);   // no rows: nothing in range
    depth = depth_;
    const int tid = threadIdx.x;
    const int row = tid / CPR, pos = tid % CPR;
    my_chunk = pos ^ ((row / RP) % CPR);
    voff0 = (uint32_t)(row * ld + my_chunk * 8) * 2u;
  }

  // GATHER: the tile's row r is row rows[r] of the tensor at `tensor_base` (of tensor_rows rows)
  // when `rows` is given, row first_row + r otherwise; rows past rows_valid_ are out of range.
  __device__ __forceinline__ void setup_gather(const char* tensor_base, uint32_t tensor_bytes,
                                               const int32_t* rows, uint32_t tensor_rows, int first_row, int ld_,
                                               int rows_valid_, int depth_) {
    base = tensor_base;
    ld = ld_;
    span = 0;
    depth = depth_;
    total_bytes = tensor_bytes;
    const int tid = threadIdx.x;
    const int row = tid / CPR, pos = tid % CPR;
    my_chunk = pos ^ ((row / RP) % CPR);
    voff0 = 0;
#pragma unroll
    for (int i = 0; i < (GATHER ? NI : 1); ++i) {
      const int r = row + i * ROWS_PER_INSTR;
      uint32_t v = kOutOfRangeIndexed;
      if (r < rows_valid_) {
        const uint32_t src = rows != nullptr ? (uint32_t)rows[r] : (uint32_t)(first_row + r);
        // (an index that names no row of the tensor, negative ones included: a row of zeros)
        if (src < tensor_rows) v = (src * (uint32_t)ld_ + (uint32_t)(my_chunk * 8)) * 2u;
      }
      vrow[i] = v;
    }
  }

  // GATE_UP: `tile_base` is the tile's first gate row; rows_valid_ counts rows to the end of the
  // up rows of the group, so that the descriptor ends where the group's b ends.
  __device__ __forceinline__ void setup_gate_up(const char* tile_base, int ld_, int rows_valid_, int depth_,
                                                int out_cols) {
    setup(tile_base, ld_, rows_valid_, depth_);
    up_step = (uint32_t)out_cols * (uint32_t)ld_ * 2u;
  }

  // Skip the first `slices` depth slices.
  __device__ __forceinline__ void skip(int slices) {
    base += (int64_t)slices * (BK * 2);
    depth -= slices * BK;
    if constexpr (GATHER) total_bytes = total_bytes > (uint32_t)slices * (BK * 2) ? total_bytes - (uint32_t)slices * (BK * 2) : 0u;
  }
  // What all loads of a depth slice share.
  struct Slice {
    rsrc_words rsrc;
    uint32_t v0;   // this lane's offset for load 0, or out of range in the depth tail
  };
  // The next slice (past the depth: empty).
  __device__ __forceinline__ Slice slice() {
    const int left = depth = uniform(depth);
    base = uniform_ptr(base);
    Slice sl;
    if constexpr (GATHER) {
      // the descriptor spans the tensor from this slice's first byte on; v0 is 0 for a chunk
      // inside the depth and out of range for one past it
      sl.rsrc = make_rsrc_words(base, left > 0 ? total_bytes : 0u);
      sl.v0 = (left >= BK || my_chunk * 8 < left) ? 0u : kOutOfRangeIndexed;
    } else {
      const int elems = left > 0 ? span + left : 0;
      sl.rsrc = make_rsrc_words(base, elems > 0 ? (uint32_t)elems * 2u : 0u);
      sl.v0 = (left >= BK || my_chunk * 8 < left) ? voff0 : kOutOfRange;
    }
    skip(1);
    return sl;
  }
  // Load I of the NI that make up one slice goes kOffset<I> bytes behind wave_at of this wave in the LDS tile.
  __device__ static constexpr __forceinline__ int wave_at(int wave) { return wave * 64 * 16; }
  template <int I>
  static constexpr int kOffset = I * NT * 16;
  template <int I, bool RIGHT_BEHIND>
  __device__ __forceinline__ void load(const Slice& sl) const {
    const uint32_t step = (uint32_t)(ROWS_PER_INSTR * ld) * 2u;
    uint32_t v;
    if constexpr (GATHER) {
      v = vrow[I] | sl.v0;   // either flag pushes the offset out of range
    } else if constexpr (GATE_UP) {
      static_assert(ROWS_PER_INSTR == 32, "one load instruction per 32-row block");
      v = sl.v0 + (I / 2) * step + (I % 2) * up_step;
    } else {
      v = sl.v0 + I * step;
    }
    load_to_lds_16<RIGHT_BEHIND>(sl.rsrc, v);
  }

  // A depth that is even but no multiple of 8: the 16-byte chunk that holds a row's last depth
  // values also holds the first values of the next row in memory (only behind the last row does the
  // descriptor end).  Once the slice with that chunk has landed, every thread clears the foreign
  // dwords of its rows' chunks in the LDS tile at `tile`, so that nothing of another row, not even
  // a NaN against a zero, reaches a sum.  tail = depth values of the slice that exist.
  __device__ static __forceinline__ void clear_depth_tail(char* tile, int tail) {
    const int chunk = tail >> 3, first_dword = (tail & 7) >> 1;
    for (int row = threadIdx.x; row < R; row += NT) {
      uint32_t* at = reinterpret_cast<uint32_t*>(tile + row * (BK * 2) + ((chunk ^ ((row / RP) % CPR)) << 4));
#pragma unroll
      for (int d = 1; d < 4; ++d)
        if (d >= first_dword) at[d] = 0u;
    }
  }
};

// F8 (one-byte elements, seen two to one as W two-byte elements per depth row): 32-byte segment
// s of depth row k sits at segment slot s ^ (k & 7), so the 8 depth rows one byte-wise
// transposing read touches land in 8 distinct groups of 8 banks.
constexpr int width_major_bytes(int W, int BK, bool f8) { return W * BK * 2 + (f8 ? 0 : BK / 16 * 64); }
//
// The offset of a lane's chunk differs from load to load by whole rows only, so ONE_OFFSET holds that of load 0 and adds the rest.  An
// addition ahead of every load costs full tiles of many slices 3 % (8 x 4096 rows, 4096 x 14336: 2621 us against 2720), and is
// for the kernel that would spill the offsets: reading, adding and writing fp32 leaves no registers for them.
template <int W, int BK, int NT, bool F8 = false, bool ONE_OFFSET = false>
struct WidthMajor {
  static constexpr int CPRW = W / 8;                  // chunks per depth row
  static constexpr int ROWS_PER_INSTR = NT / CPRW;
  static constexpr int ROWS_PER_WAVE = 64 / CPRW;     // ... of them by one wave
  static constexpr int NI = BK * CPRW / NT;
  static constexpr int BYTES = width_major_bytes(W, BK, F8);
  static constexpr int PITCH = W * 2;
  static_assert(NT % CPRW == 0 && (BK * CPRW) % NT == 0, "tile does not split over the block");
  static_assert(CPRW >= 16 && 8 % ROWS_PER_WAVE == 0, "at least 4 segments of 64 bytes; a wave's rows are all shifted or none");

  // where depth row k starts in LDS
  __device__ static constexpr __forceinline__ int row_at(int k) {
    return F8 ? k * PITCH : k * PITCH + 32 * ((k >> 3) & 1) + 64 * (k >> 4);
  }
  // which 16-byte chunk of depth row krow the lane whose LDS slot is chunk p fetches
  __device__ static __forceinline__ int chunk_for_slot(int p, int krow) {
    if constexpr (F8) {
      static_assert(!F8 || CPRW == 16, "8 segments of 32 bytes per depth row");
      return (((p >> 1) ^ (krow & 7)) << 1) | (p & 1);
    } else {
      return (((p >> 2) ^ (krow & 3)) << 2) | (p & 3);
    }
  }

  const char* base;      // depth row of the next slice, column 0
  int ld;                // elements between depth rows
  int depth;             // depth rows of the group ahead of the cursor (below 0: past the end)
  uint32_t voff[ONE_OFFSET ? 1 : NI];   // byte offset of this lane's chunk per load (kOutOfRange past the width)

  __device__ __forceinline__ void setup(const char* group_base, int ld_, int depth_, int col0,
                                        int width) {
    base = group_base;
    ld = ld_;
    depth = depth_;
    const int tid = threadIdx.x;
    const int krow0 = tid / CPRW, p = tid % CPRW;
#pragma unroll
    for (int i = 0; i < (ONE_OFFSET ? 1 : NI); ++i) {
      const int krow = krow0 + i * ROWS_PER_INSTR;
      const int c = chunk_for_slot(p, krow);
      const int col = col0 + c * 8;
      voff[i] = col < width ? (uint32_t)(krow * ld + col) * 2u : kOutOfRange;
    }
  }

  // B of the NN layout with gate | up columns: the tile's W columns are 32-column blocks taken
  // alternately from the gate columns [0, out_cols) and the up columns [out_cols, 2 out_cols) of
  // the group's b; col0 is the tile's first output column, ld_ = 2 * out_cols.
  __device__ __forceinline__ void setup_gate_up(const char* group_base, int ld_, int depth_, int col0,
                                                int out_cols) {
    base = group_base;
    ld = ld_;
    depth = depth_;
    const int tid = threadIdx.x;
    const int krow0 = tid / CPRW, p = tid % CPRW;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int krow = krow0 + i * ROWS_PER_INSTR;
      static_assert(!F8 && !ONE_OFFSET, "gate | up columns are for two-byte elements");
      const int c = chunk_for_slot(p, krow);   // 16-byte chunk of the tile row
      const int block = c >> 2;                                        // 32-column block of the tile
      const int out = col0 + (block >> 1) * 32 + (c & 3) * 8;          // output column it belongs to
      const int col = (block & 1) * out_cols + out;
      voff[i] = out < out_cols ? (uint32_t)(krow * ld + col) * 2u : kOutOfRange;
    }
  }

  __device__ __forceinline__ void skip(int slices) {
    base += (int64_t)slices * BK * ld * 2;
    depth -= slices * BK;
  }
  struct Slice {
    rsrc_words rsrc;
  };
  __device__ __forceinline__ Slice slice() {
    const int left = uniform(depth), row = uniform(ld) * 2;
    base = uniform_ptr(base);
    Slice sl;
    int rows;   // 0 .. BK (in assembly: the compiler would work it out in vector registers)
    asm("s_min_i32 %0, %1, %2\n\ts_max_i32 %0, %0, 0" : "=&s"(rows) : "s"(left), "n"(BK) : "scc");
    sl.rsrc = make_rsrc_words(base, (uint32_t)(rows * row));
    base += BK * row;
    depth = left - BK;
    return sl;
  }
  // (the rows of an instruction are a multiple of 8 apart from those of the next one)
  static_assert(ROWS_PER_INSTR % 8 == 0 && (F8 || ROWS_PER_INSTR % 16 == 0 || ROWS_PER_INSTR * 2 == 16), "");
  __device__ static constexpr __forceinline__ int wave_at(int wave) { return row_at(wave * ROWS_PER_WAVE); }
  template <int I>
  static constexpr int kOffset = row_at(I * ROWS_PER_INSTR);
  template <int I, bool RIGHT_BEHIND>
  __device__ __forceinline__ void load(const Slice& sl) const {
    if constexpr (ONE_OFFSET) {
      // (rows of up to 2^22 values: past the width it stays between 2^31 and 2^32, beyond every descriptor)
      static_assert((uint64_t)(BK - 1) * (F8 ? 1 : 2) * (1 << 22) < kOutOfRange, "");
      load_to_lds_16<RIGHT_BEHIND>(sl.rsrc, voff[0] + I * ((uint32_t)(ROWS_PER_INSTR * ld) * 2u));
    } else {
      load_to_lds_16<RIGHT_BEHIND>(sl.rsrc, voff[I]);
    }
  }
};

// ---------------------------------------------------------------- fragment readers
// A fragment is the operand of one 16x16x32 MFMA: lane l holds 8 depth values
// 8*(l/16) .. +7 of row (or column) l % 16.  A wave's rows and columns come in blocks of 32, so the two
// fragments of a block and of 32 depth values are numbered by "step": 2 s + h is half h (rows 16 h .. +15) of the
// block at 32-deep step s.

// STRIDE: distance between the blocks a wave owns, in 32-wide blocks (the waves along a
// dimension take blocks alternately when STRIDE is their number, contiguously when it is 1).
// F8: one-byte elements.  A row of the tile is then 128 depth values, and the fragment of one
// 32x32x64 instruction is 32 consecutive bytes of it (depth 32 (l / 32) .. +31 of a 64-deep step),
// read as two 16-byte halves: "step" 2 s + h below is half h of 64-deep step s.
template <int BK, int STRIDE, bool F8 = false>
struct DepthMajorFrag {
  static constexpr int CPR = BK / 8;
  static constexpr int RP = (BK * 2 >= 256) ? 1 : 256 / (BK * 2);
  static_assert((16 / RP) % CPR == 0, "blocks and their halves must share the swizzle of block 0");
  static constexpr int OFFSETS = F8 ? BK / 16 : BK / 32;
  uint32_t off[OFFSETS];   // lane offset per step (two-byte elements: per pair of them), block 0

  __device__ __forceinline__ void setup(int first_row) {
    const int lane = threadIdx.x & 63;
    const int row = first_row + (F8 ? lane & 31 : lane & 15);
    const int sw = (row / RP) % CPR;
#pragma unroll
    for (int n = 0; n < OFFSETS; ++n) {
      const int chunk = F8 ? 4 * (n / 2) + 2 * (lane >> 5) + n % 2 : 4 * n + (lane >> 4);
      off[n] = (uint32_t)(row * (BK * 2) + ((chunk ^ sw) << 4));
    }
  }
  __device__ __forceinline__ bf16x8 read(const char* tile, int ks, int blk) const {
    const int first = blk * (STRIDE * 32) + (F8 ? 0 : 16 * (ks % 2));
    return *reinterpret_cast<const bf16x8*>(tile + off[F8 ? ks : ks / 2] + first * (BK * 2));
  }
};

template <int W, int BK, int NBLK, int STRIDE>
struct WidthMajorFrag {
  static constexpr int PITCH = W * 2;
  using Tile = WidthMajor<W, BK, 256>;
  // blocks whose segments differ in what the swizzle changes; the others are whole groups of 4 segments behind them
  static constexpr int OFFSETS = 4 / STRIDE < NBLK ? 4 / STRIDE : NBLK;
  static_assert(4 % STRIDE == 0, "");
  uint32_t off[OFFSETS];   // lane offset per 32-wide block, its first half, 32-deep step 0

  // (16 lanes hand in the addresses of a block of 4 depth rows x 16 columns, lane i: depth row i / 4, columns
  // 4 (i % 4) .. +3, and lane j of them receives column j)
  __device__ __forceinline__ void setup(int first_col) {
    const int lane = threadIdx.x & 63;
    const int l16 = lane & 15;
    const int krow = 8 * (lane >> 4) + (l16 >> 2);   // (+ 4, + multiples of 32: neither changes swizzle or shift)
#pragma unroll
    for (int j = 0; j < OFFSETS; ++j) {
      const int seg = (first_col >> 5) + j * STRIDE;
      off[j] = (uint32_t)(Tile::row_at(krow) + ((seg ^ (krow & 3)) << 6) + 8 * (l16 & 3));
    }
  }
  __device__ __forceinline__ bf16x8 read(const char* tile, int ks, int blk) const {
    const char* p = tile + off[blk % OFFSETS] + (blk / OFFSETS) * 256 + 32 * (ks % 2) + (ks / 2) * Tile::row_at(32);
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        (__attribute__((address_space(3))) bf16x4*)GG_LDS_PTR(p));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        (__attribute__((address_space(3))) bf16x4*)GG_LDS_PTR(p + 4 * PITCH));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// One-byte elements, width-major tile of W bytes per depth row (128 depth rows a slice).  The
// fragment of a 32x32x64 instruction is, per lane, 32 consecutive depth values of one column
// (depth 32 (l / 32) .. +31 of the 64-deep step, column l % 32), carried as two 16-byte halves
// like the depth-major one: "step" 2 s + h is half h of 64-deep step s.  ds_read_b64_tr_b8 gives
// a lane 8 consecutive depth values of its column: 16 lanes hand in the addresses of an 8 x 16
// byte block (lane i: depth row i / 2, bytes 8 (i % 2) .. +7) and lane j of them receives column
// j.  Two such reads make a half.
template <int W, int NBLK, int STRIDE>
struct WidthMajorFrag8 {
  static constexpr int PITCH = W;
  uint32_t off[NBLK];   // lane offset per 32-wide block, 64-deep step 0, half 0, first read

  __device__ __forceinline__ void setup(int first_col) {
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, i = lane & 15;
    const int krow = 32 * (g >> 1) + (i >> 1);   // (+ multiples of 8: the swizzle sees i / 2 only)
#pragma unroll
    for (int j = 0; j < NBLK; ++j) {
      const int col = first_col + j * STRIDE * 32 + 16 * (g & 1) + 8 * (i & 1);
      off[j] = (uint32_t)(krow * PITCH + ((((col >> 5) ^ (krow & 7)) << 5) | (col & 31)));
    }
  }
  __device__ __forceinline__ bf16x8 read(const char* tile, int ks, int blk) const {
    using i32x2 = __attribute__((ext_vector_type(2))) int;
    using i32x4 = __attribute__((ext_vector_type(4))) int;
    const char* p = tile + off[blk] + (64 * (ks / 2) + 16 * (ks % 2)) * PITCH;
    const i32x2 lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) i32x2*)GG_LDS_PTR(p));
    const i32x2 hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
        (__attribute__((address_space(3))) i32x2*)GG_LDS_PTR(p + 8 * PITCH));
    return __builtin_bit_cast(bf16x8, i32x4{lo[0], lo[1], hi[0], hi[1]});
  }
};

// ------------------------------------------------------------------------ kernel

// Compile-time loop: f(integral_constant<int, 0>{}), ..., f(integral_constant<int, N-1>{}).
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  [&]<int... I>(std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
  }(std::make_integer_sequence<int, N>{});
}

// Where the LOADS global loads that begin in a depth slice of S matrix instructions go: spread evenly from FROM to TO, beyond S
// among the instructions of the slice after.
template <int LOADS, int FROM, int WAIT, int TO, int S>
struct LoadSlots {
  // loads sent ahead of instruction m
  static constexpr int before(int m) { return m <= FROM ? 0 : (m >= TO ? LOADS : LOADS * (m - FROM) / (TO - FROM)); }
  // one load goes behind instruction m, and there is an instruction ahead of that one with no wait or branch in between
  static constexpr bool alone(int m) { return m > FROM && m != WAIT && m != S && before(m + 1) == before(m) + 1; }
};

constexpr int kTileInfoDwords = 24;   // a tile's description on its way through LDS (pack_tile)

template <int LAYOUT, int BM, int BN, int BK, int STAGES, int WAVES_M, int WAVES_N>
struct GmmConfig {
  static constexpr int NT = WAVES_M * WAVES_N * 64;
  static constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
  static constexpr int MB = WTM / 32, NB = WTN / 32;
  static constexpr bool A_DEPTH_MAJOR = LAYOUT != kTN;
  static constexpr bool B_DEPTH_MAJOR = LAYOUT == kNT;
  // (fp8 tiles of the same bytes without the shifts: a little less than this)
  static constexpr int A_BYTES = A_DEPTH_MAJOR ? BM * BK * 2 : width_major_bytes(BM, BK, false);
  static constexpr int B_BYTES = B_DEPTH_MAJOR ? BN * BK * 2 : width_major_bytes(BN, BK, false);
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  // after the tile buffers: the schedule, then one strip per wave for the epilogue
  static constexpr int SCHED_OFFSET = STAGES * STAGE_BYTES;
  static constexpr int EPILOGUE_OFFSET = (SCHED_OFFSET + (int)sizeof(Sched) + 15) / 16 * 16;
  static constexpr int EPILOGUE_PITCH = 64 * 2 + 16;            // 64 bf16 columns + padding
  static constexpr int EPILOGUE_WAVE_BYTES = 32 * EPILOGUE_PITCH;
  static_assert(NB % 2 == 0, "the epilogue's strips are 64 columns wide");
  // last: per wave, the descriptions of the tiles between the fetch and the compute cursor
  static constexpr int TILE_RING_SLOTS = 4;
  static constexpr int TILE_RING_OFFSET =
      (EPILOGUE_OFFSET + WAVES_M * WAVES_N * EPILOGUE_WAVE_BYTES + 15) / 16 * 16;
  static constexpr int LDS_BYTES = TILE_RING_OFFSET + WAVES_M * WAVES_N * TILE_RING_SLOTS * kTileInfoDwords * 4;
  static_assert(LDS_BYTES <= 160 * 1024, "a compute unit has 160 KiB of LDS");
  static constexpr int WORKGROUPS_PER_CU = 2 * LDS_BYTES <= 160 * 1024 ? 2 : 1;
  static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile is made of 32x32 MFMA blocks");
  static_assert(BK % 16 == 0 && STAGES >= 2, "");
};

// One output tile (or one piece of a tile of the last round) as the scheduler hands it out.
struct TileInfo {
  GroupGeom g;
  int m0, n0;       // first row and column of the tile inside its group's output
  int rows_valid;   // rows of the tile that exist (0: no tile)
  int blocks;       // 32-row blocks the tile's rows take (MFMAs are issued for these only)
  int depth;        // depth to fetch (0: nothing to fetch, the tile multiplies zeros)
  int k0;           // first depth slice (not 0 only for a depth piece)
  int nk;           // depth slices, at least 1 so that an empty group still stores zeros
  int pieces;       // depth pieces this tile is cut into (1: whole depth, store directly)
  int piece;        // which of them this is
  int rank;         // index of the tile among the tiles that are cut
  int slot, slots_apart;   // where its pieces' partial tiles are in the workspace
  bool valid;
};

// Where a tile cursor stands: group and class.  Tile indices only grow, so inside a class the
// group only moves forward; it starts over once, when the indices pass into the runt class.
struct TileCursor {
  int e = 0;
  int cls = 0;
};

// A tile's description as 24 dwords, for the trip through LDS from the fetch cursor, which works
// it out, to the compute cursor, which needs the same one or two tiles later.
__device__ __forceinline__ void pack_tile(const TileInfo& t, int32_t* w) {
  w[0] = (int32_t)t.g.a_off, w[1] = (int32_t)(t.g.a_off >> 32);
  w[2] = (int32_t)t.g.b_off, w[3] = (int32_t)(t.g.b_off >> 32);
  w[4] = (int32_t)t.g.c_off, w[5] = (int32_t)(t.g.c_off >> 32);
  w[6] = t.g.m, w[7] = t.g.n, w[8] = t.g.k, w[9] = t.g.row0;
  w[10] = t.m0, w[11] = t.n0, w[12] = t.rows_valid, w[13] = t.blocks, w[14] = t.depth, w[15] = t.k0;
  w[16] = t.nk, w[17] = t.pieces, w[18] = t.piece, w[19] = t.rank, w[20] = t.valid ? 1 : 0;
  w[21] = t.slot, w[22] = t.slots_apart, w[23] = 0;
}
__device__ __forceinline__ TileInfo unpack_tile(const int32_t* w) {
  auto u = [&](int i) { return uniform(w[i]); };
  auto u64 = [&](int i) { return (int64_t)(((uint64_t)(uint32_t)u(i + 1) << 32) | (uint32_t)u(i)); };
  TileInfo t;
  t.g.a_off = u64(0), t.g.b_off = u64(2), t.g.c_off = u64(4);
  t.g.m = u(6), t.g.n = u(7), t.g.k = u(8), t.g.row0 = u(9);
  t.m0 = u(10), t.n0 = u(11), t.rows_valid = u(12), t.blocks = u(13), t.depth = u(14), t.k0 = u(15);
  t.nk = u(16), t.pieces = u(17), t.piece = u(18), t.rank = u(19), t.valid = u(20) != 0, t.slot = u(21), t.slots_apart = u(22);
  return t;
}

// Smallest position e >= from with t < start[e + 1], for an exclusive prefix sum `start` of n
// positions with t < start[n] (so start[e] <= t: positions without tiles are passed over).  A
// gallop, then a bisection: two probes when the answer is the next position, the common case of a
// cursor that moves on, and about 2 log2 of the distance for a workgroup's first tile, where a
// walk position by position, one LDS round trip each, took 15 to 30 us of a launch with 256 to 512
// groups.
__device__ __forceinline__ int advance_to(const int32_t* start, int n, int from, int t) {
  if (t < uniform(start[from + 1])) return from;
  int lo = from + 1, step = 1;   // t >= start[lo]
  while (lo + step < n && t >= uniform(start[lo + step])) {
    lo += step;
    step <<= 1;
  }
  int hi = lo + step < n ? lo + step : n;   // t < start[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (t >= uniform(start[mid])) {
      lo = mid;
    } else {
      hi = mid;
    }
  }
  return lo;
}

// Tile index -> group and position.  Indices past plan.main_tiles name pieces of the last
// round's tiles: piece (t - main) % pieces of tile main + (t - main) / pieces.
template <int LAYOUT, int BM, int BN, int BK>
__device__ __forceinline__ TileInfo find_tile(const Sched* sched, const GmmParams& p, int t,
                                              const TailPlan& plan, TileCursor& cur) {
  TileInfo ti;
  ti.k0 = 0;
  ti.pieces = 1;
  ti.piece = 0;
  ti.rank = 0;
  ti.slot = 0;
  ti.slots_apart = 1;
  if (t >= plan.total) {
    ti.g = GroupGeom{0, 0, 0, 0, 0, 0, 0};
    ti.m0 = ti.n0 = ti.rows_valid = ti.depth = 0;
    ti.blocks = 1;
    ti.nk = 1;
    ti.valid = false;
    return ti;
  }
  int piece = -1;
  int pieces = plan.pieces;
  const int front_tiles = LAYOUT == kTN ? uniform(sched->front_tiles) : 0;
  if (front_tiles > 0) {
    const int front_pieces = uniform(sched->front_pieces);
    const int cut = front_tiles * front_pieces;
    if (front_pieces == 0) {   // (plan_pieces_by_length)
      const int per_group = uniform(sched->group_tiles), groups = uniform(sched->cut_groups);
      if (t < front_tiles) {
        // (positions whose pieces end at t or before; no loop here, see tile_body)
        int q = 0;
#pragma unroll
        for (int i = 0; i < kMaxGroups; i += 64)
          if (i < groups) {
            const int lane = threadIdx.x & 63, at = i + lane;
            q += __popcll(__ballot(at < groups && sched->tile_start[at + 1] <= t));
          }
        q = uniform(q);
        const PieceAt at = piece_at(t, uniform(sched->tile_start[q]), per_group);
        pieces = uniform(sched->runt_start[q]);
        piece = at.piece;
        ti.slot = at.slot;
        ti.slots_apart = per_group;
        t = q * per_group + at.tile;
        ti.rank = t;
      } else {
        t = t - front_tiles + groups * per_group;
      }
    } else if (t < cut) {
      pieces = front_pieces;
      piece = t % pieces;
      ti.rank = t / pieces;
      ti.slot = t - piece;
      t = ti.rank;
    } else {
      t = t - cut + front_tiles;
    }
  } else if (t >= plan.main_tiles) {
    const int r = t - plan.main_tiles;
    piece = r % plan.pieces;
    ti.rank = r / plan.pieces;
    ti.slot = r - piece;
    t = plan.main_tiles + ti.rank;
  }
  const int first_class = uniform(sched->tile_start[p.num_groups]);
  int u;
  if (LAYOUT == kTN) {
    // (every group has the same number of tiles, and there are no runt rows)
    const int per_group = uniform(sched->group_tiles);
    cur.e = t / per_group;
    u = t - cur.e * per_group;
  } else if (t < first_class) {
    cur.e = advance_to(sched->tile_start, p.num_groups, cur.e, t);
    u = t - uniform(sched->tile_start[cur.e]);
  } else {
    if (cur.cls == 0) {
      cur.cls = 1;
      cur.e = 0;
    }
    t -= first_class;
    cur.e = advance_to(sched->runt_start, p.num_groups, cur.e, t);
    u = t - uniform(sched->runt_start[cur.e]);
  }
  // (the cursor walks positions of the order the groups are handed out in.  Weight-gradient layout:
  // all groups have the same number of tiles, so the tile prefix sums serve positions as they are;
  // by tile rows: the prefix sums were counted in that order)
  const bool ordered = LAYOUT == kTN || (p.flags & kFlagByTileRows) != 0;
  const int e = ordered ? uniform((int)sched->order[cur.e]) : cur.e;
  // read through the first lane: everything derived from these stays in scalar registers
  const int rows = uniform(sched->rows[e]);
  ti.g = group_geometry<LAYOUT>(p, p.first_group + e, uniform(sched->row_start[e]), rows);
  GroupTiles gt = group_tiles<LAYOUT, BM, BN>(rows, p.hidden_in, p.hidden_out, p.flags);
  gt.height = uniform(gt.height);
  gt.main_rows = uniform(gt.main_rows);
  int tm, tn;
  if (cur.cls == 0) {
    tile_coords(u, gt.main_rows, gt.tiles_n, p.group_m, &tm, &tn);
  } else {
    tm = gt.tiles_m - 1;
    tn = u;
  }
  ti.m0 = uniform(tm) * gt.height;
  ti.n0 = uniform(tn) * BN;
  ti.rows_valid = min(gt.height, ti.g.m - ti.m0);
  ti.depth = ti.g.k;
  const int nk = (ti.g.k + BK - 1) / BK;
  ti.nk = nk < 1 ? 1 : nk;
  if (piece >= 0 && plan.by_depth) {
    // this piece's share of the depth slices; a piece without slices contributes zeros
    const int first = piece * ti.nk / pieces, last = (piece + 1) * ti.nk / pieces;
    ti.pieces = pieces;
    ti.piece = piece;
    ti.k0 = first;
    ti.nk = last - first;
    if (ti.nk <= 0) {
      ti.k0 = 0;
      ti.nk = 1;
      ti.depth = 0;
    }
  } else if (piece >= 0) {
    // this piece's share of the tile's 32-row blocks; a piece past the rows is an empty tile
    const int all = (ti.rows_valid + 31) / 32;
    const int per = (all + pieces - 1) / pieces;
    const int skip = piece * per * 32;
    ti.m0 += skip;
    ti.rows_valid = min(per * 32, ti.rows_valid - skip);
    if (ti.rows_valid <= 0) {
      ti.rows_valid = 0;
      ti.depth = 0;
      ti.nk = 1;
    }
  }
  ti.blocks = LAYOUT == kTN ? BM / 32 : max(1, (ti.rows_valid + 31) / 32);
  ti.valid = true;
  return ti;
}

// What a launch does beside this product (the PART of gmm_tiles).
template <int WGS_PER_CU_>
struct Alone {   // nothing
  static constexpr int WGS_PER_CU = WGS_PER_CU_;   // workgroups a compute unit has room for
  static constexpr bool FIRST = false, SECOND = false;
};
template <int WGS_PER_CU_>
struct FirstOfPair {   // its workgroups are followed by those of a second product (gmm_pair_kernel)
  static constexpr int WGS_PER_CU = WGS_PER_CU_;
  static constexpr bool FIRST = true, SECOND = false;
};
// ... and this is the second one: a weight gradient whose workgroups start where the first product's have ended.
// The first one's last round leaves `early` workgroups per XCD without a tile; as many of the second's, the
// first of each XCD (an XCD starts its workgroups in order as its compute units become free), begin a tile of the
// first earlier than the rest, and are given `extra` more tiles: as many as end both soonest.
// Costs of a tile in depth slices of full tiles: the slices left to a piece and 3 of tile turnover for the first
// product, 4 of stores for the second one; short tiles' slices are five eighths as long.
// 8 x 1024 rows, 5464 -> 2048 and the weight gradient: 461 us in two launches, 409 in one without extra tiles, 376.
struct Head {
  int early, extra;
};
// None where tiles of the second are shallow: they are bound by their stores, and slow the first down (32 x 128 rows,
// 2048 -> 768: 62 us without, 65 to 72 with 1 to 4 extra tiles).
constexpr int kHeadSlices = 8;
constexpr int kMaxExtra = 12;
template <int WGS_PER_CU_, int LAYOUT1, int BM1, int BN1>
struct SecondOfPair {
  static constexpr int WGS_PER_CU = WGS_PER_CU_;
  static constexpr bool FIRST = false, SECOND = true;
  const GmmParams& first;

  // (after build_schedule and a barrier; the same answer in every wave)
  __device__ __forceinline__ Head head(const Sched* s, const GmmParams& p, int grid, int bk) const {
    int tile_rows = 0;
    for (int e = threadIdx.x & 63; e < p.num_groups; e += 64) tile_rows += (s->rows[e] + BM1 - 1) / BM1;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) tile_rows += __shfl_xor(tile_rows, d);
    const TailPlan plan = plan_tail<LAYOUT1, BM1, BN1, WGS_PER_CU>(uniform(tile_rows) * ((first.hidden_out + BN1 - 1) / BN1),
                                                                    grid, first, bk);
    Head h{0, 0};
    if (grid % 8 != 0) return h;
    h.early = grid / 8 - (plan.total % grid + 7) / 8;
    const int slices2 = ((int)(p.tokens / p.num_groups) + bk - 1) / bk;
    if (h.early == 0 || slices2 < kHeadSlices) return h;
    const int slices1 = (first.hidden_in + bk - 1) / bk / (plan.by_depth ? plan.pieces : 1);
    const int cost1 = (BM1 > 128 ? slices1 : slices1 * 5 / 8) + 3, cost2 = slices2 + 4;
    const int tiles = uniform(s->tile_start[p.num_groups]), n = h.early * 8;
    int best = 1 << 30;
    for (int extra = 0; extra <= kMaxExtra && extra * n <= tiles; ++extra) {
      const int rounds = (tiles - extra * n) / grid, rest = (tiles - extra * n) % grid;   // (of the last round, the early ones first)
      const int late = (rounds + (rest > n ? 1 : 0)) * cost2;
      const int soon = (extra + rounds + (rest > 0 ? 1 : 0)) * cost2 - cost1;
      const int end = late > soon ? late : soon;
      if (end < best) best = end, h.extra = extra;
    }
    return h;
  }
};

// The tiles of one product that workgroup w of G works on.
// DT: element type of a and b (and of c unless it is the fp32 accumulator).
// EPI: what happens to a finished tile (kEpi*): stored in the element type; added to an fp32 c
// (gradient accumulation, weight-gradient layout); or, with gate | up columns in b, combined to
// silu(gate) * up and stored half as wide.
// INDEXED: rows of a are fetched and rows of c stored through p.a_rows / p.c_rows (NN and NT).
// RAGGED_DEPTH: hidden_in is even but no multiple of 8 (NN and NT, two-byte elements, plain store).
template <int DT, int LAYOUT, int BM, int BN, int BK, int STAGES, int WAVES_M, int WAVES_N,
          int EPI, bool INDEXED, bool RAGGED_DEPTH, typename PART>
__device__ __forceinline__ void gmm_tiles(const GmmParams& given, const HostSizes& hs, char* smem, const int w, const int G, const PART& part) {
  GmmParams p = given;
  // Words that the kernel arguments are read in together, told apart: the first of these pairs otherwise spills eight of them as one and
  // reads all eight back wherever it wants one (1950 reads of spilled words, with this 710 to 1560, by what else the
  // kernel holds); in the other pairs they are spilled one by one as it is.
  if constexpr (PART::FIRST && LAYOUT == kNT && BM == 256) {
    if constexpr (DT == kBF16) {
      asm volatile("" : "+s"(p.hidden_in), "+s"(p.hidden_out), "+s"(p.ws_slots), "+s"(p.flags), "+s"(p.lda), "+s"(p.ldb));
    } else {
      asm volatile("" : "+s"(p.hidden_in), "+s"(p.hidden_out), "+s"(p.ws_slots), "+s"(p.flags));
    }
  }
  using Cfg = GmmConfig<LAYOUT, BM, BN, BK, STAGES, WAVES_M, WAVES_N>;
  constexpr int NT = Cfg::NT, MB = Cfg::MB, NB = Cfg::NB, KS = BK / 16;
  constexpr bool ACC_F32 = EPI == kEpiAccF32 || EPI == kEpiAccF32Atomic, KEEP = EPI == kEpiSwiGLUKeep, GATE_UP = EPI == kEpiSwiGLU || KEEP;
  // One-byte elements (NT layout only: both operands depth-contiguous).  The tile movers see them
  // as two-byte elements, two to one: same bytes per row and slice, BK_ELEMS depth values a slice.
  constexpr bool F8 = is_f8(DT);
  constexpr int ES = F8 ? 1 : 2, BK_ELEMS = BK * 2 / ES, OUT_DT = DT == kF16 ? kF16 : kBF16;
  static_assert(!F8 || !GATE_UP || LAYOUT == kNT, "fp8 with gate | up rows streams in the NT layout only");
  static_assert(!ACC_F32 || LAYOUT == kTN, "the fp32 accumulator is the weight gradient's");
  static_assert(!(GATE_UP || INDEXED) || LAYOUT != kTN, "row indices and gate | up are for the NN and NT layouts");
  static_assert(!KEEP || (!F8 && !INDEXED), "gate | up are kept for two-byte elements and rows in place");
  static_assert(!GATE_UP || NB % 2 == 0, "a wave needs the gate and the up block of its columns");
  constexpr int BNS = GATE_UP ? BN / 2 : BN;   // output columns per tile, what the schedule counts in
  // fp32 accumulation by reading, adding and writing in full tiles, whose epilogue holds a block row of c (16 values of 16 bytes).  With
  // every load's offset held beside it 19 registers spill, and each block row begins with a reload that waits for the stores of
  // the one before.  us with / without: 234 groups, 12160 rows, 1152 x 296: 201 / 186; 49, 7883 rows, 1920 x 8920: 1639 / 1614; 22,
  // 18760 rows, 960 x 1496: 105 / 101.
  constexpr bool ONE_OFFSET = EPI == kEpiAccF32 && BM == 256;
  // (width-major tiles of one-byte elements: half as many two-byte elements per depth row, twice
  // the depth rows)
  using ALoad = std::conditional_t<Cfg::A_DEPTH_MAJOR, DepthMajor<BM, BK, NT, INDEXED>,
                                   WidthMajor<BM * ES / 2, BK_ELEMS, NT, F8, ONE_OFFSET>>;
  using BLoad = std::conditional_t<Cfg::B_DEPTH_MAJOR, DepthMajor<BN, BK, NT, false, GATE_UP>,
                                   WidthMajor<BN * ES / 2, BK_ELEMS, NT, F8, ONE_OFFSET>>;
  using AFrag = std::conditional_t<Cfg::A_DEPTH_MAJOR, DepthMajorFrag<BK, WAVES_M, F8>,
                                   std::conditional_t<F8, WidthMajorFrag8<BM, MB, WAVES_M>, WidthMajorFrag<BM, BK, MB, WAVES_M>>>;
  using BFrag = std::conditional_t<Cfg::B_DEPTH_MAJOR, DepthMajorFrag<BK, 1, F8>,
                                   std::conditional_t<F8, WidthMajorFrag8<BN, NB, 1>, WidthMajorFrag<BN, BK, NB, 1>>>;
  constexpr int LOADS_PER_STAGE = ALoad::NI + BLoad::NI;   // per lane, per depth slice
  static_assert(KS == 4 && STAGES == 2, "the schedule of a slice (tile_body) is written for BK = 64 and two buffers");
  static_assert(LOADS_PER_STAGE >= 4 && LOADS_PER_STAGE < 32, "");
  // The positions of a slice's schedule (see tile_body) in 32nds of its matrix instructions.  A buffer is handed over as
  // early as LDS can deliver its fragments: what a fetch has time for counts for more than an even load on LDS
  // (released at 8, 10, 13 and 14, ready at 24, 22, 19 and 18, us: 8 x 4096 rows, 4096 -> 14336, NN 2913 / 2943 / 2986 / 2978;
  // 256 x 256, 7168 -> 2048, NT 2079 / 2030 / 2100 / 2160).  Tiles of few rows, whose launches are bound by latency: earlier still
  // (6 and 26 against 8 and 24: 16 x 256 rows, 3072 -> 768: 32.8 / 34.1, NT 33.8 / 35.7; 32 x 128, 2048 -> 768: 28.5 / 28.4;
  // against 10 and 22: 36.2, 37.7, 31.9).  Not short tiles of the NN layout, which mostly stream weights: 128 groups x 30 rows, 4096 ->
  // 2048: 358 / 351, 16 rows: 353 / 345; 64 x 50, 7168 -> 2048: 314 / 308; 8 x 40, 4096 -> 14336: 170 / 168; but as the first of a pair,
  // which is bound by latency again (16 x 200, 1024 -> 3072 transposed, forward and both gradients: 104 / 106).
  constexpr bool EARLY = LAYOUT != kTN && BM < 256 && !F8 && !(LAYOUT == kNN && BM == 128 && !PART::FIRST);
  constexpr int AT_READ_END = EARLY ? 6 : 8, AT_RELEASE = AT_READ_END, AT_READY = EARLY ? 26 : 24;
  // Loads that reach into the next slice are steadier: ended at 32, 36 and 40, us: 8 x 4096 rows, 4096 -> 14336, NN 2743 / 2749 /
  // 2779, input gradient 2685 / 2665 / 2675, 256 x 256 NT 1917 / 1897 / 1947, NN 1987 / 1921 / 1930.  Not where
  // tiles are shallow or their launch is bound by memory (weight gradients, tiles of few rows): with loads behind the
  // stores of a tile the first wait of the next one waits for the memory to take the whole tile, without it lets the
  // stores pass (counters go down in the order of issue): 256 groups x 256 rows, 2048 x 7168: 2555 -> 2502 us.  fp8, ended at 32 and
  // 36: 8 Zipf (1.2) groups, 22637 rows, 4720 -> 352, one tile to a workgroup: 54.1 / 51.4; 8 x 4096 rows, 4096 -> 14336, NT 1394 / 1399,
  // 8 x 2048, 4096 -> 3072 NN 174 / 174, 16 x 1024, 2048 -> 2048 NT 68.7 / 68.6.
  constexpr bool LATE_LOADS = LAYOUT != kTN && BM == 256;
  constexpr int AT_LOAD_END = LATE_LOADS ? 36 : 32;
  constexpr int FIRST_LOADS = LoadSlots<LOADS_PER_STAGE, AT_RELEASE, AT_READY, AT_LOAD_END, 32>::before(32);   // ... by a slice's end
  constexpr int UNITS = MB + NB;    // fragments of one set

  Sched* sched = reinterpret_cast<Sched*>(smem + Cfg::SCHED_OFFSET);
  build_schedule<LAYOUT, BM, BNS>(sched, p, hs, w);
  __syncthreads();
  if constexpr (LAYOUT == kTN) {
    order_groups_by_depth(sched, p.num_groups, reinterpret_cast<uint64_t*>(smem));
  } else {
    if (p.flags & kFlagByTileRows) order_groups_by_tile_rows<LAYOUT, BM, BNS>(sched, p);
  }

  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;

  AFrag afrag;
  BFrag bfrag;
  afrag.setup(wm * 32);   // wave row wm owns row blocks wm, wm + WAVES_M, ...
  bfrag.setup(wn * Cfg::WTN);

  // (tiles that are combined or scattered on their way out are cut along the depth in the shapes for
  // few rows and few tiles only: full ones would pay for it with the fix-up's scalar registers)
  constexpr bool DEPTH_PIECES = !((GATE_UP || INDEXED) && BM > 128);
  const int all_tiles = uniform(sched->tile_start[p.num_groups]) + uniform(sched->runt_start[p.num_groups]);
  // SECOND: indices below head_tiles go to the workgroups that start early, the others to all of them
  Head head{0, 0};
  if constexpr (PART::SECOND) head = part.head(sched, p, G, BK_ELEMS);
  int head_step = uniform(head.early) * 8, head_tiles = head_step * uniform(head.extra);
  TailPlan plan = plan_tail<LAYOUT, BM, BN, PART::WGS_PER_CU, DEPTH_PIECES>(all_tiles - head_tiles, G, p, BK_ELEMS);
  if constexpr (PART::SECOND) plan.main_tiles += head_tiles, plan.total += head_tiles;
  if constexpr (!DEPTH_PIECES) plan.by_depth = false;   // (known at compile time: no depth-piece code is kept)
  if constexpr (LAYOUT == kTN && DEPTH_PIECES) {
    if (p.flags & kFlagPiecesByLength) {
      plan_pieces_by_length<BM, BN, PART::WGS_PER_CU>(sched, p, G, BK_ELEMS, reinterpret_cast<uint32_t*>(smem), &plan);
    } else {
      plan_deep_tiles<BM, BN>(sched, p, G, BK_ELEMS, &plan);
    }
    plan.pieces = uniform(plan.pieces), plan.main_tiles = uniform(plan.main_tiles), plan.total = uniform(plan.total);
    // (cut deep tiles go out first, at most one piece to a workgroup)
    if (PART::SECOND && uniform(sched->front_tiles) > 0) head_tiles = 0;
  }
  const int total_tiles = plan.total;

  // Workgroups are dealt to the 8 XCDs round-robin; give each XCD a contiguous run of tile indices
  // so that its private L2 sees neighbouring tiles.  A launch with fewer tiles than workgroups
  // deals them evenly to all XCDs: runs of G / 8 would put them on the first few, each of which
  // reaches only its share of the memory bandwidth (6 tiles of 128 depth slices, all on one XCD:
  // 51 us, one to an XCD: 36 us; 30 tiles of 100 slices: 141 -> 83 us; 200 tiles and more, and tiles
  // of a few slices, within 2 % either way).  In a pair the last round is dealt evenly as well, so that the
  // workgroups without a tile in it are spread over the XCDs (alone that is neutral, 0.98 to 1.01 of the time).
  int first_t = w;
  const int full = head_tiles + (total_tiles - head_tiles) / G * G;   // (pairs) where the last round begins
  int last_t = full + w;                                              // (pairs) this workgroup's index in it
  if (G % 8 == 0) {
    const int x = w % 8, s = w / 8;
    if constexpr (PART::FIRST || PART::SECOND) {
      const int run = (total_tiles - full + 7) / 8;
      last_t = s < run ? full + x * run + s : total_tiles;
      first_t = head_tiles + x * (G / 8) + s;
      if (first_t >= full) first_t = last_t;
      if (PART::SECOND && head_tiles > 0 && s < head_step / 8) first_t = x * (head_step / 8) + s;
    } else {
      const int run = total_tiles < G ? (total_tiles + 7) / 8 : G / 8;
      first_t = s < run ? x * run + s : total_tiles;
    }
  }
  if (first_t >= total_tiles) return;
  first_t = uniform(first_t);
  // The index of this workgroup's tile after tile t (total_tiles and more: none)
  auto next_index = [&](int t) {
    if constexpr (!PART::FIRST && !PART::SECOND) return uniform(t + G);
    if (PART::SECOND && t < head_tiles) {
      const int mine = head_tiles + (G % 8 == 0 ? (w % 8) * (G / 8) + w / 8 : w);
      return uniform(t + head_step < head_tiles ? t + head_step : (mine < full ? mine : last_t));
    }
    return uniform(t + G < full ? t + G : (t < full ? last_t : total_tiles));
  };

  // Two cursors walk this workgroup's tiles: the fetch cursor runs STAGES depth slices
  // ahead of the compute cursor and crosses into the next tile on its own, so the first
  // slices of a tile are already in flight while the previous tile is being stored.
  ALoad aload;
  BLoad bload;
  int fetch_t = first_t, fetch_kt = 0;
  TileCursor fetch_cur;
  TileInfo fti;
  // The compute cursor does not look its tiles up again: the fetch cursor, which is one or two
  // tiles ahead, leaves each description in a ring in LDS (one ring per wave, written by its first
  // lane and read back by the same wave: no barrier involved).
  int32_t* tile_ring = reinterpret_cast<int32_t*>(smem + Cfg::TILE_RING_OFFSET) +
                       wave * (Cfg::TILE_RING_SLOTS * kTileInfoDwords);
  int fetch_n = 0;   // tiles the fetch cursor has set up
  auto fetch_setup = [&]() {
    fti = find_tile<LAYOUT, BM, BNS, BK_ELEMS>(sched, p, fetch_t, plan, fetch_cur);
    {
      int32_t words[kTileInfoDwords];
      pack_tile(fti, words);
      int32_t* slot = tile_ring + (fetch_n % Cfg::TILE_RING_SLOTS) * kTileInfoDwords;
      if (lane == 0) {
#pragma unroll
        for (int i = 0; i < kTileInfoDwords; i += 4)
          *reinterpret_cast<u32x4*>(slot + i) = u32x4{(uint32_t)words[i], (uint32_t)words[i + 1],
                                                      (uint32_t)words[i + 2], (uint32_t)words[i + 3]};
      }
      fetch_n = uniform(fetch_n + 1);
    }
    const int depth = fti.depth;
    // (an odd depth has a zero behind it: buffers end after whole dwords)
    const int along = ES == 2 ? depth + (depth & 1) : depth / 2;   // depth of rows along it, in two-byte elements
    if constexpr (INDEXED) {
      const int first = fti.g.row0 + fti.m0;
      aload.setup_gather(p.a, p.a_bytes, p.a_rows != nullptr ? p.a_rows + first : nullptr, p.a_index_rows, first,
                         fti.g.k * ES / 2, depth > 0 ? fti.rows_valid : 0, depth * ES / 2);
    } else if constexpr (Cfg::A_DEPTH_MAJOR) {
      aload.setup(p.a + (fti.g.a_off + (int64_t)fti.m0 * p.lda) * ES, p.lda * ES / 2, fti.rows_valid, along);
    } else {
      aload.setup(p.a + fti.g.a_off * ES, p.lda * ES / 2, depth, fti.m0 * ES / 2, fti.g.m * ES / 2);
    }
    if constexpr (GATE_UP && Cfg::B_DEPTH_MAJOR) {
      bload.setup_gate_up(p.b + (fti.g.b_off + (int64_t)fti.n0 * fti.g.k) * ES, fti.g.k * ES / 2,
                          fti.valid && depth > 0 ? 2 * fti.g.n - fti.n0 : 0, depth * ES / 2, fti.g.n);
    } else if constexpr (GATE_UP) {
      bload.setup_gate_up(p.b + fti.g.b_off * 2, 2 * fti.g.n, depth, fti.n0, fti.g.n);
    } else if constexpr (Cfg::B_DEPTH_MAJOR) {
      bload.setup(p.b + (fti.g.b_off + (int64_t)fti.n0 * p.ldb) * ES, p.ldb * ES / 2,
                  fti.valid && depth > 0 ? min(BN, fti.g.n - fti.n0) : 0, along);
    } else {
      // (rows of b are as long as they are apart where row indices are used: a scalar register less)
      bload.setup(p.b + fti.g.b_off * ES, (INDEXED ? fti.g.n : p.ldb) * ES / 2, depth, fti.n0 * ES / 2, fti.g.n * ES / 2);
    }
    if (fti.k0 != 0) {
      aload.skip(fti.k0);
      bload.skip(fti.k0);
    }
  };
  // Slices past the depth (or past the last tile) are fetched with an empty descriptor:
  // zeros, no traffic, and the number of loads in flight is the same at every step.
  typename ALoad::Slice a_slice;
  typename BLoad::Slice b_slice;
  // Load J of the cursor's slice (A's loads first, then B's) into buffer `buf`: fetch_aim, then fetch_load.  A's descriptor
  // comes with fetch_begin (then a wait, a barrier, a matrix instruction, fetch_aim and another instruction precede the first
  // load), B's ahead of A's last load (then that load and two of each precede B's first).
  bool tail_fetched = false;   // RAGGED_DEPTH: the cursor's slice holds the end of the depth
  auto fetch_begin = [&]() {
    if constexpr (RAGGED_DEPTH) tail_fetched = uniform(aload.depth) > 0 && uniform(aload.depth) < BK;
    a_slice = aload.slice();
    settle(a_slice.rsrc);
  };
  const uint32_t a_first = uniform(lds_address(smem) + ALoad::wave_at(wave)), b_first = uniform(lds_address(smem) + BLoad::wave_at(wave));
  auto fetch_aim = [&](auto j_tag, int buf) {
    constexpr int J = decltype(j_tag)::value;
    const uint32_t at = uniform(buf) * Cfg::STAGE_BYTES;
    if constexpr (J == ALoad::NI - 1) {
      b_slice = bload.slice();
      settle(b_slice.rsrc);
    }
    if constexpr (J < ALoad::NI) {
      aim_lds<ALoad::template kOffset<J>>(uniform(a_first + at));
    } else {
      aim_lds<Cfg::A_BYTES + BLoad::template kOffset<J - ALoad::NI>>(uniform(b_first + at));
    }
  };
  auto fetch_load = [&](auto j_tag, auto right_behind) {
    constexpr int J = decltype(j_tag)::value;
    if constexpr (J < ALoad::NI) {
      aload.template load<J, decltype(right_behind)::value>(a_slice);
    } else {
      bload.template load<J - ALoad::NI, decltype(right_behind)::value>(b_slice);
    }
  };
  auto fetch_whole = [&](auto j_tag, int buf) {
    fetch_aim(j_tag, buf);
    fetch_load(j_tag, std::true_type{});
  };
  auto fetch_advance = [&]() {
    // (said to be the same in every lane once more: where the compiler loses track of that, the
    // slice descriptors below are computed lane by lane and the branch becomes a masked one)
    fetch_kt = uniform(fetch_kt + 1);
    // (once a tile: kept out of the loop's instructions, which a jump over it would fetch anew every slice)
    if (__builtin_expect(fetch_kt == uniform(fti.nk) && uniform((int)fti.valid) != 0, 0)) {
      fetch_t = next_index(fetch_t);
      fetch_kt = 0;
      fetch_setup();
    }
  };

  // Fragments: sets 0 and 1 are the halves of the first 32-deep (fp8: 64-deep) step of a slice, 2 and 3 those of the
  // second.  A "unit" is one fragment (one ds_read_b128, or two transposing 64-bit reads).  Unit U of the pair of
  // sets that begins with set SET, in the order in which the matrix instructions want them: B's first block, the
  // first ML of A's, the rest of B's NB, both halves of each.
  bf16x8 fa[KS][MB], fb[KS][NB];
  auto read_unit = [&](auto u_tag, auto set_tag, auto ml_tag, int buf) {
    constexpr int U = decltype(u_tag)::value / 2, SET = decltype(set_tag)::value + decltype(u_tag)::value % 2;
    constexpr int ML = decltype(ml_tag)::value;
    const char* sa = smem + buf * Cfg::STAGE_BYTES;
    if constexpr (U >= 1 && U <= ML) {
      fa[SET][U - 1] = afrag.read(sa, SET, U - 1);
    } else {
      constexpr int J = U == 0 ? 0 : U - ML;
      fb[SET][J] = bfrag.read(sa + Cfg::A_BYTES, SET, J);
    }
  };

  using I0 = std::integral_constant<int, 0>;
  using I2 = std::integral_constant<int, 2>;
  using IMB = std::integral_constant<int, MB>;

  // Both buffers are requested up front, except what the first slice's instructions send.
  fetch_setup();
  fetch_begin();
  asm volatile("s_nop 4");
  static_for<LOADS_PER_STAGE>([&](auto j) { fetch_whole(j, 0); });
  const bool tail_first = tail_fetched;
  fetch_advance();
  fetch_begin();
  bool tail_next = tail_fetched;   // ... the slice after the one that is multiplied does
  asm volatile("s_nop 4");
  static_for<FIRST_LOADS>([&](auto j) { fetch_whole(j, 1); });

  int tile_t = first_t;
  int tile_n = 0;   // tiles this workgroup has finished
  auto next_tile = [&]() {
    int32_t words[kTileInfoDwords];
    const int32_t* slot = tile_ring + (tile_n % Cfg::TILE_RING_SLOTS) * kTileInfoDwords;
#pragma unroll
    for (int i = 0; i < kTileInfoDwords; i += 4) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(slot + i);
      words[i] = (int32_t)v[0], words[i + 1] = (int32_t)v[1], words[i + 2] = (int32_t)v[2], words[i + 3] = (int32_t)v[3];
    }
    return unpack_tile(words);
  };
  TileInfo ti = next_tile();
  // RAGGED_DEPTH: hidden_in is even but no multiple of 8.  The ragged chunks are in the slice that ends the depth, which
  // the fetch cursor knows by what is left of it (a depth piece may begin anywhere and has that slice only if it is
  // its tile's last).  Once a buffer holds that slice, complete for every wave, what its ragged chunks picked up from
  // the rows behind is cleared before any wave reads a fragment from it.
  // Whole tiles / pieces, us: 28 Zipf (1.2) groups, 5434 rows, 13374 -> 272, fp16, b transposed: 314 / 201, not: 223 / 182;
  // 16 groups, 8192 rows, 9998 -> 2048: 542 / 466.
  static_assert(!RAGGED_DEPTH || (LAYOUT != kTN && !F8 && !GATE_UP && !INDEXED), "");
  auto clear_tail = [&](int buf) {
    if constexpr (RAGGED_DEPTH) {
      char* st = smem + uniform(buf) * Cfg::STAGE_BYTES;
      const int tail = p.hidden_in % BK;
      if constexpr (Cfg::A_DEPTH_MAJOR) ALoad::clear_depth_tail(st, tail);
      if constexpr (Cfg::B_DEPTH_MAJOR) BLoad::clear_depth_tail(st + Cfg::A_BYTES, tail);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      block_barrier();
    }
  };
  wait_vmcnt<FIRST_LOADS>();   // the first slice is in
  block_barrier();
  if (RAGGED_DEPTH && tail_first) clear_tail(0);
  static_for<2 * UNITS>([&](auto u) {
    read_unit(u, I0{}, IMB{}, 0);
  });

  int x = 0;   // buffer of the slice being multiplied

  // What a lane holds of a 32 x 32 block of the result: four groups q of 4 consecutive columns of a row.
  auto group_row_of = [&](int at_lane, int q) { return F8 ? at_lane & 31 : 16 * (q / 2) + (at_lane & 15); };
  auto group_col_of = [&](int at_lane, int q) { return F8 ? 8 * q + 4 * (at_lane >> 5) : 16 * (q % 2) + 4 * (at_lane >> 4); };
  auto group_row = [&](int q) { return group_row_of(lane, q); };
  auto group_col = [&](int q) { return group_col_of(lane, q); };

  // Partial tile of depth piece `piece` of the tile `ti` names: a lane's 16-byte group (i, j, q) sits
  // at ((i * NB + j) * 4 + q) * NT + thread, so one instruction of a wave moves 1 KiB of consecutive
  // bytes.
  auto partial_rsrc = [&](const TileInfo& tile, int piece) {
    return make_rsrc(p.workspace + kWsCounterBytes + (int64_t)(tile.slot + piece * tile.slots_apart) * (BM * BN * 4),
                     piece < tile.pieces ? BM * BN * 4 : 0);   // (no such piece: zeros)
  };
  auto partial_at = [&](int i, int j, int q) -> uint32_t { return (((i * NB + j) * 4 + q) * NT + threadIdx.x) * 16; };
  bool fix_pending = false;   // this workgroup's depth piece was the last of its tile to arrive

  // Where a tile's rows of c are: a descriptor of them, or of all of c when rows go through an
  // index, the byte offset of row `row` of the tile in it and that of one of its columns (C_OOR: no
  // such row or column, nothing is stored).
  constexpr int CE = ACC_F32 ? 4 : 2;   // bytes per element of c
  constexpr uint32_t C_OOR = INDEXED || KEEP ? kOutOfRangeIndexed : kOutOfRange;
  // (the rows of a tile, of the largest width, end before it: 256 x 2^22 elements of c, twice as many of gate | up, whose
  // widths are multiples of 8)
  static_assert(INDEXED || (uint64_t)BM * (ACC_F32 ? 1 << 20 : (KEEP ? (1 << 22) - 8 : 1 << 22)) * (KEEP ? 4 : CE) <= C_OOR, "");
  auto c_rsrc = [&](const TileInfo& tile) {
    if constexpr (INDEXED) return make_rsrc(p.c, p.c_bytes);
    return make_rsrc(p.c + (tile.g.c_off + (int64_t)tile.m0 * tile.g.n) * CE,
                     tile.rows_valid > 0 ? (uint32_t)(tile.rows_valid * tile.g.n) * (uint32_t)CE : 0u);
  };
  // ... and, KEEP, of the gate | up rows beside them, twice as long
  auto gate_up_rsrc = [&](const TileInfo& tile) {
    return make_rsrc(p.gate_up + (tile.g.c_off + (int64_t)tile.m0 * tile.g.n) * 4,
                     tile.rows_valid > 0 ? (uint32_t)(tile.rows_valid * tile.g.n) * 4u : 0u);
  };
  auto c_row = [&](const TileInfo& tile, int row) -> uint32_t {
    if constexpr (INDEXED) {
      if (row >= tile.rows_valid) return C_OOR;
      const int r = tile.g.row0 + tile.m0 + row;
      const uint32_t dst = p.c_rows != nullptr ? (uint32_t)p.c_rows[r] : (uint32_t)r;
      return dst < p.c_index_rows ? dst * (uint32_t)tile.g.n * 2u : C_OOR;   // no such row: not stored
    } else {
      return (uint32_t)(row * tile.g.n) * (uint32_t)CE;
    }
  };
  auto c_at = [&](const TileInfo& tile, uint32_t row_off, int col) -> uint32_t {
    return col < tile.g.n && (!INDEXED || row_off != C_OOR) ? row_off + (uint32_t)col * (uint32_t)CE : C_OOR;
  };
  // Rows of c on 2-byte boundaries and of any length (outputs of odd width, written where they belong: a padded
  // copy of them costs a pass more than the product's own): whole chunks at once, which global memory takes on
  // any boundary, the last ones of a row by elements.  8 x 1024 rows, 2047 -> 5461, forward and gradients: 834 us with
  // padded results copied back (120 of them the copies), 760 so.
  constexpr bool ANY_ROWS = EPI == kEpiStore && !INDEXED && !RAGGED_DEPTH && !F8;
  // ... or that are no whole groups of 4 columns, which the fix-up of depth pieces stores (whole tiles / pieces, us: weight
  // gradients of 21 Zipf (1.2) groups, 51204 rows, 128 x 558: 125 / 38; 64, 49152 rows, 2046 x 1406: 492 / 364; 16 groups, 600 rows,
  // 6144 -> 518: 46.8 / 33.8).
  constexpr bool FIX_ANY_ROWS = EPI == kEpiStore && !INDEXED && !F8;
  auto store_any = [&](const TileInfo& tile, uint32_t row_off, int col, int most, u32x4 v) {
    struct Chunk {
      u32x4 v;
    } __attribute__((packed, aligned(2)));
    const int left = row_off < (uint32_t)(tile.rows_valid * tile.g.n) * 2u ? tile.g.n - col : 0;
    uint16_t* to = reinterpret_cast<uint16_t*>(p.c + (tile.g.c_off + (int64_t)tile.m0 * tile.g.n) * 2 + row_off) + col;
    if (most == 8 && left >= 8) {
      reinterpret_cast<Chunk*>(to)->v = v;
    } else {
      uint64_t low = (uint64_t)v[1] << 32 | v[0], high = (uint64_t)v[3] << 32 | v[2];
#pragma unroll 1
      for (int e = left < most ? left : most; e > 0; --e) {
        *to++ = (uint16_t)low;
        low = low >> 16 | high << 48;
        high >>= 16;
      }
    }
  };
  // silu(gate) * up of four element pairs, rounded.  gate / (1 + exp(-gate)), the division by Markstein's
  // scheme: the hardware's reciprocal (one unit in the last place; of a quarter of the divisor, whose reciprocal
  // is normal), a quotient from it and one correction by the quotient's remainder, which a fused multiply-add
  // gives exactly.  That is as good as the compiler's division in six instructions instead of ten.  The remainder
  // is not a number where the divisor or gate is infinite: the maximum then puts a number in its place, and the
  // quotient keeps its 0 or infinity.  (16 x 1024 rows, 2048 -> 4096, forward and backward, and decode, 8 x 16 rows,
  // 4096 -> 14336: within 0.3 % of the bare reciprocal, whose results are off by a unit and more.)
  auto combine4 = [](const float* gate, const float* up) {
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float d = 1.0f + __expf(-gate[r]), inverse = 0.25f * __builtin_amdgcn_rcpf(0.25f * d);
      const float q = gate[r] * inverse, remainder = __builtin_fmaf(-d, q, gate[r]);
      o[r] = __builtin_fmaf(__builtin_fmaxf(remainder, -__FLT_MAX__), inverse, q) * up[r];
    }
    return round4<OUT_DT>(o[0], o[1], o[2], o[3]);
  };
  // Row blocks this wave has stored of the tile before (0: none, or all of it has arrived), and the
  // store instructions of one (at least; more of them only make the wait that counts them stricter).
  int stored = 0;
  constexpr int STORES = ACC_F32 ? 8 : (GATE_UP ? Cfg::WTN / 32 : NB / 2 * 4);
  static_assert(LOADS_PER_STAGE + STORES * MB < 64, "vmcnt is a 6-bit field");

  // One tile, for a wave that has ML row blocks with rows in them (the tile's row blocks go to
  // the wave rows alternately).  One copy of this body exists per value of ML; a tile picks
  // its copy once, so no accumulator ever lives across a choice.
  //
  // A slice (buffer X, the other buffer Y holds the next slice) is S matrix instructions; the first half multiplies
  // fragment sets 0 and 1, which are there when it begins, the second half sets 2 and 3:
  //   to READ_END     the fragments of sets 2 and 3 are read from X
  //   at RELEASE      all waves have them: X goes to the fetch cursor, which starts the slice two ahead into it, all
  //                   of its loads by the end of this slice, i.e. ahead of the stores of a tile that ends with it
  //   from READY      Y is complete for every wave: the fragments of the next slice's sets 0 and 1 are read from it
  //                   (all MB of A's: the next slice may be the next tile's)
  // Reads and loads are spread evenly over their spans.  LDS delivers the fragments of full tiles in half of a slice's
  // matrix time and takes the loads in a quarter of it.
  auto tile_body = [&](auto ml_tag) {
    constexpr int ML = decltype(ml_tag)::value;
    // MFMAs: blocks of 32 x 32 outputs for fp8, of 16 x 16 for two-byte elements
    constexpr int EDGE = F8 ? 1 : 2, MFMA_M = ML * EDGE, MFMA_N = NB * EDGE;
    std::conditional_t<F8, f32x16, f32x4> acc[MFMA_M][MFMA_N];
#pragma unroll
    for (int i = 0; i < MFMA_M; ++i)
#pragma unroll
      for (int j = 0; j < MFMA_N; ++j)
#pragma unroll
        for (int r = 0; r < (F8 ? 16 : 4); ++r) acc[i][j][r] = 0.0f;
    // Group q (see group_row) of the 32 x 32 block (i, j), moved out of the accumulation registers here and no earlier:
    // all of them at once would not fit beside the next tile's fragments.  (How that is said decides what the compiler
    // makes of it: read in assembly, the plain epilogues of full tiles get by without moves and spills; tied
    // to the accumulation registers, those that combine two products do.  Small tiles have room.)
    auto take = [&](int i, int j, int q, float* v) {
      auto& from = F8 ? acc[i][j] : acc[2 * i + q / 2][2 * j + q % 2];
      constexpr bool TIED = !F8 && (GATE_UP || ((INDEXED || RAGGED_DEPTH) && BM > 128));
      if constexpr (TIED) asm volatile("" : "+a"(from));
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = from[F8 ? 4 * q + r : r];
        if constexpr (F8 || (MB * NB > 4 && !TIED)) {
          asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v[r]) : "a"(x));
        } else {
          asm volatile("" : "+v"(x));
          v[r] = x;
        }
      }
    };

    constexpr int S = 2 * MFMA_M * MFMA_N;
    constexpr int READ_END = S * AT_READ_END / 32, RELEASE = S * AT_RELEASE / 32, READY = S * AT_READY / 32, LOAD_END = S * AT_LOAD_END / 32;
    static_assert(READ_END <= RELEASE && RELEASE <= READY && 2 * READY >= S && READ_END > 0 && READY < S && LOAD_END - S <= READ_END, "");
    using Loads = LoadSlots<LOADS_PER_STAGE, RELEASE, READY, LOAD_END, S>;
    static_assert(Loads::before(S) == FIRST_LOADS, "the copies of this body take over from one another");
    // Matrix instructions FIRST .. LAST - 1, with the LDS reads and global loads placed behind them, in this
    // order, so they run under the matrix pipe.
    auto slots = [&](auto first_tag, auto last_tag, int y) {
      constexpr int FIRST = decltype(first_tag)::value, LAST = decltype(last_tag)::value;
      static_for<LAST - FIRST>([&](auto m_tag) {
        constexpr int m = FIRST + decltype(m_tag)::value, n = m % (S / 2), set = m < S / 2 ? 0 : 2;
        // serpentine over the 32 x 32 blocks and over the 16 x 16 ones in them: consecutive MFMAs share one operand, and the
        // fragments are wanted no faster than they come (columns of 16 x 16 blocks want all of A's at once)
        constexpr int quarter = F8 ? 0 : n % 4, block = F8 ? n : n / 4;
        constexpr int j = block / ML, i = (j % 2 == 0) ? block % ML : ML - 1 - block % ML;
        constexpr int hi = quarter / 2, hj = quarter == 1 || quarter == 2 ? 1 : 0;   // halves of A's and of B's block
        // operands swapped: the result block is held transposed, so a lane owns four
        // consecutive columns of one output row
        if constexpr (F8) {   // (takes both halves of both fragments)
          acc[i][j] = mfma_32x32x64_f8<DT>(fb[set][j], fb[set + 1][j], fa[set][i], fa[set + 1][i], acc[i][j]);
        } else {
          f32x4& sum = acc[2 * i + hi][2 * j + hj];
          sum = mfma_16x16x32<DT>(fb[set + hj][j], fa[set + hi][i], sum);
          // (the first slice of a weight gradient's tile is a copy of the loop's, see the wait below: said to be in accumulation registers
          // from there on, half as many of its sums are moved to others and back, each behind a matrix result.  One slice, 128
          // groups x 30 rows, 2048 x 1408: 132.3 / 129.5 us; two, 64 x 64, 4096 x 4096: 389.7 / 385.2; four or more: the same.  As
          // the second of a pair, where there are 12 moves either way, and with the epilogues that accumulate it gains nothing.)
          if constexpr (LAYOUT == kTN && BM == 256 && EPI == kEpiStore && !PART::SECOND && m < S / 2) asm volatile("" : "+a"(sum));
        }
        if constexpr (m < READ_END) {
          constexpr int U = 2 * (ML + NB), u0 = U * m / READ_END, u1 = U * (m + 1) / READ_END;
          static_for<u1 - u0>([&](auto d) { read_unit(std::integral_constant<int, u0 + decltype(d)::value>{}, I2{}, ml_tag, x); });
        } else if constexpr (m >= READY) {
          constexpr int U = 2 * (MB + NB), u0 = U * (m - READY) / (S - READY), u1 = U * (m + 1 - READY) / (S - READY);
          static_for<u1 - u0>([&](auto d) { read_unit(std::integral_constant<int, u0 + decltype(d)::value>{}, I0{}, IMB{}, y); });
        }
        // (a load on its own is aimed behind the instruction before: all of it behind one of 16 cycles would hold up the next)
        constexpr int at = m < READ_END ? m + S : m;   // (loads of the slice before reach up to there)
        const int to = m < READ_END ? y : x;
        constexpr int l0 = Loads::before(at), l1 = Loads::before(at + 1);
        if constexpr (Loads::alone(at)) {
          __builtin_amdgcn_sched_barrier(0);   // (the instruction stays between the two)
          fetch_load(std::integral_constant<int, l0>{}, std::false_type{});
        } else {
          static_for<l1 - l0>([&](auto d) { fetch_whole(std::integral_constant<int, l0 + decltype(d)::value>{}, to); });
        }
        if constexpr (m + 1 != READ_END && Loads::alone(at + 1)) fetch_aim(std::integral_constant<int, l1>{}, to);
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    using IReadEnd = std::integral_constant<int, READ_END>;
    using IRelease = std::integral_constant<int, RELEASE>;
    using IReady = std::integral_constant<int, READY>;
    using IAll = std::integral_constant<int, S>;

    for (int kt = 0; kt < ti.nk; ++kt) {
      const int y = uniform(x ^ 1);   // (the same in every lane: keeps the LDS addresses scalar)
      if constexpr (LATE_LOADS) {
        // (the descriptor of the last loads comes from the iteration before, for all the compiler knows in vector
        // registers; the first of them is behind a matrix instruction, fetch_aim and a wait)
#pragma unroll
        for (int w = 0; w < 4; ++w) b_slice.rsrc[w] = uniform(b_slice.rsrc[w]);
        settle<2>(b_slice.rsrc);
      }
      slots(I0{}, IReadEnd{}, y);
      fetch_advance();
      fetch_begin();
      slots(IReadEnd{}, IRelease{}, y);
      // every wave has all fragments of this slice in registers
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      block_barrier();
      slots(IRelease{}, IReady{}, y);
      // the next slice has landed for every wave (only the loads just issued may be pending and, in the first
      // slice after a tile that was stored, its stores)
      constexpr int PENDING = Loads::before(READY);
      // (in the weight-gradient layout the condition is one of the first slice's, which the compiler then takes out of the
      // loop, as long as there is no loop in this one: with that wait in the loop it moves accumulators in and out of it, 332
      // moves a slice.  Without a copy and without a move, the waits chosen among in assembly and every accumulator's zeros its
      // own, the loop is slower for the branches in each slice: 8 x 4096 rows, 4096 x 14336: 2632 / 2702 us; 256 x 256, 2048 x 7168:
      // 2561 / 2600)
      if (LATE_LOADS || (LAYOUT == kTN && kt > 0) || __builtin_expect(uniform(stored) == 0, 1)) {
        wait_vmcnt<PENDING>();
      } else {
        if (uniform(stored) == MB) {
          wait_vmcnt<PENDING + STORES * MB>();
        } else {
          wait_vmcnt<PENDING + STORES>();
        }
        if (LAYOUT != kTN) stored = 0;   // (the next wait is for them too)
      }
      block_barrier();
      if constexpr (RAGGED_DEPTH) {
        if (tail_next) clear_tail(y);
        tail_next = tail_fetched;
      }
      slots(IReady{}, IAll{}, y);
      x = uniform(y);
    }

    // A depth piece of a tile of the last round: park the partial tile in the workspace and
    // count the arrival.  The piece that arrives last adds the partial tiles up and stores the
    // sum, after the tile loop (fix_up below), where no accumulator is live any more.
    if (DEPTH_PIECES && ti.pieces > 1) {
      const __amdgpu_buffer_rsrc_t mine = partial_rsrc(ti, ti.piece);
#pragma unroll
      for (int i = 0; i < ML; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            f32x4 v;
            if constexpr (F8) {
              v = f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            } else {
              v = acc[2 * i + q / 2][2 * j + q % 2];
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), mine, partial_at(i, j, q), 0, kDeviceScope);
          }
      wait_vmcnt<0>();   // every wave's part has arrived before the arrival is counted
      stored = 0;
      block_barrier();
      if (threadIdx.x == 0) sched->arrived = __hip_atomic_fetch_add(reinterpret_cast<int*>(p.workspace) + ti.rank, 1, __ATOMIC_RELAXED,
                                                                        __HIP_MEMORY_SCOPE_AGENT);
      // (the barrier alone orders nothing: without the wait another wave could read the word before
      // it is written, and would then add up a tile that is not complete, or leave its part out)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      block_barrier();
      fix_pending = uniform(sched->arrived) == ti.pieces - 1;
      if (fix_pending) {
        // Keep the tile's description for the fix-up after the tile loop (a piece of the last
        // round is this workgroup's last tile, one of a deep tile its first): copied from the
        // slot of the tile ring it was read from, which the fetch cursor, at most two tiles
        // ahead, has not reached again.  (Packing it from registers would keep every field live
        // through the depth loop, which has no scalar registers to spare.)
        static_assert(sizeof(sched->fix_tile) == kTileInfoDwords * 4 && kTileInfoDwords <= 64, "");
        if (threadIdx.x < kTileInfoDwords)
          sched->fix_tile[threadIdx.x] = tile_ring[(tile_n % Cfg::TILE_RING_SLOTS) * kTileInfoDwords + threadIdx.x];
      }
      return;
    }

    // Epilogue.  A lane owns four groups of 4 columns of each 32x32 block (group_row, group_col).
    // The accumulators stay in the accumulation registers; each value is moved out right
    // where it is converted, so the epilogue needs only a few vector registers.
    {
      constexpr uint32_t OOR = C_OOR;
      const __amdgpu_buffer_rsrc_t rc = c_rsrc(ti);
      auto row_offset = [&](int row) { return c_row(ti, row); };
      auto at = [&](uint32_t row_off, int col) { return c_at(ti, row_off, col); };
      auto take4 = [&](int i, int j, int q) {
        float v[4];
        take(i, j, q, v);
        return round4<OUT_DT>(v[0], v[1], v[2], v[3]);
      };
      if constexpr (GATE_UP) {
        // Blocks 2 jp and 2 jp + 1 of a wave hold the gate and the up value of the same 32 output
        // columns, element for element: silu(gate) * up in fp32, one rounding, then through the wave's
        // LDS strip (32 rows x the wave's output columns) so that stores are 16 bytes per lane and
        // whole lines: the 8-byte pieces the lanes hold, 16 bytes of a line per row and instruction,
        // were written at that size past L2 (16 x 1024 rows, 2048 -> 4096: 637 -> 574 us; decode,
        // 8 x 16 rows, 4096 -> 14336: 357 -> 348).
        constexpr int OUTW = Cfg::WTN / 2, CHUNKS = OUTW / 8, ROWS = 64 / CHUNKS, PITCH = Cfg::EPILOGUE_PITCH;
        char* strip = smem + Cfg::EPILOGUE_OFFSET + wave * Cfg::EPILOGUE_WAVE_BYTES;
        const int out_row = lane / CHUNKS, out_chunk = lane % CHUNKS;
        const int col = ti.n0 + wn * OUTW + out_chunk * 8;
        u32x4 held[32 / ROWS];   // (one strip behind, as below)
        uint32_t held_off[32 / ROWS];
        const bool merge = uniform(p.flags & kFlagMergeStores) != 0;
        // What is held, to columns at_col .. +7 of the rows at held_off.
        auto store_held_to = [&](const __amdgpu_buffer_rsrc_t& to, int at_col) {
          auto chunk_at = [&](int r) {
            return col < ti.g.n && (!INDEXED || held_off[r] != C_OOR) ? held_off[r] + (uint32_t)at_col * 2u : OOR;
          };
          if (merge) {
#pragma unroll
            for (int r = 0; r < 32 / ROWS; ++r)
              __builtin_amdgcn_raw_buffer_store_b128(held[r], to, chunk_at(r), 0, kStoreMerging);
          } else {
#pragma unroll
            for (int r = 0; r < 32 / ROWS; ++r)
              __builtin_amdgcn_raw_buffer_store_b128(held[r], to, chunk_at(r), 0, kStoreStreaming);
          }
        };
        auto hold_strip = [&](const uint32_t* row_off) {
#pragma unroll
          for (int r = 0; r < 32 / ROWS; ++r) {
            held[r] = *reinterpret_cast<const u32x4*>(strip + (r * ROWS + out_row) * PITCH + out_chunk * 16);
            held_off[r] = row_off[r];
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        auto into_strip = [&](int jp, int q, u32x2 v) {
          *reinterpret_cast<u32x2*>(strip + group_row(q) * PITCH + (jp * 32 + group_col(q)) * 2) = v;
        };
#pragma unroll
        for (int i = 0; i < ML; ++i) {
          uint32_t row_off[32 / ROWS];
#pragma unroll
          for (int r = 0; r < 32 / ROWS; ++r) row_off[r] = row_offset((wm + i * WAVES_M) * 32 + r * ROWS + out_row);
          if constexpr (KEEP) {
            // The gate columns, then the up columns, as the plain epilogue would store them (16 x 1024 rows,
            // 2048 -> 4096: 520 us, 590 with them; the product that the backward would run for them: 490).
            const __amdgpu_buffer_rsrc_t rg = gate_up_rsrc(ti);
            uint32_t keep_off[32 / ROWS];
#pragma unroll
            for (int r = 0; r < 32 / ROWS; ++r) keep_off[r] = 2 * row_off[r];
#pragma unroll
            for (int part = 0; part < 2; ++part) {
#pragma unroll
              for (int jp = 0; jp < NB / 2; ++jp)
#pragma unroll
                for (int q = 0; q < 4; ++q) into_strip(jp, q, take4(i, 2 * jp + part, q));
              if (part == 1) {
                store_held_to(rg, col);
              } else if (i > 0) {
                store_held_to(rc, col);
              }
              hold_strip(keep_off);
            }
          }
#pragma unroll
          for (int jp = 0; jp < NB / 2; ++jp) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              float gate[4], up[4];
              take(i, 2 * jp, q, gate);
              take(i, 2 * jp + 1, q, up);
              into_strip(jp, q, combine4(gate, up));
            }
          }
          if constexpr (KEEP) {
            store_held_to(gate_up_rsrc(ti), ti.g.n + col);
          } else {
            if (i > 0) store_held_to(rc, col);
          }
          hold_strip(row_off);
        }
        store_held_to(rc, col);
      } else if constexpr (ACC_F32) {
        if constexpr (EPI == kEpiAccF32Atomic) {
          // c += product in fp32, by atomic additions that return nothing: the wave fires them and
          // moves on, where a read-add-write would wait for the reads (every element of c belongs
          // to one tile, so each gets exactly one addition per call and the result is the same).
          // One 32 x 32 block at a time goes through the wave's LDS strip, in as the 16-byte pieces
          // the lanes hold, out as one float per lane, 32 lanes to a row: an instruction then adds
          // to two complete 128-byte lines.
          char* strip = smem + Cfg::EPILOGUE_OFFSET + wave * Cfg::EPILOGUE_WAVE_BYTES;
          constexpr int PITCH = Cfg::EPILOGUE_PITCH;   // 32 floats and 16 bytes of padding
#pragma unroll
          for (int i = 0; i < ML; ++i) {
#pragma unroll
            for (int j = 0; j < NB; ++j) {
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                float v[4];
                take(i, j, q, v);
                *reinterpret_cast<f32x4*>(strip + group_row(q) * PITCH + group_col(q) * 4) = f32x4{v[0], v[1], v[2], v[3]};
              }
              // (offsets from one per block on: worked out per instruction they do not change from tile to
              // tile, and the compiler keeps them in more registers than there are: reloading those it
              // spilled waits for the atomics ahead of them: 2.9 % of 8 x 4096 rows, 4096 x 14336)
              int at_lane = lane;
              asm volatile("" : "+v"(at_lane));
              const int col = ti.n0 + wn * Cfg::WTN + j * 32 + (at_lane & 31);
              uint32_t off = col < ti.g.n ? (uint32_t)(((wm + i * WAVES_M) * 32 + (at_lane >> 5)) * ti.g.n + col) * 4u : kOutOfRange;
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const float v = *reinterpret_cast<const float*>(strip + (r * 2 + (lane >> 5)) * PITCH + (lane & 31) * 4);
                __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(v, rc, off, 0, 0);
                off += (uint32_t)ti.g.n * 8u;   // two rows (stays out of range: widths are below 2^20 here)
              }
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        } else {
          // c += product in fp32.  The 4 consecutive columns a lane holds are 16 bytes of c:
          // read them, add, write them back; the lanes of an instruction cover 64 (fp8: 32) contiguous bytes of a
          // row, the instructions of a block 128-byte lines.  All reads of a 32-row block row are
          // issued before the first addition: 16 in flight per lane measured faster than a
          // rolling 8 + 8.
#pragma unroll
          for (int i = 0; i < ML; ++i) {
            // (offsets are worked out again for the stores: kept, they take more registers than there are)
            auto offset = [&](int at_lane, int j, int q) {
              const int row = (wm + i * WAVES_M) * 32 + group_row_of(at_lane, q);
              const int col = ti.n0 + wn * Cfg::WTN + j * 32 + group_col_of(at_lane, q);
              return col < ti.g.n ? (uint32_t)(row * ti.g.n + col) * 4u : kOutOfRange;
            };
            u32x4 old[NB][4];
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
              for (int q = 0; q < 4; ++q) old[j][q] = __builtin_amdgcn_raw_buffer_load_b128(rc, offset(lane, j, q), 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            int at_lane = lane;
            asm volatile("" : "+v"(at_lane));
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                float v[4];
                take(i, j, q, v);
                const f32x4 sum = __builtin_bit_cast(f32x4, old[j][q]) + f32x4{v[0], v[1], v[2], v[3]};
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum), rc, offset(at_lane, j, q), 0, 0);
              }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      } else {
        // Through a strip of LDS private to the wave: 32 rows x 64 columns go in as the
        // 8-byte pieces the lanes hold and come out as 16 bytes per lane, 8 lanes per row, so
        // that one store instruction writes 8 complete 128-byte lines.
        char* strip = smem + Cfg::EPILOGUE_OFFSET + wave * Cfg::EPILOGUE_WAVE_BYTES;
        constexpr int PITCH = Cfg::EPILOGUE_PITCH;
        const int out_row = lane >> 3, out_chunk = lane & 7;
        // an even width that is not a multiple of 8: rows of c then start on 4-byte boundaries
        // only, and the last 16-byte chunk of a row holds 2, 4 or 6 columns
        const bool ragged_width = uniform(ti.g.n & 7) != 0;
        const bool any_rows = ANY_ROWS && uniform(p.flags & kFlagAnyRows) != 0;
        const bool merge = uniform(p.flags & kFlagMergeStores) != 0;
        // One strip behind: the reads of a strip return while the next one is converted (the LDS
        // serves a wave in order, so the next strip's writes need not wait for them).
        u32x4 held[4];
        uint32_t held_off[4];
        int held_col = 0;
        auto store_held = [&]() {
          if (any_rows) {
#pragma unroll
            for (int r = 0; r < 4; ++r) store_any(ti, held_off[r], held_col, 8, held[r]);
            return;
          }
          // (whole chunks only: for widths that are multiples of 8 the same as col < n)
          auto chunk_at = [&](int r) { return held_col + 8 <= ti.g.n ? at(held_off[r], held_col) : OOR; };
          if (merge) {
#pragma unroll
            for (int r = 0; r < 4; ++r) __builtin_amdgcn_raw_buffer_store_b128(held[r], rc, chunk_at(r), 0, kStoreMerging);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              __builtin_amdgcn_raw_buffer_store_b128(held[r], rc, chunk_at(r), 0, kStoreStreaming);
          }
          if (ragged_width) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const u32x4 v = held[r];
              const int valid = ti.g.n - held_col;   // columns of this lane's chunk that exist
              const uint32_t off = at(held_off[r], held_col);
              if (valid > 0 && valid < 8 && off != OOR) {
                if (valid & 4) __builtin_amdgcn_raw_buffer_store_b64(u32x2{v[0], v[1]}, rc, off, 0, kStoreMerging);
                if (valid & 2)
                  __builtin_amdgcn_raw_buffer_store_b32((valid & 4) ? v[2] : v[0], rc, off + ((valid & 4) ? 8u : 0u), 0,
                                                        kStoreMerging);
              }
            }
          }
        };
#pragma unroll
        for (int i = 0; i < ML; ++i) {
          uint32_t row_off[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) row_off[r] = row_offset((wm + i * WAVES_M) * 32 + r * 8 + out_row);
#pragma unroll
          for (int jp = 0; jp < NB / 2; ++jp) {
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
              for (int q = 0; q < 4; ++q)
                *reinterpret_cast<u32x2*>(strip + group_row(q) * PITCH + (jj * 32 + group_col(q)) * 2) =
                    take4(i, 2 * jp + jj, q);
            if (i + jp > 0) store_held();
            held_col = ti.n0 + wn * Cfg::WTN + jp * 64 + out_chunk * 8;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              held[r] = *reinterpret_cast<const u32x4*>(strip + (r * 8 + out_row) * PITCH + out_chunk * 16);
              held_off[r] = row_off[r];
            }
            // keep the conversion of one strip from being hoisted over the stores of the
            // previous one: few accumulators are live in vector registers at a time
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        store_held();
      }
      stored = ANY_ROWS && (p.flags & kFlagAnyRows) != 0 ? 0 : ML;   // (not every store is sent there: nothing to count on)
    }
  };

  while (true) {
    // row blocks of this tile that fall to this wave row: blocks wm, wm + WAVES_M, ...
    const int live = uniform((ti.blocks - wm + WAVES_M - 1) / WAVES_M);
    if constexpr (LAYOUT == kTN || MB == 1) {
      tile_body(IMB{});
    } else {
      static_assert(MB == 4, "one copy of the tile body per live block count 1..4");
      if (live >= 4) {
        tile_body(std::integral_constant<int, 4>{});
      } else if (live == 3) {
        tile_body(std::integral_constant<int, 3>{});
      } else if (live == 2) {
        tile_body(std::integral_constant<int, 2>{});
      } else {
        tile_body(std::integral_constant<int, 1>{});
      }
    }
    tile_t = next_index(tile_t);
    if (tile_t >= total_tiles) break;
    tile_n = uniform(tile_n + 1);
    ti = next_tile();
  }
  wait_vmcnt<0>();   // the zero-filling fetches past the last tile still write LDS

  // Fix-up of a tile that was cut along the depth: the tile this workgroup left in
  // Sched::fix_tile when its piece arrived last (a workgroup has at most one).  The partial tiles
  // are added up in piece order, two per step, whichever piece does the
  // adding, so the result does not depend on timing.  One block row of 32 rows at a time: NB * 4
  // groups of 16 bytes per lane and piece.
  if (DEPTH_PIECES && fix_pending) {
    __syncthreads();   // (the description was written by the first threads of the workgroup)
    int32_t words[kTileInfoDwords];
#pragma unroll
    for (int i = 0; i < kTileInfoDwords; ++i) words[i] = sched->fix_tile[i];
    const TileInfo ft = unpack_tile(words);
    if (threadIdx.x == 0) reinterpret_cast<int*>(p.workspace)[ft.rank] = 0;   // leave the counters as they were found
    const __amdgpu_buffer_rsrc_t rc = c_rsrc(ft);
    const int live = LAYOUT == kTN ? MB : (ft.blocks - wm + WAVES_M - 1) / WAVES_M;
    for (int i = 0; i < live; ++i) {
      f32x4 sum[NB][4];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) sum[j][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      for (int piece = 0; piece < ft.pieces; piece += 2) {
        const __amdgpu_buffer_rsrc_t from0 = partial_rsrc(ft, piece), from1 = partial_rsrc(ft, piece + 1);
        f32x4 v0[NB][4], v1[NB][4];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            v0[j][q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from0, partial_at(i, j, q), 0, kDeviceScope));
            v1[j][q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from1, partial_at(i, j, q), 0, kDeviceScope));
          }
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) sum[j][q] = (sum[j][q] + v0[j][q]) + v1[j][q];
      }
      // (groups 0 and 1 of a lane share their row, and 2 and 3; for fp8 all four)
      const uint32_t rows_off[2] = {c_row(ft, (wm + i * WAVES_M) * 32 + group_row(0)), c_row(ft, (wm + i * WAVES_M) * 32 + group_row(2))};
      if constexpr (GATE_UP) {
#pragma unroll
        for (int jp = 0; jp < NB / 2; ++jp)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float gate[4], up[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) gate[r] = sum[2 * jp][q][r], up[r] = sum[2 * jp + 1][q][r];
            const uint32_t row_off = rows_off[q / 2];
            const int col = ft.n0 + wn * (Cfg::WTN / 2) + jp * 32 + group_col(q);
            __builtin_amdgcn_raw_buffer_store_b64(combine4(gate, up), rc, c_at(ft, row_off, col), 0, kStoreMerging);
            if constexpr (KEEP) {
              const __amdgpu_buffer_rsrc_t rg = gate_up_rsrc(ft);
              const uint32_t gate_off = col < ft.g.n ? 2 * row_off + (uint32_t)col * 2u : C_OOR;
              const uint32_t up_off = col < ft.g.n ? 2 * row_off + (uint32_t)(ft.g.n + col) * 2u : C_OOR;
              __builtin_amdgcn_raw_buffer_store_b64(round4<OUT_DT>(gate[0], gate[1], gate[2], gate[3]), rg, gate_off, 0, kStoreMerging);
              __builtin_amdgcn_raw_buffer_store_b64(round4<OUT_DT>(up[0], up[1], up[2], up[3]), rg, up_off, 0, kStoreMerging);
            }
          }
      } else {
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t row_off = rows_off[q / 2];
            const int col = ft.n0 + wn * Cfg::WTN + j * 32 + group_col(q);
            const uint32_t off = c_at(ft, row_off, col);
            if (FIX_ANY_ROWS && ((p.flags & kFlagAnyRows) != 0 || uniform(ft.g.n & 3) != 0)) {
              const u32x2 v = round4<OUT_DT>(sum[j][q][0], sum[j][q][1], sum[j][q][2], sum[j][q][3]);
              store_any(ft, row_off, col, 4, u32x4{v[0], v[1], 0u, 0u});
            } else if constexpr (ACC_F32) {
              const f32x4 old = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rc, off, 0, 0));
              __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, old + sum[j][q]), rc, off, 0, 0);
            } else {
              __builtin_amdgcn_raw_buffer_store_b64(
                  round4<OUT_DT>(sum[j][q][0], sum[j][q][1], sum[j][q][2], sum[j][q][3]), rc, off, 0, kStoreMerging);
            }
          }
      }
    }
  }
}

template <int DT, int LAYOUT, int BM, int BN, int BK, int STAGES, int WAVES_M, int WAVES_N,
          int EPI = kEpiStore, bool INDEXED = false, bool RAGGED_DEPTH = false>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64,
                             (GmmConfig<LAYOUT, BM, BN, BK, STAGES, WAVES_M, WAVES_N>::WORKGROUPS_PER_CU)) void
gmm_kernel(GmmParams p, HostSizes hs) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub
  using Cfg = GmmConfig<LAYOUT, BM, BN, BK, STAGES, WAVES_M, WAVES_N>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  gmm_tiles<DT, LAYOUT, BM, BN, BK, STAGES, WAVES_M, WAVES_N, EPI, INDEXED, RAGGED_DEPTH>(p, hs, smem, (int)blockIdx.x,
                                                                                        (int)gridDim.x, Alone<Cfg::WORKGROUPS_PER_CU>{});
#endif
}

// Both gradients of a product in one launch: workgroups 0 .. G - 1 work on the input gradient (shape S1, layout
// LAYOUT1), G .. 2 G - 1 on the weight gradient (S2).  A compute unit has room for one of them, so the
// second half starts as the first half ends: compute units that the first product's last round leaves idle begin
// the second product at once, and what a launch takes to start and to drain (4 of the 8 us of a small one)
// passes once.  Us, two launches and one: 8 x 128 rows, 128 x 128: 15.6 / 11.2; 32 x 128, 768 x 2048: 67 / 61; 8 x
// 1024, 2048 x 5464: 461 / 376; 64 Zipf groups, 49152 rows, 2048 x 1408: 623 / 611; 43 x 848, 5696 x 2752: 2097 / 2110.
template <int LAYOUT1, typename S1, typename S2, int BK, int STAGES>
struct PairConfig {
  using First = GmmConfig<LAYOUT1, S1::BM, S1::BN, BK, STAGES, S1::WAVES_M, S1::WAVES_N>;
  using Second = GmmConfig<kTN, S2::BM, S2::BN, BK, STAGES, S2::WAVES_M, S2::WAVES_N>;
  static_assert(First::NT == Second::NT, "");
  static constexpr int NT = First::NT;
  static constexpr int LDS_BYTES = First::LDS_BYTES > Second::LDS_BYTES ? First::LDS_BYTES : Second::LDS_BYTES;
  static constexpr int WORKGROUPS_PER_CU = 2 * LDS_BYTES <= 160 * 1024 ? 2 : 1;
};
template <int DT, int LAYOUT1, typename S1, typename S2, int BK, int STAGES>
__global__ __launch_bounds__((PairConfig<LAYOUT1, S1, S2, BK, STAGES>::NT), (PairConfig<LAYOUT1, S1, S2, BK, STAGES>::WORKGROUPS_PER_CU)) void
gmm_pair_kernel(GmmParams p1, GmmParams p2, HostSizes hs) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int WGS = PairConfig<LAYOUT1, S1, S2, BK, STAGES>::WORKGROUPS_PER_CU;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int G = (int)gridDim.x / 2, w = (int)blockIdx.x;
  if (w < G) {
    gmm_tiles<DT, LAYOUT1, S1::BM, S1::BN, BK, STAGES, S1::WAVES_M, S1::WAVES_N, kEpiStore, false, false>(
        p1, hs, smem, w, G, FirstOfPair<WGS>{});
  } else {
    gmm_tiles<DT, kTN, S2::BM, S2::BN, BK, STAGES, S2::WAVES_M, S2::WAVES_N, kEpiStore, false, false>(
        p2, hs, smem, w - G, G, SecondOfPair<WGS, LAYOUT1, S1::BM, S1::BN>{p1});
  }
#endif
}

}  // namespace gg
