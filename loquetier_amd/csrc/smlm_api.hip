// C ABI of libsmlm_hip (see include/smlm.h): argument checks, workspace
// carving, launch-shape choice and kernel dispatch.  No allocation, no host
// synchronisation, no state.
#include <hip/hip_runtime.h>

#include <string.h>

#include <atomic>

#include "put_words.hpp"
#include "rms_norm.hpp"
#include "segments.hpp"
#include "smlm.h"
#include "smlm_backward.hpp"
#include "smlm_common.hpp"
#include "smlm_decode.hpp"
#include "smlm_forward.hpp"
#include "smlm_plan.hpp"

using namespace smlm;

// Scratch of smlm_gemm_static (file scope; see static_scratch below).
static __device__ __align__(256) unsigned char scratch[SMLM_STATIC_SCRATCH_BYTES];

namespace {

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
inline int round_up(int a, int b) { return ceil_div(a, b) * b; }

// Every kernel takes one argument struct.  hipLaunchKernel hands back the
// status of this launch itself; the thread's "last error" slot is shared with
// every other HIP user in the process (torch leaves benign codes there), so it
// is neither read nor cleared here.
template <typename A>
int launch(void (*kernel)(A), dim3 grid, dim3 block, hipStream_t st, const A& a) {
  void* params[] = {const_cast<A*>(&a)};
  return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, params, 0, st) ==
                 hipSuccess
             ? SMLM_OK
             : SMLM_ERR_LAUNCH;
}

// ---- launch shapes: functions of (T, d_in, d_out) only, never of the
// segmentation, so re-segmenting a batch cannot change a bit of any row. ----
// Tiles per work item: single 16-row tiles for batches of few rows, tile blocks (up to kBlkTiles tiles of one
// adapter, their weights staged once in LDS) for larger ones.  Where the forward changes over depends on the
// rank -- the tile-block kernels save weight traffic in proportion to it.  Single tiles / tile blocks in us, one
// projection 4096 -> 4096: rank 16 at 2000 rows 18.4 / 20.8, at 3072 rows 26.0 / 24.5; rank 32 at 1024 rows
// 15.6 / 17.8, at 1536 rows 21.7 / 19.2; rank 64 at 256 rows 17.0 / 16.3, at 1000 rows 22.9 / 18.8.  A launch of
// several projections, whose workgroups fill the chip together, would change over earlier (q/k/v/o: rank 16 at
// 1024 rows 30.9 / 30.9, at 2048 rows 53.1 / 47.5; rank 32 at 384 rows 24.5 / 25.3, at 768 rows 34.6 / 30.7;
// rank 64 at 128 rows 27.6 / 24.7); the rule lies between the two and does not look at the number of
// projections, so that a launch of several gives the bits that launches of one give.
// Ranks above 64: rank 128, 4096 -> 4096, prompts of 512 rows 22.9 / 20.2, of 640 rows 34.7 / 21.7, q/k/v/o at 512
// rows 62.3 / 34.5, 1024 -> 4096 at 768 rows 23.6 / 18.8; the tile blocks lose where more than 512 segments take their
// plan out of the launch and k is short (1024 -> 4096, 768 decoded rows 37.5 / 43.0).
// Up to rank 96 the second block of 64 columns is at most half full, and the
// line also looks at the shortest k of the launch (h_in; projections of one input, as a group's, share it): rank 72,
// 4096 -> 4096, 512 rows 17.0 / 18.3, q/k/v/o 45.5 / 30.4; 2048 -> 2048, 768 rows 16.3 / 17.5; 1024 -> 4096, 1000
// rows 17.0 / 20.0.
constexpr int kNoShrink = 1 << 30;  // k of an expand by itself
inline int tiles_per_wave(int T, int r, int k) {
  int from;
  if (r <= 32) from = r <= 16 ? 2048 : 768;
  else if (r <= 64) from = r <= 48 ? 512 : 128;
  else from = (r <= 96 && k < 4096) ? 1024 : 512;
  return T >= from ? kBlkTiles : 1;
}
// (The backward runs on tile blocks at every size and rank: they read the weights the other way round as they lie
// in memory, where single tiles would need transposed copies of them first.  64 rows at rank 64, single tiles / tile
// blocks: 25.0 / 18.8 us; 1024 rows at rank 16: 28.3 / 25.3 us.)

// Upper bound of the number of work units along the tile axis.  `groups` bounds
// the number of distinct plan keys (adapters): every group ends in at most one
// partly filled tile and one partly filled tile block.
inline int tile_units_max(int T, int S, int groups, int mt) {
  const int g = (groups > 0 && groups < S) ? groups : S;
  const int nt = T / kTileRows + g + 1;  // never above the plan's own bound plan_nt_max(T, S)
  const int nb = nt / kBlkTiles + g + 2;
  return (mt == 1 || nb > nt) ? nt : nb;  // there are never more tile blocks than tiles
}

// Launches of at most this many items run one item per workgroup (direct mode); measured
// faster than the persistent walk at every size tried (up to ~130k workgroups), so the walk
// is only the fallback for batches far beyond those.
constexpr long kDirectItems = 1L << 22;
constexpr int kMaxGridY = 65535;  // tile units are the y axis of a direct launch

// persistent 1-D grid: a multiple of the XCD count, no larger than the work bound
constexpr int kMaxGrid = 2048;
inline dim3 work_grid(long bound) {
  const long cap = kMaxGrid;
  long g = bound < cap ? bound : cap;
  g = (g + kNumXcd - 1) / kNumXcd * kNumXcd;
  return dim3((unsigned)g);
}

struct ShrinkCfg {
  int NB, U, MT, NW, ksplit, k_per_wave, zblocks;
};

constexpr int kDecodeWaves = 8;  // waves of the decode shrink's workgroups ...
constexpr int kDecodeSplit = 4;  // ... and its k split over workgroups, folded by the expand kernel
constexpr int kMaxExpandFold = kMaxVsplit;  // most partials the expand kernel folds itself

// waves per shrink workgroup, one choice for all projections of a launch: small
// batches whose every projection has a long enough k use eight waves and split k in four
int shrink_waves(int mt, int nproj, const int* d_in, int d_out) {
  const int kq = 32 * (d_out > 32 ? 2 : 4);  // k per wave and load batch of the decode kernels
  bool all_long = mt == 1;
  for (int i = 0; i < nproj; ++i) all_long = all_long && d_in[i] >= 16 * kq;
  return all_long ? kDecodeWaves : kFwdWaves;
}

// Which of the two tile-block shrinks: shrink_block_kernel, whose waves read x and the weights for themselves, or
// shrink_wide_kernel, whose workgroups stage the weights once for four waves.  Shrink and fold, us, wide / block, h_in =
// 4096: one projection at rank 16, 2048 rows 13.0 / 11.6, 3000 rows 13.5 / 12.7; three at rank 32, 3000 rows 30 / 26.3; at
// rank 64 1500 rows 21 / 24.0, 2048 rows 23.5 / 25.8, 3000 rows 36 / 36, 7675 rows 68 / 60.
// Above rank 64 x would be read once for every 64 columns.
// Fewer rows belong to adapters of few rows each, and the block kernel reads 64 rows for however few.  What it loses and
// gains between 1024 and 2048 rows depends on that and on the number of projections, neither of which the rule may look
// at.  Whole forwards at rank 32, three projections: 1024 rows over 64 adapters 42.5 / 46.0, over 24 32.0 / 34.4, over 4
// 30.1 / 29.4, 1400 over 64 48.0 / 49.6; one: 1024 rows over 64 25.1 / 23.1, 1400 over 24 22.2 / 21.1; add_lora, 1300
// rows over 64 28.9 / 34.3.  Backwards, three projections at rank 16, 1024 rows over 64 69.1 / 73.6.  At ranks 17 to 32 it
// goes on to 3072 rows: 4096 -> 11008 twice and back, 2112 rows, the whole pass 79.7 / 81.5; two projections, 2048 rows
// over 100 47.9 / 50.3; 3072 rows over 4 to 64, three projections, 59.9 to 74.3 / 54.2 to 69.2.
// Under dropout the
// generator keeps the vector units busy and the wide kernel's waves, more of them on a CU, share it better: 2436 rows, two
// projections at rank 16 21.7 / 28.3.
inline bool block_shrink(int mt, int T, int d_out, bool drop = false) {
  return mt > 1 && !drop && T >= (d_out <= 16 ? 2048 : 3072) && d_out <= 64;
}
// ... of a launch: its weight rows must be within the block kernel's reach too (the slices are the same either way).
// Whoever decides on the plan's route asks this, as the launch does: the wide kernel needs the splits even where two
// groups of waves share a workgroup, and would store a slice past the last one.
inline bool block_shrink(int mt, int T, int d_out, bool drop, int nproj, const int* ldw) {
  bool near = block_shrink(mt, T, d_out, drop);
  for (int i = 0; i < nproj; ++i) near = near && ldw[i] <= kBlockMaxLd;
  return near;
}
inline bool block_shrink(int mt, const ShrinkArgs& a) {
  int ldw[kMaxProj];
  for (int i = 0; i < a.items.nproj; ++i) ldw[i] = a.p[i].ldw;
  return block_shrink(mt, a.T, a.p[0].d_out, a.drop.seg_p != nullptr, a.items.nproj, ldw);
}

// k slices of a tile-block shrink, in pieces of 256 of k (64 a wave): the split with the shortest time in steps of a
// piece -- rounds of workgroups over the 256 CUs times (pieces of a slice + what starting one costs), an eighth more where
// a CU has one workgroup only, the partial sums, and the fold, which costs as much as three pieces.  An uneven last
// round is what costs most: 4096 rows, h_in = 11008 at rank 64, k in five 44.4 us, in four 30.4, in eight 33.6.
// us with k in 1 / 2 / 4 / 8 / 16, one projection of h_in = 4096 at rank 64: 4096 rows - / 20.0 / 17.3 / 19.1 / 24.6;
// 8192 rows 27.1 / 29.3 / 27.0 / 30.9, at rank 16 20.2 / 25.3 / 22.1 / 21.5.  From about 7000 rows on slices of up to
// 4608 fill the chip without being split, and a launch of several projections has no use for more workgroups
// (8192 rows over 64 adapters, six projections at rank 64: 127 / 142 / 146 us); between 4096 and 8192 rows the line at
// 112 units (7105 rows) is not measured.  The units are those of full tile blocks; with many adapters there are more, and a
// split that just fills 256 workgroups runs over: 3200 rows over eight adapters, h_in = 11008 at rank 64, in five 51.7 us,
// in four 39.8 -- but 4096 rows over 64 adapters in four 67.8, in three 78.0, so the count has no margin.
// Never more slices than `most`, which what callers' scratch holds was sized for.  `solo`: the backward's products,
// whose fold leaves by-products behind and is wanted for that.
int block_pieces(int T, int d_in, int d_out, int most, bool solo) {
  const int P = ceil_div(d_in, 256), units = ceil_div(T > 0 ? T : 1, kTileRows * kBlkTiles);
  if (most > kMaxKsplit) most = kMaxKsplit;
  if (units >= 112 && !solo) {
    const int ks = ceil_div(P, 18);
    return ceil_div(P, ks < most ? ks : most);
  }
  int best = P;
  float least = 0.0f;
  for (int want = 1; want <= most && want <= P; ++want) {
    const int m = ceil_div(P, want), ks = ceil_div(P, m);
    const long wgs = (long)units * ks;
    if ((ks > 2 && wgs > 512) || (solo && ks == 1 && P > 1 && most > 1)) continue;
    const float cost = (wgs + 255) / 256 * (m + 0.3f) * (wgs <= 256 ? 1.12f : 1.0f) + (0.1f + d_out / 160.0f) * ks + (ks > 1 ? 3.0f : 0.0f);
    if (least == 0.0f || cost < least) least = cost, best = m;
  }
  return best;
}

// solo: the product is only ever launched by itself (the backward's dV and v products) and may take the
// splits that suit a launch of one projection; the forward's projections keep one rule
// whether they are launched alone or together, so that either way gives the same bits
// plain: a product of smlm_gemm or smlm_gemm_planned; drop: of x under dropout
ShrinkCfg shrink_cfg(int T, int d_in, int d_out, int nw, bool solo, int mt, bool plain = false, bool drop = false) {
  ShrinkCfg c;
  c.MT = mt;
  c.NB = d_out <= 16 ? 1 : (d_out <= 32 ? 2 : 4);  // (run_shrink may turn 4 into 8: shrink_wide)
  c.zblocks = ceil_div(d_out, 64);
  // 32-wide k steps per load batch (the tile-block kernel stages four per batch in LDS)
  c.U = c.MT > 1 ? 4 : (c.NB == 4 ? 2 : 4);
  // k of a load batch of one wave, the unit the split is made in.  (Tile blocks: four steps, also for 128 columns a
  // workgroup, whose batches are two: slices of 256 of k instead of 512 double the partial sums, past
  // smlm_gemm_static's scratch at 1024 rows and 128 columns.)  Above 64 columns the slices of a fused call come in
  // multiples of 64 of k, so that 11008 falls into 16 instead of 15: an even number keeps batches of more than 256
  // segments on the route that plans in the launch (896 rows in 298 segments at rank 256: 54.2 -> 42.6 us) and the
  // same slices of the weights on an XCD (in three segments: 43.2 -> 37.5).  Plain products keep the fewer partial
  // sums that smlm_gemm_static has room for.
  const int kq = c.MT > 1 ? 128 : 32 * c.U;
  c.NW = nw;
  const int units = ceil_div(T > 0 ? T : 1, kTileRows * c.MT);
  // k split over workgroups: enough of them to fill the chip, but every split writes and
  // re-reads an fp32 partial of the output (8*r bytes a row against 2*d_in of input), so
  // beyond 256 workgroups the split stops where the partials reach an eighth of the input.
  // Eight-wave workgroups (decode batches: few tiles) split k in four, which quadruples the
  // number of CUs at work; the expand kernel adds the four partials.
  // (A launch of one projection fills the chip twice over from 4096 rows on: 8192 rows at rank 64, h_in =
  // 4096, k in four instead of two: 27.6 -> 23.3 us; 4096 rows, h_in = 11008, in eight instead of five: 44.4
  // -> 35.6 us.  In a launch of several projections the same splits were 2-20 % slower: cfg5 180 -> 190 us.)
  int want = c.NW == kDecodeWaves ? kDecodeSplit : ceil_div(1024, units);
  const int cheap = d_in / (32 * d_out), fill = ceil_div((solo && c.MT > 1 && units >= 64) ? 512 : 256, units);
  const int cap = cheap > fill ? cheap : fill;
  if (want > cap) want = cap;
  int max_split = d_in / (c.NW * kq);
  if (max_split < 1) max_split = 1;
  if (max_split > kMaxKsplit) max_split = kMaxKsplit;
  const int ks = want < 1 ? 1 : (want > max_split ? max_split : want);
  if (block_shrink(c.MT, T, d_out, drop)) {
    c.k_per_wave = 64 * block_pieces(T, d_in, d_out, ks, solo);
    c.ksplit = ceil_div(d_in, c.NW * c.k_per_wave);
    return c;
  }
  // (the single-tile kernels' waves take a k range each: whole load batches a wave; a tile block's four
  // waves walk one slice together, which is cut to whole load batches, so its slices come out nearly equal:
  // k = 11008 in eight is seven slices of 1408 and one of 1152 instead of seven of 1536 and one of 256)
  const int step = c.MT == 1 ? kq : (d_out > 64 && !plain ? 64 : 128) / c.NW;
  c.k_per_wave = round_up(ceil_div(d_in, c.NW * ks), step);
  c.ksplit = ceil_div(d_in, c.NW * c.k_per_wave);
  // An odd split (h_in = 14336 falls into seven slices of 2048) gives way to an even one of equal slices that
  // still fills the chip twice: 8192 rows, h_in = 14336, k in four instead of seven: rank 16 61.6 -> 53.1 us,
  // rank 64 80.0 -> 67.8 us (six, eight, ten ... fourteen slices: 56-65 and 77-87 us).
  if (solo && c.MT > 1 && c.ksplit > 1 && (c.ksplit & 1) && d_in % (c.NW * kq) == 0) {
    const int pieces = d_in / (c.NW * kq);
    for (int e = c.ksplit - 1; e >= 2; --e)
      if (e % 2 == 0 && pieces % e == 0 && units * e >= 512) {
        c.k_per_wave = pieces / e * kq;
        c.ksplit = e;
        break;
      }
  }
  return c;
}

// Tile-block shrinks of more than 64 columns: 128 columns a workgroup, which then reads x once for them, instead of
// 64 -- when that leaves workgroups enough (`wgs`, of 128 columns, over all projections of the launch; a tile block per
// 64 rows and half a one per adapter).  The batches are two k steps then (four would take 70 KB of LDS, two workgroups
// a CU: 27.5 us instead of 20.7 in the first line).  The choice does not touch the order of any sum, so it may look at
// the segmentation.  64 / 128 columns, us (forward: the whole call; [k][n]: the product), workgroups in parentheses:
//   forward, 2064 rows, two projections 4096 -> 4096 at rank 128 (528): the shrink 25.5 / 20.7
//   forward at rank 128, 4096 -> 4096: 512 rows (72) 20.2 / 23.0, 1024 rows (144) 23.0 / 25.7, 2048 rows (288)
//     31.7 / 32.2, 3000 rows (306) 43.7 / 40.8; 11008 -> 4096: 512 rows (160) 25.5 / 27.8, 640 rows (192) 30.8 / 29.2,
//     1024 rows (320) 34.4 / 31.5, 512 decoded rows over 32 adapters (384) 47.8 / 38.2; q/k/v/o: 512 rows (320)
//     38.7 / 34.5
//   weights [k][n], 4096 -> 128: 16 rows (16) 10.3 / 13.8, 1024 rows (144) 14.4 / 17.5, 4096 rows (264) 22.6 / 24.6;
//     4096 -> 1024: 128 rows (256) 32.7 / 34.6, 512 rows (640) 41.2 / 39.4, 4096 rows (2112) 107.7 / 87.1
inline bool shrink_wide(int mt, int d_out, bool w_kn, long wgs) {
  return mt > 1 && d_out > 64 && (w_kn ? wgs > 300 : wgs >= 180);
}

// most k-split partials a shrink of this shape can leave behind, whichever wave count it runs with (`either`: and
// whichever of the tile-block shrinks)
int fwd_ksplit_bound(int T, int d_in, int d_out, bool plain = false, bool either = true) {
  const bool two = either && block_shrink(kBlkTiles, T, d_out);
  int most = shrink_cfg(T, d_in, d_out, kFwdWaves, false, 1, plain).ksplit;
  auto also = [&](int ks) { most = ks > most ? ks : most; };
  also(shrink_cfg(T, d_in, d_out, kDecodeWaves, false, 1, plain).ksplit);
  for (int solo = 0; solo < 2; ++solo) {
    also(shrink_cfg(T, d_in, d_out, kFwdWaves, solo != 0, kBlkTiles, plain).ksplit);
    if (two) also(shrink_cfg(T, d_in, d_out, kFwdWaves, solo != 0, kBlkTiles, plain, true).ksplit);
  }
  return most;
}

int expand_nq(int T, int d_out) {
  (void)T;
  // 32-column blocks per wave: four (a workgroup then covers 512 columns) unless the
  // projection is narrower than that
  return d_out >= 512 ? 4 : 2;
}

TileArgs tile_args(const PlanView& pv, int n_weights) {
  TileArgs t{pv.hdr, pv.tile_row, pv.tile_rseg, pv.tile_wid, pv.blk};
  t.n_weights = n_weights;  // 0: unknown
  return t;
}

// grid of a launch: (chunk row, tile unit, projection), or (chunk row over all projections,
// tile unit) when flat, in direct mode; else the persistent one-dimensional grid
inline dim3 item_grid(const ItemSpace& sp, long items) {
  if (!sp.units_max) return work_grid(items);
  if (sp.flat) return dim3((unsigned)sp.row_start[sp.nproj], (unsigned)sp.units_max, 1u);
  int rows = 1;
  for (int i = 0; i < sp.nproj; ++i)
    if (sp.row_start[i + 1] - sp.row_start[i] > rows) rows = sp.row_start[i + 1] - sp.row_start[i];
  return dim3((unsigned)rows, (unsigned)sp.units_max, (unsigned)sp.nproj);
}

template <int DT, int NW, bool DIRECT, bool DROP = false>
int launch_shrink_nb(int NB, dim3 grid, hipStream_t st, const ShrinkArgs& a) {
  const dim3 block(NW * kWaveSize);  // U must match shrink_cfg
  if (NB == 1) return launch(shrink_kernel<DT, 1, 4, NW, DIRECT, DROP>, grid, block, st, a);
  if (NB == 2) return launch(shrink_kernel<DT, 2, 4, NW, DIRECT, DROP>, grid, block, st, a);
  return launch(shrink_kernel<DT, 4, 2, NW, DIRECT, DROP>, grid, block, st, a);
}

template <int DT, bool DIRECT, bool WKN, bool DROP = false>
int launch_shrink_wide(int NB, dim3 grid, hipStream_t st, const ShrinkArgs& a) {
  const dim3 block(kFwdThreads);  // U must match run_shrink
  if (NB == 1) return launch(shrink_wide_kernel<DT, 1, 4, DIRECT, WKN, DROP>, grid, block, st, a);
  if (NB == 2) return launch(shrink_wide_kernel<DT, 2, 4, DIRECT, WKN, DROP>, grid, block, st, a);
  if (NB == 8) return launch(shrink_wide_kernel<DT, 8, 2, DIRECT, WKN, DROP>, grid, block, st, a);
  return launch(shrink_wide_kernel<DT, 4, 4, DIRECT, WKN, DROP>, grid, block, st, a);
}

template <int DT, bool WKN>
int launch_shrink_block(int NB, dim3 grid, hipStream_t st, const ShrinkArgs& a) {
  const dim3 block(kFwdThreads);
  if (NB == 1) return launch(shrink_block_kernel<DT, 1, WKN>, grid, block, st, a);
  if (NB == 2) return launch(shrink_block_kernel<DT, 2, WKN>, grid, block, st, a);
  return launch(shrink_block_kernel<DT, 4, WKN>, grid, block, st, a);
}

// Lists the chunk rows of a tile block are dealt out into, a workgroup (of four waves) each: what leaves the fewest
// rounds of chunk rows a CU, within one generation of resident workgroups where that costs nothing, and the most
// workgroups of those.  us, four / six / twelve lists, three projections of h_in = 4096 at rank 64, k in four: 4096 rows
// 36.5 / 42.6 / 35.9, 8192 rows 59.4 / 64.4 / 61.7.
// pairs: plans keyed by pairs of addresses, whose table has an entry per segment, so that it says little about how many
// tile blocks are partly filled (2100 rows of 64 adapters in 256 segments at rank 16: 32.4 us, counting 128 of them, 30.0).
int shrink_lists(int T, int S, int groups, int rows, bool pairs = false) {
  float partly = 0.5f * (groups > 0 && groups < S ? groups : S);  // filled tile blocks
  if (pairs && partly > 32) partly = 32;
  const float units = ceil_div(T, kTileRows * kBlkTiles) + partly;
  int best = rows;
  float least = units * rows / 256 + 0.4f;
  for (int lists = rows - 1; lists >= 1; --lists) {
    const float cost = (float)((int)(1.05f * units * lists / 256) + 1) * ceil_div(rows, lists);
    if (cost < least) least = cost, best = lists;
  }
  return best;
}

template <int DT, bool DIRECT>
int launch_shrink_dt(int NB, int MT, int NW, dim3 grid, hipStream_t st,
                     const ShrinkArgs& a) {
  if (a.drop.seg_p) {  // dropout of the training rows: x in the usual layout, weights [n][k]
    if (MT == 1)
      return NW == kDecodeWaves ? launch_shrink_nb<DT, kDecodeWaves, DIRECT, true>(NB, grid, st, a)
                                : launch_shrink_nb<DT, kFwdWaves, DIRECT, true>(NB, grid, st, a);
    return launch_shrink_wide<DT, DIRECT, false, true>(NB, grid, st, a);
  }
  if (MT == 1)
    return NW == kDecodeWaves ? launch_shrink_nb<DT, kDecodeWaves, DIRECT>(NB, grid, st, a)
                              : launch_shrink_nb<DT, kFwdWaves, DIRECT>(NB, grid, st, a);
  return a.w_kn ? launch_shrink_wide<DT, DIRECT, true>(NB, grid, st, a)
                : launch_shrink_wide<DT, DIRECT, false>(NB, grid, st, a);
}

template <int DT>
int launch_shrink_block_dt(int NB, dim3 grid, hipStream_t st, const ShrinkArgs& a) {
  return a.w_kn ? launch_shrink_block<DT, true>(NB, grid, st, a) : launch_shrink_block<DT, false>(NB, grid, st, a);
}

// all projections of one launch share NB / U / MT / NW (same rank, same T)
int launch_shrink(int dtype, const ShrinkCfg& c, int S, int groups, hipStream_t st,
                  ShrinkArgs& a) {
  const int MT = c.MT;
  a.items.interleave = 1;
  const int units = tile_units_max(a.T, S, groups, MT);
  const bool f16 = dtype == SMLM_DTYPE_F16;
  if (block_shrink(MT, a)) {
    a.items.units_max = units;
    const int y = units < kMaxGridY ? units : kMaxGridY;
    const dim3 grid((unsigned)shrink_lists(a.T, S, groups, a.items.row_start[a.items.nproj]), (unsigned)y,
                    (unsigned)ceil_div(units, y));
    return f16 ? launch_shrink_block_dt<SMLM_DTYPE_F16>(c.NB, grid, st, a)
               : launch_shrink_block_dt<SMLM_DTYPE_BF16>(c.NB, grid, st, a);
  }
  const long items = (long)units * a.items.row_start[a.items.nproj];
  a.items.units_max = (items <= kDirectItems && units <= kMaxGridY) ? units : 0;
  const dim3 grid = item_grid(a.items, items);
  if (a.items.units_max)
    return f16 ? launch_shrink_dt<SMLM_DTYPE_F16, true>(c.NB, MT, c.NW, grid, st, a)
               : launch_shrink_dt<SMLM_DTYPE_BF16, true>(c.NB, MT, c.NW, grid, st, a);
  return f16 ? launch_shrink_dt<SMLM_DTYPE_F16, false>(c.NB, MT, c.NW, grid, st, a)
             : launch_shrink_dt<SMLM_DTYPE_BF16, false>(c.NB, MT, c.NW, grid, st, a);
}

// Whether the single-tile shrinks that build their plan request x and the weights along the rows, at up to 32 columns.
// It pays where the segments are few: 4096 -> 4096, us, in the MFMA's layout / along the rows: one adapter in four
// segments at rank 32, 64 rows 11.4 / 10.8, 700 rows 14.4 / 13.6; three projections, eight segments, 500 rows at rank 16
// 18.0 / 17.2, at rank 32 22.9 / 21.1; 32 segments, 300 rows at rank 16 18.5 / 17.9; but 64 one-row segments 18.6 / 20.9,
// 1400 rows in 256 segments at rank 16, one projection, 19.8 / 21.0.  Keyed by pairs, whose finder holds more registers:
// one adapter in four segments, 300 rows at rank 32 13.2 / 12.5, 32 segments of 500 rows at rank 16 11.9 / 12.4, 192
// segments of 700 rows at rank 32 17.8 / 19.0.  Wider shrinks gain at every number of segments; two workgroups of sixteen
// waves fill a CU and lose (q/k/v/o of 900 decoded rows at rank 16 32.4 / 35.2).
inline bool shrink_lines(int S, bool pairs) { return S <= (pairs ? 8 : 32); }

template <int DT, int THREADS, bool PAIRS, bool DROP = false>
int launch_self_planned_nb(int NB, dim3 grid, hipStream_t st, const SelfPlanArgs& a) {
  const dim3 block(THREADS);  // U must match shrink_cfg
  constexpr bool kMay = THREADS == kSelfPlanThreads;
  if (kMay && NB <= 2 && shrink_lines(a.plan.S, PAIRS)) {
    if (NB == 1) return launch(shrink_self_planned_kernel<DT, 1, 4, THREADS, kMay, PAIRS, DROP>, grid, block, st, a);
    return launch(shrink_self_planned_kernel<DT, 2, 4, THREADS, kMay, PAIRS, DROP>, grid, block, st, a);
  }
  if (NB == 1) return launch(shrink_self_planned_kernel<DT, 1, 4, THREADS, false, PAIRS, DROP>, grid, block, st, a);
  if (NB == 2) return launch(shrink_self_planned_kernel<DT, 2, 4, THREADS, false, PAIRS, DROP>, grid, block, st, a);
  return launch(shrink_self_planned_kernel<DT, 4, 2, THREADS, kMay, PAIRS, DROP>, grid, block, st, a);
}

template <int DT, bool WKN, int THREADS, bool PAIRS, bool DROP = false>
int launch_self_planned_block_nb(int NB, dim3 grid, hipStream_t st, const SelfPlanArgs& a) {
  const dim3 block(THREADS);  // U must match shrink_cfg
  if constexpr (!DROP) {
    if (block_shrink(kBlkTiles, a.sh)) {
      if (NB == 1) return launch(shrink_block_self_planned_kernel<DT, 1, WKN, THREADS, PAIRS>, grid, block, st, a);
      if (NB == 2) return launch(shrink_block_self_planned_kernel<DT, 2, WKN, THREADS, PAIRS>, grid, block, st, a);
      return launch(shrink_block_self_planned_kernel<DT, 4, WKN, THREADS, PAIRS>, grid, block, st, a);
    }
  }
  if (NB == 1) return launch(shrink_wide_self_planned_kernel<DT, 1, 4, WKN, THREADS, PAIRS, DROP>, grid, block, st, a);
  if (NB == 2) return launch(shrink_wide_self_planned_kernel<DT, 2, 4, WKN, THREADS, PAIRS, DROP>, grid, block, st, a);
  if (NB == 8) return launch(shrink_wide_self_planned_kernel<DT, 8, 2, WKN, THREADS, PAIRS, DROP>, grid, block, st, a);
  return launch(shrink_wide_self_planned_kernel<DT, 4, 4, WKN, THREADS, PAIRS, DROP>, grid, block, st, a);
}
template <int DT, bool WKN, bool PAIRS, bool DROP = false>
int launch_self_planned_block(int NB, int S, dim3 grid, hipStream_t st, const SelfPlanArgs& a) {
  if (S <= kFwdThreads) return launch_self_planned_block_nb<DT, WKN, kFwdThreads, PAIRS, DROP>(NB, grid, st, a);
  // more segments than the four-wave workgroup has threads: two such groups a workgroup, each taking a list of chunk
  // rows or (the wide kernel) one of two neighbouring k slices (the caller has checked that the splits are even)
  grid.x = (grid.x + 1) / 2;
  return launch_self_planned_block_nb<DT, WKN, 2 * kFwdThreads, PAIRS, DROP>(NB, grid, st, a);
}

// batches this route takes: few enough segments for the plan-building workgroups of the launch
// (one segment per thread: 512 or 1024 in the decode shrink, 256 or 512 in the tile-block shrink),
// adapter ids that index a table of at most kSelfPlanWeights entries
bool self_planned_ok(int T, int S, int n_weights, int nt_max, int mt) {
  const int segs = mt > 1 ? (S <= kFwdThreads ? kFwdThreads : kSelfPlanBlkSegs)
                          : (S <= kSelfPlanThreads ? kSelfPlanThreads : kSelfPlanSegs);
  return S <= segs && nt_max <= 4 * segs && n_weights >= 1 && n_weights <= kSelfPlanWeights &&
         tile_units_max(T, S, n_weights, mt) < kMaxGridY;
}

template <int DT>
int launch_self_planned_dt(bool pairs, const ShrinkCfg& c, int S, dim3 grid, hipStream_t st, const SelfPlanArgs& sp) {
  const bool drop = sp.sh.drop.seg_p != nullptr;
  if (drop && (pairs || sp.sh.w_kn)) return SMLM_ERR_ARG;  // (no caller: their plans are built with a launch)
  if (c.MT == 1 && S > kSelfPlanThreads) {
    // more segments than the eight-wave workgroup has threads: workgroups of two such groups of
    // waves, each taking two neighbouring k slices (the caller has checked that the splits are even)
    grid.x = (grid.x + 1) / 2;
    if (drop) return launch_self_planned_nb<DT, 2 * kSelfPlanThreads, false, true>(c.NB, grid, st, sp);
    return pairs ? launch_self_planned_nb<DT, 2 * kSelfPlanThreads, true>(c.NB, grid, st, sp)
                 : launch_self_planned_nb<DT, 2 * kSelfPlanThreads, false>(c.NB, grid, st, sp);
  }
  if (c.MT > 1 && sp.sh.w_kn) return launch_self_planned_block<DT, true, false>(c.NB, S, grid, st, sp);
  if (c.MT > 1 && drop) return launch_self_planned_block<DT, false, false, true>(c.NB, S, grid, st, sp);
  if (c.MT > 1)
    return pairs ? launch_self_planned_block<DT, false, true>(c.NB, S, grid, st, sp)
                 : launch_self_planned_block<DT, false, false>(c.NB, S, grid, st, sp);
  if (drop) return launch_self_planned_nb<DT, kSelfPlanThreads, false, true>(c.NB, grid, st, sp);
  return pairs ? launch_self_planned_nb<DT, kSelfPlanThreads, true>(c.NB, grid, st, sp)
               : launch_self_planned_nb<DT, kSelfPlanThreads, false>(c.NB, grid, st, sp);
}

int launch_shrink_self_planned(int dtype, const ShrinkCfg& c, int S, int groups, const PlanSortArgs& build,
                               hipStream_t st, const ShrinkArgs& a) {
  if (c.MT == 1 && c.NW * kWaveSize != kSelfPlanThreads) return SMLM_ERR_ARG;
  if (c.MT > 1 && c.NW != kFwdWaves) return SMLM_ERR_ARG;
  SelfPlanArgs sp{};
  sp.sh = a;
  sp.plan = build;
  sp.n_weights = groups;
  // rows of workgroups: one per unit the batch can have.  Plans keyed by pairs of addresses (a table entry per
  // segment, so nearly all of those rows would find no unit) get no more than the batch's rows in whole units
  // plus 32 part-filled ones; their kernels take the units beyond that in further rounds.
  const bool pairs = build.key_kind == SMLM_KEY_PTR2;
  sp.units = tile_units_max(a.T, S, groups, c.MT);
  const int usual = a.T / (kTileRows * c.MT) + 1 + 32;
  if (pairs && sp.units > usual) sp.units = usual;
  if (pairs && a.w_kn) return SMLM_ERR_ARG;  // (no caller: the row-major products build their plan with a launch)
  int rows = 1;
  for (int i = 0; i < a.items.nproj; ++i)
    if (a.items.row_start[i + 1] - a.items.row_start[i] > rows) rows = a.items.row_start[i + 1] - a.items.row_start[i];
  dim3 grid((unsigned)rows, (unsigned)sp.units + 1u, (unsigned)a.items.nproj);
  if (block_shrink(c.MT, a)) {
    const int lists = shrink_lists(a.T, S, groups, a.items.row_start[a.items.nproj], pairs);
    sp.builder_rows = ceil_div(kSelfPlanBuilders, S <= kFwdThreads ? lists : ceil_div(lists, 2));
    grid = dim3((unsigned)lists, (unsigned)(sp.units + sp.builder_rows));
  }
  return dtype == SMLM_DTYPE_F16 ? launch_self_planned_dt<SMLM_DTYPE_F16>(pairs, c, S, grid, st, sp)
                                 : launch_self_planned_dt<SMLM_DTYPE_BF16>(pairs, c, S, grid, st, sp);
}

template <int DT>
int launch_side_fold(int ks, dim3 grid, hipStream_t st, const ReduceArgs& a) {
  if (ks <= 4) return launch(side_fold_kernel<DT, 4>, grid, dim3(kSideThreads), st, a);
  if (ks <= 8) return launch(side_fold_kernel<DT, 8>, grid, dim3(kSideThreads), st, a);
  return launch(side_fold_kernel<DT, kMaxKsplit>, grid, dim3(kSideThreads), st, a);
}
template <int DT>
int launch_reduce_rows(int ks, dim3 grid, hipStream_t st, const ReduceArgs& a) {
  if (ks <= 4) return launch(reduce_rows_kernel<DT, 4>, grid, dim3(256), st, a);
  if (ks <= 8) return launch(reduce_rows_kernel<DT, 8>, grid, dim3(256), st, a);
  return launch(reduce_rows_kernel<DT, kMaxKsplit>, grid, dim3(256), st, a);
}

int launch_reduce(int dtype, int S, int groups, hipStream_t st, ReduceArgs& a, bool side = false) {
  const bool f16 = dtype == SMLM_DTYPE_F16;
  int ks = 1;
  for (int i = 0; i < a.nproj; ++i) ks = a.p[i].ksplit > ks ? a.p[i].ksplit : ks;
  if (side) {  // by tile slot: the by-products are stored in slot order
    const int units = tile_units_max(a.T, S, groups, 1);
    const long items = (long)ceil_div(units, kBlkTiles) * ceil_div(a.d_out, 64) * a.nproj;
    a.units_max = items <= kDirectItems ? units : 0;
    const int zero_blocks = a.zero.n ? a.zero.first[a.zero.n] : 0, bit_blocks = a.bits.n ? a.bits.first[a.bits.n] : 0;
    if (!a.units_max) {  // (a launch that walks its items has no workgroups to spare)
      int rc = SMLM_OK;
      if (zero_blocks) rc = launch(zero_spans_kernel, dim3((unsigned)zero_blocks), dim3(256), st, a.zero);
      if (!rc && bit_blocks)
        rc = launch(tile_bits_kernel, dim3((unsigned)bit_blocks), dim3(256), st, TileBitsArgs{a.bits, a.plan.tile_row});
      if (rc) return rc;
    }
    const dim3 grid = a.units_max ? dim3((unsigned)(items + ceil_div(zero_blocks + bit_blocks, kBlkTiles))) : work_grid(items);
    return f16 ? launch_side_fold<SMLM_DTYPE_F16>(ks, grid, st, a) : launch_side_fold<SMLM_DTYPE_BF16>(ks, grid, st, a);
  }
  const long fours = ((long)a.T * (a.d_out / 4) + 255) / 256;
  if (!a.seg_scale && fours <= (1L << 23)) {  // no scale to look up: fold row by row
    const dim3 grid((unsigned)fours, (unsigned)a.nproj);
    return f16 ? launch_reduce_rows<SMLM_DTYPE_F16>(ks, grid, st, a) : launch_reduce_rows<SMLM_DTYPE_BF16>(ks, grid, st, a);
  }
  const int units = tile_units_max(a.T, S, groups, 1);
  const long items = (long)units * a.nproj;
  a.units_max = items <= kDirectItems ? units : 0;
  const dim3 grid = a.units_max ? dim3((unsigned)items) : work_grid(items);
  return f16 ? launch(reduce_kernel<SMLM_DTYPE_F16>, grid, dim3(256), st, a)
             : launch(reduce_kernel<SMLM_DTYPE_BF16>, grid, dim3(256), st, a);
}

template <int DT, int NQ, bool DIRECT>
int launch_expand_wave(int KS, bool vfold, dim3 grid, hipStream_t st, const ExpandArgs& a) {
  const dim3 block(kFwdThreads);
  if (vfold) {
    if (KS == 1) return launch(expand_wave_kernel<DT, NQ, 1, DIRECT, true>, grid, block, st, a);
    if (KS == 2) return launch(expand_wave_kernel<DT, NQ, 2, DIRECT, true>, grid, block, st, a);
    return launch(expand_wave_kernel<DT, NQ, 0, DIRECT, true>, grid, block, st, a);
  }
  if (KS == 1) return launch(expand_wave_kernel<DT, NQ, 1, DIRECT, false>, grid, block, st, a);
  if (KS == 2) return launch(expand_wave_kernel<DT, NQ, 2, DIRECT, false>, grid, block, st, a);
  return launch(expand_wave_kernel<DT, NQ, 0, DIRECT, false>, grid, block, st, a);
}

template <int DT, bool DIRECT>
int launch_expand_dt(bool block, int nq, int KS, dim3 grid, hipStream_t st,
                     const ExpandArgs& a) {
  if (a.drop.seg_p) {  // the backward's dX with the dropout of x undone: no fold
    const dim3 bl(kFwdThreads);  // (launch_expand admits only tile blocks with [k][n] weights here)
    if (KS == 4) return launch(expand_block_kernel<DT, 4, 4, DIRECT, true, true>, grid, bl, st, a);
    return KS == 1 ? launch(expand_block_kernel<DT, 4, 1, DIRECT, true, true>, grid, bl, st, a)
                   : launch(expand_block_kernel<DT, 4, 2, DIRECT, true, true>, grid, bl, st, a);
  }
  if (block && KS == 4)
    return a.w_kn ? launch(expand_block_kernel<DT, 4, 4, DIRECT, true>, grid, dim3(kFwdThreads), st, a)
                  : launch(expand_block_kernel<DT, 4, 4, DIRECT, false>, grid, dim3(kFwdThreads), st, a);
  if (block && a.w_kn)
    return KS == 1 ? launch(expand_block_kernel<DT, 4, 1, DIRECT, true>, grid, dim3(kFwdThreads), st, a)
                   : launch(expand_block_kernel<DT, 4, 2, DIRECT, true>, grid, dim3(kFwdThreads), st, a);
  if (block && nq == 8)
    return KS == 1 ? launch(expand_block_kernel<DT, 8, 1, DIRECT, false>, grid, dim3(kFwdThreads), st, a)
                   : launch(expand_block_kernel<DT, 8, 2, DIRECT, false>, grid, dim3(kFwdThreads), st, a);
  if (block)
    return KS == 1 ? launch(expand_block_kernel<DT, 4, 1, DIRECT, false>, grid, dim3(kFwdThreads), st, a)
                   : launch(expand_block_kernel<DT, 4, 2, DIRECT, false>, grid, dim3(kFwdThreads), st, a);
  const bool vfold = a.p[0].vsplit > 0;  // set for all projections of a launch or for none
  return nq == 4 ? launch_expand_wave<DT, 4, DIRECT>(KS, vfold, grid, st, a)
                 : launch_expand_wave<DT, 2, DIRECT>(KS, vfold, grid, st, a);
}

// the chunk rows of an expand launch, `chunk` columns each
void expand_rows(ExpandArgs& a, int nproj, int chunk) {
  a.items.nproj = nproj;
  a.items.interleave = 0;
  a.items.row_start[0] = 0;
  // Workgroups go to the XCDs in turn (workgroup number modulo eight, whatever the XCDs' load).  With an odd
  // number of chunk rows a tile unit, the workgroups of one column chunk visit all eight XCDs from unit to
  // unit and each L2 fetches that chunk of an adapter's weights for itself: a launch of one projection gets one
  // empty row then (8192 rows at rank 64: h_out = 11136, 87 chunks of 128 columns, 83.4 -> 73.3 us; h_out =
  // 11008, 43 chunks of 256, 87.8 -> 71.7 us).  Launches of several projections are left as they are: empty
  // workgroups there can fall on the same few XCDs in every unit and leave the others with all the work
  // (measured on the shrink launch of five and six projections: up to 2.2 x slower).
  for (int i = 0; i < nproj; ++i) {
    int rows = ceil_div(a.p[i].d_out, chunk);
    if (nproj == 1 && rows > 1 && (rows & 1)) rows += 1;
    a.items.row_start[i + 1] = a.items.row_start[i] + rows;
  }
}

// all projections of one launch share the rank (d_in); d_out may differ
int launch_expand(int dtype, int nq, int MT, int S, int groups, int nproj, int max_d_in,
                  hipStream_t st, ExpandArgs& a) {
  const bool block = MT > 1;  // tile blocks with the weights staged in LDS
  // (ranks above 64: 128 of k at a time on tile blocks, the general loop over k on single tiles)
  const int KS = max_d_in <= 32 ? 1 : (max_d_in <= 64 ? 2 : (block ? 4 : 0));
  if (a.drop.seg_p && !(block && a.w_kn)) return SMLM_ERR_ARG;
  if (a.w_kn && !block) return SMLM_ERR_ARG;  // (no caller: the single-tile kernel reads [n][k] weights)
  // Tile blocks: 128 columns a workgroup, or 256 where measured better (rank 64, 8192 rows: 5-13 % at every
  // width; a row stride that is a multiple of 4 KiB, e.g. h_out = 14336, from 4096 rows on at every rank:
  // the 64 rows of a tile block then meet in few HBM channels and pieces of 512 bytes spread them over
  // twice as many).  Elsewhere 256 columns lose 1-12 % (fewer workgroups a CU; h_out = 11008, the
  // backward's dX, whose weights lie [k][n]).
  if (block) {
    int wide = 0;
    for (int i = 0; i < nproj; ++i) wide = a.p[i].d_out > wide ? a.p[i].d_out : wide;
    const bool aligned = (wide * 2) % 4096 == 0;
    const bool wider = !a.w_kn && !a.drop.seg_p &&
                       ((KS == 2 && a.T >= 8192) || (aligned && wide >= 8192 && a.T >= 4096));
    nq = wider && KS <= 2 ? 8 : 4;
  }
  const int chunk = block ? 32 * nq : kFwdWaves * 32 * nq;  // columns per workgroup
  expand_rows(a, nproj, chunk);
  const int units = tile_units_max(a.T, S, groups, block ? kBlkTiles : 1);
  const long items = (long)units * a.items.row_start[nproj];
  bool same_rows = true;
  for (int i = 1; i < nproj; ++i)
    same_rows = same_rows && (a.items.row_start[i + 1] - a.items.row_start[i] == a.items.row_start[1]);
  a.items.flat = same_rows ? 0 : 1;
  a.items.units_max = (items <= kDirectItems && units <= kMaxGridY) ? units : 0;
  const dim3 grid = item_grid(a.items, items);
  const bool f16 = dtype == SMLM_DTYPE_F16;
  if (a.items.units_max)
    return f16 ? launch_expand_dt<SMLM_DTYPE_F16, true>(block, nq, KS, grid, st, a)
               : launch_expand_dt<SMLM_DTYPE_BF16, true>(block, nq, KS, grid, st, a);
  return f16 ? launch_expand_dt<SMLM_DTYPE_F16, false>(block, nq, KS, grid, st, a)
             : launch_expand_dt<SMLM_DTYPE_BF16, false>(block, nq, KS, grid, st, a);
}

int check_common(int T, int S, int dtype) {
  if (T < 0 || S < 0) return SMLM_ERR_ARG;
  if (dtype != SMLM_DTYPE_F16 && dtype != SMLM_DTYPE_BF16) return SMLM_ERR_DTYPE;
  if (S >= kMaxSegments || T > (1 << 30)) return SMLM_ERR_LIMIT;
  return SMLM_OK;
}

int plan_build_impl(const PlanView& pv, const int32_t* seg_indptr, const void* seg_key,
                    int key_kind, int S, hipStream_t st, const void* seg_key2 = nullptr) {
  const int N = next_pow2(S);
  const PlanSortArgs sa{pv, seg_indptr, seg_key, key_kind, S, N, seg_key2};
  if (S <= kPlanSmallSegs && pv.nt_max <= kPlanSmallTiles)
    return launch(plan_small_kernel, dim3(1), dim3(kPlanThreads), st, sa);
  int rc = (N <= kPlanLdsKeys)
               ? launch(plan_sort_kernel<true>, dim3(1), dim3(kPlanThreads), st, sa)
               : launch(plan_sort_kernel<false>, dim3(1), dim3(kPlanThreads), st, sa);
  if (rc) return rc;
  const long slots = (long)pv.nt_max * kTileRows;
  const PlanFillArgs fa{pv, seg_indptr, S};
  return launch(plan_fill_kernel, dim3((unsigned)((slots + 255) / 256)), dim3(256), st, fa);
}

// shrink of one or more projections that share row routing and output width:
// out[i] = beta*out[i] + scale * x[i] W_i^T in 16 bits, via k-split fp32 partial
// sums folded by a second launch when the split is wider than one workgroup
// (fold = false leaves every projection's fp32 partials, one or more, for the consumer to fold)
// by-products a fold may leave behind (ReduceProj::pt_a ...)
struct SideOut {
  uint16_t* pt_a[kMaxProj];
  uint16_t* pt_b[kMaxProj];
  const uint16_t* v2[kMaxProj];
  const float* scale;
  ZeroSpans zero;  // memory the fold's launch is to clear as well (n = 0: none)
  TileBits bits;   // keep bits it is to turn (n = 0: none)
};

int run_shrink(int dtype, const PlanView& pv, int T, int S, int groups, int nproj,
               const void* const* x, const void* const* const* w_ptrs, float* const* partial,
               void* const* out, const int* d_in, int d_out, const int* ldw, float beta,
               const float* seg_scale, int mt, hipStream_t st, bool fold = true, bool w_kn = false,
               const DropArgs* drop = nullptr, const int32_t* w_rank = nullptr, int packed = 0,
               const PlanSortArgs* build = nullptr, bool solo = false, const SideOut* side = nullptr,
               bool* side_done = nullptr, bool plain = false) {
  if (drop && drop->seg_p && w_kn) return SMLM_ERR_ARG;
  if (side_done) *side_done = false;
  ShrinkArgs a{};
  if (drop) a.drop = *drop;
  a.w_kn = w_kn ? 1 : 0;
  a.plan = tile_args(pv, groups);
  a.plan.w_rank = w_rank;  // the output columns are the rank
  a.plan.packed = packed;
  a.seg_scale = seg_scale;
  a.beta = beta;
  a.T = T;
  a.items.nproj = nproj;
  a.items.row_start[0] = 0;
  ReduceArgs ra{};
  bool need_reduce = false, all_reduce = true;
  ShrinkCfg c0{};
  size_t bits_off = 0;
  const int nw = shrink_waves(mt, nproj, d_in, d_out);
  const bool dropped = drop && drop->seg_p;
  long wgs = 0;  // workgroups of 128 columns
  for (int i = 0; mt > 1 && d_out > 64 && i < nproj; ++i)
    wgs += (long)(ceil_div(T, kTileRows * mt) + (groups > 0 && groups < S ? groups : S) / 2) *
           shrink_cfg(T, d_in[i], d_out, nw, solo, mt, plain, dropped).ksplit *
           ceil_div(d_out, 128);
  const bool wide = shrink_wide(mt, d_out, w_kn, wgs);
  for (int i = 0; i < nproj; ++i) {
    ShrinkCfg c = shrink_cfg(T, d_in[i], d_out, nw, solo, mt, plain, dropped);
    if (wide) c.NB = 8, c.U = 2, c.zblocks = ceil_div(d_out, 128);
    if (i == 0) c0 = c;
    ShrinkProj& P = a.p[i];
    P.x = reinterpret_cast<const uint16_t*>(x[i]);
    P.w_ptrs = w_ptrs[i];
    P.partial = partial[i];
    P.out = reinterpret_cast<uint16_t*>(out[i]);
    P.d_in = d_in[i]; P.d_out = d_out; P.ldw = ldw[i];
    P.k_per_wave = c.k_per_wave; P.ksplit = c.ksplit; P.zblocks = c.zblocks;
    P.to_partial = fold ? 0 : 1;
    if (drop && drop->bits) {  // projections' masks lie end to end
      P.drop_bits = drop->bits + bits_off;
      bits_off += (size_t)drop->rows * (d_in[i] / 8);
    }
    // (a launch of one projection with an odd number of chunk rows a tile unit gets one empty row, as the
    // expand launch does and for its reason: 8192 rows at rank 64, h_in = 11008, k split in five: 75.5 ->
    // 59.6 us; 6144 rows, h_in = 4096, in three: 27.2 -> 25.0; launches of several projections and those that
    // build their plan keep their grid)
    int rows = c.ksplit * c.zblocks;
    if (nproj == 1 && !build && !block_shrink(mt, T, d_out, dropped) && rows > 1 && (rows & 1)) rows += 1;
    a.items.row_start[i + 1] = a.items.row_start[i] + rows;
    ra.p[i] = ReduceProj{partial[i], P.out, c.ksplit, side ? side->pt_a[i] : nullptr, side ? side->pt_b[i] : nullptr,
                         side ? side->v2[i] : nullptr};
    need_reduce = need_reduce || c.ksplit > 1;
    all_reduce = all_reduce && c.ksplit > 1;
  }
  // Folding the k-split partials inside the shrink launch (last-arriving workgroup, ticket
  // counters) was measured and dropped: the device-scope release/acquire it needs writes back
  // and invalidates a whole L2 per workgroup on this multi-XCD part and cost 5-10x the launch
  // it saves.
  // `build`: the plan does not exist yet -- the decode shrink whose workgroups find their
  // own tile, with one more workgroup that builds the plan (the caller has checked the limits)
  int rc = build ? launch_shrink_self_planned(dtype, c0, S, groups, *build, st, a)
                 : launch_shrink(dtype, c0, S, groups, st, a);
  if (rc || !need_reduce || !fold) return rc;
  ra.plan = a.plan;
  ra.seg_scale = seg_scale;
  ra.beta = beta;
  ra.T = T; ra.d_out = d_out; ra.nproj = nproj;
  // the by-products go with the fold when every projection is folded (else they are left to the caller)
  const bool with_side = side && all_reduce;
  if (with_side) {
    ra.side_scale = side->scale;
    ra.zero = side->zero;
    ra.bits = side->bits;
  }
  if (side_done) *side_done = with_side;
  return launch_reduce(dtype, S, groups, st, ra, with_side);
}

template <int DT, bool DROP>
int launch_wgrad(int nbj, bool split, dim3 grid, hipStream_t st, const WgradArgs& wa) {
  const dim3 bl(split ? 256 : 64);
  if (wa.zcount > 1)  // several workgroups along the rank: NBJ = 4
    return split ? launch(wgrad_kernel<DT, 4, 4, DROP, true>, grid, bl, st, wa)
                 : launch(wgrad_kernel<DT, 4, 1, DROP, true>, grid, bl, st, wa);
  if (split) {
    if (nbj == 1) return launch(wgrad_kernel<DT, 1, 4, DROP, false>, grid, bl, st, wa);
    if (nbj == 2) return launch(wgrad_kernel<DT, 2, 4, DROP, false>, grid, bl, st, wa);
    return launch(wgrad_kernel<DT, 4, 4, DROP, false>, grid, bl, st, wa);
  }
  if (nbj == 1) return launch(wgrad_kernel<DT, 1, 1, DROP, false>, grid, bl, st, wa);
  if (nbj == 2) return launch(wgrad_kernel<DT, 2, 1, DROP, false>, grid, bl, st, wa);
  return launch(wgrad_kernel<DT, 4, 1, DROP, false>, grid, bl, st, wa);
}

template <int DT, bool DROP, int NW>
int launch_bwd_tail(int nbj, dim3 grid, hipStream_t st, const BwdTailArgs& a) {
  const dim3 bl(kFwdThreads);
  if (a.e.p[0].d_in > 64) return launch(bwd_tail_kernel<DT, 4, NW, DROP, true, 4>, grid, bl, st, a);
  if (nbj == 1) return launch(bwd_tail_kernel<DT, 1, NW, DROP, false, 1>, grid, bl, st, a);
  if (nbj == 2) return launch(bwd_tail_kernel<DT, 2, NW, DROP, false, 1>, grid, bl, st, a);
  return launch(bwd_tail_kernel<DT, 4, NW, DROP, false, 2>, grid, bl, st, a);
}
template <int DT>
int launch_bwd_tail_dt(int nbj, bool split, dim3 grid, hipStream_t st, const BwdTailArgs& a) {
  if (a.w.drop.seg_p)
    return split ? launch_bwd_tail<DT, true, 4>(nbj, grid, st, a) : launch_bwd_tail<DT, true, 1>(nbj, grid, st, a);
  return split ? launch_bwd_tail<DT, false, 4>(nbj, grid, st, a) : launch_bwd_tail<DT, false, 1>(nbj, grid, st, a);
}

// Whether the weight gradients' workgroups are four waves that share an adapter's rows, or one: from how many rows an
// adapter on.  Four waves take a quarter of the steps but fill a CU sooner (their registers: four workgroups at ranks up
// to 16, three up to 32, two above, fewer under dropout), so the line rises with the workgroups, one an adapter (and 64
// ranks) for each 64 columns.  us, one wave / four, two projections 4096 -> 4096 (256 such pieces): one adapter at rank
// 16, 128 rows 7.3 / 6.8, 512 rows 14.3 / 8.7, 1024 rows 24.4 / 12.3; two of 256 rows 10.2 / 8.6, at rank 32 10.7 / 9.4,
// at rank 64 12.0 / 10.9, at rank 128 13.1 / 16.1; four of 512 rows at rank 32 22.0 / 21.7, at rank 128 24.2 / 34.8; eight
// of 512 rows at rank 16 30.9 / 31.4, at rank 32 32.6 / 36.3; sixteen of 512 at rank 128 113 / 132.
// It ends at 512 rows: the rule is given the average, and an adapter of several times that, alone in a wave, is what the
// launch waits for.  Equal adapters, then the longest four (eight) times the average: eight of 768 rows at rank 64, one
// projection, 31.7 / 31.2 and 81.8 / 33.4; sixteen of 1024 at rank 32 61.3 / 64.0 and 114 / 66.7 (190 / 77.0), at rank 128
// 109 / 115 and 142 / 119 (234 / 120), two projections 202 / 214 and 203 / 223 (281 / 234).
// Under dropout four waves pay sooner, and with adapters of unequal rows sooner still.  One projection, then two: four
// adapters of 256 rows at rank 16 13.2 / 9.5 and 15.1 / 14.6, at rank 64 15.4 / 12.4 and 18.1 / 19.7; eight of 384 at rank
// 16 20.6 / 19.4 and 27.3 / 29.6, at rank 64 24.3 / 25.1 and 32.9 / 42.8, the longest six times the shortest 38.7 / 24.3
// and 43.6 / 42.5; at rank 128, where 64 ranks are a workgroup, 27.5 / 37.4 and 52.5 / 73.6, unequal 38.7 / 37.8 and 52.6 /
// 74.4, so up to 512 rows the line goes on rising there.
// A launch of several projections has more pieces and would change over later, of one sooner (four adapters of 384 rows at
// rank 32: one 14.4 / 10.8, two 18.2 / 19.0; two of 300 rows at rank 64: one 12.5 / 9.4, four 17.4 / 20.2); the rule does
// not look at their number, so that it gives the bits that launches of one give.
bool wgrad_split(int rows, int NA, int r, bool drop) {
  const long m = (long)NA * ceil_div(r, 64);
  auto least = [](long a, long b) { return a < b ? a : b; };
  auto most = [](long a, long b) { return a > b ? a : b; };
  long line;
  if (r <= 16) line = drop ? least(48 * m, 256) : 48 * m;
  else if (r <= 32) line = drop ? 64 * m : 96 * m;
  else line = drop ? (r <= 64 ? least(64 * m, 256) : 64 * m) : 128 * m;
  return rows >= most(r > 32 && !drop ? 192 : 128, least(line, 512));
}

// Whether dX and the weight gradients (`waves`: their workgroups, of one wave or four) go out in one launch: while what
// they move takes little longer than starting and draining two.  Together they hold as many registers and as much LDS as
// the weight gradients, so fewer of dX's workgroups are resident, which costs where both run at the memory's rate.  Same
// bits.  us, whole backward, two launches / one, h_in = h_out = 4096, operands from memory (700 MB of them in turn; the
// numbers in parentheses: MB of x, dY and dX, then of the weights):
//   up to rank 64, by the bytes of both: two adapters of 1024 rows at rank 16, two projections (101 + 2) 40.6 / 38.3, one of
//     646 at rank 32, six (95 + 5) 45.1 / 42.3; sixteen of 128 at rank 32, two (101 + 25) 46.6 / 47.6, four of 512 at rank
//     64, two (101 + 13) 52.4 / 53.1
//   ... and where they are workgroups of one wave, by their number (3072 are resident at rank 16, 2048 above; dX's own
//     kernel keeps five or six waves a SIMD, here three or two): at rank 16 4096 26.4 / 23.9, 16384 47.1 / 48.6; at rank 32
//     3584 28.2 / 27.9, 4096 28.5 / 29.6, 32768 113 / 132; at rank 64 4096 of few rows 34.2 / 34.7, of 64 rows and the
//     longest of eight times that 50.0 / 47.7; under dropout 4096 at rank 32 48.2 / 48.4, at rank 64 48.0 / 43.8
//   above rank 64, where dX's own kernel keeps no more than three waves a SIMD, by the rows alone: one adapter of 1024 rows
//     at rank 128 (25 + 3) 36.3 / 31.4, two, two projections (101 + 13) 76.3 / 72.6, 64 of 32 rows, two (101 + 403, 32768
//     workgroups) 173 / 169, unequal ones alike (sixteen averaging 128 rows, the longest eight times that 75.1 / 66.6);
//     sixteen of 512 rows (201 + 50) 141 / 144, 64 of 128 (201 + 201) 158 / 163
//   under dropout dX and the gradients have more to do between their loads: two of 1377 rows, two projections at rank 16
//     (135 + 2) 56.0 / 52.5, at rank 32 62.6 / 63.0, eight of 1000 at rank 32 (197 + 6) 76.2 / 80.6; sixteen of 128, two at
//     rank 128 (101 + 101) 99.2 / 92.2, 32 of 96 (151 + 201) 168 / 176
bool bwd_one_launch(int n_proj, int n_rows, int NA, int r, const int* h_in, const int* h_out, bool drop, bool split,
                    long waves) {
  double rows = 0, weights = 0;  // bytes
  for (int i = 0; i < n_proj; ++i) {
    rows += 2.0 * n_rows * (2.0 * h_in[i] + h_out[i]);
    weights += 2.0 * NA * r * (2.0 * h_in[i] + h_out[i]);
  }
  if (r > 64) return rows < 200e6 && (!drop || rows + weights < 330e6);
  return (split || waves <= (drop || r <= 16 || r > 32 ? 4096 : 3584)) && rows + weights < (drop ? 140e6 : 105e6);
}

struct BwdProjLayout {
  size_t partial, dv16, v16, pt_a, pt_b, bits;
};
struct BwdLayout {
  BwdProjLayout p[kMaxProj];
  size_t total;
};

// the projections' areas lie end to end, each laid out as a backward of that projection alone
BwdLayout bwd_layout(int n_proj, int n_rows, int P, int NA, const int* h_in, const int* h_out, int r) {
  BwdLayout L;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    size_t o = off;
    off = align_up(off + bytes, 256);
    return o;
  };
  const size_t slots = (size_t)plan_nt_max(n_rows, P) * kTileRows;
  for (int i = 0; i < n_proj; ++i) {
    BwdProjLayout& Q = L.p[i];
    const int ks_dv = fwd_ksplit_bound(n_rows, h_out[i], r), ks_v = fwd_ksplit_bound(n_rows, h_in[i], r);
    const int ks = ks_dv > ks_v ? ks_dv : ks_v;
    Q.partial = take((size_t)ks * n_rows * r * 4);
    Q.dv16 = take((size_t)n_rows * r * 2);
    Q.v16 = take((size_t)n_rows * r * 2);
    Q.pt_a = take(r * slots * 2);
    Q.pt_b = take(r * slots * 2);
    Q.bits = take(slots * ceil_div(h_in[i], 64) * 8);  // keep bits of x's dropout mask, by tile slot
  }
  L.total = off;
  return L;
}

template <int DT>
int launch_expand_found_dt(int nq, int KS, dim3 grid, hipStream_t st, const FoundExpandArgs& a) {
  const dim3 block(kFwdThreads);
  if (nq == 4) {
    if (KS == 1) return launch(expand_found_kernel<DT, 4, 1>, grid, block, st, a);
    if (KS == 2) return launch(expand_found_kernel<DT, 4, 2>, grid, block, st, a);
    return launch(expand_found_kernel<DT, 4, 0>, grid, block, st, a);
  }
  if (KS == 1) return launch(expand_found_kernel<DT, 2, 1>, grid, block, st, a);
  if (KS == 2) return launch(expand_found_kernel<DT, 2, 2>, grid, block, st, a);
  return launch(expand_found_kernel<DT, 2, 0>, grid, block, st, a);
}
int launch_expand_found(int dtype, int T, int S, hipStream_t st, FoundExpandArgs& a) {
  const int nq = expand_nq(T, a.p.d_out);
  const int KS = a.p.d_in <= 32 ? 1 : (a.p.d_in <= 64 ? 2 : 0);
  a.chunks = ceil_div(a.p.d_out, kFwdWaves * 32 * nq);
  const long items = (long)tile_units_max(T, S, S, 1) * a.chunks, wgs = 256 * found_wgs(nq, KS);
  a.lists = items <= wgs ? a.chunks : 0;  // (a workgroup for every chunk there can be)
  const dim3 grid((unsigned)(items < wgs ? items : wgs));
  return dtype == SMLM_DTYPE_F16 ? launch_expand_found_dt<SMLM_DTYPE_F16>(nq, KS, grid, st, a)
                                 : launch_expand_found_dt<SMLM_DTYPE_BF16>(nq, KS, grid, st, a);
}

// Scratch of smlm_gemm_static: part of the code object, so every device the library is loaded
// on has its own copy at its own address.  In host code the name is only a handle for
// hipGetSymbolAddress; kernels and copies get the looked-up device address.
constexpr int kMaxDevices = 64;
std::atomic<void*> scratch_addr[kMaxDevices];

// device address of `scratch` on the current device (looked up once per device), or null
void* static_scratch() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  void* p = scratch_addr[dev].load(std::memory_order_acquire);
  if (!p) {
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
    scratch_addr[dev].store(p, std::memory_order_release);  // every thread finds the same address
  }
  return p;
}

// Columns a workgroup of the RMSNorm backward's fold takes: 16 where a row is short, so that its workgroups fill the
// chip; of wider rows 32 and 64, as the pieces of 64 bytes that 16 columns read of every partial row fetch the lines
// twice.  Whole backward, us, 16 / 32 / 64 columns: 4096 x 2048 16.9 / 16.9 / -, 1000 x 4096 12.4 / 11.0 / -,
// 1000 x 8192 21.8 / 18.8 / 18.6, 1000 x 11008 28.7 / 25.1 / 24.8, 64 x 20480 16.9 / - / 14.5.
template <int DT>
int launch_rms_fold(hipStream_t st, const RmsFoldArgs& a) {
  const dim3 bl(256);
  if (a.cols <= 2048) return launch(rms_fold_kernel<DT, 4>, dim3((unsigned)ceil_div(a.cols, 16)), bl, st, a);
  if (a.cols <= 4096) return launch(rms_fold_kernel<DT, 8>, dim3((unsigned)ceil_div(a.cols, 32)), bl, st, a);
  return launch(rms_fold_kernel<DT, 16>, dim3((unsigned)ceil_div(a.cols, 64)), bl, st, a);
}

}  // namespace

extern "C" {

SMLM_API int smlm_abi_version(void) { return SMLM_ABI_VERSION; }

SMLM_API const char* smlm_strerror(int code) {
  switch (code) {
    case SMLM_OK: return "ok";
    case SMLM_ERR_ARG: return "invalid argument";
    case SMLM_ERR_DTYPE: return "No suitable kernel.";
    case SMLM_ERR_ALIGN: return "dimension not a multiple of 8 or pointer not 16-byte aligned";
    case SMLM_ERR_WORKSPACE: return "workspace too small";
    case SMLM_ERR_LAUNCH: return "kernel launch failed";
    case SMLM_ERR_LIMIT: return "size beyond the supported range";
    case SMLM_ERR_SCRATCH: return "the call needs more scratch than the library's static array holds";
    default: return "unknown error";
  }
}

SMLM_API int smlm_tmp_size(int num_problems, size_t* bytes) {
  if (num_problems < 0 || !bytes) return SMLM_ERR_ARG;
  *bytes = (size_t)64 * (size_t)num_problems;
  return SMLM_OK;
}

SMLM_API int smlm_plan_size(int T, int S, size_t* bytes) {
  if (T < 0 || S < 0 || !bytes) return SMLM_ERR_ARG;
  if (S >= kMaxSegments || T > (1 << 30)) return SMLM_ERR_LIMIT;
  *bytes = plan_carve(nullptr, T, S, nullptr);
  return SMLM_OK;
}

SMLM_API int smlm_plan_build(void* plan, size_t plan_bytes, const int32_t* seg_indptr,
                             const void* seg_key, int key_kind, int T, int S, void* stream) {
  if (T < 0 || S < 0) return SMLM_ERR_ARG;
  if (S >= kMaxSegments || T > (1 << 30)) return SMLM_ERR_LIMIT;
  if (key_kind != SMLM_KEY_NONE && key_kind != SMLM_KEY_I32 && key_kind != SMLM_KEY_PTR)
    return SMLM_ERR_ARG;
  if (S == 0) return SMLM_OK;
  if (!plan || !seg_indptr || (key_kind != SMLM_KEY_NONE && !seg_key)) return SMLM_ERR_ARG;
  if (!aligned16(plan)) return SMLM_ERR_ALIGN;
  PlanView pv;
  if (plan_carve(plan, T, S, &pv) > plan_bytes) return SMLM_ERR_WORKSPACE;
  return plan_build_impl(pv, seg_indptr, seg_key, key_kind, S, (hipStream_t)stream);
}

SMLM_API int smlm_plan_build2(void* plan, size_t plan_bytes, const int32_t* seg_indptr,
                              const void* const* seg_key_a, const void* const* seg_key_b, int T, int S,
                              void* stream) {
  if (T < 0 || S < 0) return SMLM_ERR_ARG;
  if (S >= kMaxSegments || T > (1 << 30)) return SMLM_ERR_LIMIT;
  if (S == 0) return SMLM_OK;
  if (!plan || !seg_indptr || !seg_key_a || !seg_key_b) return SMLM_ERR_ARG;
  if (!aligned16(plan)) return SMLM_ERR_ALIGN;
  PlanView pv;
  if (plan_carve(plan, T, S, &pv) > plan_bytes) return SMLM_ERR_WORKSPACE;
  return plan_build_impl(pv, seg_indptr, seg_key_a, SMLM_KEY_PTR2, S, (hipStream_t)stream, seg_key_b);
}

// Scratch of one product: what it uses, or (`asked`) what the queries say.  They count both tile-block shrinks: from the
// row number on at which the block kernel takes over, with fewer slices, a size would otherwise fall to less than half,
// below what fewer rows use, and a buffer sized for the largest batch alone would be refused for a smaller one.
static size_t gemm_scratch(int T, int d_in, int d_out, bool asked) {
  const int ks = d_in >= d_out ? fwd_ksplit_bound(T, d_in, d_out, true, asked) : 1;
  return ks > 1 ? align_up((size_t)ks * T * d_out * 4, 256) : 256;
}

SMLM_API int smlm_gemm_planned_workspace_size(int T, int d_in, int d_out, size_t* bytes) {
  if (T < 0 || d_in <= 0 || d_out <= 0 || !bytes) return SMLM_ERR_ARG;
  if (T > (1 << 30)) return SMLM_ERR_LIMIT;
  *bytes = gemm_scratch(T, d_in, d_out, true);
  return SMLM_OK;
}

SMLM_API int smlm_gemm_planned(void* y, const void* x, const void* const* w_ptrs, int n_weights,
                               const void* plan, void* workspace, size_t workspace_bytes, int T,
                               int S, int d_in, int d_out, int w_ld, int w_row_major, int dtype,
                               float beta, const float* seg_scale, void* stream) {
  int rc = check_common(T, S, dtype);
  if (rc) return rc;
  if (d_in <= 0 || d_out <= 0 || w_ld <= 0) return SMLM_ERR_ARG;
  if ((d_in & 7) || (d_out & 7) || (w_ld & 7)) return SMLM_ERR_ALIGN;
  if (w_ld < (w_row_major ? d_out : d_in)) return SMLM_ERR_ARG;
  if (T == 0 || S == 0) return SMLM_OK;
  if (!y || !x || !w_ptrs || !plan || !workspace) return SMLM_ERR_ARG;
  if (!aligned16(y) || !aligned16(x) || !aligned16(workspace) || !aligned16(plan))
    return SMLM_ERR_ALIGN;
  if (workspace_bytes < gemm_scratch(T, d_in, d_out, false)) return SMLM_ERR_WORKSPACE;

  hipStream_t st = (hipStream_t)stream;
  PlanView pv;
  plan_carve(const_cast<void*>(plan), T, S, &pv);

  if (d_in < d_out) {  // the reference's "expand" branch (smlm_forward_cutlass.cuh:82)
    ExpandArgs a{};
    a.plan = tile_args(pv, n_weights);
    a.seg_scale = seg_scale;
    a.beta = beta;
    a.T = T; a.nt_max = pv.nt_max;
    ExpandProj& P = a.p[0];
    P.y = reinterpret_cast<uint16_t*>(y);
    P.v = reinterpret_cast<const uint16_t*>(x);
    P.w_ptrs = w_ptrs;
    P.d_in = d_in; P.d_out = d_out; P.ldw = w_ld;
    // Row-major weights (element (k, n) at w[k * w_ld + n]) are the [k][n] layout the tile-block kernels read
    // as it lies (as the backward's dX = dV A does): they run at every size, as they do for the backward.
    if (w_row_major) {
      a.w_kn = 1;
      return launch_expand(dtype, expand_nq(T, d_out), kBlkTiles, S, n_weights, 1, d_in, st, a);
    }
    return launch_expand(dtype, expand_nq(T, d_out), tiles_per_wave(T, d_in, kNoShrink), S, n_weights,
                         1, d_in, st, a);
  }
  float* partial = reinterpret_cast<float*>(workspace);
  if (w_row_major)  // the tile-block shrink stages [k][n] weights as they lie (as the backward's dV = dY B does)
    return run_shrink(dtype, pv, T, S, n_weights, 1, &x, &w_ptrs, &partial, &y, &d_in, d_out, &w_ld, beta,
                      seg_scale, kBlkTiles, st, true, true, nullptr, nullptr, 0, nullptr, false, nullptr, nullptr, true);
  return run_shrink(dtype, pv, T, S, n_weights, 1, &x, &w_ptrs, &partial, &y, &d_in,
                    d_out, &w_ld, beta, seg_scale, tiles_per_wave(T, d_out, d_in), st, true, false, nullptr, nullptr, 0,
                    nullptr, false, nullptr, nullptr, true);
}

SMLM_API int smlm_gemm_workspace_size(int T, int S, int d_in, int d_out, size_t* bytes) {
  if (T < 0 || S < 0 || d_in <= 0 || d_out <= 0 || !bytes) return SMLM_ERR_ARG;
  if (S >= kMaxSegments || T > (1 << 30)) return SMLM_ERR_LIMIT;
  size_t extra = 0;
  int rc = smlm_gemm_planned_workspace_size(T, d_in, d_out, &extra);
  if (rc) return rc;
  *bytes = plan_carve(nullptr, T, S, nullptr) + extra;
  return SMLM_OK;
}

SMLM_API int smlm_gemm(void* y, const void* x, const void* const* w_ptrs, const int32_t* seg_indptr,
                       void* workspace, size_t workspace_bytes, int T, int S, int d_in, int d_out,
                       int w_ld, int w_row_major, int dtype, float beta, const float* seg_scale,
                       void* stream) {
  int rc = check_common(T, S, dtype);
  if (rc) return rc;
  if (d_in <= 0 || d_out <= 0 || w_ld <= 0) return SMLM_ERR_ARG;
  if ((d_in & 7) || (d_out & 7) || (w_ld & 7)) return SMLM_ERR_ALIGN;
  if (w_ld < (w_row_major ? d_out : d_in)) return SMLM_ERR_ARG;
  if (T == 0 || S == 0) return SMLM_OK;
  if (!y || !x || !w_ptrs || !seg_indptr || !workspace) return SMLM_ERR_ARG;
  if (!aligned16(y) || !aligned16(x) || !aligned16(workspace)) return SMLM_ERR_ALIGN;
  PlanView pv;
  const size_t plan_bytes = plan_carve(workspace, T, S, &pv);
  if (workspace_bytes < plan_bytes + gemm_scratch(T, d_in, d_out, false)) return SMLM_ERR_WORKSPACE;

  hipStream_t st = (hipStream_t)stream;
  // The plan groups the segments by their weight address.  A product that runs on the shrink kernels
  // (d_in >= d_out, weights [n][k]) over few enough segments builds it inside its own launch: every
  // workgroup numbers the addresses by their first occurrence and finds its tile itself, a few more
  // write the plan for the fold launch behind it (as the fused forward does with adapter ids).
  const int mt = tiles_per_wave(T, d_out, d_in);
  const int nw = shrink_waves(mt, 1, &d_in, d_out);
  const int ks = shrink_cfg(T, d_in, d_out, nw, false, mt, true).ksplit;
  const bool in_launch = d_in >= d_out && !w_row_major && self_planned_ok(T, S, S, pv.nt_max, mt) &&
                         (mt > 1 ? (S <= kFwdThreads || block_shrink(mt, T, d_out, false, 1, &w_ld) || ks % 2 == 0)
                                 : (nw == kDecodeWaves && (S <= kSelfPlanThreads || ks % 2 == 0)));
  if (in_launch) {
    if (!aligned16(y) || !aligned16(x)) return SMLM_ERR_ALIGN;
    const PlanSortArgs build{pv, seg_indptr, w_ptrs, SMLM_KEY_PTR2, S, next_pow2(S), w_ptrs};
    float* partial = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + plan_bytes);
    return run_shrink(dtype, pv, T, S, S, 1, &x, &w_ptrs, &partial, &y, &d_in, d_out, &w_ld, beta,
                      seg_scale, mt, st, true, false, nullptr, nullptr, 0, &build, false, nullptr, nullptr, true);
  }
  // An expanding product on single tiles finds them itself, up to a segment a thread.  Larger batches, on tile blocks,
  // keep the plan's launch: it is the smaller part of theirs.
  if (d_in < d_out && !w_row_major && S <= kFoundSegs && tiles_per_wave(T, d_in, kNoShrink) == 1) {
    FoundExpandArgs a{};
    a.plan = PlanSortArgs{pv, seg_indptr, w_ptrs, SMLM_KEY_PTR2, S, next_pow2(S), w_ptrs};
    a.seg_scale = seg_scale;
    a.beta = beta;
    a.p.y = reinterpret_cast<uint16_t*>(y);
    a.p.v = reinterpret_cast<const uint16_t*>(x);
    a.p.w_ptrs = w_ptrs;
    a.p.d_in = d_in; a.p.d_out = d_out; a.p.ldw = w_ld;
    return launch_expand_found(dtype, T, S, st, a);
  }
  rc = plan_build_impl(pv, seg_indptr, w_ptrs, SMLM_KEY_PTR, S, st);
  if (rc) return rc;
  return smlm_gemm_planned(y, x, w_ptrs, S, workspace, reinterpret_cast<char*>(workspace) + plan_bytes,
                           workspace_bytes - plan_bytes, T, S, d_in, d_out, w_ld, w_row_major, dtype,
                           beta, seg_scale, stream);
}

SMLM_API int smlm_gemm_static(void* y, const void* x, const void* const* w_ptrs,
                              const int32_t* seg_indptr, int T, int S, int d_in, int d_out, int w_ld,
                              int w_row_major, int dtype, float beta, const float* seg_scale,
                              void* stream) {
  int rc = check_common(T, S, dtype);
  if (rc) return rc;
  if (d_in <= 0 || d_out <= 0) return SMLM_ERR_ARG;
  if (plan_carve(nullptr, T, S, nullptr) + gemm_scratch(T, d_in, d_out, false) > SMLM_STATIC_SCRATCH_BYTES)
    return SMLM_ERR_SCRATCH;
  // an empty batch launches nothing (smlm_gemm validates the rest and returns): no device needed
  void* ws = (T == 0 || S == 0) ? nullptr : static_scratch();
  if (!ws && T != 0 && S != 0) return SMLM_ERR_LAUNCH;
  return smlm_gemm(y, x, w_ptrs, seg_indptr, ws, SMLM_STATIC_SCRATCH_BYTES, T, S, d_in, d_out, w_ld,
                   w_row_major, dtype, beta, seg_scale, stream);
}

SMLM_API int smlm_lora_fwd_multi_workspace_size(int n_proj, int T, const int* h_in, int r,
                                                size_t* bytes) {
  if (n_proj < 1 || n_proj > kMaxProj || T < 0 || !h_in || r <= 0 || !bytes) return SMLM_ERR_ARG;
  size_t n = 0;
  for (int i = 0; i < n_proj; ++i) {
    if (h_in[i] <= 0) return SMLM_ERR_ARG;
    const size_t rows = T > 0 ? T : 1;
    n += align_up((size_t)fwd_ksplit_bound(T, h_in[i], r) * rows * r * 4, 256) + align_up(rows * r * 2, 256);
  }
  *bytes = n;
  return SMLM_OK;
}

// the library's view of the caller's dropout descriptor; nullptr or seg_p == nullptr: none
static int drop_args(const smlm_dropout* d, DropArgs* out) {
  *out = DropArgs{};
  if (!d || !d->seg_p) return SMLM_OK;
  if (d->rows < 0) return SMLM_ERR_ARG;
  out->seg_p = d->seg_p;
  out->rows = d->rows;
  out->k0 = (uint32_t)d->seed; out->k1 = (uint32_t)(d->seed >> 32);
  out->o0 = (uint32_t)d->offset; out->o1 = (uint32_t)(d->offset >> 32);
  out->bits = reinterpret_cast<uint8_t*>(d->mask_bits);
  return SMLM_OK;
}

SMLM_API int smlm_lora_fwd_multi(int n_proj, void* const* y, const void* const* x,
                                 void* const* v_out, const void* const* const* a_ptrs,
                                 const void* const* const* b_ptrs, int n_weights, const int* h_in,
                                 const int* h_out, const void* plan, void* workspace,
                                 size_t workspace_bytes, int T, int S, int r, int dtype, float beta,
                                 const float* seg_scale, int stages, void* stream) {
  return smlm_lora_fwd_multi_ex(n_proj, y, x, v_out, a_ptrs, b_ptrs, n_weights, h_in, h_out, plan,
                                workspace, workspace_bytes, T, S, r, dtype, beta, seg_scale, stages,
                                nullptr, stream);
}

SMLM_API int smlm_lora_fwd_multi_ex(int n_proj, void* const* y, const void* const* x,
                                    void* const* v_out, const void* const* const* a_ptrs,
                                    const void* const* const* b_ptrs, int n_weights,
                                    const int* h_in, const int* h_out, const void* plan,
                                    void* workspace, size_t workspace_bytes, int T, int S, int r,
                                    int dtype, float beta, const float* seg_scale, int stages,
                                    const smlm_lora_opts* opts, void* stream) {
  int rc = check_common(T, S, dtype);
  if (rc) return rc;
  DropArgs drop;
  if ((rc = drop_args(opts ? opts->dropout : nullptr, &drop))) return rc;
  const int32_t* w_rank = opts ? opts->adapter_rank : nullptr;
  const int packed = (opts && opts->adapter_rank) ? opts->packed_ranks : 0;
  const int32_t* build_s = opts ? opts->build_seg_indptr : nullptr;
  const void* build_k = opts ? opts->build_seg_adapter : nullptr;
  const void* build_k2 = nullptr;
  int build_kind = SMLM_KEY_I32;
  if (opts && (opts->build_seg_key_a || opts->build_seg_key_b)) {  // grouped by pairs of addresses instead of ids
    if (build_k || !opts->build_seg_key_a || !opts->build_seg_key_b) return SMLM_ERR_ARG;
    build_k = opts->build_seg_key_a;
    build_k2 = opts->build_seg_key_b;
    build_kind = SMLM_KEY_PTR2;
  }
  if ((build_s != nullptr) != (build_k != nullptr)) return SMLM_ERR_ARG;
  if (build_s && !(stages & SMLM_STAGE_SHRINK)) return SMLM_ERR_ARG;  // the plan is built with the shrink
  if (n_proj < 1 || n_proj > kMaxProj || r <= 0 || !y || !x || !a_ptrs || !b_ptrs || !h_in || !h_out)
    return SMLM_ERR_ARG;
  if (stages < 1 || stages > (SMLM_STAGE_SHRINK | SMLM_STAGE_EXPAND)) return SMLM_ERR_ARG;
  if (r & 7) return SMLM_ERR_ALIGN;
  for (int i = 0; i < n_proj; ++i) {
    if (h_in[i] <= 0 || h_out[i] <= 0) return SMLM_ERR_ARG;
    if ((h_in[i] & 7) || (h_out[i] & 7)) return SMLM_ERR_ALIGN;
  }
  if (T == 0 || S == 0) return SMLM_OK;
  if (!plan || !workspace) return SMLM_ERR_ARG;
  if (!aligned16(workspace) || !aligned16(plan)) return SMLM_ERR_ALIGN;
  // A call that runs one stage only need not name what the other stage works on: a shrink-only
  // call no y, an expand-only call no x -- and an expand-only call skips the projections whose y
  // is NULL (the projections of one shrink call may be expanded one at a time, each when its y
  // is ready).
  const bool shrink_only = stages == SMLM_STAGE_SHRINK, expand_only = stages == SMLM_STAGE_EXPAND;
  for (int i = 0; i < n_proj; ++i) {
    if (!a_ptrs[i] || !b_ptrs[i]) return SMLM_ERR_ARG;
    if ((!y[i] && !shrink_only && !expand_only) || (!x[i] && !expand_only)) return SMLM_ERR_ARG;
    if (!aligned16(y[i]) || !aligned16(x[i]) || (v_out && v_out[i] && !aligned16(v_out[i])))
      return SMLM_ERR_ALIGN;
  }
  size_t need = 0;
  rc = smlm_lora_fwd_multi_workspace_size(n_proj, T, h_in, r, &need);
  if (rc) return rc;
  if (workspace_bytes < need) return SMLM_ERR_WORKSPACE;

  hipStream_t st = (hipStream_t)stream;
  PlanView pv;
  plan_carve(const_cast<void*>(plan), T, S, &pv);

  // shrink: every projection's v, rounded to 16 bits (into v_out when the caller wants it).
  // Decode batches (eight-wave shrink, one-tile expand) skip the fold launch: the expand
  // kernel adds the few partials while it loads v.
  float* partial[kMaxProj];
  void* v16[kMaxProj];
  int vsplit[kMaxProj];
  int k_min = h_in[0];
  for (int i = 1; i < n_proj; ++i) k_min = h_in[i] < k_min ? h_in[i] : k_min;
  const int mt = tiles_per_wave(T, r, k_min);
  const int nw = shrink_waves(mt, n_proj, h_in, r);
  bool expand_folds = nw == kDecodeWaves && mt == 1;
  {
    char* w = reinterpret_cast<char*>(workspace);
    for (int i = 0; i < n_proj; ++i) {
      vsplit[i] = shrink_cfg(T, h_in[i], r, nw, false, mt, false, drop.seg_p != nullptr).ksplit;
      expand_folds = expand_folds && vsplit[i] <= kMaxExpandFold;
      partial[i] = reinterpret_cast<float*>(w);
      w += align_up((size_t)fwd_ksplit_bound(T, h_in[i], r) * T * r * 4, 256);
      v16[i] = (v_out && v_out[i]) ? v_out[i] : w;
      w += align_up((size_t)T * r * 2, 256);
    }
  }
  // A plan still to be built (opts->build_*): inside the shrink launch where the batch is within its limits, else
  // with the plan launch first -- as under dropout with plans keyed by pairs of addresses, which no kernel of that
  // kind takes.  (2786 rows, two projections 4096 -> 4096 and 1024 at rank 32, dropout: forward + backward with two
  // plan launches of 5.6 us 116.0 us, both plans built in the shrinks 106.0 us.)
  PlanSortArgs build{pv, build_s, build_k, build_kind, S, next_pow2(S), build_k2};
  bool even_splits = true;  // (the decode route pairs k slices up beyond 512 segments)
  for (int i = 0; i < n_proj; ++i) even_splits = even_splits && (vsplit[i] % 2 == 0);
  // (both routes pair k slices up in one workgroup beyond 512 / 256 segments)
  const bool self_planned = build_s && (!drop.seg_p || build_kind == SMLM_KEY_I32) &&
                            self_planned_ok(T, S, n_weights, pv.nt_max, mt) &&
                            (mt > 1 ? (S <= kFwdThreads ||
                                       block_shrink(mt, T, r, drop.seg_p != nullptr, n_proj, h_in) || even_splits)
                                    : (expand_folds && (S <= kSelfPlanThreads || even_splits)));
  if (build_s && !self_planned && (rc = plan_build_impl(pv, build_s, build_k, build_kind, S, st, build_k2))) return rc;
  if (stages & SMLM_STAGE_SHRINK) {
    rc = run_shrink(dtype, pv, T, S, n_weights, n_proj, x, a_ptrs, partial, v16, h_in, r, h_in,
                    0.0f, nullptr, mt, st, !expand_folds, false, &drop, w_rank, packed,
                    self_planned ? &build : nullptr);
    if (rc) return rc;
  }
  if (!(stages & SMLM_STAGE_EXPAND)) return SMLM_OK;

  ExpandArgs ea{};
  ea.plan = tile_args(pv, n_weights);
  ea.plan.w_rank = w_rank;
  ea.plan.packed = packed;
  ea.seg_scale = seg_scale;
  ea.beta = beta;
  ea.T = T; ea.nt_max = pv.nt_max;
  int n_exp = 0, exp_h_out = 0;  // an expand-only call launches only the projections it names a y for
  for (int i = 0; i < n_proj; ++i) {
    if (!y[i]) continue;
    ExpandProj& P = ea.p[n_exp++];
    P.y = reinterpret_cast<uint16_t*>(y[i]);
    P.v = reinterpret_cast<const uint16_t*>(v16[i]);
    P.w_ptrs = b_ptrs[i];
    P.d_in = r; P.d_out = h_out[i]; P.ldw = r;
    if (h_out[i] > exp_h_out) exp_h_out = h_out[i];
    if (expand_folds) {
      P.vpart = partial[i];
      P.vsplit = vsplit[i];
      // the rounded v exists only inside the expand kernel: it writes the caller's copy
      if (v_out && v_out[i]) P.v_out = reinterpret_cast<uint16_t*>(v_out[i]);
    }
  }
  if (n_exp == 0) return SMLM_OK;
  return launch_expand(dtype, expand_nq(T, exp_h_out), mt, S, n_weights, n_exp, r, st, ea);
}

SMLM_API int smlm_lora_fwd_workspace_size(int T, int S, int h_in, int h_out, int r, size_t* bytes) {
  if (S < 0 || h_out <= 0) return SMLM_ERR_ARG;
  return smlm_lora_fwd_multi_workspace_size(1, T, &h_in, r, bytes);
}

SMLM_API int smlm_lora_fwd(void* y, const void* x, void* v_out, const void* const* a_ptrs,
                           const void* const* b_ptrs, int n_weights, const void* plan, void* workspace,
                           size_t workspace_bytes, int T, int S, int h_in, int h_out, int r, int dtype,
                           float beta, const float* seg_scale, void* stream) {
  return smlm_lora_fwd_multi(1, &y, &x, v_out ? &v_out : nullptr, &a_ptrs, &b_ptrs, n_weights, &h_in,
                             &h_out, plan,
                             workspace, workspace_bytes, T, S, r, dtype, beta, seg_scale,
                             SMLM_STAGE_SHRINK | SMLM_STAGE_EXPAND, stream);
}

SMLM_API int smlm_lora_bwd_multi_workspace_size(int n_proj, int n_rows, int P, int NA, const int* h_in,
                                                const int* h_out, int r, size_t* bytes) {
  if (n_proj < 1 || n_proj > kMaxProj || n_rows < 0 || P < 0 || NA < 0 || !h_in || !h_out || r <= 0 || !bytes)
    return SMLM_ERR_ARG;
  for (int i = 0; i < n_proj; ++i)
    if (h_in[i] <= 0 || h_out[i] <= 0) return SMLM_ERR_ARG;
  *bytes = bwd_layout(n_proj, n_rows > 0 ? n_rows : 1, P, NA > 0 ? NA : 1, h_in, h_out, r).total;
  return SMLM_OK;
}

SMLM_API int smlm_lora_bwd_workspace_size(int n_rows, int P, int NA, int h_in, int h_out, int r,
                                          size_t* bytes) {
  return smlm_lora_bwd_multi_workspace_size(1, n_rows, P, NA, &h_in, &h_out, r, bytes);
}

SMLM_API int smlm_lora_bwd(void* dx, void* const* da_ptrs, void* const* db_ptrs, const void* dy,
                           const void* x, const void* v, const void* const* a_ptrs,
                           const void* const* b_ptrs, const void* plan, void* workspace,
                           size_t workspace_bytes, int n_rows, int P, int NA, int h_in, int h_out,
                           int r, int dtype, const float* part_scale, void* stream) {
  return smlm_lora_bwd_ex(dx, da_ptrs, db_ptrs, dy, x, v, a_ptrs, b_ptrs, plan, workspace,
                          workspace_bytes, n_rows, P, NA, h_in, h_out, r, dtype, part_scale, nullptr, stream);
}

SMLM_API int smlm_lora_bwd_ex(void* dx, void* const* da_ptrs, void* const* db_ptrs,
                              const void* dy, const void* x, const void* v,
                              const void* const* a_ptrs, const void* const* b_ptrs,
                              const void* plan, void* workspace, size_t workspace_bytes,
                              int n_rows, int P, int NA, int h_in, int h_out, int r, int dtype,
                              const float* part_scale, const smlm_lora_opts* opts, void* stream) {
  return smlm_lora_bwd_multi_ex(1, &dx, &da_ptrs, &db_ptrs, &dy, &x, v ? &v : nullptr, &a_ptrs, &b_ptrs, plan,
                                workspace, workspace_bytes, n_rows, P, NA, &h_in, &h_out, r, dtype, part_scale,
                                opts, stream);
}

// every projection's dV product is folded from k-split partials: the fold then writes what the weight gradients read
static bool bwd_all_folded(int n_proj, int n_rows, const int* h_out, int r) {
  for (int i = 0; i < n_proj; ++i)
    if (shrink_cfg(n_rows, h_out[i], r, kFwdWaves, true, kBlkTiles).ksplit <= 1) return false;
  return true;
}

SMLM_API int smlm_lora_bwd_multi_ex(int n_proj, void* const* dx, void* const* const* da_ptrs,
                                    void* const* const* db_ptrs, const void* const* dy,
                                    const void* const* x, const void* const* v,
                                    const void* const* const* a_ptrs, const void* const* const* b_ptrs,
                                    const void* plan, void* workspace, size_t workspace_bytes,
                                    int n_rows, int P, int NA, const int* h_in, const int* h_out, int r,
                                    int dtype, const float* part_scale, const smlm_lora_opts* opts,
                                    void* stream) {
  int rc = check_common(n_rows, P, dtype);
  if (rc) return rc;
  DropArgs drop;
  if ((rc = drop_args(opts ? opts->dropout : nullptr, &drop))) return rc;
  const int32_t* w_rank = opts ? opts->adapter_rank : nullptr;
  const int packed = (opts && opts->adapter_rank) ? opts->packed_ranks : 0;
  const int stages = (opts && opts->bwd_stages) ? opts->bwd_stages : (SMLM_BWD_PRODUCTS | SMLM_BWD_DX | SMLM_BWD_WGRAD);
  // the other weight layout (the reference's is_row_major = True): A_a [h_in, r], B_a [r, h_out], and so are dA_a, dB_a
  const bool rm = opts && opts->w_row_major;
  const int dx_rows = opts ? opts->dx_rows : 0;
  if (dx_rows != 0 && dx_rows < n_rows) return SMLM_ERR_ARG;
  if (rm && (drop.seg_p || packed)) return SMLM_ERR_ARG;
  if (stages < 0 || stages > (SMLM_BWD_PRODUCTS | SMLM_BWD_DX | SMLM_BWD_WGRAD)) return SMLM_ERR_ARG;
  if (n_proj < 1 || n_proj > kMaxProj || NA < 0 || r <= 0 || !h_in || !h_out) return SMLM_ERR_ARG;
  if (r & 7) return SMLM_ERR_ALIGN;
  if (NA == 0 || n_rows == 0 || P == 0) return SMLM_ERR_ARG;
  if (!dx || !da_ptrs || !db_ptrs || !dy || !x || !a_ptrs || !b_ptrs || !workspace || !plan) return SMLM_ERR_ARG;
  if (!aligned16(workspace) || !aligned16(plan)) return SMLM_ERR_ALIGN;
  bool have_v = v != nullptr && v[0] != nullptr;
  for (int i = 0; i < n_proj; ++i) {
    if (h_in[i] <= 0 || h_out[i] <= 0) return SMLM_ERR_ARG;
    if ((h_in[i] & 7) || (h_out[i] & 7)) return SMLM_ERR_ALIGN;
    if (!da_ptrs[i] || !db_ptrs[i] || !a_ptrs[i] || !b_ptrs[i] || !dx[i] || !dy[i] || !x[i]) return SMLM_ERR_ARG;
    if (have_v != (v != nullptr && v[i] != nullptr)) return SMLM_ERR_ARG;  // v of every projection or of none
    if (!aligned16(dx[i]) || !aligned16(dy[i]) || !aligned16(x[i]) || (have_v && !aligned16(v[i])))
      return SMLM_ERR_ALIGN;
  }
  const BwdLayout L = bwd_layout(n_proj, n_rows, P, NA, h_in, h_out, r);
  if (workspace_bytes < L.total) return SMLM_ERR_WORKSPACE;

  hipStream_t st = (hipStream_t)stream;
  char* ws = reinterpret_cast<char*>(workspace);
  PlanView pv{};
  plan_carve(const_cast<void*>(plan), n_rows, P, &pv);

  // A plan still to be built (opts->build_*): the dV shrink builds it inside its launch when it is
  // the first launch to use it (tile-block route, v given, the mask's keep bits given under dropout); else the
  // plan launch first.
  const int32_t* build_s = opts ? opts->build_seg_indptr : nullptr;
  const int32_t* build_k = opts ? opts->build_seg_adapter : nullptr;
  if ((build_s != nullptr) != (build_k != nullptr)) return SMLM_ERR_ARG;
  if (build_s && !(stages & SMLM_BWD_PRODUCTS)) return SMLM_ERR_ARG;  // the plan is built with the first stage
  PlanSortArgs build{pv, build_s, build_k, SMLM_KEY_I32, P, next_pow2(P)};
  constexpr int mt = kBlkTiles;
  bool even_dv = true;  // (k slices in pairs beyond 256 partitions)
  for (int i = 0; i < n_proj; ++i) even_dv = even_dv && shrink_cfg(n_rows, h_out[i], r, kFwdWaves, true, mt).ksplit % 2 == 0;
  const bool self_planned = build_s && have_v && (!drop.seg_p || drop.bits) &&
                            self_planned_ok(n_rows, P, NA, pv.nt_max, mt) && (P <= kFwdThreads || block_shrink(mt, n_rows, r) || even_dv);
  const bool products = (stages & SMLM_BWD_PRODUCTS) != 0;
  if (build_s && !self_planned && (rc = plan_build_impl(pv, build_s, build_k, SMLM_KEY_I32, P, st))) return rc;

  // 1. The backward multiplies by B and A where the forward multiplies by A^T and B^T.  The
  // tile-block kernels read the weights as they lie in memory: B [h_out, r] and A [r, h_in] as [k][n].
  // (In the row-major layout dV = dY B^T and dX = dV A^T read B [r, h_out] and A [h_in, r] the way the
  // forward reads A [r, h_in] and B [h_out, r], and v = x A reads A as [k][n].)

  // The keep bits of x's dropout mask by tile slot (projection i: the stream offset + i; the caller's bits of the
  // projections lie end to end, by row): the forward's when the caller kept them, turned behind the dV shrink, else made
  // here (same stream, same bits), so that the kernels below apply a stored mask either way.
  uint8_t* bits[kMaxProj] = {};
  TileBits turn{};
  if (drop.seg_p) {
    size_t bits_off = 0;
    const int tiles = tile_units_max(n_rows, P, NA, 1);
    for (int i = 0; i < n_proj; ++i) {
      bits[i] = reinterpret_cast<uint8_t*>(ws + L.p[i].bits);
      if (drop.bits) {
        turn.rows_bits[i] = drop.bits + bits_off;
        turn.out[i] = bits[i];
        turn.pitch[i] = h_in[i] / 8;
        turn.chunks[i] = ceil_div(h_in[i], 64);
        const long end = turn.first[i] + (long)tiles * ceil_div(turn.chunks[i], 16);
        if (end > (1L << 30)) return SMLM_ERR_LIMIT;
        turn.first[i + 1] = (int)end;
        bits_off += (size_t)drop.rows * (h_in[i] / 8);
      } else {
        DropArgs di = drop;
        const uint64_t off = (((uint64_t)drop.o1 << 32) | drop.o0) + (uint32_t)i;
        di.o0 = (uint32_t)off; di.o1 = (uint32_t)(off >> 32);
        di.bits = bits[i];
        di.bits_pitch = h_in[i] / 8;
        const DropBitsArgs ba{pv.hdr, pv.tile_row, pv.tile_rseg, di};
        if (products && (rc = launch(drop_bits_kernel, dim3((unsigned)pv.nt_max), dim3(256), st, ba))) return rc;
      }
    }
    if (drop.bits) turn.n = n_proj, turn.rows = drop.rows < n_rows ? drop.rows : n_rows, turn.tiles = tiles;
  }

  float* partial[kMaxProj];
  void* dv16[kMaxProj];
  void* v16[kMaxProj];
  const void* vv[kMaxProj];
  for (int i = 0; i < n_proj; ++i) {
    partial[i] = reinterpret_cast<float*>(ws + L.p[i].partial);
    dv16[i] = ws + L.p[i].dv16;
    v16[i] = ws + L.p[i].v16;
    vv[i] = have_v ? v[i] : v16[i];
  }

  // 2. v = round16(x A^T) unless the forward saved it
  if (!have_v && products) {
    DropArgs vdrop = drop;
    vdrop.bits = nullptr;  // the shrink kernels run the generator themselves; nothing to store here
    if (rm) {  // A [h_in, r] is [k][n]: the tile-block shrink at every size
      int a_ld[kMaxProj];
      for (int i = 0; i < n_proj; ++i) a_ld[i] = r;
      if ((rc = run_shrink(dtype, pv, n_rows, P, NA, n_proj, x, a_ptrs, partial, v16, h_in, r, a_ld, 0.0f,
                           nullptr, kBlkTiles, st, true, true, nullptr, w_rank, 0, nullptr, true)))
        return rc;
    } else if ((rc = run_shrink(dtype, pv, n_rows, P, NA, n_proj, x, a_ptrs, partial, v16, h_in, r, h_in,
                                0.0f, nullptr, mt, st, true, false, &vdrop, w_rank, 0, nullptr, true)))  // v of the dropped x, as the forward made it
      return rc;
  }

  // 3. dV = round16(dY B)
  int b_ld[kMaxProj];
  for (int i = 0; i < n_proj; ++i) b_ld[i] = rm ? h_out[i] : r;  // B [h_out, r] read as [k][n]; B [r, h_out] as [n][k]
  // The weight gradients read s*dV and s*v by tile slot, transposed.  The fold of dV leaves them behind when there is
  // one for every projection (cheaper there than among dX's stores: cfg4-like batch dV 12.5 -> 13.5, dX 10.8 -> 8.2 us;
  // ragged 32-row partitions over six projections dV 84 -> 91, dX 90 -> 74 us); else dX's launch writes them.
  // (With them out of dX's launch, dX and the weight gradients need nothing of each other.  Issuing the weight
  // gradients on a second stream, forked after the fold and joined at the end, was measured under graph replay and
  // dropped: the two launches did not overlap to any gain and the fork and join cost 6 us.)
  SideOut side{};
  for (int i = 0; i < n_proj; ++i) {
    side.pt_a[i] = reinterpret_cast<uint16_t*>(ws + L.p[i].pt_a);
    side.pt_b[i] = reinterpret_cast<uint16_t*>(ws + L.p[i].pt_b);
    side.v2[i] = reinterpret_cast<const uint16_t*>(vv[i]);
  }
  side.scale = part_scale;
  // rows of dX past the backward's own (opts->dx_rows): cleared by the fold's launch when it runs in direct mode,
  // else by a launch of their own
  ZeroSpans tail{};
  if (dx_rows > n_rows) {
    for (int i = 0; i < n_proj; ++i) {
      tail.ptr[i] = reinterpret_cast<char*>(dx[i]) + (size_t)n_rows * h_in[i] * 2;
      tail.bytes[i] = (long)(dx_rows - n_rows) * h_in[i] * 2;  // (h_in is a multiple of 8: whole 16-byte pieces)
      tail.first[i + 1] = tail.first[i] + (int)((tail.bytes[i] + kZeroBlockBytes - 1) / kZeroBlockBytes);
    }
    tail.n = n_proj;
  }
  // (a function of the shapes and the option: the same in every call of a staged backward)
  const bool side_in_fold = bwd_all_folded(n_proj, n_rows, h_out, r);
  if (side_in_fold) side.zero = tail, side.bits = turn;
  else if (tail.n && products &&
           (rc = launch(zero_spans_kernel, dim3((unsigned)tail.first[tail.n]), dim3(256), st, tail)))
    return rc;
  bool side_done = false;
  if (products && (rc = run_shrink(dtype, pv, n_rows, P, NA, n_proj, dy, b_ptrs, partial, dv16, h_out, r, b_ld,
                                   0.0f, nullptr, mt, st, true, !rm, nullptr, w_rank, packed,
                                   self_planned ? &build : nullptr, true, side_in_fold ? &side : nullptr, &side_done)))
    return rc;
  if (products && side_done != side_in_fold) return SMLM_ERR_ARG;  // (cannot happen: both follow shrink_cfg)
  if (products && turn.n && !side_in_fold &&
      (rc = launch(tile_bits_kernel, dim3((unsigned)turn.first[turn.n]), dim3(256), st, TileBitsArgs{turn, pv.tile_row})))
    return rc;

  // 4. dX = s dV A, and the slot-ordered transposed s*dV, s*v for step 5
  ExpandArgs ea{};
  ea.plan = tile_args(pv, NA);
  ea.plan.w_rank = w_rank;
  ea.seg_scale = part_scale;
  ea.beta = 0.0f;
  ea.T = n_rows; ea.nt_max = pv.nt_max;
  int widest = 0;
  for (int i = 0; i < n_proj; ++i) {
    ExpandProj& E = ea.p[i];
    E.y = reinterpret_cast<uint16_t*>(dx[i]);
    E.v = reinterpret_cast<const uint16_t*>(dv16[i]);
    E.w_ptrs = a_ptrs[i];
    E.d_in = r; E.d_out = h_in[i]; E.ldw = rm ? r : h_in[i];  // A [r, h_in] as [k][n]; A [h_in, r] as [n][k]
    E.pt_a = side_in_fold ? nullptr : side.pt_a[i];
    E.pt_b = side_in_fold ? nullptr : side.pt_b[i];
    E.v2 = side.v2[i];
    E.drop_bits = bits[i];
    if (h_in[i] > widest) widest = h_in[i];
  }
  ea.w_kn = rm ? 0 : 1;
  ea.drop = drop;  // dX is the gradient with respect to x before its dropout
  auto launch_dx = [&] { return launch_expand(dtype, expand_nq(n_rows, widest), mt, P, NA, n_proj, r, st, ea); };
  if (!(stages & SMLM_BWD_WGRAD)) return (stages & SMLM_BWD_DX) ? launch_dx() : SMLM_OK;

  // 5. dA_a, dB_a for every adapter (zeros when it has no rows)
  WgradArgs wa{};
  wa.hdr = pv.hdr;
  wa.grp_tile = pv.grp_tile;
  wa.grp_id = pv.grp_id;
  wa.tile_row = pv.tile_row;
  wa.nproj = n_proj;
  const bool split = wgrad_split(n_rows / NA, NA, r, drop.seg_p != nullptr);
  // one-wave workgroups take several neighbouring chunks in turn when there are chunks enough to keep the
  // chip busy anyway: about 8192 workgroups are left
  long all_chunks = 0;
  for (int i = 0; i < n_proj; ++i) all_chunks += ceil_div(h_in[i], kWgCols) + ceil_div(h_out[i], kWgCols);
  int walk = 1;
  if (!split) {
    const long want = all_chunks * NA * ceil_div(r, 64) / 8192;
    walk = want < 1 ? 1 : (want > 8 ? 8 : (int)want);
  }
  wa.walk = walk;
  int units = 0;
  for (int i = 0; i < n_proj; ++i) {
    WgradProj& Q = wa.p[i];
    Q.q_a = reinterpret_cast<const uint16_t*>(x[i]);
    Q.q_b = reinterpret_cast<const uint16_t*>(dy[i]);
    Q.pt_a = reinterpret_cast<const uint16_t*>(ws + L.p[i].pt_a);
    Q.pt_b = reinterpret_cast<const uint16_t*>(ws + L.p[i].pt_b);
    Q.da_ptrs = da_ptrs[i];
    Q.db_ptrs = db_ptrs[i];
    Q.h_in = h_in[i]; Q.h_out = h_out[i];
    if (rm) {
      // dB [r, h_out] = sum (s v)^T dY has the shape the kernel's first product writes ([rank, columns]) and
      // dA [h_in, r] = sum x^T (s dV) the shape of its second ([columns, rank]): the two change places
      Q.q_a = reinterpret_cast<const uint16_t*>(dy[i]);
      Q.q_b = reinterpret_cast<const uint16_t*>(x[i]);
      Q.pt_a = reinterpret_cast<const uint16_t*>(ws + L.p[i].pt_b);
      Q.pt_b = reinterpret_cast<const uint16_t*>(ws + L.p[i].pt_a);
      Q.da_ptrs = db_ptrs[i];
      Q.db_ptrs = da_ptrs[i];
      Q.h_in = h_out[i]; Q.h_out = h_in[i];
    }
    Q.chunks_a = ceil_div(Q.h_in, kWgCols);
    Q.units_a = ceil_div(Q.chunks_a, walk);
    Q.unit0 = units;
    Q.drop_bits = bits[i];
    units += Q.units_a + ceil_div(ceil_div(Q.h_out, kWgCols), walk);
  }
  wa.r = r;
  wa.n_parts = P;
  wa.grp_seg = pv.grp_seg;
  wa.w_rank = w_rank;
  wa.packed = packed;
  wa.drop = drop;  // dA against the dropped x
  // ranks above 64 are covered 64 at a time by workgroups of their own
  const int nbj = r <= 16 ? 1 : (r <= 32 ? 2 : 4);  // what launch_wgrad has kernels for
  wa.units = units;
  wa.zcount = ceil_div(r, 64);
  dim3 grid(wa.zcount > 1 ? round_up(units, kWgXcd) * wa.zcount : units, NA);
  if (stages & SMLM_BWD_DX) {
    const int dx_units = tile_units_max(n_rows, P, NA, kBlkTiles);
    ExpandArgs e = ea;
    expand_rows(e, n_proj, 32 * 4);
    const long dx_items = (long)dx_units * e.items.row_start[n_proj];
    // (what passes between the two, dV's by-products, must have been left by the fold; dX of the other weight layout is
    // another kernel)
    if (side_in_fold && !rm && dx_items <= kDirectItems &&
        bwd_one_launch(n_proj, n_rows, NA, r, h_in, h_out, drop.seg_p != nullptr, split, (long)grid.x * NA)) {
      BwdTailArgs ta;
      ta.w = wa;
      ta.e = e;
      ta.wx = (int)grid.x;
      ta.wy = NA;
      ta.wgrad = round_up(ceil_div((int)grid.x * NA, split ? 1 : kFwdWaves), kWgXcd);
      const dim3 all((unsigned)(ta.wgrad + dx_items));
      return dtype == SMLM_DTYPE_F16 ? launch_bwd_tail_dt<SMLM_DTYPE_F16>(nbj, split, all, st, ta)
                                     : launch_bwd_tail_dt<SMLM_DTYPE_BF16>(nbj, split, all, st, ta);
    }
    if ((rc = launch_dx())) return rc;
  }
  if (drop.seg_p)
    return dtype == SMLM_DTYPE_F16 ? launch_wgrad<SMLM_DTYPE_F16, true>(nbj, split, grid, st, wa)
                                   : launch_wgrad<SMLM_DTYPE_BF16, true>(nbj, split, grid, st, wa);
  return dtype == SMLM_DTYPE_F16 ? launch_wgrad<SMLM_DTYPE_F16, false>(nbj, split, grid, st, wa)
                                 : launch_wgrad<SMLM_DTYPE_BF16, false>(nbj, split, grid, st, wa);
}

static int rms_bwd_threads(int cols) {
  const int pieces = cols / 8;  // a piece a thread, or two where a row has more than 1024
  return round_up(pieces <= 1024 ? pieces : ceil_div(pieces, 2), kWaveSize);
}
// workgroups of the RMSNorm kernels: the forward gives every row group its own workgroup; the backward's fill the
// chip once (up to 512 threads a CU, the same number on every CU) with two rows each or more, so that the partial sums
// of dw stay small next to x and g.  (4096 x 3072, 384 threads: 341 workgroups 21.9 us, 512 23.5, 256 19.2.)
static int rms_blocks(int rows, int cols, bool backward) {
  int nb, cap = 1 << 22;
  if (cols > kRmsMaxCols) {  // wide rows: a workgroup per row; the backward's partial rows are whole rows of floats
    nb = rows;
    if (backward) cap = 128;
  } else if (backward) {
    const int threads = rms_bwd_threads(cols);
    nb = ceil_div(rows, 2);
    cap = 256 * (threads >= 512 ? 1 : 512 / threads);
  } else {
    nb = ceil_div(rows, cols <= kRmsWaveCols ? 4 : 1);
  }
  if (nb > cap) nb = cap;
  return nb < 1 ? 1 : nb;
}
static int rms_bwd_blocks(int rows, int cols) { return rms_blocks(rows, cols, true); }

static int rms_check(int rows, int cols, int dtype) {
  if (rows < 0 || cols <= 0) return SMLM_ERR_ARG;
  if (dtype != SMLM_DTYPE_F16 && dtype != SMLM_DTYPE_BF16) return SMLM_ERR_DTYPE;
  if (cols & 7) return SMLM_ERR_ALIGN;
  if (cols > (1 << 24) || rows > (1 << 30)) return SMLM_ERR_LIMIT;
  return SMLM_OK;
}

SMLM_API int smlm_rms_norm_fwd(void* out, float* rms, const void* x, const void* w, int rows,
                               int cols, float eps, int dtype, void* stream) {
  int rc = rms_check(rows, cols, dtype);
  if (rc) return rc;
  if (rows == 0) return SMLM_OK;
  if (!out || !rms || !x || !w) return SMLM_ERR_ARG;
  if (!aligned16(out) || !aligned16(x) || !aligned16(w)) return SMLM_ERR_ALIGN;
  const RmsFwdArgs a{reinterpret_cast<uint16_t*>(out), rms, reinterpret_cast<const uint16_t*>(x),
                     reinterpret_cast<const uint16_t*>(w), rows, cols, eps};
  hipStream_t st = (hipStream_t)stream;
  const bool f16 = dtype == SMLM_DTYPE_F16;
  const int nb = rms_blocks(rows, cols, false);
  const dim3 grid((unsigned)nb);
  const int rows_per_step = cols <= kRmsWaveCols ? 4 : 1;
  const bool one_turn = (long)nb * rows_per_step >= rows;  // every workgroup sees one row group
  const dim3 bl(256);
  if (cols > kRmsMaxCols)
    return f16 ? launch(rms_fwd_wide_kernel<SMLM_DTYPE_F16>, grid, bl, st, a)
               : launch(rms_fwd_wide_kernel<SMLM_DTYPE_BF16>, grid, bl, st, a);
  if (cols <= kRmsWaveCols) {
    if (one_turn)
      return f16 ? launch(rms_fwd_kernel<SMLM_DTYPE_F16, 1, true>, grid, bl, st, a)
                 : launch(rms_fwd_kernel<SMLM_DTYPE_BF16, 1, true>, grid, bl, st, a);
    return f16 ? launch(rms_fwd_kernel<SMLM_DTYPE_F16, 1, false>, grid, bl, st, a)
               : launch(rms_fwd_kernel<SMLM_DTYPE_BF16, 1, false>, grid, bl, st, a);
  }
  if (one_turn)
    return f16 ? launch(rms_fwd_kernel<SMLM_DTYPE_F16, 4, true>, grid, bl, st, a)
               : launch(rms_fwd_kernel<SMLM_DTYPE_BF16, 4, true>, grid, bl, st, a);
  return f16 ? launch(rms_fwd_kernel<SMLM_DTYPE_F16, 4, false>, grid, bl, st, a)
             : launch(rms_fwd_kernel<SMLM_DTYPE_BF16, 4, false>, grid, bl, st, a);
}

SMLM_API int smlm_rms_norm_bwd_workspace_size(int rows, int cols, size_t* bytes) {
  if (!bytes) return SMLM_ERR_ARG;
  int rc = rms_check(rows, cols, SMLM_DTYPE_F16);
  if (rc) return rc;
  *bytes = align_up((size_t)rms_bwd_blocks(rows > 0 ? rows : 1, cols) * cols * 4, 256);
  return SMLM_OK;
}

SMLM_API int smlm_rms_norm_bwd(void* dx, void* dw, const void* g, const void* x, const void* w,
                               const float* rms, void* workspace, size_t workspace_bytes, int rows,
                               int cols, int dtype, void* stream) {
  int rc = rms_check(rows, cols, dtype);
  if (rc) return rc;
  if (!dx || !dw || !g || !x || !w || !rms || !workspace) return SMLM_ERR_ARG;
  if (!aligned16(dx) || !aligned16(dw) || !aligned16(g) || !aligned16(x) || !aligned16(w) ||
      !aligned16(workspace))
    return SMLM_ERR_ALIGN;
  if (rows == 0) return SMLM_ERR_ARG;  // dw would have nothing to sum
  const int nb = rms_bwd_blocks(rows, cols);
  if (workspace_bytes < (size_t)nb * cols * 4) return SMLM_ERR_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const bool f16 = dtype == SMLM_DTYPE_F16;
  const RmsBwdArgs a{reinterpret_cast<uint16_t*>(dx), reinterpret_cast<float*>(workspace),
                     reinterpret_cast<const uint16_t*>(g), reinterpret_cast<const uint16_t*>(x),
                     reinterpret_cast<const uint16_t*>(w), rms, rows, cols};
  const dim3 grid((unsigned)nb);
  if (cols > kRmsMaxCols)
    rc = f16 ? launch(rms_bwd_wide_kernel<SMLM_DTYPE_F16>, grid, dim3(256), st, a)
             : launch(rms_bwd_wide_kernel<SMLM_DTYPE_BF16>, grid, dim3(256), st, a);
  else if (cols <= 8192)
    rc = f16 ? launch(rms_bwd_kernel<SMLM_DTYPE_F16, 1, 2>, grid, dim3(rms_bwd_threads(cols)), st, a)
             : launch(rms_bwd_kernel<SMLM_DTYPE_BF16, 1, 2>, grid, dim3(rms_bwd_threads(cols)), st, a);
  else
    rc = f16 ? launch(rms_bwd_kernel<SMLM_DTYPE_F16, 2, 1>, grid, dim3(rms_bwd_threads(cols)), st, a)
             : launch(rms_bwd_kernel<SMLM_DTYPE_BF16, 2, 1>, grid, dim3(rms_bwd_threads(cols)), st, a);
  if (rc) return rc;
  const RmsFoldArgs fa{reinterpret_cast<uint16_t*>(dw), reinterpret_cast<const float*>(workspace), nb, cols};
  return f16 ? launch_rms_fold<SMLM_DTYPE_F16>(st, fa) : launch_rms_fold<SMLM_DTYPE_BF16>(st, fa);
}

SMLM_API int smlm_segments_build(const int32_t* req_adapter, const int32_t* req_len, int R,
                                 int32_t* seg_adapter, int32_t* seg_len, int32_t* seg_indptr,
                                 int32_t* n_seg, void* stream) {
  if (R < 0 || !seg_indptr || !n_seg) return SMLM_ERR_ARG;
  if (R > 0 && (!req_adapter || !req_len || !seg_adapter || !seg_len)) return SMLM_ERR_ARG;
  if (R > kMaxSegments) return SMLM_ERR_LIMIT;
  const SegmentsArgs a{req_adapter, req_len, seg_adapter, seg_len, seg_indptr, n_seg, R};
  return launch(segments_kernel, dim3(1), dim3(kPlanThreads), (hipStream_t)stream, a);
}

SMLM_API int smlm_segment_scales(const int32_t* seg_adapter, int S, const float* table, int n_table, float* seg_out,
                                 const int32_t* seg_indptr, const int32_t* starts, int P, int64_t* part_seg,
                                 float* part_out, void* stream) {
  if (S < 0 || P < 0 || n_table < 0) return SMLM_ERR_ARG;
  if (S > kMaxSegments || P > kMaxSegments) return SMLM_ERR_LIMIT;
  if (S == 0) return P == 0 ? SMLM_OK : SMLM_ERR_ARG;
  if (seg_out && (!seg_adapter || !table || n_table == 0)) return SMLM_ERR_ARG;
  if (P > 0 && (!part_seg || (starts && !seg_indptr) || (part_out && !seg_out))) return SMLM_ERR_ARG;
  const int n = S > P ? S : P;
  const SegmentScalesArgs a{seg_adapter, table, seg_out, seg_indptr, starts, part_seg, part_out, S, n_table, P};
  return launch(segment_scales_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), (hipStream_t)stream, a);
}

SMLM_API int smlm_put_words(void* dst, const void* src, size_t bytes, void* stream) {
  if (bytes == 0) return SMLM_OK;
  if (!dst || !src) return SMLM_ERR_ARG;
  if ((bytes & 3) || (reinterpret_cast<uintptr_t>(dst) & 3)) return SMLM_ERR_ALIGN;
  uint32_t* d = reinterpret_cast<uint32_t*>(dst);
  const char* from = reinterpret_cast<const char*>(src);
  for (size_t words = bytes / 4; words;) {
    const int n = words < (size_t)kPutLarge ? (int)words : kPutLarge;
    int rc;
    if (n <= kPutSmall) {
      PutArgs<kPutSmall> a;
      a.dst = d;
      a.n = n;
      memcpy(a.words, from, (size_t)n * 4);
      rc = launch(put_words_kernel<kPutSmall>, dim3(1), dim3(256), (hipStream_t)stream, a);
    } else {
      PutArgs<kPutLarge> a;
      a.dst = d;
      a.n = n;
      memcpy(a.words, from, (size_t)n * 4);
      rc = launch(put_words_kernel<kPutLarge>, dim3(1), dim3(256), (hipStream_t)stream, a);
    }
    if (rc) return rc;
    d += n;
    from += (size_t)n * 4;
    words -= n;
  }
  return SMLM_OK;
}

}  // extern "C"
