// Shrink (skinny-N, long-K) and expand (skinny-K, wide-N) tile kernels.
//
// Both take the place of the CUTLASS GemmGrouped instantiations of
// kernel_src/csrc/smlm_forward/smlm_forward_cutlass.cuh:84-171.  The unit of
// work is a 16-row plan tile of one adapter (or a tile block of up to four).
// v_mfma_f32_16x16x32 runs with the tokens as the MFMA *columns* and the weight
// rows as the MFMA *rows*, so a lane ends up with consecutive output columns of
// one token.  x fragments are 16-byte global loads straight into registers (x
// is contiguous along the contraction); weight fragments come straight from
// global memory in the one-tile kernels and from an LDS-staged chunk shared by
// the tiles of a block in the tile-block kernels.
//
// Every output element is produced by the same sequence of MFMA steps over k
// whatever other rows share its tile or its workgroup, so regrouping or
// re-segmenting rows never changes a bit of any row.
//
// The number of tiles is only known on the device (plan header).  Launches are
// sized on the host over an upper bound of it, one work item per workgroup
// ("direct" mode); items past the real count find an empty entry in the plan
// and leave.  A persistent one-dimensional walk over the exact count (one
// contiguous range of items per XCD, or plain round robin) remains as the
// fallback for batches beyond the direct grid's limits.
#pragma once
#include "dropout.hpp"
#include "smlm_common.hpp"

namespace smlm {

constexpr int kFwdThreads = 256;
constexpr int kFwdWaves = kFwdThreads / kWaveSize;
constexpr int kMaxProj = 8;   // projections one launch can serve
constexpr int kNumXcd = 8;

struct TileArgs {
  const int32_t* hdr;        // 0 n_tiles, 4 n_blocks
  const int32_t* tile_row;
  const int32_t* tile_rseg;
  const int32_t* tile_wid;
  const int32_t* blk;        // (first tile << 3) | tile count, per tile block
  const int32_t* w_rank;     // optional, indexed like the weight tables: true rank of each adapter
  int packed;                // with w_rank: the weights are STORED at their true rank (rounded up to 8),
                             //   A_a [r_a, h_in], B_a [h_out, r_a], instead of zero-padded to the launch's rank
  int n_weights;             // entries of the caller's weight tables (0: unknown): a tile whose index is not
                             //   below it is left alone, like a tile of a negative adapter id
};

// whether tile index `wid` of a plan names an entry of the caller's weight tables (negative: a segment no
// adapter serves; at or past the table length: an id the caller's tables do not hold -- never dereferenced)
__device__ __forceinline__ bool wid_ok(const TileArgs& p, int wid) {
  return wid >= 0 && (p.n_weights <= 0 || wid < p.n_weights);
}

// Adapters of different ranks live zero-padded to one rank (the reference pads every adapter
// of a layer to the layer's maximum, src/loquetier_src/models/mixed_lora.py:501-521).  With the
// true ranks at hand the padding is not read: loads at or past the rank (rounded up to the
// 8-element load width) are predicated off and read zeros, which is what the padding holds.
__device__ __forceinline__ int rank_limit(const TileArgs& p, int wid, int d) {
  if (!p.w_rank) return d;
  const int r = (uload(p.w_rank, wid) + 7) & ~7;
  return r < d ? r : d;
}
// Leading dimension of a weight matrix whose contiguous dimension is the rank (B [h_out, r], read
// by the expand and by the backward's dV product): the launch's rank for zero-padded storage, the
// adapter's own (rank_limit) for packed storage -- a rank-8 adapter beside rank-64 ones then costs
// 16 bytes a row instead of a 128-byte line.
__device__ __forceinline__ int rank_ld(const TileArgs& p, int ld, int lim) {
  return (p.w_rank && p.packed) ? lim : ld;
}

// Items [first, last) of this workgroup, visited with stride `step`.  The grid
// size is a multiple of kNumXcd.
struct WorkRange {
  int first, last, step;
};
__device__ __forceinline__ WorkRange work_range(int n_work, bool interleave) {
  if (interleave) return WorkRange{(int)blockIdx.x, n_work, (int)gridDim.x};
  const int xcd = blockIdx.x % kNumXcd, local = blockIdx.x / kNumXcd;
  const int base = n_work / kNumXcd, extra = n_work % kNumXcd;
  const int start = xcd * base + (xcd < extra ? xcd : extra);
  const int count = base + (xcd < extra ? 1 : 0);
  return WorkRange{start + local, start + count, (int)gridDim.x / kNumXcd};
}

// Items are numbered (chunk row, tile unit) with the tile unit fastest; the
// chunk rows of all projections are laid end to end (row_start[p] = first chunk
// row of projection p), so there are no empty items to skew the XCD ranges.
// units_max > 0 selects the direct mode used for small launches: one item per
// workgroup, numbered over the host's upper bound of the tile units, so the
// kernel need not wait for the plan header; units past the real count are
// marked empty in the plan (tile_wid < 0, blk == 0).
struct ItemSpace {
  int row_start[kMaxProj + 1];
  int nproj;
  int interleave;  // plain round-robin items instead of one range per XCD
  int units_max;
  int flat;        // direct mode: projections end to end along x instead of on z
};
__device__ __forceinline__ void item_decode(const ItemSpace& sp, int V, int units, int* pj, int* yy,
                                            int* tb) {
  const int cr = V / units;
  *tb = V - cr * units;
  int p = 0;
#pragma unroll
  for (int i = 1; i < kMaxProj; ++i) p += (i < sp.nproj && cr >= sp.row_start[i]) ? 1 : 0;
  *pj = p;
  *yy = cr - sp.row_start[p];
}
// DIRECT launches put the chunk rows on x and the tile units on y.  Chunk rows
// are the fast axis: the workgroups in flight at one time then cover whole
// output rows of a few tile units, which the memory system serves better than a
// few columns of all rows.  The projections are either the z axis (x then spans
// the longest projection and shorter ones leave empty workgroups, but the
// projection's arguments are known at once) or, with `flat`, laid end to end
// along x (row_start; no empty workgroups -- better when the projections differ
// much in width).  (Re-indexing the plane so that the workgroups sharing a
// weight chunk share an XCD's L2 was measured: it removes the repeated weight
// fetches and is no faster, or much slower when it spreads the rows in flight.)
template <bool DIRECT>
__device__ __forceinline__ WorkRange item_range(const ItemSpace& sp, int units) {
  if (DIRECT) return WorkRange{0, 1, 1};
  return work_range(units * sp.row_start[sp.nproj], sp.interleave != 0);
}
template <bool DIRECT>
__device__ __forceinline__ bool item_get(const ItemSpace& sp, int V, int units, int* pj, int* yy,
                                         int* tb) {
  if (DIRECT && !sp.flat) {
    *pj = blockIdx.z;
    *yy = blockIdx.x;
    *tb = blockIdx.y;
    return *yy < sp.row_start[*pj + 1] - sp.row_start[*pj];
  }
  if (DIRECT) {
    const int cr = blockIdx.x;
    int p = 0;
#pragma unroll
    for (int i = 1; i < kMaxProj; ++i) p += (i < sp.nproj && cr >= sp.row_start[i]) ? 1 : 0;
    *pj = p;
    *yy = cr - sp.row_start[p];
    *tb = blockIdx.y;
    return true;
  }
  item_decode(sp, V, units, pj, yy, tb);
  return true;
}

// number of units along the tile axis: single tiles (MT == 1) or the plan's tile
// blocks (tiles of one adapter, up to kBlkTiles each)
template <int MT>
__device__ __forceinline__ int tile_units(const TileArgs& p, int units_max) {
  if (units_max > 0) return units_max;
  return MT == 1 ? p.hdr[0] : p.hdr[4];
}
// tiles of unit tb and their weight index; cnt == 0 for a unit past the end
template <int MT>
__device__ __forceinline__ void pick_tiles(const TileArgs& p, int tb, int* t0, int* cnt, int* wid) {
  if (MT == 1) {
    *t0 = tb;
    *wid = uload(p.tile_wid, tb);
    *cnt = wid_ok(p, *wid) ? 1 : 0;
  } else {
    const int packed = uload(p.blk, tb);
    *t0 = packed >> 3;
    *cnt = packed & 7;
    *wid = *cnt ? uload(p.tile_wid, *t0) : -1;
    if (!wid_ok(p, *wid)) *cnt = 0;  // a negative adapter id (rows that no adapter serves) or one past the tables
  }
}

// eight consecutive-k elements of weight column n (zeros when !ok).  A function of its own for the order it gives the
// single-tile shrink's loads: with the address written out at the call, q/k/v/o of 256 rows at rank 16 take 9.2 us
// instead of 9.0, of 1000 rows 15.2 instead of 14.8, 11008 -> 16 of 256 rows 9.5 instead of 9.3.
__device__ __forceinline__ u32x4 load_w8(const uint16_t* W, int n, int k, int ldw, bool ok, const uint16_t* zeros) {
  return ldg16_or(W + (long)n * ldw + k, ok, zeros);
}

// out = beta*old + scale*acc for four consecutive columns of one row
template <int DT>
__device__ __forceinline__ void store4(uint16_t* dst, f32x4 a, float scale, float beta) {
  u32x2 o;
  if (beta != 0.0f) {
    const u32x2 old = *reinterpret_cast<const u32x2*>(dst);
    o[0] = pack2<DT>(beta * Num<DT>::lo(old[0]) + scale * a[0], beta * Num<DT>::hi(old[0]) + scale * a[1]);
    o[1] = pack2<DT>(beta * Num<DT>::lo(old[1]) + scale * a[2], beta * Num<DT>::hi(old[1]) + scale * a[3]);
  } else {
    o[0] = pack2<DT>(scale * a[0], scale * a[1]);
    o[1] = pack2<DT>(scale * a[2], scale * a[3]);
  }
  *reinterpret_cast<u32x2*>(dst) = o;
}

// ------------------------------------------------------------------ shrink --
struct ShrinkProj {
  const uint16_t* x;          // [T, d_in]
  const void* const* w_ptrs;  // indexed by the plan's tile_wid
  float* partial;             // [ksplit, T, d_out] fp32 when ksplit > 1
  uint16_t* out;              // [T, d_out] when ksplit == 1
  int d_in, d_out, ldw, k_per_wave, ksplit, zblocks;
  int to_partial;             // write the fp32 partial even when ksplit == 1 (the consumer rounds)
  uint8_t* drop_bits;         // DROP kernels, optional: [rows, d_in / 8] keep bits of this projection's mask
};

struct ShrinkArgs {
  TileArgs plan;
  ShrinkProj p[kMaxProj];
  const float* seg_scale;     // applied when ksplit == 1
  float beta;
  int T;
  ItemSpace items;            // chunk rows of projection p: ksplit*zblocks
  int w_kn;                   // tile-block kernel only: weights are stored [k][n]
  DropArgs drop;              // DROP kernels: dropout of the training rows of x
};

// a wave's own LDS accesses are served in order; the compiler must keep them in order too
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sixteen rows of 32 * U of k on their way from memory to the MFMA.  They are requested along the rows, load i of a lane
// piece `piece` of row `row(i)`, and change layout in an LDS area of the wave's own: afterwards register u of lane (c, g)
// holds row c, k 32 u + 8 g .. + 7.  Requested in that layout, sixteen rows to sixteen neighbouring lanes, a load occupies
// the CU's address unit for 64 cycles instead of 19.
template <int U>
struct LineTurn {
  static constexpr int kRow = 4 * U;  // 16-byte pieces of a row
  static constexpr int kBytes = kTileRows * kRow * 16;
  static_assert(U == 2 || U == 4, "rows of one or two lines");
  static __device__ __forceinline__ int row(int lane, int i) { return (lane + kWaveSize * i) / kRow; }
  static __device__ __forceinline__ int piece(int lane) { return lane % kRow; }
  // (pieces change places within their row so that reads and writes touch each bank once)
  static __device__ __forceinline__ int at(int r, int p) { return r * kRow + (p ^ (U == 4 ? r : (r >> 1) & 7)); }
  static __device__ __forceinline__ void turn(char* lds, int lane, u32x4 (&v)[U]) {
    u32x4* a = reinterpret_cast<u32x4*>(lds);
#pragma unroll
    for (int i = 0; i < U; ++i) a[at(row(lane, i), piece(lane))] = v[i];
    lds_order();
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = a[at(lane & 15, 4 * u + (lane >> 4))];
    lds_order();
  }
};

// Shrink for single tiles (batches of few rows).  Work item -> (projection, k
// slice, 64-column block, tile).  The NW waves of a workgroup take consecutive k
// ranges; their accumulators are summed through LDS in wave order and written
// either as an fp32 partial (k split over workgroups, or a consumer that folds)
// or as the final 16-bit value.  NW = 8 is for decode batches: few tiles, long k.
template <int DT, int NB, int U, int NW, bool DIRECT, bool DROP = false>
__global__ __launch_bounds__(NW * kWaveSize) void shrink_kernel(ShrinkArgs a) {
  typedef LineTurn<U> Turn;
  // a wave's part: x and the weights on their way to the MFMA, then its sums
  constexpr int kSums = NB * kWaveSize;
  __shared__ __attribute__((aligned(16))) char area[NW][Turn::kBytes > kSums * 16 ? Turn::kBytes : kSums * 16];
  auto red = [&](int w, int nb) -> f32x4& { return reinterpret_cast<f32x4*>(area[w])[nb * kWaveSize + (threadIdx.x & 63)]; };
  const int units = DIRECT ? 0 : tile_units<1>(a.plan, 0);
  const WorkRange wr = item_range<DIRECT>(a.items, units);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;

  for (int V = wr.first; V < wr.last; V += wr.step) {
    int pj, yy, tile;
    if (!item_get<DIRECT>(a.items, V, units, &pj, &yy, &tile)) break;
    const ShrinkProj P = a.p[pj];
    const int kz = yy % P.ksplit, zb = yy / P.ksplit;
    if (zb >= P.zblocks) continue;  // a chunk row added to make the count even (uniform over the workgroup)
    const int wid = uload(a.plan.tile_wid, tile);
    if (!wid_ok(a.plan, wid)) continue;  // past the last tile (direct mode), or no such adapter; uniform over the workgroup
    const int n0 = zb * 64;
    const int slot = tile * kTileRows + c;
    const int row = a.plan.tile_row[slot];
    int lrow[U];  // the rows this lane requests
#pragma unroll
    for (int i = 0; i < U; ++i) lrow[i] = a.plan.tile_row[tile * kTileRows + Turn::row(lane, i)];
    const uint16_t* W = uload_ptr(P.w_ptrs, wid);
    const int nlim = rank_limit(a.plan, wid, P.d_out);  // weight rows at or past it are zero padding
    const int rseg = DROP ? a.plan.tile_rseg[slot] : -1;

    const int kbeg = (kz * NW + wave) * P.k_per_wave;
    const int kend = min(kbeg + P.k_per_wave, P.d_in);
    const uint16_t* zeros = reinterpret_cast<const uint16_t*>(a.plan.hdr + kHdrZeros);
    const DropArgs dp = DROP ? drop_proj(a.drop, pj) : DropArgs{};
    const float prob = DROP ? drop_prob(dp, row, rseg, zeros) : 0.0f;
    uint8_t* const bits_out = zb == 0 ? P.drop_bits : nullptr;
    const bool words = drop_words<U>(bits_out, P.d_in >> 3);
    DropRow dr{};
    bool dropped = false;

    f32x4 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto load_batch = [&](int k, u32x4 (&xf)[U], u32x4 (&wf)[NB][U]) {
      const int kk = k + 8 * Turn::piece(lane);
      const bool kin = kk < kend;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < U; ++i) {
          const int n = n0 + 16 * nb + Turn::row(lane, i);
          wf[nb][i] = load_w8(W, n, kk, P.ldw, kin && n < nlim, zeros);
        }
#pragma unroll
      for (int i = 0; i < U; ++i)
        xf[i] = ldg16_or(P.x + (long)lrow[i] * P.d_in + kk, kin && lrow[i] >= 0, zeros);
    };
    auto multiply = [&](int k, u32x4 (&xf)[U], u32x4 (&wf)[NB][U]) {
      DropMasks<U> dm;
      if (DROP && dropped) {  // (x is on its way)
        dm.make(dp, dr, row, k >> 3, g, bits_out, P.d_in >> 3, kend >> 3, words);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) Turn::turn(area[wave], lane, wf[nb]);
      Turn::turn(area[wave], lane, xf);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (DROP && dropped) xf[u] = dm.template apply<DT>(xf[u], u, dr);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb] = Num<DT>::mfma(wf[nb][u], xf[u], acc[nb]);
      }
    };
    {
      // two load batches in turn: one is on its way while the other is multiplied
      u32x4 xa[U], wa[NB][U], xb[U], wb[NB][U];
      load_batch(kbeg, xa, wa);
      if (DROP) dr = drop_params(prob), dropped = __builtin_amdgcn_ballot_w64(dr.on) != 0;  // (uniform over the wave)
#pragma unroll 1
      for (int k = kbeg; k < kend; k += 64 * U) {
        const bool more = k + 32 * U < kend;  // uniform over the wave
        if (more) load_batch(k + 32 * U, xb, wb);
        multiply(k, xa, wa);
        if (!more) break;
        if (k + 64 * U < kend) load_batch(k + 64 * U, xa, wa);
        multiply(k + 32 * U, xb, wb);
      }
    }

    // cross-wave sum in wave order; wave 0 writes the tile
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) red(wave, nb) = acc[nb];
    __syncthreads();
    if (wave == 0 && row >= 0) {
      float scale = 1.0f;
      const bool as_partial = P.ksplit > 1 || P.to_partial;
      if (!as_partial && a.seg_scale) scale = a.seg_scale[a.plan.tile_rseg[slot]];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        // all NW reads are issued before the first add waits for one (left to itself the
        // compiler keeps two in flight, and a many-wave kernel spends as long here as
        // in its k loop)
        f32x4 part[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) part[w] = red(w, nb);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 sum = part[0];
#pragma unroll
        for (int w = 1; w < NW; ++w) sum += part[w];
        const int n = n0 + 16 * nb + 4 * g;  // lane holds columns n .. n+3 of its token
        if (n >= P.d_out) continue;
        if (as_partial)
          *(SMLM_GLOBAL f32x4*)(P.partial + ((long)kz * a.T + row) * P.d_out + n) = sum;
        else
          store4<DT>(P.out + (long)row * P.d_out + n, sum, scale, a.beta);
      }
    }
    __syncthreads();  // red is free again (persistent walk)
  }
}

// Shrink for tile blocks (larger batches, and the backward) where block_shrink() does not choose the other kernel.  Work
// item -> (projection, k slice, column block of 16 * NB, tile block) as above, but here wave w owns tile w of the block
// and all four waves walk the whole k slice together: each 32*U-wide batch of the weight
// rows is staged once in LDS (two buffers in turn, one barrier a batch) and shared by the
// four tiles, while every wave loads the x fragments of its own tile straight into
// registers one batch ahead.  The weights are read from L2 once per workgroup, not once per
// wave, and there is no cross-wave sum.
//
// WKN: the weight matrices are stored [k][n] (k rows of d_out contiguous columns, as B
// [h_out, r] is for the backward's dV = dY B) instead of [n][k]: a batch is then staged as
// it lies in memory and the MFMA operand, which wants eight consecutive k of one column,
// is read out of LDS with the transposing read.
template <int DT, int NB, int U, bool DIRECT, bool WKN, bool DROP = false>
__global__ __launch_bounds__(kFwdThreads) void shrink_wide_kernel(ShrinkArgs a) {
  constexpr int KB = 32 * U;                 // k per batch
  constexpr int kRowsW = 16 * NB;            // weight rows (output columns) per workgroup
  constexpr int kPitch = WKN ? kRowsW + 8 : KB + 8;  // LDS row pitch in elements
  constexpr int kPieces = kRowsW * (KB / 8); // 16-byte pieces of one staged batch
  constexpr int kPer = (kPieces + kFwdThreads - 1) / kFwdThreads;
  __shared__ __attribute__((aligned(16))) uint16_t wlds[2][(WKN ? KB : kRowsW) * kPitch];
  const int units = DIRECT ? 0 : tile_units<kBlkTiles>(a.plan, 0);
  const WorkRange wr = item_range<DIRECT>(a.items, units);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const uint16_t* zeros = reinterpret_cast<const uint16_t*>(a.plan.hdr + kHdrZeros);

  for (int V = wr.first; V < wr.last; V += wr.step) {
    int pj, yy, tb;
    if (!item_get<DIRECT>(a.items, V, units, &pj, &yy, &tb)) break;
    const ShrinkProj P = a.p[pj];
    const int kz = yy % P.ksplit, zb = yy / P.ksplit;
    if (zb >= P.zblocks) continue;  // a chunk row added to make the count even (uniform over the workgroup)
    int t0, cnt, wid;
    pick_tiles<kBlkTiles>(a.plan, tb, &t0, &cnt, &wid);
    if (cnt == 0) continue;  // uniform over the workgroup
    const int n0 = zb * 16 * NB;  // (several column blocks only where NB = 4 or 8)
    const bool active = wave < cnt;
    const int slot = (t0 + (active ? wave : 0)) * kTileRows + c;
    const int row = active ? a.plan.tile_row[slot] : -1;
    const uint16_t* W = uload_ptr(P.w_ptrs, wid);
    const int nlim = rank_limit(a.plan, wid, P.d_out);  // weight rows at or past it are zero padding
    const int ldw = WKN ? rank_ld(a.plan, P.ldw, nlim) : P.ldw;  // [k][n] weights (B) have the rank contiguous
    const int kbeg = kz * kFwdWaves * P.k_per_wave;
    const int kend = min(kbeg + kFwdWaves * P.k_per_wave, P.d_in);
    const uint16_t* xrow = P.x + (long)(row < 0 ? 0 : row) * P.d_in;
    const DropArgs dp = DROP ? drop_proj(a.drop, pj) : DropArgs{};
    const float prob = DROP ? drop_prob(dp, row, a.plan.tile_rseg[slot], zeros) : 0.0f;
    DropRow dr{};
    bool dropped = false;
    uint8_t* const bits_out = zb == 0 ? P.drop_bits : nullptr;
    const bool words = drop_words<U>(bits_out, P.d_in >> 3);
    DropMasks<U> dm;
    auto make_masks = [&](int kb) { dm.make(dp, dr, row, kb >> 3, g, bits_out, P.d_in >> 3, kend >> 3, words); };

    auto load_x = [&](int kb, u32x4 (&xf)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int kk = kb + 32 * u + 8 * g;
        xf[u] = ldg16_or(xrow + kk, row >= 0 && kk < kend, zeros);
      }
    };
    auto load_w = [&](int kb, u32x4 (&st)[kPer]) {
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const int idx = threadIdx.x + j * kFwdThreads;
        if (WKN) {
          const int kl = idx / (kRowsW / 8), n8 = (idx % (kRowsW / 8)) * 8;
          st[j] = ldg16_or(W + (long)(kb + kl) * ldw + n0 + n8,
                           idx < kPieces && n0 + n8 < nlim && kb + kl < kend, zeros);
        } else {
          const int nl = idx / (KB / 8), k8 = (idx % (KB / 8)) * 8;
          st[j] = ldg16_or(W + (long)(n0 + nl) * ldw + kb + k8,
                           idx < kPieces && n0 + nl < nlim && kb + k8 < kend, zeros);
        }
      }
    };
    auto stage_w = [&](int buf, const u32x4 (&st)[kPer]) {
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const int idx = threadIdx.x + j * kFwdThreads;
        const int r_ = WKN ? idx / (kRowsW / 8) : idx / (KB / 8);
        const int c_ = WKN ? (idx % (kRowsW / 8)) * 8 : (idx % (KB / 8)) * 8;
        if (idx < kPieces) *reinterpret_cast<u32x4*>(&wlds[buf][r_ * kPitch + c_]) = st[j];
      }
    };
    auto weight_frag = [&](int buf, int u, int nb) -> u32x4 {
      if (WKN) {
        // lane c names k row 32u + 8g (+4) + c/4 and columns 16nb + 4(c%4) .. +3; it receives
        // column 16nb + c of four consecutive k rows per read
        const uint16_t* base = &wlds[buf][(32 * u + 8 * g + (c >> 2)) * kPitch + 16 * nb + 4 * (c & 3)];
        const u32x2 q0 = lds_read_tr16(base), q1 = lds_read_tr16(base + 4 * kPitch);
        return u32x4{q0[0], q0[1], q1[0], q1[1]};
      }
      return *reinterpret_cast<const u32x4*>(&wlds[buf][(16 * nb + c) * kPitch + 32 * u + 8 * g]);
    };

    f32x4 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};

    u32x4 xf[U], wst[kPer];
    load_x(kbeg, xf);
    load_w(kbeg, wst);
    if (DROP) {
      dr = drop_params(prob);
      dropped = __builtin_amdgcn_ballot_w64(dr.on) != 0;  // (uniform over the wave)
      if (dropped) make_masks(kbeg);                      // (x is on its way)
    }
    __syncthreads();  // every wave is done with both LDS buffers of the previous item
    stage_w(0, wst);
    int buf = 0;
#pragma unroll 1
    for (int kb = kbeg; kb < kend; kb += KB) {
      u32x4 xn[U], wn[kPer];
      // the next batch is requested before this one is multiplied (past the end: zeros)
      load_x(kb + KB, xn);
      load_w(kb + KB, wn);
      __syncthreads();  // buffer `buf` is written; buffer `buf ^ 1` is no longer read
      if (active) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (DROP && dropped) xf[u] = dm.template apply<DT>(xf[u], u, dr);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc[nb] = Num<DT>::mfma(weight_frag(buf, u, nb), xf[u], acc[nb]);
        }
      }
      if (DROP && dropped && kb + KB < kend) make_masks(kb + KB);  // (the next batch is on its way)
      stage_w(buf ^ 1, wn);
      buf ^= 1;
#pragma unroll
      for (int u = 0; u < U; ++u) xf[u] = xn[u];
    }

    if (row >= 0) {
      const bool as_partial = P.ksplit > 1 || P.to_partial;
      float scale = 1.0f;
      if (!as_partial && a.seg_scale) scale = a.seg_scale[a.plan.tile_rseg[slot]];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int n = n0 + 16 * nb + 4 * g;  // lane holds columns n .. n+3 of its token
        if (n >= P.d_out) continue;
        if (as_partial)
          *(SMLM_GLOBAL f32x4*)(P.partial + ((long)kz * a.T + row) * P.d_out + n) = acc[nb];
        else
          store4<DT>(P.out + (long)row * P.d_out + n, acc[nb], scale, a.beta);
      }
    }
  }
}

// ---- the products of a tile block: x [64 rows, k slice] W^T, for one or more (projection, k slice) ----
// Each of the four waves multiplies all four tiles of the block (64 rows) with 16 * NB weight columns over its own part
// of the k slice -- pieces of 64 of k, the four waves' pieces side by side, so that the workgroup reads 512 consecutive
// bytes of every row at a time -- and the waves' sums are added through LDS, in wave order, at the end of the slice.  No
// wave waits for another before that: two pieces are held in registers in turn, of which one or two are on their way at
// any time, the first of the next slice among them while a slice is finished.
//
// x and the weights are requested in full lines, eight lanes to 128 bytes of a row, and change layout through an LDS area
// of the wave's own.  Requested as the MFMA wants them, sixteen rows to the sixteen neighbouring lanes, a load occupies
// the CU's address unit for 64 cycles instead of 19 (measured with data out of L2), which alone holds x and the weights
// together to 9.4 TB/s.
//
// Bound by HBM and by what surrounds it: 7675 rows, three projections 4096 -> 64: 59.4 us with the weights staged for
// four waves at a barrier a batch, 50 so (189 MB of x; 245 MB fetched from beyond the L2s); whole pass of 7675 rows at
// rank 64, 4096 -> 14336 twice and back, 281 -> 259 us; 8600 rows over 64 adapters, six projections, 826 -> 809 us.
//
// WKN: the weight matrices are stored [k][n] (k rows of d_out contiguous columns, as B
// [h_out, r] is for the backward's dV = dY B) instead of [n][k]: a piece lies in LDS as it does in memory and the MFMA
// operand, which wants eight consecutive k of one column, is read out of it with the transposing read.
//
// Slots without a row multiply the block's first row and columns at or past the adapter's rank another column's
// weights: MFMA columns and rows do not mix, the former are not stored and the latter are stored as zeros.
__device__ __attribute__((aligned(16))) uint32_t product_zeros[4];  // what loads past the end of a slice read, and
                                                                    // predicated-off ones of kernels without a plan

constexpr int kBlockMaxLd = 1 << 25;  // longest weight row, in elements: a lane's offset in the weights has 32 bits

// waves a SIMD the registers are held to
constexpr int block_product_waves(int NB) { return NB >= 4 ? 2 : 3; }

template <int DT, int NB, bool WKN>
struct BlockProduct {
  static constexpr int KB = 64, U = KB / 32;      // k of a wave's piece, its 32-wide steps
  static constexpr int kPitch = 16 * NB + 8;      // WKN: LDS row pitch of the weights in elements
  static constexpr int kTileBytes = kTileRows * KB * 2;             // 16 rows of x (or of the weights) on their way
  static constexpr int kWBytes = WKN ? KB * kPitch * 2 : NB * kTileBytes;
  static constexpr int kStageBytes = kWBytes + 2 * kTileBytes;      // of a wave
  static constexpr int kRedBytes = kFwdWaves * kBlkTiles * NB * kWaveSize * 16;
  static constexpr int kLdsBytes = kFwdWaves * kStageBytes > kRedBytes ? kFwdWaves * kStageBytes : kRedBytes;

  struct Stage {
    u32x4 x[kBlkTiles][2], w[2 * NB];  // as they are loaded: eight rows of eight 16-byte pieces an element
    int k0;
  };
  struct Item {  // (all uniform over the four waves)
    int pj, kz, kbeg, kend, n;  // n: pieces a wave takes
  };

  const ShrinkArgs& a;
  const int lane, wave, c, g;
  const int wid, nlim;       // the block's adapter; weight rows at or past nlim are zero padding
  const int tiles;           // tiles of the block
  const int nlists;          // the chunk rows r, r + nlists ... are this group's
  int lrow[kBlkTiles][2];    // the rows this lane loads: 8 i + lane / 8 of tile t (the block's first row: none)
  int rw;                    // its row of tile `wave`, which it stores
  float scale;               //   ... and what that is scaled with when no partial sums are stored
  f32x4 acc[kBlkTiles][NB];
  // what is loaded next
  int r, s;
  Item li;
  const uint16_t *wbase, *xbase;
  int d_in, ldw;
  uint32_t woff;             // the lane's byte offset in the weights (up to 31 rows: ldw <= kBlockMaxLd)

  __device__ __forceinline__ BlockProduct(const ShrinkArgs& args, int thread, int wid_, int nlim_, int tiles_, int list,
                                          int lists)
      : a(args), lane(thread & 63), wave(__builtin_amdgcn_readfirstlane(thread >> 6)), c(thread & 15),
        g((thread & 63) >> 4), wid(wid_), nlim(nlim_), tiles(tiles_), nlists(lists), rw(-1), scale(1.0f), r(list), s(0) {
#pragma unroll
    for (int t = 0; t < kBlkTiles; ++t)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[t][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // the rows of the block, row_of(slot): row of slot 16 t + i of the block, -1 where there is none (not slot 0)
  template <typename F>
  __device__ __forceinline__ void set_rows(const F& row_of) {
#pragma unroll
    for (int t = 0; t < kBlkTiles; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) lrow[t][i] = row_of(kTileRows * t + 8 * i + (lane >> 3));
    rw = row_of(kTileRows * wave + c);
  }

  __device__ __forceinline__ bool exists(int row_) const { return row_ < a.items.row_start[a.items.nproj]; }
  __device__ __forceinline__ Item item(int row_) const {
    Item it;
    it.pj = 0;
#pragma unroll
    for (int i = 1; i < kMaxProj; ++i) it.pj += (i < a.items.nproj && row_ >= a.items.row_start[i]) ? 1 : 0;
    const ShrinkProj& P = a.p[it.pj];
    it.kz = row_ - a.items.row_start[it.pj];
    it.kbeg = it.kz * kFwdWaves * P.k_per_wave;
    it.kend = min(it.kbeg + kFwdWaves * P.k_per_wave, P.d_in);
    it.n = (it.kend - it.kbeg + kFwdWaves * KB - 1) / (kFwdWaves * KB);
    return it;
  }
  // the weights of chunk row r; `W`: their address where the caller already knows it
  __device__ __forceinline__ void open_w(const uint16_t* W = nullptr) {
    li = item(r);
    const ShrinkProj& P = a.p[li.pj];
    if (!W) W = uload_ptr(P.w_ptrs, wid);
    ldw = WKN ? rank_ld(a.plan, P.ldw, nlim) : P.ldw;  // [k][n] weights (B) have the rank contiguous
    if (WKN) {
      wbase = W;
      const int n8 = (lane % (2 * NB)) * 8;
      woff = ((uint32_t)(lane / (2 * NB)) * (uint32_t)ldw + (uint32_t)(n8 < nlim ? n8 : 0)) * 2u;
    } else {
      wbase = W;
      woff = ((uint32_t)(lane >> 3) * (uint32_t)ldw + 8u * (lane & 7)) * 2u;
    }
    s = 0;
  }
  __device__ __forceinline__ void open_x() {
    const ShrinkProj& P = a.p[li.pj];
    d_in = P.d_in;
    xbase = P.x + 8 * (lane & 7);
  }
  // slots without a row load the block's first row
  __device__ __forceinline__ void fill_rows() {
    const int any = max(__builtin_amdgcn_readfirstlane(lrow[0][0]), 0);
#pragma unroll
    for (int t = 0; t < kBlkTiles; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) lrow[t][i] = lrow[t][i] >= 0 ? lrow[t][i] : any;
  }
  __device__ __forceinline__ int piece_k() const {
    int k0 = li.kbeg + (wave + kFwdWaves * s) * KB;
    // (opaque: the compiler otherwise keeps an induction register pair for every address)
    asm volatile("" : "+s"(k0));
    return k0;
  }
  // a piece past the end of its slice (every wave takes as many) or the list reads zeros, as does its part past the end
  __device__ __forceinline__ void load_w(Stage& st) {
    const int k0 = st.k0 = piece_k();
    const uint16_t* zeros = reinterpret_cast<const uint16_t*>(product_zeros);
    const int kend = nlim > 0 ? li.kend : 0;  // (an adapter of rank 0 has no weights)
#pragma unroll
    for (int j = 0; j < 2 * NB; ++j) {
      if (WKN) {
        const int kj = k0 + (32 / NB) * j;
        const uint16_t* p = reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(wbase + (long)kj * ldw) + woff);
        st.w[j] = ldg16_or(p, kj + lane / (2 * NB) < kend, zeros);
      } else {
        const uint16_t* p = reinterpret_cast<const uint16_t*>(
            reinterpret_cast<const char*>(wbase + (long)(8 * j < nlim ? 8 * j : 0) * ldw + k0) + woff);
        st.w[j] = ldg16_or(p, k0 + 8 * (lane & 7) < kend, zeros);
      }
    }
  }
  __device__ __forceinline__ void load_x(Stage& st) {
    const uint16_t* zeros = reinterpret_cast<const uint16_t*>(product_zeros);
    const bool in = st.k0 + 8 * (lane & 7) < li.kend;
    const uint16_t* base = in ? xbase + st.k0 : zeros;
    const uint32_t pitch = in ? (uint32_t)d_in * 2u : 0u;
#pragma unroll
    for (int t = 0; t < kBlkTiles; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        st.x[t][i] = ldg16(reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(base) +
                                                             (uint64_t)(uint32_t)lrow[t][i] * pitch));
    ++s;
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void load(Stage& st) {
    if (s >= li.n) {  // (no vector memory access in here: the compiler would wait for the loads in flight)
      r += nlists;
      if (exists(r)) {
        open_w();
        open_x();
      } else {
        li.kend = 0;  // zeros from here on
      }
    }
    load_w(st);
    load_x(st);
  }
  // Through the wave's LDS area from rows of full lines, as they are loaded, to MFMA operands.  Piece p of row i lies in
  // place p ^ (i / 2) of its row: both ways every instruction touches each bank once.
  __device__ __forceinline__ void put(char* lds, int i, u32x4 v) const {
    const int row = 8 * i + (lane >> 3);
    *reinterpret_cast<u32x4*>(lds + row * (KB * 2) + (((lane & 7) ^ ((row >> 1) & 7)) << 4)) = v;
  }
  __device__ __forceinline__ u32x4 get(const char* lds, int u) const {
    return *reinterpret_cast<const u32x4*>(lds + c * (KB * 2) + (((4 * u + g) ^ ((c >> 1) & 7)) << 4));
  }
  __device__ __forceinline__ void multiply(const Stage& st, char* lds) {
    uint16_t* wl = reinterpret_cast<uint16_t*>(lds);
#pragma unroll
    for (int j = 0; j < 2 * NB; ++j) {
      if (WKN) *reinterpret_cast<u32x4*>(&wl[((32 / NB) * j + lane / (2 * NB)) * kPitch + (lane % (2 * NB)) * 8]) = st.w[j];
      else put(lds + (j >> 1) * kTileBytes, j & 1, st.w[j]);
    }
    u32x4 wf[NB][U];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h == 1 && tiles <= 2) break;  // (uniform over the four waves)
#pragma unroll
      for (int e = 0; e < 4; ++e) put(lds + kWBytes + (e >> 1) * kTileBytes, e & 1, st.x[2 * h + (e >> 1)][e & 1]);
      lds_order();
      if (h == 0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            if (WKN) {
              // lane c names k row 32u + 8g (+4) + c/4 and columns 16nb + 4(c%4) .. +3; it receives
              // column 16nb + c of four consecutive k rows per read
              const uint16_t* base = &wl[(32 * u + 8 * g + (c >> 2)) * kPitch + 16 * nb + 4 * (c & 3)];
              const u32x2 q0 = lds_read_tr16(base), q1 = lds_read_tr16(base + 4 * kPitch);
              wf[nb][u] = u32x4{q0[0], q0[1], q1[0], q1[1]};
            } else {
              wf[nb][u] = get(lds + nb * kTileBytes, u);
            }
          }
      }
      u32x4 xf[2][U];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 2; ++e) xf[e][u] = get(lds + kWBytes + e * kTileBytes, u);
      lds_order();
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int e = 0; e < 2; ++e) acc[2 * h + e][nb] = Num<DT>::mfma(wf[nb][u], xf[e][u], acc[2 * h + e][nb]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // Sum over the waves and store: wave w the rows of tile w.  Every thread of the four waves calls it.
  __device__ __forceinline__ void finish(char* smem, const Item& it, bool real) {
    f32x4(*red)[kBlkTiles][NB][kWaveSize] = reinterpret_cast<f32x4(*)[kBlkTiles][NB][kWaveSize]>(smem);
    const ShrinkProj& P = a.p[it.pj];
    const bool as_partial = P.ksplit > 1 || P.to_partial;
    __syncthreads();  // every wave is done with the area
#pragma unroll
    for (int t = 0; t < kBlkTiles; ++t)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        red[wave][t][nb][lane] = acc[t][nb];
        acc[t][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    __syncthreads();
    if (rw >= 0 && real) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        f32x4 part[kFwdWaves];
#pragma unroll
        for (int w = 0; w < kFwdWaves; ++w) part[w] = red[w][wave][nb][lane];
        f32x4 sum = part[0];
#pragma unroll
        for (int w = 1; w < kFwdWaves; ++w) sum += part[w];
        const int n = 16 * nb + 4 * g;  // lane holds columns n .. n+3 of its token
        if (n >= P.d_out) continue;
        if (n >= nlim) sum = f32x4{0.f, 0.f, 0.f, 0.f};
        if (as_partial)
          *(SMLM_GLOBAL f32x4*)(P.partial + ((long)it.kz * a.T + rw) * P.d_out + n) = sum;
        else
          store4<DT>(P.out + (long)rw * P.d_out + n, sum, scale, a.beta);
      }
    }
    __syncthreads();  // the sums are read: the area takes rows again
  }
  // The products of the group's chunk rows, the weights of the first piece (`sa`) already requested.  `turns`: how many,
  // turns past the group's last row among them (every group of a workgroup takes as many: there are barriers inside).
  __device__ __forceinline__ void run(Stage& sa, char* smem, int turns) {
    char* lds = smem + wave * kStageBytes;
    int mr = r, ms = 0;  // what is multiplied: chunk row, piece
    Item mi = li;
    auto next = [&] {
      if (++ms < mi.n) return;
      finish(smem, mi, exists(mr));
      mr += nlists;
      --turns;
      ms = 0;
      if (exists(mr)) mi = item(mr);
      else mi.n = 1;
    };
    Stage sb;
    load_x(sa);
    // (all loads are unconditional: where branches join the compiler waits for every load in flight)
#pragma unroll 1
    while (true) {
      load(sb);
      multiply(sa, lds);
      next();
      if (turns <= 0) break;
      load(sa);
      multiply(sb, lds);
      next();
      if (turns <= 0) break;
    }
  }
};

// Shrink for tile blocks where block_shrink() chooses it.  Grid (lists, tile blocks): a workgroup takes the chunk rows
// (projection, k slice) blockIdx.x, blockIdx.x + gridDim.x ... of its tile block; NB blocks of 16 columns hold the rank.
template <int DT, int NB, bool WKN>
__global__ __launch_bounds__(kFwdThreads) __attribute__((amdgpu_waves_per_eu(block_product_waves(NB))))
void shrink_block_kernel(ShrinkArgs a) {
  typedef BlockProduct<DT, NB, WKN> Product;
  __shared__ __attribute__((aligned(16))) char smem[Product::kLdsBytes];
  const int tb = (int)(blockIdx.y + blockIdx.z * gridDim.y);
  if (tb >= a.items.units_max) return;
  int t0, cnt, wid;
  pick_tiles<kBlkTiles>(a.plan, tb, &t0, &cnt, &wid);
  if (cnt == 0) return;  // uniform over the workgroup
  const int c = threadIdx.x & 15, wave = threadIdx.x >> 6;
  const int nlim = rank_limit(a.plan, wid, a.p[0].d_out);
  Product pr(a, threadIdx.x, wid, nlim, cnt, blockIdx.x, gridDim.x);
  pr.set_rows([&](int i) {
    const int row = a.plan.tile_row[(i < cnt * kTileRows ? t0 * kTileRows : t0 * kTileRows - i) + i];
    return i < cnt * kTileRows ? row : -1;
  });
  const int slot = (t0 + wave) * kTileRows + c;
  typename Product::Stage first;
  pr.open_w();
  pr.load_w(first);
  if (a.seg_scale && pr.rw >= 0) pr.scale = a.seg_scale[a.plan.tile_rseg[slot]];
  pr.fill_rows();
  pr.open_x();
  const int rows = a.items.row_start[a.items.nproj];
  pr.run(first, smem, (rows - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x);
}

constexpr int kMaxKsplit = 16;  // upper bound of the k split over workgroups

// Spans of memory to be cleared by workgroups of 256 threads, kZeroBlockBytes each: span i takes blocks
// [first[i], first[i + 1]).
constexpr int kZeroBlockBytes = 32768;
struct ZeroSpans {
  char* ptr[kMaxProj];
  long bytes[kMaxProj];     // multiples of 16
  int first[kMaxProj + 1];
  int n;
};
__device__ __forceinline__ void zero_span_block(const ZeroSpans& z, int block, int thread) {
  int i = 0;
#pragma unroll
  for (int j = 1; j < kMaxProj; ++j) i += (j < z.n && block >= z.first[j]) ? 1 : 0;
  const long off0 = (long)(block - z.first[i]) * kZeroBlockBytes;
  const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < kZeroBlockBytes / (256 * 16); ++e) {
    const long off = off0 + ((long)e * 256 + thread) * 16;
    if (off < z.bytes[i]) stg16(reinterpret_cast<uint16_t*>(z.ptr[i] + off), zero);
  }
}
__global__ __launch_bounds__(256) void zero_spans_kernel(ZeroSpans z) { zero_span_block(z, (int)blockIdx.x, threadIdx.x); }

struct ReduceProj {
  const float* partial;  // [ksplit, T, d_out]
  uint16_t* out;         // [T, d_out]
  int ksplit;            // 1: nothing to fold for this projection
  // SIDE folds (the backward's dV): side_scale * out by tile slot, transposed (side_piece), and the
  // same treatment of v2 (a second [T, d_out] matrix) -- what the weight-gradient kernel reads
  uint16_t* pt_a;
  uint16_t* pt_b;
  const uint16_t* v2;
};

struct ReduceArgs {
  TileArgs plan;
  ReduceProj p[kMaxProj];
  const float* seg_scale;
  float beta;
  int T, d_out, nproj;
  int units_max;  // > 0: direct mode, one (projection, tile) per workgroup over this tile bound
  const float* side_scale;  // SIDE folds: per segment, or null for 1
  ZeroSpans zero;           // SIDE folds, direct mode: memory the launch's last workgroups clear (the rows of dX
                            //   past the backward's own)
  TileBits bits;            // ... and keep bits they bring into the order of the tiles
};

// Folds the k-split partial sums of a shrink launch, in split order, into the
// 16-bit result (the reference's "v in the I/O dtype"), scaled per segment: work item -> (projection,
// tile), 16 threads per row.
template <int DT>
__global__ __launch_bounds__(256) void reduce_kernel(ReduceArgs a) {
  const int units = tile_units<1>(a.plan, a.units_max);
  const int c = threadIdx.x >> 4, q = threadIdx.x & 15;
  const int last = a.units_max > 0 ? (int)blockIdx.x + 1 : units * a.nproj;
  for (int V = blockIdx.x; V < last; V += gridDim.x) {
    const int pj = V / units, tile = V - pj * units;
    const ReduceProj P = a.p[pj];
    if (P.ksplit <= 1) continue;
    if (!wid_ok(a.plan, uload(a.plan.tile_wid, tile))) continue;  // past the last tile (direct mode), or no such adapter
    const int slot = tile * kTileRows + c;
    const int row = a.plan.tile_row[slot];
    if (row < 0) continue;
    const float scale = a.seg_scale ? a.seg_scale[a.plan.tile_rseg[slot]] : 1.0f;
    const float* zf = reinterpret_cast<const float*>(a.plan.hdr + kHdrZeros);
    for (int n = 4 * q; n < a.d_out; n += 64) {
      // all partials are requested before the first add waits for one; past ksplit the loads
      // read zeros (the k split never exceeds kMaxKsplit)
      f32x4 part[kMaxKsplit];
#pragma unroll
      for (int z = 0; z < kMaxKsplit; ++z)
        part[z] = ldg_f4(z < P.ksplit ? P.partial + ((long)z * a.T + row) * a.d_out + n : zf);
      f32x4 sum = part[0];
#pragma unroll
      for (int z = 1; z < kMaxKsplit; ++z) sum += part[z];
      store4<DT>(P.out + (long)row * a.d_out + n, sum, scale, a.beta);
    }
  }
}

// The same fold without a scale, four columns a thread over all rows in order instead of through the plan's
// tiles: grid (T * d_out / 4 threads, projections).  Nothing is
// looked up before the partials are requested; the rows that belong to a segment are the
// range [hdr[5], hdr[5] + hdr[2]) (segments lie end to end) and only those are stored.
// KS: upper bound of the launch's k splits.  Bound by its one round trip to memory: sixteen loads a thread whatever the
// split, a row on sixteen lanes of which only d_out / 4 worked, 8600 rows, six projections at rank 64: 14.1 us, so 9.7;
// 4224 rows, one projection at rank 16: 4.2 and 3.0.
template <int DT, int KS>
__global__ __launch_bounds__(256) void reduce_rows_kernel(ReduceArgs a) {
  const ReduceProj P = a.p[blockIdx.y];
  if (P.ksplit <= 1) return;
  const long i = (long)blockIdx.x * 256 + threadIdx.x, total = (long)a.T * (a.d_out / 4);
  const int row = (int)(i / (a.d_out / 4));
  const int first = uload(a.plan.hdr, 5), count = uload(a.plan.hdr, 2);
  const float* zf = reinterpret_cast<const float*>(a.plan.hdr + kHdrZeros);
  f32x4 part[KS];
#pragma unroll
  for (int z = 0; z < KS; ++z) part[z] = ldg_f4((i < total && z < P.ksplit) ? P.partial + (z * total + i) * 4 : zf);
  f32x4 sum = part[0];
#pragma unroll
  for (int z = 1; z < KS; ++z) sum += part[z];
  if (i < total && row >= first && row < first + count) store4<DT>(P.out + i * 4, sum, 1.0f, a.beta);
}

// The fold of the backward's dV, which also leaves the by-products of write_side (further down) behind: the rounded
// sums and v2, scaled, by tile slot and transposed; slots without a row get zeros.  Work item -> (projection, 64
// columns, four tiles), a thread per slot and four columns.  The transposed rows go through LDS, so that they are
// written 128 bytes at a time: two bytes a lane straight from the registers, 268 partitions of 2080 rows, six
// projections at ranks up to 64: 16.0 us, so 12.0; 2048 rows, two projections at rank 128: 11.3 and 7.5.  The
// launch's workgroups past its items clear a.zero and turn a.bits.
constexpr int kSideThreads = kBlkTiles * 256;
template <int DT, int KS>
__global__ __launch_bounds__(kSideThreads) void side_fold_kernel(ReduceArgs a) {
  constexpr int kSlots = kBlkTiles * kTileRows, kCols = 64;
  constexpr int kTPitch = kSlots + 2;  // elements: columns 33 banks apart
  __shared__ __attribute__((aligned(4))) uint16_t tr[2][kCols * kTPitch];
  const int tiles = tile_units<1>(a.plan, a.units_max);
  const int groups = (tiles + kBlkTiles - 1) / kBlkTiles, cols = (a.d_out + kCols - 1) / kCols;
  const int items = groups * a.nproj * cols;
  if (a.units_max > 0 && (int)blockIdx.x >= items) {  // (uniform over the workgroup)
    const int block = ((int)blockIdx.x - items) * kBlkTiles + (int)(threadIdx.x >> 8), zeros = a.zero.first[a.zero.n];
    if (block < zeros) zero_span_block(a.zero, block, threadIdx.x & 255);
    else if (block - zeros < a.bits.first[a.bits.n]) tile_bits_item(a.bits, a.plan.tile_row, block - zeros, threadIdx.x & 255);
    return;
  }
  const int slot = threadIdx.x >> 4, q = threadIdx.x & 15;
  const float* zf = reinterpret_cast<const float*>(a.plan.hdr + kHdrZeros);
  const int last = a.units_max > 0 ? (int)blockIdx.x + 1 : items;
  for (int V = blockIdx.x; V < last; V += gridDim.x) {
    const int pj = V / (groups * cols), in = V - pj * groups * cols;
    const int n0 = in % cols * kCols, tile0 = in / cols * kBlkTiles;
    const ReduceProj P = a.p[pj];
    const int n = n0 + 4 * q;
    // a tile past the last one or of no such adapter is left alone
    auto tile_ok = [&](int t) {
      return tile0 + t < tiles && wid_ok(a.plan, a.plan.tile_wid[tile0 + t < tiles ? tile0 + t : tile0]);
    };
    const int at = tile0 * kTileRows + (tile0 + (slot >> 4) < tiles ? slot : slot & 15);
    int row = a.plan.tile_row[at];
    const int seg = a.side_scale ? a.plan.tile_rseg[at] : -1;
    if (!tile_ok(slot >> 4) || n >= a.d_out) row = -1;
    f32x4 part[KS];
#pragma unroll
    for (int z = 0; z < KS; ++z)
      part[z] = ldg_f4((z < P.ksplit && row >= 0) ? P.partial + ((long)z * a.T + row) * a.d_out + n : zf);
    u32x2 second = {0u, 0u};
    if (P.pt_b && row >= 0) second = *reinterpret_cast<const u32x2*>(P.v2 + (long)row * a.d_out + n);
    const float ss = (row >= 0 && a.side_scale) ? a.side_scale[seg] : 1.0f;
    f32x4 sum = part[0];
#pragma unroll
    for (int z = 1; z < KS; ++z) sum += part[z];
    if (row >= 0) store4<DT>(P.out + (long)row * a.d_out + n, sum, 1.0f, a.beta);
    // (from the rounded value, as a reader of `out` would scale it)
    const u32x2 one = {pack2<DT>(sum[0], sum[1]), pack2<DT>(sum[2], sum[3])};
    __syncthreads();  // (the LDS of the previous item is read)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      tr[0][(4 * q + 2 * e) * kTPitch + slot] = (uint16_t)Num<DT>::bits(ss * Num<DT>::lo(one[e]));
      tr[0][(4 * q + 2 * e + 1) * kTPitch + slot] = (uint16_t)Num<DT>::bits(ss * Num<DT>::hi(one[e]));
      tr[1][(4 * q + 2 * e) * kTPitch + slot] = (uint16_t)Num<DT>::bits(ss * Num<DT>::lo(second[e]));
      tr[1][(4 * q + 2 * e + 1) * kTPitch + slot] = (uint16_t)Num<DT>::bits(ss * Num<DT>::hi(second[e]));
    }
    __syncthreads();
    // piece: half a tile; eight neighbouring threads write a line
    const int which = threadIdx.x >> 9, m = (threadIdx.x >> 3 & 56) | (threadIdx.x & 7), piece = threadIdx.x >> 3 & 7;
    uint16_t* pt = which ? P.pt_b : P.pt_a;
    if (pt && n0 + m < a.d_out && tile_ok(piece >> 1)) {
      const uint32_t* src = reinterpret_cast<const uint32_t*>(&tr[which][m * kTPitch + 8 * piece]);
      stg16(pt + side_piece(a.d_out, tile0 + (piece >> 1), n0 + m, piece & 1), u32x4{src[0], src[1], src[2], src[3]});
    }
  }
}

// ------------------------------------------------------------------ expand --
struct ExpandProj {
  uint16_t* y;                // [T, d_out]
  const uint16_t* v;          // [T, d_in]
  const void* const* w_ptrs;  // indexed by the plan's tile_wid
  uint16_t* v_out;            // wave kernels, optional [T, d_in]: copy of v, by row
  const float* vpart;         // VFOLD wave kernels: v arrives as vsplit (1..4) fp32 k-split partials
  int vsplit;                 //   [vsplit, T, d_in], summed here in split order and rounded
  int d_in, d_out, ldw;
  uint16_t* pt_a;             // block kernels, optional: scale*v by tile slot, transposed (side_piece)
  uint16_t* pt_b;             // optional: same treatment of v2 (a second [T, d_in] matrix)
  const uint16_t* v2;
  const uint8_t* drop_bits;   // DROP kernels: keep bits of this projection's mask, by tile slot (tile_bits)
};

constexpr int kMaxVsplit = 4;  // most k-split partials of v the wave kernel folds itself

struct ExpandArgs {
  TileArgs plan;
  ExpandProj p[kMaxProj];
  const float* seg_scale;
  float beta;
  int T, nt_max;
  ItemSpace items;           // chunk rows of projection p: its column chunks
  int w_kn;                  // tile-block kernel only: weights are stored [k][n]
  DropArgs drop;             // DROP kernels (the backward's dX): the mask and factor applied to the stored values
                             //   (probabilities and row count; the keep bits are each projection's own)
};

// by-products one wave per tile writes: scale*v / scale*v2 by tile slot, transposed (side_piece),
// which the weight-gradient kernel reads with the token index innermost
template <int DT>
__device__ __forceinline__ void write_side(const ExpandArgs& a, const ExpandProj& P, int slot, int row,
                                           int kk, u32x4 vf, float scale) {
  const u32x4 zero = {0u, 0u, 0u, 0u};
  const long at = side_piece(P.d_in, slot / kTileRows, kk, slot >> 3 & 1) + (slot & 7);
  u32x4 v2f = zero;
  if (P.pt_b && row >= 0) v2f = ldg16(P.v2 + (long)row * P.d_in + kk);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    P.pt_a[at + 16 * e] = (uint16_t)Num<DT>::bits(scale * Num<DT>::lo(vf[e]));
    P.pt_a[at + 16 * e + 8] = (uint16_t)Num<DT>::bits(scale * Num<DT>::hi(vf[e]));
    if (P.pt_b) {
      P.pt_b[at + 16 * e] = (uint16_t)Num<DT>::bits(scale * Num<DT>::lo(v2f[e]));
      P.pt_b[at + 16 * e + 8] = (uint16_t)Num<DT>::bits(scale * Num<DT>::hi(v2f[e]));
    }
  }
}

// ---- y in full lines ------------------------------------------------------
// The MFMA leaves a tile's accumulators as 64-byte pieces per row (lane (c, g):
// row c, eight columns at 32q + 8g).  y is read and written a full 128-byte line
// per row and instruction instead: lane -> row lane/8 (+8), eight columns at
// (lane%8)*8 of a 64-column half chunk; the accumulators change layout through
// a per-wave LDS area on the way.  Measured on a read-modify-write of gathered
// rows: 4.4 TB/s with 64-byte pieces, 4.8 with full lines.
constexpr int kOPitch = 64 + 4;  // floats: staging rows 4 banks apart, conflict-free both ways

struct LineLane {
  int orow, ocol;     // lane's row (0..7, +8 for the second instruction) and column offset
  int srow[2];        // the two y rows of the lane, -1 = none
  float scale[2];
  uint16_t* yrow[2];  // &y[srow[j]][chunk column + ocol]
  DropRow drop[2];    // DROP kernels: dropout parameters of the two rows ...
  uint32_t keep[2][2];  // ... and the keep bits of their 64-column pieces [h][j]
};

// keep bits of the pieces a lane will store (DROP kernels): requested with the other loads of
// the item; what rows that are not dropped find there is never applied
template <int NQ>
__device__ __forceinline__ void load_keep_bits(LineLane& L, const uint8_t* bits, int tile, int ncol0, int d_out,
                                               const uint16_t* zeros) {
  const int chunks = (d_out + 63) / 64;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int h = 0; h < NQ / 2; ++h) {
      const bool ok = ncol0 + 64 * h < d_out;
      L.keep[h][j] = *(const SMLM_GLOBAL uint8_t*)(
          ok ? bits + tile_bits(tile, ncol0 / 64 + h, chunks, L.orow + 8 * j, L.ocol >> 3)
             : reinterpret_cast<const uint8_t*>(zeros));
    }
}

// y is read and written once per launch, so its accesses are marked non-temporal: left to the
// default policy its lines crowd the weights out of L2 and leave dirty lines behind that the next
// launch has to wait for (measured: 4-12 % of a step on the large batches, 3.5 % on the decode
// step).  A reader that follows at once is not slowed down as long as the data fits the caches
// (measured with a writer / reader pair: 2 and 8 MB read back equally fast, 32 MB 9 % slower).
template <int NQ>
__device__ __forceinline__ void load_y_lines(u32x4 (&yold)[NQ / 2][2], const LineLane& L, int ncol0, int d_out,
                                             bool read_y, const uint16_t* zeros) {
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int h = 0; h < NQ / 2; ++h)
      yold[h][j] = ldg16_or_nt(L.yrow[j] + 64 * h, read_y && L.srow[j] >= 0 && ncol0 + 64 * h + L.ocol < d_out, zeros);
}

// DROP: what is stored is the gradient with respect to x before its dropout: the value as it
// would be stored otherwise, times the row's factor where the element was kept, zero elsewhere
template <int DT, int NQ, bool DROP = false>
__device__ __forceinline__ void store_y_lines(float* stg, const f32x4 (&acc)[NQ][2], const u32x4 (&yold)[NQ / 2][2],
                                              const LineLane& L, int c, int g, int ncol0, int d_out, float beta) {
#pragma unroll
  for (int h = 0; h < NQ / 2; ++h) {
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
      *reinterpret_cast<f32x4*>(&stg[c * kOPitch + 32 * qq + 8 * g]) = acc[2 * h + qq][0];
      *reinterpret_cast<f32x4*>(&stg[c * kOPitch + 32 * qq + 8 * g + 4]) = acc[2 * h + qq][1];
    }
    // a wave's own LDS accesses are served in order; the compiler must keep them in order too
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    f32x4 lo4[2], hi4[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      lo4[j] = *reinterpret_cast<const f32x4*>(&stg[(L.orow + 8 * j) * kOPitch + L.ocol]);
      hi4[j] = *reinterpret_cast<const f32x4*>(&stg[(L.orow + 8 * j) * kOPitch + L.ocol + 4]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (L.srow[j] < 0 || ncol0 + 64 * h + L.ocol >= d_out) continue;
      const u32x4 old = yold[h][j];
      const float sc = L.scale[j];
      u32x4 o;
      if (beta != 0.0f) {
        o[0] = pack2<DT>(beta * Num<DT>::lo(old[0]) + sc * lo4[j][0], beta * Num<DT>::hi(old[0]) + sc * lo4[j][1]);
        o[1] = pack2<DT>(beta * Num<DT>::lo(old[1]) + sc * lo4[j][2], beta * Num<DT>::hi(old[1]) + sc * lo4[j][3]);
        o[2] = pack2<DT>(beta * Num<DT>::lo(old[2]) + sc * hi4[j][0], beta * Num<DT>::hi(old[2]) + sc * hi4[j][1]);
        o[3] = pack2<DT>(beta * Num<DT>::lo(old[3]) + sc * hi4[j][2], beta * Num<DT>::hi(old[3]) + sc * hi4[j][3]);
      } else {
        o[0] = pack2<DT>(sc * lo4[j][0], sc * lo4[j][1]);
        o[1] = pack2<DT>(sc * lo4[j][2], sc * lo4[j][3]);
        o[2] = pack2<DT>(sc * hi4[j][0], sc * hi4[j][1]);
        o[3] = pack2<DT>(sc * hi4[j][2], sc * hi4[j][3]);
      }
      if (DROP) o = drop8_bits<DT>(o, L.drop[j], L.keep[h][j]);
      stg16_nt(L.yrow[j] + 64 * h, o);
    }
  }
}

// Expand, one tile per work item (small batches, decode): work item -> (projection,
// column chunk, tile); each wave of the workgroup owns 32*NQ output columns and
// loads its weight fragments straight into registers.  K (= LoRA rank) is
// short: KS > 0 unrolls KS 32-wide k steps, KS == 0 is the general loop over k.
// Bound by the chain of dependent loads (tile -> adapter and row numbers -> y, v, weights): the weights need the
// adapter alone and up to rank 32 (KS = 1) are requested ahead of the row numbers' arrival.  Whole forward, us, weights
// after the row numbers / before: six times q/k/v/o of 256 decoded rows at rank 16 from a graph 114.1 / 111.1, one
// projection of 64 decoded rows 10.0 / 9.0, 600 rows in four segments 10.8 / 10.0.  At KS = 2 the registers cost more
// than it gains where there are many workgroups (rank 40, twice 4096 -> 11008, 200 decoded rows: 28.1, the first step
// ahead 29.3, both 29.2), and above rank 64 the loop's first step ahead gained nothing (13.3 / 13.8).
// MFMA row m of column block (q,p) is output column 32q + 8(m/4) + 4p + m%4, so
// that a lane's eight accumulators for one q are eight consecutive columns.
template <int DT, int NQ, int KS, bool DIRECT, bool VFOLD>
// KS == 0 with the fold: two workgroups a CU at most.  Its registers would allow three, and launches of up to two
// workgroups a CU then come to lie three on some CUs and one on others (512 workgroups, q/k/v/o of 256 rows in two
// segments: rank 72 28.7 -> 25.9 us, rank 128 41.6 -> 34.8, rank 256 71.7 -> 58.4; 1024 workgroups, 256 decoded rows:
// 51.8 -> 52.6, 66.7 -> 68.6, 133.2 -> 133.0).
__global__ __launch_bounds__(kFwdThreads) __attribute__((amdgpu_waves_per_eu(1, KS == 0 && VFOLD ? 2 : 8)))
void expand_wave_kernel(ExpandArgs a) {
  __shared__ __attribute__((aligned(16))) float olds[kFwdWaves][kTileRows * kOPitch];
  const int units = DIRECT ? 0 : tile_units<1>(a.plan, 0);
  const WorkRange wr = item_range<DIRECT>(a.items, units);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const int mrow = 8 * (c >> 2) + (c & 3);  // column offset of MFMA row c inside a (q,p) block
  constexpr int KSU = KS > 0 ? KS : 1;

  for (int V = wr.first; V < wr.last; V += wr.step) {
    int pj, yy, tile;
    if (!item_get<DIRECT>(a.items, V, units, &pj, &yy, &tile)) break;
    const ExpandProj P = a.p[pj];
    if (!P.y) continue;  // a projection this call leaves out (uniform over the workgroup)
    const int ncol0 = (yy * kFwdWaves + wave) * 32 * NQ;
    if (ncol0 >= P.d_out) continue;
    const int wid = uload(a.plan.tile_wid, tile);
    if (!wid_ok(a.plan, wid)) continue;  // past the last tile (direct mode), or no such adapter
    const uint16_t* W = uload_ptr(P.w_ptrs, wid);
    const int klim = rank_limit(a.plan, wid, P.d_in);  // k at or past it: zero padding of v and the weights
    const int ldw = rank_ld(a.plan, P.ldw, klim);
    const int slot = tile * kTileRows + c;
    const int row = a.plan.tile_row[slot];
    const bool side = (yy == 0 && wave == 0);  // the one wave per tile that writes the caller's copy of v
    const uint16_t* zeros = reinterpret_cast<const uint16_t*>(a.plan.hdr + kHdrZeros);

    // Every load of the item is issued before anything waits for one: the old values of the
    // y rows this lane will update, the weight fragments and v (predicated-off loads read
    // zeros instead of being patched afterwards, which would make the wave wait in between).
    LineLane L;
    L.orow = lane >> 3;
    L.ocol = (lane & 7) * 8;
    int sseg[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      L.srow[j] = a.plan.tile_row[tile * kTileRows + L.orow + 8 * j];
      sseg[j] = a.seg_scale ? a.plan.tile_rseg[tile * kTileRows + L.orow + 8 * j] : -1;
    }
    u32x4 wf[NQ][2];
    auto load_w = [&](int ks) {
      const int kk = 32 * ks + 8 * g;
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int n = ncol0 + 32 * q + 4 * p + mrow;
          wf[q][p] = ldg16_or(W + (long)n * ldw + kk, kk < klim && n < P.d_out, zeros);
        }
    };
    if (KS == 1) {
      load_w(0);
      __builtin_amdgcn_sched_barrier(0);  // the weights are on their way before the row numbers are waited for
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      L.yrow[j] = P.y + (long)(L.srow[j] < 0 ? 0 : L.srow[j]) * P.d_out + ncol0 + L.ocol;
    }
    u32x4 yold[NQ / 2][2];
    load_y_lines<NQ>(yold, L, ncol0, P.d_out, a.beta != 0.0f, zeros);
#pragma unroll
    for (int j = 0; j < 2; ++j) L.scale[j] = sseg[j] >= 0 ? a.seg_scale[sseg[j]] : 1.0f;

    f32x4 acc[NQ][2];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q][0] = acc[q][1] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int nks = KS > 0 ? KS : (P.d_in + 31) / 32;
#pragma unroll KSU
    for (int ks = 0; ks < nks; ++ks) {
      const int kk = 32 * ks + 8 * g;
      const bool kin = kk < P.d_in, kreal = kk < klim;
      if (KS != 1) load_w(ks);
      u32x4 vf;
      const bool vok = kreal && row >= 0;
      if (VFOLD) {  // fold (and round) the shrink's fp32 partial sums as its fold launch would
        const float* zf = reinterpret_cast<const float*>(zeros);
        f32x4 part[kMaxVsplit][2];
#pragma unroll
        for (int z = 0; z < kMaxVsplit; ++z) {
          const bool ok = vok && z < P.vsplit;
          const float* pz = ok ? P.vpart + ((long)z * a.T + row) * P.d_in + kk : zf;
          part[z][0] = ldg_f4(pz);
          part[z][1] = ldg_f4(ok ? pz + 4 : zf);
        }
        f32x4 s0 = part[0][0], s1 = part[0][1];
#pragma unroll
        for (int z = 1; z < kMaxVsplit; ++z) s0 += part[z][0], s1 += part[z][1];  // + 0.0 past vsplit
        vf = u32x4{pack2<DT>(s0[0], s0[1]), pack2<DT>(s0[2], s0[3]), pack2<DT>(s1[0], s1[1]),
                   pack2<DT>(s1[2], s1[3])};
      } else {
        vf = ldg16_or(P.v + (long)row * P.d_in + kk, vok, zeros);
      }
      if (side && kin && P.v_out && row >= 0) stg16(P.v_out + (long)row * P.d_in + kk, vf);
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int p = 0; p < 2; ++p) acc[q][p] = Num<DT>::mfma(wf[q][p], vf, acc[q][p]);
    }
    store_y_lines<DT, NQ>(olds[wave], acc, yold, L, c, g, ncol0, P.d_out, a.beta);
  }
}

// Expand, one tile BLOCK per work item (prefill / fine-tuning batches): work item
// -> (projection, column chunk of 32*NQ columns, tile block).  The workgroup
// stages the chunk's weight rows in LDS once; wave w then multiplies tile w of
// the block with them, so an adapter's B chunk is read from L2 once per four
// tiles instead of once per tile.
// WKN: weights stored [k][n] (A [r, h_in] for the backward's dX = dV A): the chunk is staged
// as it lies in memory and read out of LDS with the transposing read.
// K (= LoRA rank): up to 32*KS in one piece; KS = 4 serves every rank above 64, 128 of k at a time, the
// next piece on its way while one is multiplied.
template <int NQ, int KS, bool WKN>
struct ExpandBlockLds {
  static constexpr int kPitch = WKN ? 32 * NQ + 8 : 32 * KS + 8;  // LDS row pitch in 16-bit elements
  // the staged weights and the area the accumulators change layout in share their LDS (the
  // weights are done with when the accumulators are complete): five workgroups fit a CU at rank 64 too
  static constexpr int kWBytes = (WKN ? 32 * KS : 32 * NQ) * kPitch * 2;
  static constexpr int kOBytes = kFwdWaves * kTileRows * kOPitch * 4;
  static constexpr int kBytes = kWBytes > kOBytes ? kWBytes : kOBytes;
};

// column chunk yy of projection pj, tile block tb; smem: ExpandBlockLds
template <int DT, int NQ, int KS, bool WKN, bool DROP>
__device__ __forceinline__ void expand_block_item(const ExpandArgs& a, int pj, int yy, int tb, char* smem) {
  static_assert(NQ % 2 == 0, "the output is written 64 columns at a time");
  constexpr int kPitch = ExpandBlockLds<NQ, KS, WKN>::kPitch;
  uint16_t* wlds = reinterpret_cast<uint16_t*>(smem);
  float(*olds)[kTileRows * kOPitch] = reinterpret_cast<float(*)[kTileRows * kOPitch]>(smem);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const int mrow = 8 * (c >> 2) + (c & 3);
  const ExpandProj P = a.p[pj];
  if (!P.y) return;  // a projection this call leaves out (uniform over the workgroup)
  const int ncol0 = yy * 32 * NQ;
  if (ncol0 >= P.d_out) return;  // a chunk row added to round the count up (uniform over the workgroup)
  const int packed = uload(a.plan.blk, tb);
  const int t0 = packed >> 3, cnt = packed & 7;
  if (cnt == 0) return;  // past the last block (direct mode); uniform over the workgroup
  const int wid = uload(a.plan.tile_wid, t0);
  if (!wid_ok(a.plan, wid)) return;  // a negative adapter id (rows that no adapter serves) or one past the tables
  const uint16_t* W = uload_ptr(P.w_ptrs, wid);
  const int klim = rank_limit(a.plan, wid, P.d_in);  // k at or past it: zero padding of v and the weights
  const int ldw = WKN ? P.ldw : rank_ld(a.plan, P.ldw, klim);  // [k][n] weights (A) have whole rows per rank
  const bool active = wave < cnt;
  const int tslot = (t0 + (active ? wave : 0)) * kTileRows;
  const int slot = tslot + c;
  const int row = active ? a.plan.tile_row[slot] : -1;  // row of the MFMA column this lane feeds
  LineLane L;  // rows this lane reads and writes in y
  L.orow = lane >> 3;
  L.ocol = (lane & 7) * 8;
  int sseg[2], dseg[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    L.srow[j] = active ? a.plan.tile_row[tslot + L.orow + 8 * j] : -1;
    sseg[j] = (a.seg_scale && active) ? a.plan.tile_rseg[tslot + L.orow + 8 * j] : -1;  // -1 on empty slots
    L.yrow[j] = P.y + (long)(L.srow[j] < 0 ? 0 : L.srow[j]) * P.d_out + ncol0 + L.ocol;
    dseg[j] = DROP ? a.plan.tile_rseg[tslot + L.orow + 8 * j] : -1;
  }
  const uint16_t* zeros = reinterpret_cast<const uint16_t*>(a.plan.hdr + kHdrZeros);

  // Every load of the item is issued before anything waits for one (predicated-off loads
  // read zeros instead of being patched afterwards).
  // weight chunk -> registers (written to LDS below): 32*NQ rows of 4*KS 16-byte pieces
  constexpr int kPieces = 32 * NQ * 4 * KS;
  constexpr int kPer = (kPieces + kFwdThreads - 1) / kFwdThreads;
  constexpr int kK = 32 * KS;  // k of one piece
  constexpr bool kLoop = KS > 2;
  u32x4 stage[kPer], vf[KS];
  auto load_stage = [&](int k0) {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int idx = threadIdx.x + j * kFwdThreads;
      if (WKN) {
        const int kl = k0 + idx / (4 * NQ), n8 = (idx % (4 * NQ)) * 8;
        stage[j] = ldg16_or(W + (long)kl * ldw + ncol0 + n8,
                            idx < kPieces && ncol0 + n8 < P.d_out && kl < klim, zeros);
      } else {
        const int nl = idx / (4 * KS), k8 = k0 + (idx % (4 * KS)) * 8;
        stage[j] = ldg16_or(W + (long)(ncol0 + nl) * ldw + k8,
                            idx < kPieces && ncol0 + nl < P.d_out && k8 < klim, zeros);
      }
    }
  };
  auto load_v = [&](int k0) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kk = k0 + 32 * ks + 8 * g;
      vf[ks] = ldg16_or(P.v + (long)row * P.d_in + kk, kk < klim && row >= 0, zeros);
    }
  };
  load_stage(0);
  const bool read_y = a.beta != 0.0f;
  u32x4 yold[NQ / 2][2];
  load_y_lines<NQ>(yold, L, ncol0, P.d_out, read_y, zeros);
  if (DROP) load_keep_bits<NQ>(L, P.drop_bits, tslot / kTileRows, ncol0, P.d_out, zeros);
  load_v(0);
  float prob[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) prob[j] = DROP ? drop_prob(a.drop, L.srow[j], dseg[j], zeros) : 0.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j) L.scale[j] = (sseg[j] >= 0 && L.srow[j] >= 0) ? a.seg_scale[sseg[j]] : 1.0f;

  f32x4 acc[NQ][2];
#pragma unroll
  for (int q = 0; q < NQ; ++q) acc[q][0] = acc[q][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int k0 = 0;; k0 += kK) {
    // (opaque: the compiler otherwise keeps an induction register pair for each of a hundred addresses)
    if (kLoop) asm volatile("" : "+s"(k0));
    __syncthreads();  // every wave is done reading the previous piece's (or item's) weights
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int idx = threadIdx.x + j * kFwdThreads;
      const int r_ = WKN ? idx / (4 * NQ) : idx / (4 * KS);
      const int c_ = WKN ? (idx % (4 * NQ)) * 8 : (idx % (4 * KS)) * 8;
      if (idx < kPieces) *reinterpret_cast<u32x4*>(&wlds[r_ * kPitch + c_]) = stage[j];
    }
    __syncthreads();
    // (waves without a tile multiply zeros: whole waves only, MFMA runs with every lane, and every
    // wave reaches the barriers)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          u32x4 wf;
          if (WKN) {
            // lane c names k row 32ks + 8g (+4) + c/4 and columns 32q + 4p + 8(c%4) .. +3; it
            // receives column 32q + 4p + 8(c/4) + c%4 (its MFMA row's column) of four k rows
            const uint16_t* base = &wlds[(32 * ks + 8 * g + (c >> 2)) * kPitch + 32 * q + 4 * p + 8 * (c & 3)];
            const u32x2 q0 = lds_read_tr16(base), q1 = lds_read_tr16(base + 4 * kPitch);
            wf = u32x4{q0[0], q0[1], q1[0], q1[1]};
          } else {
            wf = *reinterpret_cast<const u32x4*>(&wlds[(32 * q + 4 * p + mrow) * kPitch + 32 * ks + 8 * g]);
          }
          acc[q][p] = Num<DT>::mfma(wf, vf[ks], acc[q][p]);
        }
      // (the weight fragments of one k step at a time: all of them at once do not fit the registers)
      if (kLoop) __builtin_amdgcn_sched_barrier(0);
    }
    if (!kLoop || k0 + kK >= P.d_in) break;  // uniform over the workgroup
    load_stage(k0 + kK);
    load_v(k0 + kK);
  }

  __syncthreads();  // every wave has read its weights: the area is free for the accumulators
#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (DROP) L.drop[j] = drop_params(prob[j]);
  if (active) store_y_lines<DT, NQ, DROP>(olds[wave], acc, yold, L, c, g, ncol0, P.d_out, a.beta);
  if (P.pt_a && yy == 0 && active) {  // by-products for the backward, when no fold has written them
    const int rseg = a.seg_scale ? a.plan.tile_rseg[slot] : -1;
    const float side_scale = (rseg >= 0 && row >= 0) ? a.seg_scale[rseg] : 1.0f;
#pragma unroll 1
    for (int kk = 8 * g; kk < P.d_in; kk += 32)
      write_side<DT>(a, P, slot, row, kk, ldg16_or(P.v + (long)row * P.d_in + kk, kk < klim && row >= 0, zeros),
                     side_scale);
  }
}

template <int DT, int NQ, int KS, bool DIRECT, bool WKN, bool DROP = false>
// (five workgroups a CU instead of the four the compiler's own register budget gives: more y
// lines in flight per CU; worth 2 % on the prefill launch and 6 % on the fine-tune one)
// KS = 4: bound by HBM like the others (2064 rows, two projections 4096 -> 4096 at rank 128: 21.6 us for 80 MB, and
// the backward's dX 17.9 us for 46 MB, where the one-tile kernel's loop over k took 50.8 and 43.5 us: it fetched the
// weights once per 16 rows).  Four waves a SIMD spill (37.1 / 20.6 us), 64 columns a workgroup 24.0 / 18.0.
__global__ __launch_bounds__(kFwdThreads)
__attribute__((amdgpu_waves_per_eu(DIRECT ? ((KS > 2 || NQ > 4) ? 3 : 5) : 1)))
void expand_block_kernel(ExpandArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[ExpandBlockLds<NQ, KS, WKN>::kBytes];
  const int units = DIRECT ? 0 : tile_units<kBlkTiles>(a.plan, 0);
  const WorkRange wr = item_range<DIRECT>(a.items, units);
  for (int V = wr.first; V < wr.last; V += wr.step) {
    int pj, yy, tb;
    if (!item_get<DIRECT>(a.items, V, units, &pj, &yy, &tb)) break;
    expand_block_item<DT, NQ, KS, WKN, DROP>(a, pj, yy, tb, smem);
  }
}

}  // namespace smlm
