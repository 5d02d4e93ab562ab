// On-chip row scan of one keyroot-pair table per workgroup (gfx950, wave64).
//
// The recurrence, the orientation (rows = the short side) and the far rows in
// LDS slots are those of forest.hip's header. What this kernel does with them:
//
// Dominance form. With t = cmax-1-c and k the row index from the bottom, let
// G[k][t] = F - t - k (under a cost model F - Q(c) - V(k), Q and V the summed
// costs of the columns right of c and of the rows below and at k). Both the
// horizontal step (F[r][c+1] + cost) and the vertical one (F[r+1][c] + cost)
// leave G unchanged, so
//   G[k][t] = min over k' <= k, t' <= t of d[k'][t'] and of the boundary,
// d being the far (or, on tree cells, diagonal) term in the same coordinates.
// So a row that nobody reads as a row costs no scan at all: its terms only
// lower the per-column minima A[t] = min over k' <= k of d[k'][t]. The prefix
// minimum over t is formed on the rows whose values are needed ("full" rows):
// those saved to a slot (the row after a leaf), tree rows, and the row before
// a tree row (the diagonal). Integer minima re-associate exactly.
//
// Waves as a pipeline. Columns are cut into blocks of 64*C, one wave each,
// block 0 at the right edge. A block depends only on blocks before it, so no
// barrier orders the waves: wave w takes from wave w-1, through a ring of
// kEdgeRows entries in LDS (the edge), one entry per full row: the scan carry
// (the minimum over all earlier columns) and, for a saved row, the far values
// of earlier blocks that this block or a later one reads: one per nesting
// depth of the column keyroot's right paths, since the paths that cross a
// block edge nest. Each wave keeps its own far columns and those imports in
// its own segment of every slot row, so slots are never shared. The waves
// agree on progress every kSyncRows rows: a wave starts such a group once the
// wave before has finished it and the wave after has taken enough entries.
// DS operations of a wave are performed in program order and those of a
// compute unit in one global order, so the progress word, written after a
// group's entries, publishes them. With a barrier per row all waves paid the
// slowest wave's row plus the barrier; here rows take the time of one wave's
// own row.
//
// What bounds a row. A lone wave issues an instruction every 6 to 8 cycles
// whatever its kind, a dependent LDS read takes 52, a DPP scan step 16, a
// branch 15 (not taken) to 25 (taken); LDS writes of many lanes to one address
// cost the same as any. So the row loop spends instructions, not bytes: no
// branch depends on lanes (columns without a value to save write a sink entry,
// lanes outside a table store out of the buffer's range), rows past the
// table's end run as plain rows, and the edges cost one LDS read and one write
// a row.
//
// Measured, us per row of the root table of 1000-node deep / wide pairs, best
// form of a scan over every row with a barrier per row against this kernel's 8
// waves of 2 columns per lane: 0.40 / 0.44 against 0.21 / 0.28. Many tables at
// once (the 4096-pair batch, one stream): one wave of 16 columns 27.3 against
// 24.4 ms, of 8 18.5 against 16.2, 8 waves of 2 16.2 against 7.4; those are
// bound by TD traffic (about 2 bytes a cell, 4 TB/s over the batch's streams).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "kernels.hpp"
#include "wave.hpp"

namespace xted {

// A row's first metadata word: the byte offset of its far slot row (below
// 2^18) and flags. Its second word: the byte offset of the slot row it is
// saved to.
constexpr int32_t kRowSlot = 0x3FFFF;
constexpr int32_t kRowTree = 1 << 28;
constexpr int32_t kRowFull = 1 << 29;
constexpr int32_t kRowSaved = 1 << 30;

// Polls of a neighbour's progress before a wave gives up (never reached: the
// waves of a workgroup are resident together and wait only on the wave before
// or after them).
constexpr int kEdgePolls = 1 << 24;
constexpr int kSyncRows = 4;
static_assert(kEdgeRows == 2 * kSyncRows, "a wave may fill one group while the next takes another");

// Bytes of a TD buffer resource, from kTdPad entries before the table: more
// than any table and its padding (32767^2 entries of 2 bytes), and as an
// offset out of range whatever scalar offset (below it) is added.
constexpr int32_t kTdBytes = (int32_t)0x80000000u;

// Compiler ordering of this wave's LDS operations (the hardware keeps it).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

template <int W, int C, bool kCost>
__global__ __launch_bounds__(64 * W) void scan_kernel(DPArgs A) {
  // TD ring slots: a power of two dividing 64.
  constexpr int S = C >= 16 || (W == 1 && C >= 8) ? 4 : 8;
  constexpr int PD = S - 1;                    // rows of TD prefetched
  constexpr int NW = C == 1 ? 1 : C / 2;       // words of one row: two 16-bit entries each
  constexpr int D = kEdgeRows;
  extern __shared__ __align__(16) unsigned char lds[];

  // Workgroups go round robin over the 8 XCDs, each with its own L2; task
  // order keeps a pair's tables together, so kXcdRun consecutive tasks are
  // given to one XCD (the last, partial span keeps its order). The 4096-pair
  // batch ran 101.6 ms without, 100.1 with 16, 101.0 with 64, 104.8 with 256.
  constexpr uint32_t kXcds = 8, kXcdRun = 16, kSpan = kXcds * kXcdRun;
  uint32_t ix = blockIdx.x;
  if ((ix | (kSpan - 1)) < (uint64_t)A.ntasks)
    ix = (ix & ~(kSpan - 1)) + (ix % kXcds) * kXcdRun + (ix % kSpan) / kXcds;
  if ((int64_t)ix >= A.ntasks) return;
  const TaskDesc dsc = A.descs[ix];
  const bool rows_x = dsc.base_rx < 0;
  const int64_t offR = dsc.offR;
  const int64_t offC = dsc.offC;
  const NodeRec* __restrict__ rrecR = A.pool.rrec + offR;
  const NodeRec* __restrict__ crecC = A.pool.crec + offC;
  const int32_t* __restrict__ lrankC = A.pool.lrank + offC;
  const int32_t r0 = dsc.r0, c0 = dsc.c0;
  td_t* const TDo = A.td + dsc.tdo;  // [r][c]
  td_t* const TDt = A.td + dsc.tdt;  // [c][r]
  const int64_t ldo = dsc.ldo;
  const uint32_t ldt = (uint32_t)dsc.ldt;
  const int32_t rmax = dsc.rmax, cmax = dsc.cmax;
  const int32_t ncols = cmax - c0;
  const int32_t nrows = rmax - r0;
  const int32_t base = dsc.base_rx & 0x7FFFFFFF;
  const int32_t orl_c0 = cmax - 1;

  // Uniform over the wave, so it lives in a scalar register.
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int lane = threadIdx.x & 63;
  const int32_t tb = wave * 64 * C;      // first t of this wave's block
  const int32_t tlane = tb + lane * C;   // t of this lane's element 0
  const int32_t nw = W > 1 ? (ncols + 64 * C - 1) / (64 * C) : 1;  // waves with columns

  // Costs (kCost). Hpre / Vpre: prefix sums of the horizontal (column) and
  // vertical (row) edit costs over the column and row trees: insertions and
  // deletions when the rows are x, the other way round when they are y.
  // Q(c) = Hpre[cmax-1] - Hpre[c] takes the place of t, V(k) = Vpre[rmax] -
  // Vpre[r] that of k (with unit costs Q(c) = t and V(k) = k + 1; those forms
  // shift by k).
  const int32_t* __restrict__ Hpre = nullptr;
  const int32_t* __restrict__ Vpre = nullptr;
  int32_t hq = 0, hc = 0, vr = 0;
  if constexpr (kCost) {
    Hpre = (rows_x ? A.pool.pins : A.pool.pdel) + offC;
    Vpre = (rows_x ? A.pool.pdel : A.pool.pins) + offR;
    hq = Hpre[cmax - 1];
    hc = Hpre[cmax];
    vr = Vpre[rmax];
  }
  // The boundary column c = cmax in G's coordinates, the same on every row.
  const int32_t cin0 = kCost ? hc - hq : 2;

  // LDS (dynamic only, so that it starts at byte 0 and an offset is an
  // address): the progress words, wave w's at w + 1 as {rows done, full rows
  // done}, with words that never hold anyone up before wave 0 and after the
  // last wave; then W + 1 edges (wave w reads edge w and writes edge w + 1;
  // edge 0 holds the boundary's carry), then the slot rows. An edge entry:
  // word 0 the carry, word 1 + d the import of depth d, word 1 + kds trash. A
  // slot row holds one segment per wave: its own far columns (leaves but the
  // table's last, by leaf rank), at index wb the boundary value F[R][cmax]
  // that tree columns read, the kds imports (W > 1) and a sink that columns
  // saving nothing write.
  const int32_t lbase0 = dsc.lbase;
  const int32_t ltop = lrankC[cmax - 1];
  int32_t lbase = lbase0, wb = ltop - lbase0, seg = 0, kds = 0, kdep_c0 = 0;
  if constexpr (W > 1) {
    const int32_t chi = max(cmax - 1 - tb, c0);
    const int32_t clo = max(c0, cmax - tb - 64 * C);
    const int32_t lhi = lrankC[chi];
    lbase = lrankC[max(clo - 1, c0)];
    wb = max(0, lhi - lbase);
    kds = A.pool.kdn[offC + c0] + 1;
    kdep_c0 = A.pool.kdep[offC + c0];
    seg = (ltop - lhi) + wave * (2 + kds);
  }
  const uint32_t entry_bytes = W > 1 ? 4u * (uint32_t)(kds + 2) : 0u;
  const uint32_t edge_bytes = D * entry_bytes;
  constexpr uint32_t edges = W > 1 ? 8u * (W + 2) : 0u;  // byte offset of edge 0
  const uint32_t slot_base = edges + (W > 1 ? (W + 1) * edge_bytes : 0u) + 2u * (uint32_t)seg;
  const uint32_t row_bytes = 2u * (uint32_t)((ltop - lbase0) + W * (2 + kds));
  const int32_t sinkix = wb + 1 + kds;
  auto l16 = [&](uint32_t byte) -> uint16_t& { return *reinterpret_cast<uint16_t*>(lds + byte); };
  auto l32 = [&](uint32_t byte) -> int32_t& { return *reinterpret_cast<int32_t*>(lds + byte); };
  auto prog = [&](int w) { return reinterpret_cast<unsigned long long*>(lds + 8 * w); };
  if constexpr (W > 1) {
    if (threadIdx.x < D) l32(edges + threadIdx.x * entry_bytes) = cin0;
    if (threadIdx.x < W + 2) {
      const int w = (int)threadIdx.x - 1;
      *prog((int)threadIdx.x) = w < 0 || w >= nw ? 0x7FFFFFFF7FFFFFFFull : 0ull;
    }
    __syncthreads();
    if (wave >= nw) return;
  }
  const bool more = W > 1 && wave + 1 < nw;

  // Per-column state, element e (t = tlane + e, c = cmax-1-t).
  //   tcol: a tree column (orl_C(c) == orl_C(c0));
  //   lb:   on a tree column its label (tree cells only), else the far value
  //         on the boundary row F[rmax][orl_C(c)+1];
  //   foff: byte offset of the column's far value in this wave's segment;
  //   woff: byte offset it is saved at (c-1 a leaf of subtree(c0)), or the
  //         sink;
  //   xoff: (W > 1) byte offset in an edge entry: for a saved column whose
  //         right path's top keyroot lies in a later block the import word of
  //         the path's depth, else the trash word;
  //   Am:   the running minima A[t], shifted by T = tlane with unit costs
  //         (the per-column term -t + T is then the inline constant -e);
  //   negt: (kCost) the column's -Q(c).
  // Columns past the table (t >= ncols) come after every real column in the
  // scan order, so whatever they hold never reaches a real column; only
  // their stores are masked.
  bool tcol[C];
  uint32_t tmask = 0;  // bit e: some lane's element e is a tree column of the table
  int32_t lb[C], Am[C];
  uint32_t foff[C], woff[C];
  uint32_t tdq[S][NW];
  int32_t negt[kCost ? C : 1];
  uint32_t xoff[W > 1 ? C : 1];
  auto term = [&](int e) -> int32_t {
    if constexpr (kCost) return negt[e];
    else return -e;
  };
  const int32_t T = kCost ? 0 : tlane;
  // The columns' records are read 8 at a time and pinned, so that each is one
  // 16-byte load in flight with the others (unpinned, the compiler splits them
  // into loads of single fields in branches on lanes, each waiting for the one
  // before).
  constexpr int B = C < 8 ? C : 8;
#pragma unroll
  for (int e0 = 0; e0 < C; e0 += B) {
    NodeRec cl[B], rl[W > 1 ? B : 1];  // as a table column; (W > 1) as a row: kdep of c and c-1
    int32_t ul[W > 1 ? B : 1];         // (W > 1) the keyroot at the top of c-1's right path
    CostRec ll[kCost ? B : 1];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int32_t c = max(cmax - 1 - (tlane + e0 + b), c0);
      cl[b] = crecC[c];
      if constexpr (W > 1) {
        rl[b] = A.pool.rrec[offC + c];
        ul[b] = A.pool.rtop[offC + max(c - 1, c0)];
      }
      if constexpr (kCost) ll[b] = A.pool.ccrec[offC + c];
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int e = e0 + b;
      asm volatile("" : "+v"(cl[b].orl), "+v"(cl[b].label), "+v"(cl[b].x), "+v"(cl[b].y));
      if constexpr (W > 1) asm volatile("" : "+v"(rl[b].x), "+v"(rl[b].y), "+v"(ul[b]));
      if constexpr (kCost)
        asm volatile("" : "+v"(ll[b].del), "+v"(ll[b].ins), "+v"(ll[b].del_end),
                     "+v"(ll[b].ins_end));
      const int32_t t = tlane + e;
      const int32_t c = max(cmax - 1 - t, c0);
      // orl(c), label, leaf rank at orl(c), leaf rank of c-1 (bit 31: c-1 is a
      // leaf; only read when c > c0).
      const NodeRec cr = cl[b];
      const int32_t oc = cr.orl;
      const bool tree = oc == orl_c0;
      tcol[e] = tree;
      if (C >= 4) tmask |= (__ballot(tree & (t < ncols)) != 0 ? 1u : 0u) << e;
      int32_t hcol = 0, hfar = 0;  // (kCost) the horizontal sums at c and at orl(c) + 1
      if constexpr (kCost) {
        const CostRec cc = ll[b];
        hcol = rows_x ? cc.ins : cc.del;
        hfar = rows_x ? cc.ins_end : cc.del_end;
        negt[e] = hcol - hq;
        // Opaque to the optimiser, so that sums with it stay three-operand
        // adds (v_add3_u32) instead of becoming an add and a subtract.
        asm("" : "+v"(negt[e]));
      }
      lb[e] = tree ? cr.label : kCost ? hc - hfar : cmax - oc - 1;
      const bool writes = (t < ncols) & (c > c0) & (cr.y < 0);
      int32_t fi = tree ? wb : cr.x - lbase;
      if constexpr (W > 1) {
        const NodeRec rr = rl[b];  // x, y: kdep of c and of c-1
        if (!tree & (cmax - 2 - oc < tb)) fi = wb + 1 + (rr.x - kdep_c0);
        const int32_t u = ul[b];
        const bool out = writes & more & (cmax - 1 - u >= tb + 64 * C);
        xoff[e] = 4u * (uint32_t)(1 + (out ? (rr.y & 0x7FFFFFFF) - kdep_c0 : kds));
        if (t >= ncols) fi = wb;  // never used; inside the segment
      }
      foff[e] = slot_base + 2u * (uint32_t)fi;
      woff[e] = slot_base + 2u * (uint32_t)(writes ? (cr.y & 0x7FFFFFFF) - lbase : sinkix);
      Am[e] = cin0 + T;
    }
  }

  // TD row rr of this lane's columns: entry k of the group (column off + k)
  // is half k & 1 of word k / 2. Read through a buffer resource over the
  // table (its kTdPad entries of padding included): the row offset is a
  // scalar and each lane's column offset a VGPR fixed for the whole table.
  // Loads are unconditional, so the compiler never waits for them inside a
  // branch: a lane with no valid column reads C entries from column c0
  // instead, a partly valid one up to C-1 entries before column c0 (both
  // inside the kTdPad entries around every table).
  const __amdgpu_buffer_rsrc_t tdrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)(TDo - kTdPad), 0, kTdBytes, kBufferWord3);
  const __amdgpu_buffer_rsrc_t ttrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)TDt, 0, kTdBytes, kBufferWord3);
  const int32_t roff =
      ((tlane < ncols ? cmax - C - tlane : c0) + kTdPad) * (int32_t)sizeof(td_t);
  auto load_row = [&](int32_t rr, uint32_t* out) {
    // rr * ldo < 2^30 entries (trees of at most 32767 nodes): an unsigned
    // 32-bit byte offset.
    const int32_t so = (int32_t)((uint32_t)rr * (uint32_t)ldo * (uint32_t)sizeof(td_t));
    if constexpr (C >= 8) {
#pragma unroll
      for (int g = 0; g < C / 8; ++g) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(tdrs, roff + 16 * g, so, 0);
        out[4 * g + 0] = v.x;
        out[4 * g + 1] = v.y;
        out[4 * g + 2] = v.z;
        out[4 * g + 3] = v.w;
      }
    } else if constexpr (C == 4) {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(tdrs, roff, so, 0);
      out[0] = v.x;
      out[1] = v.y;
    } else if constexpr (C == 2) {
      out[0] = __builtin_amdgcn_raw_buffer_load_b32(tdrs, roff, so, 0);
    } else {
      out[0] = __builtin_amdgcn_raw_buffer_load_b16(tdrs, roff, so, 0);
    }
  };
  // Element e of ring slot u: column t = tlane + e is entry C-1-e.
  auto tdv = [&](int u, int e) -> int32_t {
    if constexpr (C == 1) {
      return (int32_t)(tdq[u][0] & 0xFFFFu);
    } else {
      const int k = C - 1 - e;
      const uint32_t w = tdq[u][k / 2];
      return (k & 1) ? (int32_t)(w >> 16) : (int32_t)(w & 0xFFFFu);
    }
  };
#pragma unroll
  for (int s = 0; s < PD; ++s) load_row(max(rmax - 1 - s, r0), tdq[s]);

  // Row metadata, 64 rows per chunk: lane i holds row rmax-1-(64s+i): its
  // far slot and flags, the slot it is saved to, its label and (kCost)
  // Vpre[r]; read per row with readlane; the next chunk is loaded one chunk
  // ahead.
  auto load_meta = [&](int s, int32_t& mfar, int32_t& mwr, int32_t& mlab, int32_t& mvp) {
    const int32_t rr = rmax - 1 - (64 * s + lane);
    const int32_t r = max(rr, r0);  // rows past the table read row r0
    NodeRec rc = rrecR[r];          // orl(r), label, kdep(r), kdep(r-1) | r-1 a leaf
    int32_t onext = rrecR[max(r - 1, r0)].orl;
    // Pinned, so that no load moves into a branch of its own (a branch on
    // lanes inside the row loop costs every uniform branch there its short
    // form).
    asm volatile("" : "+v"(rc.orl), "+v"(rc.x), "+v"(rc.y), "+v"(rc.label), "+v"(onext));
    // Rows past the table's end are plain rows (no flags): they lower minima
    // that nothing reads any more.
    const bool in = rr >= r0;
    const bool tree = in & (rc.orl + 1 == rmax);
    const bool saved = in & (r > r0) & (rc.y < 0);
    const bool next_tree = in & (r > r0) & (onext + 1 == rmax);
    const int32_t far_off = (rc.x - base - 1) * (int32_t)row_bytes;
    const int32_t wr_off = ((rc.y & 0x7FFFFFFF) - base - 1) * (int32_t)row_bytes;
    mfar = (far_off & -(int32_t)(in & (rc.orl + 1 < rmax))) | (kRowTree & -(int32_t)tree) |
           (kRowSaved & -(int32_t)saved) | (kRowFull & -(int32_t)(tree | saved | next_tree));
    mwr = wr_off & -(int32_t)saved;
    mlab = rc.label;
    if constexpr (kCost) {
      CostRec cr = A.pool.ccrec[offR + r];
      asm volatile("" : "+v"(cr.del), "+v"(cr.ins));
      mvp = rows_x ? cr.del : cr.ins;  // Vpre[r]
    }
  };
  const int32_t nchunks = (nrows + 63) >> 6;
  int32_t mfar, mwr, mlab, nfar = 0, nwr = 0, nlab = 0, mvp = 0, nvp = 0;
  load_meta(0, mfar, mwr, mlab, mvp);
  if (nchunks > 1) load_meta(1, nfar, nwr, nlab, nvp);

  int32_t cin = cin0;  // carry into this block on the last full row (lane 0)
  int32_t q = 0;       // full rows done
  int32_t vprev = 0;   // (kCost) V of the previous row
  // F[row below][column just before this block] without its cin part, in the
  // coordinates of the diagonal term (see the tree rows).
  int32_t qleft = tb - 2;
  if constexpr (kCost) qleft = hq - Hpre[max(cmax - tb, c0)];
  // (W > 1) Lane l takes word l of an edge entry: the carry, then imports.
  // The boundary value stands before the imports in the segment, so the same
  // lanes write the row's boundary value (lane 0) and imports to its slots;
  // on the outgoing entry lane 63, whose prefix minimum is the block's, writes
  // the carry.
  const int32_t word = min(lane, kds + 1);
  const uint32_t ein = edges + (uint32_t)wave * edge_bytes + 4u * (uint32_t)word;
  const uint32_t xout = edges + (uint32_t)(wave + 1) * edge_bytes;
  const uint32_t eout = xout + 4u * (uint32_t)(lane == 0 ? kds + 1 : lane == 63 ? 0 : word);
  const uint32_t seg_imp = slot_base + 2u * (uint32_t)(wb + word);
  uint32_t qoff = 0;  // (q % D) * entry_bytes
  int poll_limit = kEdgePolls;

  // Rows go S at a time in one flat loop with the inner loop fully unrolled,
  // so row k of the table always uses ring slot k % S and every slot index is
  // static: row k reads slot u and prefetches row k+PD into slot (u+PD) % S,
  // the slot the previous row has just finished with. Every path into the
  // loop head has issued the same loads, also past the table's end, so the
  // waits stay PD rows deep (an early exit merges into the loop's latch and
  // cuts them to two rows).
  for (int32_t k0 = 0; k0 < nrows; k0 += S) {
    const int32_t rpre = rmax - 1 - PD - k0;
    if (__builtin_expect((k0 & 63) == 0 && k0 > 0, 0)) {  // next 64-row chunk of row metadata
      mfar = nfar;
      mwr = nwr;
      mlab = nlab;
      mvp = nvp;
      if ((k0 >> 6) + 1 < nchunks) load_meta((k0 >> 6) + 1, nfar, nwr, nlab, nvp);
    }
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const int32_t k = k0 + u;
      load_row(max(rpre - u, r0), tdq[(u + PD) % S]);
      // Rows past the table's end: skipped where a row costs more than the
      // branch, else run as plain rows up to the next even one.
      if ((C < 8 && u % 2 == 1) || __builtin_expect(k < nrows, 1)) {
        if constexpr (W > 1) {
          if (u % kSyncRows == 0) {
            // This group's entries are there, and its full rows (at most
            // kSyncRows) find room in the outgoing ring.
            for (int n = 0;; ++n) {
              const unsigned long long pb = __hip_atomic_load(prog(wave), __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_WORKGROUP);
              const unsigned long long pa = __hip_atomic_load(prog(wave + 2), __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_WORKGROUP);
              const int32_t rows_before = __builtin_amdgcn_readfirstlane((int32_t)(uint32_t)pb);
              const int32_t full_after =
                  __builtin_amdgcn_readfirstlane((int32_t)(uint32_t)(pa >> 32));
              if (__builtin_expect((rows_before > k) & (full_after >= q - kSyncRows), 1)) break;
              if (n >= poll_limit) {  // raise the abort flag and wait no more
                A.xl_abort[2] = (int32_t)ix;
                A.xl_abort[3] = (2 << 24) | k;
                (void)atomicExch(A.xl_abort, 1);
                poll_limit = 0;
                break;
              }
            }
            lds_order();
          }
        }
        const int32_t i = k & 63;  // index in the metadata chunk
        const int32_t fw = __builtin_amdgcn_readlane(mfar, i);
        // The row's shift: V(k), or k with unit costs.
        int32_t vk = k, vcur = 1;
        if constexpr (kCost) {
          vk = vr - __builtin_amdgcn_readlane(mvp, i);
          vcur = vk - vprev;
          vprev = vk;
        }
        // The edge entry of the next full row: this one's, if it is full.
        int32_t edge = 0;
        if constexpr (W > 1) edge = l32(ein + qoff);
        // Terms of a plain row: far value + TD. (A tree row computes them too,
        // from slot row 0, and replaces them: kept out of an else of the branch
        // below, the common path has no taken branch. With the terms skipped on
        // tree rows instead, the root table of a deep 1000-node pair took 0.256
        // us a row against 0.212.)
        int32_t d[C];
        {
          const uint32_t fb = (uint32_t)(fw & kRowSlot);
          int32_t sv[C];
#pragma unroll
          for (int e = 0; e < C; ++e) sv[e] = l16(foff[e] + fb);
#pragma unroll
          for (int e = 0; e < C; ++e) {
            d[e] = sv[e] + tdv(u, e) + (term(e) - vk);
            asm volatile("" : "+v"(d[e]));
          }
          if constexpr (W > 1) asm volatile("" : "+v"(edge));
        }
        if (__builtin_expect((fw & kRowTree) != 0, 0)) {
          // Tree columns: the diagonal F[r+1][c+1] + rename (the row below is
          // full, so Am holds its values); other columns: the boundary row's
          // far value. Blended rather than branched per element.
          const int32_t labr = __builtin_amdgcn_readlane(mlab, i);
          const int32_t edge0 = kCost ? Am[C - 1] - term(C - 1) : Am[C - 1] + (C - 2);
          int32_t left = wave_shr1(edge0, cin + qleft);
#pragma unroll
          for (int e = 0; e < C; ++e) {
            d[e] = lb[e] + tdv(u, e) + (term(e) - vk);
            if (C >= 4 && !(tmask >> e & 1)) continue;  // uniform: no tree column among these
            int32_t diag, rename;
            if constexpr (kCost) {
              diag = (e ? Am[e ? e - 1 : 0] - term(e ? e - 1 : 0) : left) - vcur + term(e);
              // Columns off the tree path read entry 0 (one line for the wave)
              // instead of a row of the matrix.
              rename = A.ren[tcol[e] ? (rows_x ? labr * A.alphabet + lb[e]
                                               : lb[e] * A.alphabet + labr)
                                     : 0];
            } else {
              diag = e ? Am[e ? e - 1 : 0] - 2 : left;
              rename = (int32_t)(labr != lb[e]);
            }
            d[e] = tcol[e] ? diag + rename : d[e];
          }
        }
#pragma unroll
        for (int e = 0; e < C; ++e) Am[e] = min(Am[e], d[e]);
        if (fw & kRowFull) {
          // The row's values: prefix minima in the lane, then over the wave with
          // the carry of the blocks before (in lane 0; block 0's, the boundary,
          // is in A from the start).
#pragma unroll
          for (int e = 1; e < C; ++e) Am[e] = min(Am[e], Am[e - 1]);
          int32_t x = Am[C - 1] - T;
          if constexpr (W > 1) {
            x = min(x, lane == 0 ? edge : kBig);
            cin = edge;
          }
          const int32_t incl = wave_incl_min(x);
          const int32_t cg = wave_shr1(incl, W > 1 ? edge : kBig) + T;
#pragma unroll
          for (int e = 0; e < C; ++e) Am[e] = min(Am[e], cg);
          // Row values, and F[r][cmax]: the summed row costs (rmax - r = k + 1
          // with unit costs).
          int32_t v[C];
#pragma unroll
          for (int e = 0; e < C; ++e) v[e] = Am[e] - term(e) + vk;
          const int32_t frc = kCost ? vk : k + 1;
          if (__builtin_expect((fw & kRowSaved) != 0, 1)) {
            const uint32_t wbase = (uint32_t)__builtin_amdgcn_readlane(mwr, i);
#pragma unroll
            for (int e = 0; e < C; ++e) l16(woff[e] + wbase) = (uint16_t)v[e];
            if constexpr (W > 1) {
              l16(seg_imp + wbase) = (uint16_t)(lane == 0 ? frc : edge);
              if (__builtin_expect(kds >= 63, 0)) {
                for (int d0 = 63; d0 <= kds; d0 += 64) {
                  const int dd = min(d0 + lane, kds + 1);
                  const int32_t far = l32(xout - edge_bytes + qoff + 4 * dd);
                  l16(slot_base + wbase + 2 * (wb + dd)) = (uint16_t)far;
                  l32(xout + qoff + 4 * dd) = far;
                }
              }
            } else {
              l16(slot_base + wbase + 2u * wb) = (uint16_t)frc;
            }
          }
          if constexpr (W > 1) {
            // Imports pass on; then a path that starts in this block replaces
            // one of the same depth that ended in it. (Only a saved row's
            // entry is read beyond its carry.)
            l32(eout + qoff) = lane == 63 ? incl : edge;
            lds_order();
#pragma unroll
            for (int e = 0; e < C; ++e) l32(xout + qoff + xoff[e]) = v[e];
          }
          if constexpr (W > 1) {
            ++q;
            qoff += entry_bytes;
            if (qoff == edge_bytes) qoff = 0;
          }
          // (Tested afresh: one flag kept over the row costs more.)
          int32_t fw2 = fw;
          asm volatile("" : "+s"(fw2));
          if (__builtin_expect((fw2 & kRowTree) != 0, 0)) {
            // Tree cells -> TD / TD^T. Lanes without one store out of the
            // buffer's range, which drops the store (no branch on lanes, no
            // memory traffic). The column of element 0 is made opaque here so
            // that the compiler forms these rare stores' addresses when they
            // happen instead of keeping them live across the loop.
            const int32_t r = rmax - 1 - k;
            int32_t cb = cmax - 1 - tlane;
            asm volatile("" : "+v"(cb));
            const int32_t so = (int32_t)((uint32_t)r * (uint32_t)ldo * (uint32_t)sizeof(td_t));
#pragma unroll
            for (int e = 0; e < C; ++e) {
              if (C >= 4 && !(tmask >> e & 1)) continue;
              const int32_t c = cb - e;
              const bool cell = c >= c0 && tcol[e];
              const int32_t orow = cell ? (c + kTdPad) * (int32_t)sizeof(td_t) : kTdBytes;
              const int32_t ocol =
                  cell ? (int32_t)(((uint32_t)c * ldt + (uint32_t)r) * (uint32_t)sizeof(td_t))
                       : kTdBytes;
              __builtin_amdgcn_raw_buffer_store_b16((uint16_t)v[e], tdrs, orow, so, 0);
              __builtin_amdgcn_raw_buffer_store_b16((uint16_t)v[e], ttrs, ocol, 0, 0);
            }
          }
        }
      }  // k < nrows
      if constexpr (W > 1) {
        if (u % kSyncRows == kSyncRows - 1) {
          lds_order();
          __hip_atomic_store(prog(wave + 1),
                             ((unsigned long long)(uint32_t)q << 32) | (uint32_t)(k + 1),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          lds_order();
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
template <int W, int C>
static void launch_one(const DPArgs& a, int lds_bytes, hipStream_t s) {
  // One table per workgroup: a long task list goes in pieces.
  constexpr int64_t kChunk = kGridThreads / (64 * W);
  for (int64_t off = 0; off < a.ntasks; off += kChunk) {
    DPArgs c = a;
    c.tasks = a.tasks + off;
    c.descs = a.descs + off;
    c.ntasks = std::min(kChunk, a.ntasks - off);
    if (a.costs)
      hipLaunchKernelGGL((scan_kernel<W, C, true>), dim3((unsigned)c.ntasks), dim3(64 * W),
                         (size_t)lds_bytes, s, c);
    else
      hipLaunchKernelGGL((scan_kernel<W, C, false>), dim3((unsigned)c.ntasks), dim3(64 * W),
                         (size_t)lds_bytes, s, c);
  }
}

template <int W>
static void launch_c(int ci, const DPArgs& a, int lds, hipStream_t s) {
  switch (ci) {
    case 0: launch_one<W, 1>(a, lds, s); break;
    case 1: launch_one<W, 2>(a, lds, s); break;
    case 2: launch_one<W, 4>(a, lds, s); break;
    case 3: launch_one<W, 8>(a, lds, s); break;
    default: launch_one<W, 16>(a, lds, s); break;
  }
}

void launch_scan(int wi, int ci, const DPArgs& a, int lds_bytes, hipStream_t s) {
  switch (wi) {
    case 0: launch_c<1>(ci, a, lds_bytes, s); break;
    case 1: launch_c<2>(ci, a, lds_bytes, s); break;
    case 2: launch_c<4>(ci, a, lds_bytes, s); break;
    case 3: launch_c<8>(ci, a, lds_bytes, s); break;
    default: launch_c<16>(ci, a, lds_bytes, s); break;
  }
}

// Grants every instantiation the LDS it may ask for (> 64 KiB needs an
// explicit attribute).
template <int W, int C>
static hipError_t allow(int limit) {
  const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_kernel<W, C, false>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, limit);
  if (e != hipSuccess) return e;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_kernel<W, C, true>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, limit);
}
template <int W>
static hipError_t allow_c(int limit) {
  hipError_t e;
  if ((e = allow<W, 1>(limit)) != hipSuccess) return e;
  if ((e = allow<W, 2>(limit)) != hipSuccess) return e;
  if ((e = allow<W, 4>(limit)) != hipSuccess) return e;
  if ((e = allow<W, 8>(limit)) != hipSuccess) return e;
  return allow<W, 16>(limit);
}
hipError_t scan_init_attributes(int limit) {
  hipError_t e;
  if ((e = allow_c<1>(limit)) != hipSuccess) return e;
  if ((e = allow_c<2>(limit)) != hipSuccess) return e;
  if ((e = allow_c<4>(limit)) != hipSuccess) return e;
  if ((e = allow_c<8>(limit)) != hipSuccess) return e;
  return allow_c<16>(limit);
}

}  // namespace xted
