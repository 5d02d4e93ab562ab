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
// once (the 4096-pair batch, one stream, ms): one wave of 16 columns 27.3
// against 21.6, of 8 18.5 against 14.1, 8 waves of 2 16.2 against 7.4; those
// are bound by TD traffic (about 2 bytes a cell, 4 TB/s over the batch's
// streams).
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

// Bytes of a TD buffer resource, from kTdPad entries before the table: more
// than any table and its padding (32767^2 entries of 2 bytes), and as an
// offset out of range whatever scalar offset (below it) is added.
constexpr int32_t kTdBytes = (int32_t)0x80000000u;

// Compiler ordering of this wave's LDS operations (the hardware keeps it).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// ---------------------------------------------------------------------------
// Column-blocked tables (kXL): a table too wide or too LDS-hungry for one
// workgroup, cut into blocks of 64*W*C columns, one workgroup each. The edge
// between two blocks goes through device memory: wave W + 1 of the block
// before (edge_out) takes the last wave's edge entries from LDS and writes
// them out, wave W of the block after (edge_in) reads them and fills its
// block's first edge, so the other waves only ever see LDS. Per row a carry
// word (nb - 1 runs, one per edge, padded to whole 128-byte L2 lines), per
// saved row and edge a line-padded run of kds imports.
//
// Words are {epoch:32 | value:32}, written once per launch with atomic
// exchanges (performed where every XCD sees the same line; each XCD has an L2
// of its own), so nothing is cleared between launches and a word tells by
// itself whether it is there. Carries are read a line (16 rows) at a time with
// compare-exchanges against a value no word holds, which return the current
// word; once a line is complete so are the imports of its rows, as a rule,
// and these are read with plain loads. A stale word (levels share the memory,
// so a line of an earlier launch may still be in an L2; its epoch is old) is
// read again atomically.
// Workgroups take (table, block) from a ticket counter in start order, so a
// block only waits on blocks that are already running. Waits are bounded:
// after kXLWaitTicks of the 100 MHz wall clock a wave raises the abort flag
// (recording what it waited for), every waiting wave then stops waiting, and
// the call fails.
// Tables with at most xl_seq_rows rows are swept block after block by one
// workgroup; their words stay in its XCD and need no atomics.
//
// What bounds a row: the instructions of one wave, as on chip, with at most
// two or three waves to a SIMD. Measured, us a row over the blocks of an
// 8000-node RRT pair's root table, of 4096 / 2048 / 1024 / 512 columns: 0.45 /
// 0.32 / 0.27 / 0.26 (on chip 16 waves of 8 columns 0.63). With a barrier per row and every
// wave reading the words itself, a 20,000-node pair's pipelined blocks took
// 138 ms against 34 here, its tables of at most 256 rows 42 against 29.
// ---------------------------------------------------------------------------
constexpr uint64_t kXLWaitTicks = 1000000000ull;  // 10 s at 100 MHz
constexpr unsigned long long kXLNever = ~0ull;    // epoch 0xFFFFFFFF is never issued
constexpr int kXLLineRows = kXLLineWords;         // carries read at a time: one line
__device__ __forceinline__ unsigned long long xl_peek(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// (An idempotent or-with-0 would be turned back into a plain load.)
__device__ __forceinline__ unsigned long long xl_load(unsigned long long* p) {
  unsigned long long cur = kXLNever;
  (void)__hip_atomic_compare_exchange_strong(p, &cur, kXLNever, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
  return cur;
}
__device__ __forceinline__ void xl_store(unsigned long long* p, uint32_t epoch, int32_t v,
                                         bool local) {
  const unsigned long long w = ((unsigned long long)epoch << 32) | (uint32_t)v;
  if (local) __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else (void)__hip_atomic_exchange(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A bounded wait: true while it may go on. The wave that gives up records
// what = kind << 24 | row (kinds: 0 a carry, 1 an import, 2 a neighbour wave)
// in abort_flag[2..3]; others see the flag.
struct Patience {
  uint64_t t0 = 0;
  bool gone = false;
  __device__ __forceinline__ bool wait(int n, int32_t* abort_flag, int32_t ticket, int32_t what) {
    if (gone) return false;
    __builtin_amdgcn_s_sleep(1);
    if ((n & 255) != 255) return true;
    const uint64_t now = wall_clock64();
    if (n < 256) t0 = now;  // this wait's first look at the clock
    const bool raised = xl_peek(reinterpret_cast<unsigned long long*>(abort_flag)) & 0xFFFFFFFFu;
    if (raised || now - t0 > kXLWaitTicks) {
      if (!raised && atomicCAS(abort_flag + 1, 0, 1) == 0) {
        abort_flag[2] = ticket;
        abort_flag[3] = what;
      }
      (void)atomicExch(abort_flag, 1);
      gone = true;
    }
    return !gone;
  }
};

// What the edge waves need of a block: the table's rows, the first of its
// words, its edges' byte offsets in LDS.
struct XLEdge {
  const NodeRec* rrecR;
  const int32_t* lrankR;
  int32_t r0, rmax, nrows, kds, nb, blk, ticket;
  bool seq;
  unsigned long long* words;
  uint32_t epoch;
  uint32_t edge;         // LDS byte offset of the edge to fill or empty
  uint32_t entry_bytes;
};
// Flags of 64 rows (lane = row k0 + lane): bit 0 full, bit 1 saved, bit 2 the
// row is in the table; and the saved row's index (leaf rank of r-1).
__device__ __forceinline__ void xl_rows(const XLEdge& x, int32_t k0, int lane, int32_t& flags,
                                        int32_t& rid) {
  const int32_t rr = x.rmax - 1 - (k0 + lane);
  const int32_t r = max(rr, x.r0);
  NodeRec rc = x.rrecR[r];
  int32_t onext = x.rrecR[max(r - 1, x.r0)].orl;
  int32_t lr = x.lrankR[max(r - 1, x.r0)] - x.lrankR[x.r0];
  asm volatile("" : "+v"(rc.orl), "+v"(rc.y), "+v"(onext), "+v"(lr));
  const bool in = rr >= x.r0;
  const bool saved = in & (r > x.r0) & (rc.y < 0);
  const bool full = saved | (in & (rc.orl + 1 == x.rmax)) |
                    (in & (r > x.r0) & (onext + 1 == x.rmax));
  flags = (int32_t)full | ((int32_t)saved << 1) | ((int32_t)in << 2);
  rid = lr;
}

// Wave W: fills the block's first edge from the words of the block before.
template <int D, int kSync>
__device__ __forceinline__ void edge_in(const DPArgs& A, const XLEdge& x, unsigned char* lds,
                                        int lane) {
  auto l32 = [&](uint32_t byte) -> int32_t& { return *reinterpret_cast<int32_t*>(lds + byte); };
  unsigned long long* const prog = reinterpret_cast<unsigned long long*>(lds);
  const uint32_t epoch = x.epoch;
  const int32_t cstride = xl_pad(x.nrows), kdsp = xl_pad(x.kds);
  unsigned long long* const carries = x.words + (int64_t)(x.blk - 1) * cstride;
  unsigned long long* const exps = x.words + (int64_t)(x.nb - 1) * cstride;
  auto imp_word = [&](int32_t rid, int32_t d) {
    return exps + ((int64_t)rid * x.nb + (x.blk - 1)) * kdsp + d;
  };
  Patience pat;
  int32_t flags = 0, rid = 0, n_stale = 0, n_wait = 0, q = 0;
  uint32_t qoff = 0;
  const uint32_t edge_bytes = D * x.entry_bytes;
  // The line of row k: lane l holds row k + l's carry word.
  auto poll_line = [&](int32_t k) {
    const int32_t row = min(k + (lane & (kXLLineRows - 1)), x.nrows - 1);
    return x.seq ? xl_peek(carries + row) : xl_load(carries + row);
  };
  unsigned long long cw = poll_line(0);
  for (int32_t k0 = 0; k0 < x.nrows; k0 += kXLLineRows) {
    if ((k0 & 63) == 0) xl_rows(x, k0, lane, flags, rid);
    if (__ballot((uint32_t)(cw >> 32) != epoch)) {
      ++n_wait;
      for (int n = 0; __ballot((uint32_t)(cw >> 32) != epoch); ++n) {
        if (!pat.wait(n, A.xl_abort, x.ticket, k0)) break;
        cw = poll_line(k0);
      }
    }
    const int32_t carry = (int32_t)(uint32_t)cw;
    // The first 64 imports of the line's saved rows, all in flight together.
    unsigned long long iw[kXLLineRows];
#pragma unroll
    for (int i = 0; i < kXLLineRows; ++i) {
      const int at = (k0 & 63) + i;
      iw[i] = (unsigned long long)epoch << 32;  // nothing to read: valid
      if ((__builtin_amdgcn_readlane(flags, at) & 2) && lane < x.kds)
        iw[i] = xl_peek(imp_word(__builtin_amdgcn_readlane(rid, at), lane));
    }
    if (k0 + kXLLineRows < x.nrows) cw = poll_line(k0 + kXLLineRows);
#pragma unroll
    for (int i = 0; i < kXLLineRows; ++i) {
      const int32_t k = k0 + i;
      if (i % kSync == 0) {
        // The group's full rows find room once the first wave has taken
        // enough of the entries before.
        for (int n = 0;; ++n) {
          const unsigned long long pa =
              __hip_atomic_load(prog + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          if (__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)(pa >> 32)) >= q - kSync) break;
          if (!pat.wait(n, A.xl_abort, x.ticket, (2 << 24) | k)) break;
        }
        lds_order();
      }
      const int at = (k0 & 63) + i;
      const int32_t fl = __builtin_amdgcn_readlane(flags, at);
      if (fl & 1) {
        if ((fl & 2) && __ballot((uint32_t)(iw[i] >> 32) != epoch)) {
          ++n_stale;
          for (int n = 0; __ballot((uint32_t)(iw[i] >> 32) != epoch); ++n) {
            if ((uint32_t)(iw[i] >> 32) != epoch)
              iw[i] = xl_load(imp_word(__builtin_amdgcn_readlane(rid, at), lane));
            if (!pat.wait(n, A.xl_abort, x.ticket, (1 << 24) | k)) break;
          }
        }
        const uint32_t entry = x.edge + qoff;
        l32(entry + 4 * min(1 + lane, x.kds + 1)) = (int32_t)(uint32_t)iw[i];
        if (fl & 2) {
          for (int32_t d0 = 64; d0 < x.kds; d0 += 64) {
            const int32_t d = d0 + lane;
            unsigned long long w = (unsigned long long)epoch << 32;
            if (d < x.kds) w = xl_peek(imp_word(__builtin_amdgcn_readlane(rid, at), d));
            for (int n = 0; __ballot((uint32_t)(w >> 32) != epoch); ++n) {
              if ((uint32_t)(w >> 32) != epoch)
                w = xl_load(imp_word(__builtin_amdgcn_readlane(rid, at), d));
              if (!pat.wait(n, A.xl_abort, x.ticket, (1 << 24) | k)) break;
            }
            l32(entry + 4 * min(1 + d, x.kds + 1)) = (int32_t)(uint32_t)w;
          }
        }
        l32(entry) = __builtin_amdgcn_readlane(carry, i);
        ++q;
        qoff = qoff + x.entry_bytes == edge_bytes ? 0 : qoff + x.entry_bytes;
      }
      if (i % kSync == kSync - 1) {
        lds_order();
        __hip_atomic_store(prog, ((unsigned long long)(uint32_t)q << 32) | (uint32_t)(k + 1),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        lds_order();
      }
    }
  }
  if (lane == 0 && n_stale) atomicAdd(A.xl_abort + 8, n_stale);
  if (lane == 0 && n_wait) atomicAdd(A.xl_abort + 9, n_wait);
}

// Wave W + 1: empties the block's last edge into the words of this block.
template <int D, int kSync>
__device__ __forceinline__ void edge_out(const DPArgs& A, const XLEdge& x, unsigned char* lds,
                                         int W, int lane) {
  auto l32 = [&](uint32_t byte) -> int32_t& { return *reinterpret_cast<int32_t*>(lds + byte); };
  unsigned long long* const prog = reinterpret_cast<unsigned long long*>(lds);
  const uint32_t epoch = x.epoch;
  const int32_t cstride = xl_pad(x.nrows), kdsp = xl_pad(x.kds);
  unsigned long long* const carries = x.words + (int64_t)x.blk * cstride;
  unsigned long long* const exps = x.words + (int64_t)(x.nb - 1) * cstride;
  Patience pat;
  int32_t flags = 0, rid = 0, q = 0;
  uint32_t qoff = 0;
  const uint32_t edge_bytes = D * x.entry_bytes;
  for (int32_t k0 = 0; k0 < x.nrows; k0 += kSync) {
    if ((k0 & 63) == 0) xl_rows(x, k0, lane, flags, rid);
    for (int n = 0;; ++n) {
      const unsigned long long pb =
          __hip_atomic_load(prog + W, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)pb) > k0) break;
      if (!pat.wait(n, A.xl_abort, x.ticket, (2 << 24) | k0)) break;
    }
    lds_order();
    int32_t carry = 0;  // lane i: row k0 + i's (rows that are not full hand on any value)
#pragma unroll
    for (int i = 0; i < kSync; ++i) {
      const int at = (k0 & 63) + i;
      const int32_t fl = __builtin_amdgcn_readlane(flags, at);
      if (fl & 1) {
        const uint32_t entry = x.edge + qoff;
        const int32_t c = l32(entry);
        if (fl & 2) {
          const int32_t r = __builtin_amdgcn_readlane(rid, at);
          for (int32_t d0 = 0; d0 < x.kds; d0 += 64) {
            const int32_t d = d0 + lane;
            const int32_t v = l32(entry + 4 * min(1 + d, x.kds + 1));
            if (d < x.kds)
              xl_store(exps + ((int64_t)r * x.nb + x.blk) * kdsp + d, epoch, v, x.seq);
          }
        }
        carry = lane == i ? c : carry;
        ++q;
        qoff = qoff + x.entry_bytes == edge_bytes ? 0 : qoff + x.entry_bytes;
      }
    }
    // The entries are taken (their reads are done before this write).
    lds_order();
    __hip_atomic_store(prog + W + 1, ((unsigned long long)(uint32_t)q << 32) | (uint32_t)k0,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (lane < kSync && k0 + lane < x.nrows)
      xl_store(carries + k0 + lane, epoch, carry, x.seq);
  }
}

// One table (kTable), or one column block of a table: of a pipeline of
// workgroups (kBlocked) or of the sweep of one wave (kSwept). On the calling
// workgroup (64 * W threads, 128 more with kBlocked).
enum ScanMode { kTable, kBlocked, kSwept };
template <int W, int C, bool kCost, ScanMode kMode>
__device__ __forceinline__ void scan_block(const DPArgs& A, const TaskDesc& dsc, int32_t ix,
                                           int32_t blk, int32_t nb) {
  constexpr bool kXL = kMode == kBlocked;
  constexpr bool kRing = W > 1 || kXL;                // edges are rings between waves
  constexpr bool kEdges = kRing || kMode == kSwept;
  static_assert(kMode != kSwept || W == 1);
  // TD ring slots: a power of two dividing 64; 4 where 8 would leave too few
  // waves, or spill: 16 waves have 128 registers each (with costs and 8 slots
  // 34 of them spilled; 233,500 tables of a pair of 8000 and 250 nodes 7.8 ms,
  // with 4 slots and none 6.6).
  constexpr int S = C >= 16 || (C >= 8 && ((W == 1 && !kXL) || (kCost && (kXL || W == 16)))) ? 4 : 8;
  constexpr int PD = S - 1;                    // rows of TD prefetched
  constexpr int NW = C == 1 ? 1 : C / 2;       // words of one row: two 16-bit entries each
  constexpr int D = kXL ? xl_edge_rows(W) : kEdgeRows;
  constexpr int kSync = D / 2;  // a wave may fill one group while the next takes another
  extern __shared__ __align__(16) unsigned char lds[];
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
  const int wave = kRing ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int lane = threadIdx.x & 63;
  const int32_t tb0 = kMode != kTable ? blk * (64 * W * C) : 0;  // first t of the block
  const int32_t tb = tb0 + wave * 64 * C;            // and of this wave's part
  const int32_t tlane = tb + lane * C;               // t of this lane's element 0
  const int32_t nw = kRing ? min(W, (ncols - tb0 + 64 * C - 1) / (64 * C)) : 1;  // waves used

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
  const int32_t ltop = lrankC[max(cmax - 1 - tb0, c0)];  // of the block's columns
  int32_t lbase0 = dsc.lbase;
  if constexpr (kMode != kTable) lbase0 = lrankC[max(cmax - tb0 - 64 * W * C - 1, c0)];
  int32_t lbase = lbase0, wb = ltop - lbase0, seg = 0, kds = 0, kdep_c0 = 0;
  if constexpr (kEdges) {
    const int32_t chi = max(cmax - 1 - tb, c0);
    const int32_t clo = max(c0, cmax - tb - 64 * C);
    const int32_t lhi = lrankC[chi];
    lbase = lrankC[max(clo - 1, c0)];
    wb = max(0, lhi - lbase);
    kds = A.pool.kdn[offC + c0] + 1;
    kdep_c0 = A.pool.kdep[offC + c0];
    seg = (ltop - lhi) + wave * (2 + kds);
  }
  const uint32_t entry_bytes = kEdges ? 4u * (uint32_t)(kds + 2) : 0u;
  const uint32_t edge_bytes = D * entry_bytes;
  constexpr uint32_t edges = kRing ? 8u * (W + 2) : 0u;  // byte offset of edge 0
  const uint32_t all_edges = kRing ? (W + 1) * edge_bytes : (uint32_t)(nrows + 1) * entry_bytes;
  const uint32_t slot_base = edges + (kEdges ? all_edges : 0u) + 2u * (uint32_t)seg;
  const uint32_t row_bytes = 2u * (uint32_t)((ltop - lbase0) + W * (2 + kds));
  const int32_t sinkix = wb + 1 + kds;
  auto l16 = [&](uint32_t byte) -> uint16_t& { return *reinterpret_cast<uint16_t*>(lds + byte); };
  auto l32 = [&](uint32_t byte) -> int32_t& { return *reinterpret_cast<int32_t*>(lds + byte); };
  auto prog = [&](int w) { return reinterpret_cast<unsigned long long*>(lds + 8 * w); };
  if constexpr (kMode == kSwept) {
    if (blk == 0)
      for (int32_t k = lane; k <= nrows; k += 64) l32(k * entry_bytes) = cin0;
  }
  if constexpr (kRing) {
    if (threadIdx.x < D) l32(edges + threadIdx.x * entry_bytes) = cin0;
    if (threadIdx.x < W + 2) {
      const int w = (int)threadIdx.x - 1;
      const bool open = w < 0 ? blk == 0 : w >= nw && blk + 1 == nb;  // holds nobody up
      *prog((int)threadIdx.x) = open ? 0x7FFFFFFF7FFFFFFFull : 0ull;
    }
    __syncthreads();
    if constexpr (kXL) {
      if (wave >= W) {
        XLEdge x{rrecR, A.pool.lrank + offR, r0, rmax, nrows, kds, nb, blk, ix,
                 nrows <= A.xl_seq_rows, A.xl_words + A.xl_off[ix],
                 *A.xl_base + A.xl_epoch, edges, entry_bytes};
        if (wave == W && blk > 0) {
          edge_in<D, kSync>(A, x, lds, lane);
        } else if (wave > W && blk + 1 < nb) {
          x.edge = edges + W * edge_bytes;
          edge_out<D, kSync>(A, x, lds, W, lane);
        }
        return;
      }
    }
    if (wave >= nw) return;
  }
  const bool more = kEdges && (wave + 1 < nw || blk + 1 < nb);

  // Per-column state, element e (t = tlane + e, c = cmax-1-t).
  //   tcol: a tree column (orl_C(c) == orl_C(c0));
  //   lb:   on a tree column its label (tree cells only), else the far value
  //         on the boundary row F[rmax][orl_C(c)+1];
  //   foff: byte offset of the column's far value in this wave's segment;
  //   woff: byte offset it is saved at (c-1 a leaf of subtree(c0)), or the
  //         sink;
  //   xoff: (edges) byte offset in an edge entry: for a saved column whose
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
  uint32_t xoff[kEdges ? C : 1];
  auto term = [&](int e) -> int32_t {
    if constexpr (kCost) return negt[e];
    else return -e;
  };
  const int32_t T = kCost ? 0 : tlane;
  // The columns' records are read 8 at a time (4 where 8 would spill) and
  // pinned, so that each is one 16-byte load in flight with the others
  // (unpinned, the compiler splits them into loads of single fields in branches
  // on lanes, each waiting for the one before).
  constexpr int B = C < 8 ? C : kXL && kCost ? 4 : 8;
#pragma unroll
  for (int e0 = 0; e0 < C; e0 += B) {
    NodeRec cl[B], rl[kEdges ? B : 1];  // as a table column; (edges) as a row: kdep of c and c-1
    int32_t ul[kEdges ? B : 1];         // (edges) the keyroot at the top of c-1's right path
    CostRec ll[kCost ? B : 1];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int32_t c = max(cmax - 1 - (tlane + e0 + b), c0);
      cl[b] = crecC[c];
      if constexpr (kEdges) {
        rl[b] = A.pool.rrec[offC + c];
        ul[b] = A.pool.rtop[offC + max(c - 1, c0)];
      }
      if constexpr (kCost) ll[b] = A.pool.ccrec[offC + c];
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int e = e0 + b;
      asm volatile("" : "+v"(cl[b].orl), "+v"(cl[b].label), "+v"(cl[b].x), "+v"(cl[b].y));
      if constexpr (kEdges) asm volatile("" : "+v"(rl[b].x), "+v"(rl[b].y), "+v"(ul[b]));
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
      if constexpr (kEdges) {
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
  // (edges) Lane l takes word l of an edge entry: the carry, then imports.
  // The boundary value stands before the imports in the segment, so the same
  // lanes write the row's boundary value (lane 0) and imports to its slots;
  // on the outgoing entry lane 63, whose prefix minimum is the block's, writes
  // the carry.
  const int32_t word = min(lane, kds + 1);
  const uint32_t xin = edges + (kRing ? (uint32_t)wave * edge_bytes : 0u);
  const uint32_t xout = edges + (kRing ? (uint32_t)(wave + 1) * edge_bytes : 0u);
  const uint32_t ein = xin + 4u * (uint32_t)word;
  const uint32_t eout = xout + 4u * (uint32_t)(lane == 0 ? kds + 1 : lane == 63 ? 0 : word);
  const uint32_t seg_imp = slot_base + 2u * (uint32_t)(wb + word);
  uint32_t qoff = 0;  // (q % D) * entry_bytes
  Patience pat;

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
        if constexpr (kRing) {
          if (u % kSync == 0) {
            // This group's entries are there, and its full rows (at most
            // kSync) find room in the outgoing ring.
            for (int n = 0;; ++n) {
              const unsigned long long pb = __hip_atomic_load(prog(wave), __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_WORKGROUP);
              const unsigned long long pa = __hip_atomic_load(prog(wave + 2), __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_WORKGROUP);
              const int32_t rows_before = __builtin_amdgcn_readfirstlane((int32_t)(uint32_t)pb);
              const int32_t full_after =
                  __builtin_amdgcn_readfirstlane((int32_t)(uint32_t)(pa >> 32));
              if (__builtin_expect((rows_before > k) & (full_after >= q - kSync), 1)) break;
              if (!pat.wait(n, A.xl_abort, ix, (2 << 24) | k)) break;
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
        if constexpr (kEdges) edge = l32(ein + qoff);
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
          if constexpr (kEdges) asm volatile("" : "+v"(edge));
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
          if constexpr (kEdges) {
            x = min(x, lane == 0 ? edge : kBig);
            cin = edge;
          }
          const int32_t incl = wave_incl_min(x);
          const int32_t cg = wave_shr1(incl, kEdges ? edge : kBig) + T;
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
            if constexpr (kEdges) {
              l16(seg_imp + wbase) = (uint16_t)(lane == 0 ? frc : edge);
              if (__builtin_expect(kds >= 63, 0)) {
                for (int d0 = 63; d0 <= kds; d0 += 64) {
                  const int dd = min(d0 + lane, kds + 1);
                  const int32_t far = l32(xin + qoff + 4 * dd);
                  l16(slot_base + wbase + 2 * (wb + dd)) = (uint16_t)far;
                  l32(xout + qoff + 4 * dd) = far;
                }
              }
            } else {
              l16(slot_base + wbase + 2u * wb) = (uint16_t)frc;
            }
          }
          if constexpr (kEdges) {
            // Imports pass on; then a path that starts in this block replaces
            // one of the same depth that ended in it. (Only a saved row's
            // entry is read beyond its carry.)
            l32(eout + qoff) = lane == 63 ? incl : edge;
            lds_order();
#pragma unroll
            for (int e = 0; e < C; ++e) l32(xout + qoff + xoff[e]) = v[e];
          }
          if constexpr (kEdges) {
            ++q;
            qoff += entry_bytes;
            if (kRing && qoff == edge_bytes) qoff = 0;
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
      if constexpr (kRing) {
        if (u % kSync == kSync - 1) {
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

// Workgroups go round robin over the 8 XCDs, each with its own L2; task
// order keeps a pair's tables together, so kXcdRun consecutive tasks are
// given to one XCD (the last, partial span keeps its order). The 4096-pair
// batch ran 101.6 ms without, 100.1 with 16, 101.0 with 64, 104.8 with 256.
__device__ __forceinline__ uint32_t xcd_task(int64_t ntasks) {
  constexpr uint32_t kXcds = 8, kXcdRun = 16, kSpan = kXcds * kXcdRun;
  uint32_t ix = blockIdx.x;
  if ((ix | (kSpan - 1)) < (uint64_t)ntasks)
    ix = (ix & ~(kSpan - 1)) + (ix % kXcds) * kXcdRun + (ix % kSpan) / kXcds;
  return ix;
}

template <int W, int C, bool kCost>
__global__ __launch_bounds__(64 * W) void scan_kernel(DPArgs A) {
  const uint32_t ix = xcd_task(A.ntasks);
  if ((int64_t)ix >= A.ntasks) return;
  scan_block<W, C, kCost, kTable>(A, A.descs[ix], (int32_t)ix, 0, 1);
}

// One table per wave, block after block of kSweepCols columns, for wide tables
// of few rows in levels of many: the edge is one entry per full row, read by a
// block and overwritten for the next, and a slot row holds one block's far
// columns. What bounds it: the columns' records (36 bytes a column against 2 a
// cell) and the set-up of each block, of which a SIMD holds 4 at a time.
// 6165 tables of 8,000-20,000 columns and about 17 rows: 1.6 ms against 14
// in blocks of 1024 columns swept by a workgroup of 8 waves.
template <bool kCost>
__global__ __launch_bounds__(64, kCost ? 3 : 4) void scan_sweep_kernel(DPArgs A) {
  const uint32_t ix = xcd_task(A.ntasks);
  if ((int64_t)ix >= A.ntasks) return;
  const int32_t nb = (A.descs[ix].cmax - A.descs[ix].c0 + kSweepCols - 1) / kSweepCols;
  for (int32_t blk = 0; blk < nb; ++blk) {
    // (Opaque for each block, as in scan_xl_kernel.)
    uint32_t ib = ix;
    asm volatile("" : "+s"(ib));
    scan_block<1, kSweepCols / 64, kCost, kSwept>(A, A.descs[ib], (int32_t)ib, blk, nb);
    lds_order();
  }
}

// Column-blocked: W waves of C columns per lane and the two edge waves.
template <int W, int C, bool kCost>
__global__ __launch_bounds__(64 * (W + 2)) void scan_xl_kernel(DPArgs A) {
  extern __shared__ __align__(16) unsigned char lds[];
  if (threadIdx.x == 0) *reinterpret_cast<uint32_t*>(lds) = atomicAdd(A.xl_ticket, 1u);
  __syncthreads();
  const int32_t ticket = __builtin_amdgcn_readfirstlane(*reinterpret_cast<int32_t*>(lds));
  const int32_t ix = ticket / A.xl_nbmax;
  int32_t blk = ticket % A.xl_nbmax;
  if ((int64_t)ix >= A.ntasks) return;
  const int32_t ncols = A.descs[ix].cmax - A.descs[ix].c0;
  const int32_t nrows = A.descs[ix].rmax - A.descs[ix].r0;
  const int32_t nb = (ncols + 64 * W * C - 1) / (64 * W * C);
  const bool seq = nrows <= A.xl_seq_rows;
  if (blk >= nb || (seq && blk > 0)) return;
  do {
    __syncthreads();  // the LDS of the block before (or the ticket) is read
    // The task's index is made opaque for each block: what a block derives from
    // its descriptor would otherwise be kept in registers over the blocks (50
    // of them, and the widest form would spill).
    int32_t ib = ix;
    asm volatile("" : "+s"(ib));
    scan_block<W, C, kCost, kBlocked>(A, A.descs[ib], ib, blk, nb);
  } while (seq && ++blk < nb);
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

void launch_sweep(const DPArgs& a, int lds_bytes, hipStream_t s) {
  constexpr int64_t kChunk = kGridThreads / 64;
  for (int64_t off = 0; off < a.ntasks; off += kChunk) {
    DPArgs c = a;
    c.tasks = a.tasks + off;
    c.descs = a.descs + off;
    c.ntasks = std::min(kChunk, a.ntasks - off);
    if (a.costs)
      hipLaunchKernelGGL(scan_sweep_kernel<true>, dim3((unsigned)c.ntasks), dim3(64),
                         (size_t)lds_bytes, s, c);
    else
      hipLaunchKernelGGL(scan_sweep_kernel<false>, dim3((unsigned)c.ntasks), dim3(64),
                         (size_t)lds_bytes, s, c);
  }
}

template <int W, int C>
static void launch_xl_one(const DPArgs& a, int lds_bytes, hipStream_t s) {
  // Workgroups take (task, block) tickets from one counter that the pieces
  // of a long launch share: a later piece continues where the earlier one
  // stopped, and every block it waits on holds a lower ticket, taken by a
  // workgroup of an earlier (finished) piece or a running one of its own.
  constexpr int64_t kChunk = kGridThreads / (64 * (W + 2));
  const int64_t total = a.ntasks * a.xl_nbmax;
  for (int64_t off = 0; off < total; off += kChunk) {
    const dim3 grid((unsigned)std::min(kChunk, total - off));
    if (a.costs)
      hipLaunchKernelGGL((scan_xl_kernel<W, C, true>), grid, dim3(64 * (W + 2)),
                         (size_t)lds_bytes, s, a);
    else
      hipLaunchKernelGGL((scan_xl_kernel<W, C, false>), grid, dim3(64 * (W + 2)),
                         (size_t)lds_bytes, s, a);
  }
}

void launch_xl(int form, const DPArgs& a, int lds_bytes, hipStream_t s) {
  switch (form) {  // must match xl_waves / xl_cpl
    case 0: launch_xl_one<8, 8>(a, lds_bytes, s); break;
    case 1: launch_xl_one<8, 4>(a, lds_bytes, s); break;
    case 2: launch_xl_one<8, 2>(a, lds_bytes, s); break;
    case 3: launch_xl_one<4, 2>(a, lds_bytes, s); break;
    case 4: launch_xl_one<1, 4>(a, lds_bytes, s); break;
    default: launch_xl_one<1, 2>(a, lds_bytes, s); break;
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
template <int W, int C>
static hipError_t allow_xl(int limit) {
  const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_xl_kernel<W, C, false>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, limit);
  if (e != hipSuccess) return e;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_xl_kernel<W, C, true>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, limit);
}
hipError_t scan_init_attributes(int limit) {
  hipError_t e;
  const int xl_limit = limit + kXLEdgeBytes;
  for (const void* f : {reinterpret_cast<const void*>(&scan_sweep_kernel<false>),
                        reinterpret_cast<const void*>(&scan_sweep_kernel<true>)}) {
    e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, limit);
    if (e != hipSuccess) return e;
  }
  if ((e = allow_xl<8, 8>(xl_limit)) != hipSuccess) return e;
  if ((e = allow_xl<8, 4>(xl_limit)) != hipSuccess) return e;
  if ((e = allow_xl<8, 2>(xl_limit)) != hipSuccess) return e;
  if ((e = allow_xl<4, 2>(xl_limit)) != hipSuccess) return e;
  if ((e = allow_xl<1, 4>(xl_limit)) != hipSuccess) return e;
  if ((e = allow_xl<1, 2>(xl_limit)) != hipSuccess) return e;
  if ((e = allow_c<1>(limit)) != hipSuccess) return e;
  if ((e = allow_c<2>(limit)) != hipSuccess) return e;
  if ((e = allow_c<4>(limit)) != hipSuccess) return e;
  if ((e = allow_c<8>(limit)) != hipSuccess) return e;
  return allow_c<16>(limit);
}

}  // namespace xted
