// Forest-distance DP kernels for gfx950 (wave64).
//
// One keyroot-pair table (i0, j0) fills F over rows i in [i0, imax] and columns
// j in [j0, jmax], imax = orl_x(i0)+1, jmax = orl_y(j0)+1, with
//   F[imax][j] = jmax - j,  F[i][jmax] = imax - i,
//   tree cell (orl_x(i)==orl_x(i0) && orl_y(j)==orl_y(j0)):
//     F[i][j] = min(F[i+1][j+1] + (lab_x(i)!=lab_y(j)), F[i+1][j]+1, F[i][j+1]+1) = TD[i][j]
//   forest cell:
//     F[i][j] = min(F[orl_x(i)+1][orl_y(j)+1] + TD[i][j], F[i+1][j]+1, F[i][j+1]+1)
// (X-TED_CPU/parallel_computing.cpp:4-45, X-TED_GPU/parallel_X_TED.cu:5-55,97-122).
//
// The tables are computed row by row along the table's short side ("rows"),
// each row as one min-plus prefix scan along the long side ("columns"):
//   with t = jmax-1-j and a[t] = min(diag-or-far term, F[i+1][j]+1),
//   F[i][j] = t + min(imax-i+1, min_{t'<=t} (a[t'] - t')).
// Integer min/plus are associative, so this re-association is bit-exact.
// The transposed problem (rows = y) is the same recurrence on TD^T; both TD
// and TD^T are kept so each orientation reads its rows contiguously.
//
// Far reads F[orl_x(i)+1][orl_y(j)+1] only touch rows r with r-1 a leaf and
// columns c with c-1 a leaf. Such a row is written once and read by the rows
// of one right path, i.e. while the sweep is inside one keyroot's subtree, so
// it lives in an LDS slot indexed by that keyroot's nesting depth below the
// table's keyroot; columns are compacted by leaf rank. Values are < 2^16 and
// stored as uint16.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>
#include <utility>

#include "kernels.hpp"
#include "wave.hpp"

namespace xted {

// ---------------------------------------------------------------------------
// Leaf-keyroot lines in closed form. A line is a leaf keyroot v of one tree R
// of a pair; over the other tree T it is TD(v, c) = (orl(c) - c + 1) -
// [nxt(c) <= orl(c)], nxt(c) being the first position >= c whose label is
// label(v). The line is a row of TD (v of x) or of TD^T (v of y) and a column
// of the other layout.
//
// One workgroup of 4 waves takes the leaf keyroots among 64 consecutive
// nodes of one side (a tile) and walks T right to left, 64 positions per
// step, lane l at position c = top - l. For each of its lines a wave forms
// nxt as a prefix minimum over lanes plus the minimum carried from the
// positions above, writes the 64 values as one contiguous row segment and
// keeps them in an LDS tile; then the workgroup writes the tile transposed,
// one position per wave instruction with the tile's 64 nodes across the
// lanes: whole 256-byte runs of the column layout. The entries of nodes that
// are not leaf keyroots carry no value yet; they belong to tables of two
// non-leaf keyroots, which run after this kernel and overwrite them, and no
// table reads a cell before the level that writes it. Positions that are
// leaf keyroots of T are left out: their whole row is a line of the other
// side, written by its tiles.
// ---------------------------------------------------------------------------
constexpr int kLeafTile = 64;
__global__ __launch_bounds__(256) void leaf_kernel(LeafArgs A, int64_t ntiles, int64_t base) {
  // Row kLeafTile of the tile takes the values of lines past the tile's
  // count, which are computed (so a wave's lines have no branches between
  // them and their scans interleave) but never stored.
  __shared__ int32_t tile[kLeafTile + 1][kLeafTile + 1];
  __shared__ int32_t lines[kLeafTile];
  const int64_t tix = base + blockIdx.x;
  if (tix >= ntiles) return;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  int lo = 0, hi = A.npairs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (A.tile_start[mid] <= tix) lo = mid;
    else hi = mid - 1;
  }
  const PairMeta pm = A.pairs[lo];
  const TreeMeta tx = A.pool.trees[pm.tx], ty = A.pool.trees[pm.ty];
  const int32_t q = (int32_t)(tix - A.tile_start[lo]);
  const int32_t qx = (tx.n + kLeafTile - 1) / kLeafTile;
  const bool of_x = q < qx;  // nodes of x: the lines are rows of TD
  const TreeMeta& R = of_x ? tx : ty;
  const TreeMeta& T = of_x ? ty : tx;
  const int32_t v0 = (of_x ? q : q - qx) * kLeafTile;
  // This lane's node of the tile, and whether it is a leaf keyroot.
  const int32_t vl = v0 + lane;
  const int32_t vc = min(vl, R.n - 1);
  const bool is_line = vl < R.n && A.pool.orl[R.node_off + vc] == vc &&
                       A.pool.kdn[R.node_off + vc] >= 0;
  const unsigned long long lmask = __ballot(is_line);
  const int nl = __popcll(lmask);
  if (nl == 0) return;  // uniform over the workgroup
  if (wave == 0 && is_line) lines[__popcll(lmask & ((1ull << lane) - 1))] = lane;
  const int32_t laml = A.pool.label[R.node_off + vc];
  const int32_t* __restrict__ labT = A.pool.label + T.node_off;
  const int32_t* __restrict__ orlT = A.pool.orl + T.node_off;
  const int32_t* __restrict__ kdnT = A.pool.kdn + T.node_off;
  // of_x: TD[v][c] = td[td_off + v*ny + c], TD^T[c][v] = td[tdt_off + c*nx + v];
  // else: TD^T[v][c] = td[tdt_off + v*nx + c], TD[c][v] = td[td_off + c*ny + v].
  td_t* const rows = A.td + (of_x ? pm.td_off : pm.tdt_off);  // [v][c], stride T.n
  td_t* const cols = A.td + (of_x ? pm.tdt_off : pm.td_off);  // [c][v], stride R.n
  const bool col_ok = vl < R.n;
  __syncthreads();
  constexpr int kPer = kLeafTile / 4;  // lines (and positions) per wave
  int32_t carry[kPer];
#pragma unroll
  for (int m = 0; m < kPer; ++m) carry[m] = INT_MAX;
  // Positions of the next step are read one step ahead.
  int32_t top = T.n - 1;
  int32_t cc = max(top - lane, 0);
  int32_t nlab = labT[cc], norl = orlT[cc], nkdn = kdnT[cc];
  for (; top >= 0; top -= 64) {
    const int32_t c = top - lane;
    const int32_t lab = nlab, oc = norl;
    const bool c_line = oc == c && nkdn >= 0;  // c is a leaf keyroot of T
    if (top >= 64) {
      cc = max(top - 64 - lane, 0);
      nlab = labT[cc];
      norl = orlT[cc];
      nkdn = kdnT[cc];
    }
    const int32_t size = oc - c + 1;
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
      const int k = wave + 4 * m;  // lines interleaved over the waves
      const bool real = k < nl;    // uniform
      const int32_t off = real ? lines[k] : kLeafTile;
      const int32_t lam = __builtin_amdgcn_readlane(laml, real ? off : 0);
      const int32_t incl = wave_incl_min(c >= 0 && lab == lam ? c : INT_MAX);
      const int32_t nxt = min(carry[m], incl);
      carry[m] = min(carry[m], __builtin_amdgcn_readlane(incl, 63));
      const int32_t d = size - (int32_t)(nxt <= oc);
      if (real && c >= 0) rows[(int64_t)(v0 + off) * T.n + c] = (td_t)d;
      tile[off][lane] = d;
    }
    const unsigned long long skip = __ballot(c < 0 || c_line);
    __syncthreads();
    // Transposed: position p = wave + 4m of this step, node v0 + lane.
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
      const int p = wave + 4 * m;
      if (!((skip >> p) & 1ull) && col_ok)
        cols[(int64_t)(top - p) * R.n + vl] = (td_t)tile[lane][p];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Leaf-keyroot lines under a cost model (the closed form in kernels.hpp). For
// line v (a leaf of R) over the other tree T: with H the cost of T's nodes
// that are not mapped (inserted when v is x's, deleted when it is y's), w(k)
// = ren(v, k) - H(k) (ren(k, v) for v of y) and d(v) the cost of v alone,
//   TD(v, c) = H(sub c) + min(d(v), m(c)),   m(c) = min over k in sub(c) of w(k).
// One right-to-left sweep over T gives every m(c): with R(c) the minimum over
// c's subtree and the subtrees of its later siblings,
//   m(c) = w(c) for a leaf, min(w(c), R(c+1)) otherwise;
//   R(c) = min(m(c), R(next sibling)) when c has one, m(c) otherwise.
// Between a node and its previous sibling the sweep passes only the
// previous sibling's subtree, so R of a next sibling waits on a stack: pushed
// at a node that has a previous sibling, popped at a node that has a next
// one. All lines of a tile sweep the same T, so every push and pop is the
// same for all lanes and lane l keeps its line's entries in column l of the
// LDS stack, the top entry in a register (so a push followed by a pop does
// not wait on LDS). One wave per tile of 64 consecutive nodes of R (the unit
// kernel's tiles); lane l is node v0 + l. Per step of 64 positions the
// metadata of position top - i sits in lane i (read per position with
// readlane), the rename values are loaded a chunk of 16 positions ahead,
// and the 64 x 64 values (below 2^16) are written from a 16-bit LDS tile as
// the unit kernel writes them: row segments of every line, then the column
// layout.
// ---------------------------------------------------------------------------
constexpr int kCostLeafChunk = 16;
__global__ __launch_bounds__(64) void leaf_cost_kernel(LeafArgs A, int64_t ntiles, int64_t base) {
  __shared__ int16_t stk[kCostLeafStack][64];
  __shared__ uint16_t tile[kLeafTile][kLeafTile + 2];
  const int64_t tix = base + blockIdx.x;
  if (tix >= ntiles) return;
  const int lane = threadIdx.x & 63;
  int lo = 0, hi = A.npairs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (A.tile_start[mid] <= tix) lo = mid;
    else hi = mid - 1;
  }
  const PairMeta pm = A.pairs[lo];
  const TreeMeta tx = A.pool.trees[pm.tx], ty = A.pool.trees[pm.ty];
  const int32_t q = (int32_t)(tix - A.tile_start[lo]);
  const int32_t qx = (tx.n + kLeafTile - 1) / kLeafTile;
  const bool of_x = q < qx;  // nodes of x: the lines are rows of TD
  const TreeMeta& R = of_x ? tx : ty;
  const TreeMeta& T = of_x ? ty : tx;
  const int32_t v0 = (of_x ? q : q - qx) * kLeafTile;
  const int32_t vl = v0 + lane;
  const int32_t vc = min(vl, R.n - 1);
  const bool is_line = vl < R.n && A.pool.orl[R.node_off + vc] == vc &&
                       A.pool.kdn[R.node_off + vc] >= 0;
  const unsigned long long lmask = __ballot(is_line);
  if (lmask == 0) return;  // uniform (one wave)
  const int32_t labv = A.pool.label[R.node_off + vc];
  // d(v): deleting v (a node of x) or inserting it (a node of y).
  const int32_t* Pv = (of_x ? A.pool.pdel : A.pool.pins) + R.node_off;
  const int32_t dv = Pv[vc + 1] - Pv[vc];
  // T's unmapped nodes are inserted (v of x) or deleted (v of y).
  const int32_t* PT = (of_x ? A.pool.pins : A.pool.pdel) + T.node_off;
  const int32_t* HT = of_x ? A.ins : A.del;
  const int32_t* __restrict__ labT = A.pool.label + T.node_off;
  const int32_t* __restrict__ orlT = A.pool.orl + T.node_off;
  const int32_t* __restrict__ parT = A.pool.parent + T.node_off;
  const int32_t* __restrict__ kdnT = A.pool.kdn + T.node_off;
  // ren(v, k) = ren[labv * a + lab k] for v of x, ren[lab k * a + labv] for v of y.
  const int32_t* const renv = A.ren + (of_x ? (int64_t)labv * A.alphabet : labv);
  const int32_t rstride = of_x ? 1 : A.alphabet;
  td_t* const rows = A.td + (of_x ? pm.td_off : pm.tdt_off);  // [v][c], stride T.n
  td_t* const cols = A.td + (of_x ? pm.tdt_off : pm.td_off);  // [c][v], stride R.n
  const bool col_ok = vl < R.n;
  // Stack entries [0, sp-1) in LDS, entry sp-1 in tos.
  int32_t sp = 0, rprev = 0, tos = 0;
  for (int32_t top = T.n - 1; top >= 0; top -= kLeafTile) {
    // Lane i: position p = top - i (positions past 0 repeat position 0).
    const int32_t p = top - lane;
    const int32_t pc = max(p, 0);
    const int32_t lab = labT[pc], o = orlT[pc], par = parT[pc];
    const int32_t opar = par >= 0 ? orlT[par] : o;
    // bit 0: internal node; bit 1: has a previous sibling (push); bit 2: has
    // a next sibling (pop); bit 3: a leaf keyroot of T (its cells are written
    // by T's own tiles in the column layout)
    const int32_t flags = (o > p ? 1 : 0) | (p > 0 && par != p - 1 ? 2 : 0) |
                          (p > 0 && o < opar ? 4 : 0) | (o == p && kdnT[pc] >= 0 ? 8 : 0);
    const int32_t hsub = PT[o + 1] - PT[pc];  // H(sub p)
    const int32_t hk = HT[lab];               // H(p)
    const int32_t cnt = min(kLeafTile, top + 1);
    int32_t wq[2][kCostLeafChunk];
    auto issue = [&](int chunk, int32_t* dst) {
#pragma unroll
      for (int j = 0; j < kCostLeafChunk; ++j)
        dst[j] = renv[(int64_t)__builtin_amdgcn_readlane(lab, chunk * kCostLeafChunk + j) * rstride];
    };
    issue(0, wq[0]);
#pragma unroll
    for (int ch = 0; ch < kLeafTile / kCostLeafChunk; ++ch) {
      if (ch * kCostLeafChunk >= cnt) break;  // uniform
      if (ch + 1 < kLeafTile / kCostLeafChunk) issue(ch + 1, wq[(ch + 1) & 1]);
#pragma unroll
      for (int j = 0; j < kCostLeafChunk; ++j) {
        const int i = ch * kCostLeafChunk + j;
        if (i >= cnt) break;  // uniform
        const int32_t f = __builtin_amdgcn_readlane(flags, i);
        const int32_t w = wq[ch & 1][j] - __builtin_amdgcn_readlane(hk, i);
        const int32_t m = (f & 1) ? min(w, rprev) : w;
        int32_t r = m;
        if (f & 4) {  // pop
          r = min(m, tos);
          sp = max(sp - 1, 0);
          if (sp > 0) tos = stk[sp - 1][lane];
        }
        if ((f & 2) && sp < kCostLeafStack) {  // push
          if (sp > 0) stk[sp - 1][lane] = (int16_t)tos;
          tos = r;
          ++sp;
        }
        rprev = r;
        tile[i][lane] = (uint16_t)(__builtin_amdgcn_readlane(hsub, i) + min(dv, m));
      }
    }
    __syncthreads();
    // Row segments: line l's values at positions top - i, i in lanes.
    const bool pos_ok = lane < cnt;
    unsigned long long lm = lmask;
    while (lm) {
      const int l = __ffsll((long long)lm) - 1;
      lm &= lm - 1;
      if (pos_ok) rows[(int64_t)(v0 + l) * T.n + (top - lane)] = tile[lane][l];
    }
    // Column layout: position top - i across the tile's 64 nodes.
    const unsigned long long skip = __ballot(!pos_ok || (flags & 8));
    for (int i = 0; i < cnt; ++i) {
      if (!((skip >> i) & 1ull) && col_ok)
        cols[(int64_t)(top - i) * R.n + vl] = tile[i][lane];
    }
    __syncthreads();
  }
}

void launch_leaf(const LeafArgs& a, int64_t ntiles, hipStream_t s) {
  if (a.costs) {
    constexpr int64_t kChunk = kGridThreads / 64;
    for (int64_t base = 0; base < ntiles; base += kChunk)
      hipLaunchKernelGGL(leaf_cost_kernel, dim3((unsigned)std::min(kChunk, ntiles - base)),
                         dim3(64), 0, s, a, ntiles, base);
    return;
  }
  constexpr int64_t kChunk = kGridThreads / 256;
  for (int64_t base = 0; base < ntiles; base += kChunk)
    hipLaunchKernelGGL(leaf_kernel, dim3((unsigned)std::min(kChunk, ntiles - base)), dim3(256), 0,
                       s, a, ntiles, base);
}

// ---------------------------------------------------------------------------
// Arena words of one column-blocked task: nb-1 runs of carries (one per
// row, each run padded to whole 128-byte L2 lines), then for every saved row
// and source block a line-padded run of kds export words (by depth). A line
// thus only holds words of one producer, and no block that reads a run
// writes to it.
struct XLGeom {
  int32_t nrows, nb, nsaved, kds;
};
__device__ __forceinline__ XLGeom xl_geom(const PoolView& P, const PairMeta& pm, uint64_t task,
                                          int bw) {
  const TreeMeta tx = P.trees[pm.tx], ty = P.trees[pm.ty];
  const int32_t i0 = (int32_t)task_i0(task), j0 = (int32_t)task_j0(task);
  const int32_t a = P.orl[tx.node_off + i0] - i0 + 1, b = P.orl[ty.node_off + j0] - j0 + 1;
  const bool rows_x = a <= b;
  const int64_t offR = rows_x ? tx.node_off : ty.node_off;
  const int64_t offC = rows_x ? ty.node_off : tx.node_off;
  const int32_t r0 = rows_x ? i0 : j0, c0 = rows_x ? j0 : i0;
  XLGeom g;
  g.nrows = rows_x ? a : b;
  g.nb = ((rows_x ? b : a) + bw - 1) / bw;
  g.nsaved = P.lrank[offR + r0 + g.nrows] - P.lrank[offR + r0];
  g.kds = P.kdn[offC + c0] + 1;
  return g;
}
__device__ __forceinline__ int64_t xl_words(const XLGeom& g) {
  return (int64_t)(g.nb - 1) * xl_pad(g.nrows) + (int64_t)g.nsaved * g.nb * xl_pad(g.kds);
}

// ---------------------------------------------------------------------------
// Row scan with shared slot rows: one table per workgroup of W waves, kC = 8
// columns per lane, for tables whose column keyroot is so deep that the
// imports of several waves do not fit LDS (scan.hip) and that are not split
// over workgroups for being tall. Every wave reads and writes one set of slot
// rows and takes its scan carry from the totals of the waves before it, with a
// barrier per row. Columns are counted from jmax: t = jmax-1-j, lane l of wave w
// owning t in [w*512 + 8l, w*512 + 8l + 8).
// What bounds it: the barrier, at which all waves wait for the slowest one's
// row (8 waves 0.5 us a row). Against blocks of one wave, which is what such
// tables would take instead: 4 waves are faster (the tall tables of 1025 to 2048
// columns of a pair of 2000-node trees nested 250 deep, 217 ms against 321 with
// blocks), 8 waves slower (2049 to 4096 columns, 3000-node trees nested 190
// deep, 277 against 214; a burst of 64 pairs of 500-5000 nodes with 21 such
// tables 129.8 against 126.0). Blocks need words in device memory, so short
// tables, whose time is not their level's, keep to shared slot rows.
// ---------------------------------------------------------------------------
template <int W, bool kCost>
__global__ __launch_bounds__(64 * W) void rowscan_kernel(DPArgs A) {
  constexpr int C = 8;       // columns per lane
  constexpr int S = 4;       // TD ring slots (a power of two dividing 64)
  constexpr int PD = S - 1;  // rows of TD prefetched
  constexpr int NW = C / 2;  // words of one row: two 16-bit entries each
  // Unit costs keep row k's values less k (F - t + T - k): the vertical
  // step F[r+1][c] + 1 of row k+1 is then row k's value itself, with no add
  // per column and row; the terms read from the far rows and TD take the -k
  // through their (scalar) per-column constant, and stores add k back.
  extern __shared__ uint16_t slots[];
  // Per-wave scan totals, double-buffered by row parity: a wave may write
  // row r-1's total while a slower wave still reads row r's.
  __shared__ int32_t xtot[2][W];

  if ((int64_t)blockIdx.x >= A.ntasks) return;
  const TaskDesc dsc = A.descs[blockIdx.x];
  const bool rows_x = dsc.base_rx < 0;
  const int64_t offR = dsc.offR;
  const int64_t offC = dsc.offC;
  const NodeRec* __restrict__ rrecR = A.pool.rrec + offR;
  const NodeRec* __restrict__ crecC = A.pool.crec + offC;
  const int32_t* __restrict__ lrankC = A.pool.lrank + offC;
  const int32_t r0 = dsc.r0, c0 = dsc.c0;
  td_t* TDo = A.td + dsc.tdo;  // [r][c]
  td_t* TDt = A.td + dsc.tdt;  // [c][r]
  const int64_t ldo = dsc.ldo;
  const int64_t ldt = dsc.ldt;

  const int32_t rmax = dsc.rmax, cmax = dsc.cmax;
  const int32_t ncols = cmax - c0;
  const int32_t nrows = rmax - r0;
  const int32_t base = dsc.base_rx & 0x7FFFFFFF;
  const int32_t orl_c0 = cmax - 1;
  // Non-unit costs (kCost). Hpre / Vpre: prefix sums of the horizontal
  // (column) and vertical (row) edit costs over the column and row trees:
  // insertions and deletions when the rows are x, the other way round when
  // they are y. Q(c) = Hpre[cmax-1] - Hpre[c] takes the place of t (with
  // unit costs Q(c) = t), hq = Hpre[cmax-1], hc = Hpre[cmax] (so hc - hq is
  // the cost of column cmax-1) and vr = Vpre[rmax].
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
  // A slot row holds the compact far columns (leaves but the table's last, by
  // leaf rank) and at index wb F[R][cmax] = rmax - R for the tree columns.
  const int32_t lbase = dsc.lbase;
  const int32_t wb = lrankC[cmax] - lbase - 1;
  // The row's last entry is a sink: the saved-row stores of columns that
  // save nothing go there, so every column stores without a branch.
  const int32_t sinkix = wb + 1;
  const int32_t rowlen = sinkix + 1;

  // Uniform over the wave, so it lives in a scalar register.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int32_t tlane = (wave * 64 + lane) * C;  // t of this lane's element 0

  // Per-column state, element e (t = tlane + e, c = cmax-1-t).
  //   tcol: a tree column (orl_C(c) == orl_C(c0));
  //   lb:   on a tree column its label (tree cells only), else the far value
  //         on the boundary row F[rmax][orl_C(c)+1] = cmax - orl_C(c) - 1;
  //   foff: the column's far index in a slot row (wb for tree columns);
  //   woff: the index this column writes in a saved row (c-1 a leaf of
  //         subtree(c0)), or the sink entry;
  //   Fpm:  F[r+1][c] + 1 - t + T (the scan works on a[t] - t);
  //   negt: (kCost) the column's -Q(c).
  // Unit costs keep the values shifted by T = tlane: the per-column term
  // -t + T is then the constant -e (an inline operand, not a register), and
  // only the wave scan works unshifted. term(e) is that per-column term
  // (-Q(c) under a cost model, where nothing is shifted).
  // Columns past the table (t >= ncols) come after every real column in the
  // scan order, so whatever they hold never reaches a real column; only
  // their stores are masked.
  bool tcol[C];
  // tdq: the TD ring, as loaded, unpacked where a row uses it (tdv).
  int32_t lb[C], foff[C], woff[C], Fpm[C];
  uint32_t tdq[S][NW];
  int32_t negt[kCost ? C : 1];
  auto term = [&](int e) -> int32_t {
    if constexpr (kCost) return negt[e];
    else return -e;
  };
  const int32_t T = kCost ? 0 : tlane;
  // F[rmax][c] + (vertical cost of row rmax-1) - Q(c): 2 with unit costs.
  const int32_t fpm0 = kCost ? (hc - hq) + (vr - Vpre[rmax - 1]) : 2;
#pragma unroll
  for (int e = 0; e < C; ++e) {
    const int32_t t = tlane + e;
    const int32_t c = max(cmax - 1 - t, c0);
    // One record: orl(c), label, leaf rank at orl(c), leaf rank of c-1
    // (bit 31: c-1 is a leaf; only read when c > c0).
    const NodeRec cr = crecC[c];
    const int32_t oc = cr.orl;
    const int32_t lab = cr.label;
    const int32_t lro = cr.x;
    const int32_t lrm = cr.y & 0x7FFFFFFF;
    const bool prev_leaf = cr.y < 0;
    const bool tree = (oc == orl_c0);
    tcol[e] = tree;
    // (kCost) the column tree's horizontal sums at c and at orl(c) + 1
    int32_t hcol = 0, hfar = 0;
    if constexpr (kCost) {
      const CostRec cc = A.pool.ccrec[offC + c];
      hcol = rows_x ? cc.ins : cc.del;
      hfar = rows_x ? cc.ins_end : cc.del_end;
    }
    lb[e] = tree ? lab : kCost ? hc - hfar : cmax - oc - 1;
    foff[e] = tree ? wb : lro - lbase;
    const bool writes = t < ncols && c > c0 && prev_leaf;
    woff[e] = writes ? lrm - lbase : sinkix;
    // F[rmax][c] + 1 - t = cmax - c + 1 - t with unit costs, shifted
    Fpm[e] = fpm0 + T;
    if constexpr (kCost) {
      negt[e] = hcol - hq;
      // Opaque to the optimiser, so that sums with it stay three-operand
      // adds (v_add3_u32) instead of becoming an add and a subtract.
      asm("" : "+v"(negt[e]));
    }
  }

  // TD row rr of this lane's columns into out[]: entry k (column off + k) is
  // half k & 1 of word k / 2, read through a buffer resource over the table
  // (its kTdPad entries of padding included): the row offset is a scalar and
  // the lane's column offset a VGPR fixed for the whole table. Loads are
  // unconditional, so the compiler never waits for them inside a branch: a
  // lane with no valid column reads C entries from column c0 instead, a
  // partly valid one up to C-1 entries before column c0 (both inside the
  // kTdPad entries around every table).
  const __amdgpu_buffer_rsrc_t tdrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)(TDo - kTdPad), 0, -1, kBufferWord3);
  const int32_t roff =
      ((tlane < ncols ? cmax - C - tlane : c0) + kTdPad) * (int32_t)sizeof(td_t);
  auto load_row = [&](int32_t rr, uint32_t* out) {
    // rr * ldo < 2^30 entries (trees of at most 32767 nodes): an unsigned
    // 32-bit byte offset.
    const int32_t so = (int32_t)((uint32_t)rr * (uint32_t)ldo * (uint32_t)sizeof(td_t));
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(tdrs, roff, so, 0);
    out[0] = v.x;
    out[1] = v.y;
    out[2] = v.z;
    out[3] = v.w;
  };
  // Element e of ring slot u: column t = tlane + e is entry C-1-e.
  auto tdv = [&](int u, int e) -> int32_t {
    const int k = C - 1 - e;
    const uint32_t w = tdq[u][k / 2];
    return (k & 1) ? (int32_t)(w >> 16) : (int32_t)(w & 0xFFFFu);
  };
#pragma unroll
  for (int q = 0; q < PD; ++q) load_row(max(rmax - 1 - q, r0), tdq[q]);

  // Row metadata, 64 rows per chunk: lane i holds row rmax-1-(64q+i) as
  // (label, Rf = orl_R(r)+1, slots = fslot | wslot << 16 | wrow << 31); read
  // per row with readlane; the next chunk is loaded one chunk ahead.
  auto meta_rec = [&](int q) {
    return rrecR[max(rmax - 1 - (64 * q + lane), r0)];  // rows past the table read row r0
  };
  auto load_meta = [&](int q, int32_t& mlab, int32_t& mrf, int32_t& mslot, int32_t& mvp,
                       const NodeRec* pre = nullptr) {
    const int32_t r = max(rmax - 1 - (64 * q + lane), r0);
    const NodeRec rc = pre ? *pre : rrecR[r];  // orl(r), label, kdep(r), kdep(r-1) | r-1 a leaf
    const int32_t orr = rc.orl, lab = rc.label, kd = rc.x;
    const int32_t kdp = rc.y & 0x7FFFFFFF;
    const int32_t fs = (orr + 1 < rmax) ? kd - base - 1 : 0;
    const bool saved = r > r0 && rc.y < 0;
    const int32_t ws = saved ? (((kdp - base - 1) << 16) | (int32_t)0x80000000) : 0;
    mlab = lab;
    mrf = orr + 1;
    mslot = fs | ws;
    if constexpr (kCost) {
      const CostRec cr = A.pool.ccrec[offR + r];
      mvp = rows_x ? cr.del : cr.ins;  // Vpre[r]
    }
  };
  const int32_t nchunks = (nrows + 63) >> 6;
  int32_t mlab, mrf, mslot, nlab = 0, nrf = 0, nslot = 0;
  int32_t mvp = 0, nvp = 0;  // kCost: Vpre of the row
  {
    // The first two chunks' records are read before either is used (one
    // load latency in the set-up, not two), each as one whole record: with
    // kdep pinned the compiler does not load it in a branch of its own after
    // a wait for the rest.
    NodeRec rc0 = meta_rec(0), rc1 = meta_rec(1);
    asm volatile("" : "+v"(rc0.x), "+v"(rc1.x));
    load_meta(0, mlab, mrf, mslot, mvp, &rc0);
    if (nchunks > 1) load_meta(1, nlab, nrf, nslot, nvp, &rc1);
  }

  // F[r+1] at the column just before this wave's block (t = w*512 - 1) for
  // the row about to start: the boundary row's t + 1 first, then each row's
  // carry-in plus that t.
  // (With costs: Q at that column, qleft, and F[rmax] there.)
  const int32_t cleft = max(cmax - wave * 64 * C, c0);
  const int32_t qleft = kCost ? hq - Hpre[cleft] : wave * 64 * C - 1;
  int32_t left_prev = kCost ? hc - Hpre[cleft] : wave * 64 * C;
  int32_t vp_prev = vr;  // kCost: Vpre of the previous row

  // Rows go S at a time in one flat loop with the inner loop fully unrolled,
  // so row k of the table always uses ring slot k % S and every slot index is
  // static: row k reads slot u and prefetches row k+PD into slot (u+PD) % S,
  // the slot the previous row has just finished with. Rows past the table's
  // end issue their prefetches and skip their bodies, so that every path into
  // the loop head has issued the same loads and no wait there drains the
  // ring.
  for (int32_t k0 = 0; k0 < nrows; k0 += S) {
    if ((k0 & 63) == 0 && k0 > 0) {  // next 64-row chunk of row metadata
      mlab = nlab;
      mrf = nrf;
      mslot = nslot;
      mvp = nvp;
      if ((k0 >> 6) + 1 < nchunks) load_meta((k0 >> 6) + 1, nlab, nrf, nslot, nvp);
    }
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const int32_t k = k0 + u;  // rows done so far
      load_row(max(rmax - 1 - k - PD, r0), tdq[(u + PD) % S]);
      if (k >= nrows) continue;
      const int32_t i = k & 63;  // index in the metadata chunk
      const int32_t r = rmax - 1 - k;
      const int32_t ku = kCost ? 0 : k;  // the unit form's row shift

      const int32_t labr = __builtin_amdgcn_readlane(mlab, i);
      const int32_t Rf = __builtin_amdgcn_readlane(mrf, i);
      const int32_t sl = __builtin_amdgcn_readlane(mslot, i);
      const bool tree_row = (Rf == rmax);
      // Vertical costs of this row and of the next, and F[r][cmax] (unit
      // costs: 1, 1 and rmax - r).
      int32_t vcur = 1, vnext = 1, frc = rmax - r;
      if constexpr (kCost) {
        const int32_t vpr = __builtin_amdgcn_readlane(mvp, i);
        const int32_t vpn = i < 63 ? __builtin_amdgcn_readlane(mvp, i + 1)
                                   : __builtin_amdgcn_readlane(nvp, 0);
        vcur = vp_prev - vpr;
        vnext = vpr - vpn;
        frc = vr - vpr;
        vp_prev = vpr;
      }
      const uint16_t* frow = slots + (sl & 0xFFFF) * rowlen;
      const bool wrow = sl < 0;
      uint16_t* wrow_ptr = slots + ((sl >> 16) & 0x7FFF) * rowlen;

      // h = a[t] - t per element, prefix in the lane, then over the wave. Tree
      // rows (orl_R(r) == orl_R(r0)) and the other rows take separate code
      // paths on the uniform flag.
      int32_t h[C], pre, carry_w;
      auto row_terms = [&](auto tree_tag) {
        constexpr bool kTree = decltype(tree_tag)::value;
        int32_t sv[C];
        if constexpr (!kTree) {
#pragma unroll
          for (int e = 0; e < C; ++e) sv[e] = frow[foff[e]];
        }
        // Tree rows: F[r+1][c+1] of element 0, the previous row's value one
        // column to the left in t order (F = Fpm - 1 + t).
        int32_t fpr0 = 0;
        if constexpr (kTree) fpr0 = wave_shr1(Fpm[C - 1] - vcur - term(C - 1), left_prev);
#pragma unroll
        for (int e = 0; e < C; ++e) {
          int32_t dm;  // diagonal-or-far term minus t
          if constexpr (kTree) {
            // diagonal F[r+1][c+1] + rename on a tree column, else the
            // boundary-row far value. F[r+1][c+1] - t = Fpm[e-1] - 2.
            // Blended with a mask rather than a branch per element.
            int32_t fprm, rename;
            if constexpr (kCost) {
              fprm = e ? Fpm[e - 1] - vcur - term(e - 1) + term(e) : fpr0 + term(e);
              // Columns off the tree path read entry 0 (one line for the
              // wave) instead of a row of the matrix.
              rename = A.ren[tcol[e] ? (rows_x ? labr * A.alphabet + lb[e]
                                               : lb[e] * A.alphabet + labr)
                                     : 0];
            } else {
              fprm = e ? Fpm[e - 1] - 2 : fpr0 + term(e);
              rename = (int32_t)(labr != lb[e]);
            }
            const int32_t diag = fprm + rename;
            const int32_t far = lb[e] + tdv(u, e) + (term(e) - ku);
            dm = tcol[e] ? diag : far;
          } else {
            dm = sv[e] + tdv(u, e) + (term(e) - ku);
          }
          h[e] = min(dm, Fpm[e]);
          if (e) h[e] = min(h[e], h[e - 1]);
        }
        const int32_t incl = wave_incl_min(h[C - 1] - T);
        pre = wave_shr1(incl, kBig);
        carry_w = __builtin_amdgcn_readlane(incl, 63);
      };
      if (tree_row) row_terms(std::true_type{});
      else row_terms(std::false_type{});

      // Carry into this wave: the boundary F[r][cmax] - (-1), then the totals
      // of the earlier waves.
      int32_t carry = kCost ? frc + (hc - hq) : 2;  // unit: (rmax - r) + 1 - k
      int32_t* xt = xtot[r & 1];
      if (lane == 0) xt[wave] = carry_w;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < W - 1; ++w) carry = min(carry, w < wave ? xt[w] : kBig);
      // F[r][c] at the column just before this wave's block: the previous
      // wave's last element ends with h = min(its carry-in, its own total) =
      // this wave's carry-in, and F = h + t; for wave 0 this gives
      // F[r][cmax] = rmax - r.
      left_prev = carry + qleft - (kCost ? 0 : 1);  // unit: in row k+1's shift
      // h becomes G - t; Fpm = G + 1 - t = h + 1 (unit costs: row k+1 is shifted
      // by one more, so Fpm = h).
      const int32_t cg = min(carry, pre) + T;
#pragma unroll
      for (int e = 0; e < C; ++e) {
        h[e] = min(cg, h[e]);
        Fpm[e] = kCost ? h[e] + vnext : h[e];
      }

      // Tree cells -> TD / TD^T (tree rows only); saved rows -> LDS slots.
      if (tree_row) {
        // Column of element 0, made opaque here so that the compiler forms
        // these rare stores' addresses when they happen instead of keeping
        // two 64-bit addresses per element live across the loop.
        int32_t cb = cmax - 1 - tlane;
        asm volatile("" : "+v"(cb));
        td_t* const rowp = TDo + (int64_t)r * ldo;
        td_t* const colp = TDt + r;
        const uint32_t ldt32 = (uint32_t)ldt;
#pragma unroll
        for (int e = 0; e < C; ++e) {
          const int32_t c = cb - e;
          if (c >= c0 && tcol[e]) {
            // c * ldt < 2^30: trees have at most 32767 nodes
            rowp[c] = (td_t)(h[e] - term(e) + ku);
            colp[(uint32_t)c * ldt32] = (td_t)(h[e] - term(e) + ku);
          }
        }
      }
      if (wrow) {
        // Columns this lane does not save write the row's sink entry.
#pragma unroll
        for (int e = 0; e < C; ++e) wrow_ptr[woff[e]] = (uint16_t)(h[e] - term(e) + ku);
        if (threadIdx.x == 0) wrow_ptr[wb] = (uint16_t)frc;
        // The next row may read this slot row at columns of other waves.
        // (Every other LDS reuse is ordered by the barrier above: a slot
        // row is only rewritten after the rows that read it.)
        __syncthreads();
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Tiny tables (at most kSeg = 16, 32 or 64 columns, so at most kSeg rows):
// 64 / kSeg per wave, one per kSeg-lane segment, one column per lane
// (t = lane % kSeg). A segment is one or more whole 16-lane DPP rows, so the
// row's scan and shift stay in registers (row_shr, row_bcast, wave_shr) and a
// table needs no barrier and no LDS exchange. Row metadata sits in lanes:
// lane t of a table holds that of rows t % 16 + 16 s in set s (each 16-lane
// row of a segment holds every set), and row k takes set k / 16 with
// row_newbcast:(k % 16). The TD values of all rows are read up front. Tables
// of one wave run to the longest one's row count, each lane storing only
// while its table has rows left.
// ---------------------------------------------------------------------------
template <class F, int... K>
__device__ __forceinline__ void static_for(F& f, std::integer_sequence<int, K...>) {
  (f(std::integral_constant<int, K>{}), ...);
}

#define DPP_ROW_NEWBCAST(n) (0x150 + (n))

// Inclusive prefix minimum over each kSeg-lane segment (lane order).
template <int kSeg>
__device__ __forceinline__ int seg_incl_min(int v) {
  if constexpr (kSeg == 64) {
    return wave_incl_min(v);
  } else {
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_SHR(1), 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_SHR(2), 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_SHR(4), 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_SHR(8), 0xf, 0xf, false));
    if constexpr (kSeg == 32)
      v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_BCAST15, 0xa, 0xf, false));
    return v;
  }
}

// Value of the previous lane of the segment (its lane t = 0 receives fill).
template <int kSeg>
__device__ __forceinline__ int seg_shr1(int v, int fill, int t) {
  if constexpr (kSeg == 16) {
    return __builtin_amdgcn_update_dpp(fill, v, DPP_ROW_SHR(1), 0xf, 0xf, false);
  } else {
    const int u = wave_shr1(v, fill);
    return kSeg == 64 || t != 0 ? u : fill;
  }
}

// Value of set k / 16 in lane k % 16 of this lane's 16-lane row.
template <int k, int kSets>
__device__ __forceinline__ int32_t row_meta(const int32_t (&m)[kSets]) {
  return __builtin_amdgcn_update_dpp(0, m[k / 16], DPP_ROW_NEWBCAST(k % 16), 0xf, 0xf, false);
}

// kCost: the cost form, with the substitutions of the row scan (Q(c) from
// the column tree's prefix sums in place of t, the row node's vertical cost
// in place of 1, a rename gather on tree cells).
template <int kSeg, bool kCost>
__global__ __launch_bounds__(256) void tiny_kernel(DPArgs A, int32_t slot_ints) {
  constexpr int kPerGroup = 256 / kSeg;  // tables per workgroup of 4 waves
  constexpr int kSets = kSeg / 16;       // metadata registers per lane
  extern __shared__ uint16_t tslots[];
  __shared__ uint16_t sink[256];
  const int t = threadIdx.x & (kSeg - 1);  // this lane's column, t = cmax-1-c
  const int seg = threadIdx.x / kSeg;      // table of this lane in the workgroup
  const int64_t tix = (int64_t)blockIdx.x * kPerGroup + seg;
  const bool live = tix < A.ntasks;
  const TaskDesc dsc = A.descs[live ? tix : 0];  // idle segments redo task 0, storing nothing
  const int64_t offR = dsc.offR;
  const int64_t offC = dsc.offC;
  const NodeRec* __restrict__ rrecR = A.pool.rrec + offR;
  const NodeRec* __restrict__ crecC = A.pool.crec + offC;
  const int32_t* __restrict__ lrankC = A.pool.lrank + offC;
  const int32_t r0 = dsc.r0, c0 = dsc.c0;
  td_t* TDo = A.td + dsc.tdo;  // [r][c]
  td_t* TDt = A.td + dsc.tdt;  // [c][r]
  const int64_t ldo = dsc.ldo;
  const int64_t ldt = dsc.ldt;
  const int32_t rmax = dsc.rmax, cmax = dsc.cmax;
  const int32_t ncols = cmax - c0, nrows = rmax - r0;
  const int32_t base = dsc.base_rx & 0x7FFFFFFF;
  const int32_t lbase = dsc.lbase;
  const int32_t wb = lrankC[cmax] - lbase - 1;
  const bool rows_x = dsc.base_rx < 0;
  // Cost prefix sums of the column (Hpre) and row (Vpre) trees; hq, hc, vr
  // as in the row scan.
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
  const int32_t rowlen = wb + 1;
  uint16_t* slots = tslots + seg * (2 * slot_ints);

  // This lane's column (as in the row scan, one element).
  const int32_t c = max(cmax - 1 - t, c0);
  const NodeRec cr = crecC[c];  // orl(c), label, leaf rank at orl(c), leaf rank of c-1 | c-1 a leaf
  const int32_t oc = cr.orl;
  const int32_t labc = cr.label;
  const bool tree_col = oc == cmax - 1;
  int32_t hcol = 0, hfar = 0;  // (kCost) Hpre[c], Hpre[oc + 1]
  if constexpr (kCost) {
    const CostRec cc = A.pool.ccrec[offC + c];
    hcol = rows_x ? cc.ins : cc.del;
    hfar = rows_x ? cc.ins_end : cc.del_end;
  }
  const int32_t bfar = tree_col ? -1 : kCost ? hc - hfar : cmax - oc - 1;
  const int32_t foff = tree_col ? wb : cr.x - lbase;
  const bool col_ok = live && t < ncols;
  const bool writes = col_ok && c > c0 && cr.y < 0;
  uint16_t* const wdst_rel = writes ? slots + ((cr.y & 0x7FFFFFFF) - lbase) : sink + threadIdx.x;
  int32_t negt = kCost ? hcol - hq : -t;
  asm("" : "+v"(negt));

  // Metadata of rows t % 16 + 16 s (rows past the table read row r0).
  int32_t mlab[kSets], mrf[kSets], mslot[kSets], mvp[kSets];
#pragma unroll
  for (int s = 0; s < kSets; ++s) {
    const int32_t r = max(rmax - 1 - ((t & 15) + 16 * s), r0);
    const NodeRec rc = rrecR[r];  // orl(r), label, kdep(r), kdep(r-1) | r-1 a leaf
    const int32_t orr = rc.orl, kd = rc.x;
    const int32_t kdp = rc.y & 0x7FFFFFFF;
    const int32_t fs = (orr + 1 < rmax) ? kd - base - 1 : 0;
    const bool saved = r > r0 && rc.y < 0;
    mlab[s] = rc.label;
    mrf[s] = orr + 1;
    mslot[s] = fs | (saved ? (((kdp - base - 1) << 16) | (int32_t)0x80000000) : 0);
    mvp[s] = 0;
    if constexpr (kCost) {
      const CostRec vc = A.pool.ccrec[offR + r];
      mvp[s] = rows_x ? vc.del : vc.ins;  // Vpre[r]
    }
  }
  // TD of this lane's column for every row (row k at r = rmax-1-k).
  int32_t tdv[kSeg];
#pragma unroll
  for (int k = 0; k < kSeg; ++k)
    tdv[k] = k < nrows ? TDo[(int64_t)(rmax - 1 - k) * ldo + c] : 0;

  // Rows of the longest table of this wave.
  int32_t nmax = __builtin_amdgcn_readlane(nrows, 0);
#pragma unroll
  for (int s = 1; s < 64 / kSeg; ++s) nmax = max(nmax, __builtin_amdgcn_readlane(nrows, s * kSeg));

  // F[r+1][c] + (vertical cost of row r) - Q(c): 2 with unit costs.
  int32_t Fpm = kCost ? (hc - hq) + (vr - Vpre[rmax - 1]) : 2;
  int32_t left_prev = 0;    // F[r+1][cmax]
  int32_t vp_prev = vr;     // kCost: Vpre of the previous row
  // Row k (a compile-time index: it selects the DPP broadcast lane).
  auto row = [&](auto kc) {
    constexpr int k = decltype(kc)::value;
    if (k >= nmax) return;  // uniform
    const bool act = k < nrows;
    const int32_t r = rmax - 1 - k;
    const int32_t labr = row_meta<k>(mlab);
    const int32_t Rf = row_meta<k>(mrf);
    const int32_t sl = row_meta<k>(mslot);
    const bool tree_row = Rf == rmax;
    // Vertical costs of this row and of the next, and F[r][cmax] (unit
    // costs: 1, 1 and rmax - r).
    int32_t vcur = 1, vnext = 1, frc = rmax - r;
    if constexpr (kCost) {
      const int32_t vpr = row_meta<k>(mvp);
      const int32_t vpn = row_meta<k + 1 < kSeg ? k + 1 : k>(mvp);
      vcur = vp_prev - vpr;
      vnext = vpr - vpn;
      frc = vr - vpr;
      vp_prev = vpr;
    }
    // F[r+1][c+1] - Q(c+1): the left neighbour's previous F (lane t-1), or
    // the boundary F[r+1][cmax] for t = 0.
    const int32_t fpr = seg_shr1<kSeg>(Fpm - vcur - negt, left_prev, t);
    int32_t rename;
    if constexpr (kCost)
      rename = A.ren[(rows_x ? labr * A.alphabet + labc : labc * A.alphabet + labr) &
                     (tree_col ? -1 : 0)];
    else
      rename = (int32_t)(labr != labc);
    const int32_t diag = fpr + negt + rename;
    const int32_t sv = slots[(sl & 0xFFFF) * rowlen + foff];
    const int32_t far = (tree_row ? bfar : sv) + tdv[k] + negt;
    const int32_t dm = tree_row && tree_col ? diag : far;
    const int32_t carry = kCost ? frc + (hc - hq) : rmax - r + 1;
    const int32_t h = min(carry, seg_incl_min<kSeg>(min(dm, Fpm)));  // F - Q(c)
    if (act) {
      Fpm = h + vnext;
      left_prev = frc;
      if (tree_row && tree_col && col_ok) {
        TDo[(int64_t)r * ldo + c] = (td_t)(h - negt);
        TDt[(int64_t)c * ldt + r] = (td_t)(h - negt);
      }
      if (sl < 0) {
        uint16_t* wrow = slots + ((sl >> 16) & 0x7FFF) * rowlen;
        *(writes ? wdst_rel + (wrow - slots) : wdst_rel) = (uint16_t)(h - negt);
        if (t == 0) wrow[wb] = (uint16_t)frc;
      }
    }
  };
  static_for(row, std::make_integer_sequence<int, kSeg>{});
}

template <int kSeg>
void launch_tiny_seg(const DPArgs& a, int slot_bytes, hipStream_t s) {
  constexpr int kPerGroup = 256 / kSeg;
  const int slot_ints = (slot_bytes + 3) / 4;  // per table, in 4-byte units
  constexpr int64_t kChunk = kGridThreads / 256 * kPerGroup;
  for (int64_t off = 0; off < a.ntasks; off += kChunk) {
    DPArgs c = a;
    c.tasks = a.tasks + off;
    c.descs = a.descs + off;
    c.ntasks = std::min(kChunk, a.ntasks - off);
    const dim3 grid((unsigned)((c.ntasks + kPerGroup - 1) / kPerGroup));
    const size_t lds = (size_t)kPerGroup * slot_ints * 4;
    if (a.costs)
      hipLaunchKernelGGL((tiny_kernel<kSeg, true>), grid, dim3(256), lds, s, c, slot_ints);
    else
      hipLaunchKernelGGL((tiny_kernel<kSeg, false>), grid, dim3(256), lds, s, c, slot_ints);
  }
}

void launch_tiny(int form, const DPArgs& a, int slot_bytes, hipStream_t s) {
  switch (form) {
    case 0: launch_tiny_seg<16>(a, slot_bytes, s); break;
    case 1: launch_tiny_seg<32>(a, slot_bytes, s); break;
    default: launch_tiny_seg<64>(a, slot_bytes, s); break;
  }
}

// Arena offsets of every column-blocked task of a batch, in bucket order
// (level, then form), and the words of the level that takes most: levels run
// one after another and every launch has its own epoch, so each starts at
// offset 0 (one workgroup).
__global__ __launch_bounds__(1024) void xl_layout_kernel(XLLayoutArgs A) {
  __shared__ unsigned long long part[1024];
  __shared__ unsigned long long run;
  const int tid = threadIdx.x;
  unsigned long long most = 0;
  int64_t ord = 0;
  for (int L = 0; L < A.nlevels; ++L) {
    if (tid == 0) run = 0;
    __syncthreads();
    for (int k = 0; k < kNumXLForms; ++k) {
      const int bkt = bucket_of(L, kFirstXLClass + k, 0);
      const int64_t cnt = (int64_t)A.counts[bkt];
      const int64_t start = (int64_t)A.cursor[bkt] - cnt;  // cursors end past the bucket
      for (int64_t c0 = 0; c0 < cnt; c0 += 1024) {
        const int64_t idx = c0 + tid;
        unsigned long long w = 0;
        if (idx < cnt) {
          const uint64_t task = A.tasks[start + idx];
          w = (unsigned long long)xl_words(xl_geom(A.pool, A.pairs[task_pair(task)], task,
                                                   xl_bw(k)));
        }
        part[tid] = w;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {
          const unsigned long long v = tid >= off ? part[tid - off] : 0;
          __syncthreads();
          part[tid] += v;
          __syncthreads();
        }
        if (idx < cnt) A.off[ord + idx] = (int64_t)(run + part[tid] - w);
        __syncthreads();
        if (tid == 1023) run += part[1023];
        __syncthreads();
      }
      ord += cnt;
    }
    if (tid == 0) most = max(most, run);
  }
  if (tid == 0) *A.total = most;
}

void launch_xl_layout(const XLLayoutArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(xl_layout_kernel, dim3(1), dim3(1024), 0, s, a);
}

// Zero fill for a newly grown column-blocked arena (epoch 0 is never used).
__global__ void xl_zero_kernel(unsigned long long* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}
void launch_xl_zero(unsigned long long* p, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(xl_zero_kernel, dim3(1024), dim3(256), 0, s, p, n);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
template <int W>
static void launch_shared(const DPArgs& a, int lds_bytes, hipStream_t s) {
  // One table per workgroup: a long task list goes in pieces.
  constexpr int64_t kChunk = kGridThreads / (64 * W);
  for (int64_t off = 0; off < a.ntasks; off += kChunk) {
    DPArgs c = a;
    c.tasks = a.tasks + off;
    c.descs = a.descs + off;
    c.ntasks = std::min(kChunk, a.ntasks - off);
    if (a.costs)
      hipLaunchKernelGGL((rowscan_kernel<W, true>), dim3((unsigned)c.ntasks),
                         dim3(64 * W), (size_t)lds_bytes, s, c);
    else
      hipLaunchKernelGGL((rowscan_kernel<W, false>), dim3((unsigned)c.ntasks),
                         dim3(64 * W), (size_t)lds_bytes, s, c);
  }
}

// Grants every row-scan instantiation the LDS it may ask for (> 64 KiB needs
// an explicit attribute).
template <int W>
static hipError_t allow_lds(int limit) {
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&rowscan_kernel<W, false>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, limit);
  if (e != hipSuccess) return e;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&rowscan_kernel<W, true>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, limit);
}
hipError_t forest_init_attributes(int limit) {
  hipError_t e = scan_init_attributes(limit);
  if (e != hipSuccess) return e;
  if ((e = allow_lds<4>(limit)) != hipSuccess) return e;
  if ((e = allow_lds<8>(limit)) != hipSuccess) return e;
  return allow_lds<16>(limit);
}

// Launches one (class, task list). Returns false for a class without a kernel.
bool launch_forest(int cls, const DPArgs& a, int lds_bytes, hipStream_t s) {
  if (a.ntasks <= 0) return true;
  if (is_tiny(cls)) {
    launch_tiny(cls - kClassTiny, a, lds_bytes, s);
    return true;
  }
  if (cls >= 1 && cls <= kNumRowClasses) {
    launch_scan((cls - 1) / 5, (cls - 1) % 5, a, lds_bytes, s);
    return true;
  }
  if (cls == kClassSweep) {
    launch_sweep(a, lds_bytes, s);
    return true;
  }
  switch (cls - kClassShared) {
    case 0: launch_shared<4>(a, lds_bytes, s); return true;
    case 1: launch_shared<8>(a, lds_bytes, s); return true;
    case 2: launch_shared<16>(a, lds_bytes, s); return true;
    default: break;
  }
  if (cls >= kFirstXLClass && cls < kFirstXLClass + kNumXLForms) {
    launch_xl(cls - kFirstXLClass, a, lds_bytes, s);
    return true;
  }
  return false;
}

}  // namespace xted
