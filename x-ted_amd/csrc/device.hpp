// Device-side data layout shared by the HIP kernels and the host engine.
//
// Tree pool (structure of arrays, all int32, one region of n+1 entries per
// tree starting at node_off):
//   node arrays    parent/label/orl/kdep/kdn  [node_off + i], i in [0, n)
//   leaf rank      lrank                      [node_off + i], i in [0, n]
//   keyroot arrays kr/krkd/krsize/krleaf      [node_off + k], k in [0, K)
//                  (keyroots in descending preorder; K <= n)
//   sorted keyroots skr/skd/ssize/sleaf       [node_off + k], k in [0, K):
//                  the K1 leaf keyroots first, then the others by ascending
//                  nesting height d (and size band within a height), those
//                  of height d at [K1 + kdoff[d], K1 + kdoff[d+1])
//   spre           [node_off + k], k in [0, K]: prefix sums of ssize
//   kdoff          [node_off + d], d in [0, kdmax+1]
// A pair owns a tree-distance table TD (m x n, row-major, preorder) and its
// transpose TDT (n x m); both live in one arena of 16-bit entries (td_t) at
// td_off / tdt_off.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define XTED_HD __host__ __device__
#else
#define XTED_HD
#endif

namespace xted {

struct TreeMeta {
  int64_t node_off;  // offset of the tree's region (n+1 entries)
  int32_t n;         // node count
  int32_t K;         // keyroot count
  int32_t kdmax;     // keyroot nesting height of the root
  int32_t nleaves;   // leaf count
  int32_t K1;        // keyroots that are leaves
  int32_t pad;
};

// One entry of a tree-distance table in the arena. Every entry is at most
// the cost of deleting all of x and inserting all of y: with unit costs
// n_x + n_y <= 65534 (pool trees have at most 32767 nodes), under a cost
// model at most 65535 (checked per pair on the host). So 16 bits hold every
// value exactly, and each forest cell reads 2 bytes of HBM instead of 4;
// the kernels compute in int32 and the tables handed to a caller are int32.
using td_t = uint16_t;

struct PairMeta {
  int32_t tx, ty;   // tree ids (rows = x, columns = y)
  int64_t td_off;   // TD  offset (m*n entries)
  int64_t tdt_off;  // TDT offset (n*m entries)
};

// What a forest kernel needs to start one table, written by the plan next to
// the table's task word so that the kernel starts from one 64-byte read
// instead of a chain of dependent reads (task, pair, trees, subtree ends).
// The table is oriented with its short side as rows.
struct alignas(16) TaskDesc {
  int64_t tdo;       // offset of TD in the row layout ([r][c])
  int64_t tdt;       // and in the column layout ([c][r])
  int64_t offR;      // node offset of the row tree in the pool
  int64_t offC;      // and of the column tree
  int32_t ldo, ldt;  // row lengths of the two layouts
  int32_t r0, c0;    // the table's keyroots (row tree, column tree)
  int32_t rmax, cmax;
  int32_t base_rx;   // kdep of r0; bit 31 set when the rows are x's nodes
  int32_t lbase;     // leaves of the column tree before c0
};
static_assert(sizeof(TaskDesc) == 64, "TaskDesc is one 64-byte read");

// What a forest kernel reads of one node, in one 16-byte load: as a column
// of a table (crec: x = leaf rank at orl(i), y = leaf rank of i-1) or as a
// row (rrec: x = kdep(i), y = kdep(i-1)); bit 31 of y is set when i-1 is a
// leaf. Entry 0's y is 0.
struct alignas(16) NodeRec {
  int32_t orl, label, x, y;
};

// Under a cost model, a node's deletion / insertion cost prefix sums at
// itself and just past its subtree (at orl(i) + 1), in one 16-byte load.
struct alignas(16) CostRec {
  int32_t del, ins, del_end, ins_end;
};

// Pointers to the pool arrays (device addresses).
struct PoolView {
  const int32_t* parent;
  const int32_t* label;
  const int32_t* orl;
  const int32_t* kdep;   // nesting depth of the keyroot that owns node's right path
  const int32_t* kdn;    // keyroot nesting height at keyroots, -1 elsewhere
  const int32_t* lrank;  // leaves strictly before node (n+1 entries per tree)
  const int32_t* kr;     // keyroot node ids, descending
  const int32_t* krkd;   // nesting height per keyroot
  const int32_t* krsize; // subtree size per keyroot
  const int32_t* krleaf; // leaves in subtree per keyroot
  const int32_t* skr;    // sorted keyroots (leaf keyroots, then by nesting height)
  const int32_t* skd;
  const int32_t* ssize;
  const int32_t* sleaf;
  const int32_t* spre;   // prefix sums of ssize (K+1 entries)
  const int32_t* kdoff;
  const int32_t* rtop;   // keyroot at the top of node's right path
  const int32_t* pdel;   // cost mode: deletion costs of nodes [0, i) (n+1 entries per tree)
  const int32_t* pins;   // cost mode: insertion costs of nodes [0, i)
  const NodeRec* crec;   // per node, as a table column
  const NodeRec* rrec;   // per node, as a table row
  const CostRec* ccrec;  // cost mode: per node, pdel / pins at it and past its subtree
  const TreeMeta* trees;
};

// A table task: pair id (24 bits) | x keyroot node (20 bits) | 1 when the rows
// are x's nodes | y keyroot node (19 bits). Trees of a pool have at most
// 32,767 nodes and a batch at most 2^24 pairs.
constexpr int kTaskPairBits = 24;
XTED_HD inline uint64_t task_pack(uint32_t pair, uint32_t i0, uint32_t j0, bool rows_x) {
  return ((uint64_t)pair << 40) | ((uint64_t)i0 << 20) | ((uint64_t)rows_x << 19) | (uint64_t)j0;
}
XTED_HD inline uint32_t task_pair(uint64_t t) { return (uint32_t)(t >> 40); }
XTED_HD inline uint32_t task_i0(uint64_t t) { return (uint32_t)(t >> 20) & 0xFFFFFu; }
XTED_HD inline uint32_t task_j0(uint64_t t) { return (uint32_t)t & 0x7FFFFu; }

// ---- granularity classes ----------------------------------------------------
// Class 0: leaf (a table whose short side is one node, a leaf keyroot),
//   evaluated in closed form by the leaf kernel, one line per leaf keyroot.
// Classes 1..25: workgroup row scan with W = 2^wi waves and C = 2^ci columns
//   per lane, class = 1 + wi*5 + ci (wi, ci in 0..4).
// Class 26: tables no form below can hold (an error).
// Classes 27..32: column-blocked form for tables too wide or too LDS-hungry
//   for one workgroup: blocks of xl_bw(k) columns, one workgroup each,
//   chained per row through device memory, class = 27 + k.
// Classes 33..35: tiny tables of at most 16, 32 or 64 columns, one per 16-,
//   32- or 64-lane segment of a wave (four, two or one to a wave).
// Classes 36..38: on-chip tables of deep column keyroots, whose waves' imports
//   do not fit LDS beside the slot rows: slot rows shared by 4, 8 or 16 waves,
//   with a barrier per row.
// Class 39: tables swept by one wave, kSweepCols columns at a time.
constexpr int kClassLane = 0;  // the leaf class
constexpr int kNumRowClasses = 25;
constexpr int kClassXL = 26;
constexpr int kFirstXLClass = 27;
constexpr int kNumXLForms = 6;
constexpr int kClassTiny = kFirstXLClass + kNumXLForms;  // 33: the first tiny form
constexpr int kNumTinyForms = 3;
constexpr int kClassShared = kClassTiny + kNumTinyForms;  // 36: the first shared-slot form
constexpr int kNumSharedForms = 3;
constexpr int kSweepForm = 3;  // column-blocked form of the same width
constexpr int kClassSweep = kClassShared + kNumSharedForms;  // 39
constexpr int kSweepCols = 512;
constexpr int kNumClasses = kClassSweep + 1;  // 40
XTED_HD inline bool is_tiny(int cls) { return cls >= kClassTiny && cls < kClassShared; }
XTED_HD inline bool is_shared(int cls) { return cls >= kClassShared && cls < kClassSweep; }
// Shared-slot form k: 4, 8 or 16 waves of 8 columns per lane.
XTED_HD inline int shared_waves(int k) { return 4 << k; }
XTED_HD inline int shared_cols(int k) { return 64 * 8 * shared_waves(k); }
// Lanes per table (and most columns) of tiny form k.
XTED_HD inline int tiny_seg(int k) { return 16 << k; }
// Slot bytes of one table of tiny form k: 32 KiB per workgroup of 256 lanes.
XTED_HD inline int64_t tiny_max_lds(int k) { return (int64_t)2048 << k; }
// Column-blocked forms: waves and columns per lane of one block. The two
// narrowest serve deep trees, whose slot rows leave little LDS: one wave's
// edges take the least.
XTED_HD constexpr int xl_waves(int k) { return k <= 2 ? 8 : k == 3 ? 4 : 1; }
XTED_HD constexpr int xl_cpl(int k) { return k == 0 ? 8 : k == 1 || k == 4 ? 4 : 2; }
XTED_HD inline int xl_bw(int k) { return 64 * xl_waves(k) * xl_cpl(k); }  // 4096 .. 128
// Column-blocked tables with at most this many rows are swept block after
// block by one workgroup (forms of at most 1024 columns), with no waits
// between workgroups; taller ones pipeline one workgroup per block. Measured
// on the 20,000-node pair's tables of more than 8192 columns, ms a pair with
// 256, 128, 64, 32 and 16 rows: 76.9, 75.1, 74.1, 73.7, 74.0.
constexpr int32_t kXLSeqRows = 32;  // default of ClassRule::xl_seq_rows
// A table that fits one workgroup goes in blocks for being tall only above
// this: filling the pipeline of blocks takes about 16 rows and 3 us a block.
// Device time in ms of deep pairs of 5000 columns with 100, 237, 300, 400, 600,
// 1000, 2000 rows: in one workgroup 6.2, 12.4, 14.4, 17.7, 33.2, 58, 102; in
// blocks from 33 rows on 9.4, 14.2, 15.8, 18.5, 25.9, 39, 75. Of 1500 columns,
// two blocks: 2.0, 3.4, 3.8, 4.6, 7.2, 11.8, 23.4 and 2.3, 3.9, 4.2, 5.1, 8.0,
// 12.8, 23.6. Pairs of wide trees and of random ones lie alike. The lines cross
// at some 450 rows of 5000 columns and 2000 of 1500; with 256 no shape loses more
// than 15%.
constexpr int32_t kTallBlockRows = 256;
constexpr int kFirstSeqXLForm = 2;
// Far values a block takes from earlier blocks are indexed by the nesting
// depth of their right path below the column keyroot: at most this many.
constexpr int kMaxImports = 256;
XTED_HD inline int row_class(int wi, int ci) { return 1 + wi * 5 + ci; }

// Each (level, class) bucket is cut into size bands, largest tables first,
// so that a launch starts its longest tables first and its last workgroups
// are short ones (column-blocked classes use band 0 only). The plan's
// buckets are (level, class, band), and one launch covers kRowBands
// consecutive bands.
//
// A launch gives every workgroup the largest slot storage of its tables,
// and LDS is what bounds how many workgroups a CU holds. In the 4096-pair
// batch a W = 2 launch's tables need 2 KiB of slot rows on average and its
// largest 28 KiB, which held a CU to 5 workgroups where registers allow 10.
// So with mode 2 the row-scan tables that need more than light_per_wave
// bytes per wave (8 KiB is one workgroup's share of LDS at 20 waves per CU)
// go to bands of their own (kRowBands .. 2*kRowBands-1), and a (level,
// class) takes two launches: light tables and heavy ones.
constexpr int kRowBands = 4;
constexpr int kBands = 2 * kRowBands;
constexpr int kLightPerWave = 10 * 1024;  // default of Context::light_per_wave
// mode 0: band 0 (plan order); 1: row bands; 2: row bands, light / heavy.
XTED_HD inline int size_band(int cls, int rows, int64_t lds, int mode, int light_per_wave) {
  if (mode == 0) return 0;
  if (is_tiny(cls)) {
    const int q = tiny_seg(cls - kClassTiny) / 4;  // row bands of a quarter segment
    return rows > 3 * q ? 0 : rows > 2 * q ? 1 : rows > q ? 2 : 3;
  }
  if ((cls < 1 || cls > kNumRowClasses) && cls != kClassSweep) return 0;
  const int rb = rows >= 256 ? 0 : rows >= 64 ? 1 : rows >= 16 ? 2 : 3;
  const int waves = cls == kClassSweep ? 1 : 1 << ((cls - 1) / 5);
  const int64_t light = (int64_t)waves * light_per_wave;
  return mode == 2 && lds > light ? kRowBands + rb : rb;
}
XTED_HD inline int bucket_of(int level, int cls, int band) {
  return (level * kNumClasses + cls) * kBands + band;
}

// Words of a column-blocked table are laid out in whole 128-byte L2 lines.
constexpr int32_t kXLLineWords = 16;
XTED_HD inline int32_t xl_pad(int32_t w) { return (w + kXLLineWords - 1) & ~(kXLLineWords - 1); }

// Saved-row slots are uint16 (F <= |subtree x| + |subtree y| < 65536).
// LDS budget for the slots of one table, per wave of its workgroup.
constexpr int kLdsPerWave = 10 * 1024;
constexpr int kLdsMaxTable = 150 * 1024;
constexpr int kMaxRowWaves = 16;
constexpr int kMaxCols = 64 * 16 * kMaxRowWaves;  // 16384
// Widest table the on-chip forms take (W = 16 waves x 8 columns per lane;
// 16 columns per lane at 16 waves would spill); wider tables are column-blocked.
constexpr int kMaxOnChipCols = 64 * 8 * kMaxRowWaves;  // 8192

// 16-lane form only by default: with the 32-lane form as well the 96-tree
// distance matrix took 99.8 against 99.9 ms, 128 pairs of 100-600 nodes 19.0
// against 19.0, 1024 pairs under a cost model 55.4 against 53.8. The tuned
// rule of the 4096-pair batch (x-ted_amd/tuning.json) turns it on (96.5
// against 99.6 ms when it was tuned). The 64-lane form ran 8% slower there (4
// waves per SIMD for its 64 TD registers per lane).
constexpr int32_t kTinyDefault = 1;

// A row of up to 256 columns takes one wave about as long as several
// (a 120-node pair's root table 0.21 us a row either way).
constexpr int32_t kTallCols = 256;

// How a table is split, by its level's interior cells (level_cells_kernel). A
// level takes the longer of its work spread over the chip and its slowest
// table's rows, one after another. A table whose rows take longer than the
// level's work ("tall": few cells in the level per row of its own) is split
// for speed: fewer columns a lane, and past a block's width a pipeline of
// workgroups, since a row takes the less the fewer columns a lane holds and
// waves a compute unit has (1000 columns: 0.38 us with 16 a lane, 0.32 with 8,
// 0.24 with 4, 0.21 with 2; 4000: 0.39 in one workgroup of 16 waves, 0.45 /
// 0.32 / 0.27 / 0.26 in blocks of 4096 / 2048 / 1024 / 512). The others are
// split for throughput. Measured in ms with the bound for 2 columns a lane at
// 4e4, 1.2e5, 4e5 cells: 20,000-node pair 93, 91, 91; deep 1000-node pair 7.9,
// 7.7, 7.6; 128 pairs of 100-600 nodes 20.4, 20.8, 20.1. With the bound for 4
// at 3e5, 1.5e6, 3e6, 1e7: 20,000-node pair 94, 91, 91, 87; 1024 pairs of
// 100-1000 nodes under a cost model 64, 57, 55, 55; 4096 such pairs with unit
// costs 90, 90, 90, 98.
constexpr int64_t kTall2Cells = 120000;
constexpr int64_t kTall4Cells = 3000000;
constexpr int kTallRows = 64;
// A wide table that is at most this part of its level's cells is swept by one
// wave: the 20,000-node pair took, with shares of 1/64, 1/256, 1/1024, 1/8192 and
// no table swept, 91, 92, 88, 105 and 139 ms. Its edges and slot rows take at
// most kSweepLds, so that 8 such waves share a compute unit (10, 20, 40 and 80
// KiB: 66 ms each, and the matrix of 96 trees 92; few tables come near).
constexpr int64_t kSweepShare = 1024;
constexpr int kSweepLds = 20 * 1024;
constexpr int kTall2Form = 2, kTall4Form = 1;

// Tuning knobs carried by the plan builder (autotuner writes these).
struct ClassRule {
  int32_t lds_per_wave;  // bytes of slot storage one wave may own
  int32_t min_waves;     // lower bound on W for tables with >= wide_cols columns
  int32_t wide_cols;
  int32_t lds_max;       // slot bytes one workgroup may hold (device limit)
  int32_t max_cpl;       // most columns per lane before a table gets more waves
  int32_t xl_seq_rows = kXLSeqRows;  // column-blocked tables this short: one workgroup
  // Tiny forms in use (bit k: tables of at most tiny_seg(k) columns take
  // form k, the narrowest that holds them).
  int32_t tiny = kTinyDefault;
  // Widest form a pipelined column-blocked table may use (0: 4096-column
  // blocks, 1: 2048, 2: 1024, ...): narrower blocks put more workgroups on
  // one table.
  int32_t xl_first = 0;
  // Tall tables: those of at least kTallRows rows and more than kTallCols
  // columns in a level of at most tall2 (tall4) cells per row of theirs take
  // at most 2 (4) columns per lane, and where blocks is set go in blocks of at
  // most form kTall2Form (kTall4Form).
  int64_t tall2 = kTall2Cells, tall4 = kTall4Cells;
  int64_t sweep = kSweepShare;
  int32_t blocks = 1;
};

// A new context's settings (those of xted_set_tuning first). Up to 16 columns
// per lane: the distance matrix of 96 trees of 100-1000 nodes took 99.9 ms
// against 110.8 with 8, and 89.4 with level_align 1; under a cost model, whose
// 16-column form holds 204 VGPRs, 4096 pairs took 120 against 146, 1024 pairs
// 44 against 49.
constexpr ClassRule kDefaultRule{kLdsPerWave, 1, 1 << 30, kLdsMaxTable, 16};
constexpr int32_t kDefaultTailPairs = 32;
constexpr int32_t kDefaultLevelAlign = 1;
constexpr int32_t kDefaultSizeBands = 1;

XTED_HD inline int ilog2_ceil(int v) {
  int r = 0;
  while ((1 << r) < v) ++r;
  return r;
}

// On-chip row scan of w waves: entries of the ring between two waves, and the
// LDS bytes of a table whose row keyroot has nesting height slots (at least 1)
// and whose column keyroot has leaves_c leaves and nesting height kd_c: one
// uint16 row per slot with every far column (the leaves but the last), and
// per wave the boundary entry, a sink and, with several waves, the kd_c + 1
// values imported from earlier blocks; and w + 1 rings of a carry, the
// imports and a trash word per entry, and w + 2 progress words.
constexpr int kEdgeRows = 8;
XTED_HD inline int64_t scan_lds_need(int slots, int leaves_c, int kd_c, int w) {
  if (w == 1) return (int64_t)slots * (leaves_c + 1) * 2;
  return (int64_t)slots * (leaves_c - 1 + w * (kd_c + 3)) * 2 +
         (int64_t)(w + 1) * kEdgeRows * (kd_c + 3) * 4 + 8 * (w + 2);
}

// The same of one block of a column-blocked table of form k, whose blocks
// have at most own far columns of their own each.
XTED_HD constexpr int xl_edge_rows(int w) { return w == 1 ? 4 : kEdgeRows; }
XTED_HD inline int64_t xl_lds_need(int slots, int own, int kd_c, int k) {
  const int w = xl_waves(k);
  return (int64_t)slots * (own + w * (kd_c + 3)) * 2 +
         (int64_t)(w + 1) * xl_edge_rows(w) * (kd_c + 3) * 4 + 8 * (w + 2);
}
// The same of a swept table (kClassSweep) of that many rows: the slot rows of
// one block, and one edge entry per row.
XTED_HD inline int64_t sweep_lds_need(int slots, int own, int kd_c, int rows) {
  return (int64_t)slots * (own + kd_c + 3) * 2 + (int64_t)(rows + 1) * (kd_c + 3) * 4;
}
// Which of these forms, from form k on, takes a table: the widest whose blocks
// fit lds_max; the narrowest takes every table whose slot rows fit it by the
// bound min(leaves, columns) on a block's far columns, its edges (at most
// kXLEdgeBytes) coming on top of lds_max (a workgroup may have 160 KiB). -1:
// none. own(k): the most far columns of any one block of form k. *need
// receives the form's bytes.
constexpr int kXLEdgeBytes = 2 * xl_edge_rows(1) * (kMaxImports + 2) * 4 + 8 * 3;
template <class Own>
XTED_HD inline int xl_form(int slots, int kd_c, int leaves_c, int k, int lds_max, const Own& own,
                           int64_t* need) {
  constexpr int kLast = kNumXLForms - 1;
  const int most = leaves_c < xl_bw(kLast) ? leaves_c : xl_bw(kLast);
  if (kd_c + 1 > kMaxImports || (int64_t)slots * (most + kd_c + 3) * 2 > lds_max) return -1;
  for (; k < kLast; ++k) {
    *need = xl_lds_need(slots, own(k), kd_c, k);
    if (*need <= lds_max) return k;
  }
  *need = xl_lds_need(slots, most, kd_c, kLast);
  return kLast;
}

// Class of table (a x b): kd_r / kd_c / leaves_c (row keyroot height, column
// keyroot height and leaves) of its oriented form size its LDS storage, with
// own (xl_form) as blocks; level_cells(): the interior cells of its level. Single-row tables are the leaf class when leaf_form
// is set. *need receives the slot bytes of the chosen form.
template <class Cells, class Own>
XTED_HD inline int table_class(int a, int b, int kd_r, int kd_c, int leaves_c, bool leaf_form,
                               const ClassRule& rule, const Cells& level_cells, const Own& own,
                               int64_t* need) {
  const int rows = a <= b ? a : b;
  const int cols = a <= b ? b : a;
  const int slots = kd_r > 1 ? kd_r : 1;
  const int64_t lds_need = scan_lds_need(slots, leaves_c, kd_c, 1);
  *need = lds_need;
  if (rows == 1 && leaf_form) return kClassLane;
  for (int k = 0; k < kNumTinyForms; ++k)
    if ((rule.tiny >> k & 1) && cols <= tiny_seg(k) && lds_need <= tiny_max_lds(k))
      return kClassTiny + k;
  const int cpl_cap = rule.max_cpl < 8 ? rule.max_cpl : 8;
  int wi = 0;
  while (wi < 4 && lds_need > (int64_t)rule.lds_per_wave * (1 << wi)) ++wi;
  while (wi < 4 && cols > 64 * rule.max_cpl * (1 << wi)) ++wi;
  int tall = 0;
  const int64_t cells = cols > kTallCols ? level_cells() : 0;
  if (rows >= kTallRows && cols > kTallCols) {
    tall = cells <= rows * rule.tall2 ? 2 : cells <= rows * rule.tall4 ? 4 : 0;
    while (tall && wi < 4 && cols > 64 * tall * (1 << wi)) ++wi;
  }
  // Waves a table gets at least, by its columns (a power of two).
  const int wide = cols >= rule.wide_cols ? rule.min_waves : 1;
  int least = 1;
  while (least < kMaxRowWaves && (least < wide || cols > 64 * rule.max_cpl * least)) least *= 2;
  if (wide <= 1 && rule.max_cpl >= kSweepCols / 64 && !tall && wi > 0 && cols > 2 * kSweepCols &&
      cells >= (int64_t)rows * cols * rule.sweep) {
    const int64_t n = sweep_lds_need(slots, own(kSweepForm), kd_c, rows);
    if (n <= kSweepLds && n <= rule.lds_max) {
      *need = n;
      return kClassSweep;
    }
  }
  while (wi < 4 && (1 << wi) < least) ++wi;
  // More waves hold more imports: no more than fit, down to the least.
  while ((1 << wi) > least && scan_lds_need(slots, leaves_c, kd_c, 1 << wi) > rule.lds_max) --wi;
  const int first_tall = tall == 2 ? kTall2Form : tall == 4 ? kTall4Form : 0;
  const int first = rule.xl_first > first_tall ? rule.xl_first : first_tall;
  auto blocked = [&](int k) {
    const int form = xl_form(slots, kd_c, leaves_c, k, rule.lds_max, own, need);
    return form < 0 ? kClassXL : kFirstXLClass + form;
  };
  // Tall tables go in blocks where they are wider than one, and where LDS
  // leaves them more columns per lane; in blocks of one wave, the forms for
  // deep trees, only above what 4 waves sharing their slot rows hold. (Pairs of
  // trees nested about 250 deep, ms with such blocks for narrower tables too
  // against one workgroup: 500 x 500 nodes 82 against 33, 1000 x 1000 150
  // against 83, 2000 x 2000 321 against 217. One of 3000 x 3000 nodes, 190
  // deep, above: 214 with blocks, 277 with 8 waves sharing slot rows.)
  if (tall && rule.blocks && rows > kTallBlockRows && rows > rule.xl_seq_rows &&
      (cols > xl_bw(first_tall) || cols > 64 * tall * (1 << wi))) {
    const int cls = blocked(first), k = cls - kFirstXLClass;
    if (cls != kClassXL && (xl_waves(k) > 1 || cols > shared_cols(0)) &&
        (cols + xl_bw(k) - 1) / xl_bw(k) * xl_waves(k) >= least)
      return cls;
  }
  *need = scan_lds_need(slots, leaves_c, kd_c, 1 << wi);
  if (*need > rule.lds_max && lds_need <= rule.lds_max) {
    for (int k = 0; k < kNumSharedForms; ++k) {
      if (cols <= shared_cols(k) && shared_waves(k) >= least) {
        *need = lds_need;
        return kClassShared + k;
      }
    }
  }
  // Short tables take the forms one workgroup sweeps.
  if (cols > 64 * cpl_cap * kMaxRowWaves || *need > rule.lds_max)
    return blocked(rows <= rule.xl_seq_rows ? kFirstSeqXLForm : first);
  int w = 1 << wi;
  int c = (cols + 64 * w - 1) / (64 * w);
  int ci = ilog2_ceil(c);
  return row_class(wi, ci);
}

// The class of a table of class cls while class force is forced: force where
// the table is neither the leaf kernel's nor without a form and fits it,
// whatever the rule chose (a row-scan class takes tables of up to
// kMaxOnChipCols columns), else cls.
template <class Own>
XTED_HD inline int forced_class(int force, int cls, int a, int b, int kd_r, int kd_c, int leaves_c,
                                const ClassRule& rule, const Own& own, int64_t* need) {
  const int cols = a <= b ? b : a;
  const int slots = kd_r > 1 ? kd_r : 1;
  if (cls < 1 || cls == kClassXL) return cls;
  int64_t n = 0;
  bool fits = false;
  if (force >= kFirstXLClass && force < kFirstXLClass + kNumXLForms) {
    const int k = force - kFirstXLClass;
    fits = xl_form(slots, kd_c, leaves_c, k, rule.lds_max, own, &n) == k;
  } else if (is_tiny(force)) {
    n = scan_lds_need(slots, leaves_c, 0, 1);
    fits = cols <= tiny_seg(force - kClassTiny) && n <= tiny_max_lds(force - kClassTiny);
  } else if (force >= 1 && force <= kNumRowClasses) {
    const int w = 1 << (force - 1) / 5, c = 1 << (force - 1) % 5;
    n = scan_lds_need(slots, leaves_c, kd_c, w);
    fits = cols <= 64 * w * c && cols <= kMaxOnChipCols && n <= rule.lds_max;
  }
  if (fits) *need = n;
  return fits ? force : cls;
}

}  // namespace xted
