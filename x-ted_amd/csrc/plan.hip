// Device-side level scheduler: every keyroot-pair table of every pair in a
// batch is assigned level = depth_x(k) + depth_y(l) and a granularity class,
// then scattered into (level, class) buckets, all on the device.
//
// Replaces the reference's per-level host loop (X-TED_GPU/parallel_X_TED.cu:
// 214-220 level array, :304-385 fetch_task / fetch_size_queue /
// thrust::sort_by_key / filter_new with several host syncs per level, and
// X-TED_GPU/function.cu:18-57). Here the whole plan is built once per batch
// by three kernels (count, scan, scatter) and read back with one copy of the
// bucket counts. Counts and appends are aggregated per wave and then per
// workgroup: each distinct bucket of a workgroup costs one global atomic, and
// a wave's tables of one bucket land contiguously.
#include <hip/hip_runtime.h>
#include <algorithm>

#include "kernels.hpp"

namespace xted {

constexpr int kPlanThreads = 256;

__device__ __forceinline__ int find_pair(const int64_t* blk_start, int npairs, int64_t b) {
  int lo = 0, hi = npairs - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (blk_start[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Per-table classification shared by both passes.
__device__ __forceinline__ void classify(const PlanArgs& A, const TreeMeta& tx,
                                         const TreeMeta& ty, int32_t loff, bool leaf_form, int k,
                                         int l, int* bucket,
                                         int* lds, uint32_t* i0, uint32_t* j0,
                                         unsigned long long* cells) {
  const int64_t kx = tx.node_off + k, ly = ty.node_off + l;
  const int32_t a = A.pool.ssize[kx], b = A.pool.ssize[ly];
  *cells = (unsigned long long)a * (unsigned long long)b;
  const int32_t kdx = A.pool.skd[kx], kdy = A.pool.skd[ly];
  const int32_t level = kdx + kdy + loff;
  const ClassRule& rule = A.tail_level[level] ? A.rule_tail : A.rule;
  const int32_t leaves_c = a <= b ? A.pool.sleaf[ly] : A.pool.sleaf[kx];
  int64_t need = 0;
  // With the leaf kernel off, single-row tables take the row-scan forms.
  const int64_t offC = a <= b ? ty.node_off : tx.node_off;
  const int32_t c0 = A.pool.skr[a <= b ? ly : kx], cmax = c0 + max(a, b);
  auto own = [&](int k) {
    const int32_t bw = xl_bw(k);
    int32_t most = 0;
    for (int32_t c = cmax; c > c0; c -= bw)  // the block of columns [c - bw, c)
      most = max(most, A.pool.lrank[offC + c - 1] - A.pool.lrank[offC + max(c - bw - 1, c0)]);
    return most;
  };
  auto level_cells = [&] {
    return (int64_t)(A.level_cells ? A.level_cells[level] : A.mean_cells);
  };
  int cls = table_class(a, b, a <= b ? kdx : kdy, a <= b ? kdy : kdx, leaves_c, leaf_form, rule,
                        level_cells, own, &need);
  if (A.force_class >= 0)
    cls = forced_class(A.force_class, cls, a, b, a <= b ? kdx : kdy, a <= b ? kdy : kdx, leaves_c,
                       A.rule, own, &need);
  *bucket = bucket_of(level, cls, size_band(cls, a <= b ? a : b, need, A.bands, A.light_per_wave));
  *lds = (int)need;
  *i0 = (uint32_t)A.pool.skr[kx];
  *j0 = (uint32_t)A.pool.skr[ly];
}

// Per-workgroup bucket table in LDS: the plan's global atomics go to a few
// thousand (level, class) buckets and device-scope atomics are performed
// memory-side, so they are first combined per workgroup (open addressing on
// the bucket id), and each workgroup then makes one global atomic per bucket
// it touched. A bucket that finds the table full takes the global atomics
// directly.
constexpr int kHTBits = 8;
constexpr int kHT = 1 << kHTBits;
struct PlanLds {
  int32_t key[kHT];  // bucket id, or -1
  uint32_t cnt[kHT];
  int32_t lds[kHT];
  unsigned long long cells[kHT];  // count pass: cells; scatter pass: base
};

__device__ __forceinline__ int ht_slot(PlanLds& T, int bucket, bool insert) {
  int h = (int)(((uint32_t)bucket * 0x9E3779B1u) >> (32 - kHTBits));
  for (int probe = 0; probe < kHT; ++probe) {
    int k = __hip_atomic_load(&T.key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (k == -1 && insert) {
      k = atomicCAS(&T.key[h], -1, bucket);
      if (k == -1) return h;
    }
    if (k == bucket) return h;
    if (k == -1) return -1;  // lookup: absent
    h = (h + 1) & (kHT - 1);
  }
  return -1;  // full
}

__device__ __forceinline__ void ht_clear(PlanLds& T) {
  for (int i = threadIdx.x; i < kHT; i += kPlanThreads) {
    T.key[i] = -1;
    T.cnt[i] = 0;
    T.lds[i] = 0;
    T.cells[i] = 0;
  }
}

// The tables of this workgroup: y keyroots [l_lo, l_lo + rows) of the
// pair's sorted list against all Kx x keyroots, total of them.
struct PlanChunk {
  int p, kbase, lbase, Kx, l_lo;
  int64_t total;
};
__device__ __forceinline__ PlanChunk plan_chunk(const PlanArgs& A, const TreeMeta& tx,
                                                const TreeMeta& ty, int p) {
  PlanChunk c;
  c.p = p;
  // With the leaf kernel on, tables with a leaf keyroot are not planned here
  // (the leaf kernel writes them): only the non-leaf keyroots [K1, K) of the
  // sorted lists take part.
  const bool le = A.pair_leaf ? A.pair_leaf[p] != 0 : A.lane_enable != 0;
  c.kbase = le ? tx.K1 : 0;
  c.lbase = le ? ty.K1 : 0;
  c.Kx = tx.K - c.kbase;
  const int Ky = ty.K - c.lbase;
  const int lper = max(1, A.lchunk_tables / max(c.Kx, 1));  // same as plan_blocks()
  c.l_lo = (int)(blockIdx.x - A.blk_start[p]) * lper;
  const int l_hi = min(Ky, c.l_lo + lper);
  c.total = (int64_t)max(0, l_hi - c.l_lo) * c.Kx;
  return c;
}

// Count pass: one table's count, interior cells and slot-storage need, into
// the workgroup's table. (LDS atomics of lanes on one entry are performed one
// after another, a cycle each: less than the wave-wide sums per distinct
// bucket that would merge them, with some 6 distinct buckets among 64 tables.)
__device__ __forceinline__ void count_table(const PlanArgs& A, PlanLds& T, int bucket,
                                            unsigned long long cells, int32_t lds) {
  const int h = ht_slot(T, bucket, true);
  if (h >= 0) {
    atomicAdd(&T.cnt[h], 1u);
    atomicAdd(&T.cells[h], cells);
    atomicMax(&T.lds[h], lds);
  } else {
    atomicAdd(&A.counts[bucket], 1ull);
    atomicAdd(&A.cells[bucket], cells);
    if (lds > 0) atomicMax(&A.maxlds[bucket], lds);
  }
}

// Scatter pass, first sweep: tables per bucket into the table.
__device__ __forceinline__ void tally_table(PlanLds& T, int bucket) {
  const int h = ht_slot(T, bucket, true);
  if (h >= 0) atomicAdd(&T.cnt[h], 1u);
}

// Scatter pass, second sweep: this lane's slot, from the workgroup's range
// of the bucket (or, for a bucket not in the table, a global reservation).
__device__ __forceinline__ unsigned long long reserve_table(const PlanArgs& A, PlanLds& T,
                                                            int bucket) {
  const int h = ht_slot(T, bucket, false);
  return h >= 0 ? T.cells[h] + atomicAdd(&T.cnt[h], 1u) : atomicAdd(&A.cursor[bucket], 1ull);
}

// The start-up values of table (i0, j0) of a pair.
__device__ __forceinline__ TaskDesc make_desc(const PlanArgs& A, const PairMeta& pm,
                                              const TreeMeta& tx, const TreeMeta& ty, int32_t i0,
                                              int32_t j0) {
  const int32_t a = A.pool.orl[tx.node_off + i0] - i0 + 1;
  const int32_t b = A.pool.orl[ty.node_off + j0] - j0 + 1;
  const bool rows_x = a <= b;
  TaskDesc d;
  d.tdo = rows_x ? pm.td_off : pm.tdt_off;
  d.tdt = rows_x ? pm.tdt_off : pm.td_off;
  d.offR = rows_x ? tx.node_off : ty.node_off;
  d.offC = rows_x ? ty.node_off : tx.node_off;
  d.ldo = rows_x ? ty.n : tx.n;
  d.ldt = rows_x ? tx.n : ty.n;
  d.r0 = rows_x ? i0 : j0;
  d.c0 = rows_x ? j0 : i0;
  d.rmax = d.r0 + (rows_x ? a : b);
  d.cmax = d.c0 + (rows_x ? b : a);
  d.base_rx = A.pool.kdep[d.offR + d.r0] | (rows_x ? (int32_t)0x80000000 : 0);
  d.lbase = A.pool.lrank[d.offC + d.c0];
  return d;
}

// What bounds the passes: the loads that classify a table. So the scatter pass
// keeps its tables' buckets in LDS between its two sweeps, and a plan of few
// tables goes in small chunks (plan_chunk_tables).
// Count and scatter pass, us, with wave-wide sums per distinct bucket, every
// sweep classifying, and 2048 tables a chunk whatever the plan, against now:
// RRT 100-node pair 31 + 48, now 7 + 8; deep 1000-node pair 68 + 105, 12 + 10;
// 4096 pairs of 100-1000 nodes 2764 + 3259, 1188 + 2539 (the scatter writes 72
// bytes a table).
template <bool kScatter>
__global__ __launch_bounds__(kPlanThreads) void plan_kernel(PlanArgs A) {
  __shared__ PlanLds T;
  __shared__ int32_t bucket_at[kScatter ? kPlanChunk : 1];
  const int p = find_pair(A.blk_start, A.npairs, blockIdx.x);
  const PairMeta pm = A.pairs[p];
  const TreeMeta tx = A.pool.trees[pm.tx], ty = A.pool.trees[pm.ty];
  const PlanChunk ch = plan_chunk(A, tx, ty, p);
  const int32_t loff = A.level_off ? A.level_off[p] : 0;
  const bool leaf_form = A.pair_leaf ? A.pair_leaf[p] != 0 : A.lane_enable != 0;
  ht_clear(T);
  __syncthreads();
  // Table idx of the chunk is (l, k) = (idx / Kx, idx % Kx); a chunk holds
  // at most max(lchunk_tables, Kx) < 2^15 tables. One division per thread,
  // then each step of kPlanThreads tables adds (dl, dk) with one carry.
  const bool kept = ch.total <= kPlanChunk;  // in bucket_at (a lane reads back what it wrote)
  auto sweep = [&](bool again, auto body) {
    const int32_t total = (int32_t)ch.total;
    const int32_t kx = max(ch.Kx, 1);
    const int32_t dl = kPlanThreads / kx, dk = kPlanThreads % kx;
    int32_t lq = (int32_t)threadIdx.x / kx, kr = (int32_t)threadIdx.x % kx;
    for (int32_t base = 0; base < total; base += kPlanThreads) {
      const bool active = base + (int32_t)threadIdx.x < total;
      int bucket = 0, lds = 0;
      uint32_t i0 = 0, j0 = 0;
      unsigned long long cells = 0;
      const int k = ch.kbase + kr, l = ch.lbase + ch.l_lo + lq;
      if (active && again && kept) {
        bucket = bucket_at[base + threadIdx.x];
        i0 = (uint32_t)A.pool.skr[tx.node_off + k];
        j0 = (uint32_t)A.pool.skr[ty.node_off + l];
      } else if (active) {
        classify(A, tx, ty, loff, leaf_form, k, l, &bucket, &lds, &i0, &j0, &cells);
        if (kScatter && kept) bucket_at[base + threadIdx.x] = bucket;
      }
      body(active, bucket, lds, i0, j0, cells);
      lq += dl;
      kr += dk;
      if (kr >= kx) {
        kr -= kx;
        ++lq;
      }
    }
  };
  if (!kScatter) {
    sweep(false, [&](bool active, int bucket, int lds, uint32_t, uint32_t, unsigned long long cells) {
      if (active) count_table(A, T, bucket, cells, lds);
    });
    __syncthreads();
    for (int h = threadIdx.x; h < kHT; h += kPlanThreads) {
      const int b = T.key[h];
      if (b < 0) continue;
      atomicAdd(&A.counts[b], (unsigned long long)T.cnt[h]);
      atomicAdd(&A.cells[b], T.cells[h]);
      if (T.lds[h] > 0) atomicMax(&A.maxlds[b], T.lds[h]);
    }
  } else {
    sweep(false, [&](bool active, int bucket, int, uint32_t, uint32_t, unsigned long long) {
      if (active) tally_table(T, bucket);
    });
    __syncthreads();
    // One range per bucket for the workgroup; cnt becomes its cursor.
    for (int h = threadIdx.x; h < kHT; h += kPlanThreads) {
      const int b = T.key[h];
      if (b < 0) continue;
      T.cells[h] = atomicAdd(&A.cursor[b], (unsigned long long)T.cnt[h]);
      T.cnt[h] = 0;
    }
    __syncthreads();
    sweep(true, [&](bool active, int bucket, int, uint32_t i0, uint32_t j0, unsigned long long) {
      if (active) {
        const unsigned long long pos = reserve_table(A, T, bucket);
        const TaskDesc d = make_desc(A, pm, tx, ty, (int32_t)i0, (int32_t)j0);
        A.descs[pos] = d;
        A.tasks[pos] = task_pack((uint32_t)ch.p, i0, j0, d.base_rx < 0);
      }
    });
  }
}

// Exclusive scan of the bucket counts into the scatter cursors (one block):
// 4096 buckets a round, 4 a thread in one 32-byte read, so that the reads are
// whole lines in flight together. (A contiguous run of buckets per thread, one
// dependent read after another, took 433 us for the 38,720 buckets of the
// 4096-pair batch and 37 us for a deep 1000-node pair's 21,120; now 85 and 14.)
__global__ __launch_bounds__(1024) void plan_scan_kernel(const unsigned long long* counts,
                                                          unsigned long long* cursor, int nb) {
  __shared__ unsigned long long part[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  unsigned long long before = 0;  // the counts of earlier rounds
  for (int b0 = 0, r = 0; b0 < nb; b0 += 4096, r ^= 1) {
    const int b = b0 + 4 * tid;
    unsigned long long c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = b + i < nb ? counts[b + i] : 0;
    const unsigned long long sum = c[0] + c[1] + c[2] + c[3];
    unsigned long long incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned long long v = __shfl_up(incl, d);
      if (lane >= d) incl += v;
    }
    if (lane == 63) part[r][wave] = incl;
    __syncthreads();  // (two parts: the round before may still be read)
    unsigned long long run = before + incl - sum;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      run += w < wave ? part[r][w] : 0;
      before += part[r][w];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (b + i < nb) cursor[b + i] = run;
      run += c[i];
    }
  }
}

// Clears the count / max / ticket arrays and the abort flag (a kernel rather
// than a memset so the plan can be captured into a graph).
__global__ void plan_clear_kernel(PlanArgs a, int nb) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nb) {
    a.counts[i] = 0;
    a.cells[i] = 0;
    a.maxlds[i] = 0;
    a.tickets[i] = 0;
  }
  if (a.level_cells && i < a.nlevels) a.level_cells[i] = 0;
  if (i < kAbortInts) a.abort_flag[i] = 0;
  if (i == 0) {
    // Every column-blocked launch of the group tags its words with the base
    // and its ordinal: past those of the last plan (whose end the second word
    // holds), never 0 nor 0xFFFFFFFF.
    const uint32_t next = a.xl_base[1];
    const uint32_t base = next == 0 || next > 0xF0000000u ? 1 : next;
    a.xl_base[0] = base;
    a.xl_base[1] = base + (uint32_t)a.nlevels * kNumXLForms;
  }
}

// Interior cells of every level over all pairs, leaf keyroots' tables not
// counted: a pair's level L holds the tables of x's keyroots of height h
// against y's of height L - h, whose cells are the product of their summed
// sizes (one workgroup per pair, one level per thread).
__global__ __launch_bounds__(256) void level_cells_kernel(PlanArgs A) {
  const int p = blockIdx.x;
  const PairMeta pm = A.pairs[p];
  const TreeMeta tx = A.pool.trees[pm.tx], ty = A.pool.trees[pm.ty];
  const int32_t loff = A.level_off ? A.level_off[p] : 0;
  auto sum = [&](const TreeMeta& t, int h) {
    const int32_t* pre = A.pool.spre + t.node_off + t.K1;
    const int32_t* off = A.pool.kdoff + t.node_off;
    return (unsigned long long)(pre[off[h + 1]] - pre[off[h]]);
  };
  for (int L = threadIdx.x; L <= tx.kdmax + ty.kdmax; L += 256) {
    unsigned long long cells = 0;
    for (int h = max(0, L - ty.kdmax); h <= min(L, tx.kdmax); ++h)
      cells += sum(tx, h) * sum(ty, L - h);
    if (cells) atomicAdd(&A.level_cells[L + loff], cells);
  }
}

void launch_plan(const PlanArgs& a, int64_t nblocks, hipStream_t s) {
  const int nb = a.nlevels * kNumClasses * kBands;
  hipLaunchKernelGGL(plan_clear_kernel, dim3((nb + 255) / 256), dim3(256), 0, s, a, nb);
  if (a.level_cells)
    hipLaunchKernelGGL(level_cells_kernel, dim3((unsigned)a.npairs), dim3(256), 0, s, a);
  if (nblocks > 0)
    hipLaunchKernelGGL(plan_kernel<false>, dim3((unsigned)nblocks), dim3(kPlanThreads), 0, s, a);
  hipLaunchKernelGGL(plan_scan_kernel, dim3(1), dim3(1024), 0, s, a.counts, a.cursor, nb);
  if (nblocks > 0)
    hipLaunchKernelGGL(plan_kernel<true>, dim3((unsigned)nblocks), dim3(kPlanThreads), 0, s, a);
}

// Distances TD[0][0] of every pair into dist[], or kDistAborted everywhere
// when a wait of the group's kernels gave up.
__global__ void gather_dist_kernel(const PairMeta* pairs, const td_t* td, int32_t npairs,
                                   const int32_t* abort_flag, int32_t* dist) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < npairs) dist[i] = abort_flag[0] ? kDistAborted : td[pairs[i].td_off];
}

void launch_gather_dist(const PairMeta* pairs, const td_t* td, int32_t npairs,
                        const int32_t* abort_flag, int32_t* dist, hipStream_t s) {
  if (npairs <= 0) return;
  hipLaunchKernelGGL(gather_dist_kernel, dim3((npairs + 255) / 256), dim3(256), 0, s, pairs, td,
                     npairs, abort_flag, dist);
}

}  // namespace xted
