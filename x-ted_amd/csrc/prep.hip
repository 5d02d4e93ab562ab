// Device-side tree preprocessing: outermost-right leaves (orl), keyroots,
// keyroot nesting heights (the level scheduler's depths), per-node path
// keyroot depth, leaf ranks and the descending keyroot list.
//
// Replaces the host loops of X-TED_GPU/TED.cu:21-75 (outermost_right_leaves,
// key_roots) and X-TED_GPU/parallel_X_TED.cu:184-212 (O(K^2) keyroot depth).
// One workgroup per tree; every phase is a data-parallel pass separated by
// workgroup barriers, with pointer jumping for the ancestor-chain quantities.
//
// What bounds it: some 60 dependent passes, each of them one memory round trip
// and a barrier. So the working arrays live in LDS (trees of up to
// kPrepLdsNodes nodes; wider ones work in scratch memory), and no pass is left
// to one thread. In device memory, with the keyroots sorted by one thread, a
// pair of wide 1000-node trees took 779 us and of RRT 100-node trees 93; now 30
// and 19 (of RRT 20,000-node trees, in scratch memory, 712).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"

namespace xted {

constexpr int kPrepThreads = 1024;
constexpr int kSizeBands = 5;

// A working array's entry, read past this compute unit's L1 where the array
// is in device memory (its atomics are performed beyond it).
template <bool kLds>
__device__ __forceinline__ int32_t wld(const int32_t* p) {
  if constexpr (kLds) return *p;
  else return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroup-wide exclusive prefix sum: out(i, sum of in(0..i-1), in(i)) for
// i < n, each thread taking a contiguous chunk; returns the total. in is read
// twice, and out(i) comes after the thread's own second in(i).
template <class In, class Out>
__device__ __forceinline__ int32_t block_scan(int32_t n, int32_t* part, const In& in,
                                              const Out& out) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = blockDim.x >> 6;
  const int per = (n + (int)blockDim.x - 1) / (int)blockDim.x;
  const int lo = min(n, tid * per), hi = min(n, lo + per);
  int32_t s = 0;
  for (int i = lo; i < hi; ++i) s += in(i);
  int32_t incl = s;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  __syncthreads();  // part is free (and in's arrays are written)
  if (lane == 63) part[wave] = incl;
  __syncthreads();
  int32_t run = incl - s, total = 0;
  for (int w = 0; w < nwaves; ++w) {
    run += w < wave ? part[w] : 0;
    total += part[w];
  }
  for (int i = lo; i < hi; ++i) {
    const int32_t v = in(i);
    out(i, run, v);
    run += v;
  }
  __syncthreads();
  return total;
}

// m: kPrepArrays * (n + 1) working entries, part: 16 in LDS.
template <bool kLds>
__device__ __forceinline__ void prep_tree(const PrepArgs& A, int t, int32_t n, int64_t off,
                                          int32_t* m, int32_t* part) {
  const int32_t* parent = A.parent + off;
  const int32_t* label = A.label + off;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int n1 = n + 1;
  int32_t* const orl = m;           // last-child chains -> outermost right leaf
  int32_t* const kd = m + n1;       // nesting height of keyroots
  int32_t* const lrank = m + 2 * n1;
  int32_t* const list = m + 3 * n1; // block maxima, then keyroots in descending preorder
  int32_t* const anc = m + 4 * n1;  // keyroot flag | ancestor + 1 | keyroots on the way to it
  int32_t* const top = m + 5 * n1;  // path tops, then kdep
  int32_t* const hist = anc;        // 3 * (n + 1) entries, once anc and top are done with
  auto jump = [&](int32_t* p) {     // p[i] = end of the chain i, p[i], p[p[i]], ...
    for (;;) {
      int any = 0;
      for (int i = tid; i < n; i += nt) {
        const int32_t a = wld<kLds>(p + i), b = wld<kLds>(p + a);
        if (a != b) {
          p[i] = b;
          any = 1;
        }
      }
      if (!__syncthreads_or(any)) break;
    }
  };

  // ---- orl: follow last children to the outermost right leaf ---------------
  // In preorder the last child of v is its largest child id.
  for (int i = tid; i < n; i += nt) orl[i] = i;
  __syncthreads();
  for (int i = tid + 1; i < n; i += nt) atomicMax(&orl[parent[i]], i);
  __syncthreads();
  jump(orl);

  // ---- keyroot flags: the root and every node that is not a last child ----
  // anc packs, per node: bit 31 the flag, bits 16..30 an ancestor's id + 1 (0:
  // past the root), bits 0..15 the keyroots among the ancestors up to it.
  for (int i = tid; i < n; i += nt) {
    const int32_t p = i ? parent[i] : -1;
    const bool key = i == 0 || orl[p] != orl[i];
    A.orl[off + i] = orl[i];
    top[i] = key ? i : p;
    anc[i] = (key ? (int32_t)0x80000000 : 0) | ((p + 1) << 16);
  }
  __syncthreads();
  for (int i = tid + 1; i < n; i += nt) {
    const int32_t v = anc[i];
    anc[i] = v | (anc[((v >> 16) & 0x7FFF) - 1] < 0 ? 1 : 0);
  }
  __syncthreads();

  // ---- kanc(v): keyroots among the proper ancestors of v ---------------------
  // Pointer jumping; a packed entry is right whenever it is read.
  for (;;) {
    int any = 0;
    for (int i = tid; i < n; i += nt) {
      const int32_t v = wld<kLds>(anc + i), a = ((v >> 16) & 0x7FFF) - 1;
      if (a >= 0) {
        const int32_t w = wld<kLds>(anc + a);
        anc[i] = (v & (int32_t)0x80000000) | (w & 0x7FFF0000) | ((v & 0xFFFF) + (w & 0xFFFF));
        any = 1;
      }
    }
    if (!__syncthreads_or(any)) break;
  }
  auto kanc = [&](int i) { return anc[i] & 0xFFFF; };

  // ---- path top of v (keyroot owning v's right path) and kdep ---------------
  jump(top);
  for (int i = tid; i < n; i += nt) {
    const int32_t r = top[i], d = kanc(r);
    A.rtop[off + i] = r;
    A.kdep[off + i] = d;
    top[i] = d;
  }
  int32_t* const kdep = top;

  // ---- keyroot nesting height ------------------------------------------------
  // kd(t) = max over keyroots u in (t, orl(t)] of kanc(u) - kanc(t), 0 if none.
  // Maxima of kanc over keyroots, of 16 and of 256 nodes, shorten the scans.
  const int nb1 = (n + 15) / 16, nb2 = (nb1 + 15) / 16;
  int32_t *const max1 = list, *const max2 = list + nb1;
  auto most = [&](int32_t v, int32_t i) { return anc[i] < 0 ? max(v, kanc(i)) : v; };
  for (int b = tid; b < nb1; b += nt) {
    int32_t v = -1;
    for (int i = b * 16; i < min(n, b * 16 + 16); ++i) v = most(v, i);
    max1[b] = v;
  }
  __syncthreads();
  for (int b = tid; b < nb2; b += nt) {
    int32_t v = -1;
    for (int i = b * 16; i < min(nb1, b * 16 + 16); ++i) v = max(v, max1[i]);
    max2[b] = v;
  }
  __syncthreads();
  for (int i = tid; i < n; i += nt) {
    int32_t d = -1;
    if (anc[i] < 0) {
      const int32_t hi = orl[i];  // the range is i+1 .. hi
      int32_t v = -1, j = i + 1;
      for (; j <= hi && (j & 15); ++j) v = most(v, j);
      for (; j + 15 <= hi && (j & 255); j += 16) v = max(v, max1[j >> 4]);
      for (; j + 255 <= hi; j += 256) v = max(v, max2[j >> 8]);
      for (; j + 15 <= hi; j += 16) v = max(v, max1[j >> 4]);
      for (; j <= hi; ++j) v = most(v, j);
      d = v < 0 ? 0 : v - kanc(i);
    }
    kd[i] = d;
    A.kdn[off + i] = d;
  }
  __syncthreads();

  // ---- keyroot list, descending preorder -------------------------------------
  int32_t* const before = lrank;  // keyroots before a node
  const int32_t K =
      block_scan(n, part, [&](int i) { return anc[i] < 0 ? 1 : 0; },
                 [&](int i, int32_t run, int32_t) { before[i] = run; });
  for (int i = tid; i < n; i += nt) {
    if (anc[i] < 0) {
      const int32_t k = K - 1 - before[i];
      list[k] = i;
      A.kr[off + k] = i;
      A.krkd[off + k] = kd[i];
      A.krsize[off + k] = orl[i] - i + 1;
    }
  }
  __syncthreads();

  // ---- leaf ranks ----------------------------------------------------------
  const int32_t nleaves =
      block_scan(n, part, [&](int i) { return orl[i] == i ? 1 : 0; },
                 [&](int i, int32_t run, int32_t) {
                   lrank[i] = run;
                   A.lrank[off + i] = run;
                 });
  if (tid == 0) {
    lrank[n] = nleaves;
    A.lrank[off + n] = nleaves;
  }
  __syncthreads();
  auto leaves = [&](int i) { return lrank[orl[i] + 1] - lrank[i]; };
  for (int k = tid; k < K; k += nt) A.krleaf[off + k] = leaves(list[k]);

  // ---- per-node records of the forest kernels ------------------------------
  for (int i = tid; i < n; i += nt) {
    const int32_t prev_leaf = i > 0 && orl[i - 1] == i - 1 ? (int32_t)0x80000000 : 0;
    const int32_t o = orl[i], lab = label[i];
    A.crec[off + i] = NodeRec{o, lab, lrank[o], (i > 0 ? lrank[i - 1] : 0) | prev_leaf};
    A.rrec[off + i] = NodeRec{o, lab, kdep[i], (i > 0 ? kdep[i - 1] : 0) | prev_leaf};
  }
  __syncthreads();

  // ---- keyroots sorted for the scheduler -----------------------------------
  // Leaf keyroots first, then the other keyroots by ascending nesting height
  // and, within a height, by subtree size band (<= 16, 64, 256, 1024, more
  // nodes): a stable counting sort over the descending list. The plan gives
  // a wave consecutive keyroots of this order, so its tables fall into few
  // (level, class) buckets. Keys are counted by all threads, and places given
  // out by one wave, 64 keyroots of the list at a time.
  const int32_t kdmax = kd[0], nkeys = (kdmax + 1) * kSizeBands;  // <= 3 * (n + 1)
  auto key = [&](int i) {
    const int32_t sz = orl[i] - i + 1;
    return kd[i] * kSizeBands + (sz > 16) + (sz > 64) + (sz > 256) + (sz > 1024);
  };
  auto place = [&](int32_t pos, int i) {
    A.skr[off + pos] = i;
    A.skd[off + pos] = kd[i];
    A.ssize[off + pos] = orl[i] - i + 1;
    A.sleaf[off + pos] = leaves(i);
  };
  for (int d = tid; d < nkeys; d += nt) hist[d] = 0;
  __syncthreads();
  for (int k = tid; k < K; k += nt) {
    const int i = list[k];
    if (orl[i] != i) atomicAdd(&hist[key(i)], 1);
  }
  const int32_t K1 =
      block_scan(K, part, [&](int k) { return orl[list[k]] == list[k] ? 1 : 0; },
                 [&](int k, int32_t run, int32_t leaf) {
                   if (leaf) place(run, list[k]);
                 });
  block_scan(nkeys, part, [&](int d) { return wld<kLds>(hist + d); },
             [&](int d, int32_t run, int32_t) {
               hist[d] = run;
               if (d % kSizeBands == 0) A.kdoff[off + d / kSizeBands] = run;
             });
  if (tid == 0) A.kdoff[off + kdmax + 1] = K - K1;
  if (tid < 64) {
    for (int k0 = 0; k0 < K; k0 += 64) {
      const int i = list[min(k0 + tid, K - 1)];
      const bool mine = k0 + tid < K && orl[i] != i;
      const int32_t ky = mine ? key(i) : -1;
      // Lanes of one key: their number, this lane's rank among them, the first.
      int32_t count = 0, rank = 0, first = 0;
      for (unsigned long long todo = __ballot(mine); todo;) {
        const int lead = __ffsll((long long)todo) - 1;
        const unsigned long long same = __ballot(ky == __shfl(ky, lead));
        if ((same >> tid) & 1) {
          count = __popcll(same);
          rank = __popcll(same & ((1ull << tid) - 1));
          first = lead;
        }
        todo &= ~same;
      }
      int32_t base = 0;
      if (mine && rank == 0) base = atomicAdd(&hist[ky], count);
      base = __shfl(base, first);
      if (mine) place(K1 + base + rank, i);
    }
  }
  __syncthreads();
  const int32_t sum =
      block_scan(K, part, [&](int k) { return A.ssize[off + k]; },
                 [&](int k, int32_t run, int32_t) { A.spre[off + k] = run; });
  if (tid == 0) {
    A.spre[off + K] = sum;
    A.trees[t].K = K;
    A.trees[t].kdmax = kdmax;
    A.trees[t].nleaves = nleaves;
    A.trees[t].K1 = K1;
  }
}

__global__ __launch_bounds__(kPrepThreads) void tree_prep_kernel(PrepArgs A) {
  extern __shared__ int32_t work[];
  __shared__ int32_t part[kPrepThreads / 64];
  const int t = A.first_tree + blockIdx.x;
  const int32_t n = A.trees[t].n;
  const int64_t off = A.trees[t].node_off;
  if (n <= kPrepLdsNodes) prep_tree<true>(A, t, n, off, work, part);
  else prep_tree<false>(A, t, n, off, A.scratch + A.scratch_off[blockIdx.x], part);
}

__global__ __launch_bounds__(kPrepThreads) void cost_prefix_kernel(CostPrefixArgs A) {
  __shared__ int32_t lds_tmp[kPrepThreads];
  const TreeMeta meta = A.trees[A.first_tree + blockIdx.x];
  const int32_t n = meta.n;
  const int32_t* lab = A.label + meta.node_off;
  // A pool tree added before the cost model may hold labels outside its
  // alphabet; such a tree's sums are meaningless (pairs using it are
  // rejected on the host) but its reads stay inside the cost arrays.
  const uint32_t amax = (uint32_t)A.alphabet - 1;
  for (int pass = 0; pass < 2; ++pass) {
    const int32_t* cost = pass ? A.ins : A.del;
    int32_t* out = (pass ? A.pins : A.pdel) + meta.node_off;
    // Each thread owns a contiguous chunk of nodes; a scan of the chunk sums.
    const int per = (n + kPrepThreads - 1) / kPrepThreads;
    const int lo = min(n, (int)threadIdx.x * per), hi = min(n, lo + per);
    int32_t s = 0;
    for (int i = lo; i < hi; ++i) s += cost[min((uint32_t)lab[i], amax)];
    lds_tmp[threadIdx.x] = s;
    __syncthreads();
    for (int off = 1; off < kPrepThreads; off <<= 1) {
      const int32_t v = (int)threadIdx.x >= off ? lds_tmp[threadIdx.x - off] : 0;
      __syncthreads();
      lds_tmp[threadIdx.x] += v;
      __syncthreads();
    }
    int32_t run = threadIdx.x ? lds_tmp[threadIdx.x - 1] : 0;
    for (int i = lo; i < hi; ++i) {
      out[i] = run;
      run += cost[min((uint32_t)lab[i], amax)];
    }
    if (threadIdx.x == kPrepThreads - 1) {
      out[n] = lds_tmp[kPrepThreads - 1];
      A.totals[2 * blockIdx.x + pass] = lds_tmp[kPrepThreads - 1];
    }
    __syncthreads();
  }
  const int32_t* orl = A.orl + meta.node_off;
  const int32_t* pd = A.pdel + meta.node_off;
  const int32_t* pi = A.pins + meta.node_off;
  for (int i = threadIdx.x; i < n; i += kPrepThreads) {
    const int32_t e = orl[i] + 1;
    A.rec[meta.node_off + i] = CostRec{pd[i], pi[i], pd[e], pi[e]};
  }
}

void launch_cost_prefix(const CostPrefixArgs& a, int ntrees, hipStream_t s) {
  if (ntrees <= 0) return;
  hipLaunchKernelGGL(cost_prefix_kernel, dim3(ntrees), dim3(kPrepThreads), 0, s, a);
}

void launch_tree_prep(const PrepArgs& a, int ntrees, int maxn, hipStream_t s) {
  if (ntrees <= 0) return;
  // Fewer waves for small trees, whose passes are all barrier.
  const int threads = maxn <= 256 ? 256 : kPrepThreads;
  const size_t lds = sizeof(int32_t) * kPrepArrays * (std::min(maxn, kPrepLdsNodes) + 1);
  hipLaunchKernelGGL(tree_prep_kernel, dim3(ntrees), dim3(threads), lds, s, a);
}

hipError_t prep_init_attributes() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&tree_prep_kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             sizeof(int32_t) * kPrepArrays * (kPrepLdsNodes + 1));
}

}  // namespace xted
