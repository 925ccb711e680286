// Level-synchronous reverse Cuthill-McKee on the device, bit-exact to the sequential
// 3DRCM order (InchingLiteInteger/Fuel/Coordinate/T1.py:171-323).
//
// The sequential algorithm appends, for each dequeued node in queue order, its unvisited
// neighbours (scanned in descending index order) and sorts those new children stably by
// degree; when the queue runs dry, the first unvisited node in the caller's seed order
// starts the next connected component. Queue order is level order, so level L+1 consists of
// the unvisited neighbours of level L, each one the child of the first level-L node (lowest
// queue position) adjacent to it, and inside one parent's group the children are ordered by
// (degree ascending, index descending). One level is built per round:
//   claim   : claim[j] = min position of a level-L neighbour           (atomicMin)
//   count   : cnt[p]   = number of nodes claimed by the node at position p
//   scan    : off      = exclusive prefix sum of cnt
//   scatter : the children's keys (degree, -index) written into their parent's slot range
//   place   : each child at its key's rank in its group
// The level's bounds stay on the device: the kernels of kRounds levels are launched at a time,
// each over a fixed grid that reads the bounds, and the host looks at them once per batch (a
// level past the last one finds no nodes and does nothing).
// Components do not interact, so all of them advance in the same rounds: the components
// are found first (union-find), each one's seed is its first node in the seed order, and
// the components, ordered by their seeds' places in the seed order, are the order in which
// the sequential algorithm visits them. A round's frontier holds the components' levels one
// after another in that order, so inside each component positions compare as in the
// sequential run; every node's final position is its component's start plus its rank in
// the component (levels before its own, then its place in its own level). The number of
// rounds is the deepest component's level count, not the sum over components.
#include <hip/hip_runtime.h>

#include <climits>
#include <vector>

#include "common.h"
#include "scan.h"

#define HIP_TRY(expr)                                                                      \
  do {                                                                                     \
    hipError_t _e = (expr);                                                                \
    if (_e != hipSuccess) INCH_FAIL(INCH_ERR_HIP, "%s: %s", #expr, hipGetErrorString(_e)); \
  } while (0)

namespace {

constexpr int kG = 32;  // lanes per level node in the neighbour scans

__global__ void k_rcm_init(int64_t n, int32_t *__restrict__ claim) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) claim[i] = INT_MAX;
}

__global__ void k_rcm_zero(int32_t L, int32_t *__restrict__ a) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < L) a[i] = 0;
}

// The state of the level loop on the device, a ring of one per round: the level holds the positions
// [s, e), its children will be [e, e + next).
struct Level {
  int32_t s, e, next, bad;
};

// claim[j]: the position of j's parent (the first of its neighbours), -1 for a seed, INT_MAX while not reached. A
// node of an earlier or of this level holds a smaller position than the level's own, so it is never claimed again
// and never counted, without a look at its own position (a level of about 5,000 nodes takes 33 us in 5 launches; 37
// in 7 with that second gather per edge and with the sort and the advance in kernels of their own).
// Claims of the level's nodes, and the nodes' final positions (their component's start plus its
// nodes of earlier levels plus the place in this level's segment).
__global__ void __launch_bounds__(256) k_rcm_claim(const Level *__restrict__ lv, const int32_t *__restrict__ ord,
                                                   const int64_t *__restrict__ indptr,
                                                   const int32_t *__restrict__ indices, int32_t *__restrict__ claim,
                                                   const int32_t *__restrict__ cv, const int32_t *__restrict__ cstart,
                                                   const int32_t *__restrict__ done,
                                                   const int32_t *__restrict__ first, int32_t *__restrict__ fin) {
  const int32_t e = lv->e;
  const int lane = (int)(threadIdx.x % kG);
  for (int64_t p = lv->s + (blockIdx.x * 256 + (int)threadIdx.x) / kG; p < e; p += gridDim.x * (256 / kG)) {
    const int32_t i = ord[p];
    if (lane == 0) {
      const int32_t c = cv[i];
      fin[p] = cstart[c] + done[c] + ((int32_t)p - first[c]);
    }
    for (int64_t b = indptr[i] + lane; b < indptr[i + 1]; b += kG) {
      const int32_t j = indices[b];
      // a cached load drops earlier levels' nodes; one past the L1 sees other groups' claims: most nodes are
      // claimed by the first few positions, and the rest need no atomic
      if (claim[j] > (int32_t)p &&
          __hip_atomic_load(&claim[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > (int32_t)p)
        atomicMin(&claim[j], (int32_t)p);
    }
  }
}

__global__ void __launch_bounds__(256) k_rcm_count(const Level *__restrict__ lv, const int32_t *__restrict__ ord,
                                                   const int64_t *__restrict__ indptr,
                                                   const int32_t *__restrict__ indices,
                                                   const int32_t *__restrict__ claim, int32_t *__restrict__ cnt) {
  const int32_t s = lv->s, e = lv->e;
  const int lane = (int)(threadIdx.x % kG);
  for (int64_t p = s + (blockIdx.x * 256 + (int)threadIdx.x) / kG; p < e; p += gridDim.x * (256 / kG)) {
    const int32_t i = ord[p];
    int32_t c = 0;
    for (int64_t b = indptr[i] + lane; b < indptr[i + 1]; b += kG) {
      const int32_t j = indices[b];
      if (claim[j] == (int32_t)p) ++c;
    }
#pragma unroll
    for (int o = kG / 2; o > 0; o >>= 1) c += __shfl_xor(c, o, kG);
    if (lane == 0) cnt[p - s] = c;
  }
}

// off[q] = nodes claimed by the level's first q nodes; lv->next = all of them, and `after` the next round's level.
// One workgroup.
__global__ void __launch_bounds__(1024) k_rcm_scan(Level *__restrict__ lv, Level *__restrict__ after, int64_t n,
                                                   const int32_t *__restrict__ cnt, int32_t *__restrict__ off) {
  __shared__ int32_t sums[16];
  const int32_t L = lv->e - lv->s;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int32_t carry = 0;
  for (int32_t b = 0; b < L; b += 8192) {
    int32_t v[8], t = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int32_t i = b + 8 * tid + q;
      v[q] = i < L ? cnt[i] : 0;
      t += v[q];
    }
    int32_t inc = t;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t x = __shfl_up(inc, o, 64);
      if (lane >= o) inc += x;
    }
    __syncthreads();
    if (lane == 63) sums[w] = inc;
    __syncthreads();
    int32_t before = carry;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int32_t x = sums[q];
      if (q < w) before += x;
      carry += x;
    }
    before += inc - t;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int32_t i = b + 8 * tid + q;
      if (i < L) off[i] = before;
      before += v[q];
    }
  }
  if (tid == 0) {
    off[L] = carry;
    // more children than nodes: an inconsistent graph (an edge without its reverse); none are taken
    int32_t bad = lv->bad;
    if ((int64_t)lv->e + carry > n) {
      bad = 1;
      carry = 0;
    }
    lv->next = carry;
    *after = Level{lv->e, lv->e + carry, 0, bad};
  }
}

// The children of the level's nodes, grouped by parent, as keys of the order inside a group: ascending degree,
// then descending index.
__global__ void __launch_bounds__(256) k_rcm_scatter(const Level *__restrict__ lv, const int32_t *__restrict__ ord,
                                                     const int64_t *__restrict__ indptr,
                                                     const int32_t *__restrict__ indices,
                                                     const int32_t *__restrict__ claim,
                                                     const int32_t *__restrict__ off, uint64_t *__restrict__ key) {
  const int32_t s = lv->s, e = lv->e;
  if (lv->next == 0) return;
  const int lane = (int)(threadIdx.x % kG);
  const int sh = (int)(threadIdx.x & 63) & ~(kG - 1);      // the group's first lane in its wave
  for (int64_t p0 = s + (blockIdx.x * 256 + (int)threadIdx.x) / kG; p0 - (int)(threadIdx.x / kG) < e;
       p0 += gridDim.x * (256 / kG)) {
    const bool on = p0 < e;
    const int64_t p = on ? p0 : s;
    const int32_t i = ord[p];
    const int64_t b1 = indptr[i + 1];
    uint64_t *out = key + off[p - s];
    // lanes past their own row stay in the loop for the group's ballots
    for (int64_t b = indptr[i]; b < b1; b += kG) {
      bool mine = false;
      int32_t j = 0;
      if (on && b + lane < b1) {
        j = indices[b + lane];
        mine = claim[j] == (int32_t)p;
      }
      const uint32_t m = (uint32_t)((__ballot(mine) >> sh) & ((1ull << kG) - 1));
      if (mine)
        out[__popc(m & ((1u << lane) - 1))] =
            ((uint64_t)(indptr[j + 1] - indptr[j]) << 32) | (uint64_t)(0xffffffffu - (uint32_t)j);
      out += __popc(m);
    }
  }
}

// The new level [e, e + next): a thread per child ranks its key among its parent's children (neighbouring threads
// read the same keys; a kernel of its own for this took 4 us per level and a launch), and its components' segments:
// a level's nodes of component c are consecutive (the frontier is grouped by component, in component order, so
// their children are too), and the segment's bounds come from comparing neighbours: one writer
// each, no atomics. The first node's thread also closes c's previous segment, whose end the
// other half of lend holds.
__global__ void __launch_bounds__(256) k_rcm_place(const Level *__restrict__ lv, int32_t *__restrict__ ord,
                                                   const int32_t *__restrict__ claim, const int32_t *__restrict__ off,
                                                   const uint64_t *__restrict__ key, const int32_t *__restrict__ cv,
                                                   int32_t *__restrict__ first, const int32_t *__restrict__ lend_old,
                                                   int32_t *__restrict__ lend, int32_t *__restrict__ done) {
  const int32_t s = lv->s, e = lv->e, L1 = lv->next;
  auto node = [](uint64_t k) { return (int32_t)(0xffffffffu - (uint32_t)k); };
  for (int32_t t = blockIdx.x * 256 + threadIdx.x; t < L1; t += gridDim.x * 256) {
    const uint64_t k = key[t];
    const int32_t v = node(k), c = cv[v], p = claim[v] - s;
    const int32_t g0 = off[p], g1 = off[p + 1];
    int32_t r = g0;
#pragma unroll 8
    for (int32_t b = g0; b < g1; ++b) r += key[b] < k || (key[b] == k && b < t);
    ord[e + r] = v;
    // which of a group's children stands at t does not matter here: they share the component
    const int32_t q = e + t;
    if (t == 0 || cv[node(key[t - 1])] != c) {
      done[c] += lend_old[c] - first[c];
      first[c] = q;
    }
    if (t == L1 - 1 || cv[node(key[t + 1])] != c) lend[c] = q + 1;   // one past the segment's end
  }
}

// ---- components: union-find over the edges. A root is only ever hooked (CAS) onto a
// smaller root, so parent[v] <= v throughout and each component ends with its smallest node
// as root; finds shorten the paths they walk (the ECL-CC scheme, Jaiganesh and Burtscher,
// 2018). The finds' loads may see a stale parent: any value ever stored is an ancestor in
// the same component, and a hook only succeeds on a node that is a root at the CAS (which
// returns the current parent otherwise), so they are relaxed atomics of workgroup scope
// (cacheable); the final flattening runs after the hooking kernel has completed. ----
__device__ __forceinline__ int32_t cc_load(const int32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void cc_store(int32_t *p, int32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ int32_t cc_find(int32_t *parent, int32_t v) {
  int32_t par = cc_load(parent + v);
  if (par != v) {
    int32_t prev = v, next;
    while (par > (next = cc_load(parent + par))) {
      cc_store(parent + prev, next);
      prev = par;
      par = next;
    }
  }
  return par;
}

// Lanes per node of the two edge passes: a node's row is read by kCcLanes consecutive lanes
// (coalesced), not by one lane walking it alone.
constexpr int kCcLanes = 16;

// parent[v] = v's smallest neighbour when that is smaller than v (a valid hook: parent[v] <=
// v and in v's component), which leaves most trees shallow before any CAS
__global__ void k_cc_init(int64_t n, const int64_t *__restrict__ indptr, const int32_t *__restrict__ indices,
                          int32_t *__restrict__ parent) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t v = t / kCcLanes;
  const int lane = (int)(t % kCcLanes);
  if (v >= n) return;  // a node's lanes leave together
  int32_t m = (int32_t)v;
  for (int64_t b = indptr[v] + lane; b < indptr[v + 1]; b += kCcLanes) m = indices[b] < m ? indices[b] : m;
#pragma unroll
  for (int off = kCcLanes / 2; off > 0; off >>= 1) {
    const int32_t o = __shfl_xor(m, off, kCcLanes);
    m = o < m ? o : m;
  }
  if (lane == 0) parent[v] = m;
}

__device__ __forceinline__ void cc_link(int32_t *parent, int32_t vr, int32_t u) {
  int32_t ur = cc_find(parent, u);
  while (vr != ur) {
    const int32_t lo = vr < ur ? vr : ur, hi = vr < ur ? ur : vr;
    const int32_t r = atomicCAS(parent + hi, hi, lo);
    if (r == hi) return;
    vr = lo;
    ur = r;  // hi was hooked meanwhile: continue from its new parent
  }
}

// Two edges of every stride-th node whose ends have different parents. Joining a few nodes first
// and flattening leaves the later passes almost nothing to link: linking two edges of every node
// at once took 0.76 ms on 150,000 atoms, most of it walking trees that others were hooking.
__global__ void k_cc_link_some(int64_t n, int stride, const int64_t *__restrict__ indptr,
                               const int32_t *__restrict__ indices, int32_t *parent) {
  const int64_t v = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) * stride;
  if (v >= n) return;
  const int64_t b = indptr[v], len = indptr[v + 1] - b;
  if (len == 0) return;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int32_t u = indices[b + (k ? len - 1 : len / 2)];
    const int32_t pv = cc_load(parent + v);
    if (cc_load(parent + u) != pv) cc_link(parent, cc_find(parent, (int32_t)v), u);
  }
}

// Every edge from both ends: labels (flattened before) that differ are linked. Linking every edge
// from scratch took 2.5 ms on a 150,000-atom graph in random order, with its finds and hooks of
// 17 million edges; the two linking passes and the comparison take 0.1.
__global__ void k_cc_hook(int64_t n, const int64_t *__restrict__ indptr, const int32_t *__restrict__ indices,
                          const int32_t *__restrict__ label, int32_t *parent) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t v = t / kCcLanes;
  const int lane = (int)(t % kCcLanes);
  if (v >= n) return;
  const int32_t lv = label[v];
  for (int64_t b = indptr[v] + lane; b < indptr[v + 1]; b += kCcLanes) {
    const int32_t u = indices[b];
    if (label[u] != lv) cc_link(parent, cc_find(parent, (int32_t)v), u);
  }
}

// label[v] = root of v (in place over parent: writing a root only shortens paths)
__global__ void k_cc_flatten(int64_t n, int32_t *parent) {
  const int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (v >= n) return;
  int32_t r = (int32_t)v, p;
  while ((p = cc_load(parent + r)) != r) r = p;
  cc_store(parent + v, r);
}

// rank[seeds[k]] = k; minr[root] = smallest rank in the component (minr starts at INT_MAX)
__global__ void k_cc_rank(int64_t n, const int64_t *__restrict__ seeds, int32_t *__restrict__ rank,
                          int32_t *__restrict__ minr) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) {
    rank[seeds[k]] = (int32_t)k;
    minr[k] = INT_MAX;
  }
}

__global__ void k_cc_minrank(int64_t n, const int32_t *__restrict__ label, const int32_t *__restrict__ rank,
                             int32_t *__restrict__ minr) {
  // one atomic per run of a wave's lanes that share a component (one component: all 64), and
  // none where the minimum so far is lower: 150,000 nodes of one component took 1.7 ms one by one
  const int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const int32_t c = v < n ? label[v] : -1;
  int32_t r = v < n ? rank[v] : INT_MAX;
  // minimum over the lanes of the same run from this lane on (segmented)
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t oc = __shfl_down(c, o, 64), orr = __shfl_down(r, o, 64);
    if (lane + o < 64 && oc == c && orr < r) r = orr;
  }
  const int32_t cp = __shfl_up(c, 1, 64);
  if (c >= 0 && (lane == 0 || cp != c) && r < minr[c]) atomicMin(&minr[c], r);
}

// flag[k] = 1 when seeds[k] is the first node of its component in the seed order
__global__ void k_cc_flag(int64_t n, const int64_t *__restrict__ seeds, const int32_t *__restrict__ label,
                          const int32_t *__restrict__ minr, int32_t *__restrict__ flag) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) flag[k] = minr[label[seeds[k]]] == (int32_t)k ? 1 : 0;
}

// component c (in seed order) starts from S[c]; croot[root] = c; csize zeroed
__global__ void k_cc_seeds(int64_t n, const int64_t *__restrict__ seeds, const int32_t *__restrict__ label,
                           const int32_t *__restrict__ flag, const int32_t *__restrict__ cidx,
                           int32_t *__restrict__ S, int32_t *__restrict__ croot, int32_t *__restrict__ csize) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  csize[k] = 0;
  if (flag[k]) {
    const int32_t v = (int32_t)seeds[k];
    S[cidx[k]] = v;
    croot[label[v]] = cidx[k];
  }
}

// cv[v] = component of v; csize[c] += 1 per node, one atomic per run of a wave's lanes that
// share a component (nodes of a component tend to be consecutive: few counters, heavy
// contention otherwise)
__global__ void __launch_bounds__(256) k_cc_vertex(int64_t n, const int32_t *__restrict__ label,
                                                   const int32_t *__restrict__ croot, int32_t *__restrict__ cv,
                                                   int32_t *__restrict__ csize) {
  const int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const int32_t c = v < n ? croot[label[v]] : -1;
  if (v < n) cv[v] = c;
  const int32_t cp = __shfl_up(c, 1, 64);
  const bool head = c >= 0 && (lane == 0 || cp != c);
  // run length: lanes up to the next head (or the wave's end)
  const uint64_t heads = __ballot(head);
  if (head) {
    const uint64_t later = lane < 63 ? heads >> (lane + 1) : 0;
    int run = later ? __ffsll((unsigned long long)later) : 64 - lane;
    if (v + run > n) run = (int)(n - v);
    atomicAdd(&csize[c], run);
  }
}

// round 0: the seeds, one per component, each first in its component
__global__ void k_rcm_seed_level(int32_t C, const int32_t *__restrict__ S, int32_t *__restrict__ ord,
                                 int32_t *__restrict__ claim, int32_t *__restrict__ done, int32_t *__restrict__ first,
                                 int32_t *__restrict__ lend, Level *__restrict__ lv) {
  const int32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c == 0) *lv = Level{0, C, 0, 0};
  if (c >= C) return;
  ord[c] = S[c];
  claim[S[c]] = -1;
  done[c] = 0;
  first[c] = c;
  lend[c] = c + 1;
}

__global__ void k_rcm_finish(int64_t n, const int32_t *__restrict__ ord, const int32_t *__restrict__ fin,
                             int32_t reverse, int32_t *__restrict__ order, int64_t *__restrict__ undo) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int64_t p = reverse ? n - 1 - fin[q] : fin[q];
  const int32_t v = ord[q];
  order[p] = v;
  undo[v] = p;
}

// Input validation before any indexed access: seeds in [0, n), indptr non-decreasing from 0,
// columns in [0, n). Sets *bad to 1 on a violation.
__global__ void k_rcm_check(int64_t n, const int64_t *__restrict__ indptr, const int32_t *__restrict__ indices,
                            const int64_t *__restrict__ seeds, int32_t *__restrict__ bad) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < n) {
    const int64_t sd = seeds[t];
    if (sd < 0 || sd >= n) *bad = 1;
    if (indptr[t + 1] < indptr[t] || (t == 0 && indptr[0] != 0)) *bad = 1;
  }
}

__global__ void k_rcm_check_cols(int64_t nnz, int64_t n, const int32_t *__restrict__ indices,
                                 int32_t *__restrict__ bad) {
  for (int64_t b = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; b < nnz; b += (int64_t)gridDim.x * blockDim.x) {
    const int32_t j = indices[b];
    if (j < 0 || j >= n) *bad = 1;
  }
}

__global__ void k_rcm_flag_init(int32_t *bad) { *bad = 0; }

__global__ void k_rcm_seed_hist(int64_t n, const int64_t *__restrict__ seeds, int32_t *__restrict__ cnt) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < n) atomicAdd(&cnt[seeds[t]], 1);
}

__global__ void k_rcm_seed_perm(int64_t n, const int32_t *__restrict__ cnt, int32_t *__restrict__ bad) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < n && cnt[t] != 1) *bad = 1;
}

unsigned blocks_for(int64_t threads, int bs) { return (unsigned)((threads + bs - 1) / bs); }

}  // namespace

extern "C" {

constexpr int kRcmArrays = 20;  // int32 arrays of n + 2 entries in the work buffer
constexpr int kRcmHead = 256;   // bytes before them: the levels' states and a flag
constexpr int kRounds = 8;      // levels per look at their bounds

int64_t inch_rcm_device_work_size(int64_t n) {
  return (kRcmArrays * (n + 2) + 2 * (scan_tiles(n + 1) + 2)) * (int64_t)sizeof(int32_t) + kRcmHead;
}

inch_status inch_rcm_device(int64_t n, const int64_t *indptr, const int32_t *indices, const int64_t *seeds,
                            int32_t reverse, int32_t *order, int64_t *undo, void *work, int64_t work_bytes,
                            int64_t *comp_ptr, int64_t comp_cap, int64_t *n_comp, void *stream) {
  INCH_REQUIRE(!comp_ptr || comp_cap >= 2, "inch_rcm_device: comp_cap must be >= 2");
  INCH_REQUIRE(n > 0 && n < INT_MAX - 2 && indptr && indices && seeds && order && undo && work,
               "inch_rcm_device: bad args");
  INCH_REQUIRE(work_bytes >= inch_rcm_device_work_size(n), "inch_rcm_device: work too small (%lld < %lld)",
               (long long)work_bytes, (long long)inch_rcm_device_work_size(n));
  hipStream_t st = (hipStream_t)stream;
  int32_t *arr[kRcmArrays];
  for (int q = 0; q < kRcmArrays; ++q) arr[q] = (int32_t *)((char *)work + kRcmHead) + q * (n + 2);
  uint64_t *key = (uint64_t *)arr[0];   // two arrays
  int32_t *cnt = arr[2], *off = arr[3], *label2 = arr[4], *claim = label2, *ord = arr[5];   // claim once label2 is used
  int32_t *label = arr[6], *rank = arr[7], *minr = arr[8], *flag = arr[9], *cidx = arr[10], *croot = arr[11];
  int32_t *cv = arr[12], *csize = arr[13], *cstart = arr[14], *fin = arr[15], *first = arr[16], *lend = arr[17];
  int32_t *done = arr[18], *S = arr[19], *lend2 = flag;   // flag is free once the seeds are known
  Level *lv = (Level *)((char *)work + 16);   // kRounds of them
  int32_t *tsum = arr[kRcmArrays - 1] + (n + 2), *toff = tsum + scan_tiles(n + 1) + 2;
  const int bs = 256;
  int32_t *bad = (int32_t *)((char *)work + 8);
  k_rcm_flag_init<<<1, 1, 0, st>>>(bad);
  k_rcm_check<<<blocks_for(n, bs), bs, 0, st>>>(n, indptr, indices, seeds, bad);
  int64_t nnz = 0;
  HIP_TRY(hipMemcpyAsync(&nnz, indptr + n, sizeof(nnz), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  INCH_REQUIRE(nnz >= 0, "inch_rcm_device: indptr[n] < 0");
  if (nnz > 0) k_rcm_check_cols<<<blocks_for(nnz < 4096 * 256 ? nnz : 4096 * 256, bs), bs, 0, st>>>(nnz, n, indices, bad);
  int32_t bad_h = 0;
  HIP_TRY(hipMemcpyAsync(&bad_h, bad, sizeof(bad_h), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  INCH_REQUIRE(!bad_h, "inch_rcm_device: seeds, indptr or column indices out of range");
  k_rcm_zero<<<blocks_for(n, bs), bs, 0, st>>>((int32_t)n, cnt);
  k_rcm_seed_hist<<<blocks_for(n, bs), bs, 0, st>>>(n, seeds, cnt);
  k_rcm_seed_perm<<<blocks_for(n, bs), bs, 0, st>>>(n, cnt, bad);
  HIP_TRY(hipMemcpyAsync(&bad_h, bad, sizeof(bad_h), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  INCH_REQUIRE(!bad_h, "inch_rcm_device: seeds is not a permutation");
  // components, their seeds (first node in the seed order) and sizes, in seed order
  k_cc_init<<<blocks_for(n * kCcLanes, bs), bs, 0, st>>>(n, indptr, indices, label);
  k_cc_flatten<<<blocks_for(n, bs), bs, 0, st>>>(n, label);
  for (int stride : {64, 8}) {
    k_cc_link_some<<<blocks_for((n + stride - 1) / stride, bs), bs, 0, st>>>(n, stride, indptr, indices, label);
    k_cc_flatten<<<blocks_for(n, bs), bs, 0, st>>>(n, label);
  }
  HIP_TRY(hipMemcpyAsync(label2, label, n * sizeof(int32_t), hipMemcpyDeviceToDevice, st));
  k_cc_hook<<<blocks_for(n * kCcLanes, bs), bs, 0, st>>>(n, indptr, indices, label2, label);
  k_cc_flatten<<<blocks_for(n, bs), bs, 0, st>>>(n, label);
  k_rcm_init<<<blocks_for(n, bs), bs, 0, st>>>(n, claim);
  k_cc_rank<<<blocks_for(n, bs), bs, 0, st>>>(n, seeds, rank, minr);
  k_cc_minrank<<<blocks_for(n, bs), bs, 0, st>>>(n, label, rank, minr);
  k_cc_flag<<<blocks_for(n, bs), bs, 0, st>>>(n, seeds, label, minr, flag);
  HIP_TRY(scan_exclusive_into<int32_t>(n, flag, cidx, tsum, toff, st));
  k_cc_seeds<<<blocks_for(n, bs), bs, 0, st>>>(n, seeds, label, flag, cidx, S, croot, csize);
  k_cc_vertex<<<blocks_for(n, bs), bs, 0, st>>>(n, label, croot, cv, csize);
  HIP_TRY(hipGetLastError());
  int32_t C = 0;
  HIP_TRY(hipMemcpyAsync(&C, cidx + n, sizeof(C), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (C < 1 || C > n) INCH_FAIL(INCH_ERR_INVALID, "inch_rcm_device: %d components", C);
  HIP_TRY(scan_exclusive_into<int32_t>(C, csize, cstart, tsum, toff, st));
  k_rcm_seed_level<<<blocks_for(C, bs), bs, 0, st>>>(C, S, ord, claim, done, first, lend, lv);
  HIP_TRY(hipGetLastError());
  // all components' levels advance together, kRounds levels per look at the bounds
  const unsigned gg = blocks_for(n * kG, bs) < 2048 ? blocks_for(n * kG, bs) : 2048;
  const unsigned gn = blocks_for(n, bs) < 1024 ? blocks_for(n, bs) : 1024;
  Level h{0, C, 0, 0};
  while (true) {
    for (int r = 0; r < kRounds; ++r) {
      Level *now = lv + r;
      k_rcm_claim<<<gg, bs, 0, st>>>(now, ord, indptr, indices, claim, cv, cstart, done, first, fin);
      k_rcm_count<<<gg, bs, 0, st>>>(now, ord, indptr, indices, claim, cnt);
      k_rcm_scan<<<1, 1024, 0, st>>>(now, lv + (r + 1) % kRounds, n, cnt, off);
      k_rcm_scatter<<<gg, bs, 0, st>>>(now, ord, indptr, indices, claim, off, key);
      k_rcm_place<<<gn, bs, 0, st>>>(now, ord, claim, off, key, cv, first, lend, lend2, done);
      int32_t *swap = lend;
      lend = lend2;
      lend2 = swap;
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(&h, lv, sizeof(h), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (h.bad) INCH_FAIL(INCH_ERR_INVALID, "inch_rcm_device: inconsistent graph (more than %lld nodes reached)", (long long)n);
    if (h.s == h.e) break;
  }
  if (h.e != n) INCH_FAIL(INCH_ERR_INVALID, "inch_rcm_device: %d of %lld nodes ordered", h.e, (long long)n);
  k_rcm_finish<<<blocks_for(n, bs), bs, 0, st>>>(n, ord, fin, reverse, order, undo);
  HIP_TRY(hipGetLastError());
  std::vector<int32_t> cs;
  if (comp_ptr) {
    cs.resize((size_t)C + 1);
    HIP_TRY(hipMemcpyAsync(cs.data(), cstart, (C + 1) * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  }
  HIP_TRY(hipStreamSynchronize(st));
  // components are contiguous in the output order: their start offsets, ascending, then n
  if (n_comp) *n_comp = C;
  if (comp_ptr) {
    if (C + 1 > comp_cap) INCH_FAIL(INCH_ERR_CAPACITY, "inch_rcm_device: %d components exceed comp_cap", C);
    for (int64_t c = 0; c < C; ++c) {
      const int64_t s0 = cs[c], s1 = cs[c + 1];
      comp_ptr[reverse ? C - 1 - c : c] = reverse ? n - s1 : s0;
    }
    comp_ptr[C] = n;
  }
  return INCH_OK;
}

}  // extern "C"
