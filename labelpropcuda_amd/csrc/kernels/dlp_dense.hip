/*
 * dlp_dense.hip -- propagation iterations over a flagged frontier.
 *
 * The same iteration as k_propagate (dlp_propagate.hip; reference
 * iterativePropagation.cu:63-217), with the frontier as one byte per vertex
 * instead of a queue: the flags of frontier k are in the array of k's parity.
 * A launch walks the vertices in id order; a flagged, eligible vertex is
 * updated and, if its label moved by more than delta, stores a 1 to the flag
 * of every neighbour and its own in the other array.
 *
 * Against the queue this takes the claim out: no returning atomic per
 * neighbour (about 26 G/s on this GPU, against 80 to 200 G/s for stores), no
 * staging, no block-wide barrier and no global append at the end, so a
 * launch's chain of dependent round trips is flags and rows, columns,
 * neighbour labels.  It pays for walking all N flags, so it is used on
 * frontiers that are not too thin (dlp_dense_worth).
 *
 * Eligibility is looked up when a flagged vertex is met (a neighbour is
 * flagged without looking).  The list of vertices that entered a frontier is
 * not kept up: such a vertex's stamp is at least stampBase, and the list is
 * made from the stamps once the propagation has ended (k_dense_touched).
 *
 * Bound by the launch and three dependent round trips on graphs that the
 * caches hold, by the lines of labels, flags and row places beyond (6,000,000
 * vertices: five of six requests miss the L2s).  us a launch, queue and this,
 * over frontiers of one vertex in ten: 5,000 vertices 6.8 and 3.9, 50,000 7.4
 * and 4.8, 500,000 15.9 and 9.7, 6,000,000 (one in thirteen) 97.7 and 68.5.
 */
#include <algorithm>

#include "../dlp_kernels.h"
#include "../dlp_rowsum.h"

namespace {

constexpr int kDT = 256;
constexpr int kDW = kDT / 64;
constexpr int kDG = 8; /* lanes per vertex */

/* sizes of the last frontiers: 4 x kDenseSlots words a cache line apart, so
 * that the waves' additions to one of them do not queue on one address */
__device__ __forceinline__ int *dense_slot(const PropArgs &a, int k, int s) {
  return a.denseCount + ((k & 3) * kDenseSlots + s) * kDenseStride;
}

/* value of the lane n above in the row of 16 lanes (DPP row_shl:n) */
template <int N>
__device__ __forceinline__ float lane_above(float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x100 + N, 0xf, 0xf, true));
}

/* the last three levels of the row tree, over the group's 8 lanes; valid in
 * its first lane */
__device__ __forceinline__ float group_sum8(float x) {
  x = x + lane_above<4>(x);
  x = x + lane_above<2>(x);
  return x + lane_above<1>(x);
}

/* flag words of N vertices (N + 3 is beyond INT_MAX on the largest graphs) */
__host__ __device__ constexpr int dense_words(int N) { return (int)(((unsigned)N + 3u) / 4u); }
static_assert(dense_words(DLP_INT_MAX) == 1 << 29, "the largest graph's flags");

struct DenseProf {
  unsigned E = 0, C = 0, A = 0;
};

/* One vertex per group of 8 lanes (all 64 lanes of the wave call it; `act`,
 * u, beg and len are group-uniform, oldLabel, and `cur`, the label that the
 * new one replaces, are valid in the group's first lane): the new label, the
 * flags of the next frontier, and whether a label bit changed. */
__device__ __forceinline__ void dense_update(const PropArgs &a, const float *Fold, float *Fnew,
                                             uint8_t *next, bool act, int u, int beg, int len,
                                             float oldLabel, float cur, int lane, bool &diff,
                                             DenseProf &prof) {
  const int gl = lane & (kDG - 1), grp = lane / kDG;
  const dlp::GlobalPos pos{a.colInd, a.values, Fold, a.status, beg};
  if (!act) len = 0;
  float W, S;
  int c0 = -1, c1 = -1;
  const bool wide = __any(len > 2 * kDG);  // wave-uniform
  if (!wide) {
    /* at most two entries a lane, all columns and weights in flight
     * together; the slots they leave empty add +0.0 once */
    float w0 = 0.0f, w1 = 0.0f, s0 = 0.0f, s1 = 0.0f;
    if (gl < len) {
      c0 = a.colInd[beg + gl];
      w0 = a.values[beg + gl];
    }
    if (gl + kDG < len) {
      c1 = a.colInd[beg + gl + kDG];
      w1 = a.values[beg + gl + kDG];
    }
    const bool on0 = c0 >= 0 && !(a.status && a.status[c0] == DLP_VERTEX_DELETED);
    const bool on1 = c1 >= 0 && !(a.status && a.status[c1] == DLP_VERTEX_DELETED);
    const float f0 = on0 ? Fold[c0] : 0.0f, f1 = on1 ? Fold[c1] : 0.0f;
    w0 = on0 ? w0 : 0.0f;
    w1 = on1 ? w1 : 0.0f;
    s0 = on0 ? w0 * f0 : 0.0f;
    s1 = on1 ? w1 * f1 : 0.0f;
    W = group_sum8((w0 + 0.0f) + (w1 + 0.0f));
    S = group_sum8((s0 + 0.0f) + (s1 + 0.0f));
  } else {
    const bool longRow = len > 64;
    dlp::group_short_row_sums<kDG>(gl, longRow ? 0 : len, pos, W, S);
    unsigned long long longMask = dlp_ballot(longRow && gl == 0);
    while (longMask) {  // wave-uniform
      const int src = __ffsll((long long)longMask) - 1;
      longMask &= longMask - 1;
      const int lbeg = __shfl(beg, src, 64), llen = __shfl(len, src, 64);
      float LW, LS;
      dlp::group_row_sums<64>(lane, llen,
                              dlp::GlobalPos{a.colInd, a.values, Fold, a.status, lbeg}, LW, LS);
      LW = __shfl(LW, 0, 64);
      LS = __shfl(LS, 0, 64);
      if (lane == src) {
        W = LW;
        S = LS;
      }
    }
  }
  bool changed = false;
  if (act && gl == 0) {
    const float nl = dlp::new_label(W, S, oldLabel);
    Fnew[u] = nl;
    changed = fabsf(nl - oldLabel) > a.delta;
    diff = diff || __float_as_int(nl) != __float_as_int(cur);
    prof.E += (unsigned)len;
    prof.A += 1u;
    if (changed) {
      prof.C += (unsigned)len + 1u;
      next[u] = 1;
    }
  }
  if ((dlp_ballot(changed) >> (grp * kDG)) & 1ull) {  // group-uniform
    if (!wide) {
      if (c0 >= 0) next[c0] = 1;
      if (c1 >= 0) next[c1] = 1;
    } else {
      for (int p = gl; p < len; p += kDG) {
        const int v = a.colInd[beg + p];
        if (v >= 0) next[v] = 1;
      }
    }
  }
}

__device__ __forceinline__ void dense_row(const PropArgs &a, int u, int &beg, int &len) {
  if (a.rowInfo) {
    const int2 r = a.rowInfo[u];
    beg = r.x;
    len = r.y;
  } else {
    beg = a.rowBeg[u];
    len = a.rowLen ? a.rowLen[u] : a.rowEnd[u] - beg;
  }
}

/* what a queue launch records at its start, for the finished iteration k:
 * its frontier size, the iteration and update counters.  One wave. */
__device__ __forceinline__ void dense_fold(const PropArgs &a, int k, int lane) {
  DevCounters *c = a.ctr;
  if (c->denseFolded >= k) return;  // wave-uniform
  const int n = __builtin_amdgcn_readlane(
      dlp_wave_inclusive_sum(lane < kDenseSlots ? *dense_slot(a, k, lane) : 0), 63);
  if (lane != 0) return;
  c->denseFolded = k;
  c->denseSize[k & 3] = n;
  if (k == 0) c->frontier0 = n;
  if (n == 0) return;
  if (a.iterSizes && k < a.iterSizesCap) a.iterSizes[k] = n;
  c->iterUsed = k + 1;
  c->updates += (unsigned long long)n;
}

/* Iteration k.  Each wave takes tiles of `span` consecutive vertices: 64 * VPL,
 * VPL flags a lane, or fewer than 64 (dlp_dense_span).  VPL 1 (thick
 * frontiers): every lane loads the row place,
 * label and stamp of its vertex together with its flag, so meeting a flagged
 * vertex costs no further round trip; the groups fetch them from the lanes.
 * VPL > 1 (thin ones): flags only, then the loads of the flagged vertices.
 *
 * WATCH (from kCycleFrom on) is the cycle test (dlp_cycle_skip).  Iteration k
 * compares every label it writes with the one it replaces (lastDiff) and,
 * once labels stand still, marks the vertices of its frontier by generation
 * cycleBase + 1 + k in the array of k's parity, where the generation found
 * tells whether a vertex was in frontier k - 2 (lastMiss if not).  Frontier
 * k - 2 made of vertices of frontier k - 4 and as large, and no label changed
 * by iterations k - 4 and later: the state of k - 2 is that of k - 4, and so
 * is that of k the one of k - 2.  Every reader of the words takes the same
 * decision although iteration k itself writes them: it writes only when there
 * is no cycle, only the value k, and no value that large gives a cycle. */
template <int VPL, bool WATCH>
__global__ __launch_bounds__(kDT) void k_dense(PropArgs a, int k, int N, int tiles, int span) {
  __shared__ unsigned short lists[kDW][64 * VPL];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int gl = lane & (kDG - 1), grp = lane / kDG;
  unsigned short *list = lists[wv];
  uint8_t *cur = (k & 1) ? a.flag1 : a.flag0;
  uint8_t *next = (k & 1) ? a.flag0 : a.flag1;
  const float *Fold = (k & 1) ? a.lab1 : a.lab0;
  float *Fnew = (k & 1) ? a.lab0 : a.lab1;
  const int gwave = (int)((blockIdx.x * kDT + threadIdx.x) >> 6);
  const int nwaves = (int)(((gridDim.x - 1) * kDT) >> 6);
  DevCounters *c = a.ctr;
  const int stampBase = c->stampBase;
  bool look = false, mark = false, diff = false, miss = false;
  int lastDiff = 0, tag = 0;
  int *marks = (k & 1) ? a.mark1 : a.mark0;
  if (WATCH) {
    const int base = c->cycleBase, n2 = c->denseSize[(k - 2) & 3];
    lastDiff = c->lastDiff;
    look = base >= 0;
    tag = base + 1 + k;
    const bool cycle = look && n2 > 0 && n2 == c->denseSize[(k - 4) & 3] && lastDiff < k - 4 &&
                       c->lastMiss < k - 2;
    if (c->cycleIter > 0 || cycle) {  // grid-uniform: found before, or here
      if (blockIdx.x == 0 && threadIdx.x == 0 && c->cycleIter == 0) c->cycleIter = k;
      return;
    }
    mark = look && lastDiff < k - 1;
  }
  int count = 0; /* wave-uniform: vertices of frontier k */
  DenseProf prof;
  if (blockIdx.x == gridDim.x - 1) {  // the last block keeps the books
    if (wv == 0) dense_fold(a, k - 1, lane);
    if (wv == 1 && lane < kDenseSlots) *dense_slot(a, k + 1, lane) = 0;
    if (WATCH && !mark && threadIdx.x == 0) c->lastMiss = k;
    return;
  }
  for (int tile = gwave; tile < tiles; tile += nwaves) {  // wave-uniform
    const int base = tile * span;
    if constexpr (VPL == 1) {
      const int v = base + lane;
      const bool in = lane < span && v < N;
      const int f = in ? cur[v] : 0;
      const int stamp = in ? a.iterStamp[v] : DLP_INT_MAX;
      const float old = in ? Fold[v] : 0.0f;
      const float now = (WATCH && in) ? Fnew[v] : 0.0f;
      int beg = 0, len = 0;
      if (in) dense_row(a, v, beg, len);
      if (f) cur[v] = 0;
      const bool act = f && stamp != DLP_INT_MAX;
      const unsigned long long m = dlp_ballot(act);
      if (m == 0ull) continue;
      if (act && stamp < stampBase) a.iterStamp[v] = stampBase; /* entered a frontier */
      if (WATCH && mark && act) {
        miss = miss || marks[v] != tag - 2;
        marks[v] = tag;
      }
      const int n = __popcll(m);
      count += n;
      if (act) list[dlp_rank_below(m)] = (unsigned short)lane;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      for (int i0 = 0; i0 < n; i0 += 64 / kDG) {  // wave-uniform
        const bool on = i0 + grp < n;
        const int src = on ? list[i0 + grp] : lane;
        const int rb = __shfl(beg, src, 64), rl = __shfl(len, src, 64);
        const float ol = __shfl(old, src, 64);
        const float cl = WATCH ? __shfl(now, src, 64) : 0.0f;
        dense_update(a, Fold, Fnew, next, on, base + src, rb, rl, ol, cl, lane, diff, prof);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // read before the next tile
    } else {
      static_assert(VPL == 1 || VPL % 4 == 0, "flags are loaded as words");
      constexpr int WPL = VPL / 4;
      unsigned w[WPL];
      int c = 0;
      const int v0 = base + lane * VPL;
#pragma unroll
      for (int j = 0; j < WPL; ++j) {  // the arrays are padded to whole words
        w[j] = v0 + 4 * j < N ? reinterpret_cast<const unsigned *>(cur)[(v0 >> 2) + j] : 0u;
        c += __popc(w[j]);  // a flag byte is 0 or 1
      }
      const int incl = dlp_wave_inclusive_sum(c);
      const int n = __builtin_amdgcn_readlane(incl, 63);
      if (n == 0) continue;  // wave-uniform
      int p = incl - c;
#pragma unroll
      for (int j = 0; j < WPL; ++j) {
        if (!w[j]) continue;
        reinterpret_cast<unsigned *>(cur)[(v0 >> 2) + j] = 0u;
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if ((w[j] >> (8 * b)) & 1u) list[p++] = (unsigned short)(lane * VPL + 4 * j + b);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      for (int i0 = 0; i0 < n; i0 += 64 / kDG) {  // wave-uniform
        const bool on = i0 + grp < n;
        const int u = base + (on ? list[i0 + grp] : 0);
        int beg = 0, len = 0, stamp = DLP_INT_MAX;
        float old = 0.0f, now = 0.0f;
        if (on) {
          stamp = a.iterStamp[u];
          dense_row(a, u, beg, len);
          old = Fold[u];
          if (WATCH) now = Fnew[u];
        }
        const bool act = stamp != DLP_INT_MAX;
        if (act && gl == 0 && stamp < stampBase) a.iterStamp[u] = stampBase;
        if (WATCH && mark && act && gl == 0) {
          miss = miss || marks[u] != tag - 2;
          marks[u] = tag;
        }
        count += __popcll(dlp_ballot(act && gl == 0));
        dense_update(a, Fold, Fnew, next, act, u, beg, len, old, now, lane, diff, prof);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // read before the next tile
    }
  }
  if (lane == 0 && count) atomicAdd(dense_slot(a, k, gwave & (kDenseSlots - 1)), count);
  if (WATCH) {
    const bool anyDiff = __any(diff), anyMiss = __any(miss);
    /* a wave that met iteration k's own lastDiff has marked nothing */
    if (lane == 0 && anyDiff) c->lastDiff = k;
    if (lane == 0 && (anyMiss || lastDiff >= k)) c->lastMiss = k;
  }
  if (a.profile) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      prof.E += __shfl_xor(prof.E, off, 64);
      prof.C += __shfl_xor(prof.C, off, 64);
      prof.A += __shfl_xor(prof.A, off, 64);
    }
    if (lane == 0 && prof.A) {
      atomicAdd(&a.ctr->profFlagUpdates, (unsigned long long)prof.A);
      atomicAdd(&a.ctr->profFlagEdges, (unsigned long long)prof.E);
      atomicAdd(&a.ctr->profFlagChangedEdges, (unsigned long long)prof.C);
    }
  }
}

/* iteration k - 1 recorded for the host (a cycle was found: the last one that
 * ran); the queue counts, which the flagged iterations do not use, start from
 * zero */
__global__ __launch_bounds__(64) void k_dense_fold(PropArgs a, int k) {
  const int kc = a.ctr->cycleIter;
  dense_fold(a, (kc > 0 ? kc : k) - 1, threadIdx.x);
  if (threadIdx.x < 3) a.ctr->qcount[threadIdx.x] = 0;
}

/* flags and counts to zero before iteration k */
__global__ __launch_bounds__(kDT) void k_dense_clear(PropArgs a, int k, int N) {
  const int i = (int)(blockIdx.x * kDT + threadIdx.x), stride = (int)(gridDim.x * kDT);
  for (int w = i; w < dense_words(N); w += stride) {
    reinterpret_cast<unsigned *>(a.flag0)[w] = 0u;
    reinterpret_cast<unsigned *>(a.flag1)[w] = 0u;
  }
  for (int w = i; w < 4 * kDenseSlots; w += stride) a.denseCount[w * kDenseStride] = 0;
  if (i == 0) {
    a.ctr->denseFolded = k - 1;
    a.ctr->denseSize[(k - 1) & 3] = a.ctr->denseSize[(k - 2) & 3] = DLP_INT_MAX;  // not known
    a.ctr->lastDiff = a.ctr->lastMiss = k > kCycleFrom ? k : kCycleFrom;
  }
}

/* the queue of iteration k -> flags */
__global__ __launch_bounds__(kDT) void k_dense_enter(PropArgs a, int k) {
  const int n = a.ctr->qcount[k % 3];
  const int *q = (k & 1) ? a.q1 : a.q0;
  uint8_t *cur = (k & 1) ? a.flag1 : a.flag0;
  for (int i = (int)(blockIdx.x * kDT + threadIdx.x); i < n; i += (int)(gridDim.x * kDT))
    cur[q[i]] = 1;
}

/* Flags of iteration k -> the queue of iteration kOut and the stamps a claim
 * would have left.  kOut > k (even distance): iteration k is in the state of
 * k - 2, the frontiers up to kOut alternate in size as the last two did. */
__global__ __launch_bounds__(kDT) void k_dense_exit(PropArgs a, int k, int kOut, int N) {
  if (blockIdx.x == 0 && threadIdx.x == 0 && a.ctr->cycleIter > 0) {
    DevCounters *c = a.ctr;
    const unsigned long long sum =
        (unsigned long long)((kOut - k) / 2) *
        ((unsigned long long)c->denseSize[(k - 2) & 3] +
         (unsigned long long)c->denseSize[(k - 1) & 3]);
    if (kOut > k) c->iterUsed = kOut;
    c->updates += sum;
    c->skippedIterations += (unsigned long long)(kOut - k);
    c->skippedUpdates += sum;
    c->cycleIter = 0;
    c->cycleBase = -1;  // at most one iteration is left
  }
  const uint8_t *cur = (k & 1) ? a.flag1 : a.flag0;
  int *q = (k & 1) ? a.q1 : a.q0;
  const int stamp = a.ctr->stampBase + kOut;
  const int words = dense_words(N);
  const int wave0 = (int)((blockIdx.x * kDT + threadIdx.x) & ~63u);
  const int lane = threadIdx.x & 63, stride = (int)(gridDim.x * kDT);
  for (int b = wave0; b < words; b += stride) {  // wave-uniform
    const int i = b + lane;
    const unsigned w = i < words ? reinterpret_cast<const unsigned *>(cur)[i] : 0u;
    if (!__any(w != 0u)) continue;  // wave-uniform
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int v = 4 * i + j;
      const bool in = ((w >> (8 * j)) & 1u) && a.iterStamp[v] != DLP_INT_MAX;
      const int slot = dlp_wave_append(&a.ctr->qcount[kOut % 3], in);
      if (in) {
        q[slot] = v;
        a.iterStamp[v] = stamp;
      }
    }
  }
}

__global__ void k_dense_touched_clear(DevCounters *c) { c->touched = 0; }

/* the vertices that entered a frontier in this batch: eligible, stamped at
 * or above stampBase */
__global__ __launch_bounds__(kDT) void k_dense_touched(PropArgs a, int N) {
  constexpr int R = 8; /* vertices per thread and round */
  __shared__ int waveSum[kDW];
  __shared__ int blockBase;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int base0 = a.ctr->stampBase;
  for (long long b = (long long)blockIdx.x * (kDT * R); b < N;
       b += (long long)gridDim.x * (kDT * R)) {  // block-uniform
    unsigned hit = 0u;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const long long v = b + j * kDT + threadIdx.x;
      const int st = v < N ? a.iterStamp[v] : DLP_INT_MAX;
      hit |= (st >= base0 && st != DLP_INT_MAX ? 1u : 0u) << j;
    }
    const int c = __popc(hit);
    const int incl = dlp_wave_inclusive_sum(c);
    if (lane == 63) waveSum[wv] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
      int run = 0;
      for (int w = 0; w < kDW; ++w) {
        const int t = waveSum[w];
        waveSum[w] = run;
        run += t;
      }
      blockBase = run ? atomicAdd(&a.ctr->touched, run) : 0;
    }
    __syncthreads();
    int p = blockBase + waveSum[wv] + incl - c;
#pragma unroll
    for (int j = 0; j < R; ++j)
      if ((hit >> j) & 1u) a.touched[p++] = (int)(b + j * kDT + threadIdx.x);
    __syncthreads();  // waveSum and blockBase are rewritten in the next round
  }
}

int dense_grid(long long threads, int cap) {
  return (int)std::max<long long>(1, std::min<long long>((threads + kDT - 1) / kDT, cap));
}

}  // namespace

int dlp_launch_dense_enter(const PropArgs &a, int k, int N, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_dense_clear, dim3(dense_grid(((long long)N + 3) / 4, 2048)), dim3(kDT), 0, s,
                     a, k, N);
  DLP_LAUNCHED("k_dense_clear");
  hipLaunchKernelGGL(k_dense_enter, dim3(dense_grid(n, 2048)), dim3(kDT), 0, s, a, k);
  DLP_LAUNCHED("k_dense_enter");
  return DLP_OK;
}

int dlp_launch_dense(const PropArgs &a, int k, int N, bool thick, hipStream_t s) {
  const int span = thick ? dlp_dense_span(N) : 64 * kDenseThinFlags;
  const int tiles = (int)(((long long)N + span - 1) / span);
  const int blocks = dense_grid((long long)tiles * 64, kDenseMaxBlocks) + 1;
  const bool watch = a.cycles && a.mark0 && k >= kCycleFrom;
#define DLP_LAUNCH_DENSE(V, W) \
  hipLaunchKernelGGL((k_dense<V, W>), dim3(blocks), dim3(kDT), 0, s, a, k, N, tiles, span)
  if (thick && watch)
    DLP_LAUNCH_DENSE(1, true);
  else if (thick)
    DLP_LAUNCH_DENSE(1, false);
  else if (watch)
    DLP_LAUNCH_DENSE(kDenseThinFlags, true);
  else
    DLP_LAUNCH_DENSE(kDenseThinFlags, false);
#undef DLP_LAUNCH_DENSE
  DLP_LAUNCHED("k_dense");
  return DLP_OK;
}

int dlp_launch_dense_fold(const PropArgs &a, int k, hipStream_t s) {
  hipLaunchKernelGGL(k_dense_fold, dim3(1), dim3(64), 0, s, a, k);
  DLP_LAUNCHED("k_dense_fold");
  return DLP_OK;
}

int dlp_launch_dense_exit(const PropArgs &a, int k, int kOut, int N, hipStream_t s) {
  hipLaunchKernelGGL(k_dense_exit, dim3(dense_grid(((long long)N + 3) / 4, 2048)), dim3(kDT), 0, s,
                     a, k, kOut, N);
  DLP_LAUNCHED("k_dense_exit");
  return DLP_OK;
}

int dlp_launch_dense_touched(const PropArgs &a, int N, hipStream_t s) {
  hipLaunchKernelGGL(k_dense_touched_clear, dim3(1), dim3(1), 0, s, a.ctr);
  DLP_LAUNCHED("k_dense_touched_clear");
  hipLaunchKernelGGL(k_dense_touched, dim3(dense_grid(((long long)N + 7) / 8, 2048)), dim3(kDT), 0,
                     s, a, N);
  DLP_LAUNCHED("k_dense_touched");
  return DLP_OK;
}
