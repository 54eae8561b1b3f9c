// Phase unwrapping, DEROUL 1 with VOLKOV 0 (Herraez: phaseUnwrapping_Mat,
// pretraitement_hors_axe_CPU/deroulement_herraez.cpp:32-75).
//
// The reference computes a reliability per pixel (second differences of the
// wrapped phase, :382-404; border pixels keep 9999999 + rand(), :348), one
// per edge (the sum of its two pixels', :409-452), sorts the edges with its
// own merge sort (:160-195) and then merges pixel groups edge by edge in that
// order (:455-552): Kruskal's algorithm, so the edges that merge groups form
// the minimum spanning tree of the grid for the edge weights "position in
// the sorted order" (all distinct). The unwrapped phase is the wrapped one
// plus 2 pi times an integer increment that makes every tree edge step the
// wrapped difference (find_wrap, :370-380).
//
// GPU restructuring (same tree, same increments up to one global 2 pi k):
//  - No sort. The reference's merge sort halves a range of s edges into two
//    runs of s / 2 and leaves an odd range's last element where it is. A
//    two-pointer merge of runs orders elements as a stable merge of the runs'
//    running maxima; an element's running max is its own key, except for a
//    left-out last element, whose running max is the largest key of its whole
//    range from the moment the range is merged on. So the sorted order is
//    the plain stable order of (key', edge index), where key' is the key, or
//    for the left-out elements the largest key of their range. Kruskal and
//    Boruvka only compare edges: the 64-bit pair (key', index) does that
//    without the positions.
//  - k_herr_edges: wrapped phase (atan2 of the demodulated field),
//    reliabilities and edge keys, a tile with its halo in LDS; border values
//    from the host (the reference's unseeded rand() stream, restated there);
//  - k_herr_tails: key' of the left-out edges. All ranges of one depth have
//    the same size: blocks take ranges of at most 2048 edges and the ranges'
//    maxima go up the recursion; one block per angle takes the depths above;
//  - k_herr_tile: Boruvka inside 32 x 32 tiles in LDS. Every component takes
//    its lowest edge, leaving the tile or not, and hooks along it if it stays
//    inside (that edge is in the minimum spanning tree whatever happens
//    elsewhere), until every component's lowest edge leaves the tile;
//  - k_herr_finish: the rest of the tree, one block per angle on the tiles'
//    components (a few per cent of the pixels) and the edges between them.
//    Each pixel keeps its increment relative to its component's root; a hook
//    stores the root's increment relative to the new root, fixed by the edge's
//    wrap count. The tree is the unique minimum one, the reference's; only
//    the root whose increment is 0 may differ, a constant 2 pi k that the
//    polynomial fit which always follows unwrapping (its constant monomial)
//    removes.
// All of it waits on LDS and L2 latency, not on bandwidth (about 60 bytes per
// pixel). Measured on 100 crops of 128^2: the reference's sort replayed level
// by level in one block per angle, then Boruvka in 75 launches over global
// memory, 5560 us; this form 190 us (tiles 89, finish 40, tails 32, edges 17).
#include <hip/hip_runtime.h>

#include <cmath>

#include "internal.hpp"

namespace mtd {

constexpr float kHerrPi = 3.141592654f;     // deroulement_herraez.cpp:9
constexpr float kHerrTwoPi = 6.283185307f;  // :10

__device__ __forceinline__ float herr_wrap(float x) {
  return x > kHerrPi ? x - kHerrTwoPi : (x < -kHerrPi ? x + kHerrTwoPi : x);
}

// edge e of the C x C grid: horizontal edges row-major first, then vertical
__device__ __forceinline__ void herr_edge(int e, int C, int& p1, int& p2) {
  const int nh = C * (C - 1);
  if (e < nh) {
    const int y = e / (C - 1), x = e - y * (C - 1);
    p1 = y * C + x;
    p2 = p1 + 1;
  } else {
    p1 = e - nh;
    p2 = p1 + C;
  }
}

// number of 2 pi between the two pixels of an edge (find_wrap)
__device__ __forceinline__ int herr_wrapcount(float v1, float v2) {
  const float d = v1 - v2;
  return d > kHerrPi ? -1 : (d < -kHerrPi ? 1 : 0);
}

// index of border pixel (y, x) in the packed border table: row 0, row C-1,
// then columns 0 and C-1 of rows 1 .. C-2
__device__ __forceinline__ int herr_border_slot(int y, int x, int C) {
  if (y == 0) return x;
  if (y == C - 1) return C + x;
  return 2 * C + 2 * (y - 1) + (x == 0 ? 0 : 1);
}

// ---------------------------------------------------------------------------
// phase, reliabilities, edge keys: a block per 32 x 8 pixels
// ---------------------------------------------------------------------------
constexpr int kEx = 32, kEy = 8;

__global__ void __launch_bounds__(kEx * kEy)
k_herr_edges(const float2* __restrict__ iu, int C, const float* __restrict__ border,
             float* __restrict__ ph, float* __restrict__ key) {
  // the reliability sums are the reference's float products and sums: no
  // fused multiply-add
#pragma clang fp contract(off)
  __shared__ float lp[kEy + 3][kEx + 3];  // phases of rows y0 - 1 .., columns x0 - 1 ..
  __shared__ float lr[kEy + 1][kEx + 1];  // reliabilities of rows y0 .., columns x0 ..
  const int a = blockIdx.z, x0 = blockIdx.x * kEx, y0 = blockIdx.y * kEy, tid = threadIdx.x;
  const size_t n = (size_t)C * C, nh = (size_t)C * (C - 1);
  const float2* iu_a = iu + a * n;
  for (int t = tid; t < (kEy + 3) * (kEx + 3); t += kEx * kEy) {
    const int j = t / (kEx + 3), i = t - j * (kEx + 3);
    const int y = y0 + j - 1, x = x0 + i - 1;
    if (y >= 0 && y < C && x >= 0 && x < C) {
      const float2 u = iu_a[(size_t)((y + C / 2) % C) * C + (x + C / 2) % C];
      lp[j][i] = atan2f(u.y, u.x);
    }
  }
  __syncthreads();
  for (int t = tid; t < (kEy + 1) * (kEx + 1); t += kEx * kEy) {
    const int j = t / (kEx + 1), i = t - j * (kEx + 1);
    const int y = y0 + j, x = x0 + i;
    if (y >= C || x >= C) continue;
    float r;
    if (y == 0 || y == C - 1 || x == 0 || x == C - 1) {
      r = border[(size_t)a * (4 * C - 4) + herr_border_slot(y, x, C)];
    } else {
      // calculate_reliability (:392-398): second differences of wrapped
      // first differences, summed in float in the reference's order
      auto P = [&](int dy, int dx) { return lp[j + 1 + dy][i + 1 + dx]; };
      const float c = P(0, 0);
      const float H = herr_wrap(P(0, -1) - c) - herr_wrap(c - P(0, 1));
      const float V = herr_wrap(P(-1, 0) - c) - herr_wrap(c - P(1, 0));
      const float D1 = herr_wrap(P(-1, -1) - c) - herr_wrap(c - P(1, 1));
      const float D2 = herr_wrap(P(-1, 1) - c) - herr_wrap(c - P(1, -1));
      r = ((H * H + V * V) + D1 * D1) + D2 * D2;
    }
    lr[j][i] = r;
  }
  __syncthreads();
  const int i = tid % kEx, j = tid / kEx, y = y0 + j, x = x0 + i;
  if (y >= C || x >= C) return;
  const size_t p = (size_t)y * C + x;
  ph[a * n + p] = lp[j + 1][i + 1];
  // edge reliabilities (:418, :443): float sum of the two pixels'
  float* k = key + a * 2 * nh;
  if (x < C - 1) k[(size_t)y * (C - 1) + x] = lr[j][i] + lr[j][i + 1];
  if (y < C - 1) k[nh + p] = lr[j][i] + lr[j + 1][i];
}

// ---------------------------------------------------------------------------
// the left-out edges' keys
// ---------------------------------------------------------------------------
constexpr int kMaxDepth = 40;
constexpr int kTailThreads = 512, kTailN = 2048;

struct SortLevels {
  int s[kMaxDepth + 1];  // range size at each depth (s[0] = edge count)
  int deepest;           // last depth whose ranges (size >= 2) are merged
};

// start of the j-th range (left to right) of depth d, within the range of
// depth d0 it belongs to
__device__ __forceinline__ int herr_range_at(int j, int d, int d0, const SortLevels& L) {
  int start = 0;
  for (int i = d0 + 1; i <= d; ++i)
    if ((j >> (d - i)) & 1) start += L.s[i];
  return start;
}

// Block x: the x-th range of depth d0 (at most kTailN edges), its left-out
// edges at that depth and below, and its largest key. A NaN key counts as
// -infinity (fmaxf), as in the merge's comparisons.
__global__ void __launch_bounds__(kTailThreads)
k_herr_tails(float* __restrict__ key, int m, SortLevels L, int d0, float* __restrict__ top) {
  __shared__ float k[kTailN], mx[2][kTailN];
  const int a = blockIdx.y, tid = threadIdx.x, n = L.s[d0];
  float* ka = key + (size_t)a * m + herr_range_at(blockIdx.x, d0, 0, L);
  for (int p = tid; p < n; p += kTailThreads) k[p] = fmaxf(-INFINITY, ka[p]);
  __syncthreads();
  int cur = 0;
  for (int d = L.deepest + 1; d >= d0; --d) {  // uniform
    const int s = L.s[d];
    for (int j = tid; j < 1 << (d - d0); j += kTailThreads) {
      const int start = herr_range_at(j, d, d0, L);
      float v = s & 1 ? k[start + s - 1] : -INFINITY;
      if (d <= L.deepest) {
        v = fmaxf(v, fmaxf(mx[cur][2 * j], mx[cur][2 * j + 1]));
        if (s & 1) ka[start + s - 1] = v;
      }
      mx[cur ^ 1][j] = v;
    }
    cur ^= 1;
    __syncthreads();
  }
  if (tid == 0) top[(size_t)a * gridDim.x + blockIdx.x] = mx[cur][0];
}

// The depths above d0, one block per angle: the ranges' maxima in place, a
// chunk of ranges at a time (range j reads 2j and 2j + 1, all of them read
// before any of the chunk is written, later chunks read further on).
__global__ void __launch_bounds__(kTailThreads)
k_herr_tails_top(float* __restrict__ key, int m, SortLevels L, int d0, float* top) {
  const int a = blockIdx.x, tid = threadIdx.x;
  float* ka = key + (size_t)a * m;
  float* t = top + ((size_t)a << d0);
  for (int d = d0 - 1; d >= 0; --d) {
    const int s = L.s[d];
    for (int j0 = 0; j0 < 1 << d; j0 += kTailThreads) {
      const int j = j0 + tid;
      float v = -INFINITY;
      if (j < 1 << d) {
        v = fmaxf(t[2 * j], t[2 * j + 1]);
        if (s & 1) {
          float* tail = ka + herr_range_at(j, d, 0, L) + s - 1;
          v = fmaxf(v, *tail);
          *tail = v;
        }
      }
      __syncthreads();
      if (j < 1 << d) t[j] = v;
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
// Boruvka
// ---------------------------------------------------------------------------
using u64 = unsigned long long;
constexpr u64 kNoEdge = ~0ull;

// (key', edge index) as one integer: floats in their order (-0 as +0, NaN as
// -infinity), then the index
__device__ __forceinline__ u64 herr_pair(float k, int e) {
  const unsigned b = __float_as_uint(fmaxf(-INFINITY, k) + 0.f);
  return (u64)(b ^ ((b >> 31) ? 0xFFFFFFFFu : 0x80000000u)) << 32 | (unsigned)e;
}

// link of a root: (root it hooks to, its increment relative to that root)
__device__ __forceinline__ u64 bor_pack(int up, int off) {
  return (u64)(unsigned)up | ((u64)(unsigned)off << 32);
}
__device__ __forceinline__ int bor_up(u64 v) { return (int)(unsigned)v; }
__device__ __forceinline__ int bor_off(u64 v) { return (int)(unsigned)(v >> 32); }

template <int SCOPE>
__device__ __forceinline__ u64 bor_load(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, SCOPE);
}
template <int SCOPE>
__device__ __forceinline__ void bor_store(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, SCOPE);
}
// lowers *p to v; the read first only saves atomics (*p only falls, so a
// stale value is never too low)
template <int SCOPE>
__device__ __forceinline__ void bor_offer(u64* p, u64 v) {
  if (v < bor_load<SCOPE>(p)) __hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, SCOPE);
}
// Follows root i's links to the root of its new component, accumulating the
// increments; only this thread writes link[i] (64-bit stores), so every link
// read is some valid ancestor of its root with a consistent increment.
template <int SCOPE>
__device__ __forceinline__ void bor_jump(u64* link, int i) {
  u64 v = bor_load<SCOPE>(link + i);
  while (bor_up(v) != i) {
    const u64 w = bor_load<SCOPE>(link + bor_up(v));
    if (bor_up(w) == bor_up(v)) break;  // the new root
    v = bor_pack(bor_up(w), bor_off(v) + bor_off(w));
    bor_store<SCOPE>(link + i, v);
  }
}
constexpr int kBlockScope = __HIP_MEMORY_SCOPE_WORKGROUP;

// tiles of 32 x 32 pixels, one per thread (100 crops of 128^2: 89 us, 102 with
// two pixels per thread and 131 with four: the rounds wait on LDS, which the
// waves of two such blocks per CU hide best)
constexpr int kTile = 32, kTileN = kTile * kTile, kTileThreads = 1024;
constexpr int kTileE = kTileN / kTileThreads;

__global__ void __launch_bounds__(kTileThreads)
k_herr_tile(const float* __restrict__ key, const float* __restrict__ ph, int C,
            unsigned short* __restrict__ comp, int* __restrict__ inc, int* __restrict__ nroots,
            u64* __restrict__ edges, int* __restrict__ nedges) {
  __shared__ float lph[kTileN];
  // keys of the edges to the right of columns -1 .. 31 and below rows -1 .. 31
  __shared__ float kr[kTile][kTile + 1], kd[kTile + 1][kTile];
  __shared__ u64 best[kTileN], link[kTileN];
  __shared__ int cmp[kTileN], linc[kTileN], cnt[2], ebase;
  const int a = blockIdx.y, nt = (C + kTile - 1) / kTile, tid = threadIdx.x;
  const int X0 = (blockIdx.x % nt) * kTile, Y0 = (blockIdx.x / nt) * kTile;
  const int w = min(kTile, C - X0), h = min(kTile, C - Y0);  // the tile's pixels
  const int nh = C * (C - 1);
  const float* ka = key + (size_t)a * 2 * nh;
  const size_t base = (size_t)a * C * C;
  for (int t = tid; t < kTile * (kTile + 1); t += kTileThreads) {
    const int y = t / (kTile + 1), x = t - y * (kTile + 1);
    const int gx = X0 + x - 1;
    if (y < h && gx >= 0 && gx < C - 1 && x <= w) kr[y][x] = ka[(Y0 + y) * (C - 1) + gx];
  }
  for (int t = tid; t < kTile * (kTile + 1); t += kTileThreads) {
    const int y = t / kTile, x = t % kTile;
    const int gy = Y0 + y - 1;
    if (x < w && gy >= 0 && gy < C - 1 && y <= h) kd[y][x] = ka[nh + gy * C + X0 + x];
  }
  if (tid < 2) cnt[tid] = 0;
#pragma unroll
  for (int i = 0; i < kTileE; ++i) {
    const int q = tid + i * kTileThreads, x = q % kTile, y = q / kTile;
    linc[q] = 0;
    cmp[q] = q;
    if (x < w && y < h) lph[q] = ph[base + (size_t)(Y0 + y) * C + X0 + x];
  }
  // edge s (0: right, 1: below, 2: left, 3: above) of the pixel at (x, y):
  // whether the image has it, its pair, and the tile pixel at its other end
  // (-1: outside the tile)
  auto edge = [&](int x, int y, int s, u64& pair, int& other) {
    const int gx = X0 + x, gy = Y0 + y;
    switch (s) {
      case 0:
        if (gx >= C - 1) return false;
        pair = herr_pair(kr[y][x + 1], gy * (C - 1) + gx);
        other = x + 1 < w ? y * kTile + x + 1 : -1;
        return true;
      case 1:
        if (gy >= C - 1) return false;
        pair = herr_pair(kd[y + 1][x], nh + gy * C + gx);
        other = y + 1 < h ? (y + 1) * kTile + x : -1;
        return true;
      case 2:
        if (gx == 0) return false;
        pair = herr_pair(kr[y][x], gy * (C - 1) + gx - 1);
        other = x > 0 ? y * kTile + x - 1 : -1;
        return true;
      default:
        if (gy == 0) return false;
        pair = herr_pair(kd[y][x], nh + (gy - 1) * C + gx);
        other = y > 0 ? (y - 1) * kTile + x : -1;
        return true;
    }
  };
  // edges of each pixel not yet inside its component (edges inside one stay
  // there: the rounds look at fewer and fewer)
  unsigned open[kTileE];
#pragma unroll
  for (int i = 0; i < kTileE; ++i) {
    const int q = tid + i * kTileThreads;
    open[i] = q % kTile < w && q / kTile < h ? 15u : 0u;
  }
  while (true) {  // each round with a hook leaves fewer components
    u64 mine[kTileE];
    int side[kTileE];
#pragma unroll
    for (int i = 0; i < kTileE; ++i) {
      const int q = tid + i * kTileThreads;
      best[q] = kNoEdge;
      link[q] = bor_pack(q, 0);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTileE; ++i) {
      const int q = tid + i * kTileThreads;
      mine[i] = kNoEdge;
      side[i] = 0;
      if (!open[i]) continue;
      const int c = cmp[q];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (!(open[i] >> s & 1)) continue;
        u64 pr;
        int o;
        if (!edge(q % kTile, q / kTile, s, pr, o) || (o >= 0 && cmp[o] == c)) {
          open[i] &= ~(1u << s);
        } else if (pr < mine[i]) {
          mine[i] = pr;
          side[i] = s;
        }
      }
      if (mine[i] != kNoEdge) bor_offer<kBlockScope>(best + c, mine[i]);
    }
    __syncthreads();
    // the pixel whose edge its component took hooks the component's root
    bool hooked = false;
#pragma unroll
    for (int i = 0; i < kTileE; ++i) {
      const int q = tid + i * kTileThreads, s = side[i];
      if (mine[i] == kNoEdge) continue;
      const int c = cmp[q];
      if (best[c] != mine[i]) continue;
      u64 pr;
      int o;
      edge(q % kTile, q / kTile, s, pr, o);
      if (o < 0) continue;  // the component waits for the whole image's rounds
      const int c2 = cmp[o];
      // both ends took this edge: the lower root stays
      if (best[c2] == mine[i] && c < c2) continue;
      // inc(p2) = inc(p1) - wrapcount(p1, p2) across the edge (gatherPIXELs,
      // :482, :495), p1 its left or upper pixel
      const int d = s < 2 ? linc[o] - linc[q] + herr_wrapcount(lph[q], lph[o])
                          : linc[o] - linc[q] - herr_wrapcount(lph[o], lph[q]);
      link[c] = bor_pack(c2, d);
      hooked = true;
    }
    if (!__syncthreads_or(hooked)) break;
#pragma unroll
    for (int i = 0; i < kTileE; ++i) {
      const int q = tid + i * kTileThreads;
      if (cmp[q] == q) bor_jump<kBlockScope>(link, q);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTileE; ++i) {
      const int q = tid + i * kTileThreads;
      const u64 v = link[cmp[q]];
      cmp[q] = bor_up(v);
      linc[q] += bor_off(v);
    }
    __syncthreads();
  }
  // The tile's components get numbers 0, 1, .. in the order of their roots'
  // pixels (into best's storage, past its last use), and the edges between
  // components, or out of the tile, go to the angle's list (its order is free:
  // only the least pair of a component counts).
  int* id = (int*)best;
  const int lane = tid & 63;
  int roots = 0;
#pragma unroll
  for (int i = 0; i < kTileE; ++i) {
    const int q = tid + i * kTileThreads, x = q % kTile, y = q / kTile;
    const bool root = cmp[q] == q && x < w && y < h;
    const u64 bal = __ballot(root);
    if (lane == 0) link[q / 64] = __popcll(bal);
    if (root) id[q] = __popcll(bal & ((1ull << lane) - 1ull));
  }
  __syncthreads();
  for (int k = 0; k < kTileN / 64; ++k) roots += (int)link[k];
  if (tid == 0) nroots[(size_t)a * gridDim.x + blockIdx.x] = roots;
  int mine = 0;
#pragma unroll
  for (int i = 0; i < kTileE; ++i) {
    const int q = tid + i * kTileThreads, x = q % kTile, y = q / kTile;
    if (x >= w || y >= h) continue;
    const size_t p = base + (size_t)(Y0 + y) * C + X0 + x;
    const int c = cmp[q];
    int k = id[c];
    for (int v = 0; v < c / 64; ++v) k += (int)link[v];
    comp[p] = (unsigned short)k;
    inc[p] = linc[q];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      u64 pr;
      int o;
      if (edge(x, y, s, pr, o) && (o < 0 || cmp[o] != c)) ++mine;
    }
  }
  int at = mine ? atomicAdd(&cnt[0], mine) : 0;
  __syncthreads();
  if (tid == 0) ebase = atomicAdd(nedges + a, cnt[0]);
  __syncthreads();
  u64* ed = edges + (size_t)a * 2 * nh + ebase;
#pragma unroll
  for (int i = 0; i < kTileE; ++i) {
    const int q = tid + i * kTileThreads, x = q % kTile, y = q / kTile;
    if (x >= w || y >= h) continue;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      u64 pr;
      int o;
      if (edge(x, y, s, pr, o) && (o < 0 || cmp[o] != cmp[q])) ed[at++] = pr;
    }
  }
}

// clears the angles' edge counters ahead of the tile kernel
__global__ void k_herr_clear(int* __restrict__ nedges, int A) {
  const int a = blockIdx.x * 256 + threadIdx.x;
  if (a < A) nedges[a] = 0;
}

constexpr int kFinThreads = 1024;
constexpr int kFinN = 2048;  // components whose arrays fit in LDS

// Barrier after which the block sees each other's stores to the arrays: LDS
// needs the barrier alone, global arrays (whose minima are atomics at the L2)
// a fence as well.
template <bool LDS>
__device__ __forceinline__ void fin_sync() {
  if (!LDS) __threadfence();
  __syncthreads();
}

// The rounds of one angle over nr components: cur[i] = (current root, increment
// relative to it) of component i; ids: the components of each edge's ends.
template <bool LDS>
__device__ __forceinline__ void fin_rounds(int nr, int ne, int C, const u64* __restrict__ ed,
                                           const int2* ids,
                                           const unsigned short* __restrict__ comp,
                                           const int* __restrict__ inc,
                                           const float* __restrict__ ph,
                                           const int* tbase, u64* cur, u64* best,
                                           u64* link) {
  constexpr int SC = LDS ? kBlockScope : __HIP_MEMORY_SCOPE_AGENT;
  const int nt = (C + kTile - 1) / kTile;
  for (int i = threadIdx.x; i < nr; i += kFinThreads) bor_store<SC>(cur + i, bor_pack(i, 0));
  while (true) {  // each round but the last leaves at most half the components
    for (int i = threadIdx.x; i < nr; i += kFinThreads) bor_store<SC>(best + i, kNoEdge);
    fin_sync<LDS>();
    bool found = false;
    for (int i = threadIdx.x; i < ne; i += kFinThreads) {
      const int2 id = ids[i];
      const int r1 = bor_up(bor_load<SC>(cur + id.x)), r2 = bor_up(bor_load<SC>(cur + id.y));
      if (r1 == r2) continue;
      found = true;
      const u64 p = ed[i];
      bor_offer<SC>(best + r1, p);
      bor_offer<SC>(best + r2, p);
    }
    fin_sync<LDS>();
    if (!__syncthreads_or(found)) break;
    for (int i = threadIdx.x; i < nr; i += kFinThreads) {
      if (bor_up(bor_load<SC>(cur + i)) != i) continue;  // not a root
      const u64 b = bor_load<SC>(best + i);
      u64 v = bor_pack(i, 0);
      if (b != kNoEdge) {
        int p1, p2;
        herr_edge((int)(unsigned)b, C, p1, p2);
        auto at = [&](int p) {
          const int y = p / C, x = p - y * C;
          return bor_load<SC>(cur + tbase[(y / kTile) * nt + x / kTile] + comp[p]);
        };
        const u64 c1 = at(p1), c2 = at(p2);
        const int r1 = bor_up(c1), other = r1 == i ? bor_up(c2) : r1;
        // both ends took this edge: the lower root stays
        if (!(bor_load<SC>(best + other) == b && i < other)) {
          const int i1 = inc[p1] + bor_off(c1), i2 = inc[p2] + bor_off(c2);
          const int wr = herr_wrapcount(ph[p1], ph[p2]);
          v = bor_pack(other, r1 == i ? i2 - i1 + wr : i1 - wr - i2);
        }
      }
      bor_store<SC>(link + i, v);
    }
    fin_sync<LDS>();
    for (int i = threadIdx.x; i < nr; i += kFinThreads)
      if (bor_up(bor_load<SC>(cur + i)) == i) bor_jump<SC>(link, i);
    fin_sync<LDS>();
    for (int i = threadIdx.x; i < nr; i += kFinThreads) {
      const u64 c = bor_load<SC>(cur + i), v = bor_load<SC>(link + bor_up(c));
      bor_store<SC>(cur + i, bor_pack(bor_up(v), bor_off(c) + bor_off(v)));
    }
    fin_sync<LDS>();
  }
}

// One block per angle: the components' numbers in the angle (tbase: the first of
// each tile), the edges' components, the rounds, and each component's
// increment relative to the last root. arr: 3 arrays of C^2 per angle for
// angles with more than kFinN components.
__global__ void __launch_bounds__(kFinThreads)
k_herr_finish(int C, const int* __restrict__ nroots, const u64* __restrict__ edges,
              const int* __restrict__ nedges, const unsigned short* __restrict__ comp,
              const int* __restrict__ inc, const float* __restrict__ ph, int2* ids,
              int* tbase, int* __restrict__ off, u64* arr) {
  __shared__ u64 lcur[kFinN], lbest[kFinN], llink[kFinN];
  __shared__ int wsum[kFinThreads / 64];
  const int a = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nt = (C + kTile - 1) / kTile, tiles = nt * nt, n = C * C, m = 2 * C * (C - 1);
  int* tb = tbase + (size_t)a * tiles;
  int nr = 0;
  for (int t0 = 0; t0 < tiles; t0 += kFinThreads) {  // exclusive sums of the tiles' counts
    const int t = t0 + tid;
    const int c = t < tiles ? nroots[(size_t)a * tiles + t] : 0;
    int s = c;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(s, o, 64);
      if (lane >= o) s += v;
    }
    if (lane == 63) wsum[wave] = s;
    __syncthreads();
    int before = nr, all = nr;
    for (int k = 0; k < kFinThreads / 64; ++k) {
      if (k == wave) before = all;
      all += wsum[k];
    }
    if (t < tiles) tb[t] = before + s - c;
    nr = all;
    __syncthreads();
  }
  __threadfence_block();
  __syncthreads();
  const u64* ed = edges + (size_t)a * m;
  int2* id = ids + (size_t)a * m;
  const unsigned short* cp = comp + (size_t)a * n;
  const int* ic = inc + (size_t)a * n;
  const float* pa = ph + (size_t)a * n;
  const int ne = nedges[a];
  for (int i = tid; i < ne; i += kFinThreads) {  // read back by this thread alone
    int p1, p2;
    herr_edge((int)(unsigned)ed[i], C, p1, p2);
    auto at = [&](int p) {
      const int y = p / C, x = p - y * C;
      return tb[(y / kTile) * nt + x / kTile] + (int)cp[p];
    };
    id[i] = make_int2(at(p1), at(p2));
  }
  u64* cur;
  if (nr <= kFinN) {  // uniform
    fin_rounds<true>(nr, ne, C, ed, id, cp, ic, pa, tb, lcur, lbest, llink);
    for (int i = tid; i < nr; i += kFinThreads) off[(size_t)a * n + i] = bor_off(lcur[i]);
  } else {
    cur = arr + (size_t)a * 3 * n;
    fin_rounds<false>(nr, ne, C, ed, id, cp, ic, pa, tb, cur, cur + n, cur + 2 * (size_t)n);
    for (int i = tid; i < nr; i += kFinThreads)
      off[(size_t)a * n + i] = bor_off(bor_load<__HIP_MEMORY_SCOPE_AGENT>(cur + i));
  }
}

// unwrapImage (:555-566): value + TWOPI * increment in float
__global__ void __launch_bounds__(256)
k_herr_out(int C, const float* __restrict__ ph, const unsigned short* __restrict__ comp,
           const int* __restrict__ inc, const int* __restrict__ tbase,
           const int* __restrict__ off, float* __restrict__ phu) {
  const int a = blockIdx.y, p = blockIdx.x * 256 + threadIdx.x;
  const int n = C * C;
  if (p >= n) return;
  const int nt = (C + kTile - 1) / kTile, y = p / C, x = p - y * C;
  const size_t i = (size_t)a * n + p;
  const int c = tbase[(size_t)a * nt * nt + (y / kTile) * nt + x / kTile] + comp[i];
  phu[i] = ph[i] + kHerrTwoPi * (float)(inc[i] + off[(size_t)a * n + c]);
}

// the scratch arrays of A angles, in one walk for their sizes and addresses
struct HerrScratch {
  float *ph, *key, *top;
  unsigned short* comp;
  int *inc, *off, *nroots, *tbase, *nedges;
  u64 *edges, *arr;
  int2* ids;
  size_t bytes;
};

static SortLevels herr_levels(int C, int* d0) {
  SortLevels L{};
  L.s[0] = 2 * C * (C - 1);
  int depth = 0;
  while (depth < kMaxDepth && L.s[depth] >= 2) {
    L.s[depth + 1] = L.s[depth] / 2;
    ++depth;
  }
  L.deepest = depth - 1;
  *d0 = 0;
  while (L.s[*d0] > kTailN) ++*d0;
  return L;
}

static HerrScratch herr_scratch(void* base, int C, size_t A) {
  const size_t n = (size_t)C * C, m = 2 * (size_t)C * (C - 1);
  const size_t nt = (C + kTile - 1) / kTile, tiles = nt * nt;
  int d0;
  herr_levels(C, &d0);
  HerrScratch h{};
  size_t at = 0;
  auto take = [&](auto*& p, size_t count) {
    p = (std::decay_t<decltype(p)>)((char*)base + at);
    at += (count * sizeof(*p) + 255) / 256 * 256;
  };
  take(h.ph, A * n);
  take(h.key, A * m);
  take(h.top, A << d0);
  take(h.comp, A * n);
  take(h.inc, A * n);
  take(h.off, A * n);
  take(h.nroots, A * tiles);
  take(h.tbase, A * tiles);
  take(h.nedges, A);
  take(h.edges, A * m);
  take(h.ids, A * m);
  take(h.arr, 3 * A * n);
  h.bytes = at;
  return h;
}

size_t herraez_scratch_bytes(int C, int A) {
  return herr_scratch(nullptr, C, A > 0 ? A : 1).bytes;
}

hipError_t launch_herraez(int C, const float2* iu, int A, const float* border, void* scratch,
                          float* phu, hipStream_t s) {
  if (A <= 0) return hipSuccess;
  if (C < 3) return hipErrorInvalidValue;
  const HerrScratch h = herr_scratch(scratch, C, A);
  const int n = C * C, m = 2 * C * (C - 1), nt = (C + kTile - 1) / kTile;
  int d0;
  const SortLevels L = herr_levels(C, &d0);
  {
    Timed tm("herraez_edges", s);
    hipLaunchKernelGGL(k_herr_edges, dim3((C + kEx - 1) / kEx, (C + kEy - 1) / kEy, A),
                       dim3(kEx * kEy), 0, s, iu, C, border, h.ph, h.key);
    hipLaunchKernelGGL(k_herr_tails, dim3(1u << d0, A), dim3(kTailThreads), 0, s, h.key, m, L, d0,
                       h.top);
    if (d0 > 0)
      hipLaunchKernelGGL(k_herr_tails_top, dim3(A), dim3(kTailThreads), 0, s, h.key, m, L, d0,
                         h.top);
  }
  Timed tm("herraez_tree", s);
  hipLaunchKernelGGL(k_herr_clear, dim3((A + 255) / 256), dim3(256), 0, s, h.nedges, A);
  hipLaunchKernelGGL(k_herr_tile, dim3(nt * nt, A), dim3(kTileThreads), 0, s, h.key, h.ph, C,
                     h.comp, h.inc, h.nroots, h.edges, h.nedges);
  hipLaunchKernelGGL(k_herr_finish, dim3(A), dim3(kFinThreads), 0, s, C, h.nroots, h.edges,
                     h.nedges, h.comp, h.inc, h.ph, h.ids, h.tbase, h.off, h.arr);
  hipLaunchKernelGGL(k_herr_out, dim3((n + 255) / 256, A), dim3(256), 0, s, C, h.ph, h.comp, h.inc,
                     h.tbase, h.off, phu);
  return hipGetLastError();
}

}  // namespace mtd
