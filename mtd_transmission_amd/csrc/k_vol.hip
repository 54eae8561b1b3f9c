// Volume stage: deterministic Ewald-cap accumulation and the finalisation to
// a refractive-index volume.
//
// Accumulation (retroPropag_Born, Reconstruction/src/fonctions.cpp:875-935)
// is restated as a gather. For a lateral voxel column q = (X - V/2, Y - V/2),
// angle a contributes at most one hit: at pupil pixel fd = q + fm0(a), at
// height z = round(h(|fd|^2) - fzm0(a)) + V/2 with h(r2) = sqrt(R^2 - r2),
// provided fd lies in the [-NXMAX, NXMAX)^2 crop, |fd|^2 < coef*NXMAX^2 and the
// angle is not skipped. Each thread owns one column of a (column tile, height
// window) work item and walks the angles in order, so every voxel receives
// its hits in the reference's angle order: this is the sort-by-voxel of the
// accumulation done analytically (the scatter map is invertible per angle),
// and the sum is deterministic and equal to the sequential FP32 sum. Partial
// columns live in LDS; every voxel of the V^3 spectrum and count volume is
// written exactly once (zeros included), so no clearing pass is needed.
// Banded mode (the fused plain method): hits of all angles lie in a height
// band about V/2 of half-width about R - sqrt(R^2 - NXMAX^2) (a third of the
// volume for the usual geometry); only the windows meeting it are written and
// the inverse transform reads nothing else.
//
// Finalisation (Reconstruction/main.cpp:243-352): divide by counts (0 -> 1),
// backward 3-D FFT with both fftshift3D folded into (-1)^(x+y+z) sign flips,
// times delta_f^3 and -1/(2 n0 kv^2), split into index and absorption.
#include <algorithm>
#include <optional>

#include "dft.hpp"
#include "gen_fft.hpp"
#include "internal.hpp"
#include "passes.hpp"

namespace mtd {

// C round(): halves away from zero, exact.
__device__ __forceinline__ double round_away(double x) {
  const double t = trunc(x);
  return (fabs(x - t) >= 0.5) ? t + copysign(1.0, x) : t;
}

__device__ __forceinline__ AngleGeo angle_geo(const int* __restrict__ posx,
                                             const int* __restrict__ posy, int a, int nx,
                                             double R2, const double* __restrict__ htab,
                                             int r2tab) {
  AngleGeo g;
  g.fx = posx[a] - nx;
  g.fy = posy[a] - nx;
  const int r2 = g.fx * g.fx + g.fy * g.fy;
  const double fz2 = (R2 - (double)(g.fx * g.fx)) - (double)(g.fy * g.fy);
  g.skip = round_away(fz2) < 0.0;
  g.pad = 0;
  g.fz = (!g.skip && r2 < r2tab) ? htab[r2] : 0.0;
  return g;
}

__global__ void k_angle_geo(const int* __restrict__ posx,
                            const int* __restrict__ posy, int A, int nx,
                            double R2, const double* __restrict__ htab,
                            int r2tab, AngleGeo* __restrict__ ageo) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a < A) ageo[a] = angle_geo(posx, posy, a, nx, R2, htab, r2tab);
}

struct GatherArgs {
  const float2* spec;   // [A][C][C]
  int frame_pos;        // 1: spectra in the +posSpec frame, 0: unshifted
  const AngleGeo* ageo;
  int A, C, nx, V;
  const double* htab;   // h(r2) = sqrt(R^2 - r2)
  const float* beta;    // per r2: ((k0/PI)*(-2PI)) * h/R
  int r2max;            // largest r2 inside the pupil
  float2* vol;
  int32_t* cnt;
  uint32_t specb;       // bytes of all spectra if below 2 GiB, else 0
};

constexpr int GT = 16;  // tile side (columns per block = 256)

// ---------------------------------------------------------------------------
// Windowed gather. A prepass lists, per 16x16 column tile and in angle order,
// the angles whose pupil disc touches the tile, with a conservative height
// range derived from the tile box's nearest and farthest pupil radii (h is
// decreasing in r^2 and round is monotonic). The main kernel gives each block
// one (tile, ZW-height window); a wave tests 64 list entries against the
// window at once and takes the overlapping ones in angle order, KB at a
// time. Each column's exact hit height is computed in registers, and only
// the hits' spectrum values are loaded (a miss's buffer-load offset is out
// of range, which fetches nothing). Near the lateral origin nearly every
// angle hits the same few voxels, and those sums are serial by definition
// (angle order): the loads of KB entries are issued together so that only
// the additions stay serial, and those tiles are dispatched first (tiles in
// order of distance from the lateral origin).
// ---------------------------------------------------------------------------
struct TileEntry {
  int a;
  int zpack;  // zlo | zhi << 16, absolute heights
  int fxy;    // fxm0 & 0xffff | fym0 << 16 (signed 16-bit each)
  float fz;   // fzm0 rounded to float (the registers' height path)
};

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// h(r2) = sqrt(R^2 - r2) for 0 <= r2 <= R^2: IEEE sqrt of the same exact
// double, so the host height table's value bit for bit
__device__ __forceinline__ double height(double R2, int r2) { return sqrt(R2 - (double)r2); }

// Does angle a's pupil disc touch the 16x16 column tile at (qx0, qy0)? If so,
// the nearest and farthest pupil radii^2 of the tile box (the farthest
// clamped to the pupil edge).
__device__ __forceinline__ bool tile_touch(const GatherArgs& g, const AngleGeo& ag, int qx0,
                                           int qy0, int& dmin, int& dmax) {
  if (ag.skip) return false;
  const int cxl = max(qx0 + ag.fx, -g.nx), cxh = min(qx0 + GT - 1 + ag.fx, g.nx - 1);
  const int cyl = max(qy0 + ag.fy, -g.nx), cyh = min(qy0 + GT - 1 + ag.fy, g.nx - 1);
  if (cxl > cxh || cyl > cyh) return false;
  const int mx = cxl > 0 ? cxl : (cxh < 0 ? -cxh : 0);
  const int my = cyl > 0 ? cyl : (cyh < 0 ? -cyh : 0);
  const int Mx = max(abs(cxl), abs(cxh)), My = max(abs(cyl), abs(cyh));
  dmin = mx * mx + my * my;
  dmax = min(Mx * Mx + My * My, g.r2max);
  return dmin <= g.r2max;
}

// Prepass: one wave per 16x16 column tile lists, in angle order, the angles
// whose pupil disc touches the tile, 64 angles per ballot, with a
// conservative height range from the tile box's nearest and farthest pupil
// radii (h decreases with r^2, round is monotonic; FP64 heights and
// round-half-away, as the reference), and writes the tile's entry count and
// height range.
__global__ void __launch_bounds__(64)
k_tile_angles(GatherArgs g, int ntx, TileEntry* __restrict__ list, int4* __restrict__ tinfo) {
  const int tile = blockIdx.x, lane = threadIdx.x;
  const int qx0 = (tile % ntx) * GT - g.V / 2, qy0 = (tile / ntx) * GT - g.V / 2;
  const double R2 = g.htab[0] * g.htab[0];  // h(0) = R, an integer: exact
  TileEntry* lst = list + (size_t)tile * g.A;
  int off = 0, zmin = 0x7fffffff, zmax = -1;
  for (int a0 = 0; a0 < g.A; a0 += 64) {
    const int a = a0 + lane;
    bool act = false;
    int zl = 0, zh = 0;
    AngleGeo ag{};
    if (a < g.A) {
      ag = g.ageo[a];
      int dmin, dmax;
      if (tile_touch(g, ag, qx0, qy0, dmin, dmax)) {
        zl = clampi((int)round_away(height(R2, dmax) - ag.fz) + g.V / 2, 0, g.V - 1);
        zh = clampi((int)round_away(height(R2, dmin) - ag.fz) + g.V / 2, 0, g.V - 1);
        act = true;
        zmin = min(zmin, zl);
        zmax = max(zmax, zh);
      }
    }
    const unsigned long long bal = __ballot(act);
    if (act) {
      const int p = __popcll(bal & ((1ull << lane) - 1ull));
      lst[off + p] = TileEntry{a, zl | (zh << 16), (ag.fx & 0xffff) | (ag.fy << 16), (float)ag.fz};
    }
    off += __popcll(bal);
  }
  for (int o = 32; o > 0; o >>= 1) {
    zmin = min(zmin, __shfl_xor(zmin, o, 64));
    zmax = max(zmax, __shfl_xor(zmax, o, 64));
  }
  if (lane == 0) tinfo[tile] = make_int4(off, zmin, zmax, 0);
}

// 8 bytes at byte offset off + uni (uni uniform) from base; an offset past
// nbytes returns zeros without a memory access (a buffer load's range check)
__device__ __forceinline__ float2 load_or_zero(const float2* base, uint32_t nbytes, uint32_t off,
                                               uint32_t uni = 0) {
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)nbytes, 0x00020000);
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, (int)uni, 0);
  return make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
}
__device__ __forceinline__ float load_or_zero(const float* base, uint32_t nbytes, uint32_t off) {
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)nbytes, 0x00020000);
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
constexpr uint32_t kMissOffset = 0x80000000u;  // past every spectrum (< 2^31 bytes)

// one column's fixed data for the gather's hit tests; lengths in FP32 are exact
// integers (R^2 < 2^24: rayon is below half the volume side)
struct GatherCol {
  float qx, qy;    // lateral column (voxel - V/2)
  int zbase;       // the window's first height - V/2
  uint32_t fixed;  // byte offset of the column's element in the unshifted frame
  float R2f;       // R^2
  float xmin;      // R^2 - r2max: the smallest R^2 - |fd|^2 inside the pupil
  float half;      // 1/2 - 4 ulp(R) (see gather_fill)
  bool square;     // the pupil reaches past the crop's square: test that too
};

// A batch of KB list entries: per entry the window slot of this column's hit
// (ZW, a slot of its own, for a miss), the angle and the spectrum element's
// byte offset (kMissOffset for a miss: such a load fetches nothing and gives
// zeros) and, after issue(), the loaded value (and beta when !PRE).
template <int KB>
struct GBatch {
  int kv[KB], ea[KB];
  uint32_t el[KB], br[KB];
  float2 sp[KB];
  float b[KB];
  template <bool PRE>
  __device__ __forceinline__ void issue(const GatherArgs& g, size_t C2, uint32_t C2b) {
    // spectra below 2 GiB in all: one buffer view, the angle in the scalar
    // offset (a view per angle costs a dozen scalar instructions a load)
    if (g.specb) {
#pragma unroll
      for (int t = 0; t < KB; ++t)
        sp[t] = load_or_zero(g.spec, g.specb, el[t], (uint32_t)ea[t] * C2b);
    } else {
#pragma unroll
      for (int t = 0; t < KB; ++t) sp[t] = load_or_zero(g.spec + (size_t)ea[t] * C2, C2b, el[t]);
    }
    if constexpr (!PRE) {
#pragma unroll
      for (int t = 0; t < KB; ++t)
        b[t] = load_or_zero(g.beta, (uint32_t)(g.r2max + 1) * 4u, br[t]);
    }
    // keep the loads ahead of what follows (the other batch's sums): the
    // scheduler would otherwise sink them below those independent LDS ops
    __builtin_amdgcn_sched_barrier(0);
  }
  // The sums, four entries at a time: the four slots' old values are read
  // together, an entry whose slot an earlier one of the four also hits takes
  // that one's new sum instead (each voxel's sum still takes its hits in
  // angle order), and the new sums are written in order. One wait for LDS per
  // four entries instead of one per hit; groups without a hit in the wave
  // are skipped. Counts: one LDS add per entry, two 16-bit counts a word.
  template <bool PRE, bool COUNT, int ZW>
  __device__ __forceinline__ void apply(float2 (*acc)[256], unsigned (*cn)[256], int tid) const {
#pragma clang fp contract(off)
#pragma unroll
    for (int q = 0; q < KB; q += 4) {
      if (!__any((kv[q] < ZW) | (kv[q + 1] < ZW) | (kv[q + 2] < ZW) | (kv[q + 3] < ZW))) continue;
      float2 s[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = acc[kv[q + i]][tid];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < i; ++j)
          if (kv[q + i] == kv[q + j]) s[i] = s[j];
        // value (-b Si, b Sr)
        const float pim = PRE ? sp[q + i].y : b[q + i] * sp[q + i].y;
        const float pre = PRE ? sp[q + i].x : b[q + i] * sp[q + i].x;
        s[i].x = s[i].x + -pim;
        s[i].y = s[i].y + pre;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[kv[q + i]][tid] = s[i];
        if constexpr (COUNT)
          __hip_atomic_fetch_add(&cn[kv[q + i] >> 1][tid], 1u << ((kv[q + i] & 1) * 16),
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      }
    }
  }
};

// Entries i0 .. i0 + KB - 1 of a segment's compacted list (padded with entries
// that never hit), read from LDS at a uniform address (a broadcast), all of
// them first. Height offset of a hit: round(h(r2) - fz), FP64 and half away from
// zero in the reference. Here in FP32: R^2 - r2 is an exact float; the
// hardware square root (v_sqrt_f32, within 1 ulp, not correctly rounded) of
// it is within 1 ulp(R), fz is rounded once and the difference is rounded
// once, each within half an ulp of R (h, fz and |h - fz| are at most R): the
// FP32 difference is within 2 ulp(R) of the FP64 one. Wherever it lies within
// 1/2 - 4 ulp(R) of an integer both round to that integer; the rest (a lane in
// some ten thousands) takes the FP64 path, after the batch.
template <int ZW, bool PRE, bool POSF, int KB>
__device__ __forceinline__ void gather_fill(GBatch<KB>& B, const int4* seg, int i0,
                                            const GatherArgs& g, const GatherCol& c) {
  int4 en[KB];
  float x[KB];
  int dz[KB];
  bool in[KB];
  float worst = 0.f;
#pragma unroll
  for (int t = 0; t < KB; ++t) en[t] = seg[i0 + t];
#pragma unroll
  for (int t = 0; t < KB; ++t) {
    const float fdx = c.qx + __int_as_float(en[t].y), fdy = c.qy + __int_as_float(en[t].z);
    x[t] = __builtin_fmaf(-fdy, fdy, __builtin_fmaf(-fdx, fdx, c.R2f));  // R^2 - |fd|^2
    in[t] = x[t] >= c.xmin;
    if (c.square) {  // uniform
      const float nx = (float)g.nx;
      in[t] = in[t] && fdx >= -nx && fdx < nx && fdy >= -nx && fdy < nx;
    }
    const float d = __builtin_amdgcn_sqrtf(fmaxf(x[t], 0.f)) - __int_as_float(en[t].w);
    const float r = __builtin_rintf(d);
    worst = fmaxf(worst, fabsf(d - r));
    dz[t] = (int)r;
    B.ea[t] = __builtin_amdgcn_readfirstlane(en[t].x);
    if constexpr (POSF)
      B.el[t] = (uint32_t)__builtin_fmaf(fdy + (float)g.nx, (float)g.C, fdx + (float)g.nx) * 8u;
  }
  if (worst > c.half) {
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      const float d = __builtin_amdgcn_sqrtf(fmaxf(x[t], 0.f)) - __int_as_float(en[t].w);
      if (in[t] && fabsf(d - __builtin_rintf(d)) > c.half)
        dz[t] = (int)round_away(sqrt((double)x[t]) - g.ageo[B.ea[t]].fz);
    }
  }
#pragma unroll
  for (int t = 0; t < KB; ++t) {
    const int k = dz[t] - c.zbase;
    const bool hit = in[t] && (unsigned)k < (unsigned)ZW;
    B.kv[t] = hit ? k : ZW;
    B.el[t] = !hit ? kMissOffset : POSF ? B.el[t] : c.fixed;
    if constexpr (!PRE) B.br[t] = !hit ? kMissOffset : (uint32_t)(c.R2f - x[t]) * 4u;
  }
}

constexpr int kGatherSeg = 256;  // list entries tested (and compacted) per segment

// flags: bit0 = normalise (divide by counts, 0 -> 1) and apply the centring
// sign (-1)^(x+y+z) of the 3-D inverse FFT; counts are then not written.
// bit2 = the plain sums with that centring sign, no counts (the adjoint of
// the Born forward model; COUNT false).
// PRE: the spectra are already multiplied by the Ewald factor beta of their
// pupil pixel (the same FP32 product), so beta is not looked up here.
// POSF: spectra in the +posSpec frame. KB: list entries whose loads are issued
// together.
//
// What bounds it: the tiles at the lateral origin, which nearly every angle
// hits and whose sums are serial. Per entry and wave about 20 vector
// instructions, and one LDS round trip per four entries; before, a branch per
// entry (the rare FP64 height) and one per hit kept every list read and every
// sum's LDS round trip exposed. Those tiles also raise their waves' issue
// priority over the short lists' on the same SIMD. Gather alone, before and
// now: 100 angles into 256^3 44 -> 30 us, 600 into 512^3 243 -> 192, 200 into
// 1024^3 925 -> 807, the solver's adjoint of 400 into 256^3 125 -> 71 (a buffer
// view per angle instead of one with a scalar offset: 31, 197, 812, 76; batches
// of 16: 35, 243, 977, 81).
template <int ZW, bool PRE, bool POSF, bool COUNT, int KB>
__global__ void __launch_bounds__(256)
k_gather_win(GatherArgs g, int ntx, int w0, int nwin, int items, const int* __restrict__ order,
             const TileEntry* __restrict__ list, const int4* __restrict__ tinfo, int flags,
             const int2* __restrict__ band) {
  // The sums must be the sequential FP32 sums of the reference: no fused
  // multiply-add. The pragma is lexical, so the products and sums are written
  // here as plain operators (HIP's __fmul_rn/__fadd_rn are header functions
  // outside its scope and would still be contracted).
#pragma clang fp contract(off)
  // Blocks are dealt round-robin to the 8 XCDs. Tiles go to the XCDs in
  // order of distance from the lateral origin (order[]: the heaviest first,
  // spread over the XCDs), and the windows of one tile stay on one XCD, in
  // order (they read the same spectrum patches). A bijection when the tile
  // count is a multiple of 8. Windows w0 .. w0 + nwin - 1 are launched.
  int tile, w;
  {
    const int b = blockIdx.x, tiles = items / nwin;
    int rank;
    if (tiles % 8 == 0) {
      const int n = b / 8;
      rank = (n / nwin) * 8 + b % 8;
      w = w0 + n % nwin;
    } else {
      rank = b / nwin;
      w = w0 + b % nwin;
    }
    tile = order[rank];
  }
  const int tid = threadIdx.x;
  const int X = (tile % ntx) * GT + tid % GT, Y = (tile / ntx) * GT + tid / GT;
  const int qx = X - g.V / 2, qy = Y - g.V / 2;
  const size_t plane = (size_t)g.V * g.V;
  const size_t col = (size_t)Y * g.V + X;
  // the last tiles of a volume side that is not a multiple of the tile side
  // hold columns past the volume: they walk the lists like the others (the
  // ballots are per wave) but write nothing
  const bool inb = X < g.V && Y < g.V;
  const int z0 = w * ZW, z1 = min(z0 + ZW, g.V) - 1;
  // heights this block writes: the window, cut to the hit band when the
  // output is banded (no pass reads a plane outside the band)
  int zs0 = z0, zs1 = z1;
  if (band) {
    const int2 b = *band;
    if (z1 < b.x || z0 > b.y) return;
    zs0 = max(z0, b.x);
    zs1 = min(z1, b.y);
  }
  const int4 info = tinfo[tile];
  const bool norm = flags & 1, sgn = flags & 5;
  if (info.x == 0 || z1 < info.y || z0 > info.z) {
    if (inb) {
      for (int z = zs0; z <= zs1; ++z) {
        g.vol[z * plane + col] = make_float2(0.f, 0.f);
        if (COUNT && !sgn) g.cnt[z * plane + col] = 0;
      }
    }
    return;
  }
  if (4 * info.x > 3 * g.A) __builtin_amdgcn_s_setprio(3);
  else if (2 * info.x > g.A) __builtin_amdgcn_s_setprio(2);
  else if (4 * info.x > g.A) __builtin_amdgcn_s_setprio(1);
  // this column's ZW partial sums and hit counts (< 2^16: at most one hit
  // per angle) live in LDS, and a slot for the misses; each thread only
  // touches its own column
  __shared__ float2 acc[ZW + 1][256];
  __shared__ unsigned cn[COUNT ? ZW / 2 + 1 : 1][256];
#pragma unroll
  for (int k = 0; k <= ZW; ++k) acc[k][tid] = make_float2(0.f, 0.f);
  if constexpr (COUNT) {
#pragma unroll
    for (int k = 0; k <= ZW / 2; ++k) cn[k][tid] = 0;
  }
  const TileEntry* lst = list + (size_t)tile * g.A;
  // spectrum element read by this column: the unshifted frame holds it at
  // (qy mod C, qx mod C) for every angle; the +posSpec frame at fd + NXMAX
  const int frow = ((qy % g.C) + g.C) % g.C, fcol = ((qx % g.C) + g.C) % g.C;
  const uint32_t fixed = (uint32_t)(frow * g.C + fcol) * 8u;
  const uint32_t C2b = (uint32_t)g.C * (uint32_t)g.C * 8u;  // bytes per angle
  const size_t C2 = (size_t)g.C * g.C;
  const float Rf = (float)g.htab[0];  // h(0) = R, an integer
  const float R2f = Rf * Rf;
  const GatherCol cg{(float)qx,
                     (float)qy,
                     z0 - g.V / 2,
                     fixed,
                     R2f,
                     R2f - (float)g.r2max,
                     0.5f - ldexpf(1.f, ilogbf(Rf) - 21),
                     g.r2max >= g.nx * g.nx};
  // The tile's list in segments of kGatherSeg entries: each thread tests one
  // entry against the window, the overlapping ones are compacted into LDS in
  // list (angle) order, and every wave takes them KB at a time,
  // software-pipelined two deep: the loads of batch i + 1 are in flight
  // while the sums of batch i are applied (each voxel's sum still takes its
  // hits in angle order). Both batches always issue their KB loads (misses
  // fetch nothing), so the outstanding-load count is the same on every path.
  __shared__ int4 seg[kGatherSeg + 2 * KB];
  __shared__ int wcount[4];
  const int lane = tid & 63, wave = tid >> 6;
  for (int s0 = 0; s0 < info.x; s0 += kGatherSeg) {  // uniform
    __syncthreads();  // the previous segment is consumed
    const int j = s0 + tid;
    bool ov = false;
    TileEntry e{0, 0, 0, 0.f};
    if (j < info.x) {
      e = lst[j];
      const int zl = e.zpack & 0xffff, zh = e.zpack >> 16;
      ov = !(zh < z0 || zl > z1);
    }
    const unsigned long long bal = __ballot(ov);
    if (lane == 0) wcount[wave] = __popcll(bal);
    __syncthreads();
    int base = 0;
#pragma unroll
    for (int w2 = 0; w2 < 4; ++w2) base += w2 < wave ? wcount[w2] : 0;
    const int total = wcount[0] + wcount[1] + wcount[2] + wcount[3];
    if (ov)
      seg[base + __popcll(bal & ((1ull << lane) - 1ull))] =
          make_int4(e.a, __float_as_int((float)(short)(e.fxy & 0xffff)),
                    __float_as_int((float)(e.fxy >> 16)), __float_as_int(e.fz));
    // past the list: entries outside every pupil
    if (tid < 2 * KB) seg[total + tid] = make_int4(0, __float_as_int(1e9f), 0, 0);
    __syncthreads();
    const int nb = (total + KB - 1) / KB;
    GBatch<KB> A, B;
    gather_fill<ZW, PRE, POSF, KB>(A, seg, 0, g, cg);
    A.template issue<PRE>(g, C2, C2b);
    for (int bi = 0; bi < nb; bi += 2) {
      gather_fill<ZW, PRE, POSF, KB>(B, seg, (bi + 1) * KB, g, cg);
      B.template issue<PRE>(g, C2, C2b);
      A.template apply<PRE, COUNT, ZW>(acc, cn, tid);
      if (bi + 1 >= nb) break;
      gather_fill<ZW, PRE, POSF, KB>(A, seg, (bi + 2) * KB, g, cg);
      A.template issue<PRE>(g, C2, C2b);
      B.template apply<PRE, COUNT, ZW>(acc, cn, tid);
    }
  }
  if (!inb) return;
#pragma unroll
  for (int k = 0; k < ZW; ++k) {
    const int z = z0 + k;
    if (z > zs1) break;
    if (z < zs0) continue;
    const float2 s = acc[k][tid];
    const int c = COUNT ? (int)(cn[k >> 1][tid] >> ((k & 1) * 16) & 0xffff) : 0;
    if (sgn) {
      float2 t = s;
      if (COUNT && norm) {
        const float d = (float)(c == 0 ? 1 : c);
        t = make_float2(s.x / d, s.y / d);
      }
      if ((X + Y + z) & 1) { t.x = -t.x; t.y = -t.y; }
      g.vol[z * plane + col] = t;
    } else {
      g.vol[z * plane + col] = s;
      if (COUNT) g.cnt[z * plane + col] = c;
    }
  }
}

hipError_t launch_angle_geo(const int* posx, const int* posy, int A, int nxmax,
                            double R2, const double* htab, int r2tab,
                            AngleGeo* ageo, hipStream_t s) {
  Timed tm("angle_geo", s);
  hipLaunchKernelGGL(k_angle_geo, dim3((A + 127) / 128), dim3(128), 0, s, posx,
                     posy, A, nxmax, R2, htab, r2tab, ageo);
  return hipGetLastError();
}

// The angle table and the hit band in one launch: a single block, since a launch
// costs more than the angles (600 angles: 4.7 us each for the two, a call on
// small volumes has about 15 launches).
constexpr int kGeoThreads = 1024;
__global__ void __launch_bounds__(kGeoThreads)
k_geo_band(const int* __restrict__ posx, const int* __restrict__ posy, int A, int nx, double R2,
           const double* __restrict__ htab, int r2tab, AngleGeo* __restrict__ ageo, int V,
           int r2max, int2* __restrict__ band) {
  __shared__ int2 red[kGeoThreads / 64];
  const int tid = threadIdx.x;
  int lo = 0x7fffffff, hi = -0x7fffffff;
  const double rim = htab[r2max], top = htab[0];
  for (int a = tid; a < A; a += kGeoThreads) {
    const AngleGeo ag = angle_geo(posx, posy, a, nx, R2, htab, r2tab);
    ageo[a] = ag;
    if (ag.skip) continue;
    // hits of angle a lie between the heights at the pupil's rim and centre
    lo = min(lo, (int)round_away(rim - ag.fz) + V / 2);
    hi = max(hi, (int)round_away(top - ag.fz) + V / 2);
  }
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o, 64));
    hi = max(hi, __shfl_xor(hi, o, 64));
  }
  if (tid % 64 == 0) red[tid / 64] = make_int2(lo, hi);
  __syncthreads();
  if (tid) return;
  for (int w = 1; w < kGeoThreads / 64; ++w) {
    lo = min(lo, red[w].x);
    hi = max(hi, red[w].y);
  }
  lo = max(lo, 0);
  hi = min(hi, V - 1);
  band[0] = lo <= hi ? make_int2(lo, hi) : make_int2(1, 0);
}

hipError_t launch_geo_band(const int* posx, const int* posy, int A, int nxmax, double R2,
                           const double* htab, int r2tab, AngleGeo* ageo, int V, int r2max,
                           int2* band, hipStream_t s) {
  Timed tm("ewald_band", s);
  hipLaunchKernelGGL(k_geo_band, dim3(1), dim3(kGeoThreads), 0, s, posx, posy, A, nxmax, R2, htab,
                     r2tab, ageo, V, r2max, band);
  return hipGetLastError();
}

// zeros over planes [0, z0) and [z1, V) of the spectrum and counts, 16 bytes a
// thread (planes are multiples of 32 and 16 bytes: V is even)
__global__ void __launch_bounds__(256)
k_fill_planes(float2* __restrict__ vol, int32_t* __restrict__ cnt, int V, int z0, int z1) {
  const size_t plane = (size_t)V * V, planes = (size_t)(z0 + V - z1);
  const size_t nv = planes * plane / 2, nc = planes * plane / 4;  // 16-byte words
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  const uint4 zero = make_uint4(0, 0, 0, 0);
  if (t < nv) {
    const size_t low = z0 * plane / 2;
    ((uint4*)vol)[t < low ? t : t - low + z1 * plane / 2] = zero;
  } else if (t - nv < nc) {
    const size_t i = t - nv, low = z0 * plane / 4;
    ((uint4*)cnt)[i < low ? i : i - low + z1 * plane / 4] = zero;
  }
}

// Spectrum and counts that the fill takes a part of: beyond the 256 MiB of the last
// cache. What stays in it the gather writes beside its sums in one launch (A angles,
// gather alone / with the fill, us: 256^3 A 30 33 / 43, A 400 89 / 105; 288^3 A 60 53 / 63, A 400
// 146 / 144; 304^3 A 60 94 / 84, A 400 181 / 168; 320^3 A 1 112 / 93).
constexpr size_t kFillOver = 288u << 20;
// the windowed gather with height windows of ZW voxels (LDS: 10 B per
// voxel of the 256 x ZW block, 8 without counts) and batches of KB list entries
template <int ZW, int KB>
static hipError_t gather_windows(const GatherArgs& g, int ntx, int tiles, const int* order,
                                 const TileEntry* list, const int4* tinfo, int flags,
                                 const int2* band, int zlo, int zhi, hipStream_t s) {
  const int V = g.V;
  // only the windows that can meet the hit band are launched (the exact band
  // is only known on the device); an output without a band gets its other
  // planes from a fill, whose whole lines beat the gather's 64- and 128-byte
  // pieces: 400 angles into 512^3, 503 -> 397 us
  int w0 = std::max(zlo, 0) / ZW, w1 = std::min(zhi, V - 1) / ZW;
  if (!band) {
    const bool al = ((uintptr_t)g.vol | (g.cnt ? (uintptr_t)g.cnt : 0)) % 16 == 0;
    if (g.cnt && al && (size_t)V * V * V * 12 > kFillOver) {
      const int z1 = std::min((w1 + 1) * ZW, V);
      const size_t words = (size_t)(w0 * ZW + V - z1) * V * V / 4 * 3;
      if (words) {
        Timed tm("ewald_fill", s);
        hipLaunchKernelGGL(k_fill_planes, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s,
                           g.vol, g.cnt, V, w0 * ZW, z1);
      }
    } else {
      w0 = 0;
      w1 = (V + ZW - 1) / ZW - 1;
    }
  }
  const int nwin = w1 - w0 + 1, items = tiles * nwin;
  Timed tm("ewald_gather", s);
#define MTD_GL(PRE, POSF, COUNT)                                                              \
  hipLaunchKernelGGL((k_gather_win<ZW, PRE, POSF, COUNT, KB>), dim3(items), dim3(256), 0, s, g, \
                     ntx, w0, nwin, items, order, list, tinfo, flags, band)
  const bool pre = flags & 2, count = !(flags & 4);
  if (!g.frame_pos) {
    // unshifted spectra come from the forward column pass, pre-weighted
    if (!pre || !count) return hipErrorInvalidValue;
    MTD_GL(true, false, true);
  } else if (count) {
    if (pre) return hipErrorInvalidValue;
    MTD_GL(false, true, true);
  } else if (pre) {
    MTD_GL(true, true, false);
  } else {
    MTD_GL(false, true, false);
  }
#undef MTD_GL
  return hipGetLastError();
}

bool gather_window_supported(int zw) { return zw == 8 || zw == 16 || zw == 24; }

// scratch: [tiles][A] entries | [tiles] info
static void gather_scratch_split(void* scratch, int tiles, int A, TileEntry** list, int4** tinfo) {
  const size_t nA = (size_t)(A > 0 ? A : 1);
  *list = (TileEntry*)scratch;
  *tinfo = (int4*)((char*)scratch + (size_t)tiles * nA * sizeof(TileEntry));
}

static hipError_t tile_prepass(const GatherArgs& g, int ntx, int tiles, TileEntry* list,
                               int4* tinfo, hipStream_t s) {
  Timed tm("ewald_tiles", s);
  hipLaunchKernelGGL(k_tile_angles, dim3(tiles), dim3(64), 0, s, g, ntx, list, tinfo);
  return hipGetLastError();
}

hipError_t launch_gather(const float2* spec, int frame_pos, const AngleGeo* ageo, int A, int C,
                         int nxmax, int V, const double* htab, const float* beta, int r2max,
                         float2* vol, int32_t* cnt, void* scratch, const int* order, int flags,
                         const int2* band, int zlo, int zhi, bool prepass, int zw, int kb,
                         hipStream_t s) {
  // spectra below 2 GiB; R < V/2 with R^2 < 2^24, C^2 <= 2^24 (exact in FP32)
  if (C > 4096 || V > 8192) return hipErrorInvalidValue;
  const size_t specb = (size_t)std::max(A, 1) * C * C * sizeof(float2);
  GatherArgs g{spec, frame_pos, ageo, A, C, nxmax, V, htab, beta, r2max, vol, cnt,
               specb < ((size_t)1 << 31) ? (uint32_t)specb : 0u};
  const int ntx = (V + GT - 1) / GT, tiles = ntx * ntx;
  TileEntry* list;
  int4* tinfo;
  gather_scratch_split(scratch, tiles, A, &list, &tinfo);
  if (prepass) {
    const hipError_t e = tile_prepass(g, ntx, tiles, list, tinfo, s);
    if (e != hipSuccess) return e;
  }
#define MTD_GW(ZW, KB) \
  return gather_windows<ZW, KB>(g, ntx, tiles, order, list, tinfo, flags, band, zlo, zhi, s)
  if (kb == 16) {
    switch (zw) {
      case 8: MTD_GW(8, 16);
      case 24: MTD_GW(24, 16);
      default: MTD_GW(16, 16);
    }
  }
  switch (zw) {
    case 8: MTD_GW(8, 8);
    case 24: MTD_GW(24, 8);
    default: MTD_GW(16, 8);
  }
#undef MTD_GW
}

hipError_t launch_gather_prepass(const AngleGeo* ageo, int A, int C, int nxmax, int V,
                                 const double* htab, int r2max, void* scratch, hipStream_t s) {
  GatherArgs g{nullptr, 0, ageo, A, C, nxmax, V, htab, nullptr, r2max, nullptr, nullptr, 0u};
  const int ntx = (V + GT - 1) / GT, tiles = ntx * ntx;
  TileEntry* list;
  int4* tinfo;
  gather_scratch_split(scratch, tiles, A, &list, &tinfo);
  return tile_prepass(g, ntx, tiles, list, tinfo, s);
}

size_t gather_scratch_bytes(int V, int A) {
  const size_t tiles = (size_t)((V + GT - 1) / GT) * ((V + GT - 1) / GT);
  const size_t nA = (size_t)(A > 0 ? A : 1);
  return tiles * nA * sizeof(TileEntry) + tiles * sizeof(int4);  // 16 B per entry
}

// The gather's dispatch order of the tiles of a V^3 volume: by distance of
// the tile centre from the lateral origin, nearest first (the tiles there
// hold the longest hit lists), ties by index.
void gather_tile_order_host(int V, int* order) {
  const int ntx = (V + GT - 1) / GT, tiles = ntx * ntx;
  std::vector<std::pair<long, int>> key(tiles);
  for (int t = 0; t < tiles; ++t) {
    const long dx = 2L * ((t % ntx) * GT) + GT - V, dy = 2L * ((t / ntx) * GT) + GT - V;
    key[t] = {dx * dx + dy * dy, t};
  }
  std::sort(key.begin(), key.end());
  for (int t = 0; t < tiles; ++t) order[t] = key[t].second;
}

// ---------------------------------------------------------------------------
// finalisation passes
// ---------------------------------------------------------------------------
// heights outside [band.x, band.y] hold zeros; band == nullptr: none
__device__ __forceinline__ bool outside_band(const int2* band, int z) {
  if (!band) return false;
  const int2 b = *band;
  return z < b.x || z > b.y;
}

// A spectrum volume from outside (mtd_finalize) comes without its hit band.
// The x pass, which reads every voxel, finds out: occ[z][y] says whether the
// row's block held anything but zeros (blocks of zero rows stop there), and
// k_band_found takes the band of planes that did from it. The y pass reads no
// empty row and skips the planes outside, the height pass reads the band alone.
// On a spectrum of 400 angles at 512^3, band about a third, with the OTF: x 733 ->
// 393, y 450 -> 114, z 532 -> 280 us. Waves that found something read their counts
// ahead of the block's answer: with the counts after it, a dense spectrum took
// longer than without the look (1024^3, all three passes: 15.5 ms without, 16.7 with
// counts after, 14.8 now; 512^3 1570, 1403 and 1401 us; 512^3 with a third of the
// planes occupied 1567, 752 and 750). Sides up to kScanOver go without.
// (With every voxel's count read and divided by before the scan, the OTF stored a
// byte at a time and two atomics on one word for the band: x 557 us.)
constexpr int kBandThreads = 1024;
// occ: V^2 bytes, readable to the next multiple of 16
__global__ void __launch_bounds__(kBandThreads)
k_band_found(const uint4* __restrict__ occ, int V, int2* __restrict__ band) {
  const int n = V * V;
  int lo = n, hi = -1;  // first and last occupied row
  constexpr int KB = 8;  // words in flight
  for (int i0 = threadIdx.x; 16 * i0 < n; i0 += KB * kBandThreads) {
    uint4 w[KB];
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const int i = i0 + k * kBandThreads;
      w[k] = 16 * i < n ? occ[i] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const uint32_t q[4] = {w[k].x, w[k].y, w[k].z, w[k].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int b = 16 * (i0 + k * kBandThreads) + 4 * j;
        if (q[j] && b < n) {  // V is even: whole words
          lo = min(lo, b + __builtin_ctz(q[j]) / 8);
          hi = max(hi, b + 3 - __builtin_clz(q[j]) / 8);
        }
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o, 64));
    hi = max(hi, __shfl_xor(hi, o, 64));
  }
  __shared__ int2 red[kBandThreads / 64];
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = make_int2(lo, hi);
  __syncthreads();
  if (threadIdx.x) return;
  for (int w = 1; w < kBandThreads / 64; ++w) {
    lo = min(lo, red[w].x);
    hi = max(hi, red[w].y);
  }
  *band = hi < 0 ? make_int2(V, -1) : make_int2(lo / V, hi / V);
}

// What the x pass transforms: the gather's normalised volume, already times
// (-1)^(x+y+z); a spectrum and its counts; these without a look for their band.
enum NormKind { kNormDone, kNormScan, kNormAll };
template <int VT, NormKind KIND>
struct NormXOp {  // rows along x; a = z, line = y
  static constexpr bool kScans = KIND == kNormScan;
  const float2* vol;
  const int32_t* cnt;
  float2* out;
  uint8_t* otf;
  const float2* tw;
  const int2* band;  // kNormDone
  uint8_t* occ;      // kNormScan
  __device__ bool skip(int z) const { return KIND == kNormDone && outside_band(band, z); }
  __device__ void begin(int) {}
  // The OTF (nonzero real parts) goes through LDS to whole words, and only the
  // rows that hold something read their counts and divide.
  __device__ bool flags() const { return otf != nullptr; }
  __device__ void store_flags(int z, int y0, int n, const uint8_t* f) const {
    uint8_t* o = otf + ((size_t)z * V + y0) * V;
    if ((uintptr_t)o % 16 == 0 && n * V % 16 == 0) {  // uniform
      for (int i = threadIdx.x; i < n * V / 16; i += blockDim.x)
        ((uint4*)o)[i] = f ? ((const uint4*)f)[i] : make_uint4(0, 0, 0, 0);
    } else {
      for (int i = threadIdx.x; i < n * V; i += blockDim.x) o[i] = f ? f[i] : 0;
    }
  }
  __device__ bool keep(int z, int y0, int n, bool any) const {
    for (int i = threadIdx.x; i < n; i += blockDim.x) occ[(size_t)z * V + y0 + i] = any;
    return any;
  }
  __device__ float2 raw(int z, int y, int x) const { return vol[((size_t)z * V + y) * V + x]; }
  __device__ int part(int z, int y, int x) const { return cnt[((size_t)z * V + y) * V + x]; }
  __device__ float2 value(float2 v, int c0, int z, int y, int x) const {
    const float c = (float)(c0 == 0 ? 1 : c0);
    const float2 t = make_float2(v.x / c, v.y / c);
    return (x + y + z) & 1 ? make_float2(-t.x, -t.y) : t;
  }
  __device__ float2 load(int z, int y, int x) const {
    if constexpr (KIND == kNormDone) return raw(z, y, x);
    const float2 t = value(raw(z, y, x), part(z, y, x), z, y, x);
    if (otf) otf[((size_t)z * V + y) * V + x] = (t.x != 0.f) ? 1 : 0;
    return t;
  }
  __device__ void store(int z, int y, int x, float2 v) const {
    out[((size_t)z * V + y) * V + x] = v;
  }
  Dim<VT> V{};
};

// OCC: rows with occ 0 hold zeros and are not read. (At run time instead, a branch
// around every load: dense 1024^3 spectra 3.5 -> 7.4 ms.)
template <int VT, bool OCC>
struct PlaneYOp {  // columns of each z plane; a = z, col = x, row = y
  static constexpr int kColThreads = 512;  // complex in and out
  static constexpr bool kBalancedCols = true;
  float2* buf;
  const float2* tw;
  const int2* band;
  const uint8_t* occ;
  __device__ bool skip(int z) const { return outside_band(band, z); }
  __device__ void begin(int) {}
  __device__ float2 load(int z, int x, int y) const {
    if constexpr (OCC) {
      // a plane's view: an empty row's lanes read out of its range, without a
      // branch that would end the batch of loads
      const BufView p(buf + (size_t)z * V * V, (unsigned)V * V * sizeof(float2));
      return p.f2(occ[(size_t)z * V + y] ? ((unsigned)y * V + x) * sizeof(float2) : ~0u, 0);
    }
    return buf[((size_t)z * V + y) * V + x];
  }
  __device__ void store(int z, int x, int y, float2 v) const { buf[((size_t)z * V + y) * V + x] = v; }
  Dim<VT> V{};
};

template <int VT>
struct ZOutOp {  // lines along z; a = y, col = x, row = z
  static constexpr bool kBalancedCols = true;
  const float2* buf;
  float* re;
  float* im;
  const float2* tw;
  float df3, cte, gsign;
  const int2* band;
  int only;  // 1: launched for bands that fit the folded pass, 2: for the others
  int lo, hi;
  __device__ bool skip(int) const {
    if constexpr (cols_fold_fits<VT>()) {
      if (only) {
        const int2 b = *band;
        return cols_fold_narrow<VT>(b.x, b.y) != (only == 1);
      }
    }
    return false;
  }
  __device__ void begin(int) {
    if (band) {
      const int2 b = *band;
      lo = b.x;
      hi = b.y;
    } else {
      lo = 0;
      hi = V - 1;
    }
  }
  __device__ float2 load(int y, int x, int z) const {
    if (z < lo || z > hi) return make_float2(0.f, 0.f);
    return buf[((size_t)z * V + y) * V + x];
  }
  __device__ void store(int y, int x, int z, float2 v) const {
    const float sg = ((x + y + z) & 1) ? -gsign : gsign;
    const size_t i = ((size_t)z * V + y) * V + x;
    re[i] = (v.x * sg * df3) * cte;
    if (im) im[i] = (v.y * sg * df3) * cte;  // uniform: NULL skips the imaginary part
  }
  // the same for column x0 + c, with y, x0 and z uniform over the wave and
  // c < 64 its lane: scalar addresses
  __device__ __forceinline__ float2 load_wave(int y, int x0, int c, int z) const {
    const bool in = z >= lo && z <= hi;
    return BufView(buf + ((size_t)(in ? z : 0) * V + y) * V + x0, in ? 64 * 8 : 0).f2(c * 8, 0);
  }
  __device__ __forceinline__ void store_wave(int y, int x0, int c, int z, float2 v) const {
    const float sg = ((x0 + c + y + z) & 1) ? -gsign : gsign;
    const size_t i = ((size_t)z * V + y) * V + x0;
    (re + i)[c] = (v.x * sg * df3) * cte;
    if (im) (im + i)[c] = (v.y * sg * df3) * cte;
  }
  Dim<VT> V{};
};

// the compiled row / column pass of tile variant TV (passes.hpp)
template <int VT, bool INV, int TV, class Op>
static void vol_rows_tv(const Op& op, hipStream_t s) {
  hipLaunchKernelGGL((k_rows<VT, INV, Op, TV>), (rows_grid<VT, TV>(VT)), (rows_block<VT, TV>()),
                     0, s, op);
}
template <int VT, bool INV, int TV, class Op>
static void vol_cols_tv(const Op& op, hipStream_t s) {
  hipLaunchKernelGGL((k_cols<VT, INV, Op, TV>), (cols_grid<VT, Op, TV>(VT)),
                     (cols_block<VT, Op, TV>()), 0, s, op);
}

// A row pass or a column pass over V batches: compiled register FFTs (VT > 0)
// or the runtime-length FFTs (VT == 0). TILES: the tile variants (rows: 0, 1;
// columns: 0, 1, 2) are compiled and picked at run time; otherwise variant 0.
template <int VT, bool INV, bool TILES, class Op>
static hipError_t vol_rows(Dim<VT> V, const Op& op, const FftTab& ft, const char* name, int tile,
                           hipStream_t s) {
  Timed tm(name, s);
  if constexpr (VT > 0) {
    if (TILES && tile == 1) {
      if constexpr (TILES) vol_rows_tv<VT, INV, 1>(op, s);
    } else {
      vol_rows_tv<VT, INV, 0>(op, s);
    }
    return hipGetLastError();
  } else {
    if (!ft.gen) return hipErrorInvalidValue;
    return launch_gen<INV, true>(op, *ft.gen, V, V, s);
  }
}

template <int VT, bool INV, bool TILES, class Op>
static hipError_t vol_cols(Dim<VT> V, const Op& op, const FftTab& ft, const char* name, int tile,
                           hipStream_t s) {
  std::optional<Timed> tm;  // name NULL: the caller's
  if (name) tm.emplace(name, s);
  if constexpr (VT > 0) {
    if constexpr (op_cols_balanced<Op>::value && cols_b_fits<VT>()) {
      hipLaunchKernelGGL((k_cols_b<VT, INV, Op>), cols_b_grid<VT>(VT), cols_b_block<VT>(), 0, s,
                         op);
    } else if constexpr (TILES) {
      if (tile == 1) vol_cols_tv<VT, INV, 1>(op, s);
      else if (tile == 2) vol_cols_tv<VT, INV, 2>(op, s);
      else vol_cols_tv<VT, INV, 0>(op, s);
    } else {
      vol_cols_tv<VT, INV, 0>(op, s);
    }
    return hipGetLastError();
  } else {
    if (!ft.gen) return hipErrorInvalidValue;
    return launch_gen<INV, false>(op, *ft.gen, V, V, s);
  }
}

// The height pass. Volumes of 448, 512 and from 576 on fold the band (k_cols_fold): planes is
// the band's height expected from the geometry, 0 where there is none. Only the
// device knows the band, and a specular past the pupil's rim makes it wider than
// expected: both forms are launched, and the blocks of the one that does not apply
// return (9 us of 2110 at 512^3, 86 of 7830 at 1024^3; blocks that loop over batches
// instead return at once, but take 1.6 to 2 times as long where they are needed).
// 512^3, band 151: 335 -> 278 us; 1024^3, band 302: 5.05 -> 2.43 ms.
template <int VT>
static hipError_t vol_z(Dim<VT> V, ZOutOp<VT> z, int planes, const FftTab& ft, int tile,
                        hipStream_t s) {
  Timed tm("vol_z", s);
  if constexpr (VT > 0 && cols_fold_fits<VT>()) {
    // the band may begin at any element of its first group of T
    constexpr int T = Fft2<VT / cols_fold_r<VT>(), false>::T;
    if (planes == 0 || cols_fold_narrow<VT>(T - 1, T - 1 + planes - 1)) {
      z.only = 1;
      hipLaunchKernelGGL((k_cols_fold<VT, true, ZOutOp<VT>>), dim3(VT / cols_fold_nc<VT>(), VT),
                         dim3(cols_fold_threads<VT>()), 0, s, z);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      z.only = 2;
    }
  }
  return vol_cols<VT, true, true>(V, z, ft, nullptr, tile, s);
}

template <int VT>
static hipError_t finalize_v(Dim<VT> V, const float2* vol, const int32_t* cnt,
                             int2* band, uint8_t* occ, int planes, float2* work,
                             float df3, float cte, float gsign, float* re,
                             float* im, uint8_t* otf, const FftTab& ft, int2 tiles,
                             hipStream_t s) {
  ZOutOp<VT> z{work, re, im, ft.tw, df3, cte, gsign, band, 0, 0, V - 1, V};
  hipError_t e;
  if (occ) {
    NormXOp<VT, kNormScan> x{vol, cnt, work, otf, ft.tw, nullptr, occ, V};
    if ((e = vol_rows<VT, true, true>(V, x, ft, "vol_x", tiles.x, s)) != hipSuccess) return e;
    Timed tm("vol_band", s);
    hipLaunchKernelGGL(k_band_found, dim3(1), dim3(kBandThreads), 0, s, (const uint4*)occ, (int)V,
                       band);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    PlaneYOp<VT, true> y{work, ft.tw, band, occ, V};
    if ((e = vol_cols<VT, true, true>(V, y, ft, "vol_y", tiles.y, s)) != hipSuccess) return e;
  } else {
    if (band) {
      NormXOp<VT, kNormDone> x{vol, cnt, work, otf, ft.tw, band, nullptr, V};
      e = vol_rows<VT, true, true>(V, x, ft, "vol_x", tiles.x, s);
    } else {
      NormXOp<VT, kNormAll> x{vol, cnt, work, otf, ft.tw, nullptr, nullptr, V};
      e = vol_rows<VT, true, true>(V, x, ft, "vol_x", tiles.x, s);
    }
    if (e != hipSuccess) return e;
    PlaneYOp<VT, false> y{work, ft.tw, band, nullptr, V};
    if ((e = vol_cols<VT, true, true>(V, y, ft, "vol_y", tiles.y, s)) != hipSuccess) return e;
  }
  return vol_z<VT>(V, z, planes, ft, tiles.y, s);
}

// ---------------------------------------------------------------------------
// Born forward model (Simul_holo/main.cpp:106-109 and calcHolo,
// Simul_holo/src/fonctions.cpp:109-140): the centred 3-D spectrum of the
// index contrast, TF3D = fftshift3D(FFT3D(fftshift3D(dn))) * Tp^3
// (TF3Dcplx, Simul_holo/src/FFT_fonctions.cpp:301-318), sampled on each
// angle's Ewald cap. Both shifts are (-1)^(x+y+z) sign flips (even V), the
// output ones times (-1)^(3V/2) = gsign. The height pass runs first: it reads
// the real contrast (4 bytes per voxel) and stores only the planes of the hit
// band, the only ones the caps read, and the y and x passes then run on those
// planes alone. With the band a third of the volume that is about 16 bytes
// per voxel; x, y and z in that order with the band cut last took 39. Measured
// at 416^3, 200 angles: 606 -> 246 us, at 256^3 (400 angles) 116 -> 71 us.
// ---------------------------------------------------------------------------
template <int VT>
struct ContrastZOp {  // lines along z of the contrast volume; a = y, col = x, row = z
  static constexpr bool kBalancedCols = true;
  const float* re;
  const float* im;  // nullptr: real contrast
  float2* out;
  const float2* tw;
  const int2* band;
  int lo, hi;
  __device__ void begin(int) {
    const int2 b = *band;
    lo = b.x;
    hi = b.y;
  }
  __device__ float2 load(int y, int x, int z) const {
    const size_t i = ((size_t)z * V + y) * V + x;
    float2 t = make_float2(re[i], im ? im[i] : 0.f);
    if ((x + y + z) & 1) { t.x = -t.x; t.y = -t.y; }
    return t;
  }
  __device__ void store(int y, int x, int z, float2 v) const {
    if (z < lo || z > hi) return;
    out[((size_t)z * V + y) * V + x] = v;
  }
  Dim<VT> V{};
};

template <int VT>
struct SpectrumXOp {  // rows along x of the band's planes, in place; a = z, line = y
  float2* buf;
  const float2* tw;
  const int2* band;
  __device__ bool skip(int z) const { return outside_band(band, z); }
  __device__ void begin(int) {}
  __device__ float2 load(int z, int y, int x) const { return buf[((size_t)z * V + y) * V + x]; }
  __device__ void store(int z, int y, int x, float2 v) const {
    buf[((size_t)z * V + y) * V + x] = ((x + y + z) & 1) ? make_float2(-v.x, -v.y) : v;
  }
  Dim<VT> V{};
};

template <int VT>
static hipError_t contrast_spectrum_v(Dim<VT> V, const float* re, const float* im, float2* work,
                                      const int2* band, const FftTab& ft, hipStream_t s) {
  ContrastZOp<VT> z{re, im, work, ft.tw, band, 0, V - 1, V};
  PlaneYOp<VT, false> y{work, ft.tw, band, nullptr, V};
  SpectrumXOp<VT> x{work, ft.tw, band, V};
  hipError_t e;
  if ((e = vol_cols<VT, false, false>(V, z, ft, "fwd_vol_z", 0, s)) != hipSuccess) return e;
  if ((e = vol_cols<VT, false, false>(V, y, ft, "fwd_vol_y", 0, s)) != hipSuccess) return e;
  return vol_rows<VT, false, false>(V, x, ft, "fwd_vol_x", 0, s);
}

// calcHolo's sampling, in the frame of the per-angle spectra (+posSpec frame:
// bin (row, col) is pupil pixel fd = (col - NXMAX, row - NXMAX)): the voxel is
// retroPropag_Born's (the simulator's fobj = round(fd - fi) in centred
// coordinates is the same integer map), and the value is
// -i * q(|fd|^2) * TF3D[voxel] with q = kv / (sqrt(R^2 - |fd|^2) / R) and TF3D
// the transform in vol times fac / (kv R): one factor, rounded once to FP32.
// Error of the spectra against 64 bits over 14 lengths from 64 to 512, ten
// objects each: passes in the order x, y, z, their result scaled, then times a
// rounded q: 1; height pass first 1.04 of that; with the one factor 0.97. Bins
// outside the pupil, of skipped angles, or whose height leaves the volume
// are 0, and so are bins whose voxel would leave the volume laterally (a
// caller's specular outside the crop; the accumulation has no hit there).
// With RES the solver's weighted residual is stored instead, q * w * (S - y) (w
// NULL: 1; the real factors applied one after the other): q is the factor the
// adjoint's gather would apply per hit, so the adjoint can skip it. Bins that no
// cap reads are 0 there, and their y and w are not read. One pass in place of
// two: 400 angles of 128^2, 43 + 35 -> 55 us (blocks of 256 columns left half of
// the threads without a bin there).
constexpr int kCapX = 64, kCapY = 4;
constexpr int kCapA = 8;  // angles a thread samples, their loads in flight together
template <bool RES>
__global__ void __launch_bounds__(kCapX * kCapY)
k_cap_sample(const float2* __restrict__ vol, const AngleGeo* __restrict__ ageo, int A,
             const double* __restrict__ htab, double fac, const float* __restrict__ q2, int r2max,
             int nx, int C, int V, const float2* __restrict__ y, const float* __restrict__ w,
             float2* __restrict__ spec) {
#pragma clang fp contract(off)
  // grid (column blocks, row blocks, angle groups): no division by the runtime C
  const int col = blockIdx.x * kCapX + threadIdx.x, row = blockIdx.y * kCapY + threadIdx.y;
  if (col >= C || row >= C) return;
  const int a0 = blockIdx.z * kCapA, i = row * C + col;
  const size_t C2 = (size_t)C * C;
  const int fdx = col - nx, fdy = row - nx;
  const int r2 = fdx * fdx + fdy * fdy;
  if (r2 > r2max) {
    for (int a = a0; a < min(a0 + kCapA, A); ++a) spec[a * C2 + i] = make_float2(0.f, 0.f);
    return;
  }
  const double h = htab[r2];
  const float f = (float)(fac / h);
  const float q = RES ? q2[i] : 0.f;
  // voxel 0 stands in for a bin without one, so that no load hangs on a branch
  size_t vi[kCapA];
  bool in[kCapA], live[kCapA];
  float2 t[kCapA], m[kCapA];
  float k[kCapA];
#pragma unroll
  for (int j = 0; j < kCapA; ++j) {
    const AngleGeo ag = ageo[min(a0 + j, A - 1)];
    const int z = (int)round_away(h - ag.fz) + V / 2;
    const int X = fdx - ag.fx + V / 2, Y = fdy - ag.fy + V / 2;
    live[j] = !ag.skip;
    in[j] = !ag.skip && z >= 0 && z < V && X >= 0 && X < V && Y >= 0 && Y < V;
    vi[j] = in[j] ? ((size_t)z * V + Y) * V + X : 0;
  }
#pragma unroll
  for (int j = 0; j < kCapA; ++j) {
    t[j] = vol[vi[j]];
    if constexpr (RES) m[j] = y[min(a0 + j, A - 1) * C2 + i];
  }
  if (RES && w) {  // uniform
#pragma unroll
    for (int j = 0; j < kCapA; ++j) k[j] = w[min(a0 + j, A - 1) * C2 + i];
  } else {
#pragma unroll
    for (int j = 0; j < kCapA; ++j) k[j] = 1.f;
  }
#pragma unroll
  for (int j = 0; j < kCapA; ++j) {
    if (a0 + j >= A) break;  // uniform
    float2 s = in[j] ? make_float2(f * t[j].y, -(f * t[j].x)) : make_float2(0.f, 0.f);
    if constexpr (RES) {
      s = live[j] ? make_float2((s.x - m[j].x) * k[j] * q, (s.y - m[j].y) * k[j] * q)
                  : make_float2(0.f, 0.f);
    }
    spec[(a0 + j) * C2 + i] = s;
  }
}

// Data weights of the adjoint-iterative form: w = 1 / (q(|fd|^2)^2 * hits of
// the sample's voxel) on the cap samples, 0 elsewhere. With them A^H W A is
// Tp^6 times the centred 3-D DFT's projection on the hit voxels: the least
// squares are then as well conditioned as the plain method's count
// normalisation.
__global__ void __launch_bounds__(256)
k_cap_weights(const int32_t* __restrict__ cnt, const AngleGeo* __restrict__ ageo,
              const double* __restrict__ htab, const float* __restrict__ q, int r2max, int nx,
              int C, int V, float* __restrict__ w) {
  const int a = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= C * C) return;
  const int fdx = i % C - nx, fdy = i / C - nx;
  const int r2 = fdx * fdx + fdy * fdy;
  const AngleGeo ag = ageo[a];
  float out = 0.f;
  if (!ag.skip && r2 <= r2max) {
    const int z = (int)round_away(htab[r2] - ag.fz) + V / 2;
    const int X = fdx - ag.fx + V / 2, Y = fdy - ag.fy + V / 2;
    if (z >= 0 && z < V && X >= 0 && X < V && Y >= 0 && Y < V) {
      const int c = cnt[((size_t)z * V + Y) * V + X];  // >= 1: this sample hits it
      const float qq = q[r2];
      out = 1.f / (qq * qq * (float)c);
    }
  }
  w[(size_t)a * C * C + i] = out;
}

#define MTD_VOL_SIZES(X)                                                                   \
  X(32) X(64) X(128) X(256) X(320) X(384) X(416) X(448) X(512) X(576) X(640) X(704) X(768) \
  X(1024)

hipError_t launch_finalize(int V, const float2* vol, const int32_t* cnt,
                           int2* band, uint8_t* occ, int planes, float2* work, float df3,
                           float cte, float gsign, float* out_re, float* out_im,
                           uint8_t* otf, const FftTab& ft, int2 tiles, hipStream_t s) {
  switch (V) {
#define X(n)                                                                                   \
  case n:                                                                                      \
    return finalize_v<n>(Dim<n>{}, vol, cnt, band, occ, planes, work, df3, cte, gsign, \
                         out_re, out_im, otf, ft, tiles, s);
    MTD_VOL_SIZES(X)
#undef X
  }
  return finalize_v<0>(Dim<0>(V), vol, cnt, band, occ, planes, work, df3, cte, gsign,
                       out_re, out_im, otf, ft, tiles, s);
}

hipError_t launch_contrast_spectrum(int V, const float* re, const float* im, float2* work,
                                   const int2* band, const FftTab& ft, hipStream_t s) {
  switch (V) {
#define X(n) \
  case n: return contrast_spectrum_v<n>(Dim<n>{}, re, im, work, band, ft, s);
    MTD_VOL_SIZES(X)
#undef X
  }
  return contrast_spectrum_v<0>(Dim<0>(V), re, im, work, band, ft, s);
}

hipError_t launch_cap_sample(const float2* vol, const AngleGeo* ageo, int A, const double* htab,
                             double fac, const float* q2, int r2max, int nx, int C, int V,
                             const float2* y, const float* w, float2* spec, hipStream_t s) {
  Timed tm("cap_sample", s);
  if (A <= 0) return hipSuccess;
  const dim3 grid((C + kCapX - 1) / kCapX, (C + kCapY - 1) / kCapY, (A + kCapA - 1) / kCapA),
      block(kCapX, kCapY);
  if (y)
    hipLaunchKernelGGL((k_cap_sample<true>), grid, block, 0, s, vol, ageo, A, htab, fac, q2, r2max,
                       nx, C, V, y, w, spec);
  else
    hipLaunchKernelGGL((k_cap_sample<false>), grid, block, 0, s, vol, ageo, A, htab, fac, q2, r2max,
                       nx, C, V, nullptr, nullptr, spec);
  return hipGetLastError();
}

hipError_t launch_cap_weights(const int32_t* cnt, const AngleGeo* ageo, int A,
                              const double* htab, const float* q, int r2max, int nx, int C,
                              int V, float* w, hipStream_t s) {
  Timed tm("cap_weights", s);
  hipLaunchKernelGGL(k_cap_weights, dim3((C * C + 255) / 256, A), dim3(256), 0, s, cnt, ageo,
                     htab, q, r2max, nx, C, V, w);
  return hipGetLastError();
}

bool vol_len_supported(int V) {
  switch (V) {
#define X(n) case n: return true;
    MTD_VOL_SIZES(X)
#undef X
  }
  return false;
}

}  // namespace mtd
