// Runtime-length FFTs for the transform lengths that have no compiled
// register FFT (fft_reg.hpp): any hologram side, crop side or volume side the
// configuration files can hold, as FFTW plans any size
// (pretraitement_hors_axe_CPU/main.cpp:103, src/FFTW_init.cpp:70-71,
// Reconstruction/src/FFT_encaps.cpp:33-53).
//
// A block transforms nl lines (a power of two) held in LDS, line fastest:
//  - direct: L factors into the radices 8, 4, 2, 3, 5, 7, 11, 13, in this
//    order. Each is one Stockham autosort pass: a thread reads the values of
//    its butterflies (about 16) into registers, and after a barrier writes
//    their DFTs back to the same buffer;
//  - Bluestein (chirp-z) for lengths with a larger prime factor, written
//    from the published method: X_k = w_k sum_n (x_n w_n) conj(w_(k-n)) with
//    w_m = exp(-i pi m^2 / L), the convolution done as a cyclic one of length
//    W = a power of two >= 2L - 1 with two forward length-W FFTs (the inverse
//    through conjugation) and the host-computed spectrum of the chirp (scaled
//    1/W). The backward transform is conj(forward(conj(x))).
// Operations load and store through the same op interface as the compiled
// passes (passes.hpp): load(batch, line, element), store(batch, line,
// element, value), optional begin/skip/line.
//
// The order of the roundings is part of the result: hologram crops go through
// here to the demodulated field, and the angle and logarithm of that amplify a
// last-bit change where it is faint. Radices up to 32, Bluestein over any
// product of radices (243 points for 122) and hologram rows in pairs moved
// unwrapped fields by up to 3e-3 of their scale at single pixels and raised
// the error against 64 bits (index of 75 holograms of 2048^2, crop 202: 3.3e-5
// -> 7.5e-5; solver on a 124^3 unknown: 1.0e-7 -> 1.9e-7). Hence these radices,
// these Bluestein lengths and products spelled out (gen_cmul).
//
// What bounds it: the passes' LDS round trips and barriers, not HBM (a 364-point
// line takes about 2 ns of the chip, twice its memory time). Out of place
// between two LDS buffers with one butterfly a thread at a time, as many columns
// per block as the two buffers held (11 at 364) and integer divisions in every
// pass: 364^3 inverse passes 911 us, now 402; hologram rows of 600 219, now
// 110; crop-122 rows and columns (Bluestein over 256 points) 238, now 106.
// About 16 values a thread: 8, 24 and 32 took 928, 842 and 970 us for 48 x
// 600^2 -> 364^3, 16 takes 802; one butterfly of radices up to 32 took 807
// with the rows in pairs.
#pragma once
#include <hip/hip_runtime.h>

#include <utility>

#include "dft.hpp"
#include "passes.hpp"

namespace mtd {

constexpr int kGenMaxPasses = 8;
constexpr int kGenThreads = 512;     // most threads of a block
constexpr int kGenLdsBytes = 65536;  // most LDS of a block
constexpr int kGenMaxLen = 4096;     // most points of a line in LDS
constexpr int kGenBlocks = 256;      // blocks that give every CU one

struct GenPlan {
  int L;                   // transform length
  int W;                   // working length: L (direct) or the Bluestein length
  int nf;                  // radix passes over W
  int f[kGenMaxPasses];    // radices
  int threads;             // most threads of a pass over one line
  const float2* tw;        // exp(-2 pi i k / W), k < W
  const float2* chirp;     // Bluestein: exp(-i pi n^2 / L), n < L; nullptr: direct
  const float2* bk;        // Bluestein: FFT_W of the wrapped conj(chirp), times 1/W
};

// The lines of a block in LDS: element n of line l at p[n * pitch + l]. Rows
// are loaded along n (odd pitch: no bank conflicts), columns along l. The LDS
// address space is in the pointer's type: the passes are calls.
typedef float gen_v2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) gen_v2 gen_lds_v2;
struct GenLines {
  gen_lds_v2* p;
  int lnl, pitch;  // log2 of the lines, and the distance of two elements
  __device__ __forceinline__ int nl() const { return 1 << lnl; }
  __device__ __forceinline__ float2 get(int l, int n) const {
    const gen_v2 v = p[n * pitch + l];
    return make_float2(v.x, v.y);
  }
  __device__ __forceinline__ void set(int l, int n, float2 v) const {
    p[n * pitch + l] = gen_v2{v.x, v.y};
  }
};

inline int gen_pitch(int lnl, bool rows) { return rows && lnl > 0 ? (1 << lnl) + 1 : 1 << lnl; }

// log2 of the lines per block: up to 32 (128-byte segments of float columns)
// as far as LDS and the threads allow, 16 where 32 would leave a CU fewer than
// four blocks; fewer where the launch would leave CUs without a block (rows and
// columns of 24 crops of 20^2: 20 us with 32 lines a block, 13 with 4; with half
// or a quarter of the CUs as the aim 13 and 15; 6 of 300^2 31 and 35, now 30)
inline int gen_lnl(const GenPlan& p, bool rows, int nlines, int batches) {
  int l = 5;
  auto bytes = [&](int k) { return (size_t)gen_pitch(k, rows) * p.W * sizeof(float2); };
  if (bytes(5) > 40960) l = 4;
  while (l > 0 && (bytes(l) > (size_t)kGenLdsBytes || (p.threads << l) > kGenThreads)) --l;
  while (l > 1 && ((nlines - 1) >> l) + 1 < kGenBlocks / batches) --l;
  return l;
}

inline int gen_threads(const GenPlan& p, int lnl) { return ((p.threads << lnl) + 63) / 64 * 64; }

// a w and conj(a) w, their two roundings per part spelled out: the fused
// multiply-adds otherwise depend on what the compiler makes of the code around
// them.
__device__ __forceinline__ float2 gen_cmul(float2 a, float2 w) {
  return make_float2(__builtin_fmaf(a.x, w.x, -(a.y * w.y)), __builtin_fmaf(a.y, w.x, a.x * w.y));
}
__device__ __forceinline__ float2 gen_cmul_conj(float2 a, float2 w) {
  return make_float2(__builtin_fmaf(a.x, w.x, a.y * w.y), __builtin_fmaf(a.x, w.y, -(a.y * w.x)));
}

// Butterflies of radix R a thread holds: about 16 values in registers.
__host__ __device__ constexpr int gen_per_thread(int R) { return R < 9 ? 16 / R : 1; }

// One Stockham pass of radix R over the block's lines, Ns the product of the
// radices before it. A call: inlined into the loop over passes (with radices up
// to 32), the constants of all radices' DFTs were kept in registers across it,
// 800 of them spilled.
template <int R, bool INV>
__device__ __attribute__((noinline)) void gen_pass_r(gen_lds_v2* p, int lnl, int pitch, int W,
                                                     int Ns, const float2* __restrict__ tw) {
  constexpr int K = gen_per_thread(R);
  const GenLines x{p, lnl, pitch};
  const int nb = W / R;  // uniform: one scalar division
  const int l = threadIdx.x & (x.nl() - 1), j0 = threadIdx.x >> x.lnl;
  const int dj = blockDim.x >> x.lnl;
  float2 v[K][R];
  int d[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const int j = j0 + i * dj;
    d[i] = j * R;
    if (j >= nb) continue;
#pragma unroll
    for (int r = 0; r < R; ++r) v[i][r] = x.get(l, j + r * nb);
    if (Ns > 1) {  // uniform
      // the last pass has Ns = nb: each butterfly is its own k
      int k = j;
      d[i] = j;
      if (nb != Ns) {
        const int q = j / Ns;
        k = j - q * Ns;
        d[i] = q * Ns * R + k;
      }
      const int step = k * (W / (Ns * R));  // W_(Ns R)^(r k) = W_W^(r step)
#pragma unroll
      for (int r = 1; r < R; ++r) {
        float2 w = tw[r * step];
        if (INV) w.y = -w.y;
        v[i][r] = gen_cmul(v[i][r], w);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (j0 + i * dj >= nb) continue;
    Dft<R, INV>::run(v[i]);
#pragma unroll
    for (int r = 0; r < R; ++r) x.set(l, d[i] + r * Ns, v[i][r]);
  }
  __syncthreads();
}

template <bool INV>
__device__ __forceinline__ void gen_stockham(const GenLines& x, const GenPlan& p) {
  int Ns = 1;
  for (int i = 0; i < p.nf; ++i) {
    const int R = p.f[i];
    switch (R) {
#define X(r) \
  case r: gen_pass_r<r, INV>(x.p, x.lnl, x.pitch, p.W, Ns, p.tw); break;
      X(2) X(3) X(4) X(5) X(7) X(8) X(11) X(13)
#undef X
    }
    Ns *= R;
  }
}

// Transforms of the block's lines, in place (elements [0, L) of each). Begins
// after the caller's barrier, ends with one. Bluestein is the forward transform
// only (the caller conjugates on the way in and out for the backward one). RAW
// (Bluestein): the lines come times the chirp and with zeros from L to W, and
// are left without the conjugate and the chirp of the way out (gen_out), which
// saves two round trips through LDS.
template <bool INV, bool RAW>
__device__ __forceinline__ void gen_fft(const GenLines& x, const GenPlan& p) {
  if (!p.chirp) {
    gen_stockham<INV>(x, p);
    return;
  }
  const int L = p.L, W = p.W, l = threadIdx.x & (x.nl() - 1);
  const int n0 = threadIdx.x >> x.lnl, dn = blockDim.x >> x.lnl;
  if (!RAW) {
    // x_n w_n, zero-padded to W
    for (int n = n0; n < W; n += dn)
      x.set(l, n, n < L ? gen_cmul(x.get(l, n), p.chirp[n]) : make_float2(0.f, 0.f));
    __syncthreads();
  }
#pragma unroll 1
  for (int half = 0; half < 2; ++half) {
    gen_stockham<false>(x, p);
    if (half == 0) {
      // times the chirp's spectrum, conjugated: the inverse length-W FFT is
      // conj(FFT(conj(.)))
      for (int k = n0; k < W; k += dn) {
        const float2 z = gen_cmul(x.get(l, k), p.bk[k]);
        x.set(l, k, make_float2(z.x, -z.y));
      }
    } else if (!RAW) {
      for (int k = n0; k < L; k += dn) x.set(l, k, gen_cmul_conj(x.get(l, k), p.chirp[k]));
    } else {
      break;
    }
    __syncthreads();
  }
}

// bin k of a RAW transform
template <bool INV>
__device__ __forceinline__ float2 gen_out(const GenLines& x, const GenPlan& p, int l, int k) {
  const float2 c = x.get(l, k);
  if (!p.chirp) return c;
  const float2 y = gen_cmul_conj(c, p.chirp[k]);
  return INV ? make_float2(y.x, -y.y) : y;
}

// real and imaginary parts exchanged: before and after a forward transform,
// the backward one
__device__ __forceinline__ float2 gen_swap(float2 v) { return make_float2(v.y, v.x); }

// Calls fn(line of the block, element) for this thread's share of nl lines of
// n elements: rows run along the lines, columns across them.
template <bool ROWS, class Fn>
__device__ __forceinline__ void gen_each(int lnl, int n, Fn&& fn) {
  if (ROWS) {
    for (int l = 0; l < 1 << lnl; ++l)
      for (int i = threadIdx.x; i < n; i += blockDim.x) fn(l, i);
  } else {
    const int l = threadIdx.x & ((1 << lnl) - 1);
    for (int i = threadIdx.x >> lnl; i < n; i += blockDim.x >> lnl) fn(l, i);
  }
}

// This thread's share of nl lines of n elements, brought in KB at a time: ld(line,
// element) of all of them, then st(line, element, value). One by one, as gen_each
// goes, a load's whole latency passed before the next (one to two dozen of them:
// the most of a block's time). ld is also called on repeats of the last element.
template <bool ROWS, int KB, class Ld, class St>
__device__ __forceinline__ void gen_load(int lnl, int n, Ld&& ld, St&& st) {
  const int lm = (1 << lnl) - 1;
  const int i0 = ROWS ? threadIdx.x : threadIdx.x >> lnl;
  const int di = ROWS ? blockDim.x : blockDim.x >> lnl;
  for (int q = 0; i0 + (ROWS ? q >> lnl : q) * di < n; q += KB) {
    float2 v[KB];
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      const int l = (ROWS ? q + j : threadIdx.x) & lm;
      v[j] = ld(l, min(i0 + (ROWS ? (q + j) >> lnl : q + j) * di, n - 1));
    }
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      const int l = (ROWS ? q + j : threadIdx.x) & lm;
      const int i = i0 + (ROWS ? (q + j) >> lnl : q + j) * di;
      if (i < n) st(l, i, v[j]);
    }
  }
}

// Batched 1-D transforms of nlines lines per batch (grid: line groups, rounded
// up to 8 of them, x batches; see xcd_block). ROWS: a block's lines are
// consecutive rows and element loads run along each line; otherwise its lines
// are adjacent columns and the loads of one element index run across them
// (coalesced either way).
template <bool INV, bool ROWS, class Op>
__global__ void __launch_bounds__(kGenThreads, 4)
k_gen(Op op, GenPlan p, int nlines, int lnl, int pitch) {
  extern __shared__ float2 gen_lds[];
  const int2 ab = xcd_block();
  const int a = ab.x, line0 = ab.y << lnl;
  if (line0 >= nlines) return;
  if (skip_batch(op, a)) return;  // block-uniform, before any barrier
  op.begin(a);
  const GenLines x{(gen_lds_v2*)gen_lds, lnl, pitch};
  const int nact = min(1 << lnl, nlines - line0), L = p.L;
  static_assert(ROWS || !has_line<Op>::value, "per-line state is for rows");
  bool any = false;
  // lines past the last repeat it: they are transformed but not stored
  auto load = [&](int l, int n) {
    const int line = line0 + min(l, nact - 1);
    float2 v;
    if constexpr (has_line<Op>::value) {
      Op o = op;
      o.line(a, line);
      v = o.load(a, line, n);
    } else {
      v = op.load(a, line, n);
    }
    if constexpr (op_scans<Op>::value) any = any || v.x != 0.f || v.y != 0.f;
    return v;
  };
  constexpr int KB = has_line<Op>::value ? 4 : 8;
  auto set = [&](int l, int n, float2 v) { x.set(l, n, v); };
  if (p.chirp) {  // uniform
    gen_load<ROWS, KB>(
        lnl, L,
        [&](int l, int n) {
          const float2 v = load(l, n), w = p.chirp[n];
          return INV ? gen_cmul_conj(v, w) : gen_cmul(v, w);
        },
        set);
    gen_each<false>(lnl, p.W - L, [&](int l, int n) { x.set(l, L + n, make_float2(0.f, 0.f)); });
  } else {
    gen_load<ROWS, KB>(lnl, L, load, set);
  }
  if constexpr (op_scans<Op>::value) {
    if (!op.keep(a, line0, nact, __syncthreads_or(any))) return;
  }
  __syncthreads();
  gen_fft<INV, true>(x, p);
  gen_each<ROWS>(lnl, L, [&](int l, int n) {
    if (l < nact) op.store(a, line0 + l, n, gen_out<INV>(x, p, l, n));
  });
}

// line groups of a launch, rounded up to a multiple of 8
inline unsigned gen_groups(int nlines, int lnl) {
  return (unsigned)(((nlines + (1 << lnl) - 1) >> lnl) + 7) / 8 * 8;
}

template <bool INV, bool ROWS, class Op>
inline hipError_t launch_gen(const Op& op, const GenPlan& p, int nlines, int batches,
                             hipStream_t s) {
  if (nlines <= 0 || batches <= 0) return hipSuccess;
  const int lnl = gen_lnl(p, ROWS, nlines, batches), pitch = gen_pitch(lnl, ROWS);
  hipLaunchKernelGGL((k_gen<INV, ROWS, Op>), dim3(gen_groups(nlines, lnl), batches),
                     dim3(gen_threads(p, lnl)), (size_t)pitch * p.W * sizeof(float2), s, op, p,
                     nlines, lnl, pitch);
  return hipGetLastError();
}

}  // namespace mtd
