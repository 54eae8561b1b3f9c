// Phase unwrapping, DEROUL 1 with VOLKOV 1 (deroul_volkov4_total_sym_paire,
// pretraitement_hors_axe_CPU/src/deroulement_volkov4.cpp:14-92).
//
// For each angle the wrapped phase phi = atan2(U) of the C x C demodulated
// field is mirror-extended to 2C x 2C (Symetrise_mirror :221-240), the FFT
// gradients of phi_s and of Z = exp(i phi_s) give the gradient of the field of
// 2 pi multiples, g = (Im(grad Z / Z) - grad phi_s) / 2 pi, which is
// integrated by the FFT least-squares (Poisson) solve of integ_grad4
// (:162-191); the original quadrant of the result times 2 pi is added to phi.
//
// Two identities take this to four passes of C-point transforms:
//  - The spectral gradient and the spectral least-squares integration undo
//    each other, so integrating -grad phi_s gives mean(phi) - phi exactly:
//    the unwrapped phase is the integral of Im(grad Z / Z) plus the constant
//    mean(phi). Unwrapping only runs ahead of the polynomial phase fit, whose
//    constant monomial removes any constant (as it removes the reference's
//    arbitrary zero frequency, :189, read one element past its array), so
//    the constant is left out and phi itself is never needed: Z = U / |U|.
//  - On the even extension every transform is a cosine or sine transform of
//    the C original samples. The Nyquist terms vanish: the extension has
//    none, and a gradient's, halved by its one-sided frequency -1/2, only
//    gives an imaginary part, which the reference discards. A C-point DCT-II
//    is one C-point complex FFT of the reordered line (J. Makhoul, "A fast
//    cosine transform in one and two dimensions", IEEE Trans. ASSP 28, 1980):
//    position m holds sample n(m) = 2m (m < C/2) or 2(C-1-m)+1, and with
//    V = FFT(v), t = pi k / 2C, P = e^{-it} V[k], Q = e^{it} V[C-k] (V[C] =
//    V[0]), the DCT-II is X[k] = (P + Q) / 2 and X[C-k] = i (P - Q) / 2, for
//    complex lines too (two real lines in one transform). The DST-II of x is
//    the DCT-II of (-1)^n x, read at C - k. The inverse of real Y[k] is the
//    backward FFT of e^{it} (Y[k] - i Y[C-k]), Y[C] = 0, whose position m
//    holds Y[0] + 2 sum_k Y[k] cos(pi k (2n+1) / 2C) at n = n(m).
//  So the derivative of a line of Z is: FFT, W[k] = -(i pi / 2C)
//  ((1 - 2k/C) V[k] - e^{i pi k/C} V[C-k]), backward FFT, sign -1 on the odd
//  samples.
// Passes (C x C per angle; each one reads and writes memory once):
//  A rows     gx = Im(dZ/dx conj Z)                               8 + 4 bytes
//  B columns  gy the same way, in registers; DCT-II along y of gx and
//             DST-II along y of gy from one packed FFT: H        12 + 8
//  C rows     DST-II along x of the first, DCT-II along x of the second from
//             one packed FFT, the Poisson quotient, inverse along x: R  8 + 4
//  D columns  inverse along y, two columns in one FFT: the phase   4 + 4
// 52 bytes per pixel bound the passes. The same method on the 2C x 2C extension
// (half-empty transforms, both gradients with their trigonometry on every
// pixel three times) moved about 300. Measured, all unwrapping kernels, that
// form against this one: 300 crops of 250^2 3217 -> 536 us, 400 of 128^2 813 ->
// 144 us, 48 of 182^2 (runtime-length FFTs) 986 -> 118 us.
#include <cfloat>

#include "dft.hpp"
#include "gen_fft.hpp"
#include "internal.hpp"
#include "passes.hpp"

namespace mtd {

// sample held by position m of the reordered line (C even)
__device__ __forceinline__ int dct_src(int m, int C) { return m < C / 2 ? 2 * m : 2 * (C - 1 - m) + 1; }

// exp(i atan2(u.y, u.x)) without the angle: u / |u|. Outside the range where
// |u|^2 is a normal float (and for zeros, infinities and NaN) u is brought
// into range first, so that every value gives what the angle would.
__device__ __forceinline__ float2 unit_phasor(float2 u) {
  float m = u.x * u.x + u.y * u.y;
  if (!(m > FLT_MIN && m < FLT_MAX)) {
    if (m != m) return make_float2(m, m);
    const float s = fmaxf(fabsf(u.x), fabsf(u.y));
    if (s == 0.f) return make_float2(copysignf(1.f, u.x), u.y);
    if (s > FLT_MAX) {
      u = make_float2(copysignf(fabsf(u.x) > FLT_MAX ? 1.f : 0.f, u.x),
                      copysignf(fabsf(u.y) > FLT_MAX ? 1.f : 0.f, u.y));
    } else {
      const int e = -ilogbf(s);
      u = make_float2(ldexpf(u.x, e), ldexpf(u.y, e));
    }
    m = u.x * u.x + u.y * u.y;
  }
  const float r = __builtin_amdgcn_rsqf(m);
  return make_float2(u.x * r, u.y * r);
}

// derivative spectrum in the reordered line's terms: W[k] from V[k] and
// V[C-k]; tw4[j] = exp(-2 pi i j / 4C)
__device__ __forceinline__ float2 deriv_bin(float2 V, float2 Vr, int k, int C,
                                            const float2* __restrict__ tw4) {
  const float2 e = tw4[2 * k];  // exp(-i pi k / C)
  const float a = (float)(C - 2 * k) / (float)C;
  // a V - conj(e) Vr
  const float sx = a * V.x - (e.x * Vr.x + e.y * Vr.y);
  const float sy = a * V.y - (e.x * Vr.y - e.y * Vr.x);
  const float w = (float)(3.14159265358979323846 / 2.0) / (float)C;
  return make_float2(w * sy, -w * sx);
}

// P = e^{-it} V[k] and Q = e^{it} V[C-k], e = e^{-it}
__device__ __forceinline__ float2 dct_p(float2 V, float2 e) { return cmul(V, e); }
__device__ __forceinline__ float2 dct_q(float2 Vr, float2 e) {
  return make_float2(Vr.x * e.x + Vr.y * e.y, Vr.y * e.x - Vr.x * e.y);
}

// Bin (kx, ky) of the integration: from P and Q of the packed row transform
// (real part: DST-II along x of gx's y-cosine terms, imaginary part: DCT-II
// along x of gy's y-sine terms), the potential's cosine coefficients at kx and
// at C - kx, and the inverse transform's input e^{it} (Y[kx] - i Y[C-kx]).
__device__ __forceinline__ float2 poisson_bin(float2 P, float2 Q, float2 e, int kx, int ky, int C) {
  const float fx = (float)kx, fy = (float)ky, fr = (float)(C - kx);
  const float s = (float)(-1.0 / (2.0 * 3.14159265358979323846)) / (float)C;
  float y0 = 0.f, y1 = 0.f;
  if (kx | ky) y0 = s * ((fy - fx) * P.y + (fy + fx) * Q.y) / (fx * fx + fy * fy);
  if (kx) y1 = s * ((fy + fr) * P.x - (fy - fr) * Q.x) / (fr * fr + fy * fy);
  // e^{it} = conj(e); times (y0 - i y1)
  return make_float2(e.x * y0 - e.y * y1, -e.y * y0 - e.x * y1);
}

// Moves bins from Fft2's output layout (threads n2 < L1, u[k2] at k = n2 +
// L1 k2) to its input layout, each with its mirror bin: v[n1] at k = L2 n1 +
// n2, r[n1] at (C - k) mod C. Starts and ends with a barrier.
template <int C, class X>
__device__ __forceinline__ void bins_to_input(const float2 (&u)[Fft2<C, false>::L2],
                                              float2 (&v)[Fft2<C, false>::L1],
                                              float2 (&r)[Fft2<C, false>::L1], int n2, X x) {
  constexpr int L1 = Fft2<C, false>::L1, L2 = Fft2<C, false>::L2;
#pragma unroll
  for (int part = 0; part < 2; ++part) {
    __syncthreads();
    if (n2 < L1) {
#pragma unroll
      for (int k2 = 0; k2 < L2; ++k2) *x.lin(n2 + L1 * k2) = part ? u[k2].y : u[k2].x;
    }
    __syncthreads();
#pragma unroll
    for (int n1 = 0; n1 < L1; ++n1) {
      const int k = L2 * n1 + n2, m = k ? C - k : 0;
      (part ? v[n1].y : v[n1].x) = *x.lin(k);
      (part ? r[n1].y : r[n1].x) = *x.lin(m);
    }
  }
  __syncthreads();
}

// the line of phasors z (input layout, reordered) -> Im(dZ conj Z) without
// the odd samples' sign, at the same positions. v and u: work registers.
template <int C, class X>
__device__ __forceinline__ void line_gradient(const float2 (&z)[Fft2<C, false>::L1],
                                              float (&g)[Fft2<C, false>::L1], int n2, X x,
                                              const float2* __restrict__ tw,
                                              const float2* __restrict__ tw4) {
  using F = Fft2<C, false>;
  using B = Fft2<C, true>;
  float2 v[F::L1], u[F::L2];
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1) v[n1] = z[n1];
  F::run(v, u, n2, x, tw);
  {
    float2 r[F::L1];
    bins_to_input<C>(u, v, r, n2, x);
#pragma unroll
    for (int n1 = 0; n1 < F::L1; ++n1) v[n1] = deriv_bin(v[n1], r[n1], F::L2 * n1 + n2, C, tw4);
  }
  B::run(v, u, n2, x, tw);
  fft2_relayout<C>(u, v, n2, x);
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1) g[n1] = v[n1].y * z[n1].x - v[n1].x * z[n1].y;
}

// Column blocks: NC adjacent columns, the most of 32 (where it divides C), 16 and
// 8 that keep the block within MAXT threads (the last block may run past C). The
// gradient passes hold a line's phasors beside a transform: waves per SIMD
// that leave nearly all of it in registers (at 4 waves, crops of 160 to 256 spilled up
// to 138 of them; the column pass still keeps 16 bytes a thread in scratch at 128,
// 48 at 192, 12 at 250, 148 and 184 at 224 and 256), in blocks of at most 256 threads so that 3 fit: with 16 columns a
// 250-line block had 7 waves of the CU's 12, and one block was all that fit
// (300 crops: 321 -> 247 us with 8).
template <int C, int MAXT>
constexpr int unw_nc() {
  constexpr int T = Fft2<C, false>::T;
  return 32 * T <= MAXT && C % 32 == 0 ? 32 : 16 * T <= MAXT ? 16 : 8;
}
template <int C, int MAXT>
constexpr int unw_threads() {
  return unw_nc<C, MAXT>() * Fft2<C, false>::T;
}
template <int C>
constexpr int unw_waves() {
  return C <= 128 ? 4 : C <= 256 ? 3 : 2;
}
constexpr int kUnwGrad = 256, kUnwOut = 512;  // thread caps of passes B and D

// pass A: rows of the U frame, U[y][x] = IU[(y + C/2) % C][(x + C/2) % C]
template <int C>
__global__ void __launch_bounds__(256, unw_waves<C>())
k_unw_gx(const float2* __restrict__ iu, const float2* __restrict__ tw,
         const float2* __restrict__ tw4, float* __restrict__ gx) {
  using F = Fft2<C, false>;
  constexpr int NT = rows_nt<C>();
  __shared__ float lds[NT * F::LDS_ROW];
  const int2 ab = xcd_block();
  const int a = ab.x, t = threadIdx.x / F::T, n2 = threadIdx.x % F::T;
  const int y = ab.y * NT + t;
  const float2* row = iu + ((size_t)a * C + (y + C / 2) % C) * C;
  float2 z[F::L1];
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1)
    z[n1] = unit_phasor(row[(dct_src(F::L2 * n1 + n2, C) + C / 2) % C]);
  float g[F::L1];
  line_gradient<C>(z, g, n2, typename F::Row{lds + t * F::LDS_ROW}, tw, tw4);
  float* o = gx + ((size_t)a * C + y) * C;
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1) {
    const int m = F::L2 * n1 + n2;
    o[dct_src(m, C)] = m < C / 2 ? g[n1] : -g[n1];
  }
}

// pass B: columns; H[ky][x] = (DCT-II along y of gx, DST-II along y of gy)
template <int C>
__global__ void __launch_bounds__((unw_threads<C, kUnwGrad>()), unw_waves<C>())
k_unw_gy(const float2* __restrict__ iu, const float* __restrict__ gx,
         const float2* __restrict__ tw, const float2* __restrict__ tw4, float2* __restrict__ H) {
  using F = Fft2<C, false>;
  constexpr int NC = unw_nc<C, kUnwGrad>();
  __shared__ float lds[NC * F::LDS_COL];
  const int2 ab = xcd_block();
  const int a = ab.x, cl = threadIdx.x % NC, n2 = threadIdx.x / NC;
  const int c = ab.y * NC + cl;
  const bool live = C % NC == 0 || c < C;
  const int cc = live ? c : C - 1;
  const typename F::template Col<NC> x{lds + cl};
  const float2* col = iu + (size_t)a * C * C + (cc + C / 2) % C;
  const float* gcol = gx + (size_t)a * C * C + cc;
  float2 z[F::L1];
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1)
    z[n1] = unit_phasor(col[(size_t)((dct_src(F::L2 * n1 + n2, C) + C / 2) % C) * C]);
  float g[F::L1];
  line_gradient<C>(z, g, n2, x, tw, tw4);
  // gy's odd samples carry -1 twice: the derivative's and the DST's
  float2 v[F::L1], u[F::L2];
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1)
    v[n1] = make_float2(gcol[(size_t)dct_src(F::L2 * n1 + n2, C) * C], g[n1]);
  F::run(v, u, n2, x, tw);
  float2 r[F::L1];
  bins_to_input<C>(u, v, r, n2, x);
  if (!live) return;
  float2* o = H + (size_t)a * C * C + c;
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1) {
    const int k = F::L2 * n1 + n2;
    const float2 e = tw4[k];
    const float2 P = dct_p(v[n1], e), Q = dct_q(r[n1], e);
    o[(size_t)k * C] = make_float2(0.5f * (P.x + Q.x), 0.5f * (P.x - Q.x));
  }
}

// pass C: rows (ky); R[ky][x]
template <int C>
__global__ void __launch_bounds__(256, unw_waves<C>())
k_unw_poisson(const float2* __restrict__ H, const float2* __restrict__ tw,
              const float2* __restrict__ tw4, float* __restrict__ R) {
  using F = Fft2<C, false>;
  using B = Fft2<C, true>;
  constexpr int NT = rows_nt<C>();
  __shared__ float lds[NT * F::LDS_ROW];
  const int2 ab = xcd_block();
  const int a = ab.x, t = threadIdx.x / F::T, n2 = threadIdx.x % F::T;
  const int ky = ab.y * NT + t;
  const typename F::Row x{lds + t * F::LDS_ROW};
  const float2* h = H + ((size_t)a * C + ky) * C;
  float2 v[F::L1], u[F::L2];
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1) {
    const int m = F::L2 * n1 + n2;
    v[n1] = h[dct_src(m, C)];
    if (m >= C / 2) v[n1].x = -v[n1].x;
  }
  F::run(v, u, n2, x, tw);
  {
    float2 r[F::L1];
    bins_to_input<C>(u, v, r, n2, x);
#pragma unroll
    for (int n1 = 0; n1 < F::L1; ++n1) {
      const int k = F::L2 * n1 + n2;
      const float2 e = tw4[k];
      v[n1] = poisson_bin(dct_p(v[n1], e), dct_q(r[n1], e), e, k, ky, C);
    }
  }
  B::run(v, u, n2, x, tw);
  if (n2 < F::L1) {
    float* o = R + ((size_t)a * C + ky) * C;
#pragma unroll
    for (int k2 = 0; k2 < F::L2; ++k2) o[dct_src(n2 + F::L1 * k2, C)] = u[k2].x;
  }
}

// pass D: pairs of columns; the phase phu[y][x] of the U frame
template <int C>
__global__ void __launch_bounds__((unw_threads<C, kUnwOut>()), 4)
k_unw_out(const float* __restrict__ R, const float2* __restrict__ tw,
          const float2* __restrict__ tw4, float* __restrict__ phu) {
  using F = Fft2<C, true>;
  constexpr int NC = unw_nc<C, kUnwOut>();
  __shared__ float lds[NC * F::LDS_COL];
  const int2 ab = xcd_block();
  const int a = ab.x, cl = threadIdx.x % NC, n2 = threadIdx.x / NC;
  const int c = ab.y * NC + cl;  // columns 2c, 2c + 1
  const bool live = c < C / 2;
  const float2* q = (const float2*)(R + (size_t)a * C * C) + (live ? c : 0);
  float2 v[F::L1], u[F::L2];
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1) {
    const int k = F::L2 * n1 + n2;
    const float2 y0 = q[(size_t)k * (C / 2)];
    const float2 y1 = k ? q[(size_t)(C - k) * (C / 2)] : make_float2(0.f, 0.f);
    v[n1] = dct_q(make_float2(y0.x + y1.y, y0.y - y1.x), tw4[k]);
  }
  F::run(v, u, n2, typename F::template Col<NC>{lds + cl}, tw);
  if (!live || n2 >= F::L1) return;
  float2* o = (float2*)(phu + (size_t)a * C * C) + c;
#pragma unroll
  for (int k2 = 0; k2 < F::L2; ++k2)
    o[(size_t)dct_src(n2 + F::L1 * k2, C) * (C / 2)] = u[k2];
}

template <int C>
static hipError_t unwrap_c(const float2* iu, int A, const float2* tw, const float2* tw4,
                           float* gx, float2* H, float* phu, hipStream_t s) {
  constexpr int NB = unw_nc<C, kUnwGrad>(), ND = unw_nc<C, kUnwOut>();
  {
    Timed tm("unwrap_gx", s);
    hipLaunchKernelGGL((k_unw_gx<C>), rows_grid<C>(A), rows_block<C>(), 0, s, iu, tw, tw4, gx);
  }
  {
    Timed tm("unwrap_gy", s);
    hipLaunchKernelGGL((k_unw_gy<C>), dim3((C + NB - 1) / NB, A),
                       dim3((unw_threads<C, kUnwGrad>())), 0, s, iu, gx, tw, tw4, H);
  }
  {
    Timed tm("unwrap_poisson", s);
    hipLaunchKernelGGL((k_unw_poisson<C>), rows_grid<C>(A), rows_block<C>(), 0, s, H, tw, tw4, gx);
  }
  Timed tm("unwrap_out", s);
  hipLaunchKernelGGL((k_unw_out<C>), dim3((C / 2 + ND - 1) / ND, A),
                     dim3((unw_threads<C, kUnwOut>())), 0, s, gx, tw, tw4, phu);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Crop sides without a compiled C-point FFT: the same four passes with the
// runtime-length FFTs, nl lines in LDS per block (gen_fft.hpp), a line's
// positions reordered on load.
// ---------------------------------------------------------------------------
// Pair pass over bins k and C - k of each line, in place: fn(line, k, V[k],
// V[C-k]) gives both bins' new values (k = 0 and C/2 are their own mirrors).
template <class Fn>
__device__ __forceinline__ void gen_pairs(const GenLines& x, int C, Fn&& fn) {
  const int l = threadIdx.x & (x.nl() - 1);
  for (int k = threadIdx.x >> x.lnl; k <= C / 2; k += blockDim.x >> x.lnl) {
    const int m = k ? C - k : 0;
    const float2 a = x.get(l, k), b = x.get(l, m);
    x.set(l, k, fn(l, k, a, b));
    if (m != k) x.set(l, m, fn(l, m, b, a));
  }
  __syncthreads();
}

template <bool ROWS>
__global__ void __launch_bounds__(kGenThreads, 4)
k_unw_grad_gen(const float2* __restrict__ iu, GenPlan p, int C, const float2* __restrict__ tw4,
               float* __restrict__ gx, float2* __restrict__ H, int lnl, int pitch) {
  extern __shared__ float2 gen_lds[];
  const int2 ab = xcd_block();
  const int a = ab.x, line0 = ab.y << lnl;
  if (line0 >= C) return;
  const int nact = min(1 << lnl, C - line0);
  const GenLines x{(gen_lds_v2*)gen_lds, lnl, pitch};
  const float2* iu_a = iu + (size_t)a * C * C;
  const size_t base = (size_t)a * C * C;
  const int h = C / 2;
  auto wrap = [C](int i) { return i < C ? i : i - C; };
  auto phasor = [&](int l, int m) {
    const int i = wrap(dct_src(m, C) + h), j = wrap(line0 + l + h);
    return unit_phasor(ROWS ? iu_a[(size_t)j * C + i] : iu_a[(size_t)i * C + j]);
  };
  gen_load<ROWS, 4>(lnl, C, [&](int l, int m) { return phasor(min(l, nact - 1), m); },
                    [&](int l, int m, float2 v) { x.set(l, m, v); });
  __syncthreads();
  // forward, derivative, backward (through the exchange of parts), and for
  // the columns the packed forward transform
#pragma unroll 1
  for (int pass = 0; pass < (ROWS ? 2 : 3); ++pass) {
    gen_fft<false, false>(x, p);
    if (pass == 0) {
      gen_pairs(x, C, [&](int, int k, float2 V, float2 Vr) {
        return gen_swap(deriv_bin(V, Vr, k, C, tw4));
      });
    } else if (pass == 1) {
      gen_each<ROWS>(lnl, C, [&](int l, int m) {
        if (l >= nact) return;
        const float2 w = gen_swap(x.get(l, m)), z = phasor(l, m);
        const float g = w.y * z.x - w.x * z.y;
        const int n = dct_src(m, C);
        if (ROWS) gx[base + (size_t)(line0 + l) * C + n] = m < h ? g : -g;
        else x.set(l, m, make_float2(gx[base + (size_t)n * C + line0 + l], g));
      });
      __syncthreads();
    } else {
      gen_pairs(x, C, [&](int, int k, float2 V, float2 Vr) {
        const float2 e = tw4[k], P = dct_p(V, e), Q = dct_q(Vr, e);
        return make_float2(0.5f * (P.x + Q.x), 0.5f * (P.x - Q.x));
      });
      gen_each<ROWS>(lnl, C, [&](int l, int k) {
        if (l < nact) H[base + (size_t)k * C + line0 + l] = x.get(l, k);
      });
    }
  }
}

__global__ void __launch_bounds__(kGenThreads, 4)
k_unw_poisson_gen(const float2* __restrict__ H, GenPlan p, int C, const float2* __restrict__ tw4,
                  float* __restrict__ out, int lnl, int pitch) {
  extern __shared__ float2 gen_lds[];
  const int2 ab = xcd_block();
  const int a = ab.x, line0 = ab.y << lnl;
  if (line0 >= C) return;
  const int nact = min(1 << lnl, C - line0);
  const GenLines x{(gen_lds_v2*)gen_lds, lnl, pitch};
  const size_t base = ((size_t)a * C + line0) * C;
  gen_load<true, 8>(
      lnl, C,
      [&](int l, int m) { return H[base + (size_t)min(l, nact - 1) * C + dct_src(m, C)]; },
      [&](int l, int m, float2 v) { x.set(l, m, make_float2(m < C / 2 ? v.x : -v.x, v.y)); });
  __syncthreads();
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    gen_fft<false, false>(x, p);
    if (pass == 0) {
      gen_pairs(x, C, [&](int l, int k, float2 V, float2 Vr) {
        const float2 e = tw4[k];
        return gen_swap(poisson_bin(dct_p(V, e), dct_q(Vr, e), e, k, line0 + l, C));
      });
    }
  }
  gen_each<true>(lnl, C, [&](int l, int m) {
    if (l < nact) out[base + (size_t)l * C + dct_src(m, C)] = gen_swap(x.get(l, m)).x;
  });
}

struct UnwOutGenOp {  // pairs of columns (2 col, 2 col + 1)
  const float* R;
  const float2* tw4;
  float* phu;
  int C;
  __device__ void begin(int) {}
  __device__ float2 load(int a, int col, int k) const {
    const float2* q = (const float2*)(R + (size_t)a * C * C) + col;
    const float2 y0 = q[(size_t)k * (C / 2)];
    const float2 y1 = k ? q[(size_t)(C - k) * (C / 2)] : make_float2(0.f, 0.f);
    return dct_q(make_float2(y0.x + y1.y, y0.y - y1.x), tw4[k]);
  }
  __device__ void store(int a, int col, int m, float2 v) const {
    ((float2*)(phu + (size_t)a * C * C))[(size_t)dct_src(m, C) * (C / 2) + col] = v;
  }
};

static hipError_t unwrap_gen(int C, const float2* iu, int A, const GenPlan& p, const float2* tw4,
                             float* gx, float2* H, float* phu, hipStream_t s) {
  const int lr = gen_lnl(p, true, C, A), lc = gen_lnl(p, false, C, A);
  const int pr = gen_pitch(lr, true), pc = gen_pitch(lc, false);
  const size_t mr = (size_t)pr * p.W * sizeof(float2), mc = (size_t)pc * p.W * sizeof(float2);
  const dim3 gr(gen_groups(C, lr), A), gc(gen_groups(C, lc), A);
  const dim3 br(gen_threads(p, lr)), bc(gen_threads(p, lc));
  {
    Timed tm("unwrap_gx", s);
    hipLaunchKernelGGL((k_unw_grad_gen<true>), gr, br, mr, s, iu, p, C, tw4, gx, H, lr, pr);
  }
  {
    Timed tm("unwrap_gy", s);
    hipLaunchKernelGGL((k_unw_grad_gen<false>), gc, bc, mc, s, iu, p, C, tw4, gx, H, lc, pc);
  }
  {
    Timed tm("unwrap_poisson", s);
    hipLaunchKernelGGL(k_unw_poisson_gen, gr, br, mr, s, H, p, C, tw4, gx, lr, pr);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  Timed tm("unwrap_out", s);
  return launch_gen<true, false>(UnwOutGenOp{gx, tw4, phu, C}, p, C / 2, A, s);
}

#define MTD_UNWRAP_SIZES(X) \
  X(16) X(32) X(64) X(128) X(160) X(192) X(224) X(250) X(256) X(288) X(320) X(352) X(384) \
  X(512)

hipError_t launch_unwrap(int C, const float2* iu, int A, const FftTab& ftC, const float2* tw4,
                         void* scratch, float* phu, hipStream_t s) {
  if (A <= 0) return hipSuccess;
  float2* H = (float2*)scratch;
  float* gx = (float*)(H + (size_t)A * C * C);
  switch (C) {
#define X(n) case n: return unwrap_c<n>(iu, A, ftC.tw, tw4, gx, H, phu, s);
    MTD_UNWRAP_SIZES(X)
#undef X
  }
  if (!ftC.gen) return hipErrorInvalidValue;
  return unwrap_gen(C, iu, A, *ftC.gen, tw4, gx, H, phu, s);
}

bool unwrap_len_supported(int C) {
  switch (C) {
#define X(n) case n: return true;
    MTD_UNWRAP_SIZES(X)
#undef X
  }
  return false;
}

size_t unwrap_scratch_bytes(int C, int A) {
  // H (float2), gx, then the integral's rows (float), C^2 each
  return (size_t)(A > 0 ? A : 1) * C * C * (sizeof(float2) + sizeof(float));
}

}  // namespace mtd
