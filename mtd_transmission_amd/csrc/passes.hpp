// Generic batched 1-D FFT passes over stacks of lines, parameterised by an
// operation object that maps (batch, line, element) to memory on load and on
// store. Transforms use the two-step register FFT (fft_reg.hpp): inputs are
// loaded straight from global memory into registers and outputs stored
// straight from registers, with one LDS transpose in between.
//   rows:    each transform is one contiguous line; NT lines per block.
//   columns: NC adjacent columns per block; lane = column fastest, so every
//            load and store touches NC contiguous elements of a row.
#pragma once
#include <type_traits>
#include <utility>

#include "fft_reg.hpp"

namespace mtd {

// A side length fixed at compile time (N > 0: folds into the index
// arithmetic of the compiled lengths) or held at run time (N == 0: the
// runtime-length path). Converts to int.
template <int N>
struct Dim {
  __host__ __device__ constexpr Dim(int = N) {}
  __host__ __device__ constexpr operator int() const { return N; }
};
template <>
struct Dim<0> {
  int v = 0;
  __host__ __device__ constexpr Dim(int x = 0) : v(x) {}
  __host__ __device__ constexpr operator int() const { return v; }
};

// Raw buffer view of one device array (at most 2 GiB). A load takes a 32-bit
// per-lane byte offset and a uniform byte offset held in a scalar register,
// so a run of loads at uniform strides keeps one address register in place of
// a 64-bit address per load. Offsets at or beyond `bytes` read as zero (the
// buffer range check).
struct BufView {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ BufView(const void* p, unsigned bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes,
                                            0x00020000)) {}
  __device__ __forceinline__ float2 f2(unsigned lane_bytes, unsigned uni_bytes) const {
    return __builtin_bit_cast(float2,
                              __builtin_amdgcn_raw_buffer_load_b64(r, lane_bytes, uni_bytes, 0));
  }
};

// Row passes: NT transforms per block (at most 256 threads, 64 KiB LDS).
template <int L>
constexpr int rows_nt() {
  constexpr int by_thr = 256 / Fft2<L, false>::T;
  constexpr int by_lds = kLdsBlockMax / (Fft2<L, false>::LDS_ROW * 4);
  return divisor_le(L, by_thr < by_lds ? by_thr : by_lds);
}
// Column passes: NC adjacent columns per block, up to 32 (128-byte segments
// even for float outputs), at most 1024 threads and 64 KiB LDS; lines of
// 513-1023 keep 256 threads (their register FFTs allow 3 waves per SIMD,
// which 4-wave blocks fill), lines from 1024 take 512 (2 waves per SIMD:
// one 8-wave block per CU either way, and twice the row segment).
// MAXT lowers the thread cap (see op_col_threads).
template <int L, int MAXT = 1024>
constexpr int cols_nc() {
  constexpr int cap = L >= 1024 ? 512 : L > 512 ? 256 : 1024;
  constexpr int by_thr = (MAXT < cap ? MAXT : cap) / Fft2<L, false>::T;
  constexpr int by_lds = kLdsBlockMax / (Fft2<L, false>::LDS_COL * 4);
  constexpr int m = by_thr < by_lds ? by_thr : by_lds;
  return divisor_le(L, m < 32 ? m : 32);
}
template <int L, int MAXT = 1024>
constexpr int cols_threads() {
  return cols_nc<L, MAXT>() * Fft2<L, false>::T;
}

// An operation may cap the threads of its column blocks with a static
// kColThreads: two half-size blocks per CU overlap one block's barriers with
// the other's memory traffic, which pays where the stores are whole 128-byte
// lines either way (complex outputs) but not for float outputs.
template <class Op, class = void>
struct op_col_threads {
  static constexpr int value = 1024;
};
template <class Op>
struct op_col_threads<Op, std::void_t<decltype(Op::kColThreads)>> {
  static constexpr int value = Op::kColThreads;
};
// Column blocks are up to 1024 threads; ask the compiler for at least 4
// waves per SIMD (at most 128 VGPRs) so that a CU keeps 16 waves in flight,
// 3 for lines longer than 512 and 2 from 1024 (a 32 + 32 point register FFT
// needs about 170 VGPRs: 3 waves would spill).
// (HIP's second __launch_bounds__ argument is amdgpu_waves_per_eu.)
template <int L>
constexpr int col_waves_per_simd() {
  return L >= 1024 ? 2 : L > 512 ? 3 : 4;
}

// Tile variants TV of the passes (a schedule the autotuner picks; every
// variant does the same arithmetic in the same order, so results are
// identical): TV 0 the shapes above; TV 1 half the lines (rows) or columns
// per block, twice the blocks; TV 2 twice the columns per block where the
// block still fits one CU at the pass's waves per SIMD, its LDS within
// 64 KiB and the width within 32 and dividing L (else TV 0's width).
template <int L, int TV>
constexpr int rows_nt_tv() {
  constexpr int nt = rows_nt<L>();
  return TV == 1 && nt % 2 == 0 ? nt / 2 : nt;
}
template <int L, int MAXT, int TV>
constexpr int cols_nc_tv() {
  constexpr int nc = cols_nc<L, MAXT>();
  constexpr int T = Fft2<L, false>::T;
  constexpr int waves = col_waves_per_simd<L>();
  if constexpr (TV == 1) {
    return nc % 2 == 0 ? nc / 2 : nc;
  } else if constexpr (TV == 2) {
    constexpr int w = 2 * nc;
    constexpr bool fits = w <= 32 && L % w == 0 && w * T <= 1024 && w * T <= 256 * waves &&
                          w * Fft2<L, false>::LDS_COL * 4 <= kLdsBlockMax;
    return fits ? w : nc;
  }
  return nc;
}

// Workgroups are dealt round-robin to the 8 XCDs in dispatch order (linear
// id, x fastest). Renumber them so that XCD k runs the k-th eighth of the
// line/column groups of every batch, in order: neighbouring column groups
// share that XCD's L2 for the 128-byte lines they split, and every batch
// (e.g. a z plane, some of which may be skipped) is spread over all XCDs.
// A bijection when gridDim.x is a multiple of 8; the identity otherwise.
__device__ __forceinline__ int2 xcd_block() {
  const int gx = gridDim.x;
  if (gx % 8) return make_int2(blockIdx.y, blockIdx.x);
  const int id = blockIdx.x + blockIdx.y * gx;
  const int per = gx / 8, n = id / 8;
  return make_int2(n / per, (id % 8) * per + n % per);
}

// An operation may define skip(batch): the whole batch is then left alone
// (neither read nor written) when it returns true.
template <class Op, class = void>
struct has_skip : std::false_type {};
template <class Op>
struct has_skip<Op, std::void_t<decltype(std::declval<const Op&>().skip(0))>>
    : std::true_type {};

template <class Op>
__device__ __forceinline__ bool skip_batch(const Op& op, int a) {
  if constexpr (has_skip<Op>::value) return op.skip(a);
  return false;
}

// An operation may define line(batch, line), called once per transform
// before its loads, to hoist per-line work out of load().
template <class Op, class = void>
struct has_line : std::false_type {};
template <class Op>
struct has_line<Op, std::void_t<decltype(std::declval<Op&>().line(0, 0))>> : std::true_type {};

// An operation with a static constexpr bool kScans = true defines keep(batch,
// first line, lines, any), called once by every thread of a row block after its
// loads, with whether any value of the block's lines is not zero (NaN is not
// zero): the block then leaves its lines alone when it returns false. The
// compiled row pass scans what raw(batch, line, element) reads, and makes the
// transform's input of it with value(raw, part, batch, line, element) only if the
// block goes on. part(batch, line, element) is the input's other part, read by the
// waves that found something (1 for the others); where flags() holds, store_flags(batch, first line, lines, bytes) gets
// a byte per element, 1 where the input's real part is not zero (nullptr:
// nowhere).
template <class Op, class = void>
struct op_scans : std::false_type {};
template <class Op>
struct op_scans<Op, std::void_t<decltype(Op::kScans)>>
    : std::integral_constant<bool, Op::kScans> {};

template <int L, bool INV, class Op, int TV = 0>
__global__ void __launch_bounds__(256) k_rows(Op op) {
  using F = Fft2<L, INV>;
  constexpr int NT = rows_nt_tv<L, TV>();
  __shared__ __attribute__((aligned(16))) float lds[NT * F::LDS_ROW];
  const int2 ab = xcd_block();
  const int a = ab.x;
  if (skip_batch(op, a)) return;  // block-uniform, before the barrier
  const int r = threadIdx.x / F::T, n2 = threadIdx.x % F::T;
  const int line = ab.y * NT + r;
  op.begin(a);
  if constexpr (has_line<Op>::value) op.line(a, line);
  float2 v[F::L1], u[F::L2];
  if constexpr (!op_scans<Op>::value) {
#pragma unroll
    for (int n1 = 0; n1 < F::L1; ++n1) v[n1] = op.load(a, line, F::L2 * n1 + n2);
  } else {
    bool any = false;
#pragma unroll
    for (int n1 = 0; n1 < F::L1; ++n1) v[n1] = op.raw(a, line, F::L2 * n1 + n2);
#pragma unroll
    for (int n1 = 0; n1 < F::L1; ++n1) any = any || v[n1].x != 0.f || v[n1].y != 0.f;
    int part[F::L1];
    if (__any(any)) {  // ahead of the barrier: one more trip to memory after it otherwise
#pragma unroll
      for (int n1 = 0; n1 < F::L1; ++n1) part[n1] = op.part(a, line, F::L2 * n1 + n2);
    } else {
#pragma unroll
      for (int n1 = 0; n1 < F::L1; ++n1) part[n1] = 1;
    }
    any = __syncthreads_or(any);
    const bool flags = op.flags();  // uniform
    if (flags && !any) op.store_flags(a, ab.y * NT, NT, nullptr);
    if (!op.keep(a, ab.y * NT, NT, any)) return;  // block-uniform
#pragma unroll
    for (int n1 = 0; n1 < F::L1; ++n1) v[n1] = op.value(v[n1], part[n1], a, line, F::L2 * n1 + n2);
    if (flags) {
      uint8_t* f = (uint8_t*)lds;
#pragma unroll
      for (int n1 = 0; n1 < F::L1; ++n1) f[r * L + F::L2 * n1 + n2] = v[n1].x != 0.f;
      __syncthreads();
      op.store_flags(a, ab.y * NT, NT, f);
      __syncthreads();
    }
  }
  F::run(v, u, n2, typename F::Row{lds + r * F::LDS_ROW}, op.tw);
  if (n2 < F::L1) {
#pragma unroll
    for (int k2 = 0; k2 < F::L2; ++k2) op.store(a, line, n2 + F::L1 * k2, u[k2]);
  }
}

template <int L, bool INV, class Op, int TV = 0>
__global__ void __launch_bounds__((cols_nc_tv<L, op_col_threads<Op>::value, TV>() *
                                   Fft2<L, false>::T),
                                  col_waves_per_simd<L>()) k_cols(Op op) {
  using F = Fft2<L, INV>;
  constexpr int NC = cols_nc_tv<L, op_col_threads<Op>::value, TV>();
  __shared__ float lds[NC * F::LDS_COL];
  const int2 ab = xcd_block();
  const int a = ab.x, c0 = ab.y * NC;
  if (skip_batch(op, a)) return;  // block-uniform, before the barrier
  const int c = threadIdx.x % NC, n2 = threadIdx.x / NC;
  op.begin(a);
  float2 v[F::L1], u[F::L2];
#pragma unroll
  for (int n1 = 0; n1 < F::L1; ++n1) v[n1] = op.load(a, c0 + c, F::L2 * n1 + n2);
  F::run(v, u, n2, typename F::template Col<NC>{lds + c}, op.tw);
  if (n2 < F::L1) {
#pragma unroll
    for (int k2 = 0; k2 < F::L2; ++k2) op.store(a, c0 + c, n2 + F::L1 * k2, u[k2]);
  }
}

// The column pass on the balanced transform (Fft2B): NC adjacent columns per
// block (32: 128-byte rows even for float outputs), T = L1 threads per
// column, compiled for 4 waves per SIMD: two blocks per CU at L = 512 (512
// threads, 64 KiB), where k_cols runs one 1024-thread block and leaves half
// of each column's threads idle in its second step. An operation opts in with
// a static constexpr bool kBalancedCols = true.
template <class Op, class = void>
struct op_cols_balanced : std::false_type {};
template <class Op>
struct op_cols_balanced<Op, std::void_t<decltype(Op::kBalancedCols)>>
    : std::integral_constant<bool, Op::kBalancedCols> {};

template <int L>
constexpr int cols_b_nc() {
  return 32 * L * 4 <= kLdsBlockMax ? 32 : 16;
}
// lengths that take the balanced pass: L1 | L2 with L1 < L2, where Fft2
// idles half a line's threads in its second step. At L = 1024 (32 x 32, 16
// columns per block) it took 128 VGPRs with 12-19 spilled and was slower
// than k_cols (1024^3 z pass 4.4-5.05 -> 5.4 ms, y pass 1.08 -> 1.21 ms).
template <int L>
constexpr bool cols_b_fits() {
  constexpr int l1 = fft2_l1(L), l2 = fft2_l2(L), nc = cols_b_nc<L>();
  return l1 > 1 && l2 % l1 == 0 && l1 < l2 && L % nc == 0 && nc * L * 4 <= kLdsBlockMax &&
         64 / nc <= l1;
}
template <int L, bool INV, class Op>
__global__ void __launch_bounds__((cols_b_nc<L>() * Fft2B<L, false>::T), 4) k_cols_b(Op op) {
  using F = Fft2B<L, INV>;
  constexpr int NC = cols_b_nc<L>();
  __shared__ float lds[NC * L];
  const int2 ab = xcd_block();
  const int a = ab.x, c0 = ab.y * NC;
  if (skip_batch(op, a)) return;  // block-uniform, before the barrier
  const int c = threadIdx.x % NC, t = threadIdx.x / NC;
  op.begin(a);
  float2 v[F::L2];
#pragma unroll
  for (int m = 0; m < F::L2; ++m) v[m] = op.load(a, c0 + c, F::L1 * m + t);
  F::run(v, t, typename F::template Col<NC>{lds + c}, op.tw);
#pragma unroll
  for (int j = 0; j < F::R; ++j)
#pragma unroll
    for (int k1 = 0; k1 < F::L1; ++k1)
      op.store(a, c0 + c, F::R * t + j + F::L2 * k1, v[j * F::L1 + k1]);
}
template <int L>
inline dim3 cols_b_grid(int A) {
  return dim3(L / cols_b_nc<L>(), A);
}
template <int L>
inline dim3 cols_b_block() {
  return dim3(cols_b_nc<L>() * Fft2B<L, false>::T);
}

// The column pass of a transform whose input fills a band of its elements
// [op.lo, op.hi] (set by op.begin; load() gives zeros outside): the first radix
// R = cols_fold_r is taken by decimation in frequency, X[R*q + r] being the
// (L/R)-point transform over z mod L/R of x[z] exp(+-2 pi i r z / L), folded. A
// block loads its band once into registers (NB values a thread) and then runs R
// short transforms, so it holds 64 columns where the whole transform held 16 or
// 32: the stores, one plane after the other, become 256-byte pieces. For bands of
// cols_fold_narrow only; the others take the whole transform (folded from memory,
// read once per residue, they took longer: 640^3, band 0.43 of the height, z
// pass and all 2536 -> 3271 us, 1024^3 8676 -> 10297).
//
// The float outputs' piece is what bounds the height pass. Storing two V^3 float
// volumes column by column and reading a band of 0.295 V planes, with no
// transform, takes at V = 1024 4.8, 2.85 and 2.23 ms with 16, 32 and 64 columns
// a block (64-, 128- and 256-byte pieces), at V = 512 459, 254 and 241 us.
// The lengths it is built for: those whose L/R has a square split (all threads in
// both steps) and whose whole transform left 9 to 16 columns a block, and 448 and
// 512. Height pass alone at 4.7 to 8 bins per pupil radius (96 bins): 448^3 242 ->
// 202 us, 576^3 1077 -> 473, 640^3 1136 -> 607, 704^3 1567 -> 840, 768^3 2140 -> 969.
// 256, 320 and 384 have the square split too, with 32 columns a block as they are:
// with both launches (vol_z) they measured 34 -> 31, 78 -> 66 and 145 -> 132 us and are
// not built yet.
template <int L>
constexpr int cols_fold_r() {
  return L == 512 ? 2 : L == 576 ? 4 : L == 640 ? 10 : L == 704 ? 11 : L == 768 ? 3
         : L == 1024 ? 4 : L == 448 ? 7 : 1;
}
template <int L>
constexpr int cols_fold_nc() {
  return 64;
}
// registers for a band of 0.36 L: heights span 0.3135 L at 4 bins per pupil
// radius (the smallest volume) and NA / n0 = 0.9
template <int L>
constexpr int cols_fold_nb() {
  return (36 * L / 100 + Fft2<L / cols_fold_r<L>(), false>::T - 1) /
         Fft2<L / cols_fold_r<L>(), false>::T;
}
template <int L>
constexpr bool cols_fold_fits() {
  return cols_fold_r<L>() > 1;
}
// band elements [lo, hi] in the register path
template <int L>
__host__ __device__ constexpr bool cols_fold_narrow(int lo, int hi) {
  constexpr int T = Fft2<L / cols_fold_r<L>(), false>::T;
  return hi < lo || hi / T - (lo > 0 ? lo / T : 0) + 1 <= cols_fold_nb<L>();
}
template <int L>
constexpr int cols_fold_threads() {
  return cols_fold_nc<L>() * Fft2<L / cols_fold_r<L>(), false>::T;
}
template <int L, bool INV, class Op>
__global__ void __launch_bounds__(cols_fold_threads<L>(), 4) k_cols_fold(Op op) {
  constexpr int R = cols_fold_r<L>(), M = L / R, NC = cols_fold_nc<L>(), NB = cols_fold_nb<L>();
  using F = Fft2<M, INV>;
  constexpr int L1 = F::L1, L2 = F::L2, T = F::T;
  static_assert(L1 == L2 && NC == 64, "all threads in both steps, one column element a wave");
  __shared__ float lds[NC * F::LDS_COL];
  const int2 ab = xcd_block();
  const int a = ab.x, c0 = ab.y * NC;
  if (skip_batch(op, a)) return;  // block-uniform, before the barrier
  const int c = threadIdx.x % NC;
  // the wave's element: uniform, so every twiddle is a scalar load
  const int n2 = __builtin_amdgcn_readfirstlane(threadIdx.x / NC);
  op.begin(a);
  // input index z = T*(b + j) + n2; n1 = (b + j) mod L1: the rotation by b of
  // the first step's input is a phase on its output k1, W_L1^(b k1), which the
  // step twiddle takes along
  const int b = op.lo > 0 ? op.lo / T : 0;
  float2 e[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) e[j] = op.load_wave(a, c0, c, T * (b + j) + n2);
  // the table is constant: scalar loads
  typedef float v2f __attribute__((ext_vector_type(2)));
  const auto* tw = (const __attribute__((address_space(4))) v2f*)op.tw;
  const typename F::template Col<NC> x{lds + c};
#pragma unroll 1
  for (int r = 0; r < R; ++r) {
    float2 v[L1], u[L2];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const v2f q = tw[r * (T * (b + j) + n2) % L];
      const float2 w = make_float2(q.x, INV ? -q.y : q.y);
      const float2 t = cmul(e[j], w);
      if (j < L1) v[j] = t;
      else v[j % L1] = make_float2(v[j % L1].x + t.x, v[j % L1].y + t.y);
    }
#pragma unroll
    for (int j = NB; j < L1; ++j) v[j] = make_float2(0.f, 0.f);
    RegFFT<L1, INV>::run(v);
#pragma unroll
    for (int k1 = 1; k1 < L1; ++k1) {
      const v2f q = tw[R * ((n2 + T * b) * k1) % L];
      const float2 w = make_float2(q.x, INV ? -q.y : q.y);
      v[k1] = cmul(v[k1], w);
    }
    if (r) __syncthreads();  // the last residue's reads
#pragma unroll
    for (int k1 = 0; k1 < L1; ++k1) *x.at(k1, n2) = v[k1].x;
    __syncthreads();
#pragma unroll
    for (int n = 0; n < L2; ++n) u[n].x = *x.at(n2, n);
    __syncthreads();
#pragma unroll
    for (int k1 = 0; k1 < L1; ++k1) *x.at(k1, n2) = v[k1].y;
    __syncthreads();
#pragma unroll
    for (int n = 0; n < L2; ++n) u[n].y = *x.at(n2, n);
    RegFFT<L2, INV>::run(u);
#pragma unroll
    for (int k2 = 0; k2 < L2; ++k2) op.store_wave(a, c0, c, R * (n2 + L1 * k2) + r, u[k2]);
  }
}

// An operation may define mid_line(batch, line), called once per transform
// between the first transform and its mid() calls: per-line state that only
// mid() reads is then not held in registers through the first transform.
template <class Op, class = void>
struct has_mid_line : std::false_type {};
template <class Op>
struct has_mid_line<Op, std::void_t<decltype(std::declval<Op&>().mid_line(0, 0))>>
    : std::true_type {};

// Two chained transforms per row: the INV1 transform of the loaded line,
// op.mid(batch, line, element, value) on every output element, the values
// moved back to the input layout through the exchange storage, the INV2
// transform, op.store. The line set up by op.line(batch, line) is kept for
// the whole kernel (one line per NT-th of the block).
// waves per SIMD asked of the chained row pass: 4 (at most 128 VGPRs) for
// 128- and 256-point lines, which then fit without spilling (other lengths
// of that size would spill); the rest leave the register budget to the
// compiler
template <int L>
constexpr int rows2_waves_per_simd() {
  return (L == 128 || L == 256) ? 4 : 1;
}
template <int L, bool INV1, bool INV2, class Op>
__global__ void __launch_bounds__(256, rows2_waves_per_simd<L>()) k_rows2(Op op) {
  using F1 = Fft2<L, INV1>;
  using F2 = Fft2<L, INV2>;
  constexpr int NT = rows_nt<L>();
  __shared__ float lds[NT * F1::LDS_ROW];
  const int2 ab = xcd_block();
  const int a = ab.x;
  const int r = threadIdx.x / F1::T, n2 = threadIdx.x % F1::T;
  const int line = ab.y * NT + r;
  op.begin(a);
  op.line(a, line);
  float2 v[F1::L1], u[F1::L2];
#pragma unroll
  for (int n1 = 0; n1 < F1::L1; ++n1) v[n1] = op.load(a, line, F1::L2 * n1 + n2);
  const typename F1::Row x{lds + r * F1::LDS_ROW};
  F1::run(v, u, n2, x, op.tw);
  if constexpr (has_mid_line<Op>::value) op.mid_line(a, line);
  if (n2 < F1::L1) {
#pragma unroll
    for (int k2 = 0; k2 < F1::L2; ++k2) u[k2] = op.mid(a, line, n2 + F1::L1 * k2, u[k2]);
  }
  fft2_relayout<L>(u, v, n2, x);
  F2::run(v, u, n2, x, op.tw);
  if (n2 < F2::L1) {
#pragma unroll
    for (int k2 = 0; k2 < F2::L2; ++k2) op.store(a, line, n2 + F2::L1 * k2, u[k2]);
  }
}

template <int L, int TV = 0>
inline dim3 rows_grid(int A) {
  return dim3(L / rows_nt_tv<L, TV>(), A);
}
template <int L, int TV = 0>
inline dim3 rows_block() {
  return dim3(rows_nt_tv<L, TV>() * Fft2<L, false>::T);
}
template <int L, class Op = void, int TV = 0>
inline dim3 cols_grid(int A) {
  return dim3(L / cols_nc_tv<L, op_col_threads<Op>::value, TV>(), A);
}
template <int L, class Op = void, int TV = 0>
inline dim3 cols_block() {
  return dim3(cols_nc_tv<L, op_col_threads<Op>::value, TV>() * Fft2<L, false>::T);
}

}  // namespace mtd
