// Blocked QR and basis update of the batched FP64 low-rank additions, and the core
// product of additions with more columns than rows (gfx950).
//
// QR of a panel [A1 S1 | A2 S2] (m x K): a wave holds 16 of the columns in registers,
// as NT tiles of 16 x 16 in the layout of an MFMA result: lane (j, r), j = lane & 15,
// r = lane >> 4, element e of tile t is row 16 t + 4 r + e of column j.  In this layout
//   * a column's entries sit in one lane of each 16-lane row, so a Householder step
//     inside the 16 columns broadcasts the pivot column with DPP row_newbcast (as an
//     operand of the multiply-add) and sums over rows with two permlane swaps: no LDS
//     and no barrier in a panel;
//   * the registers are MFMA operands as they are (the sum over rows of a product
//     Y^T C may take the rows in any order), so the panel goes to the waves of the
//     later columns in compact WY form, C -= Y T^T (Y^T C), as 16 x 16 x 4 MFMA
//     products, and a basis update (I - Y T Y^T) [X; 0] likewise.
// Above 128 rows (up to 64 columns) two waves share the rows of 16 columns: one wave
// would need 128 registers for the panel alone.
// Outputs per addition: the reflectors Y (column-major, rows padded to 16, unit
// diagonal and zeros above stored), the panels' triangular factors T (16 x 16
// row-major), and R.
//
// Bound by the chain of the 16 dependent steps of a panel (about 800 cycles each:
// products, a reduction, rsq and rcp with their corrections, the update; with the
// exchange between two waves 1200) and the update of the next panel's columns; in
// large batches by FP64 issue (MFMA and vector units have the same FP64 rate).
// FP64 only: in FP32 the compact WY form (T, and one more rounding of T^T W) left an
// error of the sum of 2.2e-7 at m = 256, K = 32, singular values 10^(-i/2), against
// 1.8e-7 with a reflector at a time, which the additions in FP32 keep.
// Measured, QR of both panels and basis update with every column kept, us, these
// kernels / the unblocked ones (a reflector at a time over the whole panel, two barriers
// each):
//   m    K    additions   QR             update
//   64   16   40          12.5 / 18.6    5.8 / 14.2
//   64   128  165         95.0 / 325     23.1 / 123
//   128  32   300         56.7 / 71.8    22.9 / 77.4
//   256  16   40          18.9 / 23.6    9.0 / 18.6
//   256  64   165         146 / 191      78.1 / 182
//   256  128  4           202 / 264      105 / 289
#include <hip/hip_runtime.h>

#include <stdexcept>

#include "kernels.hpp"
#include "diag64.hpp"
#include "lr_items.hpp"

namespace frk {

namespace {

template <typename T>
struct Mma;
template <>
struct Mma<double> {
  using v4 = double __attribute__((ext_vector_type(4)));
  // D[i][j] of a result: lane j + 16 (i % 4), element i / 4
  static __device__ __forceinline__ int crow(int e, int r) { return 4 * e + r; }
  // the tile row that result row i stands for, so that lane row r, element e is row 4 r + e
  static __device__ __forceinline__ int irow(int i) { return 4 * (i & 3) + (i >> 2); }
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mma<float> {
  using v4 = float __attribute__((ext_vector_type(4)));
  // D[i][j]: lane j + 16 (i / 4), element i % 4
  static __device__ __forceinline__ int crow(int e, int r) { return 4 * r + e; }
  static __device__ __forceinline__ int irow(int i) { return i; }
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// lane J of the 16-lane row, in every lane of the row
template <int J>
__device__ __forceinline__ double bcast(double v) {
  return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + J, 0xF, 0xF, true);
}
// sum over the four lane rows, in every lane
__device__ __forceinline__ double rows_sum(double v) {
  const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
  const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
  v = __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
  const auto h2 = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
  const auto l2 = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
  return __hiloint2double(h2[0], l2[0]) + __hiloint2double(h2[1], l2[1]);
}
// largest of the four lane rows' values (not NaN), in every lane
__device__ __forceinline__ double rows_max(double v) {
  const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
  const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
  v = fmax(__hiloint2double(h[0], l[0]), __hiloint2double(h[1], l[1]));
  const auto h2 = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
  const auto l2 = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
  return fmax(__hiloint2double(h2[0], l2[0]), __hiloint2double(h2[1], l2[1]));
}
// e with |v| = f 2^e, f in [1/2, 1); 0 for zero, infinity and NaN.  x 2^e.
__device__ __forceinline__ int exponent_of(double v) { return __builtin_amdgcn_frexp_exp(v); }
__device__ __forceinline__ double scaled(double x, int e) { return __builtin_ldexp(x, e); }
// v of lane row r (0..3), in every lane row
template <int R>
__device__ __forceinline__ int row_bcast(int v) {
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  const int w = a[R & 1];
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return b[R >> 1];
}
template <int R>
__device__ __forceinline__ double row_bcast(double v) {
  return __hiloint2double(row_bcast<R>(__double2hiint(v)), row_bcast<R>(__double2loint(v)));
}
// s[e] += bcast<J>(x[e]) * x[e] and x[e] += bcast<J>(x[e]) * w, one DPP multiply-add an
// element (the compiler makes a broadcast copy and a multiply-add).  The leading
// s_nop covers a DPP source written by the instruction before the block, which the
// compiler does not see; results of matrix instructions pass mma_fence() first.
#define FRK_FMAC_DPP4(O0, O1, O2, O3, A0, A1, A2, A3, B0, B1, B2, B3, IMM)              \
  "s_nop 1\n\t"                                                                         \
  "v_fmac_f64_dpp " O0 ", " A0 ", " B0 " row_newbcast:" IMM " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f64_dpp " O1 ", " A1 ", " B1 " row_newbcast:" IMM " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f64_dpp " O2 ", " A2 ", " B2 " row_newbcast:" IMM " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f64_dpp " O3 ", " A3 ", " B3 " row_newbcast:" IMM " row_mask:0xf bank_mask:0xf"
template <int J>
__device__ __forceinline__ void dot4(double& s0, double& s1, double& s2, double& s3, double x0, double x1, double x2,
                                     double x3) {
  asm(FRK_FMAC_DPP4("%0", "%1", "%2", "%3", "%4", "%5", "%6", "%7", "%4", "%5", "%6", "%7", "%8")
      : "+v"(s0), "+v"(s1), "+v"(s2), "+v"(s3)
      : "v"(x0), "v"(x1), "v"(x2), "v"(x3), "n"(J));
}
template <int J>
__device__ __forceinline__ void axpy4(double& x0, double& x1, double& x2, double& x3, double w) {
  asm(FRK_FMAC_DPP4("%0", "%1", "%2", "%3", "%0", "%1", "%2", "%3", "%4", "%4", "%4", "%4", "%5")
      : "+v"(x0), "+v"(x1), "+v"(x2), "+v"(x3)
      : "v"(w), "n"(J));
}
// a0 += g(K) t0 + g(K+2) t2, a1 likewise: g(k) lane k's value
template <int K>
__device__ __forceinline__ void tdot4(double& a0, double& a1, double g, double t0, double t1, double t2, double t3) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %2, %4 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf"
      : "+v"(a0), "+v"(a1)
      : "v"(g), "v"(t0), "v"(t1), "v"(t2), "v"(t3), "n"(K), "n"(K + 1), "n"(K + 2), "n"(K + 3));
}
// waits until a matrix instruction's result may be read by the blocks above
__device__ __forceinline__ void mma_fence(double& x0, double& x1, double& x2, double& x3) {
  asm volatile("s_nop 15\n\ts_nop 7" : "+v"(x0), "+v"(x1), "+v"(x2), "+v"(x3));
}
// 1 / sqrt(x) and 1 / x to about an ulp, without branches (x = 0 gives NaN or inf)
__device__ __forceinline__ double rsqrt_of(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * r, r, 1.0);
  return fma(r * e, fma(0.375, e, 0.5), r);
}
__device__ __forceinline__ double inv_of(double x) { return d64::rcp2(x); }

// Squared norm at and below which a pivot column counts as zero: of a column whose
// largest entry was 2^-400 or more, so 1e-30 of its norm.
constexpr double kZeroNorm2 = 1e-300;

// A wave's share of a panel: tiles x (tile t is tile t RW + rw of the column), the
// pivot rows' tile (taken out of x; zero in a wave that does not own it), row li of
// the panel's T, the diagonal of R and 1 / (alpha - beta) of this lane's column.
template <typename T, int NT>
struct Panel {
  T x[NT][4], top[4], tr[16];
  T rd, inv;
};

// Householder step J: H = I - tau' v v^T with v = x_J - beta e (rows >= J), so the
// raw pivot column below its diagonal is the reflector; one reduction gives its norm
// and its products with every column (those with earlier reflectors are the Gram
// entries that T needs).  With n = ||x_J||, a = |alpha|, s = sign(alpha): beta = -s n,
// alpha - beta = s (a + n), tau' = 1 / (n (a + n)).
// RW waves share a panel's rows: they exchange their partial sums through ex, two
// buffers, one barrier a step (0.2 us of the 0.6 us a step takes then).
template <typename T, int NT, int RW, int J>
__device__ __forceinline__ void qr_step(Panel<T, NT>& p, int li, int lr, int rw, bool owner, T* ex) {
  using M = Mma<T>;
  asm volatile("" : "+v"(li));  // lane masks are made where they are used: 32 of them held would spill
  T s0 = T(0), s1 = T(0), s2 = T(0), s3 = T(0);
#pragma unroll
  for (int t = 0; t < NT; ++t) dot4<J>(s0, s1, s2, s3, p.x[t][0], p.x[t][1], p.x[t][2], p.x[t][3]);
  T vt[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const T b = bcast<J>(p.top[e]);
    vt[e] = (4 * lr + e >= J) ? b : T(0);
  }
  s0 += vt[0] * p.top[0];
  s1 += vt[1] * p.top[1];
  s2 += vt[2] * p.top[2];
  s3 += vt[3] * p.top[3];
  T d = rows_sum((s0 + s1) + (s2 + s3));
  T xj = row_bcast<J / 4>(p.top[J % 4]);  // row J of this lane's column
  if constexpr (RW > 1) {
    T* buf = ex + (J & 1) * (RW * 32);
    if (lr < 2) buf[rw * 32 + 16 * lr + li] = (lr == 0) ? d : xj;
    __syncthreads();
    d = T(0);
    xj = T(0);
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      d += buf[r * 32 + li];
      xj += buf[r * 32 + 16 + li];
    }
  }
  const T q = bcast<J>(d), alpha = bcast<J>(xj);
  const bool ok = q > kZeroNorm2;  // a column of zeros (at its scale) is left as it is; a NaN in it stays one
  const T rn = rsqrt_of(q), nrm = q * rn;
  const T beta = (alpha >= T(0)) ? -nrm : nrm;
  const T den = fabs(alpha) + nrm, iden = inv_of(den);
  const T z = d - beta * xj;
  const T nw = (ok && li > J) ? -(z * rn) * iden : T(0);
#pragma unroll
  for (int t = 0; t < NT; ++t) axpy4<J>(p.x[t][0], p.x[t][1], p.x[t][2], p.x[t][3], nw);
  const T ab = (ok && owner) ? alpha - beta : T(0);
#pragma unroll
  for (int e = 0; e < 4; ++e) p.top[e] += nw * ((4 * lr + e == J) ? ab : vt[e]);
  const T sinv = (alpha >= T(0)) ? iden : -iden;
  if (li == J) {
    p.rd = ok ? beta : (q != q ? q : alpha);
    p.inv = ok ? sinv : T(0);
  }
  // column J of T for unit reflectors: tau = tau' (a + n)^2 = (a + n) / n, the Gram
  // entries scaled by both columns' 1 / (alpha - beta)
  T a0 = T(0), a1 = T(0);
  if constexpr (J > 0) {
    const T g = (li < J) ? z * p.inv : T(0);
    tdot4<0>(a0, a1, g, p.tr[0], p.tr[1], p.tr[2], p.tr[3]);
    if constexpr (J > 4) tdot4<4>(a0, a1, g, p.tr[4], p.tr[5], p.tr[6], p.tr[7]);
    if constexpr (J > 8) tdot4<8>(a0, a1, g, p.tr[8], p.tr[9], p.tr[10], p.tr[11]);
    if constexpr (J > 12) tdot4<12>(a0, a1, g, p.tr[12], p.tr[13], p.tr[14], p.tr[15]);
  }
  const T c = (alpha >= T(0)) ? -rn : rn;
  const T tj = (li < J) ? c * (a0 + a1) : (li == J ? rn * den : T(0));
  p.tr[J] = ok ? tj : T(0);
}
template <typename T, int NT, int RW, int J>
__device__ __forceinline__ void qr_steps(Panel<T, NT>& p, int li, int lr, int rw, bool owner, T* ex) {
  if constexpr (J < 16) {
    qr_step<T, NT, RW, J>(p, li, lr, rw, owner, ex);
    qr_steps<T, NT, RW, J + 1>(p, li, lr, rw, owner, ex);
  }
}

// Memory access through buffer descriptors: byte offsets below 2^31, and kOut for an
// element that is not there, which reads as zero and is not written.  No branch and
// no wait depends on the bounds (guarded loads through pointers become one masked
// load after the other, each waited for).
constexpr uint32_t kOut = 0x80000000u;
template <typename T>
struct Buf {
  using v4 = typename Mma<T>::v4;
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ explicit Buf(const void* p)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0x7ffffffc, 0x00020000)) {}
  __device__ __forceinline__ T load(uint32_t off) const {
    if constexpr (sizeof(T) == 8)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  }
  __device__ __forceinline__ void store(uint32_t off, T v) const {
    if constexpr (sizeof(T) == 8) {
      typedef unsigned u2 __attribute__((ext_vector_type(2)));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, off, 0, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 0);
    }
  }
  // four consecutive elements (off aligned to four bytes)
  __device__ __forceinline__ v4 load4(uint32_t off) const {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    if constexpr (sizeof(T) == 8) {
      struct P {
        u4 a, b;
      } q{__builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0), __builtin_amdgcn_raw_buffer_load_b128(r, off, 16, 0)};
      return __builtin_bit_cast(v4, q);
    } else {
      return __builtin_bit_cast(v4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    }
  }
  __device__ __forceinline__ void store4(uint32_t off, v4 v) const {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    if constexpr (sizeof(T) == 8) {
      struct P {
        u4 a, b;
      };
      const P q = __builtin_bit_cast(P, v);
      __builtin_amdgcn_raw_buffer_store_b128(q.a, r, off, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b128(q.b, r, off, 16, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, off, 0, 0);
    }
  }
};
// byte offset of element (i, j) of a strided matrix if it is there
template <typename T>
__device__ __forceinline__ uint32_t at(bool in, int i, int64_t rs, int j, int64_t cs) {
  const uint32_t o = (uint32_t)i * ((uint32_t)rs * (uint32_t)sizeof(T)) + (uint32_t)j * ((uint32_t)cs * (uint32_t)sizeof(T));
  return in ? o : kOut;
}

// Position of row 4 r + e, column c of a 16 x 16 tile of reflectors in LDS: free of
// bank conflicts for both operand forms (rows 4 r + e by lanes (c, r), and rows
// irow(i), columns crow(e, r) by lanes (i, r)).
template <typename T>
__device__ __forceinline__ int y_pos(int e, int r, int c) {
  return 64 * e + 16 * r + (c ^ (sizeof(T) == 8 ? 4 * e + r : 4 * r + e));
}
template <typename T>
__device__ __forceinline__ int y_pos_row(int i, int c) {
  return sizeof(T) == 8 ? y_pos<T>(i >> 2, i & 3, c) : y_pos<T>(i & 3, i >> 2, c);
}

// (NT = 4: two workgroups of 8 waves fit a CU)
template <typename T, int NT, int RW, int NP, class Src>
__global__ __launch_bounds__(64 * NP * RW, (NT == 4 && NP == 8) ? 4 : 1) void lr_qr_kernel(Src items) {
  using M = Mma<T>;
  using v4 = typename M::v4;
  const QrItem it = items.get(blockIdx.x);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, li = lane & 15, lr = lane >> 4;
  const int w = wid / RW, rw = wid % RW;  // 16-column group, share of the rows
  const int m = it.m, K = it.k1 + it.k2, nref = min(m, K);
  const int c = 16 * w + li;
  const bool own = c < K, act = 16 * w < K;
  // panels of reflectors and their T for the waves of the later columns: two
  // buffers, so one barrier a panel, and the next panel's wave goes on with its
  // factorization while the others still update
  __shared__ T Ys[NP > 1 ? 2 : 1][NP > 1 ? 256 * NT * RW : 1];
  __shared__ T Ts[NP > 1 ? 2 : 1][NP > 1 ? 256 : 1];
  __shared__ T Wp[RW > 1 ? 256 * NP * RW : 1];  // partial products of the row shares
  __shared__ T ex[RW > 1 ? 64 * RW : 1];
  __shared__ int ses[16 * NP * RW];  // exponents of the columns' scales
  // the sum of the RW shares of a 16 x 16 product
  auto rw_sum = [&](v4 z) {
    if constexpr (RW > 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) Wp[256 * wid + 64 * e + lane] = z[e];
      __syncthreads();
      z = v4{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < RW; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) z[e] += Wp[256 * (w * RW + r) + 64 * e + lane];
    }
    return z;
  };
  v4 x[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) x[t] = v4{0, 0, 0, 0};
  // ---- the panel ---------------------------------------------------------------
#pragma unroll 1
  for (int blk = 0; blk < 2; ++blk) {
    const void* Sp = blk ? it.S2 : it.S1;
    const Buf<T> Ab(blk ? it.A2 : it.A1), S(Sp);
    const int64_t rs = blk ? it.a2_rs : it.a1_rs, cs = blk ? it.a2_cs : it.a1_cs;
    const int sld = blk ? it.s2_ld : it.s1_ld;
    const int kc = blk ? it.k2 : it.k1, ka = blk ? it.k2a : it.k1a;
    const int cb = c - (blk ? it.k1 : 0);  // column of this block
    const bool mine = cb >= 0 && cb < kc;
    if (!__any(mine)) continue;
    if (Sp == nullptr) {
      // (the columns of a wave that belong to the other block read zeros and add up)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = 16 * (t * RW + rw) + 4 * lr + e;
          x[t][e] += Ab.load(at<T>(mine && row < m, row, rs, cb, cs));
        }
    } else {
      // KU groups of 4 columns of A in flight
      constexpr int KU = NT <= 8 ? 4 : 2;
#pragma unroll 1
      for (int s0 = 0; s0 < ka; s0 += 4 * KU) {
        T a[KU][NT], b[KU];
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int k = s0 + 4 * u + lr;
          b[u] = S.load(at<T>(mine && k < ka, k, sld, cb, 1));
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const int row = 16 * (t * RW + rw) + M::irow(li);
            a[u][t] = Ab.load(at<T>(row < m && k < ka, row, rs, k, cs));
          }
        }
#pragma unroll
        for (int u = 0; u < KU; ++u)
#pragma unroll
          for (int t = 0; t < NT; ++t) x[t] = M::mma(a[u][t], b[u], x[t]);
      }
    }
  }
  const Buf<T> Rb(it.R);
  const int ldr = it.ldr, kp = (it.P != nullptr) ? it.kp : 0;
  // ---- projection against an orthonormal P: Z = P^T X, X -= P Z, twice ---------------
  // 16 columns of P at a time, so all of Z's block is taken from the same X: one pass leaves
  // P^T X at u ||X|| however little of X remains, and what the bases lose of their
  // orthogonality grows from addition to addition (twelve in a chain, m = 256, k = 16: 6e-8,
  // against 1e-13 with the second pass, which takes P^T X to u times what remains; the block
  // LU of 16 x 16 tiles of 256 at fixed rank 16 ends 1.3 times further from the exact solution).
  if (kp > 0) {
    const Buf<T> P(it.P);
    const int nblk = (kp + 15) / 16;
#pragma unroll 1
    for (int blk = 0; blk < 2 * nblk; ++blk) {
      const bool again = blk >= nblk;
      const int s0 = 16 * (again ? blk - nblk : blk);
      v4 zs = v4{0, 0, 0, 0};
      if (act) {
        v4 z[2] = {v4{0, 0, 0, 0}, v4{0, 0, 0, 0}};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          T a[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = 16 * (t * RW + rw) + 4 * lr + e;
            a[e] = P.load(at<T>(row < m && s0 + li < kp, row, it.p_rs, s0 + li, it.p_cs));
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) z[e & 1] = M::mma(a[e], x[t][e], z[e & 1]);
        }
        zs = z[0] + z[1];
      }
      zs = rw_sum(zs);
      if (act) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int sr = s0 + M::crow(e, lr);
          const uint32_t zo = at<T>(rw == 0 && sr < kp && own, sr, ldr, c, 1);
          Rb.store(zo, again ? Rb.load(zo) + zs[e] : zs[e]);
          T a[NT];
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const int row = 16 * (t * RW + rw) + M::irow(li);
            a[t] = P.load(at<T>(row < m && sr < kp, row, it.p_rs, sr, it.p_cs));
          }
#pragma unroll
          for (int t = 0; t < NT; ++t) x[t] = M::mma(a[t], -zs[e], x[t]);
        }
      }
      if constexpr (RW > 1) __syncthreads();  // Wp free
    }
  }
  // ---- columns of extreme norm to a largest entry in [1/2, 1), by a power of two ------
  // Reflectors and T do not depend on the columns' scales, R takes them back: norms of
  // any size neither overflow nor fall under kZeroNorm2.
  {
    T mx = T(0);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmax(mx, fabs(x[t][e]));
    mx = rows_max(mx);
    if constexpr (RW > 1) {
      if (lr == 0) Wp[256 * wid + li] = mx;
      __syncthreads();
#pragma unroll
      for (int r = 0; r < RW; ++r) mx = fmax(mx, Wp[256 * (w * RW + r) + li]);
    }
    int se = exponent_of(mx);
    se = (se > -400 && se < 400) ? 0 : se;
    if (lr == 0) ses[16 * wid + li] = se;  // (a register held through the panels would spill)
    // (scaling every panel spills at NT = 8: 199 us instead of 144 at 256 rows, 64 columns,
    // 165 additions; at the others it costs nothing)
    if (NT != 8 || __any(se != 0)) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[t][e] = scaled(x[t][e], -se);
    }
  }
  // ---- factorization, panel by panel ------------------------------------------------
  const Buf<T> Y(it.Y), Tg(it.tau);
  const int64_t ldy = it.y_cs;
#pragma unroll 1
  for (int q = 0; q < NP; ++q) {
    const int j0 = 16 * q;
    if (j0 >= nref) break;
    const bool owner = (q % RW) == rw;  // of the pivot rows, tile tq of its share
    const int tq = q / RW;
    if (w == q) {
      Panel<T, NT> p;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int e = 0; e < 4; ++e) p.x[t][e] = x[t][e];
        mma_fence(p.x[t][0], p.x[t][1], p.x[t][2], p.x[t][3]);
      }
      // the pivot rows leave x: zero rows there take no part in the steps
#pragma unroll
      for (int e = 0; e < 4; ++e) p.top[e] = T(0);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p.top[e] = (owner && t == tq) ? p.x[t][e] : p.top[e];
          p.x[t][e] = (owner && t == tq) ? T(0) : p.x[t][e];
        }
#pragma unroll
      for (int k = 0; k < 16; ++k) p.tr[k] = T(0);
      p.rd = T(0);
      p.inv = T(0);
      qr_steps<T, NT, RW, 0>(p, li, lr, rw, owner, ex);
      // T, a row a lane (every lane row the same)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        Tg.store(at<T>(lr == 0 && owner, 256 * q + 16 * li + j, 1, 0, 0), p.tr[j]);
        if constexpr (NP > 1) Ts[q & 1][16 * li + j] = p.tr[j];
      }
      // R of this panel's own columns (its columns past the last pivot: every row
      // up to there), then the unit reflectors, zero in the tiles above
      const int lim = nref - j0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 4 * lr + e;
        const T rv = (row < li) ? p.top[e] : (row == li ? p.rd : T(0));
        Rb.store(at<T>(owner && own && j0 + row < K, kp + j0 + row, ldr, c, 1), (row < lim) ? scaled(rv, ses[16 * wid + li]) : T(0));
        p.top[e] = (li >= lim || row < li) ? T(0) : (row == li ? T(1) : p.top[e] * p.inv);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int tg = t * RW + rw;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[t][e] = (owner && t == tq) ? p.top[e] : p.x[t][e] * p.inv;
          if constexpr (NP > 1) Ys[q & 1][256 * tg + y_pos<T>(e, lr, li)] = x[t][e];
        }
        Y.store4(at<T>(16 * tg < m, 16 * tg + 4 * lr, 1, c, ldy), x[t]);
      }
      __builtin_amdgcn_s_setprio(0);
    } else if constexpr (RW > 1) {
      for (int j = 0; j < 16; ++j) __syncthreads();  // the steps' barriers
    }
    if constexpr (NP > 1) {
      __syncthreads();
      if (w == q + 1) __builtin_amdgcn_s_setprio(3);  // the next panel's wave: what everything waits for
      const bool trail = w > q && act;
      const T* Yq = Ys[q & 1];
      v4 ws = v4{0, 0, 0, 0}, top = v4{0, 0, 0, 0};
      if (trail) {
        // C -= Y T^T (Y^T C); rows already in R are zero in Y and in C
        v4 wa[4] = {v4{0, 0, 0, 0}, v4{0, 0, 0, 0}, v4{0, 0, 0, 0}, v4{0, 0, 0, 0}};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
          for (int e = 0; e < 4; ++e) wa[e] = M::mma(Yq[256 * (t * RW + rw) + y_pos<T>(e, lr, li)], x[t][e], wa[e]);
          if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (holding the operands of all tiles would spill)
        }
        ws = (wa[0] + wa[1]) + (wa[2] + wa[3]);
      }
      ws = rw_sum(ws);
      if (trail) {
        v4 w2 = v4{0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 4; ++e) w2 = M::mma(-Ts[q & 1][M::crow(e, lr) * 16 + li], ws[e], w2);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int yp = y_pos_row<T>(li, M::crow(e, lr));
#pragma unroll
          for (int t = 0; t < NT; ++t) x[t] = M::mma(Yq[256 * (t * RW + rw) + yp], w2[e], x[t]);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (owner) {
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              top[e] = (t == tq) ? x[t][e] : top[e];
              x[t][e] = (t == tq) ? T(0) : x[t][e];
            }
        }
      }
      if (w != q && owner) {
        // the panel's rows of this wave's columns: R (zero below the diagonal block)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = j0 + 4 * lr + e;
          Rb.store(at<T>(own && row < K, kp + row, ldr, c, 1), (row < nref) ? scaled(top[e], ses[16 * wid + li]) : T(0));
        }
      }
    }
  }
  // rows of R past the last panel
  for (int row = 16 * ((nref + 15) / 16) + lr; row < K; row += 4) Rb.store(at<T>(rw == 0 && own, kp + row, ldr, c, 1), T(0));
}

// out = Q [X; 0] (+ Base Xb), Q = (I - Y_0 T_0 Y_0^T) (I - Y_1 T_1 Y_1^T) ...: wave
// (w, rw) owns output columns [16 w, 16 w + 16) of the tiles t RW + rw.
template <typename T, int NT, int RW, int NW, class Src>
__global__ __launch_bounds__(64 * NW * RW) void lr_apply_kernel(Src items) {
  using M = Mma<T>;
  using v4 = typename M::v4;
  const ApplyQItem it = items.get(blockIdx.x);
  const int ncol = (it.ncol_ptr != nullptr) ? *it.ncol_ptr : it.ncol;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, li = lane & 15, lr = lane >> 4;
  const int w = wid / RW, rw = wid % RW;
  const int m = it.m, c = 16 * w + li;
  const bool own = c < ncol, act = 16 * w < ncol;
  const Buf<T> Y(it.Y), Tg(it.tau), X(it.X);
  const int64_t ldy = it.y_cs;
  __shared__ T Wp[RW > 1 ? 2 * 256 * NW * RW : 1];  // two buffers, one barrier a panel
  v4 x[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * (t * RW + rw) + 4 * lr + e;
      x[t][e] = X.load(at<T>(own && row < it.kx && row < m, row, it.x_rs, c, it.x_cs));
    }
#pragma unroll 1
  for (int q = (it.nref + 15) / 16 - 1; q >= 0; --q) {
    v4 ws = v4{0, 0, 0, 0};
    if (act) {
      // (the tiles above a panel's pivot rows are stored as zeros)
      v4 wa[4] = {v4{0, 0, 0, 0}, v4{0, 0, 0, 0}, v4{0, 0, 0, 0}, v4{0, 0, 0, 0}};
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int row0 = 16 * (t * RW + rw);
        const v4 y = Y.load4(at<T>(row0 < m, row0 + 4 * lr, 1, 16 * q + li, ldy));
#pragma unroll
        for (int e = 0; e < 4; ++e) wa[e] = M::mma(y[e], x[t][e], wa[e]);
      }
      ws = (wa[0] + wa[1]) + (wa[2] + wa[3]);
    }
    if constexpr (RW > 1) {
      T* wb = Wp + (q & 1) * (256 * NW * RW);
#pragma unroll
      for (int e = 0; e < 4; ++e) wb[256 * wid + 64 * e + lane] = ws[e];
      __syncthreads();
      ws = v4{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < RW; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) ws[e] += wb[256 * (w * RW + r) + 64 * e + lane];
    }
    if (act) {
      v4 w2 = v4{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 4; ++e) w2 = M::mma(-Tg.load(at<T>(true, 256 * q + 16 * li + M::crow(e, lr), 1, 0, 0)), ws[e], w2);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        T a[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int row0 = 16 * (t * RW + rw);
          a[t] = Y.load(at<T>(row0 < m, row0 + M::irow(li), 1, 16 * q + M::crow(e, lr), ldy));
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) x[t] = M::mma(a[t], w2[e], x[t]);
      }
    }
  }
  if (it.Base != nullptr && it.kb > 0) {
    const Buf<T> Bs(it.Base), Xb(it.Xb);
    if (act)
      for (int s0 = 0; s0 < it.kb; s0 += 4) {
        const int k = s0 + lr;
        const T b = Xb.load(at<T>(own && k < it.kb, k, it.xb_rs, c, it.xb_cs));
        T a[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int row = 16 * (t * RW + rw) + M::irow(li);
          a[t] = Bs.load(at<T>(row < m && k < it.kb, row, it.base_rs, k, it.base_cs));
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) x[t] = M::mma(a[t], b, x[t]);
      }
    __syncthreads();  // the base may alias the output
  }
  const Buf<T> out(it.out);
  if (it.out_rs == 1 && (m & 3) == 0) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int row = 16 * (t * RW + rw) + 4 * lr;
      out.store4(at<T>(own && row < m, row, 1, c, it.out_cs), x[t]);
    }
  } else {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * (t * RW + rw) + 4 * lr + e;
        out.store(at<T>(own && row < m, row, it.out_rs, c, it.out_cs), x[t][e]);
      }
  }
}

// M = Ru Rv^T (Ke x Ke, row stride K) of the additions whose core is smaller than
// K = kc + kx2 (a workgroup each; the others return at once).  Wave w forms the tile
// rows w and w + 4: a lane reads four consecutive columns of its row of Ru and of a
// row of Rv per tile, and the MFMA products take them as the contraction index (any
// order will do, if both operands have the same).  Both are upper trapezoidal, so a
// tile row starts at its diagonal tile.  Bound by the FP64 MFMA rate of one CU and the
// latency of the reads.  FP64, 165 cores of 64 from 128 columns: 26 us, 135 us with
// the factors staged through LDS and one FMA a pair of LDS reads.
template <typename T, int NJ>
__global__ __launch_bounds__(256) void lr_core_prod_kernel(const LrAddDesc<T>* __restrict__ d, LrBatch<T> b) {
  using M = Mma<T>;
  using v4 = typename M::v4;
  const int t = blockIdx.x;
  const LrAddDesc<T> x = d[t];
  const int K = b.K, Kt = x.kc + x.kx2, Ke = lr_core_dim(x, b);
  if (Ke >= Kt) return;
  const Buf<T> Ru(b.Ru + (size_t)t * K * K), Rv(b.Rv + (size_t)t * K * K), Mo(b.Mw + (size_t)t * K * K);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lr = lane >> 4;
  for (int i = w; 16 * i < Ke; i += 4) {
    v4 acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] = v4{0, 0, 0, 0};
#pragma unroll 1
    for (int q = 16 * i + 4 * lr; __any(q < Kt); q += 16) {
      const int ra = 16 * i + M::irow(li);
      v4 a = Ru.load4(at<T>(ra < Ke, ra, K, q, 1)), v[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) v[j] = Rv.load4(at<T>(16 * j + li < Ke, 16 * j + li, K, q, 1));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const T ae = (q + e < Kt) ? a[e] : T(0);
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[j] = M::mma(ae, (q + e < Kt) ? v[j][e] : T(0), acc[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * i + 4 * lr + e, col = 16 * j + li;
        Mo.store(at<T>(row < Ke && col < Ke, row, K, col, 1), acc[j][e]);
      }
  }
}

template <typename T, int NT, int RW, int NP>
void qr_go(const LrAddDesc<T>* d, int nd, const LrBatch<T>& b, hipStream_t s) {
  hipLaunchKernelGGL((lr_qr_kernel<T, NT, RW, NP, LrQrItems<T>>), dim3(2 * nd), dim3(64 * NP * RW), 0, s,
                     LrQrItems<T>{d, b});
}
template <typename T, int NT, int RW, int NW>
void apply_go(const LrAddDesc<T>* d, int nd, const LrBatch<T>& b, hipStream_t s) {
  hipLaunchKernelGGL((lr_apply_kernel<T, NT, RW, NW, LrApplyItems<T>>), dim3(2 * nd), dim3(64 * NW * RW), 0, s,
                     LrApplyItems<T>{d, b});
}

}  // namespace

// Up to 128 rows the blocked kernels are faster at every width and batch measured
// (m = 64, 128; K = 16 .. 128; 4 .. 590 additions: QR 1.2 to 4 times).  With 129 to 256
// rows a panel of 16 columns costs its 16 steps whatever K is, so small K in a large
// batch goes to the unblocked kernels: FP64, m = 256, K = 32: 33.1 / 52.9 us at 40
// additions, 63.7 / 65.3 at 165, 93.4 / 76.1 at 300, 164 / 131 at 590; K = 64 at 590:
// 369 / 497.  Above 256 rows the unblocked kernels stay the faster ones where they are
// used most (m = 512, K up to 32, several hundred additions, ranks below 16: 138 us a
// launch in a factorization of 64 x 64 tiles, the blocked form with four waves a
// panel 185).
bool lr_blocked_ok(int nd, int m, int k) {
  return k <= 128 && (m <= 128 || (m <= 256 && (k > 32 || nd <= 128)));
}

// Columns to waves: 16 each, so 1, 2, 4 or 8 of them; FN(number of waves)
#define FRK_LR_COLS(FN) \
  do {                  \
    if (k <= 16)        \
      FN(1);            \
    else if (k <= 32)   \
      FN(2);            \
    else if (k <= 64)   \
      FN(4);            \
    else                \
      FN(8);            \
  } while (0)

void launch_lr_qr_blocked(const LrAddDesc<double>* d, int nd, const LrBatch<double>& b, int k, hipStream_t s) {
  if (nd <= 0) return;
  const int m = std::max(b.mmax, b.nmax);
  if (m > 256 || k > 128 || b.Kp <= 0) throw std::runtime_error("lr qr: panel outside the blocked kernels");
#define FRK_QR4(NP) qr_go<double, 4, 1, NP>(d, nd, b, s)
#define FRK_QR8(NP) qr_go<double, 8, 1, NP>(d, nd, b, s)
#define FRK_QR16(NP) qr_go<double, (NP) < 8 ? 8 : 16, (NP) < 8 ? 2 : 1, NP>(d, nd, b, s)
  if (m <= 64)
    FRK_LR_COLS(FRK_QR4);
  else if (m <= 128)
    FRK_LR_COLS(FRK_QR8);
  else
    FRK_LR_COLS(FRK_QR16);
#undef FRK_QR4
#undef FRK_QR8
#undef FRK_QR16
  FRK_HIP_CHECK(hipGetLastError());
}
void launch_lr_apply_blocked(const LrAddDesc<double>* d, int nd, const LrBatch<double>& b, int k, hipStream_t s) {
  if (nd <= 0) return;
  const int m = std::max(b.mmax, b.nmax);
  if (m > 256 || k > 128 || b.Kp <= 0) throw std::runtime_error("lr apply: panel outside the blocked kernels");
#define FRK_AP4(NW) apply_go<double, 4, 1, NW>(d, nd, b, s)
#define FRK_AP8(NW) apply_go<double, 8, 1, NW>(d, nd, b, s)
#define FRK_AP16(NW) apply_go<double, (NW) < 8 ? 8 : 16, (NW) < 8 ? 2 : 1, NW>(d, nd, b, s)
  if (m <= 64)
    FRK_LR_COLS(FRK_AP4);
  else if (m <= 128)
    FRK_LR_COLS(FRK_AP8);
  else
    FRK_LR_COLS(FRK_AP16);
#undef FRK_AP4
#undef FRK_AP8
#undef FRK_AP16
  FRK_HIP_CHECK(hipGetLastError());
}

template <typename T>
void launch_lr_add_core(const LrAddDesc<T>* d, int nd, const LrBatch<T>& b, hipStream_t s) {
  if (nd <= 0 || b.Mw == nullptr) return;
  if (b.K > 128) throw std::runtime_error("lr core product: K above 128");
  if (b.Kmax_svd <= 64)
    hipLaunchKernelGGL((lr_core_prod_kernel<T, 4>), dim3(nd), dim3(256), 0, s, d, b);
  else
    hipLaunchKernelGGL((lr_core_prod_kernel<T, 8>), dim3(nd), dim3(256), 0, s, d, b);
  FRK_HIP_CHECK(hipGetLastError());
}

template void launch_lr_add_core<double>(const LrAddDesc<double>*, int, const LrBatch<double>&, hipStream_t);
template void launch_lr_add_core<float>(const LrAddDesc<float>*, int, const LrBatch<float>&, hipStream_t);

}  // namespace frk
