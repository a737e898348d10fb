// Device-side items of the batched low-rank additions.
#pragma once
#include "common.hpp"

namespace frk {

// ===========================================================================
// Item sources of the batched QR / SVD / basis-update kernels: an uploaded item
// array, or the items of a batch of low-rank additions derived on the device
// from their descriptors (the same construction the host would do, so only the
// additions' descriptors cross PCIe).  Addition t owns QR items 2t (U side) and
// 2t+1 (V side), SVD item t, basis-update items 2t and 2t+1.
// ===========================================================================
template <class Item>
struct ItemArray {
  const Item* p;
  __device__ Item get(int b) const { return p[b]; }
};

template <typename T>
__device__ __forceinline__ bool lr_fast(const LrAddDesc<T>& x, const LrBatch<T>& b) {
  return b.lra == 2 && x.eps == 0.0;
}
// the core size of a rounded addition: K = kc + kx2, or less when K exceeds a
// tile dimension (the QR factors then have min(m, K) / min(n, K) nonzero rows)
template <typename T>
__device__ __forceinline__ int lr_core_dim(const LrAddDesc<T>& x, const LrBatch<T>& b) {
  const int Kt = x.kc + x.kx2;
  if (b.Mw == nullptr || lr_fast(x, b)) return Kt;
  return max(min(x.m, Kt), min(x.n, Kt));
}

template <typename T>
struct LrQrItems {
  const LrAddDesc<T>* d;
  LrBatch<T> b;
  __device__ QrItem get(int w) const {
    const int t = w >> 1;
    const LrAddDesc<T> x = d[t];
    const int K = b.K;
    QrItem q{};
    if ((w & 1) == 0) {
      q.Y = b.Yu + (size_t)t * (b.Kp ? (size_t)b.ldu * b.Kp : (size_t)b.mmax * K);
      q.y_cs = b.Kp ? b.ldu : x.m;
      q.tau = b.tu + (size_t)t * (b.Kp ? 16 * b.Kp : K);
      q.R = b.Ru + (size_t)t * K * K;
      q.m = x.m;
    } else {
      q.Y = b.Yv + (size_t)t * (b.Kp ? (size_t)b.ldv * b.Kp : (size_t)b.nmax * K);
      q.y_cs = b.Kp ? b.ldv : x.n;
      q.tau = b.tv + (size_t)t * (b.Kp ? 16 * b.Kp : K);
      q.R = b.Rv + (size_t)t * K * K;
      q.m = x.n;
    }
    q.y_rs = 1;
    q.ldr = K;
    const bool fast = lr_fast(x, b);
    if ((w & 1) == 0) {
      if (!fast) {  // Uc = [Uc Sc | Ux Sx] (formed inside the QR kernel)
        q.A1 = x.cu;
        q.a1_rs = x.cu_rs;
        q.a1_cs = x.cu_cs;
        q.S1 = x.cs;
        q.s1_ld = x.lds;
        q.k1a = q.k1 = x.kc;
        q.A2 = x.xu;
        q.a2_rs = x.xu_rs;
        q.a2_cs = x.xu_cs;
        q.S2 = x.xs;
        q.s2_ld = x.xs_ld;
        q.k2a = x.kx1;
        q.k2 = x.kx2;
      } else {  // project X's U basis on C's, QR the remainder
        q.A1 = x.xu;
        q.a1_rs = x.xu_rs;
        q.a1_cs = x.xu_cs;
        q.S1 = x.xs;
        q.s1_ld = x.xs_ld;
        q.k1a = x.kx1;
        q.k1 = x.kx2;
        q.k2 = 0;
        q.P = x.cu;
        q.p_rs = x.cu_rs;
        q.p_cs = x.cu_cs;
        q.kp = x.kc;
      }
    } else {
      if (!fast) {  // Vc^T = [Vc^T | Vx^T]
        q.A1 = x.cv;
        q.a1_rs = x.cv_cs;
        q.a1_cs = x.cv_rs;
        q.k1a = q.k1 = x.kc;
        q.A2 = x.xv;
        q.a2_rs = x.xv_cs;
        q.a2_cs = x.xv_rs;
        q.k2a = q.k2 = x.kx2;
      } else {
        q.A1 = x.xv;
        q.a1_rs = x.xv_cs;
        q.a1_cs = x.xv_rs;
        q.k1a = q.k1 = x.kx2;
        q.k2 = 0;
        q.P = x.cv;
        q.p_rs = x.cv_cs;
        q.p_cs = x.cv_rs;
        q.kp = x.kc;
      }
    }
    return q;
  }
};

template <typename T>
struct LrSvdItems {
  const LrAddDesc<T>* d;
  LrBatch<T> b;
  int t0;  // first item of this launch (workspace slots are indexed by the item)
  __device__ SvdItem get(int tl) const {
    const int t = t0 + tl;
    const LrAddDesc<T> x = d[t];
    const int K = b.K;
    const int Kt = x.kc + x.kx2;
    const bool fast = lr_fast(x, b);
    SvdItem sv{};
    sv.mode = 1;
    sv.Ru = b.Ru + (size_t)t * K * K;
    sv.Rv = b.Rv + (size_t)t * K * K;
    sv.ldr = K;
    sv.K = Kt;
    const int Ke = lr_core_dim(x, b);
    if (Ke < Kt) {
      // the core M = Ru Rv^T was formed into Mw (lr_core_prod_kernel)
      sv.mode = 0;
      sv.M = b.Mw + (size_t)t * K * K;
      sv.m_rs = K;
      sv.m_cs = 1;
      sv.K = Ke;
    } else if (!fast) {
      sv.kx = Kt;
      sv.ka = 0;
    } else {
      sv.kx = x.kx2;
      sv.ka = x.kc;
      sv.Sa = x.cs;
      sv.lds_in = x.lds;
    }
    sv.fixed_rank = (x.eps != 0.0) ? -1 : x.kc;
    sv.kdim = min(min(x.m, Kt), min(x.n, Kt));
    sv.eps = x.eps;
    sv.S = x.cs;
    sv.lds = x.lds;
    sv.Um = b.Um + (size_t)t * K * K;
    sv.ldu = K;
    sv.Vm = b.Vm + (size_t)t * K * K;
    sv.ldv = K;
    sv.rank_out = x.d_rank;
    sv.cap = x.cap;
    sv.cap_trunc = x.cap_trunc ? 1 : 0;
    sv.stats = b.stats;
    sv.vwork = b.Vw ? b.Vw + (size_t)t * K * K : nullptr;
    return sv;
  }
};

template <typename T>
struct LrApplyItems {
  const LrAddDesc<T>* d;
  LrBatch<T> b;
  __device__ ApplyQItem get(int w) const {
    const int t = w >> 1;
    const LrAddDesc<T> x = d[t];
    const int K = b.K;
    const int Kt = x.kc + x.kx2;
    const bool fast = lr_fast(x, b);
    T* um = b.Um + (size_t)t * K * K;
    T* vm = b.Vm + (size_t)t * K * K;
    ApplyQItem a{};
    a.y_rs = 1;
    a.ncol_ptr = x.d_rank;
    a.ncol = Kt;
    a.trans = 0;
    a.x_rs = K;
    a.x_cs = 1;
    if ((w & 1) == 0) {
      a.Y = b.Yu + (size_t)t * (b.Kp ? (size_t)b.ldu * b.Kp : (size_t)b.mmax * K);
      a.y_cs = b.Kp ? b.ldu : x.m;
      a.tau = b.tu + (size_t)t * (b.Kp ? 16 * b.Kp : K);
      a.m = x.m;
      a.out = x.cu;
      a.out_rs = x.cu_rs;
      a.out_cs = x.cu_cs;
      if (!fast) {
        a.nref = min(x.m, Kt);
        a.X = um;
        a.kx = Kt;
      } else {
        a.nref = min(x.m, x.kx2);
        a.X = um + (size_t)x.kc * K;
        a.kx = x.kx2;
        a.Base = x.cu;
        a.base_rs = x.cu_rs;
        a.base_cs = x.cu_cs;
        a.Xb = um;
        a.xb_rs = K;
        a.xb_cs = 1;
        a.kb = x.kc;
      }
    } else {
      a.Y = b.Yv + (size_t)t * (b.Kp ? (size_t)b.ldv * b.Kp : (size_t)b.nmax * K);
      a.y_cs = b.Kp ? b.ldv : x.n;
      a.tau = b.tv + (size_t)t * (b.Kp ? 16 * b.Kp : K);
      a.m = x.n;
      a.out = x.cv;
      a.out_rs = x.cv_cs;
      a.out_cs = x.cv_rs;
      if (!fast) {
        a.nref = min(x.n, Kt);
        a.X = vm;
        a.kx = Kt;
      } else {
        a.nref = min(x.n, x.kx2);
        a.X = vm + (size_t)x.kc * K;
        a.kx = x.kx2;
        a.Base = x.cv;
        a.base_rs = x.cv_cs;
        a.base_cs = x.cv_rs;
        a.Xb = vm;
        a.xb_rs = K;
        a.xb_cs = 1;
        a.kb = x.kc;
      }
    }
    return a;
  }
};

}  // namespace frk
