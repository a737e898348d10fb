// Prints, for one addition per line of input (kc kx1 kx2 cap m n cu_rs cu_cs cv_rs cv_cs lds
// xu_rs xu_cs xs_ld xv_rs xv_cs), whether the FP64 and the FP32 kernels may take it.
#include <cstdio>

#include "near.hpp"

struct Desc {
  int64_t cu_rs, cu_cs, cv_rs, cv_cs, xu_rs, xu_cs, xv_rs, xv_cs;
  int32_t kc, kx1, kx2, cap, m, n, lds, xs_ld;
};

int main() {
  long long v[16];
  for (;;) {
    for (int i = 0; i < 16; ++i)
      if (std::scanf("%lld", v + i) != 1) return 0;
    Desc x{};
    x.kc = (int32_t)v[0], x.kx1 = (int32_t)v[1], x.kx2 = (int32_t)v[2], x.cap = (int32_t)v[3];
    x.m = (int32_t)v[4], x.n = (int32_t)v[5];
    x.cu_rs = v[6], x.cu_cs = v[7], x.cv_rs = v[8], x.cv_cs = v[9], x.lds = (int32_t)v[10];
    x.xu_rs = v[11], x.xu_cs = v[12], x.xs_ld = (int32_t)v[13], x.xv_rs = v[14], x.xv_cs = v[15];
    std::printf("%d %d\n", (int)frk::near_addition<double>(x), (int)frk::near_addition<float>(x));
  }
}
