// Host-side check of the small DFTs (kcommon.h), built by tests/test_small_dft.py with hipcc for the host only. For 100,000
// random inputs of every radix and direction, against the DFT in long double: the error of each output relative to the
// input, and the part of it that always points the same way (the output's gain, which adds up from stage to stage where
// rounding errors average out). Prints a line per radix and direction: radix, inverse, rms error, largest gain error, both in
// units of 2^-53.
#include <hip/hip_runtime.h>
#undef __device__
#define __device__ __attribute__((host)) __attribute__((device))
#include "kcommon.h"

#include <cmath>
#include <complex>
#include <cstdio>
#include <random>

template<int R, bool INV> void check() {
  using C = std::complex<long double>;
  const long double turn = (INV ? 2 : -2) * 3.141592653589793238462643383279502884L / R;
  C w[R];
  for (int k = 0; k < R; ++k) { w[k] = {cosl(turn * k), sinl(turn * k)}; }
  std::mt19937_64 gen(R);
  std::normal_distribution<double> normal;
  long double along[R] = {}, power[R] = {}, err = 0, all = 0;
  for (int n = 0; n < 100000; ++n) {
    T2 a[R];
    C in[R];
    for (int k = 0; k < R; ++k) {
      a[k] = make_double2(normal(gen), normal(gen));
      in[k] = {a[k].x, a[k].y};
    }
    Dft<R, INV>::run(a);
    for (int m = 0; m < R; ++m) {
      C ref = 0;
      for (int k = 0; k < R; ++k) { ref += in[k] * w[k * m % R]; }
      const C e = C(a[m].x, a[m].y) - ref;
      along[m] += (std::conj(ref) * e).real();
      power[m] += std::norm(ref);
      err += std::norm(e);
      all += std::norm(ref);
    }
  }
  long double gain = 0;
  for (int m = 0; m < R; ++m) { gain = std::max(gain, std::fabs(along[m] / power[m])); }
  const long double u = 0x1p-53L;
  std::printf("%d %d %.4Lf %.4Lf\n", R, int(INV), std::sqrt(err / all) / u, gain / u);
}
template<int... Rs> void checkAll() { (..., (check<Rs, false>(), check<Rs, true>())); }

int main() { checkAll<2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>(); }
