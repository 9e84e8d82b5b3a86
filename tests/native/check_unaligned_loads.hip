// Host check of the piecewise loads in csrc/mgq_common.h, built with the
// compiler's alignment check as a trap: two and four floats from every address aligned
// to one float, two doubles from every address aligned to one double. Exit
// status 0 iff every load gives the values that lie there.
#include <cstdio>

#include "mgq_common.h"

int main() {
  alignas(16) float f[12];
  alignas(16) double d[8];
  for (int i = 0; i < 12; ++i) f[i] = static_cast<float>(i);
  for (int i = 0; i < 8; ++i) d[i] = i;
  int bad = 0;
  for (int o = 0; o < 8; ++o) {
    const auto v = mgq::load_f32x4(f + o);
    for (int k = 0; k < 4; ++k) bad += v[k] != static_cast<float>(o + k);
    const auto u = mgq::load_f32x2(f + o);
    for (int k = 0; k < 2; ++k) bad += u[k] != static_cast<float>(o + k);
  }
  for (int o = 0; o < 6; ++o) {
    const auto v = mgq::load_f64x2(d + o);
    for (int k = 0; k < 2; ++k) bad += v[k] != static_cast<double>(o + k);
  }
  printf("mismatches=%d\n", bad);
  return bad != 0;
}
