// CPU harness for the wide kernels' host-checkable arithmetic: the exact soft
// moments (ace_bins.hpp: exact_moment_scale) and the launch geometry
// (ace_geometry.hpp: make_wide_geometry).  Built with g++ by
// tests/test_wide.py and called through ctypes.
#include <cmath>
#include <cstdint>
#include <cstring>

#include "ace_bins.hpp"
#include "ace_geometry.hpp"

namespace {
float from_bits(uint32_t b) {
  float f;
  std::memcpy(&f, &b, 4);
  return f;
}
uint32_t to_bits(float f) {
  uint32_t b;
  std::memcpy(&b, &f, 4);
  return b;
}
}  // namespace

extern "C" {

// Violations of the exact moments over every `step`-th float32 p in [0, 1] and
// every p within `width` ulp of the 2K upper half boundaries `table`: with h
// the half-bin, u = fma(p, 2^m, -(h w)) in float32 must equal the exact
// p 2^m - h w (double holds it), be non-negative and below `umax`, and for
// h >= 1 be an integer.  plant != 0 plants a base that keeps too many bits.
long long check_exact_moments(const float* table, int num_bins, int width, int step, double umax,
                              int plant) {
  ace::MomentScale s = ace::exact_moment_scale(num_bins);
  if (plant) s.w |= 1;
  const int n = 2 * num_bins;
  const float sc = std::ldexp(1.0f, s.m);
  auto check = [&](float p, bool right) -> long long {
    int h = 0;
    // upper boundaries below p (or equal, right): the kernels' half-bin
    int lo = 0, hi = n;
    while (lo < hi) {
      const int mid = (lo + hi) / 2;
      if (right ? table[mid] <= p : table[mid] < p)
        lo = mid + 1;
      else
        hi = mid;
    }
    h = lo < n ? lo : n - 1;
    const float hw = (float)h * -(float)s.w;
    if ((double)hw != (double)h * -(double)s.w) return 1;
    const float u = std::fmaf(p, sc, hw);
    const double exact = std::ldexp((double)p, s.m) - (double)h * (double)s.w;
    if ((double)u != exact || u < 0.0f || (double)u >= umax) return 1;
    if (h >= 1 && u != std::floor(u)) return 1;
    return 0;
  };
  long long bad = 0;
  const int64_t one = to_bits(1.0f);
  for (int j = 0; j < n; ++j)
    for (int64_t d = -width; d <= width; ++d) {
      const int64_t bits = (int64_t)to_bits(table[j]) + d;
      if (bits < 0 || bits > one) continue;
      for (int r = 0; r < 2; ++r) bad += check(from_bits((uint32_t)bits), r != 0);
    }
  for (int64_t bits = 0; bits <= one; bits += step) bad += check(from_bits((uint32_t)bits), false);
  return bad;
}

// out: {cmax, vec, copies, steps, lds_fwd, lds_bwd, tiles, ws_bytes, largest count of a copy}
void wide_geometry(long long B, long long C, long long N, int K, int soft, int bg, int labels, int elem,
                   int backward, long long* out) {
  const ace::Geometry g = ace::make_wide_geometry(B, C, N, K, soft != 0, bg != 0, labels != 0,
                                               (size_t)elem, backward != 0);
  out[0] = g.var.cmax;
  out[1] = g.var.vec;
  out[2] = g.copies;
  out[3] = g.steps;
  out[4] = (long long)g.lds_fwd;
  out[5] = (long long)g.lds_bwd;
  out[6] = g.tiles;
  out[7] = (long long)g.ws_bytes;
  out[8] = (long long)(g.nt / g.copies) * g.steps * g.var.vec;
}

// 1: the wide kernel takes the soft forward, 0: the generic one.
int soft_forward_wide(long long B, long long C, long long N, int K, int bg, int labels) {
  const ace::Geometry w = ace::make_wide_geometry(B, C, N, K, true, bg != 0, labels != 0, 4, false);
  const ace::Geometry g = ace::make_geometry(B, C, N, K, true, bg != 0, labels != 0);
  return ace::wide_soft_forward_pays(w, g, labels != 0) ? 1 : 0;
}

int exact_shift(long long voxels, int first) {
  return first ? ace::exact_moment_shift0(voxels) : ace::exact_moment_shift(voxels);
}

}  // extern "C"
