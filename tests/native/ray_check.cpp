// ray_can_hit (core/geometry.h) on the host.
#include "../../path_amd/csrc/core/geometry.h"

using namespace pt;

extern "C" void rays_can_hit(const float *rays, int n, unsigned char *out) {
  for (int i = 0; i < n; ++i) {
    const float *r = rays + 6 * i;
    out[i] = ray_can_hit(Ray<float>{{r[0], r[1], r[2]}, {r[3], r[4], r[5]}});
  }
}
