// Host path tracing for the estimate of an image's rays per sample.
#include "ray_estimate.h"

#include "../core/camera.h"
#include "../core/rng.h"
#include "settings.h"

#include <cmath>
#include <vector>

namespace pt {
namespace host {

namespace {

// Closest hit in the host tree; `stack` has room for the tree's depth.
Hit<float> closest_hit(const Bvh &bvh, const std::vector<TriGeom<float>> &tris,
                       const Ray<float> &ray, std::vector<uint32_t> &stack) {
  Hit<float> best = {3.4028235e38f, kNoHit, 0};
  if (bvh.nodes.empty() || !ray_can_hit(ray))
    return best;
  const V3<float> inv = inv_direction(ray.d);
  auto enters = [&](uint32_t node, float *t) {
    float t1;
    return slab_test(bvh.nodes[node].lo, bvh.nodes[node].hi, ray.o, inv, t, &t1) && t1 >= 0.f &&
           *t <= best.t;
  };
  uint32_t node = 0;
  float t;
  if (!enters(0, &t))
    return best;
  stack.clear();
  for (;;) {
    const BvhNode &n = bvh.nodes[node];
    if (n.is_leaf) {
      for (uint32_t i = n.a; i < n.b; ++i) {
        uint32_t back;
        if (intersect_triangle(ray, tris[bvh.perm[i]], &t, &back) && t < best.t)
          best = {t, bvh.perm[i], back};
      }
    } else {
      float ta, tb;
      const bool a = enters(n.a, &ta), b = enters(n.b, &tb);
      if (a || b) {
        const bool b_first = b && (!a || tb < ta);
        if (a && b)
          stack.push_back(b_first ? n.a : n.b);
        node = b_first ? n.b : n.a;
        continue;
      }
    }
    do {
      if (stack.empty())
        return best;
      node = stack.back();
      stack.pop_back();
    } while (!enters(node, &t));
  }
}

} // namespace

float rays_per_sample(const pt_scene &scene, const pt_settings &settings,
                      const float film_to_world[12], uint32_t x_dim, uint32_t y_dim, float line) {
  constexpr uint32_t kGroup = 8, kMost = 32, kVertices = 4;
  const FlatScene &f = scene.flat();
  const PackedScene &packed = scene.packed();
  const Bvh &bvh = scene.bvh();
  const IntegratorSettings s = integrator_settings(settings);
  const SceneView<float> view = {packed.shade.data(), packed.mats.data(), f.light_tris.data(),
                                 f.light_cdf.data(), uint32_t(f.light_tris.size())};
  std::vector<uint32_t> stack;
  stack.reserve(bvh.max_depth + 1);
  float sum = 0.f, squares = 0.f, mean = 0.f;
  for (uint32_t i = 0; i < kMost; ++i) {
    // (the additive recurrence of the plastic number: points in the unit square)
    float fx = 0.5f + 0.75487767f * float(i), fy = 0.5f + 0.56984029f * float(i);
    fx -= std::floor(fx);
    fy -= std::floor(fy);
    HashRng rng = make_hash_rng(i);
    Ray<float> ray =
        camera_ray(film_to_world, fx * float(x_dim), fy * float(y_dim), x_dim, y_dim);
    PathState<float> st = initial_path_state<float>();
    uint32_t rays = 0;
    for (uint32_t k = 0; k < kVertices; ++k) {
      rays += st.has_next + st.n_light;
      Hit<float> hit = {0.f, kNoHit, 0};
      if (st.has_next && k + 1 < kVertices)
        hit = closest_hit(bvh, f.tris, ray, stack);
      PathState<float> ns;
      Ray<float> light = ray, next = ray;
      if (rendering_equation_iteration(st, rng, ray, Hit<float>{0.f, kNoHit, 0}, hit, s, view,
                                       &ns, &light, &next))
        break;
      st = ns;
      ray = next;
    }
    sum += float(rays);
    squares += float(rays * rays);
    if ((i + 1) % kGroup != 0)
      continue;
    // (2.5 standard errors of the mean from the line)
    const float n = float(i + 1);
    mean = sum / n;
    const float off = mean - line, var = squares / n - mean * mean;
    if (off * off * n > 6.25f * var)
      break;
  }
  return mean;
}

} // namespace host
} // namespace pt
