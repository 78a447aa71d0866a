// Rays per sample of an image, estimated from a few of its paths.
#pragma once

#include "renderer.h"

namespace pt {
namespace host {

// Mean number of rays (camera, light and continuation) of a sample of the
// image, up to its fourth vertex: paths through points spread over the film,
// with the render's own materials, light samples and path ends, traced in the
// scene's host tree. Fewer paths are traced once the mean is clearly above or
// below `line`.
float rays_per_sample(const pt_scene &scene, const pt_settings &settings,
                      const float film_to_world[12], uint32_t x_dim, uint32_t y_dim, float line);

} // namespace host
} // namespace pt
