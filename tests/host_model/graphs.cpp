// Graphs of batched scenes, of one captured step and of scenes in one set:
// launched, tuned, reconfigured and destroyed with launches in flight.
#include <cstdio>
#include <vector>

#include "gg_internal.hpp"
#include "granular_gpu.h"
#include "runtime.hpp"

extern "C" int gg_step(gg_particles *, gg_adaptive *, int *, const gg_particles *, const int *,
                       const gg_params *, const gg_workspace *, hipStream_t) {
  return GG_OK;
}
extern "C" int gg_step_scenes(gg_particles *, int *, const gg_particles *, const int *,
                              const gg_scenes *, const gg_params *, const gg_workspace *,
                              hipStream_t) {
  return GG_OK;
}
namespace gg {
int grid_build_general(gg_particles *, gg_adaptive *, int *, int *, const gg_workspace *,
                       hipStream_t, int, const int *, int *) {
  return GG_OK;
}
int pack_boundary(const gg_particles *, const gg_workspace *, hipStream_t) { return GG_OK; }
}  // namespace gg

static int failed = 0;
static void check(int rc, const char *what) {
  if (rc != GG_OK) std::printf("%s: status %d\n", what, rc), ++failed;
  if (model().busy_releases) {
    std::printf("%s: %d releases in flight\n", what, model().busy_releases);
    model().busy_releases = 0;
    ++failed;
  }
}

int main() {
  const int kScenes = 64;
  std::vector<char> mem(1 << 20);
  int cell = 0;
  gg_batch_scene one{};
  one.set.n = 16;
  one.set.capacity = 16;
  one.cell_start = &cell;
  one.bcell_start = &cell;
  one.ws = gg_workspace{mem.data(), mem.size(), 16, 1, gg_grid{0.04f, 3, 3, 3}, 13, 4, 4};
  one.params.stab_iters = 3;
  one.params.solver_iters = 10;
  hipStream_t st = model_stream();

  std::vector<gg_batch_scene> sc(kScenes, one);
  for (int k = 0; k < kScenes; ++k) sc[k].set.n = 1 + (k * 7) % 16;
  gg_batch_config cfg{4, 0, 0, 1}, best{};
  float ms = 0.0f;
  gg_batch *b = nullptr;
  check(gg_batch_create(sc.data(), kScenes, &cfg, &b), "create");
  for (int k = 0; k < 20; ++k) check(gg_batch_step(b, st), "step");
  check(gg_batch_autotune(b, 5, st, &best, &ms), "autotune with steps in flight");
  check(gg_batch_step(b, st), "step");
  check(gg_batch_set_config(b, &cfg), "set_config with a step in flight");
  check(gg_batch_step(b, st), "step");
  gg_batch_destroy(b);
  check(GG_OK, "destroy with a step in flight");

  gg_step_graph *g = nullptr;
  check(gg_step_graph_create(&one.set, &cell, &one.boundary, &cell, &one.params, &one.ws, 2, &g),
        "create a step graph");
  check(gg_step_graph_launch(g, st), "launch");
  gg_step_graph_destroy(g);
  check(GG_OK, "destroy a step graph with a launch in flight");

  gg_scene_desc d[2] = {{2, 2, 2, 0, 0.5f, 0.4f}, {3, 2, 1, 9, 0.5f, 0.4f}};
  gg_workspace ws = one.ws;
  ws.grid = gg_grid{0.04f, 9 + 7 - 1, 1, 1};
  int of = 0;
  gg_scenes scenes{2, d, d, &of, &of, 1};
  gg_scenes_graph *s = nullptr;
  int sw = 0, nl = 0;
  check(gg_scenes_graph_create(&one.set, &cell, &one.boundary, &cell, &scenes, &one.params, &ws, 1,
                               &s), "create a scenes graph");
  for (int k = 0; k < 3; ++k) check(gg_scenes_graph_launch(s, st), "launch");
  check(gg_scenes_graph_autotune(s, 5, st, &sw, &nl, &ms), "autotune with launches in flight");
  check(gg_scenes_graph_launch(s, st), "launch");
  gg_scenes_graph_destroy(s);
  check(GG_OK, "destroy a scenes graph with a launch in flight");
  std::printf("launches %d\n", model().launches);
  return failed ? 1 : 0;
}
