// Two threads call gg_upsample_mlp on streams of their own: every wait must
// be for the waiting thread's own record.
#include <cstdio>
#include <thread>
#include <vector>

#include "granular_gpu.h"
#include "runtime.hpp"

namespace gg {
void prof_begin(int, hipStream_t) {}
void prof_end(int, hipStream_t) {}
}  // namespace gg

int main() {
  model().yield_ms = 50;
  int bad = 0;
  for (int n : {1000, 300000}) {  // flags on the caller's stream, on the side stream
    auto call = [&] {
      gg_float3 one{};
      gg_particles coarse{}, boundary{};
      coarse.n = n;
      coarse.pos = coarse.vel = &one;
      gg_upsample_params u{};
      gg_mlp_config c;
      gg_mlp_config_default(&c);
      const gg_grid g{0.04f, 8, 8, 8};
      const uint16_t w = 0;
      const float b = 0.0f;
      float f = 0.0f;
      int cell = 0;
      static char scratch[1];  // never read: kernels do nothing here
      const int rc = gg_upsample_mlp(&coarse, &cell, &boundary, &cell, g, &u, &c, &w, &b, &f, &f,
                                     scratch, gg_upsample_mlp_scratch_bytes(n), nullptr,
                                     model_stream());
      if (rc != GG_OK) std::printf("status %d\n", rc), ++bad;
    };
    std::thread a(call), b(call);
    a.join();
    b.join();
  }
  std::printf("waits %d foreign %d\n", model().waits, model().foreign_waits);
  return bad || model().waits < 8 || model().foreign_waits ? 1 : 0;
}
