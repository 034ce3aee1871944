// What the runtime model (runtime.cpp) has counted, and its one setting.
#pragma once
#include <hip/hip_runtime_api.h>

struct Model {
  int yield_ms = 0;  // how long a record waits for another thread's of the same event
  int waits = 0, foreign_waits = 0, launches = 0, busy_releases = 0;
};
Model &model();
hipStream_t model_stream();
