// A batch's launches for a made-up number of tasks (test_batch_errors.py).
#include "strip_moment.hpp"

extern "C" int launch_tasks(int backward, int waves, int n_tasks) {
  strip::MomentBatch batch;
  batch.launches.push_back({backward != 0, 8, waves, false, 1024, 0, n_tasks});
  std::string err;
  return strip::moment_batch_launch(batch, 0, backward != 0, nullptr, &err);
}
