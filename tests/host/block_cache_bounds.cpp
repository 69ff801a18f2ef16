// What a batch holds beside its jobs: idle blocks up to an eighth of its grid
// budget, and no block larger than a job's grid for that grid.
#include "fake_hip.hpp"
#include "sgtsne.h"

#include <vector>

int main() {
  sgtsne_params p;
  sgtsne_params_default(&p);
  p.d = 3;
  const int n = 2000, k = 10;
  std::vector<int32_t> rp(n + 1), col(n * k);
  std::vector<float> val(n * k, 1.0f);
  for (int i = 0; i <= n; ++i) rp[i] = i * k;
  for (int i = 0; i < n * k; ++i) col[i] = (i / k + 1 + i % k) % n;
  const int64_t budget = (int64_t)4 << 30;
  sgtsne_batch *b = nullptr;
  EXPECT(sgtsne_batch_create(&b, &p, 8, 100000, 1000000, budget) == 0);
  const size_t created = fake::live_bytes();
  int job = -1;
  auto add = [&](int ng_cap) {
    return sgtsne_batch_add(b, n, n * k, rp.data(), col.data(), val.data(), 0, nullptr, 5, ng_cap, &job);
  };
  const size_t small = (size_t)2 << 20;  // the blocks of the graph itself
  // jobs that come and go: what stays is within an eighth of the budget
  for (int ng_cap : {128, 64, 96, 80, 112, 48, 104, 72, 120}) {
    EXPECT(add(ng_cap) == 0);
    EXPECT(sgtsne_batch_remove(b, job) == 0);
  }
  EXPECT(sgtsne_batch_step(b, 0) == 0);  // idle blocks beyond the bound go back with the next call
  if (fake::live_bytes() - created > (size_t)budget / 8) {
    std::printf("%zu MB idle\n", (fake::live_bytes() - created) >> 20);
    return 1;
  }
  // each grid has a block of its own size, whatever lies idle
  for (int ng_cap : {100, 90, 76, 60}) EXPECT(add(ng_cap) == 0);
  int64_t grids = 0;
  EXPECT(sgtsne_batch_info(b, nullptr, nullptr, nullptr, &grids, nullptr) == 0);
  const size_t held = fake::live_bytes() - created;
  if (held > (size_t)grids + (size_t)budget / 8 + small) {
    std::printf("%zu MB held for %lld MB of grids\n", held >> 20, (long long)grids >> 20);
    return 1;
  }
  for (int j = 0; j < 4; ++j) EXPECT(sgtsne_batch_remove(b, j) == 0);
  // the next job of a size takes the block of the last one
  EXPECT(add(64) == 0);
  EXPECT(sgtsne_batch_remove(b, job) == 0);
  fake::reset_calls();
  EXPECT(add(64) == 0);
  EXPECT(fake::calls["hipMallocAsync"] == 0);
  EXPECT(sgtsne_batch_destroy(b) == 0);
  EXPECT(fake::live_bytes() == 0);
  return 0;
}
