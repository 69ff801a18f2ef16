// A job whose grid does not fit beside a batch's idle blocks gets their memory.
#include "fake_hip.hpp"
#include "sgtsne.h"

#include <vector>

int main() {
  sgtsne_params p;
  sgtsne_params_default(&p);
  const int n = 3000, k = 10;
  std::vector<int32_t> rp(n + 1), col(n * k);
  std::vector<float> val(n * k, 1.0f);
  for (int i = 0; i <= n; ++i) rp[i] = i * k;
  for (int i = 0; i < n * k; ++i) col[i] = (i / k + 1 + i % k) % n;
  for (int d = 2; d <= 3; ++d) {
    p.d = d;
    sgtsne_batch *b = nullptr;
    EXPECT(sgtsne_batch_create(&b, &p, 4, 100000, 1000000, 0) == 0);
    int job = -1;
    auto add = [&](int ng_cap) {
      return sgtsne_batch_add(b, n, n * k, rp.data(), col.data(), val.data(), 0, nullptr, 5, ng_cap, &job);
    };
    EXPECT(add(d == 2 ? 512 : 128) == 0);
    EXPECT(sgtsne_batch_remove(b, job) == 0);
    // a grid of another size class, with less free than it needs
    fake::capacity = fake::live_bytes() + fake::pool_bytes() + (1 << 20);
    const int st = add(d == 2 ? 256 : 64);
    if (st) std::printf("%s\n", sgtsne_last_error());
    EXPECT(st == 0);
    // and what cannot fit at all is refused, with the batch as it was
    fake::capacity = fake::live_bytes() + fake::pool_bytes() + (1 << 20);
    EXPECT(add(d == 2 ? 512 : 128) == SGTSNE_ERR_NOMEM);
    int jobs = 0;
    EXPECT(sgtsne_batch_info(b, &jobs, nullptr, nullptr, nullptr, nullptr) == 0 && jobs == 1);
    fake::capacity = ~(size_t)0 >> 2;
    EXPECT(sgtsne_batch_destroy(b) == 0);
    EXPECT(fake::live_bytes() == 0);
  }
  return 0;
}
