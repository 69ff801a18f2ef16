// The points and rows of a large search do not stay in the device's pool.
#include "fake_hip.hpp"
#include "sgtsne.h"

#include <vector>

int main() {
  sgtsne_params p;
  sgtsne_params_default(&p);
  sgtsne_ctx *c = nullptr;  // from here on the pool keeps what is freed to it
  EXPECT(sgtsne_ctx_create(&c, &p) == 0);
  const size_t limit = (size_t)256 << 20;
  for (int n : {2000, 400000}) {
    const int k = 90;
    std::vector<int32_t> I((size_t)n * (k + 1)), rp(n + 1), col((size_t)n * k);
    std::vector<double> D((size_t)n * (k + 1));
    std::vector<float> val((size_t)n * k);
    fake::pool.clear();
    EXPECT(sgtsne_perplexity_equalize(I.data(), D.data(), n, k, 30.0, rp.data(), col.data(), val.data()) == 0);
    if (fake::pool_bytes() > limit) {
      std::printf("n %d: %zu MB kept\n", n, fake::pool_bytes() >> 20);
      return 1;
    }
  }
  {  // the pool keeps the scratch of a search, as any other call's, but not X, I and D
    const int n = 1000000, k = 20, dim = 8;
    std::vector<float> X((size_t)n * dim);
    std::vector<int32_t> I((size_t)n * (k + 1));
    std::vector<double> D((size_t)n * (k + 1));
    fake::pool.clear();
    fake::reset_calls();
    EXPECT(sgtsne_knn(X.data(), n, dim, k, SGTSNE_KNN_FILTERED, I.data(), D.data(), nullptr) == 0);
    EXPECT(fake::calls["hipMalloc"] == 1 && fake::calls["hipMallocAsync"] == 1);
    EXPECT(sgtsne_knn(X.data(), 2000, dim, k, SGTSNE_KNN_FILTERED, I.data(), D.data(), nullptr) == 0);
    EXPECT(fake::calls["hipMalloc"] == 1);
  }
  EXPECT(sgtsne_ctx_destroy(c) == 0);
  EXPECT(fake::live_bytes() == 0);
  return 0;
}
