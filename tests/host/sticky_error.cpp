// An allocation that fails is reported by its own call and by no later one.
#include "fake_hip.hpp"
#include "sgtsne.h"

#include <vector>

int main() {
  sgtsne_params p;
  sgtsne_params_default(&p);
  const int n = 700, dim = 8, k = 20;
  std::vector<float> X(n * dim), val(n * k, 1.0f), Y(n * 2, 0.5f);
  for (size_t i = 0; i < X.size(); ++i) X[i] = (float)((i * 7919) % 1013);
  std::vector<int32_t> I(n * (k + 1)), rp(n + 1), col(n * k);
  std::vector<double> D(n * (k + 1));
  for (int i = 0; i <= n; ++i) rp[i] = i * k;
  for (int i = 0; i < n * k; ++i) col[i] = (i / k + 1 + i % k) % n;
  auto knn = [&] { return sgtsne_knn(X.data(), n, dim, k, SGTSNE_KNN_AUTO, I.data(), D.data(), nullptr); };
  auto equalize = [&] {
    return sgtsne_perplexity_equalize(I.data(), D.data(), n, k, 5.0, rp.data(), col.data(), val.data());
  };
  for (long at = 0; at < 3; ++at) {
    fake::fail("hipMallocAsync", at);
    const int st = knn();
    fake::succeed();
    EXPECT(at >= 2 || st != 0);
    EXPECT(knn() == 0);
  }
  fake::fail("hipMallocAsync", 0);
  EXPECT(equalize() != 0);
  fake::succeed();
  EXPECT(equalize() == 0);
  for (int i = 0; i < n * k; ++i) col[i] = (i / k + 1 + i % k) % n;  // (the copies above delivered zeros)
  for (long at = 0; at < 24; ++at) {
    sgtsne_ctx *c = nullptr;
    fake::fail("hipMalloc", at);
    int st = sgtsne_ctx_create(&c, &p);
    if (!st) st = sgtsne_ctx_upload_P(c, n, n * k, rp.data(), col.data(), val.data(), 0);
    if (!st) st = sgtsne_ctx_set_Y(c, Y.data(), SGTSNE_LAYOUT_AOS, 1);
    fake::succeed();
    if (c) EXPECT(sgtsne_ctx_destroy(c) == 0);
    sgtsne_ctx *o = nullptr;  // a context of its own, after the failure
    EXPECT(sgtsne_ctx_create(&o, &p) == 0);
    EXPECT(sgtsne_ctx_destroy(o) == 0);
  }
  return 0;
}
