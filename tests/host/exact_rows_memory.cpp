// Exact kNN rows of a job whose usual block of distances does not fit.
#include "fake_hip.hpp"
#include "sgtsne.h"

#include <vector>

int main() {
  // 128 rows of distances to 700,000 points are 717 MB
  const int n = 700000, k = 1;
  std::vector<float> X(n, 1.0f);
  std::vector<int32_t> I((size_t)n * (k + 1));
  std::vector<double> D((size_t)n * (k + 1));
  auto knn = [&] { return sgtsne_knn(X.data(), n, 1, k, SGTSNE_KNN_EXACT_FP64, I.data(), D.data(), nullptr); };
  for (size_t free : {(size_t)400 << 20, (size_t)100 << 20, (size_t)32 << 20}) {
    fake::capacity = free;
    const int st = knn();
    if (st) std::printf("%zu MB: %s\n", free >> 20, sgtsne_last_error());
    EXPECT(st == 0);
    EXPECT(fake::live_bytes() == 0);
    fake::pool.clear();
  }
  fake::capacity = (size_t)16 << 20;  // not even X, I and D
  EXPECT(knn() != 0);
  EXPECT(fake::live_bytes() == 0);
  fake::pool.clear();
  // many dimensions: the rows come from blocks of distances (655 rows of 100,000
  // are 512 MB) and not from heaps; X, I and D are 82 MB
  {
    const int n2 = 100000, dim2 = 200;
    std::vector<float> X2((size_t)n2 * dim2, 1.0f);
    for (size_t free : {(size_t)900 << 20, (size_t)300 << 20, (size_t)100 << 20}) {
      fake::capacity = free;
      const int st = sgtsne_knn(X2.data(), n2, dim2, 1, SGTSNE_KNN_EXACT_FP64, I.data(), D.data(), nullptr);
      if (st) std::printf("%zu MB: %s\n", free >> 20, sgtsne_last_error());
      EXPECT(st == 0);
      EXPECT(fake::live_bytes() == 0);
      fake::pool.clear();
    }
  }
  return 0;
}
