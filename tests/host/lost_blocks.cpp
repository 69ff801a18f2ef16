// A call that fails part of the way gives back what it had taken.
#include "fake_hip.hpp"
#include "sgtsne.h"

#include <vector>

struct Graph {
  int n;
  std::vector<int32_t> rp, col;
  std::vector<float> val;
};
static Graph ring(int n, int k) {
  Graph g{n, {}, {}, {}};
  for (int i = 0; i <= n; ++i) g.rp.push_back(i * k);
  for (int i = 0; i < n; ++i)
    for (int e = 1; e <= k; ++e) {
      g.col.push_back((i + e) % n);
      g.val.push_back(1.0f);
    }
  return g;
}

int main() {
  sgtsne_params p;
  sgtsne_params_default(&p);
  const char *kinds[] = {"hipMallocAsync", "hipLaunchKernel", "hipStreamSynchronize", "hipMemcpyAsync"};

  // a batch: the front end of a graph job, failing at its i-th allocation,
  // launch, wait or copy (up to the copy of the merged rows; the admission that
  // follows belongs to the arena)
  sgtsne_batch *b = nullptr;
  EXPECT(sgtsne_batch_create(&b, &p, 4, 100000, 10000000, 0) == 0);
  const size_t created = fake::live_bytes();
  const Graph g = ring(3000, 30), large = ring(60000, 60);
  int job = -1;
  auto add = [&](const Graph &h) {
    return sgtsne_batch_add(b, h.n, h.rp[h.n], h.rp.data(), h.col.data(), h.val.data(), 1, nullptr, 5, 0, &job);
  };
  const long front_end[] = {4, 8, 3, 4};
  for (int k = 0; k < 4; ++k)
    for (long at = 0; at < front_end[k]; ++at) {
      fake::fail(kinds[k], at);
      const int st = add(g);
      fake::succeed();
      (void)hipGetLastError();
      if (st == 0) EXPECT(sgtsne_batch_remove(b, job) == 0);
      // an allocation that cannot be had gives every idle block back: what is
      // left then was lost
      fake::fail("hipMallocAsync", 0);
      EXPECT(add(large) == SGTSNE_ERR_NOMEM);
      fake::succeed();
      (void)hipGetLastError();
      if (fake::live_bytes() != created) {
        std::printf("%s %ld: %zu bytes lost\n", kinds[k], at, fake::live_bytes() - created);
        return 1;
      }
    }
  EXPECT(sgtsne_batch_destroy(b) == 0);
  EXPECT(fake::live_bytes() == 0);

  // the calls that take their scratch from the device's pool
  const int n = 700, dim = 8, kk = 20;
  std::vector<float> X(n * dim);
  for (size_t i = 0; i < X.size(); ++i) X[i] = (float)((i * 7919) % 1013);
  std::vector<int32_t> I(n * (kk + 1));
  std::vector<double> D(n * (kk + 1));
  int fb = 0;
  for (int method : {SGTSNE_KNN_FILTERED, SGTSNE_KNN_EXACT_FP64})
    for (const char *kind : kinds)
      for (long at = 0; at < 12; ++at) {
        fake::fail(kind, at);
        (void)sgtsne_knn(X.data(), n, dim, kk, method, I.data(), D.data(), &fb);
        fake::succeed();
        (void)hipGetLastError();
        if (fake::live_bytes() != 0) {
          std::printf("knn %d %s %ld: %zu bytes\n", method, kind, at, fake::live_bytes());
          return 1;
        }
      }
  // P + P^T of a context: the pool's blocks are back although the call failed
  for (const char *kind : kinds)
    for (long at = 0; at < 12; ++at) {
      sgtsne_ctx *c = nullptr;
      p.reorder = 0;
      EXPECT(sgtsne_ctx_create(&c, &p) == 0);
      fake::fail(kind, at);
      (void)sgtsne_ctx_upload_P(c, g.n, g.rp[g.n], g.rp.data(), g.col.data(), g.val.data(), 1);
      fake::succeed();
      (void)hipGetLastError();
      size_t pooled = 0;
      for (auto &e : fake::live) pooled += e.second.pooled ? e.second.bytes : 0;
      if (pooled) {
        std::printf("upload_P %s %ld: %zu bytes of the pool\n", kind, at, pooled);
        return 1;
      }
      EXPECT(sgtsne_ctx_destroy(c) == 0);
      fake::live.clear();
    }
  return 0;
}
