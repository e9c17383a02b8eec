// The job server's admission (serve.cpp) over a model of the context calls that
// hold a job in its k-mer run until `together` jobs are in theirs, or a second
// has passed.  Built and run by test_serve_admission.py; prints "ok" or what
// was broken.
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <string>
#include <vector>

#include "crispy_hip.h"

struct crispy_ctx {
  int64_t limit = 0, scratch_limit = -1, held = 0, scratch = 0;
  int32_t n = 0;
};

namespace {
std::mutex mu;
std::condition_variable cv;
int inside = 0, most = 0, together = 0;
}  // namespace

extern "C" {
int crispy_ctx_create(int, crispy_ctx **o) {
  *o = new crispy_ctx();
  return CRISPY_OK;
}
void crispy_ctx_destroy(crispy_ctx *c) { delete c; }
const char *crispy_ctx_error(const crispy_ctx *) { return "model"; }
int crispy_ctx_sync(crispy_ctx *) { return CRISPY_OK; }
int64_t crispy_ctx_device_bytes(const crispy_ctx *c) { return c->held + c->scratch; }
int64_t crispy_ctx_scratch_bytes(const crispy_ctx *c) { return c->scratch; }
int crispy_ctx_set_mem_limit(crispy_ctx *c, int64_t b) {
  c->limit = b;
  return CRISPY_OK;
}
int crispy_ctx_set_scratch_limit(crispy_ctx *c, int64_t b) {
  c->scratch_limit = b;
  return CRISPY_OK;
}
int crispy_ctx_trim(crispy_ctx *c) {
  c->held = c->scratch = 0;
  return CRISPY_OK;
}
int crispy_host_alloc(int64_t b, void **o) {
  *o = b ? std::malloc((size_t)b) : nullptr;
  return CRISPY_OK;
}
int crispy_host_free(void *p) {
  std::free(p);
  return CRISPY_OK;
}
int crispy_reads_upload(crispy_ctx *c, int, const char *, const int64_t *, int32_t n) {
  c->n = n;
  return CRISPY_OK;
}
int crispy_kmer_run(crispy_ctx *c, int, float, int64_t, int64_t, int64_t *k) {
  c->held = c->limit;  // all that the job is charged
  if (c->scratch_limit > c->scratch) c->scratch = c->scratch_limit;
  std::unique_lock<std::mutex> lk(mu);
  most = std::max(most, ++inside);
  cv.notify_all();
  cv.wait_for(lk, std::chrono::seconds(1), [] { return most >= together; });
  --inside;
  if (k) *k = c->n;
  return CRISPY_OK;
}
int crispy_nw_run_on_kmer(crispy_ctx *, int, float, int64_t *c) {
  *c = 0;
  return CRISPY_OK;
}
int crispy_nw_fetch(crispy_ctx *, int64_t, int64_t, int32_t *, float *) { return CRISPY_OK; }
int crispy_nw_csr(crispy_ctx *, int32_t n, int64_t *r, int32_t *, float *) {
  for (int32_t q = 0; q <= n; ++q) r[q] = 0;
  return CRISPY_OK;
}
}

int main() {
  struct Reads {
    std::string bases;
    std::vector<int64_t> off{0};
    explicit Reads(int n) : bases((size_t)n * 300, 'A') {
      for (int r = 1; r <= n; ++r) off.push_back((int64_t)r * 300);
    }
    int32_t n() const { return (int32_t)off.size() - 1; }
    int64_t est() const { return crispy_server_job_bytes(bases.data(), off.data(), n(), 6, 10); }
  } small(2000), large(10000);
  // a large job and three small ones, whose estimates the budget holds together
  const int64_t budget = large.est() + 3 * small.est() + small.est() / 2;
  for (int round = 0; round < 3; ++round) {  // the second and third on slots that hold the first's buffers
    crispy_server *srv = nullptr;
    if (crispy_server_create(0, 4, budget, &srv) != CRISPY_OK) return 1;
    for (int burst = 0; burst <= round; ++burst) {
      {
        std::lock_guard<std::mutex> lk(mu);
        together = 4;
        most = inside = 0;
      }
      std::vector<int64_t> ids;
      for (int k = 0; k < 4; ++k) {
        const Reads &r = k == 0 ? large : small;
        ids.push_back(crispy_server_submit(srv, r.bases.data(), r.off.data(), nullptr, nullptr, r.n(), 6, 0.2f, 10, 0.1f));
      }
      for (int64_t id : ids) {
        int64_t est = 0, held = 0;
        if (crispy_server_wait(srv, id, nullptr, nullptr, nullptr, nullptr) != CRISPY_OK) std::printf("a job failed\n");
        crispy_server_job_times(srv, id, nullptr, nullptr, nullptr, &est, &held);
        if (crispy_server_fetch(srv, id, nullptr, nullptr) != CRISPY_OK) std::printf("no result\n");
      }
      if (most < 4) std::printf("%d of 4 jobs that fit together ran together (burst %d of %d)\n", most, burst, round);
    }
    int64_t peak = 0;
    crispy_server_status(srv, nullptr, nullptr, nullptr, &peak);
    if (peak > budget) std::printf("%lld bytes charged of %lld\n", (long long)peak, (long long)budget);
    crispy_server_destroy(srv);
  }
  std::printf("ok\n");
  return 0;
}
