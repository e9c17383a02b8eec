// run_segment (graph_segment.hpp) against a model of the HIP runtime: streams
// that run nothing until they are waited for, graphs as lists of launches.
// Built and run by test_graph_segment.py; prints "ok" or what was broken.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "graph_segment.hpp"

namespace {

struct Launch {
  const void *func;
  uintptr_t arg;
  bool operator==(const Launch &o) const { return func == o.func && arg == o.arg; }
};
struct FakeGraph {
  std::vector<Launch> nodes;
};
struct FakeExec {
  std::vector<Launch> nodes;
  bool running = false;
};

bool capturing = false;
FakeGraph captured;
std::vector<Launch> ran;          // what the stream got, in order
std::vector<FakeExec *> running;  // execs launched since the last wait
int graphs_alive = 0, execs_alive = 0, instantiations = 0, captures = 0;

void fail(const char *what) {
  std::printf("%s\n", what);
  std::exit(1);
}

}  // namespace

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  capturing = true;
  captured.nodes.clear();
  ++captures;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  capturing = false;
  *g = reinterpret_cast<hipGraph_t>(new FakeGraph(captured));
  ++graphs_alive;
  return hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t g, hipGraphNode_t *nodes, size_t *n) {
  auto *f = reinterpret_cast<FakeGraph *>(g);
  *n = f->nodes.size();
  for (size_t k = 0; nodes && k < *n; ++k) nodes[k] = reinterpret_cast<hipGraphNode_t>(&f->nodes[k]);
  return hipSuccess;
}
hipError_t hipGraphNodeGetType(hipGraphNode_t, hipGraphNodeType *t) {
  *t = hipGraphNodeTypeKernel;
  return hipSuccess;
}
hipError_t hipGraphKernelNodeGetParams(hipGraphNode_t n, hipKernelNodeParams *p) {
  p->func = const_cast<void *>(reinterpret_cast<Launch *>(n)->func);
  return hipSuccess;
}
hipError_t hipGraphExecUpdate(hipGraphExec_t e, hipGraph_t g, hipGraphNode_t *, hipGraphExecUpdateResult *r) {
  auto *x = reinterpret_cast<FakeExec *>(e);
  auto *f = reinterpret_cast<FakeGraph *>(g);
  if (x->running) fail("an exec is updated while its last launch runs");
  if (x->nodes.size() != f->nodes.size()) fail("an exec is updated with a graph of another size");
  for (size_t k = 0; k < x->nodes.size(); ++k)
    if (x->nodes[k].func != f->nodes[k].func) fail("an exec is updated with a graph of other kernels");
  x->nodes = f->nodes;
  *r = hipGraphExecUpdateSuccess;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(new FakeExec{reinterpret_cast<FakeGraph *>(g)->nodes});
  ++execs_alive;
  ++instantiations;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete reinterpret_cast<FakeGraph *>(g);
  --graphs_alive;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  auto *x = reinterpret_cast<FakeExec *>(e);
  if (x->running) fail("an exec is destroyed while its last launch runs");
  delete x;
  --execs_alive;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  auto *x = reinterpret_cast<FakeExec *>(e);
  x->running = true;
  running.push_back(x);
  ran.insert(ran.end(), x->nodes.begin(), x->nodes.end());
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  for (FakeExec *x : running) x->running = false;
  running.clear();
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }

namespace crispy {
int set_err(crispy_ctx *, int code, const char *, ...) { return code; }
int wait_main(crispy_ctx *ctx) {
  (void)hipStreamSynchronize(ctx->stream);
  ctx->settled = ctx->launches;
  return CRISPY_OK;
}
}  // namespace crispy

int main() {
  crispy_ctx ctx;
  const char kernels[4] = {};
  std::mt19937 rng(1);
  auto run = [&](GraphSegment &g, int set, uintptr_t arg) {
    std::vector<Launch> want;
    for (int k = 0; k < 4; ++k)
      if (set >> k & 1) want.push_back({&kernels[k], arg});
    const size_t before = ran.size();
    const int rc = crispy::run_segment(&ctx, g, {(uintptr_t)set, arg}, "check", [&](bool) -> int {
      auto &to = capturing ? captured.nodes : ran;
      to.insert(to.end(), want.begin(), want.end());
      return CRISPY_OK;
    });
    if (rc != CRISPY_OK) fail("a run failed");
    if (std::vector<Launch>(ran.begin() + before, ran.end()) != want) fail("a run launched something else");
  };
  {  // jobs that all differ build no graph
    GraphSegment g;
    for (uintptr_t job = 0; job < 100; ++job) {
      run(g, 1 + job % 15, job);
      if (job % 3) (void)crispy::wait_main(&ctx);
    }
    if (captures || instantiations) fail("graphs are built for runs that do not come again");
    // a run that repeats is captured once, then replayed
    for (int k = 0; k < 10; ++k) run(g, 5, 7);
    if (captures != 1 || instantiations != 1) fail("a repeated run is not replayed");
    crispy::drop_segment((crispy::wait_main(&ctx), g));
  }
  for (int round = 0; round < 200; ++round) {  // any order of runs, waits and kernel sets
    GraphSegment g[2];
    for (int k = 0; k < 200; ++k) {
      const unsigned r = rng();
      for (unsigned rep = 0; rep <= (r >> 8) % 4; ++rep) {
        run(g[r & 1], 1 + (r >> 1) % 3, (r >> 4) % 3);
        if (rng() % 3 == 0) (void)crispy::wait_main(&ctx);
      }
    }
    (void)crispy::wait_main(&ctx);
    for (GraphSegment &x : g) crispy::drop_segment(x);
    if (graphs_alive || execs_alive) fail("graphs are left over");
  }
  std::printf("ok\n");
  return 0;
}
