// Captured launch sequences.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>
#include <vector>

#include "common.hpp"

namespace crispy {

inline void drop_segment(GraphSegment &g) {
  if (g.exec) (void)hipGraphExecDestroy(g.exec);
  g = GraphSegment();
}

// The kernel functions of a captured graph's nodes, in node order (another
// node's type in its place).  A graph must hold kernels and event dependencies
// only: memset nodes, which have given wrong results on replays, are refused.
inline int graph_kernels(crispy_ctx *ctx, hipGraph_t graph, const char *what, std::vector<const void *> *kernels) {
  size_t nn = 0;
  CRISPY_HIP(ctx, hipGraphGetNodes(graph, nullptr, &nn));
  std::vector<hipGraphNode_t> nodes(nn);
  if (nn) CRISPY_HIP(ctx, hipGraphGetNodes(graph, nodes.data(), &nn));
  for (hipGraphNode_t node : nodes) {
    hipGraphNodeType t;
    CRISPY_HIP(ctx, hipGraphNodeGetType(node, &t));
    if (t == hipGraphNodeTypeMemset)
      return set_err(ctx, CRISPY_ERR_HIP, "capturing %s: the graph holds a memset node", what);
    hipKernelNodeParams params = {};
    if (t == hipGraphNodeTypeKernel) CRISPY_HIP(ctx, hipGraphKernelNodeGetParams(node, &params));
    kernels->push_back(t == hipGraphNodeTypeKernel ? params.func : reinterpret_cast<const void *>((uintptr_t)t));
  }
  return CRISPY_OK;
}

// Runs enqueue(true) on the main stream, through the segment's graph where its
// key comes a second time in a row: a program that repeats a run replays, one
// whose runs all differ (a server's jobs) builds no graph at all.  A graph of
// the same kernels takes over the instantiated one in place
// (hipGraphExecUpdate with new arguments); one of other kernels replaces it.
// Either way the last launch of the old one has ended first.  The key must
// hold every argument of the launches, and which kernels they are must
// determine their dependencies.
template <class Enqueue>
int run_segment(crispy_ctx *ctx, GraphSegment &g, std::vector<uintptr_t> key, const char *what,
                Enqueue &&enqueue) {
  if (!ctx->graphs) return enqueue(false);
  if (!g.exec || key != g.key) {
    if (key != g.seen) {
      g.seen = std::move(key);
      return enqueue(true);
    }
    g.key.clear();
    CRISPY_HIP(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    const int rc = enqueue(true);
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(ctx->stream, &graph);
    struct Graph {
      hipGraph_t g;
      ~Graph() {
        if (g) (void)hipGraphDestroy(g);
      }
    } owner{graph};
    if (rc != CRISPY_OK) return rc;
    if (e != hipSuccess) return set_err(ctx, CRISPY_ERR_HIP, "capturing %s: %s", what, hipGetErrorString(e));
    std::vector<const void *> kernels;
    CRISPY_TRY(graph_kernels(ctx, graph, what, &kernels));
    if (g.exec && g.launch > ctx->settled) CRISPY_TRY(wait_main(ctx));
    if (g.exec && kernels == g.kernels) {
      hipGraphNode_t bad = nullptr;
      hipGraphExecUpdateResult ur = hipGraphExecUpdateError;
      if (hipGraphExecUpdate(g.exec, graph, &bad, &ur) != hipSuccess || ur != hipGraphExecUpdateSuccess) {
        (void)hipGetLastError();
        drop_segment(g);
      }
    } else {
      drop_segment(g);
    }
    if (!g.exec) {
      const hipError_t ie = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
      if (ie != hipSuccess) {
        g.exec = nullptr;
        return set_err(ctx, CRISPY_ERR_HIP, "instantiating the %s graph: %s", what, hipGetErrorString(ie));
      }
    }
    g.kernels = std::move(kernels);
    g.key = std::move(key);
  }
  CRISPY_HIP(ctx, hipGraphLaunch(g.exec, ctx->stream));
  g.launch = ++ctx->launches;
  return CRISPY_OK;
}

}  // namespace crispy
