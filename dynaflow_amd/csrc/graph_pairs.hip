// Pairs the launches of two nano-batches in a captured schedule (host code).
//
// A schedule that gives every nano-batch a stream of its own launches each projection once per nano-batch, side by side.
// With few rows a launch is the time its weights take to arrive, and both launches fetch all of them: what reaches the XCDs
// from memory and the memory-side cache stays at 6 - 7 TB/s however many ask, while what two workgroups of one XCD read
// together comes at 10 - 12 TB/s.  But the two launches start some 10 us apart, the second one on other XCDs (a queue deals its
// workgroups on from where it stopped), and whoever is behind never catches up.  So they become one launch, whose workgroups
// multiply a weight with the rows of both (up to 32 rows each that stream their weights, up to 64 on tiles), or in which the
// two workgroups that read the same weights sit on the same XCD and start together (pair_block).
// [us, in a graph: 128 MB read by two launches 39 - 43, by one launch twice 24; layer of 2 x 48 tokens 126 / 90, of 2 x 12 in
// fp8 254 / 170]
//
// Where every launch of a graph is one of a pair or short, nothing is left that gains from running side by side: the graph
// becomes a chain, which saves the meetings of two queues (6 - 10 us each).  Any other graph stays as it is: also one with a
// GEMM that has no launch of two, however few its workgroups are; of kernels that are not of this library, those of up to 512
// workgroups count as short, and the caller vouches for what they are.  Short launches and
// attention over a cache pair as well (their workgroups side by side: one launch's gap less, and of attention one tail).
// A schedule with a stream per nano-batch (`side_by_side`) runs long attention of one beside the projections of the other, which
// is worth as much from 512 workgroups on: it stays.  [us of a decode step of 4 layers, sequences of 1/4 .. 1 of 4096 positions,
// streams by nano-batch / by kind / chain: 40 sequences 1036 / 1179 / 824, 64 1230 / 1410 / 1058, 128 1644 / 2030 /
// 1622 (by kind's plans 1688); 256 of 2048 positions each 2117 / 2533 / 2145 (2333)]
#include <algorithm>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "dfhip_pairs.h"

namespace {

struct Known {
  DfhipJoin join = nullptr;
  unsigned in_line = DFHIP_SHORT_BLOCKS;
};
std::mutex known_mutex;
std::unordered_map<const void*, Known>& known_kernels() {
  static std::unordered_map<const void*, Known> kernels;
  return kernels;
}
Known find_known(const void* kernel) {
  std::lock_guard<std::mutex> guard(known_mutex);
  const auto it = known_kernels().find(kernel);
  return it == known_kernels().end() ? Known{} : it->second;
}

struct Node {
  hipGraphNode_t handle;
  bool kernel;
  hipKernelNodeParams params;
  Known known;
  int pair = -1;                         // the other node of its pair
};

// (the parts of a sequence that attention cuts, grid.y, count as one)
size_t blocks_of(const Node& node) {
  const dim3& grid = node.params.gridDim;
  return node.known.join ? grid.x : (size_t)grid.x * grid.y * grid.z;
}

// A topological order of the graph whose paired nodes are one (named by the smaller index), smallest index first; empty if
// there is none.
std::vector<int> order_of(const std::vector<Node>& nodes, const std::vector<std::pair<int, int>>& edges) {
  const int n = (int)nodes.size();
  auto name = [&](int i) { return nodes[i].pair >= 0 && nodes[i].pair < i ? nodes[i].pair : i; };
  std::vector<std::vector<int>> next(n);
  std::vector<int> waits(n, 0), order;
  for (const auto& e : edges) {
    const int a = name(e.first), b = name(e.second);
    if (a == b) return {};
    next[a].push_back(b);
    ++waits[b];
  }
  std::vector<bool> done(n, false);
  for (;;) {
    int at = -1;
    for (int i = 0; i < n && at < 0; ++i)
      if (name(i) == i && !done[i] && waits[i] == 0) at = i;
    if (at < 0) break;
    done[at] = true;
    order.push_back(at);
    for (int b : next[at]) --waits[b];
  }
  for (int i = 0; i < n; ++i)
    if (name(i) == i && !done[i]) return {};
  return order;
}

}  // namespace

void dfhip_pairable(const void* kernel, DfhipJoin join, unsigned in_line) {
  std::lock_guard<std::mutex> guard(known_mutex);
  known_kernels()[kernel] = {join, in_line};
}

extern "C" int dfhip_graph_pair_launches(void* graph, int side_by_side, int* pairs) {
  if (!graph || !pairs) return DFHIP_ERR_NULL_POINTER;
  *pairs = 0;
  hipGraph_t g = static_cast<hipGraph_t>(graph);
  size_t count = 0, edge_count = 0;
  if (hipGraphGetNodes(g, nullptr, &count) != hipSuccess || hipGraphGetEdges(g, nullptr, nullptr, &edge_count) != hipSuccess)
    return DFHIP_ERR_LAUNCH;
  if (count < 2 || count > 2048) return DFHIP_OK;
  std::vector<hipGraphNode_t> handles(count), from(edge_count), to(edge_count);
  if (hipGraphGetNodes(g, handles.data(), &count) != hipSuccess) return DFHIP_ERR_LAUNCH;
  if (edge_count && hipGraphGetEdges(g, from.data(), to.data(), &edge_count) != hipSuccess) return DFHIP_ERR_LAUNCH;

  std::unordered_map<hipGraphNode_t, int> index;
  std::vector<Node> nodes(count);
  for (size_t i = 0; i < count; ++i) {
    Node& node = nodes[i];
    node.handle = handles[i];
    index[handles[i]] = (int)i;
    hipGraphNodeType type;
    if (hipGraphNodeGetType(handles[i], &type) != hipSuccess) return DFHIP_ERR_LAUNCH;
    node.kernel = type == hipGraphNodeTypeKernel;
    if (type == hipGraphNodeTypeEmpty) continue;
    if (!node.kernel) return DFHIP_OK;
    if (hipGraphKernelNodeGetParams(handles[i], &node.params) != hipSuccess) return DFHIP_ERR_LAUNCH;
    node.known = find_known(node.params.func);
    if (node.known.join && !node.params.kernelParams) node.known.join = nullptr;
    if (!node.known.join && blocks_of(node) > node.known.in_line) return DFHIP_OK;
  }
  std::vector<std::pair<int, int>> edges(edge_count);
  const size_t words = (count + 63) / 64;
  std::vector<uint64_t> paths(count * words, 0);                     // bit j of row i: a path from node i to node j
  auto reaches = [&](size_t i, size_t j) { return (paths[i * words + j / 64] >> (j % 64)) & 1; };
  for (size_t e = 0; e < edge_count; ++e) {
    edges[e] = {index[from[e]], index[to[e]]};
    paths[edges[e].first * words + edges[e].second / 64] |= (uint64_t)1 << (edges[e].second % 64);
  }
  for (size_t k = 0; k < count; ++k)
    for (size_t i = 0; i < count; ++i)
      if (reaches(i, k))
        for (size_t w = 0; w < words; ++w) paths[i * words + w] |= paths[k * words + w];

  alignas(16) unsigned char both[DFHIP_PAIR_MAX_ARGS];
  DfhipJoined joined;
  auto join_of = [&](const Node& a, const Node& b) {
    joined.lds = a.params.sharedMemBytes;
    return a.known.join(a.params.kernelParams[0], b.params.kernelParams[0], a.params.gridDim, b.params.gridDim, both, &joined);
  };
  int found = 0;
  for (size_t i = 0; i < count; ++i) {
    Node& a = nodes[i];
    if (!a.kernel || !a.known.join || a.pair >= 0) continue;
    for (size_t j = i + 1; j < count && a.pair < 0; ++j) {
      Node& b = nodes[j];
      if (!b.kernel || b.pair >= 0 || b.params.func != a.params.func || reaches(i, j) || reaches(j, i)) continue;
      if (!dfhip_same(a.params.blockDim, b.params.blockDim) || a.params.sharedMemBytes != b.params.sharedMemBytes) continue;
      if (!join_of(a, b)) continue;
      a.pair = (int)j;
      b.pair = (int)i;
      found += a.known.in_line == 0;
    }
  }
  // launches that would lose their company
  for (const Node& node : nodes)
    if (node.kernel && blocks_of(node) > node.known.in_line && (node.pair < 0 || (side_by_side && node.known.in_line > 0)))
      return DFHIP_OK;
  if (!found) return DFHIP_OK;
  const std::vector<int> order = order_of(nodes, edges);
  if (order.empty()) return DFHIP_OK;                                 // two pairs that wait for each other crosswise

  // from here on the graph changes; a failure leaves it useless, and the caller with an error
  if (edge_count && hipGraphRemoveDependencies(g, from.data(), to.data(), edge_count) != hipSuccess) return DFHIP_ERR_LAUNCH;
  hipGraphNode_t last = nullptr;
  for (int i : order) {
    Node& node = nodes[i];
    if (!node.kernel) {
      if (hipGraphDestroyNode(node.handle) != hipSuccess) return DFHIP_ERR_LAUNCH;
      continue;
    }
    if (node.pair >= 0) {
      Node& other = nodes[node.pair];
      if (!join_of(node, other)) return DFHIP_ERR_LAUNCH;
      hipKernelNodeParams params = node.params;
      void* args[1] = {both};
      params.kernelParams = args;
      params.func = const_cast<void*>(joined.kernel);
      params.gridDim = joined.grid;
      params.sharedMemBytes = joined.lds;
      if (hipGraphKernelNodeSetParams(node.handle, &params) != hipSuccess) return DFHIP_ERR_LAUNCH;
      if (hipGraphDestroyNode(other.handle) != hipSuccess) return DFHIP_ERR_LAUNCH;
    }
    if (last && hipGraphAddDependencies(g, &last, &node.handle, 1) != hipSuccess) return DFHIP_ERR_LAUNCH;
    last = node.handle;
  }
  *pairs = found;
  return DFHIP_OK;
}
