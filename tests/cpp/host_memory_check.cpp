// Which device memory the library's launches name, checked without a GPU: this
// program defines the HIP runtime calls that libfc_dem.so makes (a program's
// own definitions come before those of the libraries it loads), so that
// "device memory" is a number that is never read, an allocation can be made to
// fail, and every launch and every replay of a captured graph is checked to
// name no freed memory.
//
//   host_memory_check SCENARIO   exits 0 when the scenario holds
#include <hip/hip_runtime.h>

#include <cxxabi.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "fc_dem.h"
#include "fc_internal.hpp"
#include "row_resort.hpp"

// ---------------------------------------------------------------------------
// The stand-in runtime.
// ---------------------------------------------------------------------------
namespace {

constexpr uintptr_t kFirst = 0x500000000000ull;  // no mapping of this process lies there
struct Block {
  size_t size;
  bool live;
};
struct Node {
  std::string kernel;
  std::vector<uintptr_t> pointers;
};
struct Graph {
  std::vector<Node> nodes;
};
struct Runtime {
  std::map<uintptr_t, Block> blocks;  // addresses are never given out twice
  uintptr_t next = kFirst;
  size_t inUse = 0, most = ~(size_t)0;     // hipMalloc fails beyond `most` bytes in use
  size_t failing = 0;                      // nor for this size exactly
  hipError_t last = hipSuccess;
  hipError_t memsetError = hipSuccess;     // what the next clear returns
  int unordered = 0;                       // clears on the null stream
  std::map<const void*, std::string> names;
  Graph* capturing = nullptr;
  struct { dim3 grid, block; size_t shared; hipStream_t stream; } config;
  std::vector<std::string> launched;       // kernels run since the last clear
  int captures = 0;
  std::string fault;
};
Runtime& rt() {
  static Runtime r;
  return r;
}

hipError_t result(hipError_t e) {
  if (e != hipSuccess) rt().last = e;
  return e;
}

void check_node(const Node& n) {
  for (uintptr_t p : n.pointers) {
    auto it = rt().blocks.upper_bound(p);
    const bool inside =
        it != rt().blocks.begin() && p < std::prev(it)->first + std::prev(it)->second.size;
    if (rt().fault.empty() && (!inside || !std::prev(it)->second.live))
      rt().fault = n.kernel + " names freed memory";
  }
}

// The types of a kernel's parameters, from its demangled name.
std::vector<std::string> parameters(const std::string& name) {
  std::vector<std::string> out;
  if (name.empty() || name.back() != ')') return out;
  size_t open = name.size() - 1;
  for (int depth = 0; open > 0; --open) {
    depth += name[open] == ')' ? 1 : (name[open] == '(' ? -1 : 0);
    if (depth == 0) break;
  }
  std::string cur;
  int depth = 0;
  for (size_t i = open + 1; i + 1 < name.size(); ++i) {
    const char c = name[i];
    depth += (c == '<' || c == '(') ? 1 : ((c == '>' || c == ')') ? -1 : 0);
    if (c == ',' && depth == 0) {
      out.push_back(cur);
      cur.clear();
    } else if (!(c == ' ' && cur.empty())) {
      cur += c;
    }
  }
  if (!cur.empty()) out.push_back(cur);
  return out;
}

Node node_of(const std::string& name, void** args) {
  Node n;
  n.kernel = name.substr(0, name.find('('));
  const size_t at = name.find("::k_");
  if (at != std::string::npos) n.kernel = name.substr(at + 2, name.find_first_of("<(", at) - at - 2);
  const std::vector<std::string> types = parameters(name);
  const std::map<std::string, size_t> structs = {{"fc::RowTables", sizeof(fc::RowTables)},
                                                 {"fc::RowHists", sizeof(fc::RowHists)},
                                                 {"fc::RowOutputs", sizeof(fc::RowOutputs)},
                                                 {"fc::SortGather", sizeof(fc::SortGather)}};
  for (size_t i = 0; i < types.size(); ++i) {
    const bool pointer = types[i].find('*') != std::string::npos;
    const auto s = structs.find(types[i]);
    const size_t words = pointer ? 1 : (s != structs.end() ? s->second / sizeof(uintptr_t) : 0);
    for (size_t w = 0; w < words; ++w) {
      uintptr_t p;
      std::memcpy(&p, static_cast<char*>(args[i]) + w * sizeof(p), sizeof(p));
      if (p >= kFirst && p < rt().next) n.pointers.push_back(p);
      // the rank sort's staging arrays are always there
      if (pointer && p == 0 && n.kernel == "k_small_rank" && i >= 6)
        rt().fault = "k_small_rank without its scratch";
      if (pointer && p == 0 && n.kernel.rfind("k_collide_", 0) == 0 && (i == 7 || i == 8))
        rt().fault = n.kernel + " without cell tables";
    }
  }
  return n;
}

bool launched(const char* kernel) {
  for (const std::string& k : rt().launched)
    if (k == kernel) return true;
  return false;
}

}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  int status = 0;
  char* d = abi::__cxa_demangle(name, nullptr, nullptr, &status);
  rt().names[host] = d ? d : name;
  std::free(d);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  rt().config = {grid, block, shared, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = rt().config.grid;
  *block = rt().config.block;
  *shared = rt().config.shared;
  *stream = rt().config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
  const Node n = node_of(rt().names[f], args);
  if (rt().capturing) {
    rt().capturing->nodes.push_back(n);
  } else {
    check_node(n);
    rt().launched.push_back(n.kernel);
  }
  return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void*, dim3, dim3, void**, unsigned, hipStream_t) {
  return result(hipErrorNotSupported);
}
hipError_t hipMalloc(void** p, size_t size) {
  *p = nullptr;
  if ((size == rt().failing && size) || size > rt().most || rt().inUse > rt().most - size) return result(hipErrorOutOfMemory);
  const uintptr_t at = rt().next;
  rt().next += (size + 4096 + 255) & ~(size_t)255;
  rt().blocks[at] = Block{size, true};
  rt().inUse += size;
  *p = reinterpret_cast<void*>(at);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  auto it = rt().blocks.find(reinterpret_cast<uintptr_t>(p));
  if (it == rt().blocks.end() || !it->second.live) {
    rt().fault = "hipFree of what is not allocated";
    return result(hipErrorInvalidValue);
  }
  it->second.live = false;
  rt().inUse -= it->second.size;
  return hipSuccess;
}
hipError_t hipMemset(void*, int, size_t) {
  ++rt().unordered;
  const hipError_t e = rt().memsetError;
  rt().memsetError = hipSuccess;
  return result(e);
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) {
  if (rt().capturing) rt().fault = "hipMemsetAsync inside a capture";
  const hipError_t e = rt().memsetError;
  rt().memsetError = hipSuccess;
  return result(e);
}
hipError_t hipMemcpyAsync(void* dst, const void*, size_t size, hipMemcpyKind kind, hipStream_t) {
  if (kind == hipMemcpyDeviceToHost) std::memset(dst, 0, size);
  return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t size, hipMemcpyKind kind) {
  return hipMemcpyAsync(dst, src, size, kind, nullptr);
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  *s = rt().capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  rt().capturing = new Graph;
  ++rt().captures;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(rt().capturing);
  rt().capturing = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph*>(g)));
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete reinterpret_cast<Graph*>(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  delete reinterpret_cast<Graph*>(e);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  for (const Node& n : reinterpret_cast<Graph*>(e)->nodes) {
    check_node(n);
    rt().launched.push_back(n.kernel);
  }
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(8);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 0;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 0;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return hipMalloc(p, 64u << 20); }
hipError_t hipGetLastError(void) {
  const hipError_t e = rt().last;
  rt().last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : "error";
}
}  // extern "C"

// ---------------------------------------------------------------------------
// Scenarios.
// ---------------------------------------------------------------------------
namespace {

#define REQUIRE(cond)                                                          \
  do {                                                                         \
    const bool held = (cond);                                                  \
    if (!held || !rt().fault.empty()) {                                        \
      std::printf("line %d: %s [%s] %s\n", __LINE__, #cond, rt().fault.c_str(), \
                  fc_last_error());                                            \
      return 1;                                                                \
    }                                                                          \
  } while (0)
#define OK(call) REQUIRE((call) == FC_SUCCESS)

fc_context* context() {
  fc_context* c = nullptr;
  if (fc_context_create(0, &c) != FC_SUCCESS) std::abort();
  return c;
}

template <typename T>
T* device(size_t count) {
  void* p = nullptr;
  if (fc_allocate_array(&p, count * sizeof(T)) != FC_SUCCESS) std::abort();
  return static_cast<T*>(p);
}

// Calls that need more sort scratch than any system below has spheres.
constexpr uint32_t kLabels = 65536, kMapTriangles = 8192, kSystem = 100000, kSort = 200000;

fc_status labels(fc_context* c) {
  const uint32_t nv = 3072, nt = 6144, np = kLabels;
  return fc_mesh_signed_distance(c, device<double>(3 * nv), nv, device<uint32_t>(3 * nt), nt,
                                 device<double>(3 * np), np, device<double>(np), nullptr);
}
fc_status build_map(fc_context* c) {
  const uint32_t nv = 4096, nt = kMapTriangles;
  std::vector<double> v(3 * nv, 0.5);
  std::vector<uint32_t> f(3 * nt);
  for (uint32_t i = 0; i < 3 * nt; ++i) f[i] = i % nv;
  const int32_t cells[3] = {8, 8, 8};
  const float lo[3] = {-1.0f, -1.0f, -1.0f};
  fc_distmap* m = nullptr;
  const fc_status s = fc_distmap_build(c, v.data(), nv, f.data(), nt, cells, 0.25f, lo, &m);
  fc_distmap_destroy(m);
  return s;
}
fc_status larger_system(fc_context* c) {
  fc_system* s = nullptr;
  return fc_system_create(c, kSystem, fc_uint3{64, 64, 64}, &s);
}
fc_status larger_sort(fc_context* c) {
  static uint32_t *k = device<uint32_t>(kSort), *v = device<uint32_t>(kSort);
  return fc_sort_particles(c, k, v, kSort);
}
using Growth = fc_status (*)(fc_context*);
const Growth kGrowths[] = {labels, build_map, larger_system, larger_sort};

// A system's runs around each call that may grow the context's scratch.
int system_runs(uint32_t n, fc_uint3 grid, const char* sortKernel) {
  for (Growth grow : kGrowths) {
    fc_context* c = context();
    fc_system* s = nullptr;
    OK(fc_system_create(c, n, grid, &s));
    OK(fc_system_run(s, 0.5f, 20));
    REQUIRE(launched(sortKernel));
    const int captures = rt().captures;
    OK(fc_system_run(s, 0.5f, 20));
    REQUIRE(rt().captures == captures);  // nothing changed: the same graphs
    OK(grow(c));
    OK(fc_system_run(s, 0.5f, 20));
    OK(fc_system_update(s, 0.5f));
    OK(fc_system_destroy(s));
  }
  return 0;
}

int batch_runs(fc_uint3 grid) {
  for (Growth grow : kGrowths) {
    fc_context* c = context();
    const uint32_t counts[3] = {900, 0, 2100};
    fc_batch* b = nullptr;
    OK(fc_batch_create(c, 3, counts, grid, &b));
    OK(fc_batch_run(b, 0.5f, 20));
    const int captures = rt().captures;
    OK(fc_batch_run(b, 0.5f, 20));
    REQUIRE(rt().captures == captures);
    OK(grow(c));
    OK(fc_batch_run(b, 0.5f, 20));
    OK(fc_batch_update(b, 0.5f));
    OK(fc_batch_destroy(b));
  }
  return 0;
}

// Runs of two grid shapes with equally many cells in turn, the second's too
// short to be captured: the first's captured steps hold tables that are gone.
int row_tables(uint32_t n) {
  fc_context* c = context();
  fc_system* s = nullptr;
  OK(fc_system_create(c, n, fc_uint3{64, 64, 64}, &s));
  fc_sim_params a, b;
  OK(fc_system_get_params(s, &a));
  b = a;
  b.gridSize = fc_uint3{128, 32, 64};
  OK(fc_system_run(s, 0.5f, 20));
  REQUIRE(launched("k_row_sort"));
  const int captures = rt().captures;
  OK(fc_system_run(s, 0.5f, 20));
  REQUIRE(rt().captures == captures);
  OK(fc_system_set_params(s, &b));
  OK(fc_system_run(s, 0.5f, 2));
  OK(fc_system_set_params(s, &a));
  OK(fc_system_run(s, 0.5f, 20));
  return 0;
}

// Runs of a system that can do without row tables, while there is no memory
// for them, after a grid change with memory, and with another error.
int no_row_tables() {
  fc_context* c = context();
  fc_system* s = nullptr;
  OK(fc_system_create(c, 8000, fc_uint3{64, 64, 64}, &s));
  rt().most = rt().inUse;
  OK(fc_system_run(s, 0.5f, 20));
  REQUIRE(launched("k_rs_scatter") && !launched("k_row_sort") && !launched("k_row_reset"));
  OK(fc_system_run(s, 0.5f, 20));  // no second attempt at the same grid
  rt().most = ~(size_t)0;
  OK(fc_system_run(s, 0.5f, 20));
  REQUIRE(!launched("k_row_sort"));
  fc_sim_params p;
  OK(fc_system_get_params(s, &p));
  p.spring *= 2.0f;
  OK(fc_system_set_params(s, &p));
  OK(fc_system_run(s, 0.5f, 20));
  REQUIRE(!launched("k_row_sort"));
  p.gridSize = fc_uint3{128, 32, 64};
  OK(fc_system_set_params(s, &p));
  rt().launched.clear();
  OK(fc_system_run(s, 0.5f, 20));
  REQUIRE(launched("k_row_sort"));
  // an error that is not for want of memory is the caller's to see, and the
  // next run has its tables again
  p.gridSize = fc_uint3{32, 64, 128};
  OK(fc_system_set_params(s, &p));
  rt().memsetError = hipErrorLaunchFailure;
  REQUIRE(fc_system_run(s, 0.5f, 20) == FC_ERROR_HIP);
  rt().launched.clear();
  const size_t blocks = rt().blocks.size();
  OK(fc_system_run(s, 0.5f, 20));
  REQUIRE(launched("k_row_sort") && rt().blocks.size() > blocks);  // none that were not cleared
  return 0;
}

// The contexts' streams do not wait for the null stream: what a kernel reads is
// cleared on the stream that launches it.
int clears() {
  fc_context* c = context();
  fc_system* s = nullptr;
  OK(fc_system_create(c, 20000, fc_uint3{64, 64, 64}, &s));
  OK(fc_system_set_polydisperse(s, 1));
  OK(fc_system_run(s, 0.5f, 20));
  REQUIRE(launched("k_collide_piles") && launched("k_row_sort"));
  OK(labels(c));
  REQUIRE(rt().unordered == 0);
  return 0;
}

// The copy of a mesh too large for the tree goes with the call that made it.
int large_meshes() {
  fc_context* c = context();
  OK(build_map(c));
  const size_t before = rt().inUse;
  std::vector<double> v((size_t)3 << 24, 0.5);  // 400 MB
  std::vector<uint32_t> f(3 * kMapTriangles);
  for (uint32_t i = 0; i < f.size(); ++i) f[i] = i;
  const int32_t cells[3] = {8, 8, 8};
  const float lo[3] = {-1.0f, -1.0f, -1.0f};
  for (uint32_t triangles : {12u, kMapTriangles}) {
    fc_distmap* m = nullptr;
    rt().launched.clear();
    OK(fc_distmap_build(c, v.data(), 1u << 24, f.data(), triangles, cells, 0.25f, lo, &m));
    REQUIRE(launched("k_tree_leaves") == (triangles > 12));
    OK(fc_distmap_destroy(m));
    REQUIRE(rt().inUse < before + (64u << 20));
  }
  return 0;
}

// A grid for whose cell tables there is no memory is refused, and the system
// runs on with the one that it has; or says so, if even that one is gone.
int no_cell_tables(uint32_t n) {
  fc_context* c = context();
  fc_system* s = nullptr;
  OK(fc_system_create(c, n, fc_uint3{64, 64, 64}, &s));
  OK(fc_system_run(s, 0.5f, 20));
  fc_sim_params a, b;
  OK(fc_system_get_params(s, &a));
  b = a;
  b.gridSize = fc_uint3{256, 256, 256};
  b.numCells = 1u << 24;
  rt().failing = 4u << 24;
  REQUIRE(fc_system_set_params(s, &b) == FC_ERROR_OUT_OF_MEMORY);
  rt().failing = 0;
  OK(fc_system_update(s, 0.5f));
  OK(fc_system_run(s, 0.5f, 20));
  rt().most = rt().inUse + (4u << 24);  // room in the place of the old tables only
  OK(fc_system_set_params(s, &a));
  b.gridSize = fc_uint3{128, 64, 64};
  b.numCells = 1u << 19;
  rt().most = rt().inUse + (2u << 20);
  OK(fc_system_set_params(s, &b));
  rt().most = ~(size_t)0;
  OK(fc_system_run(s, 0.5f, 20));
  rt().most = 0;
  REQUIRE(fc_system_set_params(s, &a) == FC_ERROR_OUT_OF_MEMORY);
  REQUIRE(fc_system_update(s, 0.5f) == FC_ERROR_OUT_OF_MEMORY);
  REQUIRE(fc_system_run(s, 0.5f, 20) == FC_ERROR_OUT_OF_MEMORY);
  uint32_t most, occupied, hist[8];
  REQUIRE(fc_system_dump_grid(s, &most, &occupied) == FC_ERROR_OUT_OF_MEMORY);
  REQUIRE(fc_system_contact_histogram(s, hist, 8) == FC_ERROR_OUT_OF_MEMORY);
  rt().most = ~(size_t)0;
  OK(fc_system_set_params(s, &a));
  OK(fc_system_run(s, 0.5f, 20));
  return 0;
}

// An error that a call has returned is that call's alone.
int errors_once() {
  fc_context* c = context();
  fc_system *s = nullptr, *other = nullptr;
  OK(fc_system_create(c, 4096, fc_uint3{64, 64, 64}, &s));
  rt().most = 0;
  REQUIRE(fc_system_create(c, 4096, fc_uint3{64, 64, 64}, &other) == FC_ERROR_OUT_OF_MEMORY);
  rt().most = ~(size_t)0;
  OK(fc_system_update(s, 0.5f));
  OK(fc_system_run(s, 0.5f, 20));
  return 0;
}

// A call that finds no memory for its scratch: the mesh calls do without, the
// others say so, and the context's systems and batches run on.
int growth_fails(uint32_t n, fc_uint3 grid) {
  for (Growth grow : kGrowths) {
    fc_context* c = context();
    fc_system* s = nullptr;
    const uint32_t counts[2] = {700, 900};
    (void)larger_sort(context());  // (its arrays)
    fc_batch* b = nullptr;
    OK(fc_system_create(c, n, grid, &s));
    OK(fc_batch_create(c, 2, counts, fc_uint3{64, 64, 2}, &b));
    OK(fc_system_run(s, 0.5f, 20));
    OK(fc_batch_run(b, 0.5f, 20));
    const bool mesh = grow == labels || grow == build_map;
    rt().failing = 4 * (grow == labels ? kLabels
                                       : (grow == build_map ? kMapTriangles
                                                            : (grow == larger_system ? kSystem : kSort)));
    rt().launched.clear();
    REQUIRE(grow(c) == (mesh ? FC_SUCCESS : FC_ERROR_OUT_OF_MEMORY));
    rt().failing = 0;
    REQUIRE(!launched("k_tree_leaves") && launched("k_mesh_sdf") == mesh);
    OK(fc_system_update(s, 0.5f));
    OK(fc_system_run(s, 0.5f, 20));
    OK(fc_batch_update(b, 0.5f));
    OK(fc_batch_run(b, 0.5f, 20));
    OK(grow(c));
    REQUIRE(!mesh || launched("k_tree_leaves"));
    OK(fc_system_run(s, 0.5f, 20));
    OK(fc_batch_run(b, 0.5f, 20));
  }
  return 0;
}

// Room for the larger scratch only in the place of the smaller; and room for
// neither, where the steps return an error.
int no_room_for_both() {
  fc_context* c = context();
  fc_system* s = nullptr;
  OK(fc_system_create(c, 4096, fc_uint3{64, 64, 64}, &s));
  OK(fc_system_run(s, 0.5f, 20));
  const uint32_t n = 8192;
  uint32_t *k = device<uint32_t>(n), *v = device<uint32_t>(n);
  rt().most = rt().inUse + 16 * n;  // (the arrays take 16 n bytes and the look-back words)
  OK(fc_sort_particles(c, k, v, n));
  OK(fc_system_run(s, 0.5f, 20));
  rt().most = 0;
  REQUIRE(fc_sort_particles(c, k, v, n + 1) == FC_ERROR_OUT_OF_MEMORY);
  REQUIRE(fc_system_update(s, 0.5f) == FC_ERROR_HIP);
  REQUIRE(fc_system_run(s, 0.5f, 20) == FC_ERROR_HIP);
  rt().most = ~(size_t)0;
  OK(fc_sort_particles(c, k, v, n));
  OK(fc_system_run(s, 0.5f, 20));
  return 0;
}

int run(const std::string& name) {
  if (name == "row-tables-small") return row_tables(8000);
  if (name == "row-tables") return row_tables(40000);
  if (name == "no-row-tables") return no_row_tables();
  if (name == "clears") return clears();
  if (name == "large-meshes") return large_meshes();
  if (name == "no-cell-tables-small") return no_cell_tables(3000);
  if (name == "no-cell-tables") return no_cell_tables(40000);
  if (name == "errors-once") return errors_once();
  if (name == "growth-fails-small") return growth_fails(4096, fc_uint3{64, 64, 64});
  if (name == "growth-fails-radix") return growth_fails(8000, fc_uint3{4, 1024, 512});
  if (name == "no-room-for-both") return no_room_for_both();
  if (name == "system-small") return system_runs(4096, fc_uint3{64, 64, 64}, "k_small_rank");
  if (name == "system-radix") return system_runs(8000, fc_uint3{4, 1024, 512}, "k_rs_scatter");
  if (name == "batch-cells") return batch_runs(fc_uint3{64, 64, 2});
  if (name == "batch-radix") return batch_runs(fc_uint3{4, 4096, 2048});
  if (name == "batch-rows") return batch_runs(fc_uint3{16, 16, 16});
  std::printf("no scenario %s\n", name.c_str());
  return 2;
}

}  // namespace

int main(int argc, char** argv) {
  const int r = argc == 2 ? run(argv[1]) : 2;
  if (r == 0) std::printf("ok\n");
  std::fflush(stdout);
  std::_Exit(r);  // (the library's handles of the real runtime are not torn down)
}
