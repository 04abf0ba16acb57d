#include "fake_hip.h"

#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>

#include "mlp_gpu.h"
#include "mlp_internal.h"
#include "mlp_launch.h"

Counts counts;
std::function<int(int)> rounds_of_slot = [](int) { return 1 << 20; };
int fail_sync = 0;
static const SlotDev* last_table = nullptr;
bool left_out(int slot) {
  const int64_t* info = last_table[slot].info;
  return info[MLP_INFO_PARTIAL] > 0 && info[MLP_INFO_PARTIAL] == info[MLP_INFO_ROUNDS] + (info[MLP_INFO_ACTIVE] ? 1 : 0);
}

namespace {

using Node = std::function<void()>;
struct Stream {
  std::vector<Node>* capture = nullptr;
};
Stream* of(hipStream_t s) { return reinterpret_cast<Stream*>(s); }

void submit(hipStream_t s, Node f) {
  if (of(s)->capture) of(s)->capture->push_back(f);
  else f();
}
// an evaluation: counted when it runs
void submit_eval(hipStream_t s, int Counts::*what, Node f) {
  if (!of(s)->capture) ++counts.eager;
  submit(s, [=] {
    ++(counts.*what);
    f();
  });
}

template <typename T>
std::vector<T> listed(const T* inl, const T* dev, int count) {
  const T* p = dev ? dev : inl;
  return std::vector<T>(p, p + count);
}

}  // namespace

// --- runtime -----------------------------------------------------------------
extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  p->totalGlobalMem = (size_t)64 << 30;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 160 * 1024, hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = *t = (size_t)64 << 30, hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* sym) { return *p = const_cast<void*>(sym), hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "(fake)"; }
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipFree(void* p) { return free(p), hipSuccess; }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  return submit(st, [=] { memcpy(d, s, n); }), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
  return submit(st, [=] { memset(d, v, n); }), hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t* s) { return *s = reinterpret_cast<hipStream_t>(new Stream), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return delete of(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  return fail_sync && --fail_sync == 0 ? hipErrorUnknown : hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }

hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(new int(0)), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<int*>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1, hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  return of(s)->capture = new std::vector<Node>, hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(of(s)->capture);
  return of(s)->capture = nullptr, hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  ++counts.instantiated;
  *e = reinterpret_cast<hipGraphExec_t>(new std::vector<Node>(*reinterpret_cast<std::vector<Node>*>(g)));
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  ++counts.replayed;
  for (const Node& f : *reinterpret_cast<std::vector<Node>*>(e)) f();
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete reinterpret_cast<std::vector<Node>*>(g), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  return delete reinterpret_cast<std::vector<Node>*>(e), hipSuccess;
}
}  // extern "C"

// --- kernels -----------------------------------------------------------------
hipError_t mlp_launch_slot_init(hipStream_t st, SlotDev* table, int id, const SlotDev& d, int64_t* mem,
                                int64_t words, const SlotInitRows&) {
  submit(st, [=] {
    memset(mem, 0, 8 * (size_t)words);
    table[id] = d;
  });
  return hipSuccess;
}
hipError_t mlp_launch_dvnd_start(hipStream_t st, const SlotDev* table, const SlotListInline& inl,
                                 const int32_t* dev, int count) {
  last_table = table;
  submit(st, [=] {
    for (int32_t id : listed(inl.id, dev, count)) {
      table[id].info[MLP_INFO_ACTIVE] = 1;
      table[id].info[MLP_INFO_ROUNDS] = table[id].info[MLP_INFO_PARTIAL] = 0;
    }
  });
  return hipSuccess;
}
hipError_t mlp_launch_sweep(hipStream_t st, int tile, const SlotDev* table, const SweepSegsInline& inl,
                            const SweepSeg* dev, int nsegs, int, int*, int, int) {
  const bool fill = (tile & MLP_TILE_FILL) != 0;
  submit_eval(st, fill ? &Counts::fills : &Counts::evals, [=] {
    for (const SweepSeg& g : listed(inl.s, dev, nsegs)) {
      int64_t* info = table[g.slot].info;
      if (fill ? info[MLP_INFO_PARTIAL] == info[MLP_INFO_ROUNDS] : info[MLP_INFO_ACTIVE])
        counts.worked += __builtin_popcount(g.mask);
      if (fill) info[MLP_INFO_PARTIAL] = 0;  // (the device's word stays: nothing reads it again)
    }
  });
  return hipSuccess;
}
hipError_t mlp_launch_psweep(hipStream_t st, const SlotDev* table, const SweepSegsInline& inl,
                             const SweepSeg* dev, int nsegs, int, int, int) {
  submit_eval(st, &Counts::pruned, [=] {
    for (const SweepSeg& g : listed(inl.s, dev, nsegs))
      if (table[g.slot].info[MLP_INFO_ACTIVE]) {
        table[g.slot].info[MLP_INFO_PARTIAL] = table[g.slot].info[MLP_INFO_ROUNDS] + 1;
        ++counts.worked;
      }
  });
  return hipSuccess;
}
namespace {
void merge(const SlotDev* table, const std::vector<int32_t>& ids, int tail) {
  if (!tail) return;
  for (int32_t id : ids) {
    int64_t* info = table[id].info;
    if (!info[MLP_INFO_ACTIVE]) continue;
    const int64_t r = ++info[MLP_INFO_ROUNDS];
    if (r >= rounds_of_slot(table[id].N) || (tail > 1 && r >= tail - 1)) info[MLP_INFO_ACTIVE] = 0;
  }
}
}  // namespace
hipError_t mlp_launch_merge_apply(hipStream_t st, const SlotDev* table, const SlotListInline& inl,
                                  const int32_t* dev, int count, int, int, int, int, int flags, int tail) {
  ++(flags & MLP_MERGE_WIDE ? counts.wide : counts.narrow);
  submit(st, [=] { merge(table, listed(inl.id, dev, count), tail); });
  return hipSuccess;
}
hipError_t mlp_launch_merge_gmem(hipStream_t st, const SlotDev* table, const SlotListInline& inl,
                                 const int32_t* dev, int count, int, int, int, int tail, int) {
  submit(st, [=] { merge(table, listed(inl.id, dev, count), tail); });
  return hipSuccess;
}
hipError_t mlp_launch_gather_info(hipStream_t st, const SlotDev* table, const int32_t* ids, int count,
                                  int word, int64_t* out) {
  submit(st, [=] {
    for (int q = 0; q < count; ++q) out[q] = table[ids[q]].info[word];
  });
  return hipSuccess;
}

int mlp_prune_rows() { return 32; }
int mlp_prune_max_w(int nb) { return nb >= 2 ? 512 : 1024; }
void mlp_tile_shape(int, int* r, int* c) { *r = 8, *c = 512; }
size_t mlp_merge_lds_bytes(int pcap, int ncap) { return 10 * (size_t)pcap + 13 * (size_t)ncap; }
size_t mlp_fused_lds_bytes(int pcap, int ncap) { return mlp_merge_lds_bytes(pcap, ncap); }
size_t mlp_total_merge_lds_bytes(int N) { return 9 * (size_t)N; }
size_t mlp_total_static_lds() { return 48 * 1024; }
size_t mlp_fused_static_lds() { return 6500; }
hipError_t mlp_launch_fused(hipStream_t st, const SlotDev* table, const FusedPlan& plan, int grid) {
  counts.fused_grid = grid;
  counts.fused_lds = mlp_fused_lds_bytes(plan.pcap, plan.ncap) + mlp_fused_static_lds();
  const std::vector<int32_t> ids(plan.slots, plan.slots + plan.count);
  const int tail = plan.tail;
  submit(st, [=] { merge(table, ids, tail); });
  return hipSuccess;
}
hipError_t mlp_merge_setup(size_t) { return hipSuccess; }
hipError_t mlp_fused_setup(size_t) { return hipSuccess; }
hipError_t mlp_total_setup(size_t) { return hipSuccess; }

// launches that no check looks at
#define NOTHING(name, ...) \
  hipError_t name(__VA_ARGS__) { return hipSuccess; }
NOTHING(mlp_launch_prep, hipStream_t, const SlotDev*, const SlotListInline&, const int32_t*, int, int)
NOTHING(mlp_launch_static_begin, hipStream_t, SlotDev*, const SlotDev&)
NOTHING(mlp_launch_round_begin, hipStream_t, const SlotDev*, const SlotListInline&, const int32_t*, int, int*, int)
NOTHING(mlp_launch_round_end, hipStream_t, const SlotDev*, const SlotListInline&, const int32_t*, int, int)
NOTHING(mlp_launch_eval, hipStream_t, const SlotDev*, const EvalSegsInline&, const EvalSeg*, int, int, int, int*,
        int, int)
NOTHING(mlp_launch_total_eval, hipStream_t, const SlotDev*, int, int, int, int, int64_t*)
NOTHING(mlp_launch_total_keys, hipStream_t, const int64_t*, int64_t, int, uint64_t, uint64_t*, int32_t*)
NOTHING(mlp_launch_total_merge, hipStream_t, const SlotDev*, int, int, int, int, int64_t, uint64_t, const uint64_t*,
        const int32_t*, int)
NOTHING(mlp_sort_pairs_u64, void*, size_t*, const uint64_t*, uint64_t*, const int32_t*, int32_t*, int, int,
        hipStream_t)
NOTHING(mlp_launch_ads, hipStream_t, const SlotDev*, int, int, uint32_t*, uint32_t*)
NOTHING(mlp_launch_rows_moves64, hipStream_t, const SlotDev*, int, int, int, int, uint64_t*)
NOTHING(mlp_launch_rows_out, hipStream_t, const RowsOut&, int, int, int, int, int64_t*, int32_t*, int32_t*)
NOTHING(mlp_launch_total_moves64, hipStream_t, const int64_t*, int64_t, int, int, int, uint64_t*)
NOTHING(mlp_launch_dist_table, hipStream_t, int, int, int, int32_t*)
NOTHING(mlp_launch_dist_list, hipStream_t, const int32_t*, int, int, int32_t*)
NOTHING(mlp_launch_sqrt_selfcheck, hipStream_t, uint32_t, uint32_t, unsigned long long*)
NOTHING(mlp_launch_weights, hipStream_t, const int32_t*, const int32_t*, int, int, int32_t*)
NOTHING(mlp_launch_clear_rows, hipStream_t, const SlotDev*, const SweepSegsInline&, const SweepSeg*, int)
NOTHING(mlp_launch_probe, hipStream_t, const SlotDev*, int, int, int, int64_t*)
NOTHING(mlp_launch_fill_i64, hipStream_t, int64_t*, int64_t, int64_t)
NOTHING(mlp_launch_set_slot, hipStream_t, SlotDev*, int, const SlotDev&)
NOTHING(mlp_launch_gather_tours, hipStream_t, const SlotDev*, const int32_t*, int, int32_t*)
NOTHING(mlp_launch_scatter_tours, hipStream_t, const SlotDev*, const int32_t*, int, const int32_t*)
