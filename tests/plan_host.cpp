// Retained plans (plan.cpp) on a host without a GPU: the HIP calls and the launches are stand-ins that note what is asked of
// them.  A record named "layers" is a resident run; its parameters are the workgroups and the layers.
#include "plan.cpp"

#include <unistd.h>

namespace {
struct Graph {
  bool resident = false;
  uint32_t workgroups = 0;
  const StepWords *step = nullptr;
};
struct Launch {
  bool resident;
  uint32_t tag;
};
std::mutex lock;
std::vector<Launch> launches;
Graph *capturing = nullptr;  // (plans are made one by one)
uint32_t layer_workgroups = 0, resident_layers = 4;
bool refuse_resident_graph = false, gives_up = false;
int cleared = 0, live_graphs = 0;
uint32_t under_way = 0, most_under_way = 0;  // workgroups of resident launches
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return ++cleared, hipSuccess; }
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind) { return memcpy(to, from, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(to, from, n), hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *) { return hipErrorUnknown; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipErrorUnknown; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipErrorUnknown; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipErrorUnknown; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return capturing = new Graph, ++live_graphs, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *graph) { return *graph = reinterpret_cast<hipGraph_t>(capturing), hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t graph) { return delete reinterpret_cast<Graph *>(graph), --live_graphs, hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t executable) { return delete reinterpret_cast<Graph *>(executable), --live_graphs, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *out, hipGraph_t graph, hipGraphNode_t *, char *, size_t) {
  const Graph &of = *reinterpret_cast<Graph *>(graph);
  if (of.resident && refuse_resident_graph) return hipErrorUnknown;
  *out = reinterpret_cast<hipGraphExec_t>(new Graph(of));
  return ++live_graphs, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t executable, hipStream_t) {
  const Graph &of = *reinterpret_cast<Graph *>(executable);
  StepWords *step = const_cast<StepWords *>(of.step);
  {
    std::lock_guard<std::mutex> hold(lock);
    launches.push_back({of.resident, step->resident_tag});
    most_under_way = std::max(most_under_way, under_way += of.workgroups);
  }
  if (of.resident) usleep(500);
  step->result[0] = (int32_t)step->value + 1;
  step->result[1] = of.resident && gives_up;
  std::lock_guard<std::mutex> hold(lock);
  under_way -= of.workgroups;
  return hipSuccess;
}
}  // extern "C"

namespace llmopt {
int fail(int status, const char *, ...) { return status; }
int fail_hip(hipError_t, const char *) { return LLMOPT_ERR_FAILURE; }
void retain(RefCounted *) {}
bool release(RefCounted *) { return true; }
int use_device(llmopt_hip_context *) { return LLMOPT_OK; }
uint32_t param_u32(const DispatchRecord &, size_t) { return 0; }
uint32_t *context_counters(llmopt_hip_context *, uint32_t *count) {
  static uint32_t counter;
  return *count = 1, &counter;
}
void *context_workspace(llmopt_hip_context *, size_t) { return nullptr; }
int build_record(llmopt_hip_library *, const llmopt_hip_dispatch_item *item, DispatchRecord *out) { return out->name = item->name, LLMOPT_OK; }
int launch_record(llmopt_hip_context *, const DispatchRecord &) { return LLMOPT_OK; }
void drop_record(DispatchRecord *) {}
hipError_t launch_nan_scan(const void *, size_t, bool, uint32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_plan_begin(const StepWords *step, hipStream_t) { return capturing->step = step, hipSuccess; }
hipError_t launch_plan_result(const int32_t *, const uint32_t *, int32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_plan_state(int64_t *, int64_t, const int32_t *, uint32_t *, uint32_t, uint32_t, uint32_t *, uint32_t, hipStream_t) { return hipSuccess; }
bool find_resident_run(const std::vector<DispatchRecord> &records, ResidentRun *out) {
  out->count = 1;
  out->layers.resize(resident_layers);
  out->args.layer_count = resident_layers;
  return records[0].name == "layers";
}
uint32_t resident_workgroups(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) { return layer_workgroups; }
ResidentWords resident_words(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) {
  ResidentWords words = {};
  words.total = 16;
  return words;
}
uint32_t resident_lds(ResidentArgs &, uint32_t) { return 0; }
bool resident_fits(const ResidentArgs &, uint32_t, uint32_t) { return true; }
hipError_t launch_decode_resident(const ResidentArgs &, uint32_t workgroups, uint32_t, hipStream_t) {
  capturing->resident = true;
  return capturing->workgroups = workgroups, hipSuccess;
}
}  // namespace llmopt

extern "C" {
void llmopt_hip_release_buffer(llmopt_hip_buffer *) {}
void llmopt_hip_release_library(llmopt_hip_library *) {}

void stub_set(uint32_t workgroups, uint32_t layers, int refuse, int give_up) {
  layer_workgroups = workgroups, resident_layers = layers, refuse_resident_graph = refuse != 0, gives_up = give_up != 0;
  launches.clear();
  cleared = 0;
  most_under_way = 0;
}
void *stub_plan(const char *name) {
  llmopt_hip_library *library = new llmopt_hip_library;
  library->context = new llmopt_hip_context;
  llmopt_hip_dispatch_item item = {};
  item.name = name;
  llmopt_hip_prebaked *plan = nullptr;
  return llmopt_hip_prebaked_create(library, &item, 1, nullptr, nullptr, &plan) == LLMOPT_OK ? plan : nullptr;
}
long stub_step(void *plan, long token) {
  int64_t out = -1;
  return llmopt_hip_prebaked_execute(static_cast<llmopt_hip_prebaked *>(plan), token, 0, 0, &out) == LLMOPT_OK ? (long)out : -1;
}
void stub_recapture(void *plan) { ++static_cast<llmopt_hip_prebaked *>(plan)->library->context->workspace_generation; }
void stub_next_tag(void *plan, uint32_t tag) { static_cast<llmopt_hip_prebaked *>(plan)->resident->next_tag = tag; }
long stub_launches(uint32_t *tags, long most) {  // of each launch the step's tag, 0 of one without resident layers
  for (long i = 0; i < most && i < (long)launches.size(); ++i) tags[i] = launches[i].resident ? launches[i].tag : 0;
  return (long)launches.size();
}
int stub_cleared() { return cleared; }
uint32_t stub_most_under_way() { return most_under_way; }
int stub_live_graphs() { return live_graphs; }
}
