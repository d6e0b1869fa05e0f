// Recorded launches (record.h): the list and its entry points.
#include "record.h"

#include <new>
#include <vector>

#include "common.h"

namespace dcp {

struct RecordedCalls {
  std::vector<std::function<int(void*)>> calls;
  bool whole = true;
};

namespace {
thread_local RecordedCalls* t_recording = nullptr;
thread_local bool t_suspended = false;
}  // namespace

RecordedCalls* current_recording() { return t_suspended ? nullptr : t_recording; }
void record_call(RecordedCalls* list, std::function<int(void*)> call) { list->calls.push_back(std::move(call)); }
void recording_failed(RecordedCalls* list) { list->whole = false; }
void suspend_recording(bool suspended) { t_suspended = suspended; }

}  // namespace dcp

using dcp::RecordedCalls;

extern "C" void* dcp_record_begin(void) {
  if (dcp::t_recording != nullptr) return nullptr;
  dcp::t_recording = new (std::nothrow) RecordedCalls;
  return dcp::t_recording;
}

extern "C" int dcp_record_end(void) {
  DCP_REQUIRE(dcp::t_recording != nullptr, "record_end: this thread is not recording");
  const bool whole = dcp::t_recording->whole;
  dcp::t_recording = nullptr;
  DCP_REQUIRE(whole, "record_end: a call could not be recorded, out of host memory");
  return DCP_OK;
}

extern "C" int dcp_record_size(const void* list) { return list ? (int)static_cast<const RecordedCalls*>(list)->calls.size() : 0; }

extern "C" int dcp_record_run(const void* list, int begin, int end, void* stream) {
  DCP_REQUIRE(list != nullptr, "record_run: null list");
  DCP_REQUIRE(static_cast<const RecordedCalls*>(list)->whole, "record_run: a call is missing from the list");
  const auto& calls = static_cast<const RecordedCalls*>(list)->calls;
  DCP_REQUIRE(begin >= 0 && begin <= end && end <= (int)calls.size(), "record_run: calls %d to %d of %zu", begin, end, calls.size());
  for (int i = begin; i < end; ++i)
    if (const int status = calls[i](stream)) return status;
  return DCP_OK;
}

extern "C" void dcp_record_free(void* list) { delete static_cast<RecordedCalls*>(list); }

extern "C" int dcp_sequence_run(const dcp_sequence_op* ops, int n_ops, void* stream) {
  DCP_REQUIRE(n_ops >= 0 && (n_ops == 0 || ops != nullptr), "sequence_run: no operations");
  for (int i = 0; i < n_ops; ++i) {
    const dcp_sequence_op& op = ops[i];
    void* const on = op.on_caller ? stream : op.stream;
    if (op.kind == DCP_SEQUENCE_RUN) {
      if (const int status = dcp_record_run(op.list, op.begin, op.end, on)) return status;
      continue;
    }
    DCP_REQUIRE((op.kind == DCP_SEQUENCE_RECORD || op.kind == DCP_SEQUENCE_WAIT) && op.event != nullptr,
                "sequence_run: operation %d is of kind %d, event %p", i, op.kind, op.event);
    const hipError_t e = op.kind == DCP_SEQUENCE_RECORD ? hipEventRecord((hipEvent_t)op.event, (hipStream_t)on)
                                                        : hipStreamWaitEvent((hipStream_t)on, (hipEvent_t)op.event, 0);
    if (e != hipSuccess) return dcp::fail(DCP_ERR_LAUNCH, "sequence_run: operation %d: %s", i, hipGetErrorString(e));
  }
  return DCP_OK;
}
