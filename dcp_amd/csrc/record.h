// Recorded launches: while a thread records, every entry point that launches kernels also notes how
// to repeat its call on another stream, so that a caller with a fixed sequence of calls (a prepared
// plan) can have all of it launched again in one call.
#pragma once

#include <functional>
#include <utility>

namespace dcp {

struct RecordedCalls;
RecordedCalls* current_recording();  // of this thread; null while it does not record or is inside a recorded call
void record_call(RecordedCalls* list, std::function<int(void*)> call);
void recording_failed(RecordedCalls* list);  // a call could not be added
void suspend_recording(bool suspended);

// One per entry point, at its top.  Entry points that call each other record the outermost call.
class RecordScope {
 public:
  template <typename F>
  explicit RecordScope(F&& call) noexcept : list_(current_recording()) {
    if (list_ == nullptr) return;
    try {
      record_call(list_, std::forward<F>(call));
    } catch (...) {  // no host memory: nothing is thrown at a C caller, the list is no good
      recording_failed(list_);
    }
    suspend_recording(true);
  }
  ~RecordScope() {
    if (list_ != nullptr) suspend_recording(false);
  }
  RecordScope(const RecordScope&) = delete;

 private:
  RecordedCalls* list_;
};

// DCP_RECORDED(call): `call` repeats the entry point's own call with its parameters; in it, `stream`
// is the stream of the repetition.
#define DCP_RECORDED(...) ::dcp::RecordScope dcp_record_scope_([=](void* stream) -> int { return __VA_ARGS__; })

}  // namespace dcp
