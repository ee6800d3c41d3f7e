// Host code: issue a recorded list of kernel launches with other addresses put in.
//
// A step that is not replayed from a HIP graph records the launches of the first layer of a
// kind and launches the other layers of that kind from the list (engine/layer_replay.py).
// Each entry is an entry point in its slot form (slots.h) and its arguments as slots; a
// patch names a slot that holds an address inside one of the layer's own tensors, the
// tensor's place in `addresses`, and the offset inside it.  One call from the host language
// issues the whole layer.
//
// tk_stream_order: what is launched on `to` from now on starts when what has been launched on `from` so far is done.  As an
// entry point of its own it stands in recorded lists, and in a HIP graph that is being recorded it is the edge between two branches.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"
#include "slots.h"

typedef int (*slots_fn)(const unsigned long long*);

// Returns -1 when every call returned the status it returned when it was recorded; else the
// index of the first call that did not (its status in *got), after which nothing is issued.
extern "C" __attribute__((visibility("default"))) int tk_replay_calls(
    int ncalls, const void* const* fns, const int* first_slot, unsigned long long* slots, int npatches,
    const int* patch_slot, const int* patch_key, const long long* patch_offset,
    const unsigned long long* addresses, const int* expected, int* got) {
  for (int p = 0; p < npatches; ++p)
    slots[patch_slot[p]] = addresses[patch_key[p]] + (unsigned long long)patch_offset[p];
  for (int c = 0; c < ncalls; ++c) {
    const int status = reinterpret_cast<slots_fn>(const_cast<void*>(fns[c]))(slots + first_slot[c]);
    if (status != expected[c]) {
      *got = status;
      return c;
    }
  }
  return -1;
}

TK_API int tk_stream_order(hipStream_t from, hipStream_t to) {
  if (from == to) return 0;
  hipEvent_t event;
  hipError_t status = hipEventCreateWithFlags(&event, hipEventDisableTiming);
  if (status != hipSuccess) return (int)status;
  status = hipEventRecord(event, from);
  if (status == hipSuccess) status = hipStreamWaitEvent(to, event, 0);
  const hipError_t gone = hipEventDestroy(event);     // (its work is queued or recorded; the handle is no longer needed)
  return (int)(status != hipSuccess ? status : gone);
}

TK_SLOTS(tk_stream_order)
