// Host-side services shared by the generated entry points: error recording, per-stream reduction
// scratch, launch-heuristic knobs.  Implemented in knet8_runtime.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <mutex>

#ifndef KNET8_API
#define KNET8_API __attribute__((visibility("default")))
#endif

namespace knet8 {

// The entry points return void like the reference's (errors there are unchecked, src/libknet8/LibKnet8.jl:54);
// failures are kept as text for knet8_last_error() instead of being dropped.
void record_error(const char* what);
void check_launch(const char* name);  // records hipGetLastError() if a launch failed

// Scratch that split reductions need beyond their inputs and outputs: `partial` holds the per-workgroup
// partial results, `counters` the per-output-group tickets (all zero between launches; the kernel that
// uses them resets them).  One per stream, so launches on different streams never share it; launches on one stream are
// ordered and may.  Where a first launch leaves sums there that a second one reads, another host thread's launch must not
// come in between: a Workspace keeps the stream's scratch to its thread until it goes out of scope, so keep it until the
// last launch that uses it is queued.
struct Workspace {
  void* partial = nullptr;
  unsigned* counters = nullptr;
  std::unique_lock<std::recursive_mutex> held;
};
// optional: the caller does without when there is none, so a failure is not recorded.
// (spare_capture: nothing is allocated for a stream under capture, where an allocation may end the capture; what it has already is given out)
Workspace workspace_for(hipStream_t stream, size_t partial_bytes, size_t ncounters, bool optional = false, bool spare_capture = false);
// Where a split launch takes its scratch from: the per-stream buffers above (a null source) or a caller-supplied provider.  A provider
// that cannot serve the request records why and returns null pointers.
struct ScratchSource {
  Workspace (*get)(void* ctx, hipStream_t stream, size_t partial_bytes, size_t ncounters);
  void* ctx;
  size_t partial_capacity, counter_capacity;   // what the provider can serve at most (0: it grows as needed); launch planners that have a choice stay within it
};
inline bool scratch_fits(const ScratchSource* src, size_t partial_bytes, size_t ncounters) {
  return src == nullptr || ((src->partial_capacity == 0 || partial_bytes <= src->partial_capacity) &&
                            (src->counter_capacity == 0 || ncounters <= src->counter_capacity));
}
// Tickets of different output groups sit 256 bytes apart: atomics on one 64-byte line are carried out one after the other (11-12 ns each on MI355X,
// measured: 256 workgroups drawing from 16 counters 4 bytes apart take 1.9 us longer than from counters 256 bytes apart).
constexpr int kTicketStride = 64;   // in counters

inline Workspace take_scratch(const ScratchSource* src, hipStream_t stream, size_t partial_bytes, size_t ncounters) {
  return src ? src->get(src->ctx, stream, partial_bytes, ncounters) : workspace_for(stream, partial_bytes, ncounters);
}
// A launch split over several workgroups stores partial results and draws tickets through these pointers: without them it must not be
// issued at all (out of device memory is an error to report, src/knetarrays/kptr.jl:114-141, not a fault on the device).
inline bool scratch_ready(const Workspace& ws, const char* who) {
  if (ws.partial != nullptr && ws.counters != nullptr) return true;
  record_error(who);   // the allocation's own failure, recorded first, is the message that is kept
  return false;
}
// Slot for the result of a `_20` reduction on this stream (host memory that the kernel writes), and the wait that fetches it (4 or 8 bytes).
void* scalar_slot(hipStream_t stream);
void fetch_scalar(hipStream_t stream, const void* slot, void* host, size_t nbytes);

// `n` 4-byte words of page-locked host memory that a kernel can read, for small arrays that go with one launch: fill `host`, queue the launch that reads it, let go.
// No other thread is given the stream's buffer in between.  host is null where there is none (stream under capture, the per-thread stream, too many words, no memory).
struct StagedWords {
  unsigned* host = nullptr;
  std::unique_lock<std::recursive_mutex> held;
};
StagedWords stage_words(hipStream_t stream, size_t n);
bool stream_is_capturing(hipStream_t stream);
// Copies n words that stand in the stream's staging buffer (staged; the caller still holds them) or anywhere in host memory to the device, in order with the stream's launches.
bool bring_words(hipStream_t stream, void* dst, const void* src, size_t n, bool staged);

// Blocks of the KnetArray pool (knet8_malloc, knet8_free).
void* pool_take(size_t nbytes);
void pool_give(void* p);

// State of the default random stream (knet8_seed): hands out `blocks` consecutive generator counters under the current seed.
void rng_take(unsigned long long blocks, unsigned long long* seed, unsigned long long* offset);

enum { kTuneNumCUs = 0, kTuneSoftmaxResidentRows = 1, kTuneGemmSmallMflop = 3, kTuneDenseBackMflop = 4, kTuneFailScratch = 5, kTuneSoftmaxNoLdsSlots = 6, kTuneGemmDryRun = 7, kTuneGemmNoPrepared = 8, kTuneGemmSplit = 9, kTuneGemmSmallRule = 10, kTuneGemmMid = 11, kTuneCount = 12 };
int tuning(int key);
bool tuned(int key);   // set by the caller, not at its default (of keys whose default is not remembered: all but kTuneNumCUs)

#ifdef KNET8_TIMELINE
struct TlStamp;
TlStamp* timeline_buffer();   // measurement build: where the stamped kernels write (null: nowhere), set by knet8_timeline_set
#endif

}  // namespace knet8
