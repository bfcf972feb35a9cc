// Device-to-host copies of large results into the caller's ordinary memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace rmhd {

// One contiguous piece of a result in the caller's memory.
struct HostSpan {
    void *dst;
    size_t bytes;
};

// A handle that may download calls copy_retain once and copy_release when it
// is destroyed: the pinned buffers of the copies are kept while any handle
// lives (at most two, 32 MiB each, shared by all handles and threads).
void copy_retain();
void copy_release();

// Copies a result that the device produces piece by piece into spans[0..n).
// fill(i, &src) queues on stream s what produces the pieces i, i+1, ... and
// returns how many of them are then at src, one after another without gaps
// (0: an error, in *err); it is called again for the next piece once the copies
// of the earlier ones are queued on s, so it may reuse the memory at src.
// Returns when every span is written.
typedef int (*FillFn)(void *ctx, int i, const char **src, hipError_t *err);
hipError_t copy_out(const HostSpan *spans, int n, FillFn fill, void *ctx, hipStream_t s);

}  // namespace rmhd
