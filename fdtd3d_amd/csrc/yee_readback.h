// Device-to-host copies of whole fields (yee_readback.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace yee {

// Every handle and batch holds one reference from its creation to its destruction; the pinned
// buffers of read_back are allocated once enough has been read (kOpen) and freed with the last reference.
void readback_ref ();
void readback_unref ();

// The n values of wsize bytes at src (device memory of `device`, final once the work queued on
// `stream` is done) into out: as they are, or widened from FP32 to FP64.  Returns when out is
// complete.
hipError_t read_back (int device, hipStream_t stream, const void *src, int64_t n, size_t wsize, void *out, bool widen);

}  // namespace yee
