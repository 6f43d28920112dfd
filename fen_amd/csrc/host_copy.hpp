// host_copy.hpp -- copies of n values between a caller's FP64 array and device
// memory of element size es (8: FP64, 4: FP32, each value rounded to nearest
// once), ordered after the work queued on `stream`; done when they return.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace fen {

void copy_to_host(hipStream_t stream, double *dst, const void *src, size_t n, size_t es);
// FP64 copies of which several are queued before the caller waits for the stream
// once (a wait costs as much as a small copy); they may be done on return.
void queue_to_host(hipStream_t stream, double *dst, const double *src, size_t n);
void queue_to_device(hipStream_t stream, double *dst, const double *src, size_t n);
void copy_to_device(hipStream_t stream, void *dst, const double *src, size_t n, size_t es);
// A context is created (+1) or destroyed (-1): the last one frees the pinned pieces.
void host_copy_user(int change);

}  // namespace fen
