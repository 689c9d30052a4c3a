// devmem.hpp -- device memory, streams and pinned memory kept between
// problems.
//
// A program that solves one problem after another (bddcml_init_c ...
// bddcml_finalize_c) asks for the same buffers each time.  hipMalloc and
// hipFree of gigabytes take 0.3 ms to several hundred ms, depending on how
// the driver clears the memory, so freed blocks stay here for the next
// problem.  Bounds: an eighth of the device's memory per device; a block
// that a whole problem (until its finalize) did not use is given back then;
// everything is given back when an allocation would otherwise fail, and by a
// finalize without a problem.  All functions may be called from any thread.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace bddc {

// device block of at least `bytes` on the current device, contents undefined
void *dev_alloc(size_t bytes);
// back to the kept blocks, or to the driver beyond their bound.  Waits for
// the block's device first, as hipFree does: work on any stream may still use
// it.
void dev_free(void *p);
// mapped coherent pinned host memory (for values a kernel writes and the
// host polls)
void *pinned_alloc(size_t bytes);
void pinned_free(void *p);
// non-blocking stream of the current device, idle when given back
hipStream_t stream_get();
void stream_put(hipStream_t st);
// end of one problem: gives back what it did not use; with nothing_held,
// everything that is kept
void devmem_end_of_problem(bool nothing_held);
// bytes of device blocks handed out and kept
void devmem_bytes(double &held, double &kept);

}  // namespace bddc
