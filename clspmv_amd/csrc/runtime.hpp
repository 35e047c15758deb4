// Internal runtime types of libclspmv (context, device buffers).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "clspmv.h"

struct clspmv_ctx_s {
    int device = 0;
    hipStream_t own = nullptr;  // default-priority stream created by clspmv_init
    hipStream_t ext = nullptr;  // caller's stream, if set
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    hipStream_t stream() const { return ext ? ext : own; }
};

namespace clspmv {

int hip_status(hipError_t e, const char* what);

// One device allocation owned by a part or a Cocktail object.
struct DevBuf {
    void* ptr = nullptr;
    size_t size = 0;
    int upload(clspmv_ctx_t ctx, const void* host, size_t bytes);
    int alloc(size_t bytes);
    int put(clspmv_ctx_t ctx, size_t at, const void* host, size_t bytes);  // bytes of host to ptr + at, waits
    void release();
};

}  // namespace clspmv

extern "C" int clspmv_part_launch(clspmv_part_t p, const float* x, float* y, hipStream_t st);
// DIA parts of narrow-band square matrices: iterations {y += A x; x := y} one
// launch can take (0: other parts), the launches that so many iterations are
// dealt to (0: they go one by one), and such a launch from x, y into xout (may
// be null) and yout, which x and y must not overlap.
extern "C" int clspmv_part_step_limit(clspmv_part_t p);
extern "C" int clspmv_part_step_launches(clspmv_part_t p, int iterations);
extern "C" int clspmv_part_launch_steps(clspmv_part_t p, int steps, const float* x, const float* y, float* xout,
                                        float* yout, hipStream_t st);
