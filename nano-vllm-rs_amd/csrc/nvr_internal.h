// Host-side internals of the nano-vllm-rs HIP library: the context object,
// status plumbing and launch checks shared by every translation unit.
#pragma once

#include <hip/hip_runtime.h>
#include <hipblas/hipblas.h>
#include <stdint.h>

struct nv_context {
    int device;
    hipStream_t stream;
    hipblasHandle_t blas;
    int cu_count;
    // Device address of this device's copy of the sampler's static partials
    // (sample.hip), for nv_sample_parallel_static.
    void* static_partials;
    // The paired sampler's per-row exchange words (sample.hip): two uint64
    // per row, zero between launches (every launch leaves them zero).
    void* pair_state;
};

namespace nvr {

// Records "<operation>: <message> (<code>)" in the calling thread's error
// buffer and returns the status unchanged (0 leaves the buffer untouched).
int hip_status(hipError_t status, const char* operation);
int blas_status(hipblasStatus_t status, const char* operation);
int fail(int code, const char* fmt, ...);

// Looks up this device's copy of the sampler's static partials (called by
// nv_create with the context's device current).
int bind_static_partials(nv_context* c);

// Allocates and zeroes the paired sampler's exchange words (nv_create);
// released by nv_destroy.
int create_pair_state(nv_context* c);

// The tile form of nv_attention (attention_prefill.hip): whether the call's
// shape takes it, and its launch. Needs 16-byte aligned q, caches and out and
// blocks * bs below 2^31.
bool attention_tiles_fit(const nv_context* c, int rows, int qh, int kvh, int dim, int bs, int batch, int max_context);
void launch_attention_tiles(nv_context* c, const uint16_t* q, const uint16_t* k, const uint16_t* v, const int* p,
                            const int* s, const int* t, uint16_t* o, int rows, int qh, int kvh, int bs, int blocks,
                            int stride, int batch, int max_context);

// nv_gemm's few-row form over a wide weight (gemm_stream.hip): whether the call
// takes it, and its launch.
bool gemm_stream_fits(const nv_context* c, const void* x, const void* w, const void* y, int m, int n, int k);
void launch_gemm_stream(nv_context* c, const uint16_t* x, const uint16_t* w, uint16_t* y, int m, int n, int k);

// nv_gemm's calls that take nv_gemm_rows' kernels (gemm.hip).
bool gemm_rows_fits(const nv_context* c, const void* x, const void* w, int m, int n, int k);

// Status of the most recent launch on this thread.
inline int launch_status() { return hip_status(hipGetLastError(), "HIP kernel launch"); }

inline bool aligned(const void* p, uintptr_t bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; }

}  // namespace nvr

#define NVR_HIP(call)                                                  \
    do {                                                               \
        int nvr_error_ = ::nvr::hip_status((call), #call);             \
        if (nvr_error_) return nvr_error_;                             \
    } while (0)
#define NVR_BLAS(call)                                                 \
    do {                                                               \
        int nvr_error_ = ::nvr::blas_status((call), #call);            \
        if (nvr_error_) return nvr_error_;                             \
    } while (0)
#define NVR_ACTIVATE(c) NVR_HIP(hipSetDevice((c)->device))
