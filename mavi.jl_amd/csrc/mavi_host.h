// mavi_host.h -- host-side helpers shared by the C entry points of single
// systems (mavi_capi.hip) and replica batches (mavi_batch.hip).
#pragma once
#include <string>

#include "mavi_internal.h"

inline int set_err(mavi_ctx *ctx, int code, const std::string &msg) {
    if (ctx) ctx->err = msg;
    return code;
}

#define HIPCHK(ctx, expr)                                                                                  \
    do {                                                                                                   \
        hipError_t e_ = (expr);                                                                            \
        if (e_ != hipSuccess)                                                                              \
            return set_err((ctx), MAVI_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));           \
    } while (0)

// Allocate and zero on the context's stream: the library's stream is
// non-blocking, so a zero fill on the null stream would not be ordered
// before the stream's own work on the buffer.
template <typename T>
hipError_t dalloc(T **p, int64_t count, hipStream_t st) {
    *p = nullptr;
    if (count <= 0) count = 1;
    hipError_t e = hipMalloc((void **)p, sizeof(T) * (size_t)count);
    if (e == hipSuccess) e = hipMemsetAsync(*p, 0, sizeof(T) * (size_t)count, st);
    return e;
}

template <typename T>
void dfree(T *&p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

// Up to this many particles the chunk gather keeps eight candidates a lane in
// flight (pair_gather_deep; rings four): there are few waves a SIMD, and a
// candidate's trip to memory is what a step waits for.  Above, other waves hide it
// and the extra registers (fewer waves) cost more.  us a step, two candidates in
// flight -> eight: LJ 4k 39.5 -> 37.0, 66k 45.5 -> 40.0, 202k 59.0 -> 54.7, 393k
// 72.9 -> 68.0, 787k 99.4 -> 99.9, 1M 115.9 -> 119.7; with a walls list 160k 66.9
// -> 62.5, 292k 82.2 -> 82.8; self-propelled 32k 23.2 -> 21.2, 490k 49.0 -> 47.0;
// run-and-tumble 32k 20.3 -> 19.7, 131k 25.5 -> 25.2, 292k 34.5 -> 34.4, 490k 38.7
// -> 40.3; rings 2k 31.7 -> 28.6, 20k 34.3 -> 30.8, 200k 50.2 -> 47.2, 298k 58.3 ->
// 55.5; a batch's plain replicas, by the family's slots: 16 of 1k 36.5 -> 31.4, 16
// of 10k 54.5 -> 50.6.
constexpr int64_t kDeepGather = 300000;

inline int nblk(int64_t n, int t) { return (int)((n + t - 1) / t); }

inline bool is_pow2_wg(int32_t w) { return w == 64 || w == 128 || w == 256 || w == 512 || w == 1024; }

// Kernel timing of one launch class with HIP events (mavi_prof_enable): the
// launches inside the scope are bracketed on the stream they run on.
struct ProfScope {
    mavi_sys *s;
    int which;
    hipStream_t st;
    ProfScope(mavi_sys *s_, int w, hipStream_t st_) : s(s_), which(w), st(st_) {
        if (s->prof) (void)hipEventRecord(s->ev0, st);
    }
    ~ProfScope() {
        if (!s->prof) return;
        (void)hipEventRecord(s->ev1, st);
        if (hipEventSynchronize(s->ev1) == hipSuccess) {
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, s->ev0, s->ev1) == hipSuccess) {
                s->profs[which].ms += ms;
                s->profs[which].launches += 1;
            }
        }
    }
};
