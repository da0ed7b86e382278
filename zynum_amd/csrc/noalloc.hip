// A GEMM request entry point that allocates nothing, for callers that cannot
// call hipMalloc (code under HIP graph capture, tight serving loops).
//
// It runs the plain FP64/FP32 MFMA GEMM of zynum_gpu_gemm on device operands.
// The only device memory beyond the caller's A, B and C is the buffer of the
// K ranges' partial sums (output tiles that are split over K), which here is
// a fixed file-scope device array instead of the staging-buffer cache.  The
// plans of both scalar types are bounded by kGemmScratchMax (24 MiB); the
// 64 x 64 plan for operands that the direct loads do not take needs at most
// (512 + 127) * 4096 elements, 20.9 MB.
//
// Two arrays per device.  One is for synchronous calls, which split most
// mid-size products: a call that splits holds it (a mutex) until its work is
// done, so synchronous calls of several threads never share it in flight.  The
// other is for asynchronous calls, which split only where few tiles walk a
// long K: nobody waits for them, so those that overlap on one device race on
// it.  Nothing needs clearing: a split call writes every partial it reads.
#include <mutex>

#include "abi_common.hpp"
#include "gemm.hpp"
#include "runtime.hpp"

namespace zg {
namespace {

constexpr size_t kScratchBytes = kGemmScratchMax;
// [0] asynchronous calls, [1] synchronous ones
static __device__ __align__(256) double scratch[2][kScratchBytes / sizeof(double)];

constexpr int kMaxDevices = 64;
struct DeviceScratch {
    std::once_flag once;
    char* ptr = nullptr;
    int status = ZYNUM_GPU_OK;
    std::mutex synchronous;  // held by the synchronous call that uses its array
};
DeviceScratch g_scratch[kMaxDevices];

// The current device's arrays (each device holds its own copy): their address
// is looked up once per device with that device current.  The array's name is
// a host-side stand-in and is never passed on.
int scratch_of_device(DeviceScratch** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        (void)hipGetLastError();
        return ZYNUM_GPU_DECLINE_NO_DEVICE;
    }
    DeviceScratch& d = g_scratch[dev];
    std::call_once(d.once, [&d] {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            (void)hipGetLastError();
            d.status = ZYNUM_GPU_ERR_LAUNCH;
            return;
        }
        d.ptr = static_cast<char*>(p);
    });
    *out = &d;
    return d.status;
}

template <typename T>
int gemm_noalloc(const zynum_gpu_gemm_request* r, hipStream_t s) {
    const bool ta = r->transa != ZYNUM_GPU_NO_TRANS, tb = r->transb != ZYNUM_GPU_NO_TRANS;
    const T alpha = scalar_from_bits<T>(r->alpha_re), beta = scalar_from_bits<T>(r->beta_re);
    const int m = r->m, n = r->n, k = r->k;
    if (m <= 0 || n <= 0) return ZYNUM_GPU_OK;  // gemm.zig:1393
    if (take_forced_decline()) return ZYNUM_GPU_DECLINE_FORCED;
    if (!device_ready()) return ZYNUM_GPU_DECLINE_NO_DEVICE;
    const bool reads_ab = (k > 0) && (alpha != T(0));
    // device operands only: staging host memory would need buffers
    if (!is_device_pointer(r->c) || (reads_ab && (!is_device_pointer(r->a) || !is_device_pointer(r->b))))
        return ZYNUM_GPU_DECLINE_UNSUPPORTED;
    GemmDesc<T> d;
    d.ta = ta; d.tb = tb; d.m = m; d.n = n; d.k = k;
    d.lda = r->lda; d.ldb = r->ldb; d.ldc = r->ldc;
    d.alpha = alpha; d.beta = beta;
    d.a = static_cast<const T*>(r->a); d.b = static_cast<const T*>(r->b); d.c = static_cast<T*>(r->c);
    const int tile = r->tile == 0 ? kTileAuto : r->tile - 1;
    const bool waits = !(r->flags & ZYNUM_GPU_FLAG_ASYNC);
    const size_t want = (reads_ab && tile == kTileAuto) ? gemm_scratch_bytes<T>(d, waits) : 0;
    std::unique_lock<std::mutex> held;  // until this call's work is done
    hipError_t e;
    if (want > 0) {
        if (want > kScratchBytes) return ZYNUM_GPU_DECLINE_SCRATCH;
        DeviceScratch* scr = nullptr;
        const int st = scratch_of_device(&scr);
        if (st != ZYNUM_GPU_OK) return st;
        if (waits) held = std::unique_lock<std::mutex>(scr->synchronous);
        e = gemm_launch_scratch<T>(d, s, reinterpret_cast<T*>(scr->ptr + (waits ? kScratchBytes : 0)));
    } else {
        e = gemm_launch<T>(d, s, tile);
    }
    if (waits) {
        const hipError_t waited = hipStreamSynchronize(s);
        if (e == hipSuccess) e = waited;
    }
    return status_from_hip(e);
}

}  // namespace
}  // namespace zg

extern "C" int zynum_gpu_gemm_noalloc(const zynum_gpu_gemm_request* r) {
    if (r == nullptr) return ZYNUM_GPU_DECLINE_ARGUMENT;
    const char ta = zg::request_trans_char(r->transa, false), tb = zg::request_trans_char(r->transb, false);
    if (zg::gemm_error(ta, tb, r->m, r->n, r->k, r->lda, r->ldb, r->ldc) != 0) return ZYNUM_GPU_DECLINE_ARGUMENT;
    if (r->scalar != ZYNUM_GPU_F64 && r->scalar != ZYNUM_GPU_F32) return ZYNUM_GPU_DECLINE_UNSUPPORTED;
    if (r->mode != ZYNUM_GPU_MODE_PLAIN || r->tile > zg::kTileConfigs) return ZYNUM_GPU_DECLINE_UNSUPPORTED;
    // the request's stream, else the one set by zynum_gpu_set_stream, else the null stream
    // (the library's own stream is created on first use, so it is not taken here)
    hipStream_t s = r->stream ? reinterpret_cast<hipStream_t>(r->stream) : zg::caller_stream();
    return r->scalar == ZYNUM_GPU_F64 ? zg::gemm_noalloc<double>(r, s) : zg::gemm_noalloc<float>(r, s);
}
