// gdn_noalloc.hip -- gdn_recurrence_noalloc: the gated delta-rule steps of
// gdn_test_recurrence on caller-owned device buffers, with no allocation of
// any kind (for callers that cannot allocate: code under HIP graph capture,
// serving loops).
//
// The only memory beyond the caller's inputs and outputs is one entry per
// (step, head) of scalars.  It lives in the file-scope device array `scratch`
// below (kScratchEntries entries, 512 KiB on every GPU the library runs on,
// held until the process ends).  Steps are processed in chunks that fit it:
// one kernel fills the chunk's entries, then the recurrence reads them -- one
// launch for the whole chunk, the state in registers (gdn_scan.h), or one
// launch per step; stream order keeps the next chunk's fill behind the last
// launch that reads the previous one.  Every call on a GPU shares that GPU's
// array, so calls that overlap on one GPU race.
//
// Host code never passes `scratch` itself to a kernel: its name is a
// host-side stand-in, not a device address.  The device address is looked up
// once per device with hipGetSymbolAddress and kept in g_scratch_ptr.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <mutex>

#include "gdn_amd.h"
#include "gdn_device.h"
#include "gdn_internal.h"
#include "gdn_scan.h"

namespace {

constexpr int kScratchEntries = 16384;
constexpr int kMaxDevices = 64;
constexpr int kCols = 16;              // state columns per recurrence workgroup

// beta and decay first: the per-step kernel reads them as pairs of its own
// layout (float2 per entry, from the array's start)
struct Entry {
    gdn::f32x4 scal;  // beta, decay, alpha
    float inv[4];     // 1 / |k|, 1 / |q|
};
__device__ __align__(256) Entry scratch[kScratchEntries];

std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current device, looked up on the
// first call there.
void *scratch_ptr() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        gdn_error("gdn_recurrence_noalloc: no current device");
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void *p = nullptr;
        const hipError_t rc = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (rc != hipSuccess || p == nullptr) {
            std::fprintf(stderr, "gdn_recurrence_noalloc: hipGetSymbolAddress failed: %s\n", hipGetErrorString(rc));
            return nullptr;
        }
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

// (beta, decay) of n (step, head) pairs, from raw (a, b, a_log, dt_bias).
__global__ __launch_bounds__(gdn::kT) void k_scalars(const float *__restrict__ a, const float *__restrict__ b,
                                                     const float *__restrict__ a_log,
                                                     const float *__restrict__ dt_bias, int n,
                                                     float2 *__restrict__ out) {
    const int i = blockIdx.x * gdn::kT + threadIdx.x;
    if (i >= n) return;
    float beta, decay;
    gdn::head_scalars(a[i], b[i], a_log[i], dt_bias[i], beta, decay);
    out[i] = make_float2(beta, decay);
}

// The entries of n (step, head) pairs, a wave each: the norms and alpha in
// gdn_tree_reduce_256's order (four values in a lane, then the lanes), beta
// and decay.
__global__ __launch_bounds__(gdn::kT) void k_entries(const float *__restrict__ q, const float *__restrict__ k,
                                                     const float *__restrict__ a, const float *__restrict__ b,
                                                     const float *__restrict__ a_log,
                                                     const float *__restrict__ dt_bias, int n,
                                                     Entry *__restrict__ out) {
    using gdn::f32x4;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    const f32x4 qv = *reinterpret_cast<const f32x4 *>(q + (size_t)i * gdn::kHD + 4 * lane);
    const f32x4 kv = *reinterpret_cast<const f32x4 *>(k + (size_t)i * gdn::kHD + 4 * lane);
    auto tree = [](f32x4 x, f32x4 y) {
        return gdn::wave_tree64((x.x * y.x + x.y * y.y) + (x.z * y.z + x.w * y.w));
    };
    const float q_inv = 1.0f / __builtin_sqrtf(tree(qv, qv) + 1e-6f);
    const float k_inv = 1.0f / __builtin_sqrtf(tree(kv, kv) + 1e-6f);
    const f32x4 qn = {qv.x * q_inv, qv.y * q_inv, qv.z * q_inv, qv.w * q_inv};
    const f32x4 kn = {kv.x * k_inv, kv.y * k_inv, kv.z * k_inv, kv.w * k_inv};
    const float alpha = tree(qn, kn);
    if (lane == 0) {
        float beta, decay;
        gdn::head_scalars(a[i], b[i], a_log[i], dt_bias[i], beta, decay);
        out[i].scal = (f32x4){beta, decay, alpha, 0.0f};
        out[i].inv[0] = k_inv;
        out[i].inv[1] = q_inv;
    }
}

struct EntryScalars {
    const Entry *e;  // this head's entry of the first step
    int heads;
    __device__ __forceinline__ gdn::f32x4 get(int m) const { return e[(size_t)m * heads].scal; }
    __device__ __forceinline__ float inv(int m, int kind) const { return e[(size_t)m * heads].inv[kind]; }
};

// n_steps steps of every head: grid (256 / kScanWgCols, heads).
template <int C>
__global__ __launch_bounds__(gdn::kT) void k_scan(const float *__restrict__ q, const float *__restrict__ k,
                                                  const float *__restrict__ v, const Entry *__restrict__ entries,
                                                  int n_steps, void *__restrict__ S, float *__restrict__ o) {
    __shared__ gdn::ScanLds lds;
    const int h = blockIdx.y, heads = gridDim.y, c0 = blockIdx.x * gdn::kScanWgCols;
    gdn::ScanArgs a;
    a.q = q + (size_t)h * gdn::kHD;
    a.k = k + (size_t)h * gdn::kHD;
    a.v = v + (size_t)h * gdn::kHD + c0;
    a.o = o + (size_t)h * gdn::kHD + c0;
    a.ldq = a.ldv = a.ldo = (size_t)heads * gdn::kHD;
    a.n = n_steps;
    const size_t at = (size_t)h * gdn::kHD * gdn::kHD + c0;
    void *s = C == gdn::kRef ? static_cast<void *>(static_cast<uint16_t *>(S) + at)
                             : static_cast<void *>(static_cast<float *>(S) + at);
    gdn::scan_block<C, true>(a, EntryScalars{entries + h, heads}, s, lds);
}

// One step of every head: grid (256 / kCols, heads).
template <int C>
__global__ __launch_bounds__(gdn::kT) void k_step(const float *__restrict__ q, const float *__restrict__ k,
                                                  const float *__restrict__ v, const float2 *__restrict__ bd,
                                                  void *__restrict__ S, float *__restrict__ o) {
    const gdn::ScalarsFromPairs scal{reinterpret_cast<const float *>(bd)};
    gdn::recur_block<C, kCols, false, false, false>(q, k, v, scal, nullptr, S, o, nullptr, blockIdx.y,
                                                     blockIdx.x * kCols);
}

// Whether `steps` steps of every head run as one scan or step by step.  The
// scan reads and writes the state once, in 32-byte pieces (8 columns a
// workgroup); a step's launch moves it in whole lines but costs at least 5 us
// and the state's traffic again.  Measured (FP32 state, per-step / scan, us):
//   8 heads: 1 step 10.5 / 12.9, 2 steps 14.8 / 13.6, 100 steps 559 / 87
//   48 heads: 2 steps 27 / 35, 3 steps 40 / 36, 100 steps 1194 / 324
//   256 heads: 3 steps 140 / 129 (REF 134 / 136), 4 steps 185 / 134
//   1024 heads: 3 steps 470 / 516, 4 steps 628 / 553
// The scan's 16-byte loads of q and k need them so aligned; a caller's
// buffers at other addresses keep the per-step kernel.
bool use_scan(uint32_t heads, uint32_t steps, const float *q, const float *k) {
    const bool aligned = ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) & 15) == 0;
    return aligned && (steps >= 4 || (steps == 3 && heads <= 96) || (steps == 2 && heads <= 8));
}

}  // namespace

extern "C" int gdn_recurrence_noalloc(int contract, uint32_t n_heads, uint32_t n_steps, const float *q,
                                      const float *k, const float *v, const float *a, const float *b,
                                      const float *a_log, const float *dt_bias, void *S, float *o,
                                      void *stream) {
    if (contract < GDN_CONTRACT_REF || contract > GDN_CONTRACT_FP32) {
        std::fprintf(stderr, "gdn_recurrence_noalloc: unknown contract %d\n", contract);
        return -1;
    }
    if (n_heads == 0 || n_heads > (uint32_t)kScratchEntries) {
        std::fprintf(stderr, "gdn_recurrence_noalloc: %u heads; the scratch array holds one step of at most %d\n",
                     n_heads, kScratchEntries);
        return -1;
    }
    if (n_steps == 0) return 0;
    if (!q || !k || !v || !a || !b || !a_log || !dt_bias || !S || !o) {
        gdn_error("gdn_recurrence_noalloc: a buffer pointer is NULL");
        return -1;
    }
    void *mem = scratch_ptr();
    if (mem == nullptr) return -1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t chunk = (uint32_t)kScratchEntries / n_heads;  // steps per scratch fill
    for (uint32_t s0 = 0; s0 < n_steps; s0 += chunk) {
        const uint32_t ns = (n_steps - s0 < chunk) ? n_steps - s0 : chunk;
        const size_t first = (size_t)s0 * n_heads;
        const int n = (int)(ns * n_heads);
        if (use_scan(n_heads, ns, q, k)) {
            Entry *en = static_cast<Entry *>(mem);
            const size_t ov = first * gdn::kHD;
            const dim3 grid(gdn::kHD / gdn::kScanWgCols, n_heads), block(gdn::kT);
            hipLaunchKernelGGL(k_entries, dim3((unsigned)((n + 3) / 4)), block, 0, s, q + ov, k + ov, a + first,
                               b + first, a_log + first, dt_bias + first, n, en);
            if (contract == GDN_CONTRACT_REF)
                hipLaunchKernelGGL(k_scan<gdn::kRef>, grid, block, 0, s, q + ov, k + ov, v + ov, en, (int)ns, S,
                                   o + ov);
            else if (contract == GDN_CONTRACT_BF16W_FP32S)
                hipLaunchKernelGGL(k_scan<gdn::kBf16w>, grid, block, 0, s, q + ov, k + ov, v + ov, en, (int)ns, S,
                                   o + ov);
            else
                hipLaunchKernelGGL(k_scan<gdn::kFp32>, grid, block, 0, s, q + ov, k + ov, v + ov, en, (int)ns, S,
                                   o + ov);
            continue;
        }
        float2 *bd = static_cast<float2 *>(mem);
        const dim3 grid(gdn::kHD / kCols, n_heads), block(gdn::kT);
        hipLaunchKernelGGL(k_scalars, dim3((unsigned)((n + gdn::kT - 1) / gdn::kT)), block, 0, s, a + first,
                           b + first, a_log + first, dt_bias + first, n, bd);
        for (uint32_t st = 0; st < ns; ++st) {
            const size_t ov = (size_t)(s0 + st) * n_heads * gdn::kHD;
            const float2 *bds = bd + (size_t)st * n_heads;
            if (contract == GDN_CONTRACT_REF)
                hipLaunchKernelGGL(k_step<gdn::kRef>, grid, block, 0, s, q + ov, k + ov, v + ov, bds, S, o + ov);
            else if (contract == GDN_CONTRACT_BF16W_FP32S)
                hipLaunchKernelGGL(k_step<gdn::kBf16w>, grid, block, 0, s, q + ov, k + ov, v + ov, bds, S, o + ov);
            else
                hipLaunchKernelGGL(k_step<gdn::kFp32>, grid, block, 0, s, q + ov, k + ov, v + ov, bds, S, o + ov);
        }
    }
    const hipError_t rc = hipGetLastError();
    if (rc != hipSuccess) {
        std::fprintf(stderr, "gdn_recurrence_noalloc: launch failed: %s\n", hipGetErrorString(rc));
        return -1;
    }
    return 0;
}
