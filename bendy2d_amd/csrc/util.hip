// util.hip -- fill and device-wide exclusive scan.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/bendy2d.h"
#include "engine.h"
#include "kernels.h"

namespace bd {

__global__ void k_fill_u32(uint32_t *p, size_t n, uint32_t v) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

void launch_fill_u32(uint32_t *p, size_t n, uint32_t v, hipStream_t stream) {
    if (!n) return;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, stream, p, n, v);
}

// The parts of an engine's state one after another into dst, a word to a lane:
// whole cache lines a wavefront whether they go to HBM or over PCIe.  What bounds
// it is the launch for small scenes and the link for large ones.  A frame of 5
// polygons, read back, 135 -> 88 us against a copy per array into pageable memory,
// of 32 x 32 particles 263 -> 228; 20 updates of 1,048,576 and one readback
// 13.7 -> 11.1 ms.
__global__ void __launch_bounds__(256) k_gather_state(StateParts s, uint64_t *__restrict__ dst) {
    const size_t first = (size_t)blockIdx.x * 256u + threadIdx.x, step = (size_t)gridDim.x * 256u;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const StateParts::Part &p = s.part[k];
        const uint64_t *const src = (const uint64_t *)p.src;
        for (size_t i = first; i < p.words; i += step) dst[i] = src[p.index ? (size_t)p.index[i] : i];
        dst += p.words;
    }
}

hipError_t gather_state(const StateParts &parts, void *dst, hipStream_t stream) {
    size_t words = 0;
    for (const StateParts::Part &p : parts.part) words = std::max<size_t>(words, p.words);
    if (!words) return hipSuccess;
    // kernels go to the current device, which need not be the stream's
    int now = 0;
    hipDevice_t own = 0;
    hipError_t e = hipGetDevice(&now);
    if (e == hipSuccess) e = hipStreamGetDevice(stream, &own);
    if (e == hipSuccess && own != now) e = hipSetDevice(own);
    if (e != hipSuccess) return e;
    const size_t blocks = std::min<size_t>((words + 255) / 256, 2048);
    hipLaunchKernelGGL(k_gather_state, dim3((unsigned)blocks), dim3(256), 0, stream, parts, (uint64_t *)dst);
    e = hipGetLastError();
    if (own != now) (void)hipSetDevice(now);
    return e;
}

int Engine::download(HostScene &s, PinnedPool &pool, std::string &err) {
    const size_t words = state_count();
    const StateParts parts = state_parts();
    PinnedBuf host = pool.take(words * sizeof(float2));
    if (host.p) {
        BD_HIP(gather_state(parts, host.p, stream()));
        BD_HIP(hipStreamSynchronize(stream()));
        const int rc = unpack((const float2 *)host.p, s, err);
        pool.give(std::move(host));
        return rc;
    }
    // more than the pool holds, or no page-locked memory left: into pageable memory,
    // a part at a time where none is read by index
    DevBuf<float2> dev;
    std::vector<float2> plain(std::max<size_t>(words, 1));
    bool by_index = false;
    for (const StateParts::Part &p : parts.part) by_index |= p.index != nullptr;
    if (by_index) {
        BD_HIP(dev.alloc(plain.size()));
        BD_HIP(gather_state(parts, dev.p, stream()));
        BD_HIP(hipMemcpyAsync(plain.data(), dev.p, words * sizeof(float2), hipMemcpyDeviceToHost, stream()));
    } else {
        float2 *to = plain.data();
        for (const StateParts::Part &p : parts.part) {
            if (p.words) BD_HIP(hipMemcpyAsync(to, p.src, p.words * sizeof(float2), hipMemcpyDeviceToHost, stream()));
            to += p.words;
        }
    }
    BD_HIP(hipStreamSynchronize(stream()));
    return unpack(plain.data(), s, err);
}

std::shared_ptr<PinnedPool> PinnedPool::shared() {
    static std::mutex m;
    static std::weak_ptr<PinnedPool> pool;
    std::lock_guard<std::mutex> hold(m);
    std::shared_ptr<PinnedPool> p = pool.lock();
    if (!p) pool = p = std::make_shared<PinnedPool>();
    return p;
}

PinnedBuf PinnedPool::take(size_t bytes) {
    PinnedBuf b;
    {
        std::lock_guard<std::mutex> hold(m_);
        int best = -1;
        for (int k = 0; k < kKept; k++)
            if (kept_[k].p && kept_[k].n >= bytes && (best < 0 || kept_[k].n < kept_[best].n)) best = k;
        if (best >= 0) b = std::move(kept_[best]);
    }
    if (!b.p && bytes <= kKeptBytes) {
        // a half more, so that a growing scene does not ask anew each time, as long
        // as the buffer can be kept
        hipError_t e = b.alloc(std::max(kLeast, std::min(bytes + bytes / 2, kKeptBytes)));
        if (e != hipSuccess) e = b.alloc(std::max<size_t>(bytes, 16));
        if (e != hipSuccess) (void)hipGetLastError();
    }
    return b;
}

void PinnedPool::give(PinnedBuf &&b) {
    PinnedBuf drop[kKept + 1];  // freed after the lock
    std::lock_guard<std::mutex> hold(m_);
    drop[kKept] = std::move(b);
    if (!drop[kKept].p || drop[kKept].n > kKeptBytes) return;
    // the smallest kept ones make way
    for (int gone = 0;;) {
        size_t total = drop[kKept].n;
        int least = -1, room = -1;
        for (int k = 0; k < kKept; k++) {
            if (!kept_[k].p) { room = k; continue; }
            total += kept_[k].n;
            if (least < 0 || kept_[k].n < kept_[least].n) least = k;
        }
        if (room >= 0 && total <= kKeptBytes) {
            kept_[room] = std::move(drop[kKept]);
            return;
        }
        drop[gone++] = std::move(kept_[least]);
    }
}

// Plain streaming copy, 16 bytes per lane and iteration: the reference kernel
// for reading HBM byte counters and for the achievable copy bandwidth.
__global__ void k_copy_f4(const float4 *__restrict__ src, float4 *__restrict__ dst, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) dst[i] = src[i];
}

constexpr int kScanThreads = 256;
constexpr int kScanPerThread = 4;
constexpr int kScanTile = kScanThreads * kScanPerThread;  // 1024 words per block

// Inclusive prefix sum across the 64 lanes of a wavefront.
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

// Exclusive scan of one 1024-word tile; the tile total goes to sums[block].
__global__ void __launch_bounds__(kScanThreads) k_scan_tile(const uint32_t *in, uint32_t *out, size_t n,
                                                            uint32_t *sums) {
    __shared__ uint32_t s_wave[kScanThreads / 64];
    size_t base = (size_t)blockIdx.x * kScanTile + (size_t)threadIdx.x * kScanPerThread;
    uint32_t v[kScanPerThread];
    uint32_t local = 0;
#pragma unroll
    for (int k = 0; k < kScanPerThread; k++) {
        v[k] = (base + k < n) ? in[base + k] : 0u;
        local += v[k];
    }
    uint32_t inc = wave_inclusive_scan(local);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 63) s_wave[wave] = inc;
    __syncthreads();
    uint32_t wave_off = 0;
    for (int w = 0; w < wave; w++) wave_off += s_wave[w];
    uint32_t run = wave_off + inc - local;
#pragma unroll
    for (int k = 0; k < kScanPerThread; k++) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
    if (sums && threadIdx.x == kScanThreads - 1) sums[blockIdx.x] = run;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_add(uint32_t *out, size_t n, const uint32_t *offs) {
    size_t base = (size_t)blockIdx.x * kScanTile;
    uint32_t o = offs[blockIdx.x];
    for (int k = threadIdx.x; k < kScanTile; k += kScanThreads)
        if (base + k < n) out[base + k] += o;
}

static int scan_level(const uint32_t *in, uint32_t *out, size_t n, hipStream_t stream, ScanTemp &tmp, int lvl,
                      uint64_t &launches, std::string &err) {
    size_t blocks = (n + kScanTile - 1) / kScanTile;
    if (blocks <= 1) {
        hipLaunchKernelGGL(k_scan_tile, dim3(1), dim3(kScanThreads), 0, stream, in, out, n, (uint32_t *)nullptr);
        launches++;
        return BD_OK;
    }
    if (lvl >= 4) {
        err = "scan too large";
        return BD_ERR_CAPACITY;
    }
    BD_HIP(tmp.level[lvl].alloc(blocks));
    hipLaunchKernelGGL(k_scan_tile, dim3((unsigned)blocks), dim3(kScanThreads), 0, stream, in, out, n, tmp.level[lvl].p);
    launches++;
    int rc = scan_level(tmp.level[lvl].p, tmp.level[lvl].p, blocks, stream, tmp, lvl + 1, launches, err);
    if (rc) return rc;
    hipLaunchKernelGGL(k_scan_add, dim3((unsigned)blocks), dim3(kScanThreads), 0, stream, out, n, tmp.level[lvl].p);
    launches++;
    return BD_OK;
}

int exclusive_scan_u32(const uint32_t *in, uint32_t *out, size_t n, hipStream_t stream, ScanTemp &tmp,
                       uint64_t &launches, std::string &err) {
    if (!n) return BD_OK;
    return scan_level(in, out, n, stream, tmp, 0, launches, err);
}

}  // namespace bd

extern "C" int32_t bd_ext_copy_calibration(uint64_t bytes, float *ms) {
    if (bytes < 16 || (bytes & 15)) return BD_ERR_ARG;
    int n_dev = 0;
    if (hipGetDeviceCount(&n_dev) != hipSuccess || n_dev < 1) return BD_ERR_NODEVICE;
    void *src = nullptr, *dst = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int32_t rc = BD_OK;
    if (hipMalloc(&src, bytes) != hipSuccess || hipMalloc(&dst, bytes) != hipSuccess) rc = BD_ERR_NOMEM;
    if (rc == BD_OK && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)) rc = BD_ERR_DEVICE;
    if (rc == BD_OK) {
        const size_t n = bytes / 16;
        bd::launch_fill_u32((uint32_t *)src, bytes / 4, 0x3f800000u, nullptr);
        // one float4 per lane (the grid-stride loop only matters past 2^28 bytes)
        const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, (size_t)1 << 20);
        float t = 0.0f;
        if (hipEventRecord(e0, nullptr) != hipSuccess) rc = BD_ERR_DEVICE;
        if (rc == BD_OK) hipLaunchKernelGGL(bd::k_copy_f4, dim3(blocks), dim3(256), 0, nullptr,
                                            (const float4 *)src, (float4 *)dst, n);
        if (rc == BD_OK && (hipGetLastError() != hipSuccess || hipEventRecord(e1, nullptr) != hipSuccess ||
                            hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&t, e0, e1) != hipSuccess))
            rc = BD_ERR_DEVICE;
        if (ms) *ms = t;
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (src) (void)hipFree(src);
    if (dst) (void)hipFree(dst);
    return rc;
}
