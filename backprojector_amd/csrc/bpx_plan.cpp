// Plans: validation, structure detection, device staging and execution of one capture.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <limits>
#include <map>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>

#include "bpx_host.hpp"

namespace bpx {

// ------------------------------------------------------------------ device buffers
namespace {
struct PooledBlock {
    void* ptr;
    size_t cap;
    int device;
    uint64_t tick;   // of its release
};
// Never destroyed: plans may outlive this library's static objects.
struct Pool {
    std::mutex mutex;
    std::vector<PooledBlock> blocks;   // oldest release first
    size_t bytes = 0;
    uint64_t ticks = 0;                // allocations so far
    std::vector<std::pair<int, hipStream_t>> streams;
    std::vector<char*> slabs;
};
Pool& pool() {
    static Pool* p = new Pool;
    return *p;
}
int current_device() {
    int d = -1;
    return hipGetDevice(&d) == hipSuccess ? d : -1;
}

// Block sizes: multiples of 256 bytes up to 64 KiB, then of an eighth of the power of two below.
size_t block_size(size_t n) {
    size_t step = 256;
    if (n > (64u << 10)) {
        size_t p = 64u << 10;
        while (p <= n / 2) p *= 2;
        step = p / 8;
    }
    return (n + step - 1) / step * step;
}
// Takes the oldest blocks out until at most `room` bytes are kept and none has lain unused for
// kPooledTicks allocations; the caller frees them outside the lock.
std::vector<void*> evict(Pool& p, size_t room) {
    std::vector<void*> out;
    out.reserve(p.blocks.size());   // nothing below throws: the list and its total stay in step
    size_t n = 0;
    while (n < p.blocks.size() && (p.bytes > room || p.ticks - p.blocks[n].tick > kPooledTicks)) {
        out.push_back(p.blocks[n].ptr);
        p.bytes -= p.blocks[n].cap;
        ++n;
    }
    p.blocks.erase(p.blocks.begin(), p.blocks.begin() + (ptrdiff_t)n);
    return out;
}
}  // namespace

void DeviceBuffer::alloc(size_t n) {
    if (!try_alloc(n))
        fail(BPX_ERR_OUT_OF_MEMORY, "hipMalloc(" + std::to_string(n) + " bytes) failed: " +
                                        hipGetErrorString(hipErrorOutOfMemory));
}
bool DeviceBuffer::try_alloc(size_t n) {
    release();
    if (n == 0) n = 256;
    size_t want = block_size(n);
    Pool& p = pool();
    device = current_device();
    {
        std::lock_guard<std::mutex> lock(p.mutex);
        ++p.ticks;
        size_t best = p.blocks.size();
        for (size_t i = 0; i < p.blocks.size(); ++i)
            if (p.blocks[i].device == device && p.blocks[i].cap >= want && p.blocks[i].cap <= want + want / 4 &&
                (best == p.blocks.size() || p.blocks[i].cap < p.blocks[best].cap))
                best = i;
        if (best < p.blocks.size()) {
            ptr = p.blocks[best].ptr;
            cap = p.blocks[best].cap;
            p.bytes -= cap;
            p.blocks.erase(p.blocks.begin() + (ptrdiff_t)best);
        }
    }
    if (!ptr) {
        hipError_t e = hipMalloc(&ptr, want);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            std::vector<void*> all;
            {
                std::lock_guard<std::mutex> lock(p.mutex);
                all = evict(p, 0);
            }
            for (void* b : all) (void)hipFree(b);
            e = hipMalloc(&ptr, want);
            if (e == hipErrorOutOfMemory) {   // without the rounding for reuse
                (void)hipGetLastError();
                want = (n + 255u) / 256u * 256u;
                e = hipMalloc(&ptr, want);
            }
        }
        if (e != hipSuccess) {
            ptr = nullptr;
            (void)hipGetLastError();   // or the next launch would report it
            if (e == hipErrorOutOfMemory) return false;
            fail(BPX_ERR_OUT_OF_MEMORY, "hipMalloc(" + std::to_string(n) + " bytes) failed: " + hipGetErrorString(e));
        }
        cap = want;
    }
    bytes = n;
    return true;
}
void DeviceBuffer::release() {
    if (ptr) {
        bool kept = false;
        std::vector<void*> drop;
        if (cap <= kPooledBytes / 2 && device >= 0 && current_device() == device && hipDeviceSynchronize() == hipSuccess) {
            try {
                Pool& p = pool();
                std::lock_guard<std::mutex> lock(p.mutex);
                drop = evict(p, kPooledBytes - cap);
                p.blocks.push_back({ptr, cap, device, p.ticks});
                p.bytes += cap;
                kept = true;
            } catch (const std::bad_alloc&) {   // no host memory for the list: free it below
            }
        }
        if (!kept) (void)hipFree(ptr);
        for (void* d : drop) (void)hipFree(d);
    }
    ptr = nullptr;
    bytes = cap = 0;
}

size_t release_pooled() {
    Pool& p = pool();
    std::vector<void*> all;
    size_t bytes = 0;
    {
        std::lock_guard<std::mutex> lock(p.mutex);
        bytes = p.bytes;
        all = evict(p, 0);
    }
    for (void* b : all) (void)hipFree(b);
    return bytes;
}

hipStream_t take_stream() {
    const int device = current_device();
    {
        Pool& p = pool();
        std::lock_guard<std::mutex> lock(p.mutex);
        for (size_t i = p.streams.size(); i-- > 0;)
            if (p.streams[i].first == device) {
                const hipStream_t s = p.streams[i].second;
                p.streams.erase(p.streams.begin() + (ptrdiff_t)i);
                return s;
            }
    }
    hipStream_t s = nullptr;
    hip_check(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreate");
    return s;
}
void give_stream(hipStream_t s) {
    hipDevice_t device = -1;
    if (hipStreamGetDevice(s, &device) == hipSuccess && hipStreamSynchronize(s) == hipSuccess) {
        Pool& p = pool();
        std::lock_guard<std::mutex> lock(p.mutex);
        if (p.streams.size() < 8) {
            try {
                p.streams.emplace_back((int)device, s);
                return;
            } catch (const std::bad_alloc&) {
            }
        }
    }
    (void)hipStreamDestroy(s);
}

PlanImpl::~PlanImpl() {
    oct.reset();   // its events were recorded on `stream`: before that is given back
    for (auto& e : ev)
        if (e) (void)hipEventDestroy(e);
    if (done) (void)hipEventDestroy(done);
    if (ready) (void)hipEventDestroy(ready);
    if (stream) give_stream(stream);
}

static uint32_t round_up(uint64_t x, uint32_t m) { return (uint32_t)((x + m - 1) / m * m); }

static bool finite_pair(const bpx_pair& p) {
    for (int k = 0; k < 3; ++k)
        if (!std::isfinite(p.camera_point[k]) || !std::isfinite(p.laser_point[k])) return false;
    return std::isfinite(p.camera_wall) && std::isfinite(p.laser_wall);
}

static bool same3(const float* a, const float* b) { return std::memcmp(a, b, 12) == 0; }

// Bound on |approximate quotient - exact quotient| of the table lookup.  The approximation
// q1 = fma(d', 2/dT, c1) (confocal) or fma(t, 1/dT, c1) differs from the exact fp32 chain
// (<= 3 rounded adds, 1 sqrt of <= 2 ulp error in the hardware sqrt, 1 rounded subtract,
// 1 rounded division) by a few units of 2^-24 times the magnitudes involved; 16 * 2^-24 * Q
// with Q = (max |total| + |t0|)/dT + Tc + 2 covers every term with a wide margin.
static double tap_error_bound(double max_total, double t0, double dT, double Tc) {
    const double Q = (std::fabs(max_total) + std::fabs(t0)) / dT + Tc + 2.0;
    return 16.0 * std::ldexp(1.0, -24) * Q;
}

static double dist3(const float* a, const double* b) {
    const double x = a[0] - b[0], y = a[1] - b[1], z = a[2] - b[2];
    return std::sqrt(x * x + y * y + z * z);
}

// Voxel-grid corners of the A.1 grid (convex hull of all voxel positions).
static void grid_corners(const uint32_t n[3], const float zero[3], const float inc[9],
                         double corners[8][3]) {
    for (int m = 0; m < 8; ++m) {
        const double i[3] = {(m & 4) ? (double)(n[0] - 1) : 0.0, (m & 2) ? (double)(n[1] - 1) : 0.0,
                             (m & 1) ? (double)(n[2] - 1) : 0.0};
        for (int k = 0; k < 3; ++k)
            corners[m][k] = (double)zero[k] + inc[k] * i[0] + inc[3 + k] * i[1] + inc[6 + k] * i[2];
    }
}

// Per-pair element windows [lo, hi) of a fused confocal row (lde elements): every element a
// gather kernel can read for the pair and any voxel of the grid.  A voxel's distance d to the
// wall point lies between the distances to the nearest and farthest points of the corners'
// bounding box, the box widened by 1e-5 of the largest coordinate and the distances by a
// relative 1e-5 (the kernels' fp32 coordinates and squared distances are a few ulps off the
// exact ones); its bin is round((lw + 2 d + cw - t0) / deltaT) over that range, and the
// kernels read element bin + 1 and its neighbours (the two candidate bins of the approximate
// quotient, the second sample of a 16-bit element), so 4 elements of slack below and 5 above
// cover every read.  Bins before the row or past its end clamp to its ends (elements 0 and
// Tc, Tc + 1), so a window reaching past an end keeps that end's first 6 / last 6 elements,
// also when the whole window lies beyond it.
static std::vector<uint32_t> row_windows(const std::vector<bpx_pair>& pr, const double corners[8][3], double t0,
                                         double dT, uint32_t Tc, uint32_t lde) {
    double lo[3], hi[3], scale = 1.0;
    for (int k = 0; k < 3; ++k) lo[k] = hi[k] = corners[0][k];
    for (int m = 0; m < 8; ++m)
        for (int k = 0; k < 3; ++k) {
            lo[k] = std::min(lo[k], corners[m][k]);
            hi[k] = std::max(hi[k], corners[m][k]);
            scale = std::max(scale, std::fabs(corners[m][k]));
        }
    for (const auto& p : pr)
        for (int k = 0; k < 3; ++k) scale = std::max(scale, std::fabs((double)p.laser_point[k]));
    for (int k = 0; k < 3; ++k) {
        lo[k] -= 1e-5 * scale;
        hi[k] += 1e-5 * scale;
    }
    std::vector<uint32_t> w(2 * pr.size());
    for (size_t p = 0; p < pr.size(); ++p) {
        double near2 = 0.0, far2 = 0.0;
        for (int k = 0; k < 3; ++k) {
            const double x = pr[p].laser_point[k];
            const double c = x < lo[k] ? lo[k] - x : x > hi[k] ? x - hi[k] : 0.0;
            const double f = std::max(std::fabs(x - lo[k]), std::fabs(x - hi[k]));
            near2 += c * c;
            far2 += f * f;
        }
        const double base = (double)pr[p].laser_wall + (double)pr[p].camera_wall - t0;
        const double qlo = (base + 2.0 * std::sqrt(near2) * (1.0 - 1e-5)) / dT;
        const double qhi = (base + 2.0 * std::sqrt(far2) * (1.0 + 1e-5)) / dT;
        double elo = std::floor(qlo) + 1.0 - 4.0, ehi = std::ceil(qhi) + 1.0 + 5.0;
        if (!std::isfinite(elo) || !std::isfinite(ehi)) elo = 0.0, ehi = (double)lde;
        w[2 * p] = (uint32_t)std::clamp(elo, 0.0, (double)(Tc >= 4u ? Tc - 4u : 0u));
        w[2 * p + 1] = (uint32_t)std::clamp(ehi, (double)std::min(lde, 6u), (double)lde);
    }
    return w;
}

std::vector<uint32_t> confocal_row_windows(const bpx_pair* pairs, uint32_t P, const uint32_t n[3],
                                           const float zero[3], const float inc[9], float t0, float dT,
                                           uint32_t Tc) {
    double corners[8][3];
    grid_corners(n, zero, inc, corners);
    return row_windows(std::vector<bpx_pair>(pairs, pairs + P), corners, t0, dT, Tc, round_up((uint64_t)Tc + 2, 16));
}

static double max_total_path(const bpx_pair* pr, size_t count, const double corners[8][3]) {
    double mx = 0.0;
    for (size_t i = 0; i < count; ++i) {
        const bpx_pair& p = pr[i];
        double dl = 0, dc = 0;
        for (int m = 0; m < 8; ++m) {
            dl = std::max(dl, dist3(p.laser_point, corners[m]));
            dc = std::max(dc, dist3(p.camera_point, corners[m]));
        }
        mx = std::max(mx, std::fabs((double)p.laser_wall) + std::fabs((double)p.camera_wall) + dl + dc);
    }
    return mx;
}

double single_tap_error_bound(const bpx_pair* pairs, uint32_t P, const uint32_t n[3], const float zero[3],
                              const float inc[9], float t0, float dT, uint32_t T) {
    double corners[8][3];
    grid_corners(n, zero, inc, corners);
    return tap_error_bound(max_total_path(pairs, P, corners), t0, dT, T);
}

// Power-of-two scale s so that max|x| / s lies in [2^14, 2^15) (exact rescaling).
// Largest |sample| of the chunk (host chunk, or the copied windows of the source rows).
static float chunk_max_abs(const CaptureIn& c) {
    float m = 0.0f;
    if (c.chunk) {
        const uint64_t n = c.size * (c.cplx ? 2 : 1);
        for (uint64_t i = 0; i < n; ++i) m = std::max(m, std::fabs(c.chunk[i]));
    } else if (c.device_rows) {
        const uint64_t n = c.size * (c.cplx ? 2 : 1);
        DeviceBuffer r;
        r.alloc(sizeof(float));
        hip_check(hipMemset(r.ptr, 0, sizeof(float)), "hipMemset");
        hip_check(launch_abs_max(static_cast<const float*>(c.device_rows->ptr), n, static_cast<float*>(r.ptr),
                                 nullptr),
                  "abs max kernel");
        hip_check(hipMemcpy(&m, r.ptr, sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy");
    } else if (c.src) {
        for (uint32_t p = 0; p < c.P; ++p) {
            const float* r = c.src + (size_t)p * c.src_T + c.from;
            for (uint32_t i = 0; i < c.ncopy; ++i) m = std::max(m, std::fabs(r[i]));
        }
    }
    return m;
}

static float choose_scale(const CaptureIn& c) {
    const float m = chunk_max_abs(c);
    if (!(m > 0.0f) || !std::isfinite(m)) return 1.0f;
    int e;
    std::frexp(m, &e);  // m in [2^(e-1), 2^e)
    return std::ldexp(1.0f, e - 1 - 14);
}

static void validate_common(const CaptureIn& c, const uint32_t n[3]) {
    if (!c.chunk && !c.src && !c.device_rows && c.size) fail(BPX_ERR_INVALID_ARGUMENT, "transient_chunk is NULL");
    if (c.device_rows && c.device_rows->bytes < sizeof(float) * c.size * (c.cplx ? 2 : 1))
        fail(BPX_ERR_INVALID_ARGUMENT, "device rows smaller than the chunk");
    if (!c.chunk && c.src) {
        if (c.cplx) fail(BPX_ERR_INVALID_ARGUMENT, "device cropping takes real samples");
        if ((uint64_t)c.from + c.ncopy > c.src_T || (uint64_t)c.cfrom + c.ncopy > c.T)
            fail(BPX_ERR_INVALID_ARGUMENT, "crop window outside the source or chunk rows");
    }
    if (!c.pairs && c.P) fail(BPX_ERR_INVALID_ARGUMENT, "scanned_pairs is NULL");
    if (c.T == 0) fail(BPX_ERR_INVALID_ARGUMENT, "T must be > 0");
    if ((uint64_t)c.P * c.T != c.size)
        fail(BPX_ERR_INVALID_ARGUMENT, "transient_size (" + std::to_string(c.size) +
                                           ") != num_pairs * T (" +
                                           std::to_string((uint64_t)c.P * c.T) + ")");
    if (!std::isfinite(c.t0)) fail(BPX_ERR_INVALID_ARGUMENT, "t0 must be finite");
    if (!(c.dT > 0.0f) || !std::isfinite(c.dT) || !std::isfinite(1.0f / c.dT) ||
        c.dT < std::numeric_limits<float>::min())
        fail(BPX_ERR_INVALID_ARGUMENT, "deltaT must be a positive normal float");
    for (int k = 0; k < 3; ++k)
        if (n[k] == 0) fail(BPX_ERR_INVALID_ARGUMENT, "voxels_per_side must be > 0");
    if ((uint64_t)n[0] * n[1] * n[2] > (1ull << 32))
        fail(BPX_ERR_UNSUPPORTED, "volumes above 2^32 voxels are not supported");
    if (c.T > (1u << 22)) fail(BPX_ERR_UNSUPPORTED, "T above 2^22 bins is not supported");
}

// Pairs that take part: finite ones, minus the reference launcher's dropped tail if asked.
static std::vector<uint32_t> used_pairs(const CaptureIn& c, uint32_t flags) {
    uint32_t P = c.P;
    if (flags & BPX_FLAG_REFERENCE_PAIR_TRUNCATION) {
        const uint32_t B = std::min<uint32_t>(256u, std::max<uint32_t>(P, 1u));
        P = (P / B) * B;
    }
    std::vector<uint32_t> idx;
    idx.reserve(P);
    for (uint32_t p = 0; p < P; ++p)
        if (finite_pair(c.pairs[p])) idx.push_back(p);
    return idx;
}

// ------------------------------------------------------------------ host -> device uploads
// Large pageable host arrays go through pinned chunks (allocated once per process): host threads
// copy chunks in or out while the DMA engine works on others.  Measured on MI355X: pageable
// hipMemcpy ~30 GB/s in and, into fresh pages, 4 to 9 GB/s out; pinned ~57 GB/s; 4 host threads
// copy into pinned memory at ~60 GB/s, 8 write fresh pages at 16 (one: 3.6).
namespace {
constexpr size_t kRingChunk = 2u << 20;
constexpr size_t kRingBytes = 32u << 20;
constexpr size_t kStagedDown = 16u << 20;   // from here on an array goes through the ring
constexpr size_t kStagedUp = 64u << 20;
// One a direction, so that neither waits for the other's transfers; used by whoever holds the mutex.
struct Ring {
    struct Events {
        hipEvent_t of[kRingBytes / kRingChunk] = {};
    };
    std::mutex mutex;
    char* at = nullptr;
    std::map<int, Events> events;
    // The chunks and the current device's events (an event can be recorded on its own device alone).
    hipEvent_t* ensure() {
        if (!at) {
            void* p = nullptr;
            hip_check(hipHostMalloc(&p, kRingBytes, hipHostMallocDefault), "hipHostMalloc");
            at = static_cast<char*>(p);
        }
        Events& ev = events[current_device()];
        for (auto& e : ev.of)
            if (!e) hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
        return ev.of;
    }
};
Ring &g_up = *new Ring, &g_down = *new Ring;   // never destroyed, as the pool

// f(chunk, offset, bytes) for every chunk of an array, on up to `most` threads that take the chunks
// in turn; the first error any of them met.
template <class F>
hipError_t for_chunks(size_t bytes, uint32_t most, F&& f) {
    const uint32_t chunks = (uint32_t)((bytes + kRingChunk - 1) / kRingChunk);
    const uint32_t n = std::min({most, (chunks + 1u) / 2u, std::max(1u, std::thread::hardware_concurrency() / 2u)});
    const int device = current_device();
    std::atomic<uint32_t> next{0};
    std::atomic<int> error{(int)hipSuccess};
    auto work = [&](bool own) {
        if (!own && device >= 0) (void)hipSetDevice(device);
        for (;;) {
            const uint32_t k = next.fetch_add(1);
            if (k >= chunks || error.load() != (int)hipSuccess) break;
            const size_t off = (size_t)k * kRingChunk;
            const hipError_t e = f(k, off, std::min(kRingChunk, bytes - off));
            if (e != hipSuccess) error.store((int)e);
        }
    };
    std::vector<std::thread> th;
    th.reserve(n);
    try {
        for (uint32_t t = 1; t < n; ++t) th.emplace_back(work, false);
    } catch (const std::exception&) {   // no further thread to be had: those that started, and this one
    }
    work(true);
    for (auto& x : th) x.join();
    return (hipError_t)error.load();
}
}  // namespace

// Memory that the copy engine reaches by itself (pinned, managed, on a device): it goes in one copy.
// 128 MiB into a pinned volume: 2.36 ms, through the ring 3.75.
static bool direct_memory(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();   // ordinary host memory
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

void upload_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes < kStagedUp || direct_memory(src)) {
        hip_check(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice), "hipMemcpy(upload)");
        return;
    }
    std::lock_guard<std::mutex> lock(g_up.mutex);
    hipEvent_t* const events = g_up.ensure();
    // The ring in two halves: threads fill one while the other one's copies run.
    constexpr size_t half = kRingBytes / 2;
    hipError_t e = hipSuccess;
    uint32_t round = 0;
    for (size_t base = 0; base < bytes && e == hipSuccess; base += half, ++round) {
        char* at = g_up.at + (round & 1u) * half;
        hipEvent_t ev = events[round & 1u];
        if (round >= 2) e = hipEventSynchronize(ev);   // this half's previous copies are done
        if (e == hipSuccess)
            e = for_chunks(std::min(half, bytes - base), 4, [&](uint32_t, size_t off, size_t n) {
                std::memcpy(at + off, static_cast<const char*>(src) + base + off, n);
                return hipMemcpyAsync(static_cast<char*>(dst) + base + off, at + off, n, hipMemcpyHostToDevice, s);
            });
        if (e == hipSuccess) e = hipEventRecord(ev, s);
    }
    const hipError_t done = hipStreamSynchronize(s);   // the ring may be reused as soon as this returns
    hip_check(e, "upload");
    hip_check(done, "hipStreamSynchronize");
}

void download_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes < kStagedDown || direct_memory(dst)) {
        hip_check(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s), "hipMemcpyAsync(download)");
        hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
        return;
    }
    hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");   // other transfers may use the ring meanwhile
    std::lock_guard<std::mutex> lock(g_down.mutex);
    hipEvent_t* const events = g_down.ensure();
    for (size_t base = 0; base < bytes; base += kRingBytes) {
        const size_t part = std::min(bytes - base, kRingBytes);
        const char* from = static_cast<const char*>(src) + base;
        char* to = static_cast<char*>(dst) + base;
        hipError_t e = hipSuccess;
        for (size_t off = 0, b = 0; off < part && e == hipSuccess; off += kRingChunk, ++b) {
            e = hipMemcpyAsync(g_down.at + off, from + off, std::min(kRingChunk, part - off), hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(events[b], s);
        }
        if (e == hipSuccess)
            e = for_chunks(part, 8, [&](uint32_t k, size_t off, size_t n) {
                const hipError_t w = hipEventSynchronize(events[k]);
                if (w == hipSuccess) std::memcpy(to + off, g_down.at + off, n);
                return w;
            });
        const hipError_t done = hipStreamSynchronize(s);
        hip_check(e, "download");
        hip_check(done, "hipStreamSynchronize");
    }
}

namespace {
constexpr size_t kSlabBytes = 1u << 20;
}
void TableUploads::add(void* dst, const void* src, size_t bytes) {
    if (bytes == 0) return;
    if (bytes > kSlabBytes) {
        hip_check(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice), "hipMemcpy(table)");
        return;
    }
    if (!slab) {
        Pool& p = pool();
        std::lock_guard<std::mutex> lock(p.mutex);
        if (!p.slabs.empty()) {
            slab = p.slabs.back();
            p.slabs.pop_back();
        }
    }
    if (!slab) {
        void* m = nullptr;
        hip_check(hipHostMalloc(&m, kSlabBytes, hipHostMallocDefault), "hipHostMalloc");
        slab = static_cast<char*>(m);
    }
    if (used + bytes > kSlabBytes) {
        hip_check(hipStreamSynchronize(stream), "hipStreamSynchronize");
        used = 0;
    }
    std::memcpy(slab + used, src, bytes);
    hip_check(hipMemcpyAsync(dst, slab + used, bytes, hipMemcpyHostToDevice, stream), "hipMemcpyAsync(table)");
    used += (bytes + 255u) & ~(size_t)255u;
}
void TableUploads::finish() {
    const hipError_t e = hipStreamSynchronize(stream);
    open = false;
    hip_check(e, "hipStreamSynchronize");
}
TableUploads::~TableUploads() {
    if (open) (void)hipStreamSynchronize(stream);   // left by an exception
    if (!slab) return;
    try {
        Pool& p = pool();
        std::lock_guard<std::mutex> lock(p.mutex);
        if (p.slabs.size() < 4) {
            p.slabs.push_back(slab);
            return;
        }
    } catch (const std::bad_alloc&) {
    }
    (void)hipHostFree(slab);
}

// Stages the raw rows of the used pairs on the device (compacting when pairs were dropped).
// Device rows [rows_in][row floats] -> the plan's raw rows of the used pairs: taken over when
// every row is used, else gathered.
static void adopt_device_rows(PlanImpl& pl, DeviceBuffer& rows, uint32_t rows_in, size_t row,
                              const std::vector<uint32_t>& idx) {
    if (idx.size() == rows_in && rows_in) {
        pl.raw.release();
        pl.raw.swap(rows);
        return;
    }
    pl.raw.alloc(sizeof(float) * row * std::max<size_t>(idx.size(), 1));
    if (idx.empty()) return;
    DeviceBuffer map;
    map.alloc(sizeof(uint32_t) * idx.size());
    hip_check(hipMemcpy(map.ptr, idx.data(), sizeof(uint32_t) * idx.size(), hipMemcpyHostToDevice),
              "hipMemcpy(row map)");
    hip_check(launch_crop_rows(static_cast<const float*>(rows.ptr), (uint32_t)row, static_cast<const uint32_t*>(map.ptr),
                               (uint32_t)idx.size(), (uint32_t)row, 0u, 0u, (uint32_t)row,
                               static_cast<float*>(pl.raw.ptr), pl.stream),
              "row gather kernel");
    hip_check(hipStreamSynchronize(pl.stream), "hipStreamSynchronize");
}

void plan_replace_rows(PlanImpl& pl, DeviceBuffer& rows) {
    if (pl.path == kPathOctree) fail(BPX_ERR_UNSUPPORTED, "octree plans keep their rows");
    if (pl.P == 0 || !pl.raw.ptr) return;   // nothing staged: every execution writes zeros
    const size_t row = (size_t)pl.T * (pl.cplx ? 2 : 1);
    if (rows.bytes < sizeof(float) * row * pl.rows_in) fail(BPX_ERR_INVALID_ARGUMENT, "replacement rows too small");
    plan_wait(pl);
    adopt_device_rows(pl, rows, pl.rows_in, row, pl.used);
    if (pl.stage.ptr) {   // the staging descriptor names the raw rows: point it at the new ones
        const StageJob job = stage_job(pl);
        hip_check(hipMemcpy(pl.stage.ptr, &job, sizeof(StageJob), hipMemcpyHostToDevice), "hipMemcpy(staging job)");
    }
}

static void stage_raw(PlanImpl& pl, const CaptureIn& c, const std::vector<uint32_t>& idx) {
    const size_t comp = c.cplx ? 2 : 1;
    const size_t row = (size_t)c.T * comp;
    pl.used = idx;
    pl.rows_in = c.P;
    if (!c.chunk && c.device_rows) {
        adopt_device_rows(pl, *c.device_rows, c.P, row, idx);
        return;
    }
    pl.raw.alloc(sizeof(float) * row * std::max<size_t>(idx.size(), 1));
    if (!c.chunk) {
        if (idx.empty()) return;
        if (idx.size() == c.P && c.from == 0 && c.cfrom == 0 && c.ncopy == c.T && c.src_T == c.T) {
            upload_host(pl.raw.ptr, c.src, sizeof(float) * row * c.P, pl.stream);
            return;
        }
        // the source rows in one copy, then the crop (and compaction of dropped pairs) on the device
        DeviceBuffer full, map;
        full.alloc(sizeof(float) * (size_t)c.P * c.src_T);
        map.alloc(sizeof(uint32_t) * idx.size());
        upload_host(full.ptr, c.src, sizeof(float) * (size_t)c.P * c.src_T, pl.stream);
        hip_check(hipMemcpy(map.ptr, idx.data(), sizeof(uint32_t) * idx.size(), hipMemcpyHostToDevice),
                  "hipMemcpy(row map)");
        hip_check(launch_crop_rows(static_cast<const float*>(full.ptr), c.src_T,
                                   static_cast<const uint32_t*>(map.ptr), (uint32_t)idx.size(), c.T, c.from,
                                   c.cfrom, c.ncopy, static_cast<float*>(pl.raw.ptr), pl.stream),
                  "crop kernel");
        hip_check(hipStreamSynchronize(pl.stream), "hipStreamSynchronize");
        return;
    }
    if (idx.size() == c.P) {
        upload_host(pl.raw.ptr, c.chunk, sizeof(float) * row * c.P, pl.stream);
    } else {
        std::vector<float> tmp(row * idx.size());
        for (size_t i = 0; i < idx.size(); ++i)
            std::memcpy(&tmp[i * row], c.chunk + (size_t)idx[i] * row, sizeof(float) * row);
        if (!tmp.empty())
            hip_check(hipMemcpy(pl.raw.ptr, tmp.data(), sizeof(float) * tmp.size(),
                                hipMemcpyHostToDevice),
                      "hipMemcpy(transient)");
    }
}

static void make_events(PlanImpl& pl) {
    for (auto& e : pl.ev) hip_check(hipEventCreate(&e), "hipEventCreate");
    hip_check(hipEventCreateWithFlags(&pl.done, hipEventDisableTiming), "hipEventCreate");
    hip_check(hipEventCreateWithFlags(&pl.ready, hipEventDisableTiming), "hipEventCreate");
}

void plan_wait(const PlanImpl& pl) {
    hip_check(hipStreamSynchronize(pl.stream), "hipStreamSynchronize");
}

// Exhaustive-grid structure: p = l*C + c with laser data depending only on l and camera
// data only on c.  Returns C (0 when the list is not such a product).
static uint32_t grid_structure(const std::vector<bpx_pair>& pr) {
    const uint32_t P = (uint32_t)pr.size();
    if (P < 2) return 0;
    uint32_t C = 1;
    while (C < P && same3(pr[C].laser_point, pr[0].laser_point) &&
           pr[C].laser_wall == pr[0].laser_wall)
        ++C;
    if (C == P || P % C != 0 || C < 2) return 0;
    for (uint32_t p = 0; p < P; ++p) {
        const uint32_t l = p / C, c = p % C;
        const bpx_pair& a = pr[p];
        const bpx_pair& lb = pr[(size_t)l * C];
        const bpx_pair& cb = pr[c];
        if (!same3(a.laser_point, lb.laser_point) || a.laser_wall != lb.laser_wall) return 0;
        if (!same3(a.camera_point, cb.camera_point) || a.camera_wall != cb.camera_wall) return 0;
    }
    return C;
}

// The LDS-staged kernel of non-confocal captures where it applies: real samples, voxels of a column
// sharing x and y, points clear of the volume (its roots' range), windows that fit beside the
// threshold table.  Tiles are 16 x 16 x 8.
static void paths_lds_setup(PlanImpl& pl, const std::vector<bpx_pair>& pr, const double corners[8][3]) {
    const Grid& g = pl.g;
    if (pl.cplx || g.inc[6] != 0.0f || g.inc[7] != 0.0f || g.n[2] < 8u || pl.T + 1u > 16384u) return;
    double lo[3], hi[3];
    for (int k = 0; k < 3; ++k) {
        lo[k] = hi[k] = corners[0][k];
        for (int m = 1; m < 8; ++m) {
            lo[k] = std::min(lo[k], corners[m][k]);
            hi[k] = std::max(hi[k], corners[m][k]);
        }
        const double slack = 1e-5 * std::max(std::fabs(lo[k]), std::fabs(hi[k]));
        lo[k] -= slack;
        hi[k] += slack;
    }
    // distance of a point from the volume's box; a point inside it may be at distance 0 of a voxel
    const auto clear = [&](const float* p) {
        double d = 0.0;
        for (int k = 0; k < 3; ++k) {
            const double e = std::max({lo[k] - (double)p[k], (double)p[k] - hi[k], 0.0});
            d = std::max(d, e);
        }
        return d > 1e-9;
    };
    for (const auto& p : pr)
        if (!clear(p.laser_point) || !clear(p.camera_point)) return;
    if (!(pl.max_path < 1e9)) return;
    double d2 = 0.0;
    for (int k = 0; k < 3; ++k) {
        const double r = 15.0 * (std::fabs((double)g.inc[k]) + std::fabs((double)g.inc[3 + k])) + 7.0 * std::fabs((double)g.inc[6 + k]);
        d2 += r * r;
    }
    const double need = std::ceil(2.0 * std::sqrt(d2) / (double)pl.dT * (1.0 + 1e-6)) + 14.0;
    if (!(need <= 2048.0)) return;
    PathsLdsArgs a{};
    a.seg = round_up((uint64_t)need, 256);
    a.Tc = pl.T;
    if (paths_lds_bytes(a) > 160u * 1024u) return;
    a.L = pl.L;
    a.C = pl.C;
    a.P = pl.P;
    a.g = g;
    // blocks of 8 pairs (a stage) between compensated adds: the order of the sums differs from the
    // general kernels', and no sum should come out further from the exact one than theirs
    a.kahan_block = std::min<uint32_t>(pl.kahan_block, 8u);
    a.scale = pl.scale;
    // parts towards 2,048 work-groups of at least 8 lasers or 64 pairs, 64 MiB of partial sums
    const uint64_t tiles = (uint64_t)((g.n[0] + 15u) / 16u) * ((g.n[1] + 15u) / 16u) * ((g.n[2] + 7u) / 8u);
    const uint64_t vox = (uint64_t)g.n[0] * g.n[1] * g.n[2];
    const uint32_t units = pl.L ? pl.L : pl.P;
    uint64_t parts = std::min<uint64_t>((2048u + tiles - 1u) / tiles, units / (pl.L ? 8u : 64u));
    parts = std::max<uint64_t>(1u, std::min<uint64_t>(parts, (64ull << 20) / (8u * vox)));
    a.part_units = (uint32_t)((units + parts - 1u) / parts);
    pl.paths_parts = (units + a.part_units - 1u) / a.part_units;
    if (pl.paths_parts > 1) pl.parts.alloc((size_t)pl.paths_parts * vox * 8u);
    pl.paths = a;
}

// Default confocal kernel where the polynomial-quotient kernel does not apply: the LDS-staged one where
// it does (separable grid, flat wall, short bin windows) and has enough tiles to fill the GPU.  Real
// formats: 16^3 tiles of 256 lanes (16 voxels per lane) from 1,024 tiles, 16^3 tiles of 512 lanes (8
// per lane) from 512; else, and for complex formats, 16 x 16 x 8 tiles of 256 lanes from 512.
// Measured at 16,384 pairs (gather ms, the three shapes in that order, texture path last): 256^3
// 81.7 / 85.8 / 96.7 / 141; 128^3 16.1 / 12.8 / 14.4 / 20.0; 112^3 - / 13.2 / 12.1 / 19.4; 96^3 - / -
// / 10.2 / 10.0.
int default_variant(const PlanImpl& pl) {
    const uint32_t* n = pl.g.n;
    if (!pl.fused || !pl.sep || !pl.flat) return kDefaultVariant;
    const uint32_t seg = lds_seg_elems(pl.format);
    const uint64_t t16 = (uint64_t)((n[0] + 15) / 16) * ((n[1] + 15) / 16) * ((n[2] + 15) / 16);
    const uint64_t t8 = (uint64_t)((n[0] + 15) / 16) * ((n[1] + 15) / 16) * ((n[2] + 7) / 8);
    const bool cplx = pl.format == kCF16 || pl.format == kCBF16;   // two accumulators per voxel
    const bool fits16 = confocal_lds_fits(pl.g.inc, pl.inv2, 16, seg), fits8 = confocal_lds_fits(pl.g.inc, pl.inv2, 8, seg);
    if (!cplx && t16 >= kLdsDeepTiles && fits16) return kLdsVariant;
    if (!cplx && t16 >= kLdsMinTiles && fits16) return kLdsVariant + 2;
    return t8 >= kLdsMinTiles && fits8 ? kLdsVariant + 1 : kDefaultVariant;
}

PlanImpl* make_plan_single_tap(const CaptureIn& c, const uint32_t n[3], const float zero[3],
                               const float inc[9], const bpx_options* opt) {
    validate_common(c, n);
    for (int k = 0; k < 3; ++k)
        if (!std::isfinite(zero[k])) fail(BPX_ERR_INVALID_ARGUMENT, "volume_zero_pos must be finite");
    for (int k = 0; k < 9; ++k)
        if (!std::isfinite(inc[k])) fail(BPX_ERR_INVALID_ARGUMENT, "voxel_inc must be finite");
    if (!device_ready()) fail(BPX_ERR_NO_DEVICE, "no gfx950 device available");

    bpx_options o{BPX_STORAGE_F32, 32u, 0u, -1};
    if (opt) o = *opt;
    if (o.kahan_block == 0) o.kahan_block = 32;
    if (o.storage > BPX_STORAGE_BF16) fail(BPX_ERR_INVALID_ARGUMENT, "unknown storage format");
    if (o.variant >= variant_count()) fail(BPX_ERR_INVALID_ARGUMENT, "unknown kernel variant");

    auto pl = std::make_unique<PlanImpl>();
    pl->stream = take_stream();
    make_events(*pl);
    pl->cplx = c.cplx;
    pl->format = c.cplx ? (o.storage == BPX_STORAGE_F16 ? kCF16 : o.storage == BPX_STORAGE_BF16 ? kCBF16 : kC64)
                        : (o.storage == BPX_STORAGE_F16 ? kF16 : o.storage == BPX_STORAGE_BF16 ? kBF16 : kF32);
    pl->row_format = pl->format;
    pl->kahan_block = o.kahan_block;
    pl->t0 = c.t0;
    pl->dT = c.dT;
    pl->T = c.T;
    std::memcpy(pl->g.n, n, sizeof(uint32_t) * 3);
    std::memcpy(pl->g.zero, zero, sizeof(float) * 3);
    std::memcpy(pl->g.inc, inc, sizeof(float) * 9);

    const std::vector<uint32_t> idx = used_pairs(c, o.flags);
    std::vector<bpx_pair> pr(idx.size());
    for (size_t i = 0; i < idx.size(); ++i) pr[i] = c.pairs[idx[i]];
    pl->P = (uint32_t)pr.size();

    const size_t nvox = (size_t)n[0] * n[1] * n[2];
    pl->vol.alloc(nvox * (c.cplx ? 8 : 4));

    // structure
    bool confocal = !pr.empty();
    for (const auto& p : pr) confocal = confocal && same3(p.laser_point, p.camera_point);
    pl->C = confocal ? 0 : grid_structure(pr);
    pl->L = pl->C ? pl->P / pl->C : 0;
    pl->path = confocal ? kPathConfocal : (pl->C ? kPathGrid : kPathPairs);

    // exactness precondition of the table lookup
    double corners[8][3];
    grid_corners(n, zero, inc, corners);
    pl->max_path = max_total_path(pr.data(), pr.size(), corners);
    const double bound = tap_error_bound(pl->max_path, c.t0, c.dT, c.T);
    pl->tap_bound = bound;
    if (bound >= 0.25)
        fail(BPX_ERR_UNSUPPORTED,
             "path lengths / t0 too large relative to deltaT for the exact bin lookup (bound " +
                 std::to_string(bound) + ")");

    pl->variant = o.variant < 0 ? kDefaultVariant : o.variant;
    pl->fused = pl->path == kPathConfocal && variant_fused(pl->variant);
    pl->K = variant_k(pl->variant);
    if (pl->path == kPathPairs) pl->K = 4;
    if (pl->path == kPathGrid && pl->K == 8) pl->K = 4;
    pl->tiles = make_tiles(n, pl->K);

    if (pl->P == 0) return pl.release();

    // samples: raw rows resident on the device; scale for 16-bit storage
    pl->scale = (pl->format == kF32 || pl->format == kC64) ? 1.0f : choose_scale(c);
    stage_raw(*pl, c, idx);
    // padded rows (split) or the fused sample+threshold layout, [P][ldh] elements
    pl->ldh = round_up((uint64_t)c.T + 2, pl->fused ? 16 : 64);
    const uint64_t hbytes = (uint64_t)pl->P * pl->ldh *
                            (pl->fused ? fused_elem_bytes(pl->format) : format_bytes(pl->format));
    if (hbytes >= (1ull << 32)) fail(BPX_ERR_UNSUPPORTED, "transient rows above 4 GiB per plan");
    if (pl->path != kPathConfocal && o.variant < 0) paths_lds_setup(*pl, pr, corners);
    if (!pl->paths.seg) pl->H.alloc(hbytes);
    else if (pl->format != kF32) pl->H.alloc((size_t)pl->P * c.T * 4u);
    // fused rows staged over per-pair windows keep zeros outside them (written here only)
    if (pl->fused) hip_check(hipMemsetAsync(pl->H.ptr, 0, hbytes, pl->stream), "hipMemsetAsync(fused rows)");
    TableUploads tables(pl->stream);

    std::vector<float> p8((size_t)pl->P * 8);
    std::memcpy(p8.data(), pr.data(), sizeof(float) * p8.size());
    pl->pair8.alloc(sizeof(float) * p8.size());
    tables.add(pl->pair8.ptr, p8.data(), sizeof(float) * p8.size());

    if (pl->path == kPathConfocal) {
        pl->Z.alloc(sizeof(float) * ((size_t)c.T + 1));
        if (!pl->fused) {
            pl->lds = round_up((uint64_t)c.T + 1, 64);
            const uint64_t sbytes = (uint64_t)pl->P * pl->lds * 4;
            if (sbytes >= (1ull << 32)) fail(BPX_ERR_UNSUPPORTED, "threshold table above 4 GiB");
            pl->S.alloc(sbytes);
        } else {
            pl->win_host = row_windows(pr, corners, c.t0, c.dT, c.T, pl->ldh);
            pl->win.alloc(sizeof(uint32_t) * pl->win_host.size());
            tables.add(pl->win.ptr, pl->win_host.data(), sizeof(uint32_t) * pl->win_host.size());
            const StageJob job = stage_job(*pl);
            pl->stage_zb = stage_z_blocks(job);
            pl->stage_sb = stage_row_blocks(job);
            pl->stage.alloc(sizeof(StageJob));   // written by set_fused_variant
        }
        pl->inv2 = (float)(2.0 / (double)c.dT);
        std::vector<float> p4((size_t)pl->P * 4);
        bool flat = true;
        for (uint32_t p = 0; p < pl->P; ++p) {
            p4[4 * p + 0] = pr[p].laser_point[0];
            p4[4 * p + 1] = pr[p].laser_point[1];
            p4[4 * p + 2] = pr[p].laser_point[2];
            p4[4 * p + 3] = (float)(((double)pr[p].laser_wall + (double)pr[p].camera_wall - (double)c.t0) /
                                        (double)c.dT + 1.0);
            flat = flat && pr[p].laser_point[2] == pr[0].laser_point[2];
        }
        pl->flat = flat;
        pl->zflat = flat;
        pl->lz = pr[0].laser_point[2];
        pl->sep = inc[6] == 0.0f && inc[7] == 0.0f;
        if (!pl->sep) pl->flat = false;
        if (o.variant < 0) pl->variant = default_variant(*pl);
        pl->keep_f32 = (o.flags & BPX_FLAG_KEEP_F32_ROWS) != 0;
        pl->auto_variant = o.variant < 0;
        if (pl->fused) {
            set_fused_variant(*pl, pl->variant);
        } else {
            pl->lds_tiles = false;
            pl->rows16 = false;
        }
        pl->pair4.alloc(sizeof(float) * p4.size());
        tables.add(pl->pair4.ptr, p4.data(), sizeof(float) * p4.size());
    } else {
        if ((uint64_t)(c.T + 1) * 4 > 64 * 1024)
            fail(BPX_ERR_UNSUPPORTED, "non-confocal captures need T <= 16383 after cropping");
        pl->Z.alloc(sizeof(float) * (c.T + 1));
        pl->inv = (float)(1.0 / (double)c.dT);
        pl->c1 = (float)(1.0 - (double)c.t0 / (double)c.dT);
        if (pl->path == kPathGrid) {
            std::vector<float> las((size_t)pl->L * 4), spd((size_t)pl->C * 4);
            for (uint32_t l = 0; l < pl->L; ++l) {
                const bpx_pair& a = pr[(size_t)l * pl->C];
                las[4 * l + 0] = a.laser_point[0];
                las[4 * l + 1] = a.laser_point[1];
                las[4 * l + 2] = a.laser_point[2];
                las[4 * l + 3] = a.laser_wall;
            }
            for (uint32_t s = 0; s < pl->C; ++s) {
                spd[4 * s + 0] = pr[s].camera_point[0];
                spd[4 * s + 1] = pr[s].camera_point[1];
                spd[4 * s + 2] = pr[s].camera_point[2];
                spd[4 * s + 3] = pr[s].camera_wall;
            }
            pl->lasers.alloc(sizeof(float) * las.size());
            pl->spads.alloc(sizeof(float) * spd.size());
            tables.add(pl->lasers.ptr, las.data(), sizeof(float) * las.size());
            tables.add(pl->spads.ptr, spd.data(), sizeof(float) * spd.size());
        }
    }
    tables.finish();
    return pl.release();
}

int staged_format(const PlanImpl& pl) {
    if (!pl.fmt_flag.ptr || (!pl.rows16 && !pl.poly_counts)) return pl.row_format;
    plan_wait(pl);
    uint32_t flag = 3;
    hip_check(hipMemcpy(&flag, pl.fmt_flag.ptr, 4, hipMemcpyDeviceToHost), "hipMemcpy(row format)");
    return flag == 0u && pl.poly_counts ? kCount : pl.rows16 && !(flag & 1u) ? kF16 : pl.row_format;
}

StageJob stage_job(const PlanImpl& pl) {
    StageJob j{};
    j.src = static_cast<const float*>(pl.raw.ptr);
    j.dst = pl.H.ptr;
    j.pair8 = static_cast<const float*>(pl.pair8.ptr);
    j.Z = static_cast<float*>(pl.Z.ptr);
    j.rows = pl.P;
    j.Tc = pl.T;
    j.lde = pl.ldh;
    j.format = pl.row_format;
    j.fmt_flag = pl.rows16 || pl.poly_counts ? static_cast<const uint32_t*>(pl.fmt_flag.ptr) : nullptr;
    j.win = static_cast<const uint32_t*>(pl.win.ptr);
    j.alt_format = pl.rows16 ? kF16 : pl.row_format;
    j.count_rows = pl.poly_counts ? 1 : 0;
    j.clear_flag = j.fmt_flag ? 1u : 0u;
    j.inv_scale = 1.0f / pl.scale;
    j.t0 = pl.t0;
    j.dT = pl.dT;
    return j;
}

void set_fused_variant(PlanImpl& pl, int variant) {
    pl.variant = variant;
    pl.K = variant_k(variant);
    pl.tiles = make_tiles(pl.g.n, pl.K);
    pl.lds_tiles = variant >= kLdsVariant && pl.sep && pl.flat &&
                   confocal_lds_fits(pl.g.inc, pl.inv2, lds_shape(variant, pl.format).depth(),
                                     lds_seg_elems(pl.format));
    // fp32 rows of integer samples within fp16's exact range are staged as fp16: the same
    // values, half the LDS bytes per lookup (one 8-B read instead of an 8-B and a 4-B one).
    // Each execution checks its samples on the device first and stages and gathers in the
    // format the check allows, so the volume is the fp32 rows' bit for bit either way.  For
    // the shapes of 8 voxels per lane (gather ms at 16,384 pairs, fp32 -> fp16 rows: 128^3
    // 16^3 x 512 lanes 12.96 -> 11.67, 16 x 16 x 8 x 256 14.57 -> 13.92; 256^3 83.3 -> 83.2,
    // 91.7 -> 89.7); the 16-per-lane shape, bound by its arithmetic and the default where
    // it applies (256^3), measured slower with fp16 rows (84.5 -> 86.4), so it keeps fp32.
    pl.rows16 = pl.lds_tiles && pl.format == kF32 && lds_shape(variant, pl.format).kz == 8 && !pl.keep_f32;
    // Rows of counts: integer sums need no order and no compensation, so any split of the pairs
    // gives the volume of the fp32 rows bit for bit while a block of kahan_block counts stays
    // below 2^24 and the whole sum below 2^32.  For variants 7 and 8 (as the exact fp16 rows), and for
    // every confocal plan whose variant was left to the library.
    // The other rows (fp32, 16-bit, complex64) for every confocal plan whose variant was left to the
    // library.
    pl.poly = LdsPolyShape{};
    pl.poly_counts = pl.poly_real = false;
    pl.row_format = pl.format;
    if (!pl.keep_f32 && pl.sep && pl.flat) {
        const bool counts = pl.format == kF32 && (pl.auto_variant || variant > kLdsVariant) && pl.kahan_block <= 4096u &&
                            pl.P <= (1u << 20);
        const bool real = pl.auto_variant && (!format_complex(pl.format) || pl.format == kC64);
        const int rows = pl.format == kC64 ? (int)kC64Split : pl.format == kF32 ? (int)kF32Split : pl.format;
        if (counts || real)
            pl.poly = lds_poly_shape(pl.g, pl.inv2, pl.lz, pl.tap_bound, pl.max_path, kPolyBudget, real ? rows : (int)kCount);
        pl.poly_counts = counts && pl.poly.kz;
        pl.poly_real = real && pl.poly.kz;
        if (pl.poly_real) pl.row_format = rows;
        const size_t vox = (size_t)pl.g.n[0] * pl.g.n[1] * pl.g.n[2];
        size_t bytes = 0;
        if (pl.poly_counts) {
            pl.poly_parts = lds_poly_parts(pl.g, pl.poly, pl.P, 4u, 4u, &pl.poly_part_pairs);
            if (pl.poly_parts > 1) bytes = pl.poly_parts * vox * 4u;
        }
        if (pl.poly_real) {
            const uint32_t b = lds_poly_part_bytes(rows);
            pl.real_parts = lds_poly_parts(pl.g, pl.poly, pl.P, b, part_unit(pl.kahan_block), &pl.real_part_pairs);
            if (pl.real_parts > 1) bytes = std::max(bytes, pl.real_parts * vox * b);
        }
        if (bytes > pl.parts.bytes) pl.parts.alloc(bytes);
    }
    pl.tex_parts = 1;
    if (pl.auto_variant && !pl.poly_real && !pl.lds_tiles && variant == kDefaultVariant) {
        pl.tex_parts = split_parts(pl.tiles, pl.P, part_unit(pl.kahan_block), &pl.tex_part_pairs);
        const size_t bytes = (size_t)pl.tex_parts * pl.g.n[0] * pl.g.n[1] * pl.g.n[2] * (pl.cplx ? 16u : 8u);
        if (pl.tex_parts > 1 && bytes > pl.parts.bytes) pl.parts.alloc(bytes);
    }
    if ((pl.rows16 || pl.poly_counts) && !pl.fmt_flag.ptr) {
        pl.fmt_flag.alloc(4);
        // fp32 until run
        hip_check(hipMemsetAsync(pl.fmt_flag.ptr, 0xff, 4, pl.stream), "hipMemsetAsync(row format)");
    }
    if (pl.stage.ptr) {   // the staging descriptor names the format flag (or none)
        const StageJob job = stage_job(pl);
        hip_check(hipMemcpy(pl.stage.ptr, &job, sizeof(StageJob), hipMemcpyHostToDevice), "hipMemcpy(staging job)");
    }
}

void stage_rows(PlanImpl& pl, hipStream_t s) {
    hip_check(launch_stage(static_cast<const StageJob*>(pl.stage.ptr), 1u, pl.stage_zb, pl.stage_sb, s),
              "row staging kernels");
}

void PlanImpl::execute(hipStream_t s) {
    if (path == kPathOctree) {
        execute_octree(*this, s);
        return;
    }
    const size_t nvox = (size_t)g.n[0] * g.n[1] * g.n[2];
    // a recorded event costs the GPU about as much as a small kernel's launch
    const auto mark = [&](int k) {
        if (timed) hip_check(hipEventRecord(ev[k], s), "hipEventRecord");
    };
    if (path == kPathWindow) {
        if (P == 0 || T < 2) {
            hip_check(hipMemsetAsync(vol.ptr, 0, nvox * (cplx ? 8 : 4), s), "hipMemsetAsync");
            return;
        }
        mark(0);
        hip_check(launch_prefix(static_cast<const float*>(raw.ptr), P, T, cplx ? 1 : 0, H.ptr, ldh, s),
                  "prefix kernel");
        mark(1);
        hip_check(launch_ztable(1, t0, dT, half_width, T, static_cast<float*>(Z.ptr), s), "window table (start)");
        hip_check(launch_ztable(2, t0, dT, half_width, T, static_cast<float*>(Z2.ptr), s), "window table (end)");
        if (poly.kz) {
            WindowLdsArgs a = wlds;
            a.PS = static_cast<const double*>(H.ptr);
            a.Slo = static_cast<const double*>(win_lo.ptr);
            a.Shi = static_cast<const double*>(win_hi.ptr);
            a.Zlo = static_cast<const float*>(Z.ptr);
            a.Zhi = static_cast<const float*>(Z2.ptr);
            a.pair8 = static_cast<const float*>(pair8.ptr);
            a.pairs = static_cast<const float4*>(pair4.ptr);
            a.out = static_cast<float*>(vol.ptr);
            a.parts = poly_parts > 1 ? static_cast<double*>(parts.ptr) : nullptr;
            hip_check(launch_window_tables(a, static_cast<double*>(win_lo.ptr), static_cast<double*>(win_hi.ptr), s),
                      "window threshold kernel");
            mark(2);
            hip_check(launch_window_lds(a, poly, poly_parts, s), "window gather kernel (LDS-staged)");
            mark(3);
            return;
        }
        mark(2);
        WindowArgs a{};
        a.PS = H.ptr;
        a.pairs = static_cast<const float*>(pair8.ptr);
        a.Zlo = static_cast<const float*>(Z.ptr);
        a.Zhi = static_cast<const float*>(Z2.ptr);
        a.out = vol.ptr;
        a.P = P;
        a.T = T;
        a.ldp = ldh;
        a.ps_bytes = H.bytes;
        std::memcpy(a.n, g.n, sizeof(a.n));
        std::memcpy(a.zero, wzero, sizeof(a.zero));
        std::memcpy(a.vsize, wvs, sizeof(a.vsize));
        a.inv = inv;
        a.c1_lo = c1_lo;
        a.c1_hi = c1_hi;
        a.confocal = all_confocal ? 1u : 0u;
        hip_check(launch_window(a, cplx ? 1 : 0, s), "window gather kernel");
        mark(3);
        return;
    }
    if (P == 0) {
        hip_check(hipMemsetAsync(vol.ptr, 0, nvox * (cplx ? 8 : 4), s), "hipMemsetAsync");
        return;
    }
    // marks: ev[0] | split-layout row padding | ev[1] | tables (fused: all staging) | ev[2] |
    // gather | ev[3]
    mark(0);
    if (paths.seg) {
        if (format != kF32)
            hip_check(launch_quantise_rows(static_cast<const float*>(raw.ptr), (uint64_t)P * T, format, 1.0f / scale,
                                           static_cast<float*>(H.ptr), s),
                      "row quantisation kernel");
    } else if (!fused)
        hip_check(launch_pad_rows(static_cast<const float*>(raw.ptr), P, T, T, H.ptr, ldh, format,
                                  1.0f / scale, s),
                  "row staging kernel");
    mark(1);
    if (path == kPathConfocal) {
        if (fused) {
            const StageJob* const job = static_cast<const StageJob*>(stage.ptr);
            hip_check(launch_stage(job, 1u, stage_zb, 0u, s), "path-length table kernel");   // clears the flag
            if (rows16 || poly_counts)
                hip_check(launch_exact16_check(static_cast<const float*>(raw.ptr), (uint64_t)P * T,
                                               static_cast<uint32_t*>(fmt_flag.ptr), s),
                          "exact fp16 check kernel");
            hip_check(launch_stage(job, 1u, 0u, stage_sb, s), "row staging kernel");
        } else {
            hip_check(launch_ztable(0, t0, dT, 0.0f, T + 1, static_cast<float*>(Z.ptr), s),
                      "path-length table kernel");
            hip_check(launch_stable(static_cast<const float*>(pair8.ptr), P, T, static_cast<const float*>(Z.ptr),
                                    static_cast<float*>(S.ptr), lds, 1u, 0u, s),
                      "threshold table kernel");
        }
        mark(2);
        ConfocalArgs a{};
        a.H = H.ptr;
        a.S = static_cast<const float*>(S.ptr);
        a.pairs = static_cast<const float4*>(pair4.ptr);
        a.out = vol.ptr;
        a.P = P;
        a.Tc = T;
        a.ldh = ldh;
        a.lds = lds;
        a.h_bytes = (uint32_t)H.bytes;
        a.s_bytes = (uint32_t)(fused ? 0 : S.bytes);
        a.g = g;
        a.t = tiles;
        a.inv2 = inv2;
        a.scale = scale;
        a.lz = lz;
        a.kahan_block = kahan_block;
        const auto gather = [&](int rows) {
            const bool counts = rows == kCount;
            if (tex_parts > 1) {
                hip_check(launch_split(a, SplitPairs{parts.ptr, tex_part_pairs, 0u}, rows, tex_parts, sep, flat, s),
                          "confocal gather kernel (pairs split)");
                return;
            }
            if (!counts && !poly_real) {
                hip_check(launch_confocal(a, rows, variant, sep, flat, s), "confocal gather kernel");
                return;
            }
            LdsPolyArgs pa = lds_poly_args(a, poly);
            const uint32_t n = counts ? poly_parts : real_parts;
            pa.part_pairs = counts ? poly_part_pairs : real_part_pairs;
            pa.parts = n > 1 ? parts.ptr : nullptr;
            hip_check(launch_lds_poly(pa, poly, rows, n, s), "confocal gather kernel (polynomial quotients)");
        };
        if (rows16 || poly_counts) {
            // every instantiation launched; those the device check did not pick return at once
            a.fmt_flag = static_cast<const uint32_t*>(fmt_flag.ptr);
            if (poly_counts) {
                a.fmt_mask = 3u;
                a.fmt_want = 0u;
                gather(kCount);
            }
            if (rows16) {
                a.fmt_mask = poly_counts ? 3u : 1u;
                a.fmt_want = poly_counts ? 2u : 0u;
                gather(kF16);
            }
            a.fmt_mask = a.fmt_want = rows16 ? 1u : 2u;
        }
        gather(row_format);
        const uint32_t count_parts = poly_counts ? poly_parts : 0u, own_parts = poly_real ? real_parts : tex_parts;
        if (count_parts > 1u || own_parts > 1u)
            hip_check(launch_sum_parts(PartsSum{vol.ptr, parts.ptr, static_cast<const uint32_t*>(fmt_flag.ptr), nvox,
                                                count_parts, own_parts, cplx ? 1u : 0u, scale}, s),
                      "partial sums kernel");
    } else {
        hip_check(launch_ztable(0, t0, dT, 0.0f, T + 1, static_cast<float*>(Z.ptr), s),
                  "threshold table kernel");
        mark(2);
        if (paths.seg) {
            PathsLdsArgs a = paths;
            a.rows = static_cast<const float*>(format == kF32 ? raw.ptr : H.ptr);
            a.lasers = static_cast<const float4*>(lasers.ptr);
            a.spads = static_cast<const float4*>(spads.ptr);
            a.pairs = static_cast<const float*>(pair8.ptr);
            a.Z = static_cast<const float*>(Z.ptr);
            a.out = static_cast<float*>(vol.ptr);
            a.parts = paths_parts > 1 ? static_cast<double*>(parts.ptr) : nullptr;
            a.inv = inv;
            a.c1 = c1;
            hip_check(launch_paths_lds(a, paths_parts, s), "gather kernel (LDS-staged paths)");
        } else if (path == kPathGrid) {
            GridArgs a{};
            a.H = H.ptr;
            a.lasers = static_cast<const float4*>(lasers.ptr);
            a.spads = static_cast<const float4*>(spads.ptr);
            a.Z = static_cast<const float*>(Z.ptr);
            a.out = vol.ptr;
            a.L = L;
            a.C = C;
            a.Tc = T;
            a.ldh = ldh;
            a.h_bytes = (uint32_t)H.bytes;
            a.g = g;
            a.t = tiles;
            a.inv = inv;
            a.c1 = c1;
            a.scale = scale;
            a.kahan_block = kahan_block;
            hip_check(launch_grid(a, format, variant, s), "grid gather kernel");
        } else {
            PairsArgs a{};
            a.H = H.ptr;
            a.pairs = static_cast<const float*>(pair8.ptr);
            a.Z = static_cast<const float*>(Z.ptr);
            a.out = vol.ptr;
            a.P = P;
            a.Tc = T;
            a.ldh = ldh;
            a.h_bytes = (uint32_t)H.bytes;
            a.g = g;
            a.t = tiles;
            a.inv = inv;
            a.c1 = c1;
            a.scale = scale;
            a.kahan_block = kahan_block;
            hip_check(launch_pairs(a, format, variant, s), "pairs gather kernel");
        }
    }
    mark(3);
}

// The LDS-staged window kernel where it applies: real samples, confocal pairs on a flat wall, bin
// windows and threshold tables that fit, in LDS and in the device's memory.  Allocates the prefix sums
// then (H) and sets their row pitch; the general kernel's are the caller's.
static void window_lds_setup(PlanImpl& pl, const std::vector<bpx_pair>& pr, float width) {
    bool flat = true;
    for (const auto& p : pr) flat = flat && p.laser_point[2] == pr[0].laser_point[2];
    if (pl.cplx || !pl.all_confocal || !flat) return;
    for (int k = 0; k < 3; ++k) {
        pl.g.zero[k] = pl.wzero[k];
        pl.g.inc[4 * k] = pl.wvs[k];
    }
    pl.lz = pr[0].laser_point[2];
    pl.inv2 = (float)(2.0 / (double)pl.dT);
    const LdsPolyShape sh = lds_poly_shape(pl.g, pl.inv2, pl.lz, pl.tap_bound, pl.max_path, kWindowPolyBudget, kCount);
    const double bins = (double)width / (double)pl.dT;
    if (!sh.kz || !(bins < 1024.0)) return;
    WindowLdsArgs& a = pl.wlds;
    a.P = pl.P;
    a.T = pl.T;
    a.seg = sh.seg;
    a.shift = (uint32_t)bins & ~1u;
    a.seg_sums = round_up((uint64_t)sh.seg + a.shift + 6u, 128);
    a.ldp = round_up((uint64_t)pl.T + a.seg_sums, 32);
    a.pitch = round_up(pl.T, 32);
    if (window_lds_bytes(a) > 160u * 1024u) return;
    // tables beside the sums: 16 more bytes a bin, at most 16 GiB in all
    if ((uint64_t)pl.P * (2u * a.pitch + a.ldp) * 8u > (16ull << 30)) return;
    a.g = pl.g;
    a.inv2 = pl.inv2;
    a.lz = pl.lz;
    a.width_bins = (float)bins;
    a.hi_offset = (float)(bins - (double)a.shift + (double)a.seg);
    const LdsPolyArgs k = lds_poly_args(ConfocalArgs{.g = pl.g, .inv2 = pl.inv2}, sh);
    a.k1 = k.k1;
    a.k2 = k.k2;
    a.k3 = k.k3;
    std::vector<float> p4((size_t)pl.P * 4);
    for (uint32_t p = 0; p < pl.P; ++p) {
        p4[4 * p + 0] = pr[p].laser_point[0];
        p4[4 * p + 1] = pr[p].laser_point[1];
        p4[4 * p + 2] = pr[p].laser_point[2];
        p4[4 * p + 3] = (float)(((double)pr[p].laser_wall + (double)pr[p].camera_wall - (double)pl.half_width -
                                 (double)pl.t0) / (double)pl.dT + 1.0);
    }
    // double sums: a split changes their last bits only
    pl.poly_parts = lds_poly_parts(pl.g, sh, pl.P, 8u, 4u, &a.part_pairs);
    const size_t sums = pl.poly_parts > 1 ? (size_t)pl.poly_parts * pl.g.n[0] * pl.g.n[1] * pl.g.n[2] * 8u : 0u;
    const size_t table = (size_t)pl.P * a.pitch * 8u;
    if (!pl.pair4.try_alloc(sizeof(float) * p4.size()) || !pl.win_lo.try_alloc(table) || !pl.win_hi.try_alloc(table) ||
        (sums && !pl.parts.try_alloc(sums)) || !pl.H.try_alloc((size_t)pl.P * a.ldp * 8u)) {
        for (DeviceBuffer* b : {&pl.pair4, &pl.win_lo, &pl.win_hi, &pl.parts, &pl.H}) b->release();
        return;
    }
    hip_check(hipMemcpy(pl.pair4.ptr, p4.data(), sizeof(float) * p4.size(), hipMemcpyHostToDevice), "hipMemcpy(pairs)");
    pl.ldh = a.ldp;
    pl.poly = sh;
}

PlanImpl* make_plan_window(const CaptureIn& c, const uint32_t n[3], const float vpos[3],
                           const float vsize[3]) {
    validate_common(c, n);
    for (int k = 0; k < 3; ++k)
        if (!std::isfinite(vpos[k]) || !std::isfinite(vsize[k]))
            fail(BPX_ERR_INVALID_ARGUMENT, "volume position/size must be finite");
    if (!device_ready()) fail(BPX_ERR_NO_DEVICE, "no gfx950 device available");
    auto pl = std::make_unique<PlanImpl>();
    pl->stream = take_stream();
    make_events(*pl);
    pl->path = kPathWindow;
    pl->cplx = c.cplx;
    pl->format = c.cplx ? kC64 : kF32;
    pl->t0 = c.t0;
    pl->dT = c.dT;
    pl->T = c.T;
    std::memcpy(pl->g.n, n, sizeof(uint32_t) * 3);
    // CPU grid (octree_volume.hpp:42, 147-167) and window width (backproject.hpp:147)
    for (int k = 0; k < 3; ++k) {
        pl->wzero[k] = vpos[k] - vsize[k] / 2.0f;
        pl->wvs[k] = vsize[k] / (float)n[k];
    }
    const float a2 = pl->wvs[0] * pl->wvs[0], b2 = pl->wvs[1] * pl->wvs[1], c2 = pl->wvs[2] * pl->wvs[2];
    const float width = (float)std::sqrt(((double)a2 + (double)b2) + (double)c2);
    pl->half_width = width / 2.0f;
    const std::vector<uint32_t> idx = used_pairs(c, 0);
    std::vector<bpx_pair> pr(idx.size());
    for (size_t i = 0; i < idx.size(); ++i) pr[i] = c.pairs[idx[i]];
    pl->P = (uint32_t)pr.size();
    bool confocal = true;
    for (const auto& p : pr) confocal = confocal && same3(p.laser_point, p.camera_point);
    pl->all_confocal = confocal;
    const size_t nvox = (size_t)n[0] * n[1] * n[2];
    pl->vol.alloc(nvox * (c.cplx ? 8 : 4));
    // exactness precondition: CPU-grid corners
    double corners[8][3];
    for (int m = 0; m < 8; ++m) {
        const double i[3] = {(m & 4) ? (double)(n[0] - 1) : 0.0, (m & 2) ? (double)(n[1] - 1) : 0.0,
                             (m & 1) ? (double)(n[2] - 1) : 0.0};
        for (int k = 0; k < 3; ++k) corners[m][k] = (double)pl->wzero[k] + (double)pl->wvs[k] * i[k];
    }
    pl->max_path = max_total_path(pr.data(), pr.size(), corners);
    const double bound = tap_error_bound(pl->max_path + width, c.t0, c.dT, c.T);
    pl->tap_bound = bound;
    if (bound >= 0.25)
        fail(BPX_ERR_UNSUPPORTED, "path lengths / t0 too large relative to deltaT for the exact bin lookup");
    pl->inv = (float)(1.0 / (double)c.dT);
    pl->c1_lo = (float)(1.0 - ((double)c.t0 + (double)pl->half_width) / (double)c.dT);
    pl->c1_hi = (float)(1.0 - ((double)c.t0 - (double)pl->half_width) / (double)c.dT);
    if (pl->P == 0 || c.T < 2) return pl.release();
    stage_raw(*pl, c, idx);
    pl->ldh = round_up(c.T, 32);
    pl->Z.alloc(sizeof(float) * c.T);
    pl->Z2.alloc(sizeof(float) * c.T);
    std::vector<float> p8((size_t)pl->P * 8);
    std::memcpy(p8.data(), pr.data(), sizeof(float) * p8.size());
    pl->pair8.alloc(sizeof(float) * p8.size());
    hip_check(hipMemcpy(pl->pair8.ptr, p8.data(), sizeof(float) * p8.size(), hipMemcpyHostToDevice),
              "hipMemcpy(pairs)");
    window_lds_setup(*pl, pr, width);
    if (!pl->poly.kz) pl->H.alloc((size_t)pl->P * pl->ldh * (c.cplx ? 16 : 8));
    return pl.release();
}

}  // namespace bpx
