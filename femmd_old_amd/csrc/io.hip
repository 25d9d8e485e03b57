// io.hip -- the engine's traffic with the caller's host arrays.
//
// The boundary hands over caller-ordered host arrays (femmd2D/src/
// particles.cpp:105-199 copies whole arrays); the device holds them in the
// engine's internal order.  Kernels do the re-ordering, reading the internal
// arrays through the caller -> internal map and writing the caller's order
// straight into pinned host memory (and back), so a query is one kernel and
// one wait; the host only copies contiguous runs between that memory and the
// caller's arrays.  Large transfers go through a ring of kIoSlots slots, the
// device filling (or emptying) some while the host copies another: the pinned
// memory of an engine is bounded by kIoSlots * kIoSlotBytes.  Where no pinned
// memory can be had, a slot on the device takes its place and is copied.
//
// Bound by the latency of one kernel and one wait (13 us) for small systems
// and by the host link for large ones.  Before, each array was copied to
// pageable memory on its own and permuted on the host.  Measured, before and
// now: get_state (4 arrays) of 256 particles 98 -> 21 us, of 114,140 220 ->
// 85 us, of 1,141,760 5.5 -> 0.68 ms, of 512 replicas of 1088 42.6 -> 13.2 ms;
// energies 43 -> 13 us; set_state of 57,120 169 -> 51 us; adjoint_op of
// 57,120 273 -> 161 us.
#include <algorithm>
#include <cstring>

#include "engine.hpp"

namespace fm {

namespace {
constexpr int kIoThreads = 256;

struct StateOutArgs {
    const float *src[4];
    const int32_t *iid;  // caller id -> internal id
    uint32_t n;
};
// out[t] = value t0 + t of the arrays src[0], src[1], ... in caller order,
// one after the other (n values each).
__global__ __launch_bounds__(kIoThreads) void k_state_out(StateOutArgs a, uint64_t t0, uint32_t m,
                                                          float *out) {
    const uint32_t t = blockIdx.x * kIoThreads + threadIdx.x;
    if (t >= m) return;
    const uint64_t i = t0 + t;
    const uint32_t k = (uint32_t)(i / a.n), u = (uint32_t)(i - (uint64_t)k * a.n);
    const float *s = k == 0 ? a.src[0] : k == 1 ? a.src[1] : k == 2 ? a.src[2] : a.src[3];
    out[t] = s[a.iid[u]];
}

struct StateInArgs {
    float *dst[4];
    float wrap[4];  // box length of a position, 0: stored as given
    uint32_t stride;  // between a particle's values in dst
    const int32_t *iid;
    uint32_t n;
};
__global__ __launch_bounds__(kIoThreads) void k_state_in(StateInArgs a, uint64_t t0, uint32_t m,
                                                         const float *in) {
    const uint32_t t = blockIdx.x * kIoThreads + threadIdx.x;
    if (t >= m) return;
    const uint64_t i = t0 + t;
    const uint32_t k = (uint32_t)(i / a.n), u = (uint32_t)(i - (uint64_t)k * a.n);
    float *d = k == 0 ? a.dst[0] : k == 1 ? a.dst[1] : k == 2 ? a.dst[2] : a.dst[3];
    const float L = k == 0 ? a.wrap[0] : k == 1 ? a.wrap[1] : k == 2 ? a.wrap[2] : a.wrap[3];
    float v = in[t];
    if (L > 0.0f) {  // femmd2D/src/def.h:112 pbcCalc, FP32
        const float q = v / L;
        const float f = floorf(q);
        const float p = f * L;
        v = v - p;
    }
    d[(size_t)a.iid[u] * a.stride] = v;
}

// Total force per particle, caller order: pair force plus its corner forces
// (held in gather order), x then y.
__global__ __launch_bounds__(kIoThreads) void k_force_out(const float *fx, const float *fy,
                                                          const float2 *cf, const int32_t *goff,
                                                          const int32_t *iid, uint32_t n, uint64_t t0,
                                                          uint32_t m, float *out) {
    const uint32_t t = blockIdx.x * kIoThreads + threadIdx.x;
    if (t >= m) return;
    const uint64_t i = t0 + t;
    const bool y = i >= n;
    const int q = iid[y ? i - n : i];
    float v = y ? fy[q] : fx[q];
    if (goff)
        for (int e = goff[q]; e < goff[q + 1]; ++e) {
            const float2 c = cf[e];
            v += y ? c.y : c.x;
        }
    out[t] = v;
}

// out[t] = src[idx ? idx[t0 + t] : t0 + t]
template <class T>
__global__ __launch_bounds__(kIoThreads) void k_out(const T *src, const int32_t *idx, uint64_t t0,
                                                    uint32_t m, T *out) {
    const uint32_t t = blockIdx.x * kIoThreads + threadIdx.x;
    if (t < m) out[t] = src[idx ? (uint64_t)idx[t0 + t] : t0 + t];
}

// The error word (and the n doubles of src) to the host.
__global__ void k_report(const uint32_t *err, const double *src, int n, IoHead *h) {
    if (threadIdx.x == 0) h->err = *err;
    if ((int)threadIdx.x < n) h->obs[threadIdx.x] = src[threadIdx.x];
}

// iid[p0 + uid[q]] = q for the particles q of a span.
__global__ __launch_bounds__(kKickThreads) void k_invert(const Span *spans, const RepDesc *reps,
                                                         const int32_t *uid, int32_t *iid) {
    const Span sp = spans[blockIdx.x];
    const int q = sp.begin + (int)threadIdx.x;
    if (q < sp.end) iid[reps[sp.rep].p0 + uid[q]] = q;
}

unsigned blocks(uint32_t m) { return (m + kIoThreads - 1) / kIoThreads; }
}  // namespace

PinBuf::~PinBuf() {
    if (staged()) {
        delete[] p;
        if (d) (void)hipFree(d);
    } else if (p) {
        (void)hipHostFree(p);
    }
    for (auto &e : ev)
        if (e) (void)hipEventDestroy(e);
}

// Memory for the largest replica's state, at most a ring of slots.
hipError_t PinBuf::alloc(size_t most, bool pinned) {
    slot = std::min<size_t>(std::max<size_t>((most + 255) / 256 * 256, 1024), kIoSlotBytes);
    nslot = most > slot ? kIoSlots : 1;
    hipError_t e = hipSuccess;
    if (pinned && hipHostMalloc(reinterpret_cast<void **>(&p), sizeof(IoHead) + slot * nslot,
                                hipHostMallocDefault) == hipSuccess) {
        d = p;
    } else {
        (void)hipGetLastError();
        nslot = 1;
        p = new unsigned char[sizeof(IoHead) + slot];
        if ((e = hipMalloc(reinterpret_cast<void **>(&d), sizeof(IoHead) + slot)) != hipSuccess) {
            d = nullptr;
            return e;
        }
    }
    std::memset(p, 0, sizeof(IoHead));
    for (int k = 0; k < (nslot > 1 ? nslot : 0); ++k)
        if ((e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming)) != hipSuccess) return e;
    return hipSuccess;
}

// `count` items of `elem` bytes to the host: fill(first, n, slot) launches
// the kernel that writes items [first, first + n) into a slot (and, staged,
// its copy follows on the stream), take(first, n, slot) consumes them on the
// host, in order.
template <class Fill, class Take>
int Engine::io_read(size_t count, size_t elem, Fill &&fill, Take &&take, std::string &err) {
    std::lock_guard<std::mutex> lock(pin_.mu);
    const size_t per = pin_.slot / elem;
    auto put = [&](size_t i, size_t m, int s) -> bool {  // true: failed
        return fill((uint64_t)i, (uint32_t)m, pin_.ddata(s)) ||
               (pin_.staged() && hipMemcpyAsync(pin_.data(s), pin_.ddata(s), m * elem,
                                                hipMemcpyDeviceToHost, stream_) != hipSuccess);
    };
    if (count == 0) return FM_OK;
    if (count <= per) {
        if (put(0, count, 0)) return check(hipErrorUnknown, "read", err);
        const int rc = check(hipStreamSynchronize(stream_), "read", err);
        if (rc) return rc;
        take((uint64_t)0, (uint32_t)count, pin_.data(0));
        return FM_OK;
    }
    const size_t nchunk = (count + per - 1) / per;
    size_t issued = 0;
    for (size_t c = 0; c < nchunk; ++c) {
        for (; issued < nchunk && issued < c + (size_t)pin_.nslot; ++issued) {
            const size_t i = issued * per;
            const int s = (int)(issued % pin_.nslot);
            if (put(i, std::min(per, count - i), s) ||
                (pin_.nslot > 1 && hipEventRecord(pin_.ev[s], stream_) != hipSuccess)) {
                (void)hipStreamSynchronize(stream_);
                return check(hipErrorUnknown, "read", err);
            }
        }
        const int s = (int)(c % pin_.nslot);
        const int rc = check(pin_.nslot > 1 ? hipEventSynchronize(pin_.ev[s])
                                            : hipStreamSynchronize(stream_), "read", err);
        if (rc) return rc;
        const size_t i = c * per;
        take((uint64_t)i, (uint32_t)std::min(per, count - i), pin_.data(s));
    }
    return FM_OK;
}

// The other way: put(first, n, slot) writes items into a slot on the host,
// use(first, n, slot) launches the kernel that reads them.  Returns with the
// stream drained (the slots are free again).
template <class Put, class Use>
int Engine::io_write(size_t count, size_t elem, Put &&put, Use &&use, std::string &err) {
    std::lock_guard<std::mutex> lock(pin_.mu);
    const size_t per = pin_.slot / elem;
    size_t c = 0;
    for (size_t i = 0; i < count; i += per, ++c) {
        const int s = (int)(c % pin_.nslot);
        if (c >= (size_t)pin_.nslot) {
            const int rc = check(pin_.nslot > 1 ? hipEventSynchronize(pin_.ev[s])
                                                : hipStreamSynchronize(stream_), "write", err);
            if (rc) return rc;
        }
        const uint32_t m = (uint32_t)std::min(per, count - i);
        put((uint64_t)i, m, pin_.data(s));
        if ((pin_.staged() && hipMemcpyAsync(pin_.ddata(s), pin_.data(s), m * elem,
                                             hipMemcpyHostToDevice, stream_) != hipSuccess) ||
            use((uint64_t)i, m, pin_.ddata(s)) ||
            (pin_.nslot > 1 && hipEventRecord(pin_.ev[s], stream_) != hipSuccess)) {
            (void)hipStreamSynchronize(stream_);
            return check(hipErrorUnknown, "write", err);
        }
    }
    return check(hipStreamSynchronize(stream_), "write", err);
}

namespace {
// Copies items [i, i + m) of the concatenation of the k arrays a (n floats
// each) from (kOut) or to a slot.
template <bool kOut>
void split_copy(float *const *a, int k, size_t n, size_t i, size_t m, void *slot) {
    float *s = static_cast<float *>(slot);
    for (int q = (int)(i / n); q < k && m > 0; ++q) {
        const size_t u = i - (size_t)q * n, c = std::min(m, n - u);
        if (kOut) std::memcpy(a[q] + u, s, c * sizeof(float));
        else std::memcpy(s, a[q] + u, c * sizeof(float));
        s += c;
        i += c;
        m -= c;
    }
}
}  // namespace

int Engine::io_state_out(int r, int k, const float *const *src, float *const *dst, std::string &err) {
    const size_t n = (size_t)nparticles(r);
    StateOutArgs a{};
    for (int q = 0; q < 4; ++q) a.src[q] = src[std::min(q, k - 1)];
    a.iid = iid_.p + reps_h_[r].p0;
    a.n = (uint32_t)n;
    return io_read(
        n * k, sizeof(float),
        [&](uint64_t i, uint32_t m, void *slot) {
            hipLaunchKernelGGL(k_state_out, dim3(blocks(m)), dim3(kIoThreads), 0, stream_, a, i, m,
                               static_cast<float *>(slot));
            return hipGetLastError() != hipSuccess;
        },
        [&](uint64_t i, uint32_t m, void *slot) { split_copy<true>(dst, k, n, i, m, slot); }, err);
}

int Engine::io_state_in(int r, int k, const float *const *src, float *const *dst, const float *wrap,
                        int stride, std::string &err) {
    const size_t n = (size_t)nparticles(r);
    StateInArgs a{};
    for (int q = 0; q < 4; ++q) {
        a.dst[q] = dst[std::min(q, k - 1)];
        a.wrap[q] = wrap ? wrap[std::min(q, k - 1)] : 0.0f;
    }
    a.stride = (uint32_t)stride;
    a.iid = iid_.p + reps_h_[r].p0;
    a.n = (uint32_t)n;
    float *h[4];
    for (int q = 0; q < k; ++q) h[q] = const_cast<float *>(src[q]);
    return io_write(
        n * k, sizeof(float),
        [&](uint64_t i, uint32_t m, void *slot) { split_copy<false>(h, k, n, i, m, slot); },
        [&](uint64_t i, uint32_t m, void *slot) {
            hipLaunchKernelGGL(k_state_in, dim3(blocks(m)), dim3(kIoThreads), 0, stream_, a, i, m,
                               static_cast<const float *>(slot));
            return hipGetLastError() != hipSuccess;
        },
        err);
}

int Engine::io_force_out(int r, const float *fx, const float *fy, const float2 *cf,
                         float *ox, float *oy, std::string &err) {
    const size_t n = (size_t)nparticles(r);
    float *const dst[2] = {ox, oy};
    return io_read(
        2 * n, sizeof(float),
        [&](uint64_t i, uint32_t m, void *slot) {
            hipLaunchKernelGGL(k_force_out, dim3(blocks(m)), dim3(kIoThreads), 0, stream_, fx, fy, cf,
                               gather_ ? goff_.p : nullptr, iid_.p + reps_h_[r].p0, (uint32_t)n,
                               i, m, static_cast<float *>(slot));
            return hipGetLastError() != hipSuccess;
        },
        [&](uint64_t i, uint32_t m, void *slot) {
            float *s = static_cast<float *>(slot);
            for (int q = 0; q < 2; ++q) {  // (either may not be wanted)
                const size_t b = std::max<size_t>(i, q * n), e = std::min<size_t>(i + m, (q + 1) * n);
                if (b < e && dst[q]) std::memcpy(dst[q] + (b - q * n), s + (b - i), (e - b) * sizeof(float));
            }
        },
        err);
}

template <class T>
int Engine::io_out(size_t n, const T *src, const int32_t *idx, T *dst, std::string &err) {
    return io_read(
        n, sizeof(T),
        [&](uint64_t i, uint32_t m, void *slot) {
            hipLaunchKernelGGL(k_out<T>, dim3(blocks(m)), dim3(kIoThreads), 0, stream_, src, idx, i, m,
                               static_cast<T *>(slot));
            return hipGetLastError() != hipSuccess;
        },
        [&](uint64_t i, uint32_t m, void *slot) { std::memcpy(dst + i, slot, m * sizeof(T)); }, err);
}
template int Engine::io_out<double>(size_t, const double *, const int32_t *, double *, std::string &);
template int Engine::io_out<int32_t>(size_t, const int32_t *, const int32_t *, int32_t *, std::string &);

int Engine::io_in(size_t bytes, const void *src, void *dst, std::string &err) {
    return io_write(
        bytes, 1,
        [&](uint64_t i, uint32_t m, void *slot) {
            std::memcpy(slot, static_cast<const unsigned char *>(src) + i, m);
        },
        [&](uint64_t i, uint32_t m, void *slot) {
            return hipMemcpyAsync(static_cast<unsigned char *>(dst) + i, slot, m, hipMemcpyDefault,
                                  stream_) != hipSuccess;
        },
        err);
}

// The error word, and n <= kObsStride doubles of src, read with one kernel
// and one wait.
hipError_t Engine::launch_report(const double *src, int n) {
    hipLaunchKernelGGL(k_report, dim3(1), dim3(64), 0, stream_, err_.p, src, n, pin_.dhead());
    return hipGetLastError();
}

int Engine::io_report(const double *src, int n, std::string &err) {
    const int rc = check(launch_report(src, n), "report", err);
    return rc ? rc : io_wait(err);
}

int Engine::io_wait(std::string &err) {
    if (pin_.staged()) {
        const int rc = check(hipMemcpyAsync(pin_.p, pin_.d, sizeof(IoHead), hipMemcpyDeviceToHost, stream_),
                             "report", err);
        if (rc) return rc;
    }
    return check(hipStreamSynchronize(stream_), "step", err);
}

int Engine::launch_invert() {
    hipLaunchKernelGGL(k_invert, dim3((unsigned)kspans_h_.size()), dim3(kKickThreads), 0, stream_,
                       kspans_.p, reps_.p, uid_.p, iid_.p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace fm
