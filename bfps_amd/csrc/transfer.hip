// Host copies of fields and tracer rows.  Bound by the bus: 47 to 52 GB/s at
// 256^3 and more (pinned copies reach 57), by page faults of the caller's
// memory and threads below.
//
// The host layouts (component innermost, kx = n/2 stored, real rows ordered
// [z][y]) differ from the device's planes.  A host loop over every value,
// through a pageable buffer of the whole field, cost 60 to 90 times the
// transform it surrounded (128^3 FP32, 3 components: put + get 8.7 ms around
// 0.04 ms of transform).  Here kernels reorder: a chunk of the host layout at
// a time is written to (read from) pinned host memory, and threads copy
// between that and the caller's memory, each with a pinned slot of its own, so
// that kernels, bus transfers, page faults and copies of different chunks
// overlap.
#include <condition_variable>
#include <mutex>
#include <thread>

#include "ctx.hpp"

namespace {

constexpr size_t kSlotBytes = size_t(4) << 20;
constexpr int kMaxSlots = 8;

// Rows a chunk: a 32nd of the transfer (several chunks a thread, so that the
// last copy is short), at least 512 KB, at most a slot
size_t chunk_rows(size_t nrows, size_t row_bytes) {
    const size_t bytes = std::min(kSlotBytes, std::max(size_t(512) << 10, nrows * row_bytes / 32));
    return std::max<size_t>(1, bytes / row_bytes);
}

// Pinned slots of the process: at most kMaxSlots (32 MB), allocated when
// first needed, shared by every context (a transfer takes the free ones it
// can use and waits for the first), freed with the last context.
struct SlotPool {
    std::mutex mu;
    std::condition_variable cv;
    void* slot[kMaxSlots] = {};
    bool busy[kMaxSlots] = {};
    int users = 0;
};
SlotPool& pool() {
    static SlotPool* p = new SlotPool();  // outlives contexts destroyed at exit
    return *p;
}

// up to `want` slots; the first is waited for
int take_slots(int want, int (&got)[kMaxSlots], hipError_t* err) {
    SlotPool& P = pool();
    std::unique_lock<std::mutex> lk(P.mu);
    int n = 0;
    *err = hipSuccess;
    for (;;) {
        for (int i = 0; i < kMaxSlots && n < want; i++) {
            if (P.busy[i]) continue;
            if (!P.slot[i]) {
                *err = hipHostMalloc(&P.slot[i], kSlotBytes, hipHostMallocPortable);
                if (*err != hipSuccess) {
                    P.slot[i] = nullptr;
                    (void)hipGetLastError();
                    break;
                }
            }
            P.busy[i] = true;
            got[n++] = i;
        }
        if (n > 0) {
            *err = hipSuccess;
            return n;
        }
        bool any = false;
        for (bool b : P.busy) any |= b;
        if (!any) return 0;  // no slot could be allocated and none will be returned
        P.cv.wait(lk);
    }
}
void return_slots(const int (&got)[kMaxSlots], int n) {
    SlotPool& P = pool();
    {
        std::lock_guard<std::mutex> lk(P.mu);
        for (int i = 0; i < n; i++) P.busy[got[i]] = false;
    }
    P.cv.notify_all();
}

// Chunks 0..nchunks-1 through nt threads, thread t with slot t and chunks t,
// t + nt, ...; work(t, slot, event, k) returns a hipError_t, finish(event)
// waits for what a thread left in flight.
template <class W>
int run_chunks(bfpsh_ctx* ctx, size_t nchunks, W&& work) {
    int got[kMaxSlots];
    hipError_t err;
    const int nt = take_slots(int(std::min<size_t>(nchunks, kMaxSlots)), got, &err);
    if (nt == 0) return fail(ctx, BFPSH_EHIP, std::string("pinned staging memory: ") + hipGetErrorString(err));
    hipError_t errs[kMaxSlots] = {};
    auto body = [&](int t) {
        hipError_t e = hipSetDevice(ctx->device);
        hipEvent_t ev = nullptr;
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        for (size_t k = t; k < nchunks && e == hipSuccess; k += nt) e = work(pool().slot[got[t]], ev, k);
        // nothing of this slot stays in flight, whatever happened
        const hipError_t w = ev ? hipEventSynchronize(ev) : hipSuccess;
        if (e == hipSuccess) e = w;
        if (e != hipSuccess) (void)hipStreamSynchronize(ctx->stream);
        if (ev) (void)hipEventDestroy(ev);
        errs[t] = e;
    };
    std::thread th[kMaxSlots];
    bool here[kMaxSlots] = {};
    for (int t = 1; t < nt; t++) {
        try {
            th[t] = std::thread(body, t);
        } catch (...) {
            // no thread (or no memory for one) to be had: this one takes its
            // chunks.  Nothing may pass here: threads already started use
            // this frame
            here[t] = true;
        }
    }
    body(0);
    for (int t = 1; t < nt; t++) {
        if (here[t]) body(t);
        else th[t].join();
    }
    return_slots(got, nt);
    for (int t = 0; t < nt; t++)
        if (errs[t] != hipSuccess) return fail(ctx, BFPSH_EHIP, std::string("host copy: ") + hipGetErrorString(errs[t]));
    return BFPSH_OK;
}

// Rows of the host layout, `row_bytes` each, `nrows` of them: to the host
// through pack(slot, row0, rows), which enqueues the kernel that writes the
// rows to the slot, or from it through unpack(slot, row0, rows).
template <class F>
int rows_to_host(bfpsh_ctx* ctx, size_t nrows, size_t row_bytes, void* host, F&& pack) {
    const size_t per = chunk_rows(nrows, row_bytes);
    return run_chunks(ctx, (nrows + per - 1) / per, [&](void* slot, hipEvent_t ev, size_t k) -> hipError_t {
        const size_t r0 = k * per, nr = std::min(per, nrows - r0);
        pack(slot, r0, nr);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(ev, ctx->stream);
        if (e == hipSuccess) e = hipEventSynchronize(ev);
        if (e == hipSuccess) std::memcpy(static_cast<char*>(host) + r0 * row_bytes, slot, nr * row_bytes);
        return e;
    });
}
template <class F>
int rows_from_host(bfpsh_ctx* ctx, size_t nrows, size_t row_bytes, const void* host, F&& unpack) {
    const size_t per = chunk_rows(nrows, row_bytes);
    return run_chunks(ctx, (nrows + per - 1) / per, [&](void* slot, hipEvent_t ev, size_t k) -> hipError_t {
        const size_t r0 = k * per, nr = std::min(per, nrows - r0);
        hipError_t e = hipEventSynchronize(ev);  // the slot's previous chunk has been read
        if (e != hipSuccess) return e;
        std::memcpy(slot, static_cast<const char*>(host) + r0 * row_bytes, nr * row_bytes);
        unpack(slot, r0, nr);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(ev, ctx->stream);
        return e;
    });
}

// Host row r of a complex field, [ky][kz] = r, holds n/2 + 1 modes of NC
// components; of a real field, [z][y] = r, n points of NC components.  One
// thread per value of the host layout, so that the side on the bus is
// accessed in order; the planes are read (written) NC interleaved runs at a
// time, whole lines of which the L2 holds.  TO_HOST = false: host -> planes.
template <typename T, int NC, bool TO_HOST>
__global__ void __launch_bounds__(256)
k_rows_complex(C2<T>* planes, C2<T>* host, int n, uint32_t row0, uint32_t rows) {
    const uint32_t nxs = n / 2, len = (nxs + 1) * NC, total = rows * len;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const uint32_t r = i / len, j = i - r * len, x = j / NC, c = j - x * NC;
        C2<T>* p = planes + c * plane_size(n) + sphys(n, size_t(row0 + r) * nxs + (x < nxs ? x : 0));
        if (TO_HOST) host[i] = x < nxs ? *p : mk<T>(T(0), T(0));
        else if (x < nxs) *p = host[i];
    }
}
template <typename T, int NC, bool TO_HOST>
__global__ void __launch_bounds__(256) k_rows_real(T* planes, T* host, int n, uint32_t row0, uint32_t rows) {
    const uint32_t len = uint32_t(n) * NC, total = rows * len;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const uint32_t r = i / len, j = i - r * len, x = j / NC, c = j - x * NC;
        const uint32_t z = (row0 + r) / uint32_t(n), y = (row0 + r) - z * uint32_t(n);
        T* p = planes + (c * plane_size(n) + size_t(y) * row_stride(n)) * 2 + size_t(z) * n + x;
        if (TO_HOST) host[i] = *p;
        else *p = host[i];
    }
}
// rows of NC doubles in order[row0 ..] order
__global__ void __launch_bounds__(256)
k_gather_rows(const double* __restrict__ in, double* __restrict__ out, const uint32_t* __restrict__ order,
              uint32_t row0, uint32_t rows, uint32_t nc) {
    const uint32_t total = rows * nc;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const uint32_t r = i / nc;
        out[i] = in[size_t(order[row0 + r]) * nc + (i - r * nc)];
    }
}

unsigned grid_of(size_t values) { return unsigned(std::min<size_t>((values + 255) / 256, 4096)); }

template <typename T, int NC, bool TO_HOST>
int field_rows(bfpsh_ctx* ctx, bool real, void* planes, void* host) {
    const int n = ctx->n;
    const size_t nrows = size_t(n) * n, vals = size_t(real ? n : n / 2 + 1) * NC;
    const size_t row_bytes = vals * (real ? sizeof(T) : sizeof(C2<T>));
    auto go = [&](void* slot, size_t r0, size_t nr) {
        if (real)
            k_rows_real<T, NC, TO_HOST><<<grid_of(nr * vals), 256, 0, ctx->stream>>>((T*)planes, (T*)slot, n,
                                                                                    uint32_t(r0), uint32_t(nr));
        else
            k_rows_complex<T, NC, TO_HOST><<<grid_of(nr * vals), 256, 0, ctx->stream>>>((C2<T>*)planes, (C2<T>*)slot,
                                                                                        n, uint32_t(r0), uint32_t(nr));
    };
    if (TO_HOST) return rows_to_host(ctx, nrows, row_bytes, host, go);
    return rows_from_host(ctx, nrows, row_bytes, host, go);
}
template <typename T, bool TO_HOST>
int field_nc(bfpsh_ctx* ctx, bool real, int nc, void* planes, void* host) {
    return nc == 1   ? field_rows<T, 1, TO_HOST>(ctx, real, planes, host)
           : nc == 3 ? field_rows<T, 3, TO_HOST>(ctx, real, planes, host)
                     : field_rows<T, 9, TO_HOST>(ctx, real, planes, host);
}

}  // namespace

int bfpsh_field_to_host(bfpsh_ctx* ctx, bool real, int nc, const void* planes, void* host) {
    void* p = const_cast<void*>(planes);
    return ctx->prec == BFPSH_FP32 ? field_nc<float, true>(ctx, real, nc, p, host)
                                   : field_nc<double, true>(ctx, real, nc, p, host);
}
int bfpsh_field_from_host(bfpsh_ctx* ctx, bool real, int nc, void* planes, const void* host) {
    void* h = const_cast<void*>(host);
    return ctx->prec == BFPSH_FP32 ? field_nc<float, false>(ctx, real, nc, planes, h)
                                   : field_nc<double, false>(ctx, real, nc, planes, h);
}
int bfpsh_rows_to_host(bfpsh_ctx* ctx, const double* rows, int nc, double* host) {
    return rows_to_host(ctx, size_t(ctx->np), size_t(nc) * sizeof(double), host, [&](void* slot, size_t r0, size_t nr) {
        k_gather_rows<<<grid_of(nr * nc), 256, 0, ctx->stream>>>(rows, (double*)slot, ctx->d_order, uint32_t(r0),
                                                                 uint32_t(nr), uint32_t(nc));
    });
}
void bfpsh_transfer_open() {
    std::lock_guard<std::mutex> lk(pool().mu);
    pool().users++;
}
void bfpsh_transfer_close() {
    SlotPool& P = pool();
    std::lock_guard<std::mutex> lk(P.mu);
    if (--P.users > 0) return;
    for (int i = 0; i < kMaxSlots; i++)
        if (P.slot[i] && !P.busy[i]) {
            (void)hipHostFree(P.slot[i]);
            P.slot[i] = nullptr;
        }
}
