// Readback: particle state in id order, straight into host memory.
//
// The device keeps particles in slot order (by cell) in its working
// precision; a reader wants them by id in FP64 (Space.positions, the
// particle records engine_fromCUDA leaves, tfRunner_cuda.cu:4329-4520).  One
// kernel per chunk of ids gathers the slots, converts, and writes each field
// as contiguous rows into a pinned host buffer over the bus; the host only
// copies finished rows to the caller.  What bounds it is the bus (24 B per
// particle for positions) and, past a few MB, the page faults of the
// caller's fresh buffer, so large reads are cut into chunks that several
// threads gather and copy at the same time, each with its own buffer.
// Before, every read copied all state arrays through pageable memory and
// gathered them in one host thread: 2,000,000 positions took 87 ms.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "ensemble.h"

namespace tfg {

namespace {

// Chunks of 2 MB keep a kernel's launch small against its transfer (1 MB
// chunks: 1,000,000 positions in 1.8 ms, 2 MB 1.4 ms, 4 MB 1.4 ms, one
// thread).  Up to kReadSerial bytes the calling thread reads alone, gathering
// one chunk while it copies the one before: more threads save little there
// and wait for each other on a busy host (250,000 records, 21 MB: 1.5 ms
// alone, 1.6 to 6 ms with four).  Above it four threads read (2,000,000
// positions 2.8 -> 1.3 ms; eight 1.3 ms).
constexpr size_t kReadChunk = static_cast<size_t>(2) << 20;
constexpr size_t kReadSerial = static_cast<size_t>(24) << 20;
constexpr int kReadThreads = 4;

constexpr int kReadBlock = 256;   // particles per block

// One field of a record: rows of W values for the block's particles, laid
// out through LDS so that the block writes them contiguously.
template <int W, typename T, typename T0>
__device__ inline void put_rows(T *out, int first, int n, const T0 (&v)[W], T *lds) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < W; k++) lds[threadIdx.x * W + k] = static_cast<T>(v[k]);
    __syncthreads();
    for (int t = threadIdx.x; t < n * W; t += kReadBlock) out[static_cast<size_t>(first) * W + t] = lds[t];
}

// The rows from particle p on (kept.ns species per row).
__host__ __device__ inline ReadRows kept_at(const ReadRows &kept, size_t p) {
    ReadRows r = kept;
    r.x += 3 * p;
    r.v += 3 * p;
    r.f += 4 * p;
    r.cid += p;
    r.flags += p;
    if (r.ns > 0) {
        r.sp += r.ns * p;
        r.q += r.ns * p;
    }
    return r;
}

// Ids [id0, id0 + n) of a system into the rows of o (null fields skipped), by
// the block of ids b0 / kReadBlock.  Positions follow the host's arithmetic:
// stored + frame offset, then (origin + loc h) + x, each rounded once.
template <typename real>
__device__ inline void read_block(const KP<real> &P, const SysDesc &sd, int id0, int n, int b0, const ReadRows &o, double *lds) {
#pragma clang fp contract(off)
    const bool from_a = P.list_mode && P.lflags[3] != 0;   // in-place updates leave B behind A
    const typename V<real>::v4 *pos = from_a ? P.A.pos : P.B.pos;
    const typename V<real>::v4 *vel = from_a ? P.A.vel : P.B.vel;
    const int4 *meta = from_a ? P.A.meta : P.B.meta;
    const real *sp = from_a ? P.A.sp : P.B.sp, *q = from_a ? P.A.q : P.B.q;
    const int nb = min(kReadBlock, n - b0);
    const bool valid = static_cast<int>(threadIdx.x) < nb;
    const int slot = P.slot_of[sd.p_off + id0 + b0 + (valid ? static_cast<int>(threadIdx.x) : 0)];
    const int4 m = meta[slot];
    const int cid = m.z - sd.cell_off;
    if (o.xg || o.x) {
        const typename V<real>::v4 p = pos[slot];
        const double x[3] = {static_cast<double>(p.x) + sd.foff[0], static_cast<double>(p.y) + sd.foff[1],
                             static_cast<double>(p.z) + sd.foff[2]};
        if (o.xg) {
            int loc[3];
            cell_loc(cid, sd, loc);
            double g[3];
            for (int k = 0; k < 3; k++) g[k] = (o.origin[k] + loc[k] * sd.h[k]) + x[k];
            put_rows<3>(o.xg, b0, nb, g, lds);
        }
        if (o.x) put_rows<3>(o.x, b0, nb, x, lds);
    }
    if (o.v) {
        const typename V<real>::v4 v = vel[slot];
        const double w[3] = {static_cast<double>(v.x), static_cast<double>(v.y), static_cast<double>(v.z)};
        put_rows<3>(o.v, b0, nb, w, lds);
    }
    if (o.f) {
        const typename V<real>::v4 f = P.force[slot];
        const double w[4] = {static_cast<double>(f.x), static_cast<double>(f.y), static_cast<double>(f.z),
                             static_cast<double>(f.w)};
        put_rows<4>(o.f, b0, nb, w, lds);
    }
    if (valid) {
        const int row = b0 + static_cast<int>(threadIdx.x);
        if (o.cid) o.cid[row] = cid;
        if (o.flags) o.flags[row] = static_cast<int>(static_cast<unsigned>(m.x) >> 16);
        for (int k = 0; k < o.ns; k++) {
            if (o.sp) o.sp[static_cast<size_t>(row) * o.ns + k] = static_cast<double>(sp[static_cast<size_t>(k) * P.np + slot]);
            if (o.q) o.q[static_cast<size_t>(row) * o.ns + k] = static_cast<double>(q[static_cast<size_t>(k) * P.np + slot]);
        }
    }
}

template <typename real> __global__ __launch_bounds__(kReadBlock) void k_read(KP<real> P, int s, int id0, int n, ReadRows o) {
    __shared__ double lds[kReadBlock * 4];
    read_block<real>(P, P.sys[s], id0, n, blockIdx.x * kReadBlock, o, lds);
}

// The marked ones of kKeepGroup members into the kept arrays (id order over the
// ensemble, P.S species per row), in one launch: a launch per member cost the
// step after the reads of 49 members 0.15 ms.
constexpr int kKeepGroup = 256;
struct Marks {
    unsigned bits[kKeepGroup / 32];
};
template <typename real> __global__ __launch_bounds__(kReadBlock) void k_keep(KP<real> P, int first, Marks marks, ReadRows kept) {
    __shared__ double lds[kReadBlock * 4];
    const int g = blockIdx.y;
    if ((marks.bits[g >> 5] >> (g & 31) & 1u) == 0) return;
    const SysDesc &sd = P.sys[first + g];
    const int b0 = blockIdx.x * kReadBlock;
    if (b0 >= sd.np) return;
    read_block<real>(P, sd, 0, sd.np, b0, kept_at(kept, sd.p_off), lds);
}

int launch_read(DeviceEnsemble *E, int s, int id0, int n, const ReadRows &o, hipStream_t stream) {
    const dim3 g((n + kReadBlock - 1) / kReadBlock), b(kReadBlock);
    if (E->precision == PREC_MIXED)
        hipLaunchKernelGGL(k_read<float>, g, b, 0, stream, make_params<float>(E, 0), s, id0, n, o);
    else
        hipLaunchKernelGGL(k_read<double>, g, b, 0, stream, make_params<double>(E, 0), s, id0, n, o);
    return launch_error("readback");
}

int launch_keep(DeviceEnsemble *E, int first, int count, int most, const Marks &m) {
    const dim3 g((most + kReadBlock - 1) / kReadBlock, count), b(kReadBlock);
    if (E->precision == PREC_MIXED)
        hipLaunchKernelGGL(k_keep<float>, g, b, 0, E->stream, make_params<float>(E, 0), first, m, E->kept);
    else
        hipLaunchKernelGGL(k_keep<double>, g, b, 0, E->stream, make_params<double>(E, 0), first, m, E->kept);
    return launch_error("kept reads");
}

// The wanted fields of o (non-null) laid one after the other in a buffer for
// n particles; returns its size in bytes.
size_t place_rows(const ReadRows &want, unsigned char *base, int n, ReadRows *o) {
    *o = want;
    size_t at = 0;
    auto put = [&](auto *&p, int w) {
        if (!p) return;
        p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(base + at);
        at += (static_cast<size_t>(n) * w * sizeof(*p) + 15) & ~static_cast<size_t>(15);
    };
    put(o->xg, 3);
    put(o->x, 3);
    put(o->v, 3);
    put(o->f, 4);
    put(o->sp, o->ns);
    put(o->q, o->ns);
    put(o->cid, 1);
    put(o->flags, 1);
    return at;
}

void copy_rows(const ReadRows &from, const ReadRows &to, int first, int n) {
    auto put = [&](auto *dst, const auto *src, int w) {
        if (dst) std::memcpy(dst + static_cast<size_t>(first) * w, src, static_cast<size_t>(n) * w * sizeof(*src));
    };
    put(to.xg, from.xg, 3);
    put(to.x, from.x, 3);
    put(to.v, from.v, 3);
    put(to.f, from.f, 4);
    put(to.sp, from.sp, from.ns);
    put(to.q, from.q, from.ns);
    put(to.cid, from.cid, 1);
    put(to.flags, from.flags, 1);
}

// The calling thread's device for the length of a read.
struct OnDevice {
    int before = -1;
    explicit OnDevice(int device) {
        if (hipGetDevice(&before) != hipSuccess) before = -1;
        if (before != device) (void)hipSetDevice(device);
        else before = -1;
    }
    ~OnDevice() {
        if (before >= 0) (void)hipSetDevice(before);
    }
};

}  // namespace

// Reads every particle of system s: the wanted fields of each chunk of ids
// are gathered into a pinned buffer and handed to use(rows, first id, count),
// which may run on several threads at once for different chunks.  The caller
// holds read_lock.
template <typename Use> static int read_system(DeviceEnsemble *E, int s, ReadRows want, Use &&use) {
    const OnDevice on(E->device);
    const int n = E->sys[s].np;
    for (int k = 0; k < 3; k++) want.origin[k] = E->engines[s]->geom.origin[k];
    ReadRows probe;
    const size_t per = place_rows(want, nullptr, 1024, &probe) / 1024 + 1;   // bytes per particle, rounded up
    int chunk = static_cast<int>(kReadChunk / per) & ~(kReadBlock - 1);
    chunk = std::min(std::max(chunk, kReadBlock), n);
    const int nchunks = (n + chunk - 1) / chunk;
    int threads = 1;
    if (per * n > kReadSerial)
        threads = std::max(1, std::min({kReadThreads, static_cast<int>(std::thread::hardware_concurrency()), nchunks}));
    // pinned buffers, grown on first use, and an event each: one per thread,
    // two for a lone one
    const int depth = threads == 1 ? std::min(2, nchunks) : 1;
    const size_t need = place_rows(want, nullptr, chunk, &probe);
    for (int t = 0; t < threads * depth; t++) {
        DeviceEnsemble::ReadSlot &slot = E->read_slot[t];
        if (slot.bytes < need) {
            if (slot.ptr) (void)hipHostFree(slot.ptr);
            slot.ptr = nullptr;
            slot.bytes = 0;
            const size_t bytes = (need + 65535) & ~static_cast<size_t>(65535);
            void *p = nullptr;
            TFG_HIP(hipHostMalloc(&p, bytes, hipHostMallocDefault));
            slot.ptr = static_cast<unsigned char *>(p);
            slot.bytes = bytes;
        }
        if (!slot.done) TFG_HIP(hipEventCreateWithFlags(&slot.done, hipEventDisableTiming));
    }
    std::atomic<int> failed{TFG_OK};
    std::string msg;
    // thread t takes chunks t, t + threads, ...
    auto work = [&](int t) {
        auto slot_of = [&](int c) -> const DeviceEnsemble::ReadSlot & { return E->read_slot[t * depth + c / threads % depth]; };
        auto rows_of = [&](int c) {
            ReadRows rows;
            place_rows(want, slot_of(c).ptr, std::min(chunk, n - c * chunk), &rows);
            return rows;
        };
        int ahead = t;
        for (int c = t; c < nchunks && failed.load(std::memory_order_relaxed) == TFG_OK; c += threads) {
            int rc = TFG_OK;
            for (; rc == TFG_OK && ahead < nchunks && ahead < c + depth * threads; ahead += threads) {
                rc = launch_read(E, s, ahead * chunk, std::min(chunk, n - ahead * chunk), rows_of(ahead), E->stream);
                const hipError_t e = hipEventRecord(slot_of(ahead).done, E->stream);
                if (rc == TFG_OK && e != hipSuccess)
                    rc = set_error(TFG_E_DEVICE, std::string("readback: ") + hipGetErrorString(e));
            }
            if (rc == TFG_OK) {
                const hipError_t e = hipEventSynchronize(slot_of(c).done);
                if (e != hipSuccess) rc = set_error(TFG_E_DEVICE, std::string("readback: ") + hipGetErrorString(e));
            }
            if (rc != TFG_OK) {
                int none = TFG_OK;
                if (failed.compare_exchange_strong(none, rc)) msg = last_error();   // read after the join
                return;
            }
            use(rows_of(c), c * chunk, std::min(chunk, n - c * chunk));
        }
    };
    std::vector<std::thread> pool;
    try {
        for (int t = 1; t < threads; t++)
            pool.emplace_back([&, t] {
                (void)hipSetDevice(E->device);
                work(t);
            });
    } catch (...) {   // no more threads: the calling one takes the remaining parts
    }
    work(0);
    for (int t = static_cast<int>(pool.size()) + 1; t < threads; t++) work(t);
    for (std::thread &th : pool) th.join();
    const int rc = failed.load();
    return rc != TFG_OK ? set_error(rc, msg) : TFG_OK;
}

static void record_rows(Engine &e, const ReadRows &r, int first, int n) {
    for (int k = 0; k < n; k++) {
        HostParticle &hp = e.parts[first + k];
        for (int a = 0; a < 3; a++) {
            hp.x[a] = r.x[3 * k + a];
            hp.v[a] = r.v[3 * k + a];
        }
        for (int a = 0; a < 4; a++) hp.f[a] = r.f[4 * k + a];
        hp.cid = r.cid[k];
        hp.flags = static_cast<uint32_t>(r.flags[k]);
    }
    if (r.ns > 0) {
        std::copy(r.sp, r.sp + static_cast<size_t>(n) * r.ns, e.species.begin() + static_cast<size_t>(first) * r.ns);
        std::copy(r.q, r.q + static_cast<size_t>(n) * r.ns, e.species_q.begin() + static_cast<size_t>(first) * r.ns);
    }
}

static int read_into_engine_locked(DeviceEnsemble *E, int s) {
    Engine &e = *E->engines[s];
    double some = 0;
    int some_i = 0;
    ReadRows want;   // every field of the host record
    want.x = want.v = want.f = &some;
    want.cid = want.flags = &some_i;
    want.ns = e.nspecies;
    if (e.nspecies > 0) want.sp = want.q = &some;
    const int rc = read_system(E, s, want, [&](const ReadRows &r, int first, int n) { record_rows(e, r, first, n); });
    if (rc == TFG_OK && E->keep_reads) E->kept_sys[s] = kReadNone;   // the host record is newer
    return rc;
}

int read_into_engine(DeviceEnsemble *E, int s) {
    const std::lock_guard<std::mutex> hold(E->read_lock);
    return read_into_engine_locked(E, s);
}

void ensemble_keep_reads(DeviceEnsemble *E) {
    E->keep_reads = true;
    E->kept_sys.assign(E->nsys, kReadNone);
}

// The kept arrays, one block, on first use; false without device memory for it.
static bool kept_alloc(DeviceEnsemble *E) {
    if (E->kept.x) return true;
    const size_t n = static_cast<size_t>(E->np);
    double *p = nullptr;
    if (E->buf.alloc(&p, n * (11 + 2 * E->S)) != TFG_OK) {
        (void)hipGetLastError();   // the caller goes on without it
        return false;
    }
    ReadRows &k = E->kept;
    k.x = p;
    k.v = k.x + 3 * n;
    k.f = k.v + 3 * n;
    k.sp = k.f + 4 * n;
    k.q = k.sp + n * E->S;
    k.cid = reinterpret_cast<int *>(k.q + n * E->S);
    k.flags = k.cid + n;
    k.ns = E->S;
    return true;
}

// A read copies nothing for later: the state of the members read is kept here,
// by the next call that changes it (sweeps read every member between two
// steps, and a gather behind each read delayed the next one).  Without device
// memory the host engines take it now.
int keep_reads(DeviceEnsemble *E) {
    if (!E->keep_reads) return TFG_OK;
    const std::lock_guard<std::mutex> hold(E->read_lock);
    if (std::find(E->kept_sys.begin(), E->kept_sys.end(), kReadCurrent) == E->kept_sys.end()) return TFG_OK;
    const bool device = kept_alloc(E);
    for (int first = 0; first < E->nsys; first += kKeepGroup) {
        const int count = std::min(kKeepGroup, E->nsys - first);
        Marks marks{};
        int most = 0, rc;
        for (int g = 0; g < count; g++) {
            char &state = E->kept_sys[first + g];
            if (state != kReadCurrent) continue;
            if (!device) {
                if ((rc = read_into_engine_locked(E, first + g)) != TFG_OK) return rc;
                continue;
            }
            marks.bits[g >> 5] |= 1u << (g & 31);
            most = std::max(most, E->sys[first + g].np);
            state = kReadKept;
        }
        if (most > 0 && (rc = launch_keep(E, first, count, most, marks)) != TFG_OK) return rc;
    }
    return TFG_OK;
}

int restore_kept(DeviceEnsemble *E) {
    const std::lock_guard<std::mutex> hold(E->read_lock);
    for (int s = 0; s < static_cast<int>(E->kept_sys.size()); s++) {
        if (E->kept_sys[s] == kReadCurrent) {
            const int rc = read_into_engine_locked(E, s);
            if (rc != TFG_OK) return rc;
        }
        if (E->kept_sys[s] != kReadKept) continue;
        const OnDevice on(E->device);
        Engine &e = *E->engines[s];
        const size_t n = static_cast<size_t>(E->sys[s].np);
        const ReadRows d = kept_at(E->kept, E->sys[s].p_off);
        const size_t S = d.ns;
        std::vector<double> x(3 * n), v(3 * n), f(4 * n), sp(n * S), q(n * S);
        std::vector<int> cid(n), flags(n);
        ReadRows h;
        h.x = x.data(), h.v = v.data(), h.f = f.data(), h.sp = sp.data(), h.q = q.data();
        h.cid = cid.data(), h.flags = flags.data();
        h.ns = e.nspecies;
        TFG_HIP(hipStreamSynchronize(E->stream));
        TFG_HIP(hipMemcpy(h.x, d.x, 3 * n * sizeof(double), hipMemcpyDeviceToHost));
        TFG_HIP(hipMemcpy(h.v, d.v, 3 * n * sizeof(double), hipMemcpyDeviceToHost));
        TFG_HIP(hipMemcpy(h.f, d.f, 4 * n * sizeof(double), hipMemcpyDeviceToHost));
        TFG_HIP(hipMemcpy(h.cid, d.cid, n * sizeof(int), hipMemcpyDeviceToHost));
        TFG_HIP(hipMemcpy(h.flags, d.flags, n * sizeof(int), hipMemcpyDeviceToHost));
        if (S > 0) {
            TFG_HIP(hipMemcpy(h.sp, d.sp, n * S * sizeof(double), hipMemcpyDeviceToHost));
            TFG_HIP(hipMemcpy(h.q, d.q, n * S * sizeof(double), hipMemcpyDeviceToHost));
        }
        for (size_t p = 0, ns = h.ns; ns < S && p < n; p++)   // the ensemble's species per row: the member's
            for (size_t k = 0; k < ns; k++) {
                h.sp[p * ns + k] = h.sp[p * S + k];
                h.q[p * ns + k] = h.q[p * S + k];
            }
        record_rows(e, h, 0, static_cast<int>(n));
    }
    return TFG_OK;
}

int ensemble_read(DeviceEnsemble *E, int s, const ReadRows &out) {
    if (s < 0 || s >= E->nsys) return set_error(TFG_E_RANGE, "system index out of range");
    const std::lock_guard<std::mutex> hold(E->read_lock);
    const int rc = read_system(E, s, out, [&](const ReadRows &rows, int first, int n) { copy_rows(rows, out, first, n); });
    if (rc == TFG_OK && E->keep_reads) {
        E->kept_sys[s] = kReadCurrent;
        E->engines[s]->energies = energies_of(E->status_sums() + 5 * s);
    }
    return rc;
}

}  // namespace tfg
