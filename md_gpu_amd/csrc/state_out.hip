// state_out.hip -- the state in the caller's atom order.
//   k_state_out   gathers a range of atoms from the sorted slots, wraps the positions as
//                 the list build does and writes [n][3] rows straight into pinned host memory
//   md_state_out  copies them from there to the caller's arrays while the next ranges arrive
//
// Bound by the host's side: the device writes pinned memory at the link's rate, a thread
// fills pageable memory at a few GB/s (page faults of new arrays included), so ranges of
// the atoms go to threads of their own, each with its own part of the arrays.  (Before: six
// blocking copies of padded arrays and an unpermuting loop on one thread.)  All three
// arrays of 256 atoms 19 us (before 96), 32,768: 84 (420), 196,608: 336 (2,334), 1.2 M: 1,460 (20,950).
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <new>
#include <system_error>
#include <thread>

#include "state_out.h"

namespace {

constexpr int TB = 256;
constexpr int MAXW = 8;

__global__ __launch_bounds__(TB) void k_state_out(const StateOutArgs a, int first, int n, float* px, float* pv,
                                                  float* pf) {
    __shared__ float row[3][3 * TB];
    const int b = blockIdx.x * TB, k = b + (int)threadIdx.x;
    if (k < n) {
        const int s = a.slot_of[first + k];
        const int r = a.nrep == 1 ? 0 : a.tile_rep[s / MD_TILE];
        if (px) {   // positions run unwrapped between list builds: wrap as the build does
            const float4 v = (cur_buf(a.st[r]) ? a.pos[1] : a.pos[0])[s];
            const RepParam& p = a.rep[r];
            row[0][3 * threadIdx.x] = wrap_coord(v.x, p.L[0], p.Linv[0]);
            row[0][3 * threadIdx.x + 1] = wrap_coord(v.y, p.L[1], p.Linv[1]);
            row[0][3 * threadIdx.x + 2] = wrap_coord(v.z, p.L[2], p.Linv[2]);
        }
        if (pv) {
            const float4 v = a.vel[s];
            row[1][3 * threadIdx.x] = v.x;
            row[1][3 * threadIdx.x + 1] = v.y;
            row[1][3 * threadIdx.x + 2] = v.z;
        }
        if (pf) {
            const float4 v = a.force[s];
            row[2][3 * threadIdx.x] = v.x;
            row[2][3 * threadIdx.x + 1] = v.y;
            row[2][3 * threadIdx.x + 2] = v.z;
        }
    }
    __syncthreads();
    // whole lines over the link: consecutive lanes write consecutive words
    const int nf = 3 * min(TB, n - b);
    for (int i = threadIdx.x; i < nf; i += TB) {
        if (px) px[3 * (size_t)b + i] = row[0][i];
        if (pv) pv[3 * (size_t)b + i] = row[1][i];
        if (pf) pf[3 * (size_t)b + i] = row[2][i];
    }
}

// The atoms cut into equal parts (one per thread, or one in all) and these into chunks of a
// slot; chunk c is the (c / parts)-th of part c % parts.
struct Plan {
    int natom, parts, per, chunk, nchunk, narr;
    size_t slot;
    float* out[3];
    char* base;
    int first(int c) const { return std::min(natom, (c % parts) * per + (c / parts) * chunk); }
    int count(int c) const {
        const int end = std::min(natom, (c % parts + 1) * per);
        return std::max(0, std::min(chunk, end - ((c % parts) * per + (c / parts) * chunk)));
    }
    float* row(int c, int k, int nslot) const {   // the k-th asked array in the chunk's slot
        return (float*)(base + (c % nslot) * slot + (size_t)k * chunk * 12);
    }
    void copy(int c, int nslot) const {
        const int f = first(c), n = count(c);
        int k = 0;
        for (float* o : out)
            if (o) memcpy(o + 3 * (size_t)f, row(c, k++, nslot), (size_t)n * 12);
    }
};

int cpus() {
    cpu_set_t s;
    return sched_getaffinity(0, sizeof s, &s) == 0 ? CPU_COUNT(&s) : 1;
}

}  // namespace

void HostRing::release() {
    for (auto& e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (p) (void)hipHostFree(p);
    p = nullptr;
    bytes = 0;
}

hipError_t HostRing::open(size_t want, bool events) {
    hipError_t h = hipSuccess;
    if (bytes < want) {
        if (p) (void)hipHostFree(p);
        bytes = 0;
        want = (want + 4095) / 4096 * 4096;
        if ((h = hipHostMalloc((void**)&p, want, hipHostMallocCoherent)) != hipSuccess) {
            p = nullptr;
            return h;
        }
        bytes = want;
    }
    for (int k = 0; k < (events ? NS : 0) && h == hipSuccess; k++)
        if (!ev[k]) h = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming | hipEventReleaseToSystem);
    return h;
}

hipError_t md_state_out(const StateOutArgs& a, float* const outs[3], HostRing& ring, hipStream_t st) {
    Plan p{};
    p.natom = a.natom;
    for (int k = 0; k < 3; k++) {
        p.out[k] = outs[k];
        p.narr += outs[k] != nullptr;
    }
    if (p.narr == 0 || a.natom < 1) return hipStreamSynchronize(st);
    std::lock_guard<std::mutex> hold(ring.use);
    const size_t bytes = (size_t)a.natom * 12 * p.narr;
    const int most = (int)(HostRing::SLOT / (12 * p.narr)) & ~15;   // atoms of a chunk
    int slots = 1;
    auto cut = [&](int parts) -> hipError_t {   // multiples of 16 atoms: rows of a slot stay 64-byte aligned
        p.parts = parts;
        p.per = ((a.natom + parts - 1) / parts + 15) & ~15;
        const int rounds = (p.per + most - 1) / most;
        p.chunk = ((p.per + rounds - 1) / rounds + 15) & ~15;
        p.nchunk = parts * ((p.per + p.chunk - 1) / p.chunk);
        p.slot = (size_t)p.chunk * 12 * p.narr;
        const hipError_t e = ring.open(std::min(p.nchunk, HostRing::NS) * p.slot, p.nchunk > 1);
        slots = (int)std::min<size_t>(HostRing::NS, ring.bytes / p.slot);
        p.base = ring.p;
        return e;
    };

    // a thread per 512 KB: starting one costs some 20 us, as much as copying 100 KB
    struct Lane {
        alignas(64) std::atomic<int> ready{0};
        std::atomic<int> done{0};
    } lane[MAXW];
    std::atomic<int> go{0};   // 1: the plan is set, -1: give up
    std::thread th[MAXW];
    const int want = std::min((int)std::min<size_t>(MAXW, bytes / HostRing::SLOT), cpus() - 1);
    int nth = 0;
    hipError_t h = cut(std::max(1, want));
    if (h != hipSuccess) return h;
    if (want >= 2) {
        const Plan* pp = &p;
        for (; nth < want; nth++) {
            Lane* l = &lane[nth];
            const int w = nth;
            try {
                th[nth] = std::thread([pp, &slots, l, w, &go]() {
                    while (go.load(std::memory_order_acquire) == 0) std::this_thread::yield();
                    for (int c = w, j = 0; go.load(std::memory_order_relaxed) > 0 && c < pp->nchunk; c += pp->parts, j++) {
                        while (l->ready.load(std::memory_order_acquire) <= j) {
                            if (go.load(std::memory_order_relaxed) < 0) return;
                            std::this_thread::yield();
                        }
                        pp->copy(c, slots);
                        l->done.store(j + 1, std::memory_order_release);
                    }
                });
            } catch (const std::system_error&) {   // no more threads to be had
                break;
            } catch (const std::bad_alloc&) {
                break;
            }
        }
    }
    if (nth < want && want >= 2) h = cut(std::max(1, nth));
    if (nth) go.store(1, std::memory_order_release);

    const int ahead = p.nchunk <= slots ? p.nchunk : std::max(1, slots / 2);   // chunks queued at a time
    auto launch = [&](int c) -> hipError_t {
        const int n = p.count(c);
        if (n > 0) {
            float* o[3];
            int k = 0;
            for (int i = 0; i < 3; i++) o[i] = outs[i] ? p.row(c, k++, slots) : nullptr;
            hipLaunchKernelGGL(k_state_out, dim3((n + TB - 1) / TB), dim3(TB), 0, st, a, p.first(c), n, o[0], o[1], o[2]);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        return p.nchunk > 1 ? hipEventRecord(ring.ev[c % slots], st) : hipSuccess;
    };
    for (int c = 0; c < ahead && h == hipSuccess; c++) h = launch(c);
    for (int c = 0; c < p.nchunk && h == hipSuccess; c++) {
        h = p.nchunk > 1 ? hipEventSynchronize(ring.ev[c % slots]) : hipStreamSynchronize(st);
        if (h != hipSuccess) break;
        if (nth) {
            lane[c % p.parts].ready.store(c / p.parts + 1, std::memory_order_release);
        } else {
            p.copy(c, slots);
        }
        const int m = c + ahead;
        if (m < p.nchunk) {
            const int old = m - slots;   // the chunk that had this slot
            if (nth && old >= 0)
                while (lane[old % p.parts].done.load(std::memory_order_acquire) <= old / p.parts) std::this_thread::yield();
            h = launch(m);
        }
    }
    if (h != hipSuccess) go.store(-1, std::memory_order_release);
    for (int w = 0; w < nth; w++) th[w].join();
    if (h != hipSuccess) (void)hipStreamSynchronize(st);   // nothing queued writes the ring after this
    return h;
}
