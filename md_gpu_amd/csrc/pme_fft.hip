// pme_fft.hip -- the transforms of smooth PME with the influence function between
// them, in three kernels instead of the FFT library's four to eight and a convolution
// pass (which stay for the grids this does not take, pme.hip).
//   k_pme_fwd   a workgroup per x plane: real-to-complex along z (two real rows as one
//               complex one, so odd lengths need no special case), then along y
//   k_pme_xconv a workgroup per 16 columns: forward along x, multiplication by the
//               influence function C(m) = qfac exp(-pi^2 m^2/b^2) B(m) / (pi V m^2) with
//               the energy and traced-virial sums (when asked for), inverse along x
//   k_pme_inv   a workgroup per x plane: inverse along y, complex-to-real along z
// The passes run between two LDS buffers (md_fft.h); the spectrum is [K0][K1][K2/2 + 1].
// The forward butterflies compute in FP64 between values stored in FP32: the charges'
// spectrum is smallest where the influence function is largest (low m), so the white
// rounding noise of that half weighs most in the forces.
//
// Bound by latency: the grids are 3.5 to 8 MB, resident in cache; a plane's passes are
// LDS round trips with a barrier each, on one CU per plane, and their straight-line
// butterflies are fetched anew by every launch (so large radices, few passes, and each
// radix once per kernel: with the passes of z and y as separate code 34 us instead of 28
// for the three kernels at 96^3 in FP32).  96^3: 30 us, before 50 us (hipFFT's six
// kernels and the convolution pass); 128^3: 44 (62); 45^3: 21 (44).  512 threads per plane
// instead of 1,024: 31.5 and 47; radices up to 8 instead of 16: 36 and 55.
#include <algorithm>

#include "md_device.h"
#include "md_fft.h"
#include "md_reduce.h"

namespace {

constexpr int TP = 1024;  // threads per plane
constexpr int NV = 4;     // 16-byte loads in flight per thread of a plane
constexpr int TX = 256;   // threads per column group
constexpr int XB = 16;    // columns per workgroup (128 bytes of a row)

__device__ __forceinline__ bool go_step(const PmeArgs& a) {
    const RepState s = a.st[0];
    if (a.mode == MODE_FORCE) return !stale(s);
    if (a.mode == MODE_LF) return !stale(s) && s.step < s.target;
    return s.phase == 1 && !stale(s);
}

template <class T>
__device__ __forceinline__ fft::Cx<T> turn_at(const double2* tw, int k) { return {(T)tw[k].x, (T)tw[k].y}; }

__device__ __forceinline__ float2 swapped(float2 v) { return make_float2(v.y, v.x); }

// Pass q of plan p from LDS buffer s to d, then the two swapped: element i of line l at
// l * ls + i * es.  Called at one place per kernel, in a loop over all of its passes: the
// butterflies are straight-line code, fetched anew by every launch (the kernels of a step
// do not fit the instruction cache together), so each radix stands in a kernel once.
template <class T>
__device__ __forceinline__ void run_pass(const FftPlan& p, int q, const fft::Div& lines, int ls, int es,
                                         const fft::Cx<T>* tw, float2*& s, float2*& d) {
    const float2* src = s;
    float2* dst = d;
    fft::pass_any(p, q, lines, tw, (int)threadIdx.x, (int)blockDim.x,
                  [=](int l, int j, int t) { return src[fft::mul24(l, ls) + fft::mul24(j, es) + t * es]; },
                  [=](int l, int o, int t, float2 v) { dst[fft::mul24(l, ls) + fft::mul24(o, es) + t * es] = v; });
    __syncthreads();
    s = dst;
    d = const_cast<float2*>(src);
}

}  // namespace

__global__ __launch_bounds__(TP) void k_pme_fwd(const PmeArgs a, const PmeFftArgs f) {
    typedef fft::Cx<double> Cx;
    extern __shared__ float2 s_fft[];
    const int tid = threadIdx.x, x = blockIdx.x;
    const int K1 = a.K1, K2 = a.K2, H = K2 / 2 + 1, rows = (K1 + 1) / 2, pz = K2 | 1, py = H | 1;
    Cx* tw1 = reinterpret_cast<Cx*>(s_fft + 2 * f.plane);
    Cx* tw2 = tw1 + K1;
    float2 *s = s_fft, *d = s_fft + f.plane;
    const float* __restrict__ q = a.qgrid + (size_t)x * K1 * K2;
    const fft::Div dz = f.dk2, d4 = f.dk24, dh = f.dh;
    // rows of whole float4s: NV of them in flight per thread, the first ones with the state
    const bool vec = (K2 & 3) == 0;
    const int n4 = vec ? K1 * (K2 / 4) : 1;
    float4 v[NV];
    auto load = [&](int u0) {
#pragma unroll
        for (int k = 0; k < NV; k++) v[k] = reinterpret_cast<const float4*>(q)[min(u0 + k * TP, n4 - 1)];
    };
    if (vec) load(tid);
    for (int k = tid; k < K1 + K2; k += TP) tw1[k] = turn_at<double>(f.tw, a.K0 + k);
    if (!go_step(a)) return;   // grid-uniform
    if (vec) {
        for (int u0 = tid; u0 < n4; u0 += NV * TP) {
            if (u0 != tid) load(u0);
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const int u = u0 + k * TP;
                if (u >= n4) break;
                const int y = d4.quot(u), z = 4 * (u - y * (K2 / 4));
                float* t = reinterpret_cast<float*>(s + (y >> 1) * pz + z) + (y & 1);
                t[0] = v[k].x;
                t[2] = v[k].y;
                t[4] = v[k].z;
                t[6] = v[k].w;
            }
        }
        if (K1 & 1)
            for (int z = tid; z < K2; z += TP) s[(rows - 1) * pz + z].y = 0.0f;   // the last row has no partner
    } else {
#pragma unroll 4
        for (int u = tid; u < rows * K2; u += TP) {
            const int r = dz.quot(u), z = u - r * K2;
            const float re = q[2 * r * K2 + z];
            const float im = 2 * r + 1 < K1 ? q[(2 * r + 1) * K2 + z] : 0.0f;
            s[r * pz + z] = make_float2(re, im);
        }
    }
    __syncthreads();
    const int nz = f.p2.npass, ny = f.p1.npass;
    for (int q = 0; q < nz + ny; q++) {   // along z, then along y
        const bool z = q < nz;
        run_pass(z ? f.p2 : f.p1, z ? q : q - nz, z ? f.drow : f.dh, z ? pz : 1, z ? 1 : py, (const Cx*)(z ? tw2 : tw1), s, d);
        if (q != nz - 1) continue;
        // the two rows' half spectra: (Z(k) + conj Z(N - k)) / 2 and (Z(k) - conj Z(N - k)) / 2i
        for (int u = tid; u < rows * H; u += TP) {
            const int r = dh.quot(u), k = u - r * H;
            const float2 A = s[r * pz + k], B = s[r * pz + (k ? K2 - k : 0)];
            d[2 * r * py + k] = make_float2(0.5f * (A.x + B.x), 0.5f * (A.y - B.y));
            if (2 * r + 1 < K1) d[(2 * r + 1) * py + k] = make_float2(0.5f * (A.y + B.y), 0.5f * (B.x - A.x));
        }
        __syncthreads();
        float2* t = s;
        s = d;
        d = t;
    }
    float2* __restrict__ out = a.sgrid + (size_t)x * K1 * H;
    for (int u = tid; u < K1 * H; u += TP) {
        const int y = dh.quot(u);
        out[u] = s[y * py + u - y * H];
    }
}

template <bool EN>
__global__ __launch_bounds__(TX) void k_pme_xconv(const PmeArgs a, const PmeFftArgs f) {
    typedef fft::Cx<double> Cx;
    extern __shared__ float2 s_fft[];
    __shared__ float4 s_col[XB];   // per column: m1, m2, |b1|^2, |b2|^2
    __shared__ double s_red[TX / 64][2];
    const int tid = threadIdx.x;
    const int K0 = a.K0, H = a.K2 / 2 + 1, M = a.K1 * H, c0 = blockIdx.x * XB;
    const RepParam& p = a.rep[0];
    Cx* tw = reinterpret_cast<Cx*>(s_fft + 2 * K0 * XB);
    float2 *s = s_fft, *d = s_fft + K0 * XB;
    const int l0 = tid & (XB - 1);
    const float2* __restrict__ in = a.sgrid + min(c0 + l0, M - 1);
    float2 v[8];
    auto load = [&](int i0) {   // the first ones with the state
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = in[(size_t)min(i0 + k * (TX / XB), K0 - 1) * M];
    };
    load(tid / XB);
    for (int k = tid; k < K0; k += TX) tw[k] = turn_at<double>(f.tw, k);
    if (tid < XB) {
        const int c = min(c0 + tid, M - 1), i1 = c / H, i2 = c - i1 * H;
        const float2 u1 = a.tab[K0 + i1], u2 = a.tab[K0 + a.K1 + i2];
        s_col[tid] = make_float4(u1.x * p.Linv[1], u2.x * p.Linv[2], u1.y, u2.y);
    }
    const float Li0 = p.Linv[0];
    const float cpref = (float)((double)a.qfac / (3.14159265358979323846 * (double)p.L[0] * p.L[1] * p.L[2]));
    if (!go_step(a)) return;   // grid-uniform
    for (int i0 = tid / XB; i0 < K0; i0 += 8 * (TX / XB)) {
        if (i0 != tid / XB) load(i0);
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (i0 + k * (TX / XB) < K0) s[(i0 + k * (TX / XB)) * XB + l0] = v[k];
    }
    __syncthreads();
    double e = 0.0, w = 0.0;
    const int np = f.p0.npass;
    for (int q = 0; q < 2 * np; q++) {   // forward, then inverse
        run_pass(f.p0, q < np ? q : q - np, f.dcol, 1, XB, (const Cx*)tw, s, d);
        if (q != np - 1) continue;
        for (int u = tid; u < K0 * XB; u += TX) {   // column l0 = u mod XB of each thread
            const int i = u / XB;
            const float2 S = s[u], u0 = a.tab[i];
            const float4 c = s_col[l0];
            const float m0 = u0.x * Li0;
            const float mm = fmaf(c.y, c.y, fmaf(c.x, c.x, m0 * m0));
            float C = 0.0f;
            if (c0 + l0 + i != 0) C = cpref * expf(-a.pi2_b2 * mm) / mm * (u0.y * c.z * c.w);
            if (EN && c0 + l0 < M) {
                // the half spectrum: k2 = 0 and (K2 even) K2/2 stand for themselves,
                // the others also for their conjugate partners
                const int i2 = (c0 + l0) % H;
                const double half = (i2 == 0 || 2 * i2 == a.K2) ? 0.5 : 1.0;
                const double em = half * (double)C * ((double)S.x * S.x + (double)S.y * S.y);
                e += em;
                w += em * (1.0 - 2.0 * (double)a.pi2_b2 * (double)mm);
            }
            s[u] = make_float2(S.y * C, S.x * C);   // swapped: the inverse as a forward transform
        }
        __syncthreads();
    }
    if (c0 + l0 < M) {
        float2* __restrict__ out = a.sgrid + c0 + l0;
        for (int i = tid / XB; i < K0; i += TX / XB) out[(size_t)i * M] = swapped(s[i * XB + l0]);
    }
    if (EN) {   // the workgroup's sums in a fixed order
        e = wave_sum_d(e);
        w = wave_sum_d(w);
        if ((tid & 63) == 0) {
            s_red[tid >> 6][0] = e;
            s_red[tid >> 6][1] = w;
        }
        __syncthreads();
        if (tid < 2) {
            double t = 0.0;
            for (int v = 0; v < TX / 64; v++) t += s_red[v][tid];
            a.part[2 * (size_t)blockIdx.x + tid] = t;
        }
    }
}

__global__ __launch_bounds__(TP) void k_pme_inv(const PmeArgs a, const PmeFftArgs f) {
    typedef fft::Cx<float> Cx;
    extern __shared__ float2 s_fft[];
    const int tid = threadIdx.x, x = blockIdx.x;
    const int K1 = a.K1, K2 = a.K2, H = K2 / 2 + 1, rows = (K1 + 1) / 2, pz = K2 | 1, py = H | 1;
    Cx* tw1 = reinterpret_cast<Cx*>(s_fft + 2 * f.plane);
    Cx* tw2 = tw1 + K1;
    float2 *s = s_fft, *d = s_fft + f.plane;
    const float2* __restrict__ in = a.sgrid + (size_t)x * K1 * H;
    const fft::Div dh = f.dh;
    float2 v[2 * NV];
    auto load = [&](int u0) {   // the first ones with the state
#pragma unroll
        for (int k = 0; k < 2 * NV; k++) v[k] = in[min(u0 + k * TP, K1 * H - 1)];
    };
    load(tid);
    for (int k = tid; k < K1 + K2; k += TP) tw1[k] = turn_at<float>(f.tw, a.K0 + k);
    if (!go_step(a)) return;   // grid-uniform
    for (int u0 = tid; u0 < K1 * H; u0 += 2 * NV * TP) {
        if (u0 != tid) load(u0);
#pragma unroll
        for (int k = 0; k < 2 * NV; k++) {
            const int u = u0 + k * TP;
            if (u >= K1 * H) break;
            const int y = dh.quot(u);
            s[y * py + u - y * H] = swapped(v[k]);
        }
    }
    __syncthreads();
    const int nz = f.p2.npass, ny = f.p1.npass;
    for (int p = 0; p < ny + nz; p++) {   // along y, then along z
        const bool z = p >= ny;
        run_pass(z ? f.p2 : f.p1, z ? p - ny : p, z ? f.drow : f.dh, z ? pz : 1, z ? 1 : py, (const Cx*)(z ? tw2 : tw1), s, d);
        if (p != ny - 1) continue;
        // rows 2r and 2r + 1 as one complex row: Z(k) = R0(k) + i R1(k), Z(N - k) from the
        // conjugates (the imaginary parts at k = 0 and N / 2 are rounding, left out)
        for (int u = tid; u < rows * H; u += TP) {
            const int r = dh.quot(u), k = u - r * H;
            float2 A = swapped(s[2 * r * py + k]);
            float2 B = 2 * r + 1 < K1 ? swapped(s[(2 * r + 1) * py + k]) : make_float2(0.f, 0.f);
            if (k == 0 || 2 * k == K2) A.y = B.y = 0.0f;
            d[r * pz + k] = make_float2(A.y + B.x, A.x - B.y);
            if (k != 0 && 2 * k != K2) d[r * pz + K2 - k] = make_float2(B.x - A.y, A.x + B.y);
        }
        __syncthreads();
        float2* t = s;
        s = d;
        d = t;
    }
    float* __restrict__ q = a.qgrid + (size_t)x * K1 * K2;
    const fft::Div dz = f.dk2;
    for (int u = tid; u < rows * K2; u += TP) {
        const int r = dz.quot(u), z = u - r * K2;
        const float2 v = s[r * pz + z];
        q[2 * r * K2 + z] = v.y;
        if (2 * r + 1 < K1) q[(2 * r + 1) * K2 + z] = v.x;
    }
}

// ---------------------------------------------------------------- launchers

static size_t plane_bytes(int plane, int K1, int K2) { return 2 * (size_t)plane * sizeof(float2) + (K1 + K2) * sizeof(fft::Cx<double>); }
static size_t column_bytes(int K0) { return 2 * (size_t)K0 * XB * sizeof(float2) + K0 * sizeof(fft::Cx<double>); }

// Whether these kernels take the grid: every edge a product of 2, 3 and 5, two buffers of an x
// plane's half spectrum and of 16 columns within lds bytes of LDS.  Fills the plans, the plane
// size and the number of column groups.  (Beyond that -- about 136 points per plane edge on
// 160 KB -- the transforms are hipFFT's.)
extern "C" int md_pme_fft_plan(int K0, int K1, int K2, size_t lds, PmeFftArgs* f) {
    f->p0 = fft::plan(K0);
    f->p1 = fft::plan(K1);
    f->p2 = fft::plan(K2);
    if (!f->p0.npass || !f->p1.npass || !f->p2.npass) return 0;
    const int H = K2 / 2 + 1;
    f->plane = std::max((K1 + 1) / 2 * (K2 | 1), K1 * (H | 1));
    f->ncol = (K1 * H + XB - 1) / XB;
    f->drow = fft::Div((K1 + 1) / 2);
    f->dh = fft::Div(H);
    f->dk2 = fft::Div(K2);
    f->dk24 = fft::Div(std::max(K2 / 4, 1));
    f->dcol = fft::Div(XB);
    return plane_bytes(f->plane, K1, K2) + 1024 <= lds && column_bytes(K0) + 1024 <= lds;
}

// Permit the kernels' dynamic LDS (more than 64 KB on larger grids); outside stream capture.
extern "C" hipError_t md_pme_fft_setup(int K0, int K1, int K2, const PmeFftArgs& f) {
    const int pb = (int)plane_bytes(f.plane, K1, K2), cb = (int)column_bytes(K0);
    const struct { const void* k; int b; } all[] = {{reinterpret_cast<const void*>(k_pme_fwd), pb},
                                                    {reinterpret_cast<const void*>(k_pme_inv), pb},
                                                    {reinterpret_cast<const void*>(k_pme_xconv<false>), cb},
                                                    {reinterpret_cast<const void*>(k_pme_xconv<true>), cb}};
    for (const auto& x : all) {
        if (x.b <= 65536) continue;
        const hipError_t e = hipFuncSetAttribute(x.k, hipFuncAttributeMaxDynamicSharedMemorySize, x.b);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

extern "C" hipError_t md_launch_pme_fft(const PmeArgs& a, const PmeFftArgs& f, int energy, hipStream_t st) {
    const size_t pb = plane_bytes(f.plane, a.K1, a.K2), cb = column_bytes(a.K0);
    hipLaunchKernelGGL(k_pme_fwd, dim3(a.K0), dim3(TP), pb, st, a, f);
    if (energy) hipLaunchKernelGGL(k_pme_xconv<true>, dim3(f.ncol), dim3(TX), cb, st, a, f);
    else hipLaunchKernelGGL(k_pme_xconv<false>, dim3(f.ncol), dim3(TX), cb, st, a, f);
    hipLaunchKernelGGL(k_pme_inv, dim3(a.K0), dim3(TP), pb, st, a, f);
    return hipGetLastError();
}
