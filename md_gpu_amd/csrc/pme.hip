// pme.hip -- smooth particle-mesh Ewald (Essmann, Perera, Berkowitz, Darden, Lee,
// Pedersen, J. Chem. Phys. 103, 8577 (1995)): the reciprocal-space part that the
// damped Coulomb term (lkspace 2, src/forces.cu:97-110) leaves out, for one
// replica.  The reference vendors GROMACS' PME (src/pme.c:829-1340) without
// building it; this is the method from the paper, as the oracle's md_pme.cpp.
//
// Per step, before the step kernel (which adds frec to each atom's pair force and
// the long-range energy and virial to the replica's first tile):
//   k_pme_spread  the order-p B-spline weights of each atom's scaled coordinates
//                 u = K (x / L + 1/2) (in FP64, so the weights carry only FP32
//                 rounding), q th_x th_y th_z summed per brick of the grid in LDS in
//                 64-bit fixed point: integer sums, so the grid does not depend on the
//                 order of the adds and runs repeat bit for bit
//   R2C FFT       (hipFFT, on the engine's stream, its work area allocated up front)
//   k_pme_conv    multiply by the influence function C(m) = qfac exp(-pi^2 m^2/b^2)
//                 B(m) / (pi V m^2), summing the energy 1/2 C |S|^2 and the traced
//                 virial 1/2 C |S|^2 (1 - 2 pi^2 m^2 / b^2) over the half spectrum
//   C2R FFT       -> dE/dQ on the grid
//   k_pme_gather  four lanes per slot: F = -q grad(sum_k dE/dQ(k) th th th), plus the
//                 correction -qq erf(b r)/r of its excluded pairs
//   k_pme_sum     one workgroup: every workgroup's energy and virial in a fixed
//                 order, plus the self term and the neutralizing-background term
//                 at the step's volume.
// Every kernel first reads the replica's state and does nothing for a step the
// step kernel will not take (the same test as the step kernel), so the chain can
// sit inside a device-gated graph segment, and reads the replica's box (pressure
// coupling rescales it after each step).
#include <hipfft/hipfft.h>

#include "md_device.h"
#include "md_reduce.h"

namespace {

constexpr int PT = 256;   // threads per workgroup

__device__ __forceinline__ bool pme_go(const RepState& s, int mode) {
    if (mode == MODE_FORCE) return !stale(s);
    if (mode == MODE_LF) return !stale(s) && s.step < s.target;
    return s.phase == 1 && !stale(s);
}

// th[j] = M_P(w + j), dth[j] = M_P'(w + j), j = 0..P-1, 0 <= w <= 1:
// M_2(x) = 1 - |x - 1|, M_{k+1}(x) = [x M_k(x) + (k + 1 - x) M_k(x - 1)] / k,
// M_k'(x) = M_{k-1}(x) - M_{k-1}(x - 1).
template <int P, bool DER>
__device__ __forceinline__ void bspline(float w, float* th, float* dth) {
    float a[P];
    a[0] = w;
    a[1] = 1.0f - w;
#pragma unroll
    for (int j = 2; j < P; j++) a[j] = 0.0f;
#pragma unroll
    for (int k = 2; k < P; k++) {
        if (DER && k == P - 1) {
#pragma unroll
            for (int j = 0; j < P; j++) dth[j] = (j < k ? a[j] : 0.0f) - (j > 0 ? a[j - 1] : 0.0f);
        }
        const float rk = 1.0f / (float)k;
        float b[P];
#pragma unroll
        for (int j = 0; j <= k; j++)
            b[j] = ((w + (float)j) * (j < k ? a[j] : 0.0f) + ((float)(k + 1 - j) - w) * (j > 0 ? a[j - 1] : 0.0f)) * rk;
#pragma unroll
        for (int j = 0; j <= k; j++) a[j] = b[j];
    }
#pragma unroll
    for (int j = 0; j < P; j++) th[j] = a[j];
}

// Grid index k0 = floor(u) mod K and the fraction w = u - floor(u) of
// u = (x + L/2) K / L, in FP64: the modulo as fl - K floor(fl / K) with one
// correction by K where the rounded quotient lands on the wrong integer (no
// emulated 64-bit integer division).
__device__ __forceinline__ void grid_coord(float x, double hl, double kl, double ik, int K, int& k0, float& w) {
    double u = ((double)x + hl) * kl;
    if (!(fabs(u) < 1e9)) u = 0.0;   // a non-finite coordinate (the step kernel reports it) stays in the grid
    const double fl = floor(u);
    w = (float)(u - fl);
    double m = fl - (double)K * floor(fl * ik);
    m = m >= (double)K ? m - (double)K : (m < 0.0 ? m + (double)K : m);
    k0 = (int)m;
}

// index of stencil point j (k0 - j, periodic)
__device__ __forceinline__ int wrapk(int k, int K) { return k < 0 ? k + K : k; }

// The replica's box as the PME kernels use it, read at each launch: pressure
// coupling rescales it after every step.
struct PmeBox {
    float L[3], Li[3];
    double hl[3], kl[3];   // L / 2 and K / L
};
__device__ __forceinline__ PmeBox pme_box(const PmeArgs& a) {
    const RepParam& p = a.rep[0];
    PmeBox b;
    const int K[3] = {a.K0, a.K1, a.K2};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        b.L[d] = p.L[d];
        b.Li[d] = p.Linv[d];
        b.hl[d] = 0.5 * (double)p.L[d];
        b.kl[d] = (double)K[d] / (double)p.L[d];
    }
    return b;
}

// Charge spreading, one workgroup per brick of SB0 x SB1 x SB2 grid points summed in
// LDS.  The bricks tile the grid, so every grid point is written once, as float:
// no clearing, no device-scope atomics and no separate conversion pass.
//  1. The cells of the last list build that can hold an atom touching the brick
//     (its points grown by the spline's support and by a.margin, the most an atom
//     can have moved since the build) are tabulated, their atoms tested, and those
//     in reach collected in LDS (in any order: the sums are integers).
//  2. The collected atoms' weights are computed, a lane per atom.
//  3. A lane per (atom, x point, y point) adds its run of P z points that lie in
//     the brick, in 64-bit fixed point: the same sums bit for bit whatever the order.
// The z rows in LDS are padded by one word against bank conflicts.
// Bound by latency at 96^3 (the chain state -> cells -> atoms -> weights -> adds, once
// per brick) and by the LDS adds and their addresses at 128^3.  A wavefront per atom
// with one 8-byte global atomic per stencil point, then a conversion pass, took 30 + 5.5
// us for 32,768 ions on 96^3 and 161 + 7.4 us for 196,608 water atoms on 128^3 (the
// device's atomic units); this takes 11.4 and 28.6 us for the same grids bit for bit.
// Brick and workgroup were swept: 8 x 8 x 16 with 256 threads gives 12.0 and 31.1,
// 16 x 8 x 32 with 512 threads 12.1 and 24.8 but 15.6 instead of 10.5 us for 6,591 atoms
// on 45^3 (27 bricks), 8 x 8 x 8 with 256 threads 15.8 and 39.6.
constexpr int SB0 = 16, SB1 = 8, SB2 = 16, SBZ = SB2 + 1, ST = 512;   // ST threads per brick
constexpr int SU = 4;                 // candidates a thread tests at once (their loads in flight together)
constexpr int SLIST = (SU + 1) * ST;  // collected atoms: up to ST - 1 pending and SU ST new ones

// fixed point (units of 2^-32) of f, rounded to nearest even.  small: |f| < 2^19, where
// the rounding falls out of one FP64 fma (the integer is the low 52 bits).
__device__ __forceinline__ long long to_fixed(float f, bool small) {
    if (small) {
        const double magic = 6755399441055744.0;   // 1.5 * 2^52
        return __double_as_longlong(fma((double)f, MD_PME_QUNIT, magic)) - __double_as_longlong(magic);
    }
    return __double2ll_rn((double)f * MD_PME_QUNIT);
}

// cells of one axis that can hold an atom whose stencil meets grid points [g0, g0 + b)
struct CellSpan {
    int lo, n, nc;
    __device__ int at(int k) const { const int c = lo + k; return c >= nc ? c - nc : c; }
};
__device__ __forceinline__ CellSpan cell_span(int g0, int b, int P, float h, float margin, float cinv, int nc) {
    const float lo = (float)g0 * h - margin, hi = (float)(g0 + b + P - 1) * h + margin;
    CellSpan c;
    c.nc = nc;
    const int l = (int)floorf(lo * cinv), r = (int)floorf(hi * cinv);
    if (r - l + 1 >= nc) {
        c.lo = 0;
        c.n = nc;
    } else {
        c.lo = l < 0 ? l + nc : (l >= nc ? l - nc : l);
        c.n = r - l + 1;
    }
    return c;
}

template <int P>
__global__ __launch_bounds__(ST) void k_pme_spread(const PmeArgs a) {
    __shared__ unsigned long long s_acc[SB0 * SB1 * SBZ];
    __shared__ int s_at[SLIST];                          // slots of the collected atoms
    __shared__ float s_w[3][ST][P];                  // weights of the atoms being added
    __shared__ uint32_t s_k[ST];                         // their grid indices relative to the brick, 10 bits each
    __shared__ int s_start[ST], s_pref[ST + 1], s_wsum[ST / 64], s_cnt;
    const RepState s = a.st[0];
    const RepParam p = a.rep[0];      // in the state's round trip
    loads_issued();
    if (!pme_go(s, a.mode)) return;   // grid-uniform
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const PmeBox bx = pme_box(a);
    const float4* __restrict__ pin = a.pos[cur_buf(s)];
    const int nb1 = (a.K1 + SB1 - 1) / SB1, nb2 = (a.K2 + SB2 - 1) / SB2;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int g2 = blk % nb2 * SB2, g1 = blk / nb2 % nb1 * SB1, g0 = blk / (nb2 * nb1) * SB0;
    const int n0 = min(SB0, a.K0 - g0), n1 = min(SB1, a.K1 - g1), n2 = min(SB2, a.K2 - g2);
    for (int k = tid; k < SB0 * SB1 * SBZ; k += ST) s_acc[k] = 0ull;
    if (tid == 0) s_cnt = 0;
    float margin = a.margin;
    if (a.baro) {
        // scaled box (pressure coupling): an atom moved by less than (min m r_list - r_c) / 2
        // from its scaled build position, m = L / Lb, at the scale before the last
        // rescaling, which at most halves the box
        const float m = fminf(bx.L[0] / p.Lb[0], fminf(bx.L[1] / p.Lb[1], bx.L[2] / p.Lb[2]));
        margin = fmaxf(margin, 0.5f * (m * a.rl - 0.5f * a.rc) + 2e-3f);
    }
    const CellSpan c0 = cell_span(g0, n0, P, bx.L[0] / (float)a.K0, margin, p.cinv[0], p.nc[0]);
    const CellSpan c1 = cell_span(g1, n1, P, bx.L[1] / (float)a.K1, margin, p.cinv[1], p.nc[1]);
    const CellSpan c2 = cell_span(g2, n2, P, bx.L[2] / (float)a.K2, margin, p.cinv[2], p.nc[2]);
    const int ncell = c0.n * c1.n * c2.n;
    // FP32 reach test: floor(u) - g mod K below n + P - 1, with 0.01 of slack on both
    // sides (the points are tested exactly in step 3)
    const float kf[3] = {(float)a.K0, (float)a.K1, (float)a.K2};
    const float sc[3] = {(float)bx.kl[0], (float)bx.kl[1], (float)bx.kl[2]};
    const float gf[3] = {(float)g0, (float)g1, (float)g2};
    const float rf[3] = {(float)(n0 + P - 1), (float)(n1 + P - 1), (float)(n2 + P - 1)};
    auto reach = [&](float x, int d) {
        const float t = fmaf(x, sc[d], 0.5f * kf[d]) - gf[d] + 0.01f;
        const float r = t - kf[d] * floorf(t / kf[d]);
        return r < rf[d] + 0.02f;
    };
    const bool wr0 = a.K0 < n0 + P - 1, wr1 = a.K1 < n1 + P - 1, wr2 = a.K2 < n2 + P - 1;
    int pend = 0;   // collected atoms not yet added (workgroup-uniform)
    // add n (at most ST) collected atoms, from the list's entry base on, to the brick
    auto add = [&](int base, int n) {
        if (tid < n) {
            const float4 x = pin[s_at[base + tid]];
            int k0, k1, k2;
            float w0, w1, w2, t0[P], t1[P], t2[P];
            grid_coord(x.x, bx.hl[0], bx.kl[0], a.ik0, a.K0, k0, w0);
            grid_coord(x.y, bx.hl[1], bx.kl[1], a.ik1, a.K1, k1, w1);
            grid_coord(x.z, bx.hl[2], bx.kl[2], a.ik2, a.K2, k2, w2);
            bspline<P, false>(w0, t0, nullptr);
            bspline<P, false>(w1, t1, nullptr);
            bspline<P, false>(w2, t2, nullptr);
#pragma unroll
            for (int c = 0; c < P; c++) {
                s_w[0][tid][c] = t0[c] * x.w;   // the charge rides on the x weights
                s_w[1][tid][c] = t1[c];
                s_w[2][tid][c] = t2[c];
            }
            const uint32_t r0 = (uint32_t)wrapk(k0 - g0, a.K0), r1 = (uint32_t)wrapk(k1 - g1, a.K1),
                           r2 = (uint32_t)wrapk(k2 - g2, a.K2);
            s_k[tid] = r0 | (r1 << 10) | (r2 << 20);
        }
        __syncthreads();
        for (int u = tid; u < n * P * P; u += ST) {
            const int t = u / (P * P), ij = u % (P * P), i = ij / P, j = ij % P;
            const uint32_t k = s_k[t];
            // point v of the brick, or out of range; an axis shorter than the brick and the
            // spline's support (wrap) meets the brick from both sides
            auto point = [](uint32_t r, int c, int K, bool wrap) {
                int v = (int)r - c;
                if (wrap) v = wrapk(v, K);
                return (uint32_t)v;
            };
            const uint32_t v0 = point(k & 1023u, i, a.K0, wr0), v1 = point((k >> 10) & 1023u, j, a.K1, wr1);
            if (v0 < (uint32_t)n0 && v1 < (uint32_t)n1) {
                const float wxy = s_w[0][t][i] * s_w[1][t][j];
                float wz[P];
#pragma unroll
                for (int c = 0; c < P; c++) wz[c] = s_w[2][t][c];
                unsigned long long* row = s_acc + (v0 * SB1 + v1) * SBZ;
#pragma unroll
                for (int c = 0; c < P; c++) {
                    const uint32_t v2 = point(k >> 20, c, a.K2, wr2);
                    if (v2 < (uint32_t)n2) atomicAdd(row + v2, (unsigned long long)to_fixed(wxy * wz[c], a.small_q != 0));
                }
            }
        }
    };
    for (int b = 0; b < ncell; b += ST) {
        int cs = 0, cn = 0;
        if (b + tid < ncell) {
            const int c = b + tid, w2 = c % c2.n, w1 = c / c2.n % c1.n, w0 = c / (c2.n * c1.n);
            const int r = a.cell_rank[c0.at(w0) + p.nc[0] * (c1.at(w1) + p.nc[1] * c2.at(w2))];
            cs = a.cell_start[r];
            cn = a.cell_start[r + 1] - cs;
        }
        int inc = cn;
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(inc, o, 64);
            if (lane >= o) inc += t;
        }
        if (lane == 63) s_wsum[wave] = inc;
        __syncthreads();
        int off = inc - cn, T = 0;
#pragma unroll
        for (int w = 0; w < ST / 64; w++) {
            if (w < wave) off += s_wsum[w];
            T += s_wsum[w];
        }
        s_start[tid] = cs;
        s_pref[tid] = off;
        if (tid == 0) s_pref[ST] = T;
        __syncthreads();
        for (int q0 = 0; q0 < T; q0 += SU * ST) {
            int slot[SU];
            float4 x[SU];
#pragma unroll
            for (int u = 0; u < SU; u++) {
                const int q = min(q0 + u * ST + tid, T - 1);
                int lo = 0;   // last cell with pref <= q
#pragma unroll
                for (int h = ST / 2; h >= 1; h >>= 1) lo += s_pref[lo + h] <= q ? h : 0;
                slot[u] = s_start[lo] + (q - s_pref[lo]);
            }
#pragma unroll
            for (int u = 0; u < SU; u++) x[u] = pin[slot[u]];
#pragma unroll
            for (int u = 0; u < SU; u++) {
                const bool hit = q0 + u * ST + tid < T && x[u].w != 0.0f && reach(x[u].x, 0) && reach(x[u].y, 1) &&
                                 reach(x[u].z, 2);
                const unsigned long long m = __ballot(hit);
                if (m == 0) continue;   // wavefront-uniform
                int at = 0;
                if (lane == 0) at = atomicAdd(&s_cnt, (int)__popcll(m));
                at = __builtin_amdgcn_readfirstlane(at);
                if (hit) s_at[at + (int)__popcll(m & ((1ull << lane) - 1ull))] = slot[u];
            }
            __syncthreads();
            pend = s_cnt;
            int base = 0;
            while (pend >= ST) {   // workgroup-uniform
                add(base, ST);
                __syncthreads();
                base += ST;
                pend -= ST;
            }
            if (base > 0) {   // the atoms past the added ones move to the front
                const int k = tid < pend ? s_at[base + tid] : 0;
                __syncthreads();
                if (tid < pend) s_at[tid] = k;
                if (tid == 0) s_cnt = pend;
            }
            __syncthreads();
        }
    }
    if (pend > 0) add(0, pend);
    __syncthreads();
    for (int k = tid; k < SB0 * SB1 * SB2; k += ST) {
        const int z = k % SB2, y = k / SB2 % SB1, x = k / (SB2 * SB1);
        if (x < n0 && y < n1 && z < n2) {
            const long long v = (long long)s_acc[(x * SB1 + y) * SBZ + z];
            a.qgrid[((size_t)(g0 + x) * a.K1 + g1 + y) * a.K2 + g2 + z] = (float)((double)v * (1.0 / MD_PME_QUNIT));
        }
    }
}

// FP64 sum of (e, w) over the workgroup (fixed order) into part[k]
__device__ __forceinline__ void block_pair_sum(double e, double w, double* part, int k) {
    __shared__ double s_red[PT / 64][2];
    e = wave_sum_d(e);
    w = wave_sum_d(w);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        s_red[wave][0] = e;
        s_red[wave][1] = w;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double te = 0.0, tw = 0.0;
        for (int v = 0; v < PT / 64; v++) {
            te += s_red[v][0];
            tw += s_red[v][1];
        }
        part[2 * (size_t)k] = te;
        part[2 * (size_t)k + 1] = tw;
    }
}

__global__ __launch_bounds__(PT) void k_pme_conv(const PmeArgs a) {
    if (!pme_go(a.st[0], a.mode)) return;   // grid-uniform
    const int H = a.K2 / 2 + 1;
    const size_t n = (size_t)a.K0 * a.K1 * H;
    const float2* t1 = a.tab + a.K0;
    const float2* t2 = a.tab + a.K0 + a.K1;
    const PmeBox bx = pme_box(a);
    const float cpref = (float)((double)a.qfac / (3.14159265358979323846 * (double)bx.L[0] * bx.L[1] * bx.L[2]));
    double e = 0.0, w = 0.0;
    for (size_t i = (size_t)blockIdx.x * PT + threadIdx.x; i < n; i += (size_t)gridDim.x * PT) {
        const int i2 = (int)(i % H);
        const size_t r = i / H;
        const int i1 = (int)(r % a.K1), i0 = (int)(r / a.K1);
        const float2 u0 = a.tab[i0], u1 = t1[i1], u2 = t2[i2];
        const float m0 = u0.x * bx.Li[0], m1 = u1.x * bx.Li[1], m2 = u2.x * bx.Li[2];   // reciprocal vector
        const float mm = fmaf(m2, m2, fmaf(m1, m1, m0 * m0));
        const float2 S = a.sgrid[i];
        float C = 0.0f;
        if (i != 0) C = cpref * expf(-a.pi2_b2 * mm) / mm * (u0.y * u1.y * u2.y);
        // the half spectrum: k2 = 0 and (K2 even) K2/2 stand for themselves, the
        // others also for their conjugate partners
        const double half = (i2 == 0 || 2 * i2 == a.K2) ? 0.5 : 1.0;
        const double em = half * (double)C * ((double)S.x * S.x + (double)S.y * S.y);
        e += em;
        w += em * (1.0 - 2.0 * (double)a.pi2_b2 * (double)mm);
        a.sgrid[i] = make_float2(S.x * C, S.y * C);
    }
    block_pair_sum(e, w, a.part, blockIdx.x);
}

// Four lanes (a quad) per atom, 64 atoms per workgroup, so the load latency is
// spread over four times the wavefronts: lanes 0..2 of the quad compute the
// B-spline weights and derivatives of one axis each (into LDS, once per atom);
// then lane c of the quad reads the stencil points with z offsets c and c + 4
// and the quad's partial gradients are summed by DPP.  Lane c also takes the
// atom's c-th excluded partner.
template <int P, bool EN>
__global__ __launch_bounds__(PT) void k_pme_gather(const PmeArgs a) {
    __shared__ float s_t[PT / 4][3][P], s_d[PT / 4][3][P];
    __shared__ int s_k[PT / 4][3];
    const int sub = threadIdx.x & 3, la = threadIdx.x >> 2;   // lane in the quad, atom in the workgroup
    const int slot = blockIdx.x * (PT / 4) + la, sl = min(slot, a.nslot - 1);
    double e = 0.0, w = 0.0;
    // the state, the slot's id, its position in both buffers and the box in one round trip
    const RepState s = a.st[0];
    const int id0 = a.ids[sl];
    const float4 xa = a.pos[0][sl], xb = a.pos[1][sl];
    const PmeBox bx = pme_box(a);
    loads_issued();
    if (!pme_go(s, a.mode)) return;   // grid-uniform
    const int id = slot < a.nslot ? id0 : -1;
    const float4* __restrict__ pin = a.pos[cur_buf(s)];
    const float4 x = id >= 0 ? (cur_buf(s) ? xb : xa) : make_float4(0.f, 0.f, 0.f, 0.f);
    if (x.w != 0.0f && sub < 3) {   // this lane's axis
        const float xc = sub == 0 ? x.x : (sub == 1 ? x.y : x.z);
        // selected, not indexed by the lane's axis: an indexed private array lives in scratch
        const double hl = sub == 0 ? bx.hl[0] : (sub == 1 ? bx.hl[1] : bx.hl[2]);
        const double kl = sub == 0 ? bx.kl[0] : (sub == 1 ? bx.kl[1] : bx.kl[2]);
        const double ik = sub == 0 ? a.ik0 : (sub == 1 ? a.ik1 : a.ik2);
        const int K = sub == 0 ? a.K0 : (sub == 1 ? a.K1 : a.K2);
        int k0;
        float w0, t[P], d[P];
        grid_coord(xc, hl, kl, ik, K, k0, w0);
        bspline<P, true>(w0, t, d);
        s_k[la][sub] = k0;
#pragma unroll
        for (int m = 0; m < P; m++) {
            s_t[la][sub][m] = t[m];
            s_d[la][sub][m] = d[m];
        }
    }
    __syncthreads();
    float fx = 0.0f, fy = 0.0f, fz = 0.0f;
    if (x.w != 0.0f) {
        const int k0 = s_k[la][0], k1 = s_k[la][1], k2 = s_k[la][2];
        float t0[P], t1[P], d0[P], d1[P];
#pragma unroll
        for (int m = 0; m < P; m++) {
            t0[m] = s_t[la][0][m];
            d0[m] = s_d[la][0][m];
            t1[m] = s_t[la][1][m];
            d1[m] = s_d[la][1][m];
        }
        // this lane's z points c = sub and sub + 4 (weight 0 where c >= P)
        constexpr int NH = P > 4 ? 2 : 1;
        float tz[NH], dz[NH];
        int gz[NH];
#pragma unroll
        for (int h = 0; h < NH; h++) {
            const int c = sub + 4 * h;
            const bool in = c < P;
            tz[h] = in ? s_t[la][2][in ? c : 0] : 0.0f;
            dz[h] = in ? s_d[la][2][in ? c : 0] : 0.0f;
            gz[h] = in ? wrapk(k2 - c, a.K2) : 0;
        }
        float gx = 0.0f, gy = 0.0f, gzz = 0.0f;
#pragma unroll
        for (int i = 0; i < P; i++) {
            const int g0 = wrapk(k0 - i, a.K0);
#pragma unroll
            for (int j = 0; j < P; j++) {
                const float* row = a.qgrid + ((size_t)g0 * a.K1 + wrapk(k1 - j, a.K1)) * a.K2;
                float sz = 0.0f, sdz = 0.0f;
#pragma unroll
                for (int h = 0; h < NH; h++) {
                    const float ph = row[gz[h]];
                    sz = fmaf(ph, tz[h], sz);
                    sdz = fmaf(ph, dz[h], sdz);
                }
                gx = fmaf(d0[i] * t1[j], sz, gx);
                gy = fmaf(t0[i] * d1[j], sz, gy);
                gzz = fmaf(t0[i] * t1[j], sdz, gzz);
            }
        }
        fx = -x.w * gx * (float)bx.kl[0];
        fy = -x.w * gy * (float)bx.kl[1];
        fz = -x.w * gzz * (float)bx.kl[2];
        if (a.has_excl) {
            // excluded pairs: U = -qq erf(b r)/r, F_i = qq [c2 e^{-b^2 r^2}/r - erf(b r)/r^2] d/r
            const int4 ex = a.excl[id];
            const int pj = sub == 0 ? ex.x : (sub == 1 ? ex.y : (sub == 2 ? ex.z : ex.w));
            const float4 y = pj >= 0 ? pin[a.slot_of[pj]] : make_float4(0.f, 0.f, 0.f, 0.f);
            if (y.w != 0.0f) {
                const float c2 = a.beta * 1.1283791670955126f;   // 2 beta / sqrt(pi)
                const float dx = minimg(x.x - y.x, bx.L[0], bx.Li[0]), dy = minimg(x.y - y.y, bx.L[1], bx.Li[1]),
                            dzz = minimg(x.z - y.z, bx.L[2], bx.Li[2]);
                const float r2 = fmaf(dzz, dzz, fmaf(dy, dy, dx * dx));
                const float r = sqrtf(r2), ir = 1.0f / r;
                const float br = a.beta * r;
                const float erfv = erff(br);
                const float qq = a.qfac * x.w * y.w;
                const float fr = qq * (c2 * expf(-br * br) - erfv * ir) * ir * ir;
                fx = fmaf(fr, dx, fx);
                fy = fmaf(fr, dy, fy);
                fz = fmaf(fr, dzz, fz);
                // energy and virial in FP64: for neutral molecules these terms nearly
                // cancel the self term, each far larger than their sum
                if (EN) {
                    const double rd = sqrt((double)r2), bd = (double)a.beta * rd;
                    const double qqd = (double)a.qfac * (double)x.w * (double)y.w, erfd = erf(bd);
                    e -= 0.5 * qqd * erfd / rd;   // each pair is listed from both atoms
                    w += 0.5 * qqd * (1.1283791670955126 * bd * exp(-bd * bd) - erfd) / rd;
                }
            }
        }
    }
    fx = group_sum<4>(fx);
    fy = group_sum<4>(fy);
    fz = group_sum<4>(fz);
    if (id >= 0 && sub == 0) a.frec[slot] = make_float4(fx, fy, fz, 0.0f);
    if (EN) block_pair_sum(e, w, a.part, a.nconv + blockIdx.x);
}

// Every workgroup's (energy, virial) pair of the influence and gather kernels in
// a fixed order, plus the self and background constants.  One workgroup after
// the gather: a device-scope fence and a shared counter in each of the gather's
// thousands of workgroups cost more than this launch.
__global__ __launch_bounds__(PT) void k_pme_sum(const PmeArgs a) {
    if (!pme_go(a.st[0], a.mode)) return;
    const int np = a.nconv + a.ngather;
    double te = 0.0, tw = 0.0;
    for (int k = threadIdx.x; k < np; k += PT) {
        te += a.part[2 * (size_t)k];
        tw += a.part[2 * (size_t)k + 1];
    }
    block_pair_sum(te, tw, a.out, 0);
    if (threadIdx.x == 0) {
        // self term, and the neutralizing background at the current volume (its
        // virial -L dE/dL is three times itself)
        const RepParam& p = a.rep[0];
        const double V = (double)p.L[0] * p.L[1] * p.L[2], b = (double)a.beta;
        const double ebg = -(double)a.qfac * 3.14159265358979323846 * a.qsum2 / (2.0 * V * b * b);
        a.out[0] += a.e_self + ebg;
        a.out[1] += 3.0 * ebg;
    }
}

template <int P>
void launch_spread(const PmeArgs& a, hipStream_t st) {
    const int nb = ((a.K0 + SB0 - 1) / SB0) * ((a.K1 + SB1 - 1) / SB1) * ((a.K2 + SB2 - 1) / SB2);
    hipLaunchKernelGGL(k_pme_spread<P>, dim3(nb), dim3(ST), 0, st, a);
}

template <int P>
void launch_gather(const PmeArgs& a, int energy, hipStream_t st) {
    if (energy) hipLaunchKernelGGL((k_pme_gather<P, true>), dim3(a.ngather), dim3(PT), 0, st, a);
    else hipLaunchKernelGGL((k_pme_gather<P, false>), dim3(a.ngather), dim3(PT), 0, st, a);
}

}  // namespace

extern "C" hipError_t md_launch_pme_fft(const PmeArgs& a, const PmeFftArgs& f, int energy, hipStream_t st);

// Queue the chain for one step.  f: the plans of the engine's own transforms, or null: r2c
// and c2r.  energy = 0: no step of the run asks for energies or the virial, so their sums are
// left out (their readers, the step kernel's energy variants, do not run either).
// Returns 0, or 1 (HIP launch error) or 2 (hipFFT error).
extern "C" int md_launch_pme(const PmeArgs& a, const PmeFftArgs* f, hipfftHandle r2c, hipfftHandle c2r, int energy,
                             hipStream_t st) {
    switch (a.order) {
    case 4: launch_spread<4>(a, st); break;
    case 6: launch_spread<6>(a, st); break;
    case 8: launch_spread<8>(a, st); break;
    default: return 1;
    }
    if (hipGetLastError() != hipSuccess) return 1;
    if (f) {
        if (md_launch_pme_fft(a, *f, energy, st) != hipSuccess) return 1;
    } else {
        if (hipfftExecR2C(r2c, a.qgrid, reinterpret_cast<hipfftComplex*>(a.sgrid)) != HIPFFT_SUCCESS) return 2;
        hipLaunchKernelGGL(k_pme_conv, dim3(a.nconv), dim3(PT), 0, st, a);
        if (hipfftExecC2R(c2r, reinterpret_cast<hipfftComplex*>(a.sgrid), a.qgrid) != HIPFFT_SUCCESS) return 2;
    }
    switch (a.order) {
    case 4: launch_gather<4>(a, energy, st); break;
    case 6: launch_gather<6>(a, energy, st); break;
    default: launch_gather<8>(a, energy, st); break;
    }
    if (energy) hipLaunchKernelGGL(k_pme_sum, dim3(1), dim3(PT), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}
