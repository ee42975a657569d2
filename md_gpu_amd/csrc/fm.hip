// fm.hip -- adjoint of the pair force for force matching (no reference
// counterpart; the forward pass is the reference's pair kernel,
// src/pair_forces.cu:133-204, run by k_step in force-only mode with
// charges scaled by qscale).
//
// loss = (1/M) sum_frames sum_i |F_i - F*_i|^2,  M = 3 * atoms * frames.
// With R_i = F_i - F*_i and d_ij = x_i - x_j (full list, ordered pairs):
//   dloss/dtheta = (2/M) sum_i sum_j (R_i . d_ij) d ff_ij / d theta
//   d ff / d lj1[ti,tj] = r^-14,  d ff / d lj2[ti,tj] = -r^-8,
//   d ff / d qscale    = 2 qscale qfac q_i q_j C(r) / r^2   (C: Wolf / RF / damped factor)
// Per-pair terms are FP32; each atom's partial sums are promoted to FP64
// before they are accumulated across atoms, workgroups and frames.  The
// Coulomb factor is the force pass's cubic table (Wolf / damped).
// Work decomposition as the step kernel: one workgroup per 64-slot tile (a
// frame is a replica), the tile's neighbor set staged in LDS, G lanes per atom
// walking its row (md_rows.h).  Each workgroup stores its FP64 sums in its own
// slot of part (no atomics); k_fm_reduce adds the slots.
// Algorithmic work per ordered pair: forward 65 flop + adjoint ~45 flop.
#include <algorithm>

#include "md_reduce.h"
#include "md_rows.h"

namespace {

// Sum over the G lanes of each aligned lane group (all lanes get the sum).
template <int G>
__device__ __forceinline__ float lane_group_sum(float x) {
#pragma unroll
    for (int o = G / 2; o >= 1; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

// The same in FP64.
template <int G>
__device__ __forceinline__ double group_sum_d(double x) {
    x += dpp_d<0xB1>(x);                          // quad_perm [1, 0, 3, 2]
    x += dpp_d<0x4E>(x);                          // quad_perm [2, 3, 0, 1]
    if constexpr (G >= 8) x += dpp_d<0x141>(x);   // row_half_mirror
    if constexpr (G >= 16) x += dpp_d<0x140>(x);  // row_mirror
    return x;
}

// Prologue of the adjoint walk: the tables and the tile's set in LDS.
template <int COUL>
__device__ __forceinline__ void fm_stage(const StepArgs& a, int tile, int r, float4* s_j, float4* s_lj, float4* s_ct,
                                         float4* s_sh, const float4* __restrict__ pin) {
    const int tid = threadIdx.x;
    const RepParam& p = a.rep[r];
    if (tid < 64) s_lj[tid] = a.ljtab[tid];
    if (COUL == 1 || COUL == 2) {
        if (tid < 256) s_ct[tid] = a.ctab[tid];
        if (tid == 0) s_ct[MD_CTAB] = a.ctab[MD_CTAB];
    }
    stage_shift_table(s_sh, p.L[0], p.L[1], p.L[2]);
    __syncthreads();
    stage_tile_set(s_j, s_sh, pin, a.jset + (size_t)tile * a.jcap, min(a.jcount[tile], a.jcap));
    __syncthreads();
}

// FP64 totals of the workgroup's per-thread accumulators into part[tile][.]
template <int NW, int NACC>
__device__ __forceinline__ void fm_flush(double* acc, double (*s_red)[NACC], double* part, int tile) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int k = 0; k < NACC; k++)
        for (int o = 32; o >= 1; o >>= 1) acc[k] += __shfl_xor(acc[k], o, 64);
    if (lane == 0)
        for (int k = 0; k < NACC; k++) s_red[wave][k] = acc[k];
    __syncthreads();
    if (tid < NACC) {
        double t = s_red[0][tid];
        for (int w = 1; w < NW; w++) t += s_red[w][tid];
        part[(size_t)tile * NACC + tid] = t;
    }
}

}  // namespace

// Adjoint walk after a force pass (the force of the trial parameters is in
// a.force).  The Coulomb factor C(r)/r^2 comes from the same cubic table as the
// force pass (Wolf / damped), so the gradient is that of the force the GPU computes.
template <int G, int COUL, int NT>
__global__ __launch_bounds__(64 * G) void k_fm_adjoint(const StepArgs a, double* part) {
    constexpr int NW = G;
    constexpr int NACC = 2 + 2 * NT * NT;
    extern __shared__ float4 s_j[];
    __shared__ double s_red[NW][NACC];
    __shared__ float4 s_lj[64];
    __shared__ float4 s_ct[(COUL == 1 || COUL == 2) ? MD_CTAB + 1 : 1];
    __shared__ float4 s_sh[27];
    const int tid = threadIdx.x;
    const int sub = tid & (G - 1), ai = tid / G;
    const int tile = xcd_block(blockIdx.x, gridDim.x);
    const int slot = tile * 64 + ai;
    const int r = __builtin_amdgcn_readfirstlane(a.tile_rep[tile]);
    const float4* __restrict__ pin = a.pos[cur_buf(a.st[r])];
    fm_stage<COUL>(a, tile, r, s_j, s_lj, s_ct, s_sh, pin);
    double acc[NACC];
#pragma unroll
    for (int k = 0; k < NACC; k++) acc[k] = 0.0;
    const int id = a.ids[slot];
    const bool active = id >= 0;
    const float4 xi = pin[slot];
    const int ti = active ? a.typ[slot] : 0;
    const int nn = active ? min(a.ncount[slot], a.cap) : 0;
    const float4 F = a.force[slot], T = a.target[slot];
    const float Rx = F.x - T.x, Ry = F.y - T.y, Rz = F.z - T.z;
    float s1[NT], s2[NT], sq = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; t++) s1[t] = s2[t] = 0.0f;
    const uint4* __restrict__ row4 = reinterpret_cast<const uint4*>(a.nl16 + (size_t)slot * a.cap);
    walk_row<G>(s_j, row4, nn, sub, [&](const float4& pj) {
        const int tj = staged_type(pj);
        const float dx = xi.x - pj.x, dy = xi.y - pj.y, dz = xi.z - pj.z;
        const float rsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        const bool inside = !(rsq > a.rc2);
        const float g = inside ? fmaf(Rz, dz, fmaf(Ry, dy, Rx * dx)) : 0.0f;
        const float ri = __builtin_amdgcn_rsqf(rsq);
        const float ri2 = ri * ri;
        const float ri8 = (ri2 * ri2) * (ri2 * ri2);
        const float t8 = g * ri8;
        const float t14 = t8 * ri2 * ri2 * ri2;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            s1[t] += (tj == t) ? t14 : 0.0f;
            s2[t] -= (tj == t) ? t8 : 0.0f;
        }
        if (COUL == 0) {
            sq = fmaf(g * pj.w, (ri - a.reacf * rsq) * ri2, sq);
        } else if (COUL == 1 || COUL == 2) {
            const float hv = ctab_eval(s_ct, (rsq * ri) * a.ct_scale);
            sq = fmaf(g * pj.w, hv * (ri2 * ri), sq);   // C(r) / r^2, as in the force pass
        }
    });
    if (active) {
        double* a1 = acc + 2;
        double* a2 = acc + 2 + NT * NT;
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
            for (int ta = 0; ta < NT; ta++) {
                if (ta == ti) {
                    a1[ta * NT + t] += (double)s1[t];
                    a2[ta * NT + t] += (double)s2[t];
                }
            }
        }
        acc[1] += (double)sq * 2.0 * (double)a.qq_scale * (double)a.qfac * (double)xi.w;
        if (sub == 0) acc[0] += (double)Rx * Rx + (double)Ry * Ry + (double)Rz * Rz;
    }
    fm_flush<NW, NACC>(acc, s_red, part, tile);
}

// Single-pass form (systems without bonded terms): the rows are walked once for
// the force with the trial parameters and, on the same lanes, for the basis
// sums whose dot products with the residual R_i = F_i - F*_i give the gradient:
//   b14[t] = sum_{j of type t} r^-14 d_ij,   b8[t] = sum_{j of type t} r^-8 d_ij,
//   bc = sum_j q_j C(r)/r^2 d_ij,
//   dloss/dlj1[ti,t] = (2/M) sum_i R_i . b14[t],  dloss/dlj2[ti,t] = -(2/M) sum_i R_i . b8[t],
//   dloss/dqscale = (2/M) sum_i 2 qscale qfac q_i R_i . bc.
// Bound by VALU issue (58 instructions a pair) and, with two workgroups a CU, by the round trips
// before the rows: 4,096 ions x 64 frames 268 -> 244 us an evaluation with the loads of three
// round trips issued together (six before), rows of similar length in a wavefront, parameters
// by bit-field inserts instead of an LDS read, and the tile's sums on one wavefront (120 LDS
// permutes in each before).
// R_i . b is linear in b, so each lane dots the residual (known to all lanes of
// the atom after the force reduction) with its own partial sums; a.qq_scale
// holds qscale.
template <int G, int COUL, int NT>
__global__ __launch_bounds__(64 * G) void k_fm_fused(const StepArgs a, double* part) {
    constexpr int NACC = 2 + 2 * NT * NT;
    extern __shared__ float4 s_j[];
    __shared__ float4 s_lj[64];
    __shared__ float4 s_ct[(COUL == 1 || COUL == 2) ? MD_CTAB + 1 : 1];
    __shared__ float4 s_sh[27];
    constexpr int NTH = 64 * G, JPRE = 32 / G;
    const int tid = threadIdx.x, lane = tid & 63;
    const int sub = tid & (G - 1), ai = tid / G;
    const int tile = xcd_block(blockIdx.x, gridDim.x);
    // Three round trips before the rows are walked: the tile's order, replica, set entries (JPRE
    // a thread; those past the set are loaded and not used) and the tables; the replica's state
    // and the atom's data in both position buffers; the neighbors' positions.
    const int slot = tile * 64 + a.rperm[tile * 64 + ai];   // rows of similar length share a wavefront
    const int r = __builtin_amdgcn_readfirstlane(a.tile_rep[tile]);
    const int jn = min(a.jcount[tile], a.jcap);
    const uint32_t* __restrict__ jt = a.jset + (size_t)tile * a.jcap;
    uint32_t je[JPRE];
#pragma unroll
    for (int u = 0; u < JPRE; u++) je[u] = jt[min(tid + u * NTH, a.jcap - 1)];
    if (tid < 64) s_lj[tid] = a.ljtab[tid];
    if (COUL == 1 || COUL == 2) {
        for (int k = tid; k <= MD_CTAB; k += NTH) s_ct[k] = a.ctab[k];
    }
    const RepState st = a.st[r];
    const RepParam& p = a.rep[r];
    const float L0 = p.L[0], L1 = p.L[1], L2 = p.L[2];
    const int id = a.ids[slot], ti_s = a.typ[slot], nc_s = a.ncount[slot];
    const float4 xa = a.pos[0][slot], xb = a.pos[1][slot], T = a.target[slot];
    const uint4* __restrict__ row4 = reinterpret_cast<const uint4*>(a.nl16 + (size_t)slot * a.cap);
    const uint4 q0 = row4[sub], q1 = row4[(a.cap >= 16 * G ? G : 0) + sub];   // block 1 when the capacity holds one
    loads_issued();
    stage_shift_table(s_sh, L0, L1, L2);
    const int cb = cur_buf(st);
    const float4* __restrict__ pin = a.pos[cb];
    float4 xg[JPRE];
#pragma unroll
    for (int u = 0; u < JPRE; u++) xg[u] = pin[(tid + u * NTH < jn) ? (je[u] & MD_SLOTMASK) : 0u];
    __syncthreads();   // the shift table
#pragma unroll
    for (int u = 0; u < JPRE; u++) {
        const int k = tid + u * NTH;
        if (k < jn) {
            const float4 sv = s_sh[(je[u] >> MD_SLOTBITS) & 31u];
            s_j[k + 1] = make_float4(xg[u].x + sv.x, xg[u].y + sv.y, xg[u].z + sv.z, staged_w<true>(xg[u].w, je[u]));
        }
    }
    for (int k = tid + JPRE * NTH; k < jn; k += NTH) {   // sets beyond JPRE entries per thread
        const uint32_t e = jt[k];
        const float4 x = pin[e & MD_SLOTMASK];
        const float4 sv = s_sh[(e >> MD_SLOTBITS) & 31u];
        s_j[k + 1] = make_float4(x.x + sv.x, x.y + sv.y, x.z + sv.z, staged_w<true>(x.w, e));
    }
    if (tid == 0) s_j[0] = make_float4(MD_FAR, MD_FAR, MD_FAR, 0.0f);
    __syncthreads();
    const float qs = a.qq_scale;
    const bool active = id >= 0;
    const float4 xi = cb ? xb : xa;
    const int ti = active ? ti_s : 0;
    const int nn = active ? min(nc_s, a.cap) : 0;
    const float qi = xi.w * a.qfac * (qs * qs);
    const float4* s_lji = s_lj + ti * 8;
    float f[3] = {0.0f, 0.0f, 0.0f}, bc[3] = {0.0f, 0.0f, 0.0f}, b14[NT][3], b8[NT][3];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int c = 0; c < 3; c++) b14[t][c] = b8[t][c] = 0.0f;
    const int nn0 = longest_row(nn, a.ljfree, ti);
    const float4 lj_a = s_lji[0], lj_b = s_lji[1];
    // two types: one or the other by the type's bit, as a mask (m = ~0 for type 1)
    auto pick = [](uint32_t m, float one, float zero) {
        float z;
        asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(z) : "v"(m), "v"(one), "v"(zero));
        return z;
    };
    walk_row_sorted<G>(s_j, row4, nn, nn0, sub, q0, q1, [&](const float4& pj) {
        const int tj = staged_type(pj);
        uint32_t m = 0;
        float4 lj;
        if (NT == 1) {
            lj = lj_a;
        } else if (NT == 2) {
            asm("v_bfe_i32 %0, %1, 0, 1" : "=v"(m) : "v"(pj.w));
            lj = make_float4(pick(m, lj_b.x, lj_a.x), pick(m, lj_b.y, lj_a.y), 0.0f, 0.0f);
        } else {
            lj = s_lji[tj];
        }
        const float d[3] = {xi.x - pj.x, xi.y - pj.y, xi.z - pj.z};
        const float rsq = fmaf(d[2], d[2], fmaf(d[1], d[1], d[0] * d[0]));
        const float ri = __builtin_amdgcn_rsqf(rsq);
        const float ri2 = ri * ri, ri3 = ri2 * ri;
        const float ri6 = ri3 * ri3, ri8 = ri6 * ri2;
        float ff = fmaf(lj.x, ri6, -lj.y) * ri8;
        float u = 0.0f;   // q_j C(r) / r^2
        if (COUL == 0) {
            u = (ri - a.reacf * rsq) * ri2 * pj.w;
        } else if (COUL == 1 || COUL == 2) {
            u = ctab_eval(s_ct, (rsq * ri) * a.ct_scale) * pj.w * ri3;
        }
        if (COUL <= 2) ff = fmaf(u, qi, ff);
        const bool use = !(rsq > a.rc2);
        ff = use ? ff : 0.0f;
        const float w14 = use ? ri6 * ri8 : 0.0f, w8 = use ? ri8 : 0.0f, wc = use ? u : 0.0f;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            f[c] = fmaf(ff, d[c], f[c]);
            if (COUL <= 2) bc[c] = fmaf(wc, d[c], bc[c]);
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
            float x14, x8;
            if (NT == 1) {
                x14 = w14;
                x8 = w8;
            } else if (NT == 2) {   // the type's bit as a mask
                x14 = t ? __uint_as_float(__float_as_uint(w14) & m) : pick(m, 0.0f, w14);
                x8 = t ? __uint_as_float(__float_as_uint(w8) & m) : pick(m, 0.0f, w8);
            } else {
                x14 = tj == t ? w14 : 0.0f;
                x8 = tj == t ? w8 : 0.0f;
            }
#pragma unroll
            for (int c = 0; c < 3; c++) {
                b14[t][c] = fmaf(x14, d[c], b14[t][c]);
                b8[t][c] = fmaf(x8, d[c], b8[t][c]);
            }
        }
    });
    // the atom's force on all of its lanes, then the residual; the atom's sums go to LDS and one
    // wavefront adds the tile's, a lane per atom
    constexpr int NS = 2 + 2 * NT;   // loss, qscale, lj1 and lj2 by partner type
#pragma unroll
    for (int c = 0; c < 3; c++) f[c] = lane_group_sum<G>(f[c]);
    const float R[3] = {f[0] - T.x, f[1] - T.y, f[2] - T.z};
    double g[NS];
    g[0] = (double)R[0] * R[0] + (double)R[1] * R[1] + (double)R[2] * R[2];
    g[1] = 0.0;
    if (COUL <= 2)
        g[1] = group_sum_d<G>((double)fmaf(R[2], bc[2], fmaf(R[1], bc[1], R[0] * bc[0])) * 2.0 * (double)qs *
                              (double)a.qfac * (double)xi.w);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        g[2 + t] = group_sum_d<G>((double)fmaf(R[2], b14[t][2], fmaf(R[1], b14[t][1], R[0] * b14[t][0])));
        g[2 + NT + t] = group_sum_d<G>(-(double)fmaf(R[2], b8[t][2], fmaf(R[1], b8[t][1], R[0] * b8[t][0])));
    }
    __syncthreads();   // every row is walked: the staged set makes room
    double* s_g = reinterpret_cast<double*>(s_j);   // [NS][64]
    int* s_ti = reinterpret_cast<int*>(s_g + NS * 64);
    if (sub == 0) {
#pragma unroll
        for (int k = 0; k < NS; k++) s_g[k * 64 + ai] = active ? g[k] : 0.0;
        s_ti[ai] = ti;
    }
    __syncthreads();
    if (tid >= 64) return;
    const int tl = s_ti[lane];
#pragma unroll
    for (int k = 0; k < NS; k++) g[k] = s_g[k * 64 + lane];
    double* out = part + (size_t)tile * NACC;
    auto put = [&](int k, double v) {
        v = wave_sum_d(v);
        if (lane == 0) out[k] = v;
    };
    put(0, g[0]);
    put(1, g[1]);
#pragma unroll
    for (int ta = 0; ta < NT; ta++)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            put(2 + ta * NT + t, ta == tl ? g[2 + t] : 0.0);
            put(2 + NT * NT + ta * NT + t, ta == tl ? g[2 + NT + t] : 0.0);
        }
}

// Workgroup k: out[k] = sum over the per-tile slots of accumulator k (fixed
// order: deterministic).
__global__ __launch_bounds__(256) void k_fm_reduce(const double* part, int nslot, int nacc, double* out) {
    __shared__ double s_red[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k = blockIdx.x;
    double v = 0.0;
    for (int b = threadIdx.x; b < nslot; b += blockDim.x) v += part[(size_t)b * nacc + k];
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) out[k] = s_red[0] + s_red[1] + s_red[2] + s_red[3];
}

template <bool FUSED, int G, int NT>
static void launch_fm_g(const StepArgs& a, double* part, int coul, hipStream_t st) {
    // the staged set; afterwards (fused) the atoms' sums and types in its place
    const size_t sums = (2 + 2 * NT) * 64 * sizeof(double) + 64 * sizeof(int);
    const size_t sh = std::max((size_t)(a.jcap + 1) * sizeof(float4), FUSED ? sums : 0);
    const dim3 grid(a.ntiles), blk(64 * G);
    switch (coul) {
    case 0: hipLaunchKernelGGL((FUSED ? k_fm_fused<G, 0, NT> : k_fm_adjoint<G, 0, NT>), grid, blk, sh, st, a, part); break;
    case 1: hipLaunchKernelGGL((FUSED ? k_fm_fused<G, 1, NT> : k_fm_adjoint<G, 1, NT>), grid, blk, sh, st, a, part); break;
    case 2: hipLaunchKernelGGL((FUSED ? k_fm_fused<G, 2, NT> : k_fm_adjoint<G, 2, NT>), grid, blk, sh, st, a, part); break;
    default: hipLaunchKernelGGL((FUSED ? k_fm_fused<G, 3, NT> : k_fm_adjoint<G, 3, NT>), grid, blk, sh, st, a, part); break;
    }
}

template <bool FUSED, int NT>
static hipError_t launch_fm_nt(const StepArgs& a, double* part, int lanes, int coul, hipStream_t st) {
    switch (lanes) {
    case 4: launch_fm_g<FUSED, 4, NT>(a, part, coul, st); break;
    case 8: launch_fm_g<FUSED, 8, NT>(a, part, coul, st); break;
    case 16: launch_fm_g<FUSED, 16, NT>(a, part, coul, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ev0 / ev1 (optional): events recorded around the per-tile kernel alone
template <bool FUSED>
static hipError_t launch_fm(const StepArgs& a, double* part, double* out, int lanes, int coul, int nt, hipStream_t st,
                            hipEvent_t ev0, hipEvent_t ev1) {
    hipError_t e = hipErrorInvalidValue;
    if (ev0 && (e = hipEventRecord(ev0, st)) != hipSuccess) return e;
    e = hipErrorInvalidValue;
    if (nt == 1) e = launch_fm_nt<FUSED, 1>(a, part, lanes, coul, st);
    if (nt == 2) e = launch_fm_nt<FUSED, 2>(a, part, lanes, coul, st);
    if (nt == 4) e = launch_fm_nt<FUSED, 4>(a, part, lanes, coul, st);
    if (e != hipSuccess) return e;
    if (ev1 && (e = hipEventRecord(ev1, st)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_fm_reduce, dim3(2 + 2 * nt * nt), dim3(256), 0, st, (const double*)part, a.ntiles,
                       2 + 2 * nt * nt, out);
    return hipGetLastError();
}

// Single pass (no bonded terms): loss and gradient sums without a separate force pass.
// a.ljtab = the trial table, a.qq_scale = qscale.
// ntype must be 1, 2 or 4 (the host rounds up; unused type rows stay zero)
// part: [ntiles][2 + 2 nt^2] scratch; out: [2 + 2 nt^2] sums (loss, qscale, lj1, lj2 terms)
extern "C" hipError_t md_launch_fm_fused(const StepArgs& a, double* part, double* out, int lanes, int coul, int nt,
                                         hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    return launch_fm<true>(a, part, out, lanes, coul, nt, st, ev0, ev1);
}

extern "C" hipError_t md_launch_fm_adjoint(const StepArgs& a, double* part, double* out, int lanes, int coul, int nt,
                                           hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    return launch_fm<false>(a, part, out, lanes, coul, nt, st, ev0, ev1);
}
