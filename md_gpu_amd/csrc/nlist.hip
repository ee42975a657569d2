// nlist.hip -- binned cell-list neighbor build with space-filling-curve
// ordering of the atoms (the reference's intended neighborlist_binned,
// src/neighborlist_binned.cu:20-119 / src/neighborlist_kernel_o.cu:20-261,
// which never compiled; the list semantics are those of the O(N^2) build it
// replaces, src/neighborlist.cu:231-297).
//
// A rebuild is six kernels.  Each runs only for replicas whose list is stale
// (RepState.trip, raised by the position update when some atom moved by at
// least skin/2 since the last build: the skin criterion of
// src/neighborlist.cu:157-176), so the chain can sit in every graph segment:
//   k_nl_bin      wrap every coordinate into the box, cell of every atom (cells
//                 are ranked along a Hilbert curve), arrival rank in the cell
//   k_nl_scan     exclusive scan of cell counts -> cell_start (one block per replica)
//   k_nl_scatter  atom -> provisional slot (cell order, arrival order)
//   k_nl_permute  deterministic order inside a cell (by eighth of the cell, then
//                 original index); gathers pos/vel/force/id/type into scratch in the
//                 new order, positions wrapped into the box
//   k_nl_tbuild   one workgroup per 64-slot tile: the members of the image cells within
//                 r_list of the tile's bounding box are streamed through LDS and tested
//                 against the tile's atoms with the canonical FP32 predicate.  Candidates
//                 that some atom of the tile hits form the tile's neighbor set (in
//                 candidate order); each atom's row holds 16-bit indices into that set, in
//                 candidate order, so rows are deterministic.  Each tile stores its longest
//                 row and set size.
//   k_nl_commit   per rebuilt replica: new list epoch (or the next step kernel opens it).
// Bytes per atom per rebuild (algorithmic): read pos/vel/force/id/type 56 B,
// write them twice (scratch + copy back) 112 B, plus the rows 2*K B and the
// tile sets (4 B per set entry, about 4*K/16 B per atom).
#include <type_traits>
#include <utility>

#include "md_device.h"

namespace {

constexpr int kTab = 512;     // region cells per table batch

__device__ __forceinline__ int cell_coord(float x, float halfL, float cinv, int nc) {
    int k = (int)floorf((x + halfL) * cinv);
    return min(max(k, 0), nc - 1);
}

// floor(a / b), b > 0, without an integer division: the estimate from the rounded
// reciprocal of b is off by at most one for |a| < 2^24, and one correction step
// makes it exact.  (Region walks never come near that range.)
__device__ __forceinline__ int floor_div(int a, int b, float inv_b) {
    int q = (int)floorf(((float)a + 0.5f) * inv_b);
    const int r = a - q * b;
    return q + (r >= b ? 1 : 0) - (r < 0 ? 1 : 0);
}

// One axis of the image-cell region around a tile's bounding box [bmin, bmax].
struct Axis {
    int lo, nr, nc;
    float cedge, halfL, bmin, bmax, inv_nc, inv_nr;
    // image index k, wrapped cell w of region coordinate c; returns the gap between
    // the cell slab and the box along this axis (0 when they overlap)
    __device__ float gap(int c, int& k, int& w) const {
        k = floor_div(c, nc, inv_nc);
        w = c - k * nc;
        const float cl = c * cedge - halfL, ch = cl + cedge;
        return fmaxf(0.0f, fmaxf(cl - bmax, bmin - ch));
    }
};

__device__ __forceinline__ Axis make_axis(float bmin, float bmax, float rlp, float halfL, float cinv,
                                          float cedge, int nc) {
    Axis x;
    // image offsets beyond one box length never hold a candidate (r_list < L/2),
    // and the bounds keep the walk finite for any input
    const int l = max((int)floorf((bmin + halfL - rlp) * cinv), -nc);
    const int h = min((int)floorf((bmax + halfL + rlp) * cinv), 2 * nc - 1);
    x.lo = l;
    x.nr = max(h - l + 1, 0);
    x.nc = nc;
    x.inv_nc = 1.0f / (float)nc;
    x.inv_nr = 1.0f / (float)max(x.nr, 1);
    x.cedge = cedge;
    x.halfL = halfL;
    x.bmin = bmin;
    x.bmax = bmax;
    return x;
}

// exclusive scan over an NT-thread block; returns this thread's offset, sets total
template <int NT>
__device__ int block_scan(int v, int* s_w, int& total) {
    constexpr int NW = NT / 64;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int inc = v;
    for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) s_w[w] = inc;
    __syncthreads();
    int off = 0;
    total = 0;
    for (int k = 0; k < NW; k++) {
        const int t = s_w[k];
        if (k < w) off += t;
        total += t;
    }
    __syncthreads();
    return off + inc - v;
}

// old with lane n's value replaced by the wavefront-uniform v (no builtin: the LLVM intrinsic by name)
extern "C" __device__ int md_writelane(int v, int n, int old) __asm("llvm.amdgcn.writelane.i32");
__device__ __forceinline__ int writelane(int v, int n, int old) { return md_writelane(v, n, old); }

// second hash of an original index into the tile build's 16,384-bit exclusion filter
__device__ __forceinline__ uint32_t excl_hash(int id) { return ((uint32_t)id * 2654435761u) >> 18; }

}  // namespace

// The short rebuild kernels first read what says whether their wavefront has
// work (the gate counter, the tile's replica and that replica's state: scalar
// loads, a wavefront's 64 slots being one tile of one replica), and only the
// wavefronts of replicas being rebuilt go on to their slots' data.  In a
// batched run most replicas are not rebuilt at a given check, and their slots'
// data (tens of MB over all replicas) is then never read.
__global__ __launch_bounds__(256) void k_nl_bin(BuildArgs a) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= a.nslot) return;
    const int n_stale = a.gate->n_stale;
    const int r = __builtin_amdgcn_readfirstlane(a.tile_rep[s >> 6]);
    loads_issued();
    if (n_stale == 0) return;
    const RepState st = a.st[r];
    loads_issued();
    if (!stale(st)) return;
    const int id = a.ids[s];
    const float4 x0 = a.pos[0][s], x1 = a.pos[1][s];
    const RepParam& p = a.rep[r];
    const float h0 = p.halfL[0], h1 = p.halfL[1], h2 = p.halfL[2];
    const float c0 = p.cinv[0], c1 = p.cinv[1], c2 = p.cinv[2];
    const float L0 = p.L[0], L1 = p.L[1], L2 = p.L[2], Li0 = p.Linv[0], Li1 = p.Linv[1], Li2 = p.Linv[2];
    const int n0 = p.nc[0], n1 = p.nc[1], n2 = p.nc[2], cell_off = p.cell_off, slot_off = p.slot_off;
    loads_issued();
    if (s == slot_off) {
        a.st[r].trip[(st.nb + 1) & 1] = 0;   // the buffer the next epoch will use
        a.repw[r].Lb[0] = L0;                 // the box of this build (the skin check under pressure coupling)
        a.repw[r].Lb[1] = L1;
        a.repw[r].Lb[2] = L2;
    }
    if (id < 0) return;
    const float4 xr = cur_buf(st) ? x1 : x0;
    // the wrapped position k_nl_permute stores (same operations)
    const float x = wrap_coord(xr.x, L0, Li0), y = wrap_coord(xr.y, L1, Li1), z = wrap_coord(xr.z, L2, Li2);
    int cx = cell_coord(x, h0, c0, n0);
    int cy = cell_coord(y, h1, c1, n1);
    int cz = cell_coord(z, h2, c2, n2);
    int lin = cx + n0 * (cy + n1 * cz);
    int gc = cell_off + a.cell_rank[cell_off + lin];
    // the atom's eighth of the cell, numbered along a path through adjacent eighths
    const int sx = (x + h0) * c0 - (float)cx >= 0.5f;
    const int sy = (y + h1) * c1 - (float)cy >= 0.5f;
    const int sz = (z + h2) * c2 - (float)cz >= 0.5f;
    const int sub = (0x54672310 >> (4 * (sx | (sy << 1) | (sz << 2)))) & 7;
    a.key[s] = gc;
    a.rank[s] = atomicAdd(&a.cell_count[gc], 1) | (sub << MD_SUBSHIFT);
}

__global__ __launch_bounds__(1024) void k_nl_scan(BuildArgs a) {
    __shared__ int wsum[16];
    const int r = blockIdx.x;
    const int n_stale = a.gate->n_stale;
    const RepState st = a.st[r];
    const RepParam& p = a.rep[r];
    const int nc = p.nc[0] * p.nc[1] * p.nc[2];
    const int cell_off = p.cell_off, cs_off = p.cs_off, slot_off = p.slot_off, natom = p.natom;
    loads_issued();
    if (n_stale == 0) return;
    if (!stale(st)) return;
    const int per = (nc + 1023) / 1024;
    const int b = min(nc, (int)threadIdx.x * per), e = min(nc, b + per);
    int sum = 0;
#pragma unroll 8
    for (int k = b; k < e; k++) sum += a.cell_count[cell_off + k];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
        int v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int k = 0; k < 16; k++) { int t = wsum[k]; wsum[k] = run; run += t; }
    }
    __syncthreads();
    int run = slot_off + wsum[w] + inc - sum;
#pragma unroll 8
    for (int k = b; k < e; k++) {
        int c = a.cell_count[cell_off + k];
        a.cell_start[cs_off + k] = run;
        run += c;
        a.cell_count[cell_off + k] = 0;   // ready for the next rebuild
    }
    if (threadIdx.x == 0) a.cell_start[cs_off + nc] = slot_off + natom;
}

__global__ __launch_bounds__(256) void k_nl_scatter(BuildArgs a) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= a.nslot) return;
    const int n_stale = a.gate->n_stale;
    const int r = __builtin_amdgcn_readfirstlane(a.tile_rep[s >> 6]);
    loads_issued();
    if (n_stale == 0) return;
    const RepState st = a.st[r];   // whole (no load that waits for nb)
    loads_issued();
    if (!stale(st)) return;
    const int id = a.ids[s];
    const int gc = a.key[s];
    const int rk = a.rank[s];
    loads_issued();
    if (id < 0) return;
    int t = a.cell_start[gc + r] + (rk & ((1 << MD_SUBSHIFT) - 1));
    a.tmp[t] = s;
    a.tmpid[t] = id | ((rk >> MD_SUBSHIFT) << MD_SUBSHIFT);   // order key: eighth of the cell, then index
}

__global__ __launch_bounds__(256) void k_nl_permute(BuildArgs a) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.nslot) return;
    const int n_stale = a.gate->n_stale;
    const int r = __builtin_amdgcn_readfirstlane(a.tile_rep[t >> 6]);
    loads_issued();
    if (n_stale == 0) return;
    const RepState st = a.st[r];
    loads_issued();
    if (!stale(st)) return;
    // tmp holds a slot of this replica for every t below slot_off + natom
    const RepParam& p = a.rep[r];
    const int lim = p.slot_off + p.natom;
    if (t >= lim) return;
    const int o = a.tmp[t];
    const int mykey = a.tmpid[t];
    const float L0 = p.L[0], L1 = p.L[1], L2 = p.L[2], Li0 = p.Linv[0], Li1 = p.Linv[1], Li2 = p.Linv[2];
    loads_issued();
    const int gc = a.key[o];
    const float4 xr = cur_buf(st) ? a.pos[1][o] : a.pos[0][o];
    const float4 v = a.vel[o], f4 = a.force[o];
    const int ty = a.typ[o];
    const float4 x = make_float4(wrap_coord(xr.x, L0, Li0), wrap_coord(xr.y, L1, Li1), wrap_coord(xr.z, L2, Li2), xr.w);
    const int myid = mykey & ((1 << MD_SUBSHIFT) - 1);
    int cs = a.cell_start[gc + r], ce = a.cell_start[gc + r + 1];
    int cnt = 0;
#pragma unroll 4
    for (int u = cs; u < ce; u++) cnt += (a.tmpid[u] < mykey);
    int f = cs + cnt;
    a.pos_s[f] = x;
    a.vel_s[f] = v;
    a.force_s[f] = f4;
    a.ids_s[f] = myid;
    a.typ_s[f] = ty;
    a.slot_of[myid] = f;
}

// k_nl_bin, k_nl_scan, k_nl_scatter and k_nl_permute in one launch, a workgroup per
// replica, for replicas whose cells and order keys fit in LDS: counts, starts and keys stay
// there and the atoms' data in registers (NA atoms a thread).  The same order.
// Bound by latency (state, atoms, cell order, stores) and by one CU's share of the memory:
// 4,000 atoms 14.6 us where the four kernels take 20, idle 1.6 instead of 8.7; the forces of
// 4,096 ions with their list 392 -> 343 us, 40 steps of 4,000 atoms at constant pressure
// 803 -> 777.  Up to 4,096 atoms a replica: with 8 atoms a thread the registers do not
// hold them (6,591 atoms 31 us against 19, 64 Ar-Xe replicas 3.28 -> 3.39 ms).
// f(0), f(1), ..., f(N - 1) with constant arguments: arrays indexed by them stay in registers
template <class F, int... I>
__device__ __forceinline__ void unrolled_seq(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unrolled(F&& f) {
    unrolled_seq(std::make_integer_sequence<int, N>{}, f);
}

constexpr int SORT_NT = 1024;
template <int NA>
__global__ __launch_bounds__(SORT_NT) void k_nl_sort(BuildArgs a) {
    extern __shared__ int s_cell[];   // [nc + 1] atoms per cell, then first atom; [natom] order keys
    __shared__ int s_w[SORT_NT / 64];
    const int r = blockIdx.x, tid = threadIdx.x;
    const int n_stale = a.gate->n_stale;
    const RepState st = a.st[r];
    loads_issued();
    if (n_stale == 0) return;
    if (!stale(st)) return;
    const RepParam& p = a.rep[r];
    const float h0 = p.halfL[0], h1 = p.halfL[1], h2 = p.halfL[2];
    const float c0 = p.cinv[0], c1 = p.cinv[1], c2 = p.cinv[2];
    const float L0 = p.L[0], L1 = p.L[1], L2 = p.L[2], Li0 = p.Linv[0], Li1 = p.Linv[1], Li2 = p.Linv[2];
    const int n0 = p.nc[0], n1 = p.nc[1], n2 = p.nc[2], natom = p.natom;
    const int cell_off = p.cell_off, cs_off = p.cs_off, slot_off = p.slot_off;
    const int nc = n0 * n1 * n2;
    int* const s_key = s_cell + nc + 1;
    const float4* __restrict__ pin = (cur_buf(st) ? a.pos[1] : a.pos[0]) + slot_off;
    float4 x[NA];
    int key[NA], cell[NA], at[NA];
    unrolled<NA>([&](auto u) {
        const int k = min(tid + u * SORT_NT, natom - 1);
        x[u] = pin[k];
        key[u] = a.ids[slot_off + k];
    });
    for (int k = tid; k <= nc; k += SORT_NT) s_cell[k] = 0;
    unrolled<NA>([&](auto u) {
        x[u] = make_float4(wrap_coord(x[u].x, L0, Li0), wrap_coord(x[u].y, L1, Li1), wrap_coord(x[u].z, L2, Li2), x[u].w);
        const int cx = cell_coord(x[u].x, h0, c0, n0), cy = cell_coord(x[u].y, h1, c1, n1), cz = cell_coord(x[u].z, h2, c2, n2);
        cell[u] = a.cell_rank[cell_off + cx + n0 * (cy + n1 * cz)];
        // the atom's eighth of the cell, numbered along a path through adjacent eighths
        // (fused as the compiler fuses k_nl_bin's)
        const int sx = fmaf(x[u].x + h0, c0, -(float)cx) >= 0.5f;
        const int sy = fmaf(x[u].y + h1, c1, -(float)cy) >= 0.5f;
        const int sz = fmaf(x[u].z + h2, c2, -(float)cz) >= 0.5f;
        const int sub = (0x54672310 >> (4 * (sx | (sy << 1) | (sz << 2)))) & 7;
        key[u] |= sub << MD_SUBSHIFT;
    });
    __syncthreads();
    unrolled<NA>([&](auto u) {
        if (tid + u * SORT_NT < natom) at[u] = atomicAdd(&s_cell[cell[u]], 1);
    });
    __syncthreads();
    // first atom of every cell: contiguous runs of cells per thread
    const int per = (nc + SORT_NT - 1) / SORT_NT;
    const int b = min(nc, tid * per), e = min(nc, b + per);
    int sum = 0;
    for (int k = b; k < e; k++) sum += s_cell[k];
    int total;
    int run = block_scan<SORT_NT>(sum, s_w, total);
    for (int k = b; k < e; k++) {
        const int c = s_cell[k];
        s_cell[k] = run;
        a.cell_start[cs_off + k] = slot_off + run;
        run += c;
    }
    if (tid == 0) {
        s_cell[nc] = natom;
        a.cell_start[cs_off + nc] = slot_off + natom;
        a.st[r].trip[(st.nb + 1) & 1] = 0;   // the buffer the next epoch will use
        a.repw[r].Lb[0] = L0;                 // the box of this build (the skin check under pressure coupling)
        a.repw[r].Lb[1] = L1;
        a.repw[r].Lb[2] = L2;
    }
    __syncthreads();
    unrolled<NA>([&](auto u) {
        if (tid + u * SORT_NT < natom) s_key[s_cell[cell[u]] + at[u]] = key[u];
    });
    __syncthreads();
    // each atom's new slot (at, in order within its cell); then array by array, so that a
    // thread's loads of one are in flight together (as scalars: an array of float4 went to scratch)
    float v0[NA], v1[NA], v2[NA], v3[NA];
    int ty[NA];
    auto load = [&](const float4* from) {
        unrolled<NA>([&](auto u) {
            const float4 q = from[slot_off + min(tid + u * SORT_NT, natom - 1)];
            v0[u] = q.x;
            v1[u] = q.y;
            v2[u] = q.z;
            v3[u] = q.w;
        });
    };
    auto store = [&](float4* to) {
        unrolled<NA>([&](auto u) {
            if (tid + u * SORT_NT < natom) to[at[u]] = make_float4(v0[u], v1[u], v2[u], v3[u]);
        });
    };
    load(a.vel);
    unrolled<NA>([&](auto u) {
        ty[u] = a.typ[slot_off + min(tid + u * SORT_NT, natom - 1)];
    });
    unrolled<NA>([&](auto u) {
        const int cs = s_cell[cell[u]], ce = s_cell[cell[u] + 1];
        int cnt = 0;
#pragma unroll 4
        for (int q = cs; q < ce; q++) cnt += s_key[q] < key[u];
        at[u] = slot_off + cs + cnt;
    });
    store(a.vel_s);
    load(a.force);
    unrolled<NA>([&](auto u) {
        if (tid + u * SORT_NT >= natom) return;
        const int id = key[u] & ((1 << MD_SUBSHIFT) - 1);
        a.pos_s[at[u]] = x[u];
        a.ids_s[at[u]] = id;
        a.typ_s[at[u]] = ty[u];
        a.slot_of[id] = at[u];
    });
    store(a.force_s);
}

// Tile neighbor-set build: one workgroup of NW = 8 (16 for few tiles) wavefronts per 64-slot
// tile, 64 / NW atoms (a group of consecutive slots, so a compact one) per wavefront, their
// positions held as wavefront-uniform values.
//  1. The image cells within r_list of the tile's bounding box (region order, kTab cells a
//     round, a thread per cell) write their members' slots to LDS, 512 per chunk.
//  2. A thread per candidate finds the groups whose bounding box its image is within r_list of.
//  3. Each wavefront lists the chunk's candidates in reach of its group (in candidate
//     order) and tests them, 64 at a time (a lane each), against its 8 atoms with the
//     canonical predicate; the hit masks stay in registers (a lane per atom and 64
//     candidates).  A candidate that hits any atom of the tile gets the next local index
//     of the tile's set, and each atom's hits are appended to its row, first in LDS, then
//     64 entries at a time to memory in one contiguous store.
// So set and rows follow candidate order and do not depend on scheduling.
//
// Bound by VALU issue (75 % busy with water, 78 % with Ar-Xe replicas; 7 instructions per
// atom and 64 candidates for the test, 7 for the append, 4 to keep the mask in between),
// the rest barriers and load latency; at 32,768 ions two tiles per CU leave it latency-bound
// (40 %).  A full build (us): 196,608 water atoms 397 (660 before), 32,768 ions 77 (89), 512
// Ar-Xe replicas 912 (1,065), 64 replicas 151 (211).  Before, every wavefront tested every candidate of the tile (a barrier per 64
// of them), tested self and exclusions per atom and stored hits to memory 2 bytes at a
// time; a group's own candidates are under half of the tile's.  Groups by bounding sphere
// instead of box: 480 us (water).  80 registers keep three workgroups per CU (unbounded,
// 114: one workgroup fewer, 542 us); 64 spill (500 us).
template <bool EXCL, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 6 : 4) void k_nl_tbuild(BuildArgs a) {
    constexpr int NT = kTab, CW = NT / 64, AW = 64 / NW;   // candidates of a chunk, their wavefronts, atoms of a group
    static_assert(NW >= CW && (NT / 64) * AW <= 64, "a candidate per thread, a mask per lane");
    __shared__ uint32_t s_cand[NT];       // the next chunk's candidates: slot | image shift code << 24
    __shared__ float4 s_cx[NT];           // the chunk: candidate position (unshifted), w = bits of the set entry
    __shared__ int s_cid[EXCL ? NT : 1];  // original index of the candidate (exclusions), bit 31: may be excluded
    __shared__ uint2 s_gm[CW][NW];        // [wavefront of the candidates][group]: those in reach of the group
    __shared__ uint8_t s_hit[NT];         // the candidate hit some atom of the tile
    __shared__ uint16_t s_li[NT];         // row entry of a candidate of the set
    __shared__ uint16_t s_list[NW][NT];   // per wavefront the chunk's candidates in reach of its group
    __shared__ uint16_t s_row[64][128];   // per atom the row entries not yet stored (ring by entry mod 128)
    __shared__ uint32_t s_bloom[EXCL ? 512 : 1];   // excluded partners of the tile's atoms (16,384 bits, two hashes)
    __shared__ float4 s_shv[27];          // -k L per shift code (canonical displacement (xi - xj) + s)
    __shared__ float4 s_ax[64];           // the tile's atoms (x, y, z, bits of the id)
    __shared__ float4 s_glo[NW], s_ghi[NW];   // per group: bounding box
    __shared__ int4 s_ex[EXCL ? 64 : 1];
    __shared__ float s_bb[6];
    __shared__ int s_w[NW], s_cw[CW], s_wmax[NW];
    __shared__ int s_cnt[64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tile = blockIdx.x;
    const int slot0 = tile * 64;
    // the gate, the replica index and the tile's atoms in one round trip
    const int n_stale = a.gate->n_stale;
    const int r = __builtin_amdgcn_readfirstlane(a.tile_rep[tile]);
    int id_pre = -1;
    float4 x_pre = make_float4(0.f, 0.f, 0.f, 0.f);
    if (tid < 64) {
        id_pre = a.ids_s[slot0 + tid];
        x_pre = a.pos_s[slot0 + tid];
    }
    loads_issued();
    if (n_stale == 0) return;
    const RepState st = a.st[r];
    loads_issued();
    if (!stale(st)) return;
    const RepParam& p = a.rep[r];
    const int cb = cur_buf(st);
    const float L0 = p.L[0], L1 = p.L[1], L2 = p.L[2];
    const float rl2 = a.rl2;
    const float rlp = sqrtf(rl2) * 1.0001f + 1e-4f;
    // reach of a group's bounding box: r_list grown by what rounding of the coordinates, the
    // image shift and the test can lose
    const float reach2 = (rlp + 1e-3f + 1e-6f * (L0 + L1 + L2)) * (rlp + 1e-3f + 1e-6f * (L0 + L1 + L2));
    if (tid < 27) {
        const int kx = tid % 3 - 1, ky = (tid / 3) % 3 - 1, kz = tid / 9 - 1;
        s_shv[tid] = make_float4(-(float)kx * L0, -(float)ky * L1, -(float)kz * L2, 0.0f);
    }
    if (EXCL) {
        if (tid < 512) s_bloom[tid] = 0u;
        __syncthreads();
    }
    if (tid < 64) {
        const bool act = id_pre >= 0;
        s_ax[tid] = make_float4(act ? x_pre.x : MD_FAR, act ? x_pre.y : MD_FAR, act ? x_pre.z : MD_FAR,
                                __int_as_float(id_pre));
        if (EXCL) {
            const int4 ex = act ? a.excl[id_pre] : make_int4(-1, -1, -1, -1);
            s_ex[tid] = ex;
            for (const int q : {ex.x, ex.y, ex.z, ex.w})
                if (q >= 0) {
                    atomicOr(&s_bloom[(q >> 5) & 511], 1u << (q & 31));
                    atomicOr(&s_bloom[excl_hash(q) >> 5], 1u << (excl_hash(q) & 31));
                }
        }
        // bounding boxes over the active atoms, of the groups (8 lanes), then of the tile
        float lx = act ? x_pre.x : 3.0e38f, ly = act ? x_pre.y : 3.0e38f, lz = act ? x_pre.z : 3.0e38f;
        float hx = act ? x_pre.x : -3.0e38f, hy = act ? x_pre.y : -3.0e38f, hz = act ? x_pre.z : -3.0e38f;
        auto grow = [&](int o) {
            lx = fminf(lx, __shfl_xor(lx, o, 64)); ly = fminf(ly, __shfl_xor(ly, o, 64)); lz = fminf(lz, __shfl_xor(lz, o, 64));
            hx = fmaxf(hx, __shfl_xor(hx, o, 64)); hy = fmaxf(hy, __shfl_xor(hy, o, 64)); hz = fmaxf(hz, __shfl_xor(hz, o, 64));
        };
        for (int o = 1; o < AW; o <<= 1) grow(o);
        if ((lane & (AW - 1)) == 0) {
            s_glo[lane / AW] = make_float4(lx, ly, lz, 0.0f);
            s_ghi[lane / AW] = make_float4(hx, hy, hz, 0.0f);
        }
        for (int o = AW; o <= 32; o <<= 1) grow(o);
        if (tid == 0) {
            s_bb[0] = lx; s_bb[1] = ly; s_bb[2] = lz;
            s_bb[3] = hx; s_bb[4] = hy; s_bb[5] = hz;
        }
    }
    __syncthreads();
    // this wavefront's atoms as wavefront-uniform values; an empty slot sits far
    // outside the box, so no candidate passes the distance test for it
    float axr[AW], ayr[AW], azr[AW];
    int cnt[AW];
#pragma unroll
    for (int i = 0; i < AW; i++) {
        const float4 q = s_ax[wave * AW + i];
        axr[i] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(q.x)));
        ayr[i] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(q.y)));
        azr[i] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(q.z)));
        cnt[i] = 0;
    }
    const int gs = __builtin_ctz(a.row_g);   // row layout: lanes per atom of the step kernel, a power of 2
    const int cap = a.cap, jcap = a.jcap;
    uint16_t* const wrow = a.nl16 + (size_t)(slot0 + wave * AW) * cap;   // row of the wavefront's first atom
    uint32_t* const jset = a.jset + (size_t)tile * jcap;
    int jn = 0;     // size of the tile's set so far (workgroup-uniform)
    // where this lane's entry of a 64-entry stretch of a row goes (lpos16): entry fe of the
    // stretch to position fp, so the wavefront's stores are contiguous (G = 16: in 8-byte
    // pieces, the stretch being half a block)
    const int fe = gs == 2 ? (lane & 32) + ((lane >> 3) & 3) + 4 * (lane & 7)
                           : gs == 3 ? (lane >> 3) + 8 * (lane & 7) : (lane >> 2) + 16 * (lane & 3);
    const int fp = gs == 4 ? 8 * (lane >> 2) + (lane & 3) : lane;

    // store entries e0 .. e0 + 63 (e0 a multiple of 64) of atom i's row; past c: the dummy.
    // Rows longer than the capacity are cut (the host grows it and replays).
    auto flush = [&](int i, int e0, int c) {
        if (e0 >= cap) return;   // wavefront-uniform
        __builtin_amdgcn_wave_barrier();
        const uint16_t v = e0 + fe < c ? s_row[wave * AW + i][(e0 + fe) & 127] : (uint16_t)0;
        const int off = gs == 4 ? (e0 & ~127) + ((e0 >> 4) & 4) : e0;
        wrow[(uint32_t)(i * cap + off) + fp] = v;
        __builtin_amdgcn_wave_barrier();
    };

    {
        const int cell_off = p.cell_off, cs_off = p.cs_off;
        int nreg = 1;
        for (int b0 = 0; b0 < nreg; b0 += kTab) {
            // image-cell region covering the tile box grown by r_list (in the loop, so its
            // values need no registers during the tests; one round unless the cells are small)
            auto bb = [&](int k) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(s_bb[k]))); };
            const Axis ax = make_axis(bb(0), bb(3), rlp, p.halfL[0], p.cinv[0], p.cedge[0], p.nc[0]);
            const Axis ay = make_axis(bb(1), bb(4), rlp, p.halfL[1], p.cinv[1], p.cedge[1], p.nc[1]);
            const Axis az = make_axis(bb(2), bb(5), rlp, p.halfL[2], p.cinv[2], p.cedge[2], p.nc[2]);
            nreg = bb(0) <= bb(3) ? ax.nr * ay.nr * az.nr : 0;   // no atoms: no region
            if (nreg == 0) break;
            const int ncx = p.nc[0], ncy = p.nc[1];
            const float rlp2 = rlp * rlp;
            // region cell c -> its cell's linear index and image shift code; -1 when the
            // image cell lies r_list or farther from the box
            auto locate = [=](int c, int& code) -> int {
                int kx, ky, kz, wx, wy, wz;
                const int cyz = floor_div(c, ax.nr, ax.inv_nr), cz = floor_div(cyz, ay.nr, ay.inv_nr);
                const float ddx = ax.gap(ax.lo + (c - cyz * ax.nr), kx, wx);
                const float ddy = ay.gap(ay.lo + (cyz - cz * ay.nr), ky, wy);
                const float ddz = az.gap(az.lo + cz, kz, wz);
                if (ddx * ddx + ddy * ddy + ddz * ddz >= rlp2) return -1;
                code = shift_code(kx, ky, kz);
                return wx + ncx * (wy + ncy * wz);
            };
            // ---- a region cell per thread: its first slot and image shift (cell), members (n)
            //      and the index of its first member among the candidates (first)
            int code = 0, n = 0;
            uint32_t cell = 0;
            if (tid < NT && b0 + tid < nreg) {
                const int c = locate(b0 + tid, code);
                if (c >= 0) {
                    const int rank = a.cell_rank[cell_off + c];
                    const int cs = a.cell_start[cs_off + rank];
                    n = a.cell_start[cs_off + rank + 1] - cs;
                    cell = (uint32_t)cs | ((uint32_t)code << MD_SLOTBITS);
                }
            }
            int T;
            const int first = block_scan<64 * NW>(n, s_w, T);
            // the candidates [q0, q0 + NT) to s_cand, each cell's by its thread
            auto expand = [&](int q0) {
                const int e = min(first + n, q0 + NT);
                for (int q = max(first, q0); q < e; q++) s_cand[q - q0] = cell + (uint32_t)(q - first);
            };
            // ---- the candidates, NT per chunk.  The next chunk's loads are issued before
            //      this chunk is tested, so they are in flight during the tests.
            uint32_t nj = 0;   // slot | shift code << 24 of the candidate
            int nty = 0, nid = 0;
            float4 nx = make_float4(0.f, 0.f, 0.f, 0.f);
            auto fetch = [&]() {
                nj = s_cand[tid];
                const int j = (int)(nj & MD_SLOTMASK);
                nx = a.pos_s[j];
                nty = a.typ_s[j];
                if (EXCL) nid = a.ids_s[j];
            };
            expand(0);
            __syncthreads();
            if (tid < min(T, NT)) fetch();
            __syncthreads();   // s_cand is read before the next chunk's candidates replace it
            for (int base = 0; base < T; base += NT) {
                float4 cx = nx;
                const uint32_t info = nj | ((uint32_t)nty << MD_JBITS);
                const int cid = nid;
                // groups in reach: the image within `reach` of the group's bounding box
                if (NW == CW || tid < NT) {
                    const bool valid = base + tid < T;
                    const float4 sv = s_shv[valid ? nj >> MD_SLOTBITS : MD_SHIFT0];
                    const float ix = valid ? cx.x - sv.x : MD_FAR, iy = cx.y - sv.y, iz = cx.z - sv.z;
                    int glo = 0, ghi = 0;   // lane g: the wavefront's mask of group g
#pragma unroll 2
                    for (int g = 0; g < NW; g++) {
                        const float4 lo = s_glo[g], hi = s_ghi[g];
                        const float gx = fmaxf(0.0f, fmaxf(lo.x - ix, ix - hi.x));
                        const float gy = fmaxf(0.0f, fmaxf(lo.y - iy, iy - hi.y));
                        const float gz = fmaxf(0.0f, fmaxf(lo.z - iz, iz - hi.z));
                        const unsigned long long in =
                            __builtin_amdgcn_ballot_w64(fmaf(gz, gz, fmaf(gy, gy, gx * gx)) < reach2);
                        glo = writelane((int)(uint32_t)in, g, glo);
                        ghi = writelane((int)(uint32_t)(in >> 32), g, ghi);
                    }
                    if (lane < NW) s_gm[wave][lane] = make_uint2((uint32_t)glo, (uint32_t)ghi);
                    cx.w = __uint_as_float(info);
                    s_cx[tid] = cx;
                    s_hit[tid] = 0;
                }
                if (EXCL && (NW == CW || tid < NT)) {
                    const bool may = ((s_bloom[(cid >> 5) & 511] >> (cid & 31)) & 1u) &&
                                     ((s_bloom[excl_hash(cid) >> 5] >> (excl_hash(cid) & 31)) & 1u);
                    s_cid[tid] = cid | (may ? (int)0x80000000 : 0);
                }
                if (base + NT < T) expand(base + NT);
                __syncthreads();
                if (tid < NT && base + NT + tid < T) fetch();
                // ---- this wavefront's candidates of the chunk
                int nl = 0;
                const uint2 gm = s_gm[lane & (CW - 1)][wave];
#pragma unroll
                for (int w = 0; w < CW; w++) {
                    const uint32_t g0 = (uint32_t)__builtin_amdgcn_readlane((int)gm.x, w),
                                   g1 = (uint32_t)__builtin_amdgcn_readlane((int)gm.y, w);
                    const unsigned long long in = ((unsigned long long)g1 << 32) | g0;
                    const uint32_t e = __builtin_amdgcn_mbcnt_hi(g1, __builtin_amdgcn_mbcnt_lo(g0, (uint32_t)nl));
                    if (__builtin_amdgcn_inverse_ballot_w64(in)) s_list[wave][e] = (uint16_t)(w * 64 + lane);
                    nl += __popcll(in);
                }
                // ---- distance tests: hit masks of batch b and atom i in lane AW b + i
                int mlo = 0, mhi = 0;
                const int nbat = (nl + 63) >> 6;
                for (int b = 0; b < nbat; b++) {
                    const int k = b * 64 + lane;
                    const bool valid = k < nl;
                    const int t = s_list[wave][valid ? k : 0];
                    float4 q = s_cx[t];
                    const uint32_t qi = __float_as_uint(q.w);
                    const int qc = (int)((qi >> MD_SLOTBITS) & 31u), js = (int)(qi & MD_SLOTMASK);
                    const int jid = EXCL ? s_cid[t] : 0;
                    if (!valid) q.x = MD_FAR;   // out of everyone's reach
                    // Most batches hold no image (every shift zero: the canonical (xi - xj) - 0
                    // is xi - xj) and neither an atom of the tile nor a possibly excluded one;
                    // those conditions are only tested for batches that do (wavefront-uniform).
                    const bool shifted = __builtin_amdgcn_ballot_w64(qc != MD_SHIFT0) != 0;
                    const bool own = __builtin_amdgcn_ballot_w64((uint32_t)(js - slot0) < 64u || (EXCL && jid < 0)) != 0;
                    unsigned long long any = 0;
                    auto test = [&](auto shift_tag, auto own_tag) {
                        constexpr bool SH = decltype(shift_tag)::value, OWN = decltype(own_tag)::value;
                        float4 sv = make_float4(0.f, 0.f, 0.f, 0.f);
                        if (SH) sv = s_shv[qc];
#pragma unroll
                        for (int i = 0; i < AW; i++) {
                            float dx = axr[i] - q.x, dy = ayr[i] - q.y, dz = azr[i] - q.z;
                            if (SH) {   // (xi - xj) - k L: the canonical minimum-image displacement for this image
                                dx += sv.x;
                                dy += sv.y;
                                dz += sv.z;
                            }
                            const float rsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                            unsigned long long m = __builtin_amdgcn_ballot_w64(rsq < rl2);
                            if (OWN) {
                                m &= __builtin_amdgcn_ballot_w64(js != slot0 + wave * AW + i);
                                if (EXCL) {
                                    const int qid = jid & 0x7fffffff;
                                    const int4 ex = s_ex[wave * AW + i];
                                    m &= __builtin_amdgcn_ballot_w64(qid != ex.x && qid != ex.y && qid != ex.z && qid != ex.w);
                                }
                            }
                            any |= m;
                            mlo = writelane((int)(uint32_t)m, b * AW + i, mlo);
                            mhi = writelane((int)(uint32_t)(m >> 32), b * AW + i, mhi);
                        }
                    };
                    if (own) test(std::true_type{}, std::true_type{});
                    else if (shifted) test(std::true_type{}, std::false_type{});
                    else test(std::false_type{}, std::false_type{});
                    if (__builtin_amdgcn_inverse_ballot_w64(any)) s_hit[t] = 1;
                }
                __syncthreads();
                // ---- the chunk's set entries
                const unsigned long long hm = __builtin_amdgcn_ballot_w64(tid < NT && s_hit[tid & (NT - 1)] != 0);
                if (lane == 0 && wave < CW) s_cw[wave] = __popcll(hm);
                __syncthreads();
                int li = jn + 1 + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(hm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)hm, 0u));
#pragma unroll
                for (int w = 0; w < CW; w++) {
                    if (w < wave) li += s_cw[w];
                    jn += s_cw[w];
                }
                // a set that outgrew its capacity is rebuilt after the host grows it (the run
                // is rolled back); until then its rows point past it only at the dummy.  Row
                // entries are byte offsets of the staged entry (li x 16, li <= MD_JMAX).
                if (__builtin_amdgcn_inverse_ballot_w64(hm)) {
                    if (li - 1 < jcap) jset[li - 1] = info;
                    s_li[tid] = (uint16_t)(li - 1 < jcap ? li << 4 : 0);
                }
                __syncthreads();
                // ---- the hits to the atoms' rows in LDS (under the hit mask itself); a full
                //      stretch of 64 entries goes out
                for (int b = 0; b < nbat; b++) {
                    const int k = b * 64 + lane;
                    const uint16_t lis = s_li[s_list[wave][k < nl ? k : 0]];
#pragma unroll
                    for (int i = 0; i < AW; i++) {
                        const uint32_t m0 = (uint32_t)__builtin_amdgcn_readlane(mlo, b * AW + i),
                                       m1 = (uint32_t)__builtin_amdgcn_readlane(mhi, b * AW + i);
                        const unsigned long long mi = ((unsigned long long)m1 << 32) | m0;
                        const uint32_t e = __builtin_amdgcn_mbcnt_hi(m1, __builtin_amdgcn_mbcnt_lo(m0, (uint32_t)cnt[i]));
                        if (__builtin_amdgcn_inverse_ballot_w64(mi)) s_row[wave * AW + i][e & 127u] = lis;
                        const int c0 = cnt[i];
                        cnt[i] += __popcll(mi);
                        if ((c0 ^ cnt[i]) & 64) flush(i, c0 & ~63, cnt[i]);
                    }
                }
            }
        }
    }
    // the rows' last entries, padded to the end of the last block (the dummy, local
    // index 0), row lengths, longest row of the wavefront
    int mx = 0;
    const int my_t = a.ljfree != 0 && tid < 64 ? a.typ_s[slot0 + tid] : 0;
#pragma unroll
    for (int i = 0; i < AW; i++) {
        const int c = cnt[i];
        mx = max(mx, c);
        if (c & 63) flush(i, c & ~63, c);
        const int e1 = (c + 63) & ~63;
        if (gs == 4 && (e1 & 64)) flush(i, e1, c);
        if (lane == i) {
            const int cc = __float_as_int(s_ax[wave * AW + i].w) >= 0 ? c : 0;
            a.ncount[slot0 + wave * AW + i] = cc;
            s_cnt[wave * AW + i] = cc;
        }
    }
    if (lane == 0) s_wmax[wave] = mx;
    __syncthreads();
    // the tile's atoms, those with Lennard-Jones interactions first, by decreasing row
    // length (ties by slot): the step kernel's wavefronts then hold atoms whose rows end in
    // the same block
    if (tid < 64) {
        const int c = s_cnt[tid] + (((a.ljfree >> my_t) & 1) ? 0 : 1 << 24);
        if (a.ljfree != 0) {   // one wavefront: its LDS accesses stay in order
            s_cnt[tid] = c;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        const int add = a.ljfree != 0 ? 0 : 1 << 24;
        int rank = 0;
#pragma unroll 4
        for (int k = 0; k < 64; k++) {
            const int d = s_cnt[k] + add;
            rank += (d > c) || (d == c && k < tid);
        }
        a.rperm[slot0 + rank] = (uint8_t)tid;
    }
    // copy the tile back from scratch into the primary arrays (new order)
    if (tid < 64) {
        const int s = slot0 + tid;
        const float4 x = a.pos_s[s];
        a.pos[cb][s] = x;
        a.pos_build[s] = x;
        a.vel[s] = a.vel_s[s];
        a.force[s] = a.force_s[s];
        a.ids[s] = a.ids_s[s];
        a.typ[s] = a.typ_s[s];
    }
    if (tid == 0) {   // longest row and set size of the tile; k_nl_commit opens the new list epoch
        int m = s_wmax[0];
        for (int w = 1; w < NW; w++) m = max(m, s_wmax[w]);
        a.tilemax[tile] = max(a.tilemax[tile], m);   // running maxima since the host cleared them
        a.jmax[tile] = max(a.jmax[tile], jn);
        a.jcount[tile] = min(jn, jcap);
    }
}

// Last kernel of a rebuild chain that is not followed by a deferred-finalize
// block: every rebuilt replica (one wavefront each) opens its new list epoch
// (a deferred-finalize block's first step kernel opens it instead).  The gate
// counters change once per workgroup.  No early exit: every wavefront reaches
// the barrier.
__global__ __launch_bounds__(256) void k_nl_commit(BuildArgs a) {
    __shared__ int s_d[4][3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = blockIdx.x * 4 + wave;
    int done = 0, to_run = 0, to_force = 0;
    if (r < a.nrep) {
        const RepState st = a.st[r];
        if (stale(st)) {
            if (lane == 0) {
                a.st[r].age = 0;
                a.st[r].nb = st.nb + 1;
            }
            done = 1;
            to_run = (a.lfgate || st.phase == 0) && st.step < st.target;
            to_force = !a.lfgate && st.phase == 1;
        }
    }
    if (lane == 0) {
        s_d[wave][0] = done;
        s_d[wave][1] = to_run;
        s_d[wave][2] = to_force;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int n = 0, nr = 0, nf = 0;
        for (int w = 0; w < 4; w++) { n += s_d[w][0]; nr += s_d[w][1]; nf += s_d[w][2]; }
        if (n) atomicSub(&a.gate->n_stale, n);
        if (nr) atomicAdd(&a.gate->n_run, nr);
        if (nf) atomicAdd(&a.gate->n_force, nf);
    }
}

// Mark the lists of all replicas stale (host-requested full rebuild; force = 0: leave
// them) and clear the builds' maxima (ntmax of them).  The persistent kernel's run end
// passes its error word: the lists go stale only after a run without errors, and the
// word goes to pinned host memory.
__global__ __launch_bounds__(256) void k_force_trip(RepState* st, Gate* g, int nrep, int force, int* tmax, int ntmax,
                                                    const int* err, int* err_out) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < ntmax; i += (int)gridDim.x * 256) tmax[i] = 0;
    if (blockIdx.x != 0) return;
    if (err) {
        const int v = *err;
        if (threadIdx.x == 0) *err_out = v;
        if (v) return;
    }
    if (!force) return;
    for (int r = threadIdx.x; r < nrep; r += 256) st[r].trip[st[r].nb & 1] = 1;
    if (threadIdx.x == 0) {
        g->n_stale = nrep;
        g->n_run = 0;
        g->n_force = 0;
    }
}

// ---------------------------------------------------------------- invariants
// Consistency of the sorted atom order and the lists, checked on the device
// (test support, no counterpart in the reference).  Counts into bad[]:
//   0: an active slot s with slot_of[ids[s]] != s (the order is not a bijection)
//   1: a row entry outside the tile's set (local index 0 or beyond jcount)
//   2: a row pair (i, j) whose image distance at the build positions is not
//      below r_list, or j = i
//   3: a set entry whose slot is not an active slot of the tile's replica
//   4: a row longer than the capacity or a set larger than its capacity
//   5: a row block padding entry that is not the dummy
// One thread per atom slot; the caller has just built the lists (pos_build).
__global__ __launch_bounds__(256) void k_check_lists(BuildArgs a, int row_g, int* bad) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= a.nslot) return;
    const int tile = s >> 6;
    const int r = a.tile_rep[tile];
    const RepParam& p = a.rep[r];
    const int id = a.ids[s];
    if (id < 0) return;
    if (id >= 0 && a.slot_of[id] != s) atomicAdd(&bad[0], 1);
    const int nn = a.ncount[s];
    const int jn = a.jcount[tile];
    if (nn > a.cap || a.jmax[tile] > a.jcap) atomicAdd(&bad[4], 1);
    const float4 xi = a.pos_build[s];
    const uint16_t* row = a.nl16 + (size_t)s * a.cap;
    const uint32_t* js = a.jset + (size_t)tile * a.jcap;
    const int n = min(nn, a.cap);
    for (int e = 0; e < n; e++) {
        const int off = row[lpos16(e, row_g)];
        const int li = off >> 4;
        if ((off & 15) || li < 1 || li > jn) {
            atomicAdd(&bad[1], 1);
            continue;
        }
        const uint32_t info = js[li - 1];
        const int j = (int)(info & MD_SLOTMASK), code = (int)((info >> MD_SLOTBITS) & 31);
        if (j < p.slot_off || j >= p.slot_off + p.nslot || a.ids[j] < 0) {
            atomicAdd(&bad[3], 1);
            continue;
        }
        const float4 xj = a.pos_build[j];
        const int kx = code % 3 - 1, ky = (code / 3) % 3 - 1, kz = code / 9 - 1;
        // the image shift of the build's box (a coupled box has moved on since)
        const float dx = (xi.x - xj.x) + (-(float)kx * p.Lb[0]);
        const float dy = (xi.y - xj.y) + (-(float)ky * p.Lb[1]);
        const float dz = (xi.z - xj.z) + (-(float)kz * p.Lb[2]);
        const float rsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        if (!(rsq < a.rl2) || j == s) atomicAdd(&bad[2], 1);
    }
    const int blk = 8 * row_g;
    const int endb = min((nn + blk - 1) / blk * blk, a.cap);
    for (int e = n; e < endb; e++)
        if (row[lpos16(e, row_g)] != 0) atomicAdd(&bad[5], 1);
}

// ---------------------------------------------------------------- launchers

// commit = 0: a deferred-finalize block follows and its first step kernel opens the new lists
extern "C" hipError_t md_launch_rebuild(const BuildArgs& a, int commit, hipStream_t st) {
    const int nb = (a.nslot + 255) / 256;
    if (a.sort_lds > 0) {
        auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(a.nrep), dim3(SORT_NT), a.sort_lds, st, a); };
        if (a.sort_na <= 1) go(k_nl_sort<1>);
        else if (a.sort_na <= 2) go(k_nl_sort<2>);
        else go(k_nl_sort<4>);
    } else {
        hipLaunchKernelGGL(k_nl_bin, dim3(nb), dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_nl_scan, dim3(a.nrep), dim3(1024), 0, st, a);
        hipLaunchKernelGGL(k_nl_scatter, dim3(nb), dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_nl_permute, dim3(nb), dim3(256), 0, st, a);
    }
    const dim3 ntiles(a.nslot / 64);
    // 16 wavefronts a tile (groups of four atoms) while every tile has a CU of its own:
    // 6,591 water atoms 79 -> 65 us a build (with more tiles than CUs, two
    // workgroups of 8 share one and the wavefronts of both are in flight already).
    if (a.wide) {
        if (a.has_excl) hipLaunchKernelGGL((k_nl_tbuild<true, 16>), ntiles, dim3(1024), 0, st, a);
        else hipLaunchKernelGGL((k_nl_tbuild<false, 16>), ntiles, dim3(1024), 0, st, a);
    } else {
        if (a.has_excl) hipLaunchKernelGGL((k_nl_tbuild<true, 8>), ntiles, dim3(512), 0, st, a);
        else hipLaunchKernelGGL((k_nl_tbuild<false, 8>), ntiles, dim3(512), 0, st, a);
    }
    if (commit) hipLaunchKernelGGL(k_nl_commit, dim3((a.nrep + 3) / 4), dim3(256), 0, st, a);
    return hipGetLastError();
}

extern "C" hipError_t md_launch_force_trip(RepState* s, Gate* g, int nrep, int force, int* tmax, int ntmax,
                                           const int* err, int* err_out, hipStream_t st) {
    const int grid = std::max(1, std::min(256, (ntmax + 1023) / 1024));
    hipLaunchKernelGGL(k_force_trip, dim3(grid), dim3(256), 0, st, s, g, nrep, force, tmax, ntmax, err, err_out);
    return hipGetLastError();
}

extern "C" hipError_t md_launch_check_lists(const BuildArgs& a, int row_g, int* bad, hipStream_t st) {
    hipLaunchKernelGGL(k_check_lists, dim3((a.nslot + 255) / 256), dim3(256), 0, st, a, row_g, bad);
    return hipGetLastError();
}
