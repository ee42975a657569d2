// persist.hip -- small single systems: every step of a run in one launch.
//
// For one replica of at most MD_PK_SLOTS slots (Lennard-Jones only, no bonded
// terms) a step is microseconds of pair work spread over a handful of tiles,
// and a launch per step (plus its finalize) costs more than the step.  Here a
// few workgroups of 512 or 1024 threads, one per CU and all resident at once,
// run every step of a run and exchange positions once per step:
//   - workgroup w owns the NTH/G slots from w NTH/G (G lanes per atom) and
//     keeps their position, velocity, force and build position in registers;
//   - each step it stages the positions of the whole system into LDS (at most
//     64 KB) and walks its atoms' rows there, minimum image per pair
//     (src/neighborlist.cu:271-273), LJ force as src/pair_forces.cu:190-195;
//   - the rows are private to the lanes: lane l of an atom lists the
//     neighbors j = l (mod G) within r_list, 16-bit slot indices in LDS.  They
//     are built by a scan of the staged system at the run's first step and
//     whenever the previous step's skin check tripped anywhere (the flag rides on
//     the atom's published position, so all rebuild together); the build wraps the
//     atoms into the box, as the tile path's build does;
//   - where the Berendsen factor (src/integrator.cu:146-147, from the previous
//     step's temperature) or the statistics records need them, each workgroup also
//     publishes its FP64 partial sums (2 KE, LJ energy, virial), added in the same
//     order everywhere.
// Integrators: leapfrog (src/nve_leapfrog.cu:37-55, src/nvt_leapfrog_ber.cu:35-55)
// and NVE velocity Verlet in the leapfrog form of the step kernel (each step
// ends with the second half kick and begins the next with the first).
//
// The exchange: every published 64-bit word carries the number of its step beside
// 32 bits of data (48 of a position), stored and loaded whole at agent scope, so a
// reader that sees the number has the data and no fence, cache write-back or
// invalidation orders anything.  One wavefront waits for the workgroups' hints (a word
// each, stored once its positions are on the way), then every thread loads its
// slots and repeats those whose number is still the old one.  Two banks by step
// parity: a workgroup writes step n + 2 only after it has read every atom of step
// n + 1, and their owners had read step n before they wrote those.  Every wait is
// bounded (MD_PK_TIMEOUT ticks of the 100 MHz wall clock): a workgroup that times
// out sets MD_PK_ERR_WAIT and leaves, the others leave at their next wait, and
// the host reports the error.
//
// Bound by that latency (about 1.8 of 3.3 us a step at 864 atoms) and the walk's VALU
// work on few CUs.  While four of its CUs stay free, the workgroups are placed on one XCD (the others are
// launched for every one that works and leave: workgroups are dealt to the XCDs in turn;
// engines take the XCDs in turn, and one that finds its XCD taken replays the run on any CU
// and tries the next XCD after some runs)
// and have 512 threads, twice as many CUs.  100 steps with a download, 864 atoms: 497
// us with a grid barrier of release and acquire fences per step, 447 with agent-scope
// words instead on one XCD, 428 with 512 threads, 377 without the barrier; 256 atoms, 10
// steps: 81, 76, 71, 71.  (Every thread polling its slots instead of a hint: 376 there, but
// 863 instead of 503 at 2,048 atoms; 256 threads: 484 instead of 444 with 8 lanes.)
#include <hip/hip_ext.h>

#include <type_traits>

#include "md_device.h"
#include "md_pk_words.h"
#include "md_reduce.h"

namespace {

constexpr unsigned FL_TRIP = 1u, FL_ROWS = 2u, FL_STOP = 4u;   // flag bits below the step number

// A published word (md_pk_words.h) is stored and loaded whole.
__device__ __forceinline__ void put(uint64_t* p, uint32_t v, uint32_t tag) {
    __hip_atomic_store(p, pk::word(v, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The limit of a wait: looked at every 64 tries.
struct Wait {
    unsigned long long t0 = 0;
    unsigned tries = 0;
    __device__ __forceinline__ bool late(unsigned long long limit) {
        if ((++tries & 63u) != 0) return false;
        const unsigned long long t = wall_clock64();
        if (tries == 64u) t0 = t;
        return t - t0 > limit;
    }
};

}  // namespace

// G lanes per atom (NTH / G atoms per workgroup); NT1: one atom type (the LJ
// parameters sit in registers).
template <int G, bool NT1, int NTH>
__global__ __launch_bounds__(NTH) void k_persist(const PersistArgs a) {
    constexpr int APW = NTH / G, NW = NTH / 64;
    extern __shared__ float4 s_dyn[];
    float4* s_pos = s_dyn;                                                 // [nslot] x, y, z, type (-1: padding)
    float* s_tyf = reinterpret_cast<float*>(s_dyn + a.nslot);              // [nslot] type as a float
    // lane rows: entry p of thread t in the 16-bit half p & 1 of word (p >> 1) NTH + t
    uint16_t* s_rows = reinterpret_cast<uint16_t*>(s_tyf + a.nslot);       // [cap_l / 2][NTH] words
    __shared__ float4 s_lj[64];
    __shared__ double s_red[NW][3];
    __shared__ double s_lam;         // Berendsen factor of the current step
    __shared__ unsigned s_bits[2];   // flag bits of all atoms' last steps, by step parity
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, sub = tid & (G - 1);
    if ((int)(blockIdx.x % a.spread) != a.xcd) return;   // launched only for the placement
    const int bid = blockIdx.x / a.spread;
    const int slot = bid * APW + tid / G;
    const bool inr = slot < a.nslot;
    const int id = inr ? a.ids[slot] : -1;
    const bool active = id >= 0;
    const int ty = active ? a.typ[slot] : 0;
    const RepParam& p = a.rep[0];
    const float L0 = p.L[0], L1 = p.L[1], L2 = p.L[2];
    const float Li0 = p.Linv[0], Li1 = p.Linv[1], Li2 = p.Linv[2];
    const RepState s0 = a.st[0];
    const long long step0 = s0.step;
    const int cb0 = (int)(step0 & 1);   // between runs phase = 0: the positions of step0
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f), v = x, f = x;
    if (inr) {
        x = a.pos[cb0][slot];
        v = a.vel[slot];
        f = a.force[slot];
    }
    for (int k = tid; k < a.nslot; k += NTH) s_tyf[k] = a.ids[k] >= 0 ? (float)a.typ[k] : -1.0f;
    if (tid < 64) s_lj[tid] = a.ljtab[tid];
    const double dtd = a.dt, taud = a.tau;
    double lamd = a.leapfrog ? a.th[0].S : 1.0;   // leapfrog: the factor of the run's first step
    const bool need_lam = a.leapfrog && a.thermostat == 1;
    // The published sums have a reader.  A leapfrog run of one step exchanges no positions: it
    // publishes them so that workgroup 0 stores the new state after everyone has read the old one
    // (with the state stored by a launch of its own instead, which asks for nothing here, 100
    // steps took 1 to 4 % longer: other registers throughout).
    const bool need_ke = need_lam || a.stats != nullptr || (a.leapfrog && a.nsteps == 1);
    // the atom's position, published as step number n (into bank n & 1)
    auto publish = [&](unsigned n, float4 y, unsigned fl) {
        uint64_t* q = a.xch + ((size_t)(n & 1) * a.natom + slot) * 2;
        const unsigned iy = __float_as_uint(y.y);
        put(q, __float_as_uint(y.x), pk::pos_tag(n, fl, iy >> 16));
        put(q + 1, __float_as_uint(y.z), pk::pos_tag(n, fl, iy & 0xffffu));
    };
    // every workgroup's sums of step number n (lane w: workgroup w's); false: the wait timed out
    auto sums_of = [&](unsigned n, double& t0, double& t1, double& t2) {
        bool ok = true;
        if (lane < a.nwg) {
            const uint64_t* q = a.pub + ((size_t)(n & 1) * MD_PK_WG + lane) * 6;
            uint64_t w[6];
            Wait wait;
            for (;;) {
                bool all = true;
#pragma unroll
                for (int c = 0; c < 6; c++) w[c] = get(q + c);
#pragma unroll
                for (int c = 0; c < 6; c++) all = all && pk::sum_of_step(w[c], n);
                if (all) break;
                if (wait.late(MD_PK_TIMEOUT)) {
                    ok = false;
                    break;
                }
            }
            auto dbl = [](uint64_t hi, uint64_t lo) { return __longlong_as_double((long long)((hi << 32) | (lo & 0xffffffffull))); };
            t0 = dbl(w[1], w[0]);
            t1 = dbl(w[3], w[2]);
            t2 = dbl(w[5], w[4]);
        }
        if (__all(ok)) return true;
        if (lane == 0) atomicOr(a.err, MD_PK_ERR_WAIT);
        return false;
    };
    if (tid < 2) s_bits[tid] = 0u;
    if (!a.leapfrog) {
        // velocity Verlet: the first half kick and drift of the run's first step
        // (k_vv_kick's arithmetic with S = 1)
        if (active) {
            const float h = 0.5f * a.dt * v.w;
            v.x = fmaf(f.x, h, v.x);
            v.y = fmaf(f.y, h, v.y);
            v.z = fmaf(f.z, h, v.z);
            x = make_float4(fmaf(v.x, a.dt, x.x), fmaf(v.y, a.dt, x.y), fmaf(v.z, a.dt, x.z), x.w);
            if (sub == 0) publish(1u, x, 0u);
        }
        __syncthreads();
        if (tid == 0) put(a.hint + MD_PK_WG + bid, 1u, 0u);
    }
    float4 xb = x;                  // build position (skin check)
    int cnt = 0;                    // this lane's row length
    int nbuild = 0;
    float4 lj1 = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();                // s_lj, s_tyf
    if (NT1) lj1 = s_lj[0];
    const int nsteps = (int)a.nsteps;
    int done = 0;
    for (int k = 0; k < nsteps; k++) {
        // the positions of the step whose forces this iteration computes, step number k + 1:
        // each thread waits for its slots (leapfrog's first ones are the run's start)
        unsigned fl = 0;
        if (k > 0 || !a.leapfrog) {
            // the first exchange also shows that every workgroup has its CU: placed on one XCD they
            // may find it taken by another engine's, and the host then runs them spread out
            const unsigned long long limit = a.spread > 1 && k <= 1 ? MD_PK_TIMEOUT_FIRST : MD_PK_TIMEOUT;
            constexpr int SPT = MD_PK_SLOTS / NTH;
            const unsigned n = (unsigned)(k + 1);
            const uint64_t* bank = a.xch + (size_t)(n & 1) * a.natom * 2;
            if (wave == 0) {   // the hints: nothing relies on them but the time of the first try
                bool ok = true;
                if (lane < a.nwg) {
                    const uint64_t* q = a.hint + (n & 1) * MD_PK_WG + lane;
                    Wait wait;
                    while ((unsigned)get(q) != n) {
                        if (wait.late(limit)) {
                            ok = false;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                if (!ok) {
                    atomicOr(a.err, MD_PK_ERR_WAIT);
                    fl |= FL_STOP;
                }
            }
            __syncthreads();
            unsigned miss = 0;
#pragma unroll
            for (int u = 0; u < SPT; u++)
                if (tid + u * NTH < a.natom) miss |= 1u << u;
            Wait wait;
            while (miss) {
                uint64_t w[SPT][2];
#pragma unroll
                for (int u = 0; u < SPT; u++)
                    if ((miss >> u) & 1u) {
                        const uint64_t* q = bank + (size_t)(tid + u * NTH) * 2;
                        w[u][0] = get(q);
                        w[u][1] = get(q + 1);
                    }
#pragma unroll
                for (int u = 0; u < SPT; u++)
                    if (((miss >> u) & 1u) && pk::pos_of_step(w[u][0], n) && pk::pos_of_step(w[u][1], n)) {
                        const int q = tid + u * NTH;
                        const unsigned iy = ((unsigned)(w[u][0] >> 32) << 16) | ((unsigned)(w[u][1] >> 32) & 0xffffu);
                        s_pos[q] = make_float4(__uint_as_float((uint32_t)w[u][0]), __uint_as_float(iy),
                                               __uint_as_float((uint32_t)w[u][1]), s_tyf[q]);
                        fl |= (unsigned)(w[u][0] >> 48) & 7u;
                        miss &= ~(1u << u);
                    }
                if (miss && wait.late(limit)) {
                    atomicOr(a.err, MD_PK_ERR_WAIT);
                    fl |= FL_STOP;
                    break;
                }
            }
        } else {
            for (int q = tid; q < a.natom; q += NTH) {
                const float4 y = a.pos[cb0][q];
                s_pos[q] = make_float4(y.x, y.y, y.z, s_tyf[q]);
            }
        }
        if (fl) atomicOr(&s_bits[k & 1], fl);
        __syncthreads();
        const unsigned bits = s_bits[k & 1];
        if (tid == 0) s_bits[(k + 1) & 1] = 0u;   // read by all before this step's barriers
        if (bits & FL_STOP) break;
        // rows: at the first step and after any skin trip.  The atom's G lanes test
        // the slots j = c G + lane in chunks c and compact the hits in slot order,
        // entry e of the row going to lane e mod G: the lanes' rows differ in length
        // by at most one.
        unsigned mybits = 0;
        if (k == 0 || (bits & FL_TRIP)) {
            if (active) {
                x.x = wrap_coord(x.x, L0, Li0);
                x.y = wrap_coord(x.y, L1, Li1);
                x.z = wrap_coord(x.z, L2, Li2);
            }
            xb = x;
            const int g0 = lane & ~(G - 1);   // the group's first lane in the wavefront
            int n = 0;                        // the atom's entries so far (the same in its G lanes)
            for (int j0 = 0; j0 < a.natom; j0 += G) {
                const int j = j0 + sub;
                bool hit = false;
                if (active && j < a.natom) {
                    const float4 pj = s_pos[j];
                    const float dx = minimg(x.x - pj.x, L0, Li0);
                    const float dy = minimg(x.y - pj.y, L1, Li1);
                    const float dz = minimg(x.z - pj.z, L2, Li2);
                    const float rsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                    hit = rsq < a.rl2 && j != slot;
                }
                const unsigned gm = (unsigned)(__ballot(hit) >> g0) & ((1u << G) - 1u);
                if (hit) {
                    const int e = n + __builtin_popcount(gm & ((1u << sub) - 1u));
                    const int q = e / G;
                    if (q < a.cap_l) s_rows[((q >> 1) * NTH + (tid - sub) + (e % G)) * 2 + (q & 1)] = (uint16_t)j;
                }
                n += __builtin_popcount(gm);
            }
            cnt = n > sub ? (n - sub + G - 1) / G : 0;
            // an odd row ends in half a word: its other half names the atom itself (a
            // valid slot whose pair the walk masks)
            if ((cnt & 1) && cnt < a.cap_l) s_rows[((cnt >> 1) * NTH + tid) * 2 + 1] = (uint16_t)slot;
            if ((n + G - 1) / G > a.cap_l) mybits |= FL_ROWS;
            nbuild++;
        }
        const bool en = a.stats && a.energy_every > 0 && ((step0 + k) % a.energy_every) == 0;
        // pair forces of the own atom (this lane's share of its row), two entries per
        // LDS word so that both neighbors' loads are in flight together
        float fx = 0.f, fy = 0.f, fz = 0.f;
        double elj = 0.0, evi = 0.0;
        const int nr = min(cnt, a.cap_l);
        const float4* s_lji = s_lj + ty * 8;
        const uint32_t* s_w = reinterpret_cast<const uint32_t*>(s_rows) + tid;
        auto walk = [&](auto en_tag) {
            constexpr bool EN = decltype(en_tag)::value;
            auto pair = [&](const float4& pj, bool ok) {
                const float dx = minimg(x.x - pj.x, L0, Li0);
                const float dy = minimg(x.y - pj.y, L1, Li1);
                const float dz = minimg(x.z - pj.z, L2, Li2);
                const float rsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                const float4 lj = NT1 ? lj1 : s_lji[(int)pj.w];
                float ff = pair_ff_lj(rsq, lj);
                const bool use = ok && !(rsq > a.rc2);   // src/pair_forces.cu:195
                ff = use ? ff : 0.0f;
                fx = fmaf(ff, dx, fx);
                fy = fmaf(ff, dy, fy);
                fz = fmaf(ff, dz, fz);
                if (EN && use) {
                    const float ri2 = __builtin_amdgcn_rcpf(rsq);
                    const float ri6 = ri2 * ri2 * ri2;
                    elj += (double)(fmaf(lj.x * (1.0f / 12.0f) * ri6, ri6, -lj.y * (1.0f / 6.0f) * ri6) - lj.z);
                    evi += (double)(ff * rsq);
                }
            };
            for (int e = 0; e < nr; e += 2) {
                const uint32_t w = s_w[(e >> 1) * NTH];
                const float4 p0 = s_pos[w & 0xffffu];
                const float4 p1 = s_pos[w >> 16];
                pair(p0, true);
                pair(p1, e + 1 < nr);
            }
        };
        if (en) walk(std::true_type{});
        else walk(std::false_type{});
        fx = group_sum<G>(fx);
        fy = group_sum<G>(fy);
        fz = group_sum<G>(fz);
        // The previous step's sums, wanted by the Berendsen factor (every workgroup) and the
        // statistics record (workgroup 0): read by wavefront 0 before its atoms are published,
        // so their bank is not written again before.
        const bool want_sums = k > 0 && wave == 0 && (need_lam || (bid == 0 && a.stats));
        if (want_sums) {   // the previous step's totals: Berendsen factor and record
            double t0 = 0.0, t1 = 0.0, t2 = 0.0;
            if (!sums_of((unsigned)(k + 1), t0, t1, t2) && lane == 0) atomicOr(&s_bits[(k + 1) & 1], FL_STOP);
            t0 = wave_sum_d(t0);
            t1 = wave_sum_d(t1);
            t2 = wave_sum_d(t2);
            const double T = t0 / ((double)p.nf * MD_KB_REF);
            if (need_lam && lane == 0) s_lam = sqrt(1.0 + dtd / taud * ((double)p.T0 / T - 1.0));
            const long long ks = k - 1;
            if (bid == 0 && lane == 0 && a.stats && ks < a.stat_cap) {
                const bool en_p = a.energy_every > 0 && ((step0 + ks) % a.energy_every) == 0;
                StatRec rec;
                rec.ke = 0.5 * t0;
                rec.temp = T;
                rec.xi = a.th[0].xi;
                rec.vxi = a.th[0].vxi;
                rec.volume = (double)L0 * (double)L1 * (double)L2;
                rec.has_energy = en_p ? 1 : 0;
                rec.pad = 0;
                rec.pe_lj = en_p ? 0.5 * t1 : 0.0;
                rec.pe_coul = 0.0;
                rec.pe_bond = 0.0;
                rec.pe_angle = 0.0;
                rec.virial = en_p ? 0.5 * t2 : 0.0;
                rec.conserved = rec.ke + rec.pe_lj;
                a.stats[ks] = rec;
            }
        }
        __syncthreads();   // every row is walked: s_pos is free for the next step; s_lam
        if (need_lam && k > 0) lamd = s_lam;
        // integrate (every lane of the group holds the same bits; lane 0 stores)
        double dke = 0.0;
        const bool last = k + 1 == nsteps;
        if (active) {
            f = make_float4(fx, fy, fz, 0.0f);
            const float lam = (float)lamd;
            bool drift = true;
            if (a.leapfrog) {
                const float massif = a.dt * v.w;   // dt / m (src/nve_leapfrog.cu:38)
                v.x = fmaf(fx, massif, v.x) * lam;
                v.y = fmaf(fy, massif, v.y) * lam;
                v.z = fmaf(fz, massif, v.z) * lam;
                if (need_ke) dke = ((double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z) / (double)v.w;
            } else {
                // v(t) = v(t - dt/2) + F dt/2m ends the step; v(t + dt/2) = v(t) + F dt/2m begins the next
                const float h = 0.5f * a.dt * v.w;
                v.x = fmaf(fx, h, v.x);
                v.y = fmaf(fy, h, v.y);
                v.z = fmaf(fz, h, v.z);
                if (need_ke) dke = ((double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z) / (double)v.w;
                drift = !last;
                if (drift) {
                    v.x = fmaf(fx, h, v.x);
                    v.y = fmaf(fy, h, v.y);
                    v.z = fmaf(fz, h, v.z);
                }
            }
            if (drift) {
                x = make_float4(fmaf(v.x, a.dt, x.x), fmaf(v.y, a.dt, x.y), fmaf(v.z, a.dt, x.z), x.w);
                const float ddx = minimg(x.x - xb.x, L0, Li0), ddy = minimg(x.y - xb.y, L1, Li1),
                            ddz = minimg(x.z - xb.z, L2, Li2);
                if (fmaf(ddz, ddz, fmaf(ddy, ddy, ddx * ddx)) >= a.skin2q) mybits |= FL_TRIP;   // src/neighborlist.cu:174
                if (!(fabsf(x.x) <= L0 && fabsf(x.y) <= L1 && fabsf(x.z) <= L2)) mybits |= FL_STOP;
            }
            if (sub == 0) {
                if (mybits & FL_STOP) atomicOr(a.err, 1);   // an atom left the box: unstable
                if (mybits & FL_ROWS) {                      // the run is replayed with longer rows
                    atomicOr(a.err, MD_PK_ERR_ROWS);
                    mybits |= FL_STOP;
                }
                if (!last) publish((unsigned)(k + 2), x, mybits);
            }
            if (sub != 0) dke = 0.0;
        }
        if (need_ke) {   // the workgroup's partial sums
            const double q0 = wave_sum_d(dke);
            const double q1 = en ? wave_sum_d(elj) : 0.0;
            const double q2 = en ? wave_sum_d(evi) : 0.0;
            if (lane == 0) {
                s_red[wave][0] = q0;
                s_red[wave][1] = q1;
                s_red[wave][2] = q2;
            }
            __syncthreads();
            if (tid < 3) {
                double t = s_red[0][tid];
                for (int w = 1; w < NW; w++) t += s_red[w][tid];
                const uint64_t d = (uint64_t)__double_as_longlong(t);
                const unsigned n = (unsigned)(k + 2);
                uint64_t* q = a.pub + ((size_t)(n & 1) * MD_PK_WG + bid) * 6 + 2 * tid;
                put(q, (uint32_t)d, pk::sum_tag(n));
                put(q + 1, (uint32_t)(d >> 32), pk::sum_tag(n));
            }
        }
        if (!last) {
            __syncthreads();
            if (tid == 0) put(a.hint + (k & 1) * MD_PK_WG + bid, (unsigned)(k + 2), 0u);
        }
        done = k + 1;
    }
    // the last step's record and factor
    if (done == nsteps && nsteps > 0) {
        if (wave == 0 && bid == 0) {
            double t0 = 0.0, t1 = 0.0, t2 = 0.0;
            if (need_ke) sums_of((unsigned)(nsteps + 1), t0, t1, t2);   // every workgroup has read st and th
            t0 = wave_sum_d(t0);
            t1 = wave_sum_d(t1);
            t2 = wave_sum_d(t2);
            if (lane == 0) {
                const long long ks = nsteps - 1;
                const double T = t0 / ((double)p.nf * MD_KB_REF);
                if (a.stats && ks < a.stat_cap) {
                    const bool en = a.energy_every > 0 && ((step0 + ks) % a.energy_every) == 0;
                    StatRec rec;
                    rec.ke = 0.5 * t0;
                    rec.temp = T;
                    rec.xi = a.th[0].xi;
                    rec.vxi = a.th[0].vxi;
                    rec.volume = (double)L0 * (double)L1 * (double)L2;
                    rec.has_energy = en ? 1 : 0;
                    rec.pad = 0;
                    rec.pe_lj = en ? 0.5 * t1 : 0.0;
                    rec.pe_coul = 0.0;
                    rec.pe_bond = 0.0;
                    rec.pe_angle = 0.0;
                    rec.virial = en ? 0.5 * t2 : 0.0;
                    rec.conserved = rec.ke + rec.pe_lj;
                    a.stats[ks] = rec;
                }
                double lam = 1.0;
                if (a.leapfrog && a.thermostat == 1) lam = sqrt(1.0 + dtd / taud * ((double)p.T0 / T - 1.0));
                if (a.leapfrog) a.th[0].S = lam;
                RepState& st = a.st[0];
                st.step = step0 + nsteps;
                st.nb = s0.nb + nbuild;
            }
        }
        if (active && sub == 0) {
            a.pos[(int)((step0 + nsteps) & 1)][slot] = x;
            a.vel[slot] = v;
            a.force[slot] = f;
        }
    }
}

// nwg: working workgroups launched (a.nwg, or fewer in a test of the bounded waits)
extern "C" hipError_t md_launch_persist(const PersistArgs& a, int lanes, int nwg, size_t shmem, hipStream_t st,
                                        hipEvent_t ev0, hipEvent_t ev1) {
    const dim3 grid(nwg * a.spread), block(a.nth);
    const bool nt1 = a.ntype == 1;
    hipError_t rc = hipSuccess;
    auto go = [&](auto kern) {
        // more than 64 KB of dynamic LDS is requested (one workgroup per CU)
        rc = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)shmem);
        if (rc != hipSuccess) return;
        if (ev0) hipExtLaunchKernelGGL(kern, grid, block, shmem, st, ev0, ev1, 0, a);
        else hipLaunchKernelGGL(kern, grid, block, shmem, st, a);
    };
    auto pick = [&](auto g) {
        constexpr int G = decltype(g)::value;
        if (a.nth == 512) nt1 ? go(k_persist<G, true, 512>) : go(k_persist<G, false, 512>);
        else nt1 ? go(k_persist<G, true, 1024>) : go(k_persist<G, false, 1024>);
    };
    switch (lanes) {
    case 4: pick(std::integral_constant<int, 4>{}); break;
    case 8: pick(std::integral_constant<int, 8>{}); break;
    case 16: pick(std::integral_constant<int, 16>{}); break;
    default: return hipErrorInvalidValue;
    }
    if (rc != hipSuccess) return rc;
    return hipGetLastError();
}
