// state_out.h -- the state in the caller's atom order, from the device into the caller's
// (pageable) arrays through an engine's own pinned ring (state_out.hip).
#pragma once
#include <mutex>

#include "md_device.h"

struct StateOutArgs {
    const float4* pos[2];   // current buffer per replica: pos[cur_buf(st[r])]
    const float4* vel;
    const float4* force;
    const int* slot_of;     // [N]
    const int* tile_rep;
    const RepParam* rep;
    const RepState* st;
    int nrep, natom;
};

// Pinned memory of one engine, made by its first download (as much as that needs, at most
// NS slots of SLOT bytes) and freed with it.  A download holds it until its arrays are filled:
// downloads of one engine from several threads take turns.
struct HostRing {
    static constexpr int NS = 16;
    static constexpr size_t SLOT = 512 << 10;
    char* p = nullptr;
    size_t bytes = 0;
    hipEvent_t ev[NS] = {};
    std::mutex use;
    ~HostRing() { release(); }
    void release();
    hipError_t open(size_t want, bool events);
};

// outs: positions, velocities, forces ([natom][3]; nullptr: not asked for).  Returns when they are written.
hipError_t md_state_out(const StateOutArgs& a, float* const outs[3], HostRing& ring, hipStream_t st);
