// hp_gather.hip -- record assembly for a batch of calls: the reference's
// calc_particle_radii / _reset_potentials (src/groupies.c:212-268), which
// fills each halo's struct potential records from the FOF group's particle
// copies before compute_potential.
//
// The host walks the halo hierarchy exactly as the reference recursion does
// (the halo, its descendants depth first in sibling order, then the parent's
// subtree as potential-only records where the host rule holds) and emits one
// segment per visited halo: a contiguous run of particles that becomes a
// contiguous run of records.  The device side is one pass over the records:
// read a 32-byte particle, write a 48-byte record with r2 about the call's
// centre.  It is HBM-bound; the segments of a group of records are found on
// the device, so the host sends the segments and nothing else.

#include "hp_internal.h"

#pragma clang fp contract(off)

namespace hp {

struct GParticle {  // struct particle, src/particle.h:5-8
    int64_t id;
    float pos[6];
};
static_assert(sizeof(GParticle) == 32, "particle layout");

struct GatherSeg {
    int64_t src;     // first particle
    int32_t dst;     // first record; a segment ends where the next begins
    int32_t flags;   // 0, 1 (the call's own halo) or 2 (a small descendant), kGatherPotential
    float cen[3];    // the centre r2 is about
    int32_t pad;
};
static_assert(sizeof(GatherSeg) == 32, "segment layout");
constexpr int32_t kGatherPotential = 4;  // potential-only records

constexpr int kGatherGroup = 1024;    // records of a workgroup
constexpr int kGatherThreads = 256;

// src/groupies.c:212-233 per record: zeroed record, position and velocity,
// r2 = sum of float dx * dx about the centre, ke = -1 for potential-only
// records, flags.
//
// A workgroup takes 1024 records.  The segment of its first record is found
// 64 candidates at a time, the starts of the segments after it go to LDS and
// each record searches those.  A wavefront's 64 records go out through LDS as
// contiguous 16-byte words: 9.4M records (750 MB) in 0.161 ms, 4.7 TB/s, where
// a copy reaches 5.1; stored a record a lane (three words 48 bytes apart) it
// was 0.274 ms.
__global__ __launch_bounds__(kGatherThreads) void k_gather_records(
    const GParticle *__restrict__ parts, const GatherSeg *__restrict__ segs, int32_t nsegs,
    int32_t total, struct potential *__restrict__ po) {
    struct alignas(8) Word {  // 16 bytes of a record array that may start at 8
        uint32_t w[4];
    };
    __shared__ int32_t s_dst[kGatherGroup];
    __shared__ Word s_rec[kGatherThreads / kWave][3 * kWave];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const int32_t base = blockIdx.x * kGatherGroup;
    const int32_t end = min(base + kGatherGroup, total);
    // the last segment that starts at or before base
    int32_t lo = 0, hi = nsegs;
    while (hi - lo > 1) {
        const int32_t step = (hi - lo + kWave - 1) / kWave, i = lo + lane * step;
        const int32_t c = __popcll(ballot(i < hi && segs[i].dst <= base));
        lo += (c - 1) * step;
        hi = min(lo + step, hi);
    }
    lo = uniform(lo);
    // the starts of the segments from there on that begin before end (each
    // holds a record, so there are at most kGatherGroup)
    int32_t m = 0;
    for (int32_t k = threadIdx.x;; k += kGatherThreads) {
        const bool in = k < kGatherGroup && lo + k < nsegs && segs[lo + k].dst < end;
        if (in) s_dst[k] = segs[lo + k].dst;
        const int32_t c = __syncthreads_count(in);
        m += c;
        if (c < kGatherThreads) break;
    }
    for (int32_t r0 = base + wave * kWave; r0 < end; r0 += kGatherThreads) {
        const int32_t i = r0 + lane;
        if (i < end) {
            int32_t a = 0, b = m;
            while (b - a > 1) {
                const int32_t mid = (a + b) >> 1;
                if (s_dst[mid] <= i) a = mid;
                else b = mid;
            }
            const GatherSeg sg = segs[lo + a];
            const GParticle p = parts[sg.src + (i - sg.dst)];
            float r2 = 0.0f;
            for (int k = 0; k < 3; k++) {
                const float dx = p.pos[k] - sg.cen[k];
                r2 += dx * dx;
            }
            Word *w = &s_rec[wave][3 * lane];
            w[0] = Word{{__float_as_uint(p.pos[0]), __float_as_uint(p.pos[1]),
                         __float_as_uint(p.pos[2]), __float_as_uint(p.pos[3])}};
            w[1] = Word{{__float_as_uint(p.pos[4]), __float_as_uint(p.pos[5]),
                         __float_as_uint(r2), 0u}};
            w[2] = Word{{0u, 0u, __float_as_uint(sg.flags & kGatherPotential ? -1.0f : 0.0f),
                         (uint32_t)(sg.flags & ~kGatherPotential)}};
        }
        wave_sync();
        Word *out = reinterpret_cast<Word *>(po + r0);
        const int32_t words = 3 * min(end - r0, kWave);
        for (int32_t k = lane; k < words; k += kWave) out[k] = s_rec[wave][k];
        wave_sync();
    }
}
static_assert(sizeof(struct potential) == 48 && offsetof(struct potential, r2) == 24 &&
                  offsetof(struct potential, pe) == 32 && offsetof(struct potential, ke) == 40,
              "record layout");

}  // namespace hp
