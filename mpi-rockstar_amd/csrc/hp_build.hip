// hp_build.hip -- GPU build of the reference's potential tree and its
// multipoles, for every halo of a batch at once.
//
// The tree is MPI-Rockstar's POTENTIAL fast3tree (src/potential.c:57-64,
// src/fast3tree.c:736-908): a binary k-d tree over the finite points of one
// compute_potential call, splitting a node of more than 10 points at the float
// midpoint of the widest side of its tight box (z first, x or y only when
// strictly wider), points with pos[dim] <= lim going left.  A split that puts
// every point on one side makes the node a leaf.  Every partition puts the
// points in the order the reference's in-place swap loop leaves them
// (src/fast3tree.c:762-773, closed form in inplace_dest): each split lists
// the node's points by side (the stable order), then moves every point to
// its slot.  So the final tree order, and with it every leaf's summation
// order, is the reference's.
//
// The build runs over the whole batch at once:
//   roots     gather: records -> float4 (x, y, z, record index), tight box and
//             non-finite count per call (tiles of one call, block reductions,
//             integer atomics on order-preserving float keys); roots: one
//             thread per call writes the root node and queues it (calls with
//             non-finite points get a workgroup that moves those records to
//             the end of the call's range, stably).
//   levels    nodes of more than kSmallMax points: tiles of 1024 points,
//             count pass -> one wavefront per node (scan of the tile counts,
//             child boxes) -> scatter pass; host-driven, several levels per
//             counter read.
//   subtrees  every node of at most kSmallMax points is finished in one go:
//             65..kSmallMax points by a workgroup (a kernel each for nodes of
//             at most 256, 512 and 1,024 points), a thread per point down to
//             nodes of at most 32 points, then by its wavefronts; at most 64
//             points by one wavefront, a point per lane.  Both keep the points and the node table in LDS, compute
//             centres of mass bottom-up and dmin over the final order, and
//             write leaves straight into the final tree-order array.
// Multipoles of the nodes made by the split levels (src/potential.c:71-124):
// leaf mass and centre from f64 sums, internal centres combined in float
// from the two children (right term first) level by level, dmin over the
// node's whole range in f64 by tiles.

#include "hp_internal.h"

#pragma clang fp contract(off)

namespace hp {

__device__ __forceinline__ double d2_ref(const float *c, const float4 &p) {
    // src/potential.c:22-29: float differences, double squares, summed in
    // order (a float times a float is exact in double, so each fma rounds
    // as the separate product and sum do)
    const double dx = (double)(c[0] - p.x);
    const double dy = (double)(c[1] - p.y);
    const double dz = (double)(c[2] - p.z);
    double s = dx * dx;
    s = fma(dy, dy, s);
    s = fma(dz, dz, s);
    return s;
}

__device__ __forceinline__ void finish_dmin(Node *nd, double big, double sum, int32_t count) {
    // src/potential.c:79-81
    double b = sqrt(big) / 2.0;
    float dmin = (float)(b + sqrt(b * b + sum / ((double)count * 1.0)));
    nd->dmin = dmin;
    nd->dmin2 = dmin * dmin;
}

// ------------------------------------------------------------------ level 0

struct RootTile {
    int32_t halo;
    int32_t off;
};
// Records of one root tile: a call's box is combined by atomics, one set per
// tile, and those of a call of many tiles wait for each other (2,050 tiles:
// 161 us with 1,024 records to a tile, 56 with 4,096).
__host__ __device__ __forceinline__ int32_t root_tile_records(int64_t count) {
    return count > 256 * kTile ? 4 * kTile : kTile;
}

__global__ void k_fill_i32(int32_t *p, int32_t v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// box keys per halo: [lo0 lo1 lo2 hi0 hi1 hi2] as order-preserving ints,
// bad: non-finite count, pot: potential-only records (ke < 0) per call, and
// pot[nhalos] > 0 when some call has any
// (and the build's counters: all zero but the node count, one id per call's
// root; nothing reads them before k_roots)
__global__ void k_root_init(int32_t *box, int32_t *bad, int32_t *pot, int nhalos,
                            int32_t *counters) {
    int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h < kNumCounters) counters[h] = h == kNodeCount ? nhalos : 0;
    if (h == 0) pot[nhalos] = 0;
    if (h >= nhalos) return;
    for (int k = 0; k < 3; k++) {
        box[6 * h + k] = float_key(__int_as_float(0x7f800000));       // +inf
        box[6 * h + 3 + k] = float_key(__int_as_float((int)0xff800000));  // -inf
    }
    bad[h] = 0;
    pot[h] = 0;
}

// The records into float4 (x, y, z, record index), each call's tight box and
// non-finite and potential-only counts; and each record's sort key for the
// bound pass (potential-only flag above the r2 bits), read here where the
// records stream in order.
__global__ __launch_bounds__(kTileThreads) void k_gather(
    const struct potential *__restrict__ po, const int64_t *__restrict__ hfirst,
    const int64_t *__restrict__ hcount, const RootTile *__restrict__ tiles,
    float4 *__restrict__ A, int32_t *__restrict__ box, int32_t *__restrict__ bad,
    int32_t *__restrict__ pot, int32_t nhalos, uint64_t *__restrict__ rkey) {
    __shared__ float s_lo[3][kTileThreads / kWave], s_hi[3][kTileThreads / kWave];
    __shared__ int s_bad[kTileThreads / kWave], s_pot[kTileThreads / kWave];
    const RootTile t = tiles[blockIdx.x];
    const int64_t first = hfirst[t.halo];
    const int64_t end = first + hcount[t.halo];
    float lo[3], hi[3];
    for (int k = 0; k < 3; k++) {
        lo[k] = __int_as_float(0x7f800000);
        hi[k] = __int_as_float((int)0xff800000);
    }
    int nbad = 0, npot = 0;
    const int rounds = root_tile_records(hcount[t.halo]) / kTileThreads;
    for (int r = 0; r < rounds; r++) {
        int64_t i = first + t.off + r * kTileThreads + threadIdx.x;
        if (i >= end) break;
        const float *q = po[i].pos;
        float x = q[0], y = q[1], z = q[2];
        const bool potonly = po[i].ke < 0.0f;
        npot += potonly ? 1 : 0;
        rkey[i] = ((uint64_t)(potonly ? 1 : 0) << 32) | (uint64_t)__float_as_uint(po[i].r2);
        A[i] = make_float4(x, y, z, __int_as_float((int32_t)i));
        if (finite3(x, y, z)) {
            lo[0] = fminf(lo[0], x); hi[0] = fmaxf(hi[0], x);
            lo[1] = fminf(lo[1], y); hi[1] = fmaxf(hi[1], y);
            lo[2] = fminf(lo[2], z); hi[2] = fmaxf(hi[2], z);
        } else {
            nbad++;
        }
    }
    const int w = threadIdx.x / kWave;
    for (int k = 0; k < 3; k++) {
        float a = wave_min(lo[k]), b = wave_max(hi[k]);
        if (lane_id() == 0) {
            s_lo[k][w] = a;
            s_hi[k][w] = b;
        }
    }
    int nb = wave_sum(nbad), np_ = wave_sum(npot);
    if (lane_id() == 0) {
        s_bad[w] = nb;
        s_pot[w] = np_;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float a[3], b[3];
        int tb = 0, tp = 0;
        for (int k = 0; k < 3; k++) {
            a[k] = s_lo[k][0];
            b[k] = s_hi[k][0];
        }
        for (int j = 1; j < kTileThreads / kWave; j++) {
            for (int k = 0; k < 3; k++) {
                a[k] = fminf(a[k], s_lo[k][j]);
                b[k] = fmaxf(b[k], s_hi[k][j]);
            }
        }
        for (int j = 0; j < kTileThreads / kWave; j++) {
            tb += s_bad[j];
            tp += s_pot[j];
        }
        for (int k = 0; k < 3; k++) {
            atomicMin(&box[6 * t.halo + k], float_key(a[k]));
            atomicMax(&box[6 * t.halo + 3 + k], float_key(b[k]));
        }
        if (tb) atomicAdd(&bad[t.halo], tb);
        if (tp) {
            atomicAdd(&pot[t.halo], tp);
            atomicOr(&pot[nhalos], 1);
        }
    }
}

struct BuildArgs {
    Node *nodes;
    int32_t *parent;
    int32_t *sides;         // per position: a partition's points listed by side
    int32_t *leaf_of;
    float4 *fin;            // final tree order
    Task *small_next;       // wavefront subtree tasks
    Task *group_next;       // workgroup subtree tasks
    Task *big;              // append-only
    int2 *tiles;            // append-only (task index, offset)
    int32_t *fat;           // leaves of more than kFatLeaf points
    int32_t *counters;
    // per call-size bucket (tune_bucket): nodes above bucket_big points are
    // split by the level passes; subtrees of at most bucket_wave points are
    // built by one wavefront (32 or 64)
    int32_t bucket_big[kTuneBuckets];
    int32_t bucket_wave[kTuneBuckets];
    int32_t cap_small, cap_group, cap_big, cap_tiles, cap_nodes, cap_fat;
};

__device__ void note_fat_leaf(const BuildArgs &a, int32_t id, int32_t count) {
    if (count <= kFatLeaf) return;
    int32_t k = atomicAdd(&a.counters[kFatCount], 1);
    if (k < a.cap_fat) a.fat[k] = id;
    else atomicOr(&a.counters[kErrFlags], kErrCapacity);
}

// Node ids and small-task slots are allocated together: counters[kNodeCount]
// and counters[kSmallNext] are adjacent 32-bit halves of one 64-bit counter,
// so a split costs one atomic round trip.
__device__ __forceinline__ uint64_t alloc_nodes_and_small(const BuildArgs &a, int32_t nodes,
                                                          int32_t small) {
    static_assert(kNodeCount == 0 && kSmallNext == 1, "packed counter layout");
    return atomicAdd(reinterpret_cast<unsigned long long *>(a.counters),
                     (unsigned long long)nodes | ((unsigned long long)small << 32));
}

__device__ Task make_task(int32_t id, const float *lo, const float *hi, int32_t depth) {
    Task t;
    t.node = id;
    t.dim = split_dim(lo, hi);
    t.lim = split_lim(lo, hi, t.dim);
    t.depth = depth;
    t.tile0 = 0;
    t.ntiles = 0;
    t.pad[0] = t.pad[1] = 0;
    return t;
}

// The launch setting of a call's nodes (its size bucket's).
struct Sizes {
    int32_t big;   // nodes above this many points: split levels
    int32_t wave;  // subtrees of at most this many points: one wavefront
};
__device__ __forceinline__ Sizes sizes_of(const BuildArgs &a, int32_t bucket) {
    bucket = min(max(bucket, 0), kTuneBuckets - 1);
    return Sizes{a.bucket_big[bucket], a.bucket_wave[bucket]};
}

// Subtree tasks: a node of more than 10 and at most s.wave points is built
// by one wavefront, a larger one of at most s.big points by one workgroup.
// Each kind has its own list.
__device__ __forceinline__ bool wave_sized(const Sizes &s, int32_t n) {
    return n > kLeafPoints && n <= s.wave && n <= s.big;
}
__device__ __forceinline__ bool group_sized(const Sizes &s, int32_t n) {
    return n > s.wave && n <= s.big;
}

// Queues node `id` (tight box known) at a slot already allocated in the
// list of its kind; the task carries the node's range, so that the subtree
// kernels can pick their tasks without reading the node.
__device__ void push_task_at(const BuildArgs &a, Task *list, int32_t cap, int32_t slot, int32_t id,
                             const float *lo, const float *hi, int32_t depth, int32_t first,
                             int32_t count) {
    if (slot >= cap) {
        atomicOr(&a.counters[kErrFlags], kErrCapacity);
        return;
    }
    Task t = make_task(id, lo, hi, depth);
    t.pad[0] = first;
    t.pad[1] = count;
    list[slot] = t;
}
__device__ __forceinline__ void push_small_at(const BuildArgs &a, int32_t slot, int32_t id,
                                              const float *lo, const float *hi, int32_t depth,
                                              int32_t first, int32_t count) {
    push_task_at(a, a.small_next, a.cap_small, slot, id, lo, hi, depth, first, count);
}
__device__ __forceinline__ void push_group_at(const BuildArgs &a, int32_t slot, int32_t id,
                                              const float *lo, const float *hi, int32_t depth,
                                              int32_t first, int32_t count) {
    push_task_at(a, a.group_next, a.cap_group, slot, id, lo, hi, depth, first, count);
}

// A big-task slot and its tiles are reserved together: counters[kBigNext]
// and counters[kTileNext] are the two halves of one 64-bit counter.
__device__ __forceinline__ uint64_t alloc_big_and_tiles(const BuildArgs &a, int32_t ntiles) {
    static_assert(kTileNext == kBigNext + 1 && (kBigNext & 1) == 0, "packed counter layout");
    return atomicAdd(reinterpret_cast<unsigned long long *>(a.counters + kBigNext),
                     1ull | ((unsigned long long)ntiles << 32));
}

// Queues a node of more than its bucket's split size with its tiles; the
// task keeps the bucket (pad[0]) for its children.
__device__ void push_big(const BuildArgs &a, int32_t id, const float *lo, const float *hi,
                         int32_t count, int32_t depth, int32_t bucket) {
    Task t = make_task(id, lo, hi, depth);
    t.pad[0] = bucket;
    const int32_t nt = (count + kTile - 1) / kTile;
    const uint64_t al = alloc_big_and_tiles(a, nt);
    const int32_t bi = (int32_t)al, t0 = (int32_t)(al >> 32);
    if (bi >= a.cap_big || t0 + nt > a.cap_tiles) {
        atomicOr(&a.counters[kErrFlags], kErrCapacity);
        return;
    }
    t.tile0 = t0;
    t.ntiles = nt;
    a.big[bi] = t;
    for (int32_t j = 0; j < nt; j++) a.tiles[t0 + j] = make_int2(bi, j * kTile);
}

// A big task queued by a whole wavefront (wavefront-uniform arguments) at a
// task slot and tiles its caller reserved (alloc_big_and_tiles); the lanes
// write the tiles.
__device__ void push_big_wave_at(const BuildArgs &a, int32_t bi, int32_t t0, int32_t id,
                                 const float *lo, const float *hi, int32_t count, int32_t depth,
                                 int32_t bucket) {
    const int lane = lane_id();
    const int32_t nt = (count + kTile - 1) / kTile;
    if (bi >= a.cap_big || t0 + nt > a.cap_tiles) {
        if (lane == 0) atomicOr(&a.counters[kErrFlags], kErrCapacity);
        return;
    }
    if (lane == 0) {
        Task t = make_task(id, lo, hi, depth);
        t.tile0 = t0;
        t.ntiles = nt;
        t.pad[0] = bucket;
        a.big[bi] = t;
    }
    for (int32_t j = lane; j < nt; j += kWave) a.tiles[t0 + j] = make_int2(bi, j * kTile);
}

__device__ __forceinline__ void write_node(Node *nd, const float *lo, const float *hi, int32_t first,
                           int32_t count, int32_t skip) {
    Node n;
    for (int k = 0; k < 3; k++) {
        n.lo[k] = lo[k];
        n.hi[k] = hi[k];
        n.com[k] = 0.0f;
    }
    n.mass = 0.0f;
    n.dmin2 = 0.0f;
    n.dmin = 0.0f;
    n.first = first;
    n.count = count;
    n.left = -1;
    n.skip = skip;
    *nd = n;
}

// Root nodes, one thread per call.  A call with non-finite points is listed
// for k_roots_bad; every other call gets its root node here, its points in
// tree order when it is a single leaf, and its root queued as a task.  The
// subtree-task slots of a wavefront's calls are taken with one atomic.
__device__ __forceinline__ void root_of_call(int h, const int64_t *__restrict__ hfirst,
                                             const int64_t *__restrict__ hcount,
                                             const int32_t *__restrict__ box,
                                             const int32_t *__restrict__ bad,
                                             const float4 *__restrict__ A,
                                             int32_t *__restrict__ badlist, int nhalos,
                                             const BuildArgs &a) {
    const bool v = h < nhalos;
    int32_t first = 0, nfin = 0, bucket = 0;
    bool isbad = false;
    if (v) {
        first = (int32_t)hfirst[h];
        const int32_t count = (int32_t)hcount[h];
        const int32_t nbad = bad[h];
        nfin = count - nbad;
        isbad = nbad > 0;
        bucket = tune_bucket(count);
    }
    const bool ok = v && !isbad;
    const Sizes sz = sizes_of(a, bucket);
    const bool wsmall = ok && wave_sized(sz, nfin), gsmall = ok && group_sized(sz, nfin);
    const uint64_t ms = ballot(wsmall), mg = ballot(gsmall);
    int32_t slot0 = 0, gslot0 = 0;
    if (lane_id() == 0) {
        if (ms) slot0 = (int32_t)(alloc_nodes_and_small(a, 0, __popcll(ms)) >> 32);
        if (mg) gslot0 = atomicAdd(&a.counters[kGroupNext], __popcll(mg));
    }
    slot0 = __shfl(slot0, 0, 64);
    gslot0 = __shfl(gslot0, 0, 64);
    if (isbad) {
        const int32_t k = atomicAdd(&a.counters[kBadRoots], 1);
        badlist[k] = h;
    }
    float lo[3], hi[3];
    for (int k = 0; k < 3; k++) {
        lo[k] = ok && nfin ? key_float(box[6 * h + k]) : 0.0f;
        hi[k] = ok && nfin ? key_float(box[6 * h + 3 + k]) : 0.0f;
    }
    // roots above their split size, one after another: the lanes write the
    // tiles (one thread writing the 2,050 of a 2.1M-record call took 55 us)
    uint64_t big = ballot(ok && nfin > sz.big);
    while (big) {
        const int l = __builtin_ctzll(big);
        big &= big - 1;
        float blo[3], bhi[3];
        for (int k = 0; k < 3; k++) {
            blo[k] = lane_float(lo[k], l);
            bhi[k] = lane_float(hi[k], l);
        }
        const int32_t n = __builtin_amdgcn_readlane(nfin, l);
        uint64_t al = 0;
        if (lane_id() == 0) al = alloc_big_and_tiles(a, (n + kTile - 1) / kTile);
        al = read_lane(al, 0);
        push_big_wave_at(a, (int32_t)al, (int32_t)(al >> 32), __builtin_amdgcn_readlane(h, l), blo,
                         bhi, n, 0, __builtin_amdgcn_readlane(bucket, l));
    }
    if (!ok) return;
    if (nfin <= kLeafPoints) {
        for (int32_t i = 0; i < nfin; i++) {
            a.fin[first + i] = A[first + i];
            a.leaf_of[first + i] = h;
        }
    }
    write_node(a.nodes + h, lo, hi, first, nfin, -1);
    a.parent[h] = -1;
    if (wsmall) push_small_at(a, slot0 + rank_below(ms), h, lo, hi, 0, first, nfin);
    else if (gsmall) push_group_at(a, gslot0 + rank_below(mg), h, lo, hi, 0, first, nfin);
}

__global__ __launch_bounds__(256) void k_roots(const int64_t *__restrict__ hfirst,
                                               const int64_t *__restrict__ hcount,
                                               const int32_t *__restrict__ box,
                                               const int32_t *__restrict__ bad,
                                               const float4 *__restrict__ A,
                                               int32_t *__restrict__ badlist, int nhalos,
                                               BuildArgs a) {
    root_of_call(blockIdx.x * blockDim.x + threadIdx.x, hfirst, hcount, box, bad, A, badlist,
                 nhalos, a);
}

// The listed calls with non-finite points, one workgroup each: removal of
// the non-finite records to the tail in the order of the reference's swap
// loop (src/fast3tree.c:875-887), root node, root queued or finished as a
// leaf.
__device__ __forceinline__ void roots_of_bad_calls(const int64_t *__restrict__ hfirst,
                                                   const int64_t *__restrict__ hcount,
                                                   const int32_t *__restrict__ box,
                                                   const int32_t *__restrict__ bad,
                                                   float4 *__restrict__ A,
                                                   const int32_t *__restrict__ badlist,
                                                   int32_t nlist, const BuildArgs &a) {
    __shared__ int s_cnt[2][4];
    for (int32_t li = blockIdx.x; li < nlist; li += gridDim.x) {
        const int h = badlist[li];
        const int32_t first = (int32_t)hfirst[h];
        const int32_t count = (int32_t)hcount[h];
        const int32_t nbad = bad[h];
        const int32_t nfin = count - nbad;
        float lo[3], hi[3];
        for (int k = 0; k < 3; k++) {
            lo[k] = nfin ? key_float(box[6 * h + k]) : 0.0f;
            hi[k] = nfin ? key_float(box[6 * h + 3 + k]) : 0.0f;
        }
        // finite | non-finite in the order of the reference's swap loop
        // (inplace_dest): pass 0 lists the positions by class in the stable
        // order, pass 1 moves every point to its slot in the final array;
        // then the finite part goes back into A for splitting
        const int w = threadIdx.x / kWave;
        const int32_t *sd = a.sides + first;
        for (int pass = 0; pass < 2; pass++) {
            int32_t runf = 0, runb = 0;
            for (int32_t base = 0; base < count; base += 256) {
                int32_t i = base + threadIdx.x;
                bool vv = i < count;
                float4 p = vv ? A[first + i] : make_float4(0, 0, 0, 0);
                bool f = vv && finite3(p.x, p.y, p.z);
                bool bb = vv && !f;
                uint64_t mf = ballot(f), mb = ballot(bb);
                if (lane_id() == 0) {
                    s_cnt[0][w] = __popcll(mf);
                    s_cnt[1][w] = __popcll(mb);
                }
                __syncthreads();
                int of = 0, ob = 0, tf = 0, tb = 0;
                for (int j = 0; j < 4; j++) {
                    if (j < w) {
                        of += s_cnt[0][j];
                        ob += s_cnt[1][j];
                    }
                    tf += s_cnt[0][j];
                    tb += s_cnt[1][j];
                }
                if (vv) {
                    const int32_t rank = f ? runf + of + rank_below(mf) : runb + ob + rank_below(mb);
                    if (pass == 0) {
                        a.sides[first + (f ? rank : nfin + rank)] = i;
                    } else {
                        const int32_t d = first + inplace_dest(i, f, rank, count, nfin,
                                                               [&](int32_t k) { return sd[k]; });
                        a.fin[d] = p;
                        if (!f) a.leaf_of[d] = -1;
                    }
                }
                runf += tf;
                runb += tb;
                __syncthreads();
            }
        }
        __syncthreads();
        // A keeps the compact finite points of every call (the direct kernel
        // reads them there; the split levels read them when nfin > 10)
        for (int32_t i = threadIdx.x; i < nfin; i += 256) A[first + i] = a.fin[first + i];
        if (nfin <= kLeafPoints)
            for (int32_t i = threadIdx.x; i < nfin; i += 256) a.leaf_of[first + i] = h;
        if (threadIdx.x == 0) {
            write_node(a.nodes + h, lo, hi, first, nfin, -1);
            a.parent[h] = -1;
            const int32_t bucket = tune_bucket((int32_t)hcount[h]);
            const Sizes sz = sizes_of(a, bucket);
            if (nfin > sz.big) {
                push_big(a, h, lo, hi, nfin, 0, bucket);
            } else if (wave_sized(sz, nfin)) {
                const uint64_t old = alloc_nodes_and_small(a, 0, 1);
                push_small_at(a, (int32_t)(old >> 32), h, lo, hi, 0, first, nfin);
            } else if (group_sized(sz, nfin)) {
                push_group_at(a, atomicAdd(&a.counters[kGroupNext], 1), h, lo, hi, 0, first, nfin);
            }
        }
        __syncthreads();
    }
}
__global__ __launch_bounds__(256) void k_roots_bad(const int64_t *__restrict__ hfirst,
                                                   const int64_t *__restrict__ hcount,
                                                   const int32_t *__restrict__ box,
                                                   const int32_t *__restrict__ bad,
                                                   float4 *__restrict__ A,
                                                   const int32_t *__restrict__ badlist,
                                                   BuildArgs a) {
    roots_of_bad_calls(hfirst, hcount, box, bad, A, badlist, a.counters[kBadRoots], a);
}

// k_roots, k_roots_bad and k_levels_init of a single call, in one launch of
// one workgroup (a call of 134 records is bound by its launches).
__device__ void level_done(int32_t *c, int32_t *lv, int32_t level);
__device__ void levels_init(int32_t *c, int32_t *lv);
__global__ __launch_bounds__(256) void k_root_one(const int64_t *__restrict__ hfirst,
                                                  const int64_t *__restrict__ hcount,
                                                  const int32_t *__restrict__ box,
                                                  const int32_t *__restrict__ bad,
                                                  float4 *__restrict__ A,
                                                  int32_t *__restrict__ badlist,
                                                  int32_t *__restrict__ lv, BuildArgs a) {
    root_of_call(threadIdx.x, hfirst, hcount, box, bad, A, badlist, 1, a);
    __threadfence();
    __syncthreads();
    if (bad[0] > 0) roots_of_bad_calls(hfirst, hcount, box, bad, A, badlist, 1, a);
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) levels_init(a.counters, lv);
}

// ------------------------------------------------------------ small tasks

// Writes the two children of a split node and queues those that need a
// split: small ones at slots P, P + 1 (allocated with the node ids), big ones
// at task slots B, B + 1 with their tiles from T0.
// Called by a whole wavefront with wavefront-uniform arguments.  P, G, B
// and T0 are reserved by the caller in the wavefront and workgroup subtree
// lists and the big-task list.
__device__ void make_children(const BuildArgs &a, const Task &t, const Node &nd, int32_t L,
                              int32_t P, int32_t G, int32_t B, int32_t T0, int32_t nl,
                              const float *loL, const float *hiL, const float *loR,
                              const float *hiR) {
    const int32_t nr = nd.count - nl;
    const Sizes sz = sizes_of(a, t.pad[0]);
    if (lane_id() == 0) {
        write_node(a.nodes + L, loL, hiL, nd.first, nl, L + 1);
        write_node(a.nodes + L + 1, loR, hiR, nd.first + nl, nr, nd.skip);
        a.parent[L] = a.parent[L + 1] = t.node;
        a.nodes[t.node].left = L;
        if (wave_sized(sz, nl)) push_small_at(a, P++, L, loL, hiL, t.depth + 1, nd.first, nl);
        if (group_sized(sz, nl)) push_group_at(a, G++, L, loL, hiL, t.depth + 1, nd.first, nl);
        if (wave_sized(sz, nr)) push_small_at(a, P, L + 1, loR, hiR, t.depth + 1, nd.first + nl, nr);
        if (group_sized(sz, nr)) push_group_at(a, G, L + 1, loR, hiR, t.depth + 1, nd.first + nl, nr);
    }
    // big children at the task slots from B and the tiles from T0 (left first)
    if (nl > sz.big) push_big_wave_at(a, B, T0, L, loL, hiL, nl, t.depth + 1, t.pad[0]);
    if (nr > sz.big)
        push_big_wave_at(a, B + (nl > sz.big ? 1 : 0), T0 + (nl > sz.big ? (nl + kTile - 1) / kTile : 0),
                         L + 1, loR, hiR, nr, t.depth + 1, t.pad[0]);
}

__device__ __forceinline__ int32_t wave_pushes(const Sizes &s, int32_t nl, int32_t nr) {
    return (wave_sized(s, nl) ? 1 : 0) + (wave_sized(s, nr) ? 1 : 0);
}
__device__ __forceinline__ int32_t group_pushes(const Sizes &s, int32_t nl, int32_t nr) {
    return (group_sized(s, nl) ? 1 : 0) + (group_sized(s, nr) ? 1 : 0);
}

// ------------------------------------------------------------- subtrees
//
// A node of 65..kSmallMax points is finished by one workgroup, a node of at
// most 64 points by one wavefront.  Both keep the points in LDS.
//
// The workgroup has a thread per point and splits, level by level, only the
// nodes of more than 32 points (at most 31 at a time); each level lists the
// nodes' points by side, moves them to the in-place partition's order, and
// takes the children's tight boxes from segmented scans over runs of lanes,
// one LDS atomic per run and coordinate.  The nodes of at most 32 points are
// then finished by its wavefronts, packed up to 64 points to a wavefront, as
// the wavefront subtrees are, with no workgroup barrier: the deep levels, where most of a tree's nodes are,
// cost a wavefront's own latency.  Last come the nodes above: centres of mass
// bottom-up, dmin by a wavefront each over the final order.  (A workgroup of
// 256 threads that split every node level by level took 13 us a level and
// 162 us for a task of 1,024 points on its own; this one takes 72.  On the
// one-GPU catalogue, 6.71M points: 796 -> 731, 320 -> 249 and 281 -> 227 us
// for the three sizes, 160 -> 126 for the wavefront subtrees, whose segmented
// scans are on integers now.)
//
// Nodes are numbered locally and mapped onto a block of 2n - 2 global ids
// reserved for the subtree: the workgroup's levels first (2k ids for k
// splits), then 2m - 2 for each of its k + 1 parts of m points, in position
// order.  Ids that are not used are never referenced.

constexpr int kWaveTask = 64;   // subtrees up to this size: one wavefront
constexpr int kWaveMin = 32;    // the smallest wavefront/workgroup boundary (wave_max) used
constexpr int kRootSkip = -2;   // local skip pointer: the subtree root's own skip
constexpr uint8_t kNone8 = 0xff;
constexpr int kPart = 32;       // a workgroup splits nodes of more points than this level by level

// The workgroup subtree kernel comes in three sizes, for nodes of at most
// 256, 512 and 1,024 points: its LDS grows with the size, and the smaller
// sizes fit more workgroups on a CU.  The tasks are split by size into one
// list per kernel (k_group_classes) before the kernels run.
constexpr int kSubClasses = 3;
__host__ __device__ constexpr int sub_class(int32_t n) { return n > 512 ? 2 : (n > 256 ? 1 : 0); }
__device__ __forceinline__ uint64_t lanes_below(int i) {
    return i >= 64 ? ~0ull : ((1ull << i) - 1ull);
}

// bits [lf, lf + n) of a wavefront mask (lf + n <= 64)
__device__ __forceinline__ uint64_t lane_run(int lf, int n) {
    return (n >= 64 ? ~0ull : ((1ull << n) - 1ull)) << lf;
}

// Inclusive scan of v over this lane's run [seg, lane] of the wavefront
// (seg <= lane; runs are contiguous), on DPP moves: row_shr 1, 2, 4, 8
// within rows of 16, then row_bcast 15 and 31 across rows.
// On integers (float_key), where a move and a minimum are one instruction.
// (v_min_i32 with a lane move: 2 instructions a step against 6 on floats,
// whose minimum first makes both operands canonical.)
template <typename Op>
__device__ __forceinline__ int seg_scan(int v, int seg, Op op) {
    const int lane = lane_id(), r = lane & 15;
    int u;
    u = dpp_move<0x111>(v);
    if (r >= 1 && lane - 1 >= seg) v = op(v, u);
    u = dpp_move<0x112>(v);
    if (r >= 2 && lane - 2 >= seg) v = op(v, u);
    u = dpp_move<0x114>(v);
    if (r >= 4 && lane - 4 >= seg) v = op(v, u);
    u = dpp_move<0x118>(v);
    if (r >= 8 && lane - 8 >= seg) v = op(v, u);
    u = dpp_move<0x142>(v);  // row_bcast:15, used by rows 1 and 3
    if (((lane >> 4) & 1) && (lane & ~15) - 1 >= seg) v = op(v, u);
    u = dpp_move<0x143>(v);  // row_bcast:31, used by rows 2 and 3
    if (lane >= 32 && 31 >= seg) v = op(v, u);
    return v;
}

// ---- one wavefront, at most 64 points
//
// One point per lane, the points of one subtree or of several whose points
// follow each other.  Each level, every lane tests its point against its
// node's split plane; ballots give the left counts and the stable listing (a
// node's points occupy a contiguous run of lanes), and the children's tight
// boxes come from segmented scans across the lanes.  The node table stays in
// LDS with local ids (the roots, then children in pairs, levels in order).
// Centres of mass and dmin are computed with a lane per node, summing the
// node's points in tree order, the order of the reference's loops.

constexpr int kWaveNodes = 2 * kWaveTask;  // a tree over n points has at most 2n - 1 nodes
constexpr int kSkipRoot = 128;             // skip >= this: that of root skip - kSkipRoot
static_assert(kWaveNodes <= kSkipRoot && kSkipRoot + kWaveTask < kNone8, "local ids fit a byte");

struct WaveTree {
    union {
        float lim[kWaveNodes];     // split planes, while the levels run
        float com[3][kWaveNodes];  // then the centres of mass
    };
    float mass[kWaveNodes];
    uint8_t dim[kWaveNodes], lf[kWaveNodes], cnt[kWaveNodes];
    uint8_t left[kWaveNodes], skip[kWaveNodes];  // left: kNone8 for a leaf
    uint8_t lev[kWaveNodes];     // each node's level
    uint8_t st[kWaveTask];       // a level's points by side, node by node
};

// v, as a value that the compiler knows nothing about.
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A wavefront's LDS accesses complete in order; the compiler has to keep
// them so.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The subtrees of `nroots` nodes over the n points p of the lanes [0, n), in
// tree order from position `first` on.  Root r (id(r), its skip pointer
// skip(r)) holds the lanes from the r-th set bit of `heads` to the next; with
// one root (kMany false) its split plane (dim, lim) is given.  Node ids [base, base + 2 (n - nroots)) (fits:
// they are there; else the root stays a leaf and the error is flagged).  P: n
// points of LDS.  Writes the points' order and leaves and every node's record
// but the roots' boxes; the roots' centres and masses end in W.com[.][r],
// W.mass[r].
template <bool kMany, class Id, class Skip>
__device__ __forceinline__ void wave_subtree(const BuildArgs &a, WaveTree &W, float4 *P, float4 p, int n,
                             uint64_t heads, int nroots, int root_dim, float root_lim, int32_t first, int32_t base,
                             bool fits, double particle_mass, Id &&root_id, Skip &&root_skip) {
    const int lane = lane_id();
    const bool v = lane < n;
    const int root = kMany ? __popcll(heads & lanes_below(lane + 1)) - 1 : 0;
    // this lane's node: its run of lanes [lf, lf + c)
    int lf = 0, c = n, nid = root, M = nroots, nlev = 0;
    if constexpr (kMany) {
        lf = 63 - __builtin_clzll(heads & lanes_below(lane + 1));
        const uint64_t after = heads & ~lanes_below(lane + 1);
        c = (after ? __builtin_ctzll(after) : n) - lf;
    }
    auto gid = [&](int j) -> int32_t { return j < nroots ? root_id(j) : base + j - nroots; };
    // the tight box of each run of the lanes `in`, in its last lane
    auto boxes = [&](bool in, float (&lo)[3], float (&hi)[3]) {
        auto mn = [](int x, int y) { return min(x, y); };
        auto mx = [](int x, int y) { return max(x, y); };
        const int seg = in ? lf : lane;
        const int kx = float_key(p.x), ky = float_key(p.y), kz = float_key(p.z);
        lo[0] = key_float(seg_scan(kx, seg, mn));
        lo[1] = key_float(seg_scan(ky, seg, mn));
        lo[2] = key_float(seg_scan(kz, seg, mn));
        hi[0] = key_float(seg_scan(kx, seg, mx));
        hi[1] = key_float(seg_scan(ky, seg, mx));
        hi[2] = key_float(seg_scan(kz, seg, mx));
    };
    if constexpr (kMany) {
        float lo[3], hi[3];
        boxes(v, lo, hi);
        if (v && lane == lf + c - 1) {
            const int dm = split_dim(lo, hi);
            W.lf[root] = (uint8_t)lf;
            W.cnt[root] = (uint8_t)c;
            W.dim[root] = (uint8_t)dm;
            W.lim[root] = split_lim(lo, hi, dm);
            W.left[root] = kNone8;
            W.lev[root] = 0;
            W.skip[root] = (uint8_t)(kSkipRoot + root);
        }
    } else if (lane == 0) {
        W.lf[0] = 0;
        W.cnt[0] = (uint8_t)n;
        W.dim[0] = (uint8_t)root_dim;
        W.lim[0] = root_lim;
        W.left[0] = kNone8;
        W.lev[0] = 0;
        W.skip[0] = kSkipRoot;
    }
    wave_sync();
    bool pend = v && c > kLeafPoints;
    while (ballot(pend)) {
        // src/fast3tree.c:751-774 (partition), 805-809 (failed split)
        bool gl = false;
        if (pend) gl = comp(p, W.dim[nid]) <= W.lim[nid];
        const uint64_t mL = ballot(gl);
        const uint64_t mN = pend ? lane_run(lf, c) : 0ull;
        const int nl = __popcll(mL & mN);
        const bool split = pend && nl > 0 && nl < c;
        const uint64_t mH = ballot(split && lane == lf);
        const int C = M + 2 * __popcll(mH & lanes_below(lf));
        // the in-place partition's order (inplace_dest), from the node's
        // points listed by side
        const uint64_t below = mN & lanes_below(lane);
        const int rank = gl ? __popcll(mL & below) : __popcll(~mL & below);
        if (split) W.st[lf + (gl ? rank : nl + rank)] = (uint8_t)(lane - lf);
        wave_sync();
        if (split) {
            P[lf + inplace_dest(lane - lf, gl, rank, c, nl,
                                [&](int k) { return (int)W.st[lf + k]; })] = p;
            if (lane == lf) {
                W.lf[C] = (uint8_t)lf;
                W.cnt[C] = (uint8_t)nl;
                W.lf[C + 1] = (uint8_t)(lf + nl);
                W.cnt[C + 1] = (uint8_t)(c - nl);
                W.left[C] = W.left[C + 1] = kNone8;
                W.lev[C] = W.lev[C + 1] = (uint8_t)(nlev + 1);
                W.skip[C] = (uint8_t)(C + 1);
                W.skip[C + 1] = W.skip[nid];
                W.left[nid] = (uint8_t)C;
            }
        }
        wave_sync();
        if (split) {  // the point that came here, and its node
            p = P[lane];
            const bool right = lane - lf >= nl;
            nid = C + (right ? 1 : 0);
            lf += right ? nl : 0;
            c = right ? c - nl : nl;
        }
        if (mH) {
            M += 2 * __popcll(mH);
            nlev++;
        }
        // tight boxes of the new children
        float lo[3], hi[3];
        boxes(split, lo, hi);
        if (split && lane == lf + c - 1) {
            const int dm = split_dim(lo, hi);
            W.dim[nid] = (uint8_t)dm;
            W.lim[nid] = split_lim(lo, hi, dm);
            if (fits) {
                Node *g = a.nodes + base + nid - nroots;
                for (int d = 0; d < 3; d++) {
                    g->lo[d] = lo[d];
                    g->hi[d] = hi[d];
                }
            }
        }
        wave_sync();
        pend = split && c > kLeafPoints;
    }
    // every lane's node is a leaf now (its box is there already)
    if (M > nroots && !fits) {  // out of node ids: the root stays a leaf
        if (lane == 0) {
            atomicOr(&a.counters[kErrFlags], kErrCapacity);
            W.left[0] = kNone8;
        }
        M = nroots;
        nlev = 0;
        nid = root;
    }
    if (v) {
        P[lane] = p;
        a.fin[first + lane] = p;
        a.leaf_of[first + lane] = gid(nid);
    }
    wave_sync();
    // leaf centres: f64 sums in tree order (src/potential.c:100-107)
    for (int j = lane; j < M; j += kWave) {
        if (W.left[j] != kNone8) continue;
        const int lf = W.lf[j], c = W.cnt[j];
        double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll 5
        for (int i = lf; i < lf + c; i++) {
            const float4 q = P[i];
            sx += (double)q.x;
            sy += (double)q.y;
            sz += (double)q.z;
        }
        const double dn = (double)c;
        W.com[0][j] = sx != 0.0 ? (float)(sx / dn) : 0.0f;
        W.com[1][j] = sy != 0.0 ? (float)(sy / dn) : 0.0f;
        W.com[2][j] = sz != 0.0 ? (float)(sz / dn) : 0.0f;
        W.mass[j] = (float)(particle_mass * dn);
    }
    wave_sync();
    // internal centres, deepest level first (src/potential.c:115-122: float,
    // right term first); a lane keeps its two nodes' places, so that a level
    // is one round of table reads
    const bool two = lane + kWave < M;
    const int lev0 = lane < M ? W.lev[lane] : -1, lev1 = two ? W.lev[lane + kWave] : -1;
    const int left0 = lane < M ? W.left[lane] : kNone8, left1 = two ? W.left[lane + kWave] : kNone8;
    for (int L = nlev - 1; L >= 0; L--) {
        for (int h = 0; h < 2; h++) {
            const int cl = h ? left1 : left0;
            if ((h ? lev1 : lev0) != L || cl == kNone8) continue;
            const int j = lane + kWave * h;
            const float ml = W.mass[cl], mr = W.mass[cl + 1];
            const float m = ml + mr;
            for (int d = 0; d < 3; d++) {
                const float rr = W.com[d][cl + 1] * mr;
                const float ll = W.com[d][cl] * ml;
                W.com[d][j] = m != 0.0f ? (rr + ll) / m : 0.0f;
            }
            W.mass[j] = m;
        }
        wave_sync();
    }
    // dmin over each node's points in tree order (src/potential.c:71-82),
    // then the node records: every field but the box (the root's is its
    // creator's, the others were written with their level)
    for (int j = lane; j < M; j += kWave) {
        const int lf = W.lf[j], c = W.cnt[j];
        const float com[3] = {W.com[0][j], W.com[1][j], W.com[2][j]};
        double big = 0.0, sum = 0.0;
#pragma unroll 4
        for (int i = lf; i < lf + c; i++) {
            const double d = d2_ref(com, P[i]);
            big = d > big ? d : big;
            sum += d;
        }
        Node nd;
        finish_dmin(&nd, big, sum, c);
        const int cl = W.left[j], sk = W.skip[j];
        const int32_t id = gid(j);
        Node *g = a.nodes + id;
        for (int d = 0; d < 3; d++) g->com[d] = com[d];
        g->mass = W.mass[j];
        g->dmin2 = nd.dmin2;
        g->first = first + lf;
        g->count = c;
        g->left = cl != kNone8 ? base + cl - nroots : -1;
        g->skip = sk >= kSkipRoot ? root_skip(sk - kSkipRoot) : base + sk - nroots;
        g->dmin = nd.dmin;
        if (cl != kNone8)
            a.parent[base + cl - nroots] = a.parent[base + cl + 1 - nroots] = id;
    }
    wave_sync();
}

// Splits the workgroup subtree tasks by size into the lists of the three
// kernel sizes: list c at out + c * cap_group, counted in counters[kClassNext + c].
// Each task also gets its node ids here, 2n - 2 for n points (the most a
// subtree can need; ids it does not use are never referenced), the first
// kept in tile0: one atomic per wavefront instead of one per subtree.
__device__ __forceinline__ void group_class(int32_t k, int32_t n, const Task *__restrict__ in,
                                            const BuildArgs &a, Task *__restrict__ out) {
    if (k - lane_id() >= n) return;  // whole wavefronts past the list
    Task t;
    int c = -1;
    int32_t need = 0;
    if (k < n) {
        t = in[k];
        c = sub_class(t.pad[1]);
        need = 2 * t.pad[1] - 2;
    }
    const int32_t incl = wave_scan_add(need);
    int32_t ids = 0;
    if (lane_id() == kWave - 1)
        ids = (int32_t)alloc_nodes_and_small(a, incl, 0);
    t.tile0 = read_lane(ids, kWave - 1) + incl - need;
    for (int q = 0; q < kSubClasses; q++) {
        const uint64_t m = ballot(c == q);
        if (!m) continue;
        int32_t base = 0;
        if (lane_id() == 0) base = atomicAdd(&a.counters[kClassNext + q], __popcll(m));
        base = __shfl(base, 0, 64);
        if (c == q) out[(int64_t)q * a.cap_group + base + rank_below(m)] = t;
    }
}
__global__ __launch_bounds__(256) void k_group_classes(const Task *__restrict__ in, BuildArgs a,
                                                       Task *__restrict__ out) {
    group_class(blockIdx.x * blockDim.x + threadIdx.x, min(a.counters[kGroupNext], a.cap_group), in,
                a, out);
}

// A node of more than kPart points of the workgroup's current level.
struct SubEntry {
    float lim;          // split plane, from the node's tight box
    int16_t loc;        // local node id
    int16_t lf, n, nl;  // first point (subtree-relative), points, left count
    int16_t skip;       // local skip pointer
    uint8_t split, dim; // whether both sides hold points; split dimension
};

template <int kCap>
struct SubLds {
    static constexpr int kWaves = kCap / kWave;
    static constexpr int kAct = kCap / (kPart + 1);  // nodes of more than kPart points at a time
    static_assert(2 * kAct <= kWave, "a lane per child");
    // local nodes whose table entries fit here
    static constexpr int kTop = (3 * kCap / 16 + kWave - 1) / kWave * kWave;
    float4 P[kCap];
    WaveTree wt[kWaves];
    union {
        uint16_t st[kCap];      // a level's points by side, node by node
        float4 cm[kTop];        // then the local nodes' centres of mass
    };
    // a part (a node of at most kPart points, or a larger leaf), at its first
    // position; n: of the leaves of more than 64 points, else 0
    int16_t part_id[kCap], part_skip[kCap], wide_n[kCap];
    uint16_t lvl[kCap + 2];     // first local id of each level
    int16_t top_left[kTop], top_lf[kTop], top_n[kTop];
    SubEntry e[2][kAct];
    int32_t box[2 * kAct][6];   // the children's tight boxes, float keys
    uint8_t map[2 * kAct];      // a child slot's place among the next level's nodes
    uint64_t mask[kWaves], head[kWaves];
    int32_t na[2], M, nlev, next;
};

// One workgroup per task of the list `cls` (nodes of at most kCap points), a
// thread per point.  Bound by the latency of a task: LDS (77 KB at 1,024
// points) and registers leave 8 wavefronts per SIMD at every size.  At the 64
// registers of that a thread spills some 100 bytes (734 MB of HBM traffic a
// launch of the 1,024-point size on the one-GPU catalogue, against 315 MB for
// the kernel with 256 threads); with more registers and fewer wavefronts it was
// slower (1,162 us against 731).
template <int kCap>
__global__ __launch_bounds__(kCap, 8) void k_subtree(const float4 *__restrict__ A,
                                                     const float4 *__restrict__ B,
                                                     const Task *__restrict__ tasks, BuildArgs a,
                                                     double particle_mass, int cls) {
    constexpr int kWaves = SubLds<kCap>::kWaves, kTop = SubLds<kCap>::kTop;
    __shared__ SubLds<kCap> S;
    const int tid = threadIdx.x, lane = lane_id(), w = uniform(tid / kWave);
    const int32_t ntasks = a.counters[kClassNext + cls];
    const float inf = __int_as_float(0x7f800000);
    // A dynamic queue over the list: thread 0 takes the workgroup's next
    // entry when it starts the current one.  Entries are taken from the end
    // of the list: the largest subtrees (children of the big nodes of the
    // last split levels) are queued last and should start first.
    if (tid == 0) S.next = atomicAdd(&a.counters[kClassCursor + cls], 1);
    __syncthreads();
    for (int32_t k = uniform(S.next); k < ntasks; k = uniform(S.next)) {
        int32_t k_after = 0;
        if (tid == 0) k_after = atomicAdd(&a.counters[kClassCursor + cls], 1);
        const Task t = load_const(tasks + (ntasks - 1 - k));
        const int32_t first = t.pad[0], n = min(t.pad[1], kCap);
        const int32_t root_skip = load_const(&a.nodes[t.node].skip);
        const float4 *src = (t.depth & 1) ? B : A;
        const bool in = tid < n;
        const float4 p0 = in ? src[first + tid] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const int32_t base = t.tile0;  // 2n - 2 ids reserved by k_group_classes
        if (base + 2 * n - 2 > a.cap_nodes) {  // out of node ids: the root stays a leaf
            if (tid == 0) atomicOr(&a.counters[kErrFlags], kErrCapacity);
            if (in) {
                a.fin[first + tid] = p0;
                a.leaf_of[first + tid] = t.node;
            }
            __syncthreads();  // every wavefront has read the entry it is at
            if (tid == 0) S.next = k_after;
            __syncthreads();
            continue;
        }
        auto gid = [&](int j) { return j == 0 ? t.node : base + j - 1; };
        auto gskip = [&](int s) { return s == kRootSkip ? root_skip : gid(s); };
        if (in) S.P[tid] = p0;
        if (tid < kWaves) S.head[tid] = 0;
        __syncthreads();
        if (tid == 0) {
            S.M = 1;
            S.nlev = 0;
            S.lvl[0] = 0;
            S.lvl[1] = 1;
            S.top_left[0] = -1;
            S.top_lf[0] = 0;
            S.top_n[0] = (int16_t)n;
            if (n > kPart) {
                SubEntry e;
                e.loc = 0;
                e.lf = 0;
                e.n = (int16_t)n;
                e.nl = 0;
                e.skip = kRootSkip;
                e.split = 0;
                e.dim = (uint8_t)t.dim;
                e.lim = t.lim;
                S.e[0][0] = e;
                S.na[0] = 1;
            } else {  // one part
                S.na[0] = 0;
                S.head[0] = 1;
                S.part_id[0] = 0;
                S.wide_n[0] = 0;
                S.part_skip[0] = kRootSkip;
            }
        }
        __syncthreads();
        int cur = 0;
        int q = in && n > kPart ? 0 : -1;  // this position's node among the level's, if any
        for (int na; (na = uniform(S.na[cur])) > 0; cur ^= 1) {
            const int nxt = cur ^ 1;
            // what follows from the thread's number is found anew each level
            // (kept, it would not fit the registers)
            const int tid = opaque((int)threadIdx.x), lane = opaque(lane_id());
            SubEntry en;
            en.lf = en.n = 0;
            if (q >= 0) en = S.e[cur][q];
            float4 p = S.P[tid];
            // 1. left flags (src/fast3tree.c:751-774), one ballot per wavefront
            const bool gl = q >= 0 && comp(p, en.dim) <= en.lim;
            const uint64_t m = ballot(gl);
            if (lane == 0) S.mask[w] = m;
            for (int x = tid; x < 12 * na; x += kCap)
                (&S.box[0][0])[x] = float_key(x % 6 < 3 ? inf : -inf);
            __syncthreads();
            // 2. left flags before a position: the wavefronts' counts, scanned
            //    in every wavefront's lanes; the node's points by side
            int cnt = lane < kWaves ? __popcll(S.mask[lane]) : 0;
            const int excl = wave_scan_add(cnt) - cnt;  // lane kWaves: the total
            auto before = [&](int x) {
                const int c = x >> 6;
                const uint64_t mk = S.mask[min(c, kWaves - 1)];
                return __shfl(excl, c, 64) + (c < kWaves ? __popcll(mk & lanes_below(x & 63)) : 0);
            };
            const int s0 = before(en.lf), nl = before(en.lf + en.n) - s0;
            const int sl = __builtin_amdgcn_readlane(excl, w) + __popcll(m & lanes_below(lane)) - s0;
            // src/fast3tree.c:805-809: a split with an empty side is a leaf
            const bool split = q >= 0 && nl > 0 && nl < en.n;
            const int rel = tid - en.lf, rank = gl ? sl : rel - sl;
            if (split) S.st[en.lf + (gl ? rank : nl + rank)] = (uint16_t)rel;
            if (q >= 0 && rel == 0) {
                S.e[cur][q].nl = (int16_t)nl;
                S.e[cur][q].split = split ? 1 : 0;
            }
            __syncthreads();
            // 3. the points to the in-place partition's order (inplace_dest)
            if (split) {
                const int dst = en.lf + inplace_dest(rel, gl, rank, en.n, nl,
                                                     [&](int x) { return (int)S.st[en.lf + x]; });
                S.P[dst] = p;
            }
            __syncthreads();
            // 4. tight boxes of the children
            int slot = 0, lf = tid;
            if (split) {  // the point that came here, and its child
                p = S.P[tid];
                slot = 2 * q + (rel >= nl ? 1 : 0);
                lf = en.lf + ((slot & 1) ? nl : 0);
            }
            if (ballot(split)) {
                const int chunk0 = tid - lane;
                const int sg = split ? (lf > chunk0 ? lf - chunk0 : 0) : lane;
                auto mn = [](int x, int y) { return min(x, y); };
                auto mx = [](int x, int y) { return max(x, y); };
                const int kx = float_key(p.x), ky = float_key(p.y), kz = float_key(p.z);
                const int l0 = seg_scan(kx, sg, mn), l1 = seg_scan(ky, sg, mn),
                          l2 = seg_scan(kz, sg, mn);
                const int h0 = seg_scan(kx, sg, mx), h1 = seg_scan(ky, sg, mx),
                          h2 = seg_scan(kz, sg, mx);
                const int end = (slot & 1) ? en.lf + en.n : en.lf + nl;  // the child's
                if (split && (lane == kWave - 1 || tid + 1 == end)) {
                    atomicMin(&S.box[slot][0], l0);
                    atomicMin(&S.box[slot][1], l1);
                    atomicMin(&S.box[slot][2], l2);
                    atomicMax(&S.box[slot][3], h0);
                    atomicMax(&S.box[slot][4], h1);
                    atomicMax(&S.box[slot][5], h2);
                }
            }
            __syncthreads();
            // 5. wavefront 0, a lane per child: ids, records, the next level's
            //    nodes and the parts
            if (w == 0) {
                const bool v = lane < 2 * na;
                const int side = lane & 1;
                SubEntry pe;
                pe.split = 0;
                if (v) pe = S.e[cur][lane >> 1];
                const bool sp = v && pe.split;
                const uint64_t ms = ballot(sp);
                const int M = uniform(S.M), C = M + rank_below(ms);
                const int cn = side ? pe.n - pe.nl : pe.nl;
                const bool act = sp && cn > kPart;
                const uint64_t ma = ballot(act);
                if (sp) {
                    const int clf = pe.lf + (side ? pe.nl : 0);
                    const int skip = side ? pe.skip : C + 1;
                    float lo[3], hi[3];
                    for (int d = 0; d < 3; d++) {
                        lo[d] = key_float(S.box[lane][d]);
                        hi[d] = key_float(S.box[lane][3 + d]);
                    }
                    Node *g = a.nodes + gid(C);
                    for (int d = 0; d < 3; d++) {
                        g->lo[d] = lo[d];
                        g->hi[d] = hi[d];
                    }
                    a.parent[gid(C)] = gid(pe.loc);
                    if (!side) {
                        a.nodes[gid(pe.loc)].left = gid(C);
                        if (pe.loc < kTop) S.top_left[pe.loc] = (int16_t)C;
                    }
                    if (C < kTop) {
                        S.top_left[C] = -1;
                        S.top_lf[C] = (int16_t)clf;
                        S.top_n[C] = (int16_t)cn;
                    }
                    S.map[lane] = act ? (uint8_t)rank_below(ma) : kNone8;
                    if (act) {
                        g->first = first + clf;
                        g->count = cn;
                        g->skip = gskip(skip);
                        SubEntry ne;
                        ne.loc = (int16_t)C;
                        ne.lf = (int16_t)clf;
                        ne.n = (int16_t)cn;
                        ne.nl = 0;
                        ne.skip = (int16_t)skip;
                        ne.split = 0;
                        ne.dim = (uint8_t)split_dim(lo, hi);
                        ne.lim = split_lim(lo, hi, ne.dim);
                        S.e[nxt][rank_below(ma)] = ne;
                    } else {
                        S.part_id[clf] = (int16_t)C;
                        S.wide_n[clf] = 0;
                        S.part_skip[clf] = (int16_t)skip;
                        atomicOr((unsigned long long *)&S.head[clf >> 6], 1ull << (clf & 63));
                    }
                } else if (v && !side) {  // a failed split: a leaf
                    S.part_id[pe.lf] = pe.loc;
                    S.wide_n[pe.lf] = pe.n > kWave ? pe.n : 0;
                    S.part_skip[pe.lf] = pe.skip;
                    atomicOr((unsigned long long *)&S.head[pe.lf >> 6], 1ull << (pe.lf & 63));
                    if (pe.loc) a.nodes[gid(pe.loc)].left = -1;
                }
                if (lane == 0) {
                    S.na[nxt] = __popcll(ma);
                    if (ms) {
                        S.nlev = S.nlev + 1;
                        S.M = M + __popcll(ms);
                        S.lvl[S.nlev + 1] = (uint16_t)S.M;
                    }
                }
            }
            __syncthreads();
            q = split && S.map[slot] != kNone8 ? (int)S.map[slot] : -1;
        }
        // The parts, packed: a wavefront takes consecutive parts of together
        // at most 64 points.  A pack ends before the part that holds the 64th
        // position after its start; every wavefront follows the chain of packs
        // on the scalar unit and takes each kWaves-th.  Part i at position lf
        // has its node ids from base + (M - 1) + 2 (lf - i) on.
        const int M = uniform(S.M), nlev = uniform(S.nlev);
        auto cm_put = [&](int j, float x, float y, float z, float mass) {
            if (j < kTop) S.cm[j] = make_float4(x, y, z, mass);
        };
        const uint64_t hw = lane < kWaves ? S.head[lane] : 0ull;
        int at = 0, i0 = 0;  // a pack's first position and part
        for (int pk = 0; at < n; pk++) {
            int end = at + kWave;
            const int wide = uniform(S.wide_n[at]);
            if (wide) end = at + wide;
            if (end >= n) {
                end = n;
            } else if (!wide) {
                const int c = end >> 6;
                uint64_t hm = read_lane(hw, c) & lanes_below((end & 63) + 1);
                end = 64 * c + 63;
                if (!hm) {  // the part that holds it starts in the 64 positions before
                    hm = read_lane(hw, c - 1);
                    end -= 64;
                }
                end -= __builtin_clzll(hm);
            }
            const int m = end - at, c = at >> 6, sh = at & 63;
            // the pack's first positions, as a mask from `at` on
            uint64_t heads = read_lane(hw, c) >> sh;
            if (sh && c + 1 < kWaves) heads |= read_lane(hw, c + 1) << (64 - sh);
            if (m < kWave) heads &= lanes_below(m);
            const int nr = wide ? 1 : __popcll(heads);
            if (pk % kWaves == w) {
                if (!wide) {
                    const float4 x = lane < m ? S.P[at + lane] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    wave_subtree<true>(
                        a, S.wt[w], S.P + at, x, m, heads, nr, 0, 0.0f, first + at,
                        base + (M - 1) + 2 * (at - i0), true, particle_mass,
                        [&](int j) { return gid(S.part_id[at + S.wt[w].lf[j]]); },
                        [&](int j) { return gskip(S.part_skip[at + S.wt[w].lf[j]]); });
                    if (lane < nr)
                        cm_put(S.part_id[at + S.wt[w].lf[lane]], S.wt[w].com[0][lane],
                               S.wt[w].com[1][lane], S.wt[w].com[2][lane], S.wt[w].mass[lane]);
                } else {  // a leaf whose split failed: f64 sums in tree order
                    const int id = S.part_id[at];
                    for (int j = lane; j < m; j += kWave) {
                        a.fin[first + at + j] = S.P[at + j];
                        a.leaf_of[first + at + j] = gid(id);
                    }
                    double sx = 0.0, sy = 0.0, sz = 0.0;
                    for (int j = 0; j < m; j++) {
                        const float4 x = S.P[at + j];
                        sx += (double)x.x;
                        sy += (double)x.y;
                        sz += (double)x.z;
                    }
                    if (lane == 0) {
                        const double dn = (double)m;
                        const float cx = sx != 0.0 ? (float)(sx / dn) : 0.0f;
                        const float cy = sy != 0.0 ? (float)(sy / dn) : 0.0f;
                        const float cz = sz != 0.0 ? (float)(sz / dn) : 0.0f;
                        const float mass = (float)(particle_mass * dn);
                        Node *g = a.nodes + gid(id);
                        g->com[0] = cx;
                        g->com[1] = cy;
                        g->com[2] = cz;
                        g->mass = mass;
                        cm_put(id, cx, cy, cz, mass);
                    }
                }
            }
            at = end;
            i0 += nr;
        }
        if (tid == 0) S.next = k_after;
        if (M == 1 && n <= kWave) {  // one part: its wavefront did it all
            __syncthreads();
            continue;
        }
        __threadfence_block();
        __syncthreads();
        // the nodes above the parts: centres of mass, deepest level first
        // (src/potential.c:115-122: float, right term first), by one wavefront
        // (a level reads what this wavefront wrote at deeper levels, or the
        // parts' roots, made visible by the barrier above)
        struct Top {
            int left, lf, n;
        };
        auto top = [&](int j) {
            if (j < kTop) return Top{S.top_left[j], S.top_lf[j], S.top_n[j]};
            const Node *g = a.nodes + gid(j);
            const int32_t l = g->left;
            // a part's own children are not of the levels above
            return Top{l >= base && l < base + M - 1 ? l - base + 1 : -1, g->first - first, g->count};
        };
        auto cm_get = [&](int j) {
            if (j < kTop) return S.cm[j];
            const Node *g = a.nodes + gid(j);
            return make_float4(g->com[0], g->com[1], g->com[2], g->mass);
        };
        auto combine = [&](int j, int cl) {
            const float4 l = cm_get(cl), r = cm_get(cl + 1);
            const float m = l.w + r.w;
            float c[3];
            const float lc[3] = {l.x, l.y, l.z}, rc[3] = {r.x, r.y, r.z};
            for (int d = 0; d < 3; d++) {
                const float rr = rc[d] * r.w;
                const float ll = lc[d] * l.w;
                c[d] = m != 0.0f ? (rr + ll) / m : 0.0f;
            }
            Node *g = a.nodes + gid(j);
            for (int d = 0; d < 3; d++) g->com[d] = c[d];
            g->mass = m;
            cm_put(j, c[0], c[1], c[2], m);
        };
        if (w == 0) {
            int left[kTop / kWave];  // a lane's nodes' children, read ahead
            for (int h = 0; h < kTop / kWave; h++) {
                const int j = lane + kWave * h;
                left[h] = j < M ? S.top_left[j] : -1;
            }
            int l1 = M;
            for (int L = nlev; L >= 0; L--) {
                const int l0 = uniform(S.lvl[L]);
                for (int h = 0; h < kTop / kWave; h++) {
                    const int j = lane + kWave * h;
                    if (j >= l0 && j < l1 && left[h] >= 0) combine(j, left[h]);
                }
                for (int j = max(l0, kTop) + lane; j < l1; j += kWave) {
                    const int cl = top(j).left;
                    if (cl >= 0) combine(j, cl);
                }
                wave_sync();
                l1 = l0;
            }
        }
        __threadfence_block();
        __syncthreads();
        // their dmin (src/potential.c:71-82), a wavefront each
        for (int j0 = w; j0 < M; j0 += kWaves * kWave) {
            double my_big = 0.0, my_sum = 0.0;  // lane k's: of node j0 + k kWaves
            int my_n = 0;
            for (int k = 0; k < kWave; k++) {
                const int j = j0 + k * kWaves;
                if (j >= M) break;
                const Top tp = top(j);
                if (tp.left < 0 && tp.n <= kWave) continue;  // a part
                const float4 c4 = cm_get(j);
                const float com[3] = {c4.x, c4.y, c4.z};
                double big = 0.0, sum = 0.0;
                for (int i = lane; i < tp.n; i += kWave) {
                    const double d = d2_ref(com, S.P[tp.lf + i]);
                    big = d > big ? d : big;
                    sum += d;
                }
                big = wave_max(big);
                sum = wave_sum(sum);
                if (lane == k) {
                    my_big = big;
                    my_sum = sum;
                    my_n = tp.n;
                }
            }
            if (my_n > 0) finish_dmin(a.nodes + gid(j0 + lane * kWaves), my_big, my_sum, my_n);
        }
        __syncthreads();
    }
}

// Node ids of the wavefront subtrees, assigned before they are built: a
// subtree of n points gets 2n - 2 ids (the most it can need; ids it does not
// use are never referenced) from one block above every id in use.  Task k's
// first id is counters[kWaveIdBase] plus the exclusive prefix of the needs
// before it: k_wave_need, the library's exclusive scan, then k_wave_base.
// The subtree kernel then needs no atomic per task.
__host__ __device__ __forceinline__ int32_t wave_ids(int32_t n) { return 2 * n - 2; }
__global__ void k_wave_need(const Task *__restrict__ tasks, BuildArgs a, int32_t *__restrict__ need,
                            int32_t m) {
    const int32_t ntasks = min(a.counters[kSmallNext], a.cap_small);
    for (int32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < m; k += gridDim.x * blockDim.x)
        need[k] = k < ntasks ? wave_ids(tasks[k].pad[1]) : 0;
}
// after the scan (off holds cap_small + 1 entries): the block of ids
__global__ void k_wave_base(BuildArgs a, const int32_t *__restrict__ off) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const int32_t ntasks = min(a.counters[kSmallNext], a.cap_small);
    const int32_t base0 = a.counters[kNodeCount];
    a.counters[kWaveIdBase] = base0;
    a.counters[kNodeCount] = base0 + off[ntasks];
}

// One wavefront per task: subtrees of at most 64 points whose parent the
// split levels made.  Under 5 KB of LDS, so that 8 wavefronts fit per SIMD:
// the nodes' boxes go to their global records as they are found (only each
// node's split plane stays), parents are written from the parent's side.
__global__ __launch_bounds__(kWave, 8) void k_subtree_wave(const float4 *__restrict__ A,
                                                        const float4 *__restrict__ B,
                                                        const Task *__restrict__ tasks,
                                                        BuildArgs a, double particle_mass,
                                                        const int32_t *__restrict__ wave_off) {
    __shared__ float4 P[kWaveTask];
    __shared__ WaveTree W;
    const int lane = lane_id();
    const int32_t ntasks = min(a.counters[kSmallNext], a.cap_small);
    const int32_t id_base = a.counters[kWaveIdBase];
    // tasks k = blockIdx.x, blockIdx.x + gridDim.x, ...: they are all small
    // and alike, and a fixed stride needs no queue atomic per task
    for (int32_t k = blockIdx.x; k < ntasks; k += gridDim.x) {
        const Task t = tasks[k];
        const int32_t n = t.pad[1];
        if (n > kWaveTask) {  // never queued here; guards the lane-per-point layout
            if (lane == 0) atomicOr(&a.counters[kErrFlags], kErrBadTree);
            continue;
        }
        // the task carries the root's range and split plane, so the points
        // load at once; the root's node record is needed only at the end
        const float4 *src = (t.depth & 1) ? B : A;
        const float4 p = lane < n ? src[t.pad[0] + lane] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const int32_t skip = a.nodes[t.node].skip;
        // the task's node ids (2n - 2 from the scan); a subtree that does not
        // fit keeps its root as a leaf (checked once the levels are done)
        const int32_t base = id_base + wave_off[k];
        wave_subtree<false>(a, W, P, p, n, 1ull, 1, t.dim, t.lim, t.pad[0], base,
                            base + wave_ids(n) <= a.cap_nodes, particle_mass,
                            [&](int) { return t.node; }, [&](int) { return skip; });
    }
}

// -------------------------------------------------------------- big tasks

__device__ void block_box_reduce(float (*lo)[3], float (*hi)[3], int &nl, TilePart *out) {
    __shared__ float s_lo[2][3][kTileThreads / kWave], s_hi[2][3][kTileThreads / kWave];
    __shared__ int s_n[kTileThreads / kWave];
    const int w = threadIdx.x / kWave;
    for (int s = 0; s < 2; s++)
        for (int k = 0; k < 3; k++) {
            float a = wave_min(lo[s][k]), b = wave_max(hi[s][k]);
            if (lane_id() == 0) {
                s_lo[s][k][w] = a;
                s_hi[s][k][w] = b;
            }
        }
    int n = wave_sum(nl);
    if (lane_id() == 0) s_n[w] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        TilePart tp;
        tp.nleft = 0;
        tp.pad[0] = tp.pad[1] = tp.pad[2] = 0;
        for (int s = 0; s < 2; s++)
            for (int k = 0; k < 3; k++) {
                float a = s_lo[s][k][0], b = s_hi[s][k][0];
                for (int j = 1; j < kTileThreads / kWave; j++) {
                    a = fminf(a, s_lo[s][k][j]);
                    b = fmaxf(b, s_hi[s][k][j]);
                }
                tp.lo[s][k] = a;
                tp.hi[s][k] = b;
            }
        for (int j = 0; j < kTileThreads / kWave; j++) tp.nleft += s_n[j];
        *out = tp;
    }
    __syncthreads();
}

__device__ void big_count_tile(const float4 *__restrict__ src, const int2 *__restrict__ tiles,
                               const Task *__restrict__ big, const Node *__restrict__ nodes,
                               TilePart *__restrict__ parts, int32_t ti);

// Count pass over the tiles of split level `level`.
__global__ __launch_bounds__(kTileThreads) void k_big_count(const float4 *__restrict__ src,
                                                            const int2 *__restrict__ tiles,
                                                            const Task *__restrict__ big,
                                                            const Node *__restrict__ nodes,
                                                            TilePart *__restrict__ parts,
                                                            const int32_t *__restrict__ lv,
                                                            int32_t level) {
    const int32_t t1 = lvl_tile(lv)[level];
    for (int32_t ti = lvl_tile(lv)[level - 1] + blockIdx.x; ti < t1; ti += gridDim.x)
        big_count_tile(src, tiles, big, nodes, parts, ti);
}

__device__ void big_count_tile(const float4 *__restrict__ src, const int2 *__restrict__ tiles,
                               const Task *__restrict__ big, const Node *__restrict__ nodes,
                               TilePart *__restrict__ parts, int32_t ti) {
    const int2 tl = tiles[ti];
    const Task t = big[tl.x];
    const Node nd = nodes[t.node];
    float lo[2][3], hi[2][3];
    for (int s = 0; s < 2; s++)
        for (int k = 0; k < 3; k++) {
            lo[s][k] = __int_as_float(0x7f800000);
            hi[s][k] = __int_as_float((int)0xff800000);
        }
    int nl = 0;
    for (int r = 0; r < kTile / kTileThreads; r++) {
        int32_t i = tl.y + r * kTileThreads + threadIdx.x;
        if (i >= nd.count) break;
        float4 p = src[nd.first + i];
        int s = comp(p, t.dim) <= t.lim ? 0 : 1;
        nl += 1 - s;
        lo[s][0] = fminf(lo[s][0], p.x); hi[s][0] = fmaxf(hi[s][0], p.x);
        lo[s][1] = fminf(lo[s][1], p.y); hi[s][1] = fmaxf(hi[s][1], p.y);
        lo[s][2] = fminf(lo[s][2], p.z); hi[s][2] = fmaxf(hi[s][2], p.z);
    }
    block_box_reduce(lo, hi, nl, parts + ti);
}

// The split of big task bi (t, its node nd), by one wavefront once its
// tiles are counted: the left count and the children's boxes from the tiles'
// parts (lanes over tiles), then the children.  The node ids and subtree
// slots, the workgroup-subtree slots and the big children's task slots and
// tiles are reserved by three lanes at once (one round trip).
__device__ void split_task(const TilePart *__restrict__ parts, BigSplit *__restrict__ res,
                           const BuildArgs &a, int32_t bi, const Task &t, const Node &nd) {
    const int lane = lane_id();
    const float inf = __int_as_float(0x7f800000), ninf = __int_as_float((int)0xff800000);
    float lo[2][3] = {{inf, inf, inf}, {inf, inf, inf}};
    float hi[2][3] = {{ninf, ninf, ninf}, {ninf, ninf, ninf}};
    int32_t nl = 0;
    for (int32_t j = lane; j < t.ntiles; j += kWave) {
        const TilePart *p = parts + t.tile0 + j;
        nl += p->nleft;
        for (int s = 0; s < 2; s++)
            for (int d = 0; d < 3; d++) {
                lo[s][d] = fminf(lo[s][d], p->lo[s][d]);
                hi[s][d] = fmaxf(hi[s][d], p->hi[s][d]);
            }
    }
    nl = wave_sum(nl);
    for (int s = 0; s < 2; s++)
        for (int d = 0; d < 3; d++) {
            lo[s][d] = wave_min(lo[s][d]);
            hi[s][d] = wave_max(hi[s][d]);
        }
    // nl, nd and the reduced boxes are wavefront-uniform from here on
    BigSplit r;
    r.nleft = nl;
    r.left = -1;
    r.leafL = r.leafR = 0;
    if (nl == 0 || nl == nd.count) {
        if (lane == 0) note_fat_leaf(a, t.node, nd.count);
    } else {
        const int32_t nr = nd.count - nl;
        const Sizes sz = sizes_of(a, t.pad[0]);
        const int32_t ng = group_pushes(sz, nl, nr);
        const int32_t ntl = nl > sz.big ? (nl + kTile - 1) / kTile : 0;
        const int32_t ntr = nr > sz.big ? (nr + kTile - 1) / kTile : 0;
        const int32_t nbig = (ntl ? 1 : 0) + (ntr ? 1 : 0);
        uint64_t al = 0, bal = 0;
        int32_t G = 0;
        if (lane == 0) al = alloc_nodes_and_small(a, 2, wave_pushes(sz, nl, nr));
        if (lane == 1 && ng) G = atomicAdd(&a.counters[kGroupNext], ng);
        if (lane == 2 && nbig)
            bal = atomicAdd(reinterpret_cast<unsigned long long *>(a.counters + kBigNext),
                            (unsigned long long)nbig | ((unsigned long long)(ntl + ntr) << 32));
        al = read_lane(al, 0);
        G = read_lane(G, 1);
        bal = read_lane(bal, 2);
        const int32_t L = (int32_t)al, P = (int32_t)(al >> 32);
        if (L + 2 > a.cap_nodes) {
            if (lane == 0) atomicOr(&a.counters[kErrFlags], kErrCapacity);
        } else {
            r.left = L;
            r.leafL = nl <= kLeafPoints;
            r.leafR = nr <= kLeafPoints;
            make_children(a, t, nd, L, P, G, (int32_t)bal, (int32_t)(bal >> 32), nl, lo[0], hi[0],
                          lo[1], hi[1]);
        }
    }
    if (lane == 0) res[bi] = r;
}

// The two passes over one tile of a big task, with the points' ranks on
// their side of the plane in rounds of 256 (a block prefix of ballots):
//   kSides:   lists the node's points by side, a.sides[first + k] = the
//             position of the k-th left point, then of the right points
//             (the stable order).  Each workgroup takes its tile's left
//             prefix and the task's left total from the count pass's parts
//             (and keeps the prefix in its part for the scatter pass); the
//             workgroup of the task's first tile also splits the task.
//   kScatter: moves each point to the slot the reference's in-place
//             partition gives it (inplace_dest over that list).  Its first
//             workgroup moves the level state forward (level_done).
enum { kSides = 0, kScatter = 1 };

template <int kPass>
__device__ void big_tile_pass(const float4 *__restrict__ src, float4 *__restrict__ dst,
                              const int2 *__restrict__ tiles, const Task *__restrict__ big,
                              TilePart *__restrict__ parts, BigSplit *__restrict__ res,
                              const BuildArgs &a, int32_t ti);
__device__ void level_done(int32_t *c, int32_t *lv, int32_t level);

template <int kPass>
__global__ __launch_bounds__(kTileThreads) void k_big_tiles(
    const float4 *__restrict__ src, float4 *__restrict__ dst, const int2 *__restrict__ tiles,
    const Task *__restrict__ big, TilePart *__restrict__ parts, BigSplit *__restrict__ res,
    BuildArgs a, int32_t *__restrict__ lv, int32_t level) {
    // (the scatter pass makes no pushes: the counters it reads here are final)
    if (kPass == kScatter && blockIdx.x == 0 && threadIdx.x == 0) level_done(a.counters, lv, level);
    const int32_t t1 = lvl_tile(lv)[level];
    for (int32_t ti = lvl_tile(lv)[level - 1] + blockIdx.x; ti < t1; ti += gridDim.x)
        big_tile_pass<kPass>(src, dst, tiles, big, parts, res, a, ti);
}

template <int kPass>
__device__ void big_tile_pass(const float4 *__restrict__ src, float4 *__restrict__ dst,
                              const int2 *__restrict__ tiles, const Task *__restrict__ big,
                              TilePart *__restrict__ parts, BigSplit *__restrict__ res,
                              const BuildArgs &a, int32_t ti) {
    __shared__ int s_cnt[2][kTileThreads / kWave];
    const int2 tl = tiles[ti];
    const Task t = big[tl.x];
    const Node nd = a.nodes[t.node];
    const int w = threadIdx.x / kWave;
    int32_t lpre, nleft;
    BigSplit r;
    if (kPass == kSides) {
        // left points of the task's earlier tiles and of all its tiles (every
        // wavefront sums them: no barrier needed to share them)
        const int32_t me = tl.y / kTile;
        int32_t before = 0, all = 0;
        for (int32_t j = lane_id(); j < t.ntiles; j += kWave) {
            const int32_t c = parts[t.tile0 + j].nleft;
            before += j < me ? c : 0;
            all += c;
        }
        lpre = wave_sum(before);
        nleft = wave_sum(all);
        if (threadIdx.x == 0) parts[ti].pad[0] = lpre;
        if (me == 0 && w == 0) split_task(parts, res, a, tl.x, t, nd);
        if (nleft == 0 || nleft == nd.count) return;  // failed split: no listing
    } else {
        r = res[tl.x];
        nleft = r.nleft;
        if (r.left < 0) {  // failed split: the node is a leaf, its order unchanged
            for (int j = threadIdx.x; j < kTile; j += kTileThreads) {
                int32_t i = tl.y + j;
                if (i >= nd.count) break;
                a.fin[nd.first + i] = src[nd.first + i];
                a.leaf_of[nd.first + i] = t.node;
            }
            return;
        }
        lpre = parts[ti].pad[0];
    }
    const int32_t rpre = tl.y - lpre;
    int32_t runL = 0, runR = 0;
    for (int rr = 0; rr < kTile / kTileThreads; rr++) {
        int32_t i = tl.y + rr * kTileThreads + threadIdx.x;
        bool v = i < nd.count;
        float4 p = v ? src[nd.first + i] : make_float4(0, 0, 0, 0);
        bool f = v && comp(p, t.dim) <= t.lim;
        bool g = v && !f;
        uint64_t mL = ballot(f), mR = ballot(g);
        if (lane_id() == 0) {
            s_cnt[0][w] = __popcll(mL);
            s_cnt[1][w] = __popcll(mR);
        }
        __syncthreads();
        int oL = 0, oR = 0, tL = 0, tR = 0;
        for (int j = 0; j < kTileThreads / kWave; j++) {
            if (j < w) {
                oL += s_cnt[0][j];
                oR += s_cnt[1][j];
            }
            tL += s_cnt[0][j];
            tR += s_cnt[1][j];
        }
        if (v) {
            const int32_t rank = f ? lpre + runL + oL + rank_below(mL)
                                   : rpre + runR + oR + rank_below(mR);
            if (kPass == kSides) {
                a.sides[nd.first + (f ? rank : nleft + rank)] = i;
            } else {
                const int32_t *sd = a.sides + nd.first;
                const int32_t d = nd.first + inplace_dest(i, f, rank, nd.count, nleft,
                                                          [&](int32_t k) { return sd[k]; });
                const bool leaf = f ? r.leafL : r.leafR;  // left points land in [0, nleft)
                const int32_t id = f ? r.left : r.left + 1;
                if (leaf) {
                    a.fin[d] = p;
                    a.leaf_of[d] = id;
                } else {
                    dst[d] = p;
                }
            }
        }
        runL += tL;
        runR += tR;
        __syncthreads();
    }
}

// The level state on the device.  After the roots, level 1's big tasks and
// tiles are the pushes so far; after split level L's scatter pass (whose
// counters are final: the split happened in the sides pass), level L + 1's
// are the pushes of level L.  depth_end[L] records the node count (node
// ids grow with depth).  A dropped push (capacity) ends the levels.
__device__ void level_done(int32_t *c, int32_t *lv, int32_t level) {
    const int32_t nodes = c[kNodeCount];
    int32_t err = c[kErrFlags];
    if (level >= kMaxLevels) {
        atomicOr(&c[kErrFlags], kErrCapacity);
        err |= kErrCapacity;
    } else {
        lv[level] = nodes;
    }
    const bool stop = (err & kErrCapacity) != 0;
    int32_t *big = lvl_big(lv), *tile = lvl_tile(lv);
    big[level + 1] = stop ? big[level] : c[kBigNext];
    tile[level + 1] = stop ? tile[level] : c[kTileNext];
    c[kGlobalNodes] = nodes;
    if (level == 0 || c[kActive]) c[kLevel] = level + 1;  // a level with nothing to split adds no depth
    c[kActive] = big[level + 1] > big[level] ? 1 : 0;
}
__device__ void levels_init(int32_t *c, int32_t *lv) {
    lvl_big(lv)[0] = 0;
    lvl_tile(lv)[0] = 0;
    level_done(c, lv, 0);
}
__global__ void k_levels_init(int32_t *__restrict__ c, int32_t *__restrict__ lv) {
    if (threadIdx.x == 0 && blockIdx.x == 0) levels_init(c, lv);
}

// --------------------------------------------------------------- multipoles

// The multipole kernels take their sizes from the device counters (node
// count, fat-leaf count, per-depth node ranges, big tasks and tiles), so a
// whole build can be replayed from a graph.

// Leaves made by the split levels (at most 10 points): mass, centre
// (src/potential.c:100-107, f64 sums) and dmin (src/potential.c:71-82), one
// thread each.  Subtree nodes have ids at or above counters[kGlobalNodes]
// and are finished by their workgroup.
__global__ void k_leaf_com(Node *__restrict__ nodes, const float4 *__restrict__ fin,
                           const int32_t *__restrict__ counters, double particle_mass) {
    const int32_t nnodes = counters[kGlobalNodes];
    for (int32_t id = blockIdx.x * blockDim.x + threadIdx.x; id < nnodes;
         id += gridDim.x * blockDim.x) {
        const Node nd = nodes[id];
        if (nd.left >= 0 || nd.count <= 0 || nd.count > kLeafPoints) continue;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        for (int32_t i = 0; i < nd.count; i++) {
            const float4 p = fin[nd.first + i];
            s0 += (double)p.x;
            s1 += (double)p.y;
            s2 += (double)p.z;
        }
        const double n = (double)nd.count;
        float com[3];
        com[0] = s0 != 0.0 ? (float)(s0 / n) : 0.0f;
        com[1] = s1 != 0.0 ? (float)(s1 / n) : 0.0f;
        com[2] = s2 != 0.0 ? (float)(s2 / n) : 0.0f;
        double big = 0.0, sum = 0.0;
        for (int32_t i = 0; i < nd.count; i++) {
            const double d = d2_ref(com, fin[nd.first + i]);
            big = d > big ? d : big;
            sum += d;
        }
        Node *me = nodes + id;
        me->com[0] = com[0];
        me->com[1] = com[1];
        me->com[2] = com[2];
        me->mass = (float)(particle_mass * n);
        finish_dmin(me, big, sum, nd.count);
    }
}

// The same for leaves of more than kFatLeaf points (failed splits), one
// wavefront each.  Sums of floats in f64 are exact here, so the order of the
// wavefront reduction does not matter.
__global__ __launch_bounds__(256) void k_fat_leaf_com(Node *__restrict__ nodes,
                                                      const int32_t *__restrict__ list,
                                                      const int32_t *__restrict__ counters,
                                                      int32_t cap, const float4 *__restrict__ fin,
                                                      double particle_mass) {
    const int32_t nlist = min(counters[kFatCount], cap);
    const int32_t nw = (int32_t)(gridDim.x * blockDim.x / kWave);
    const int lane = lane_id();
    for (int32_t k = (int32_t)((blockIdx.x * blockDim.x + threadIdx.x) / kWave); k < nlist;
         k += nw) {
        const int32_t id = list[k];
        const Node nd = nodes[id];
        double s[3] = {0.0, 0.0, 0.0};
        for (int32_t i = lane; i < nd.count; i += kWave) {
            const float4 p = fin[nd.first + i];
            s[0] += (double)p.x;
            s[1] += (double)p.y;
            s[2] += (double)p.z;
        }
        for (int k2 = 0; k2 < 3; k2++) s[k2] = wave_sum(s[k2]);
        if (lane == 0) {
            const double n = (double)nd.count;
            Node *me = nodes + id;
            for (int k2 = 0; k2 < 3; k2++) me->com[k2] = s[k2] != 0.0 ? (float)(s[k2] / n) : 0.0f;
            me->mass = (float)(particle_mass * n);
        }
    }
}

// The device wall clock at this point of the stream.
__global__ void k_stamp(uint64_t *t, int i) {
    if (threadIdx.x == 0 && blockIdx.x == 0) t[i] = (uint64_t)wall_clock64();
}

// After the last split level of a recorded step: trees still being split
// need more levels than were recorded.
__global__ void k_depth_check(int32_t *__restrict__ c) {
    if (threadIdx.x == 0 && blockIdx.x == 0 && c[kActive]) c[kErrFlags] |= kErrDeep;
}

// Internal nodes of depth d: float mass and centre from the two children,
// right term first (src/potential.c:115-122).  Node ids grow with depth:
// depth d holds [depth_end[d - 1], depth_end[d]), depth 0 the roots; the
// host runs the depths deepest first.
__global__ void k_internal_com(Node *__restrict__ nodes, const int32_t *__restrict__ depth_end,
                               int32_t d) {
    const int32_t begin = d ? depth_end[d - 1] : 0, end = depth_end[d];
    for (int32_t id = begin + blockIdx.x * blockDim.x + threadIdx.x; id < end;
         id += gridDim.x * blockDim.x) {
        Node *me = nodes + id;
        const int32_t L = me->left;
        if (L < 0) continue;
        const Node *l = nodes + L, *r = nodes + L + 1;
        const float ml = l->mass, mr = r->mass;
        const float m = ml + mr;
        for (int k = 0; k < 3; k++) {
            const float rr = r->com[k] * mr;
            const float ll = l->com[k] * ml;
            me->com[k] = m != 0.0f ? (rr + ll) / m : 0.0f;
        }
        me->mass = m;
    }
}

// Tile partials of dmin for big nodes (every big task of every level), then
// k_dmin_big combines each node's.  The reference adds the points' distances
// in tree order; here a tile's are added across its threads and the tiles'
// across a wavefront's lanes, in another order but always the same.  The sums
// are f64, of terms of one sign (some 1e-15 of the sum apart), and dmin is
// rounded to a float: it moves by its last bit where the value is as near to a
// rounding boundary as that.
__global__ __launch_bounds__(kTileThreads) void k_dmin_tiles(const Node *__restrict__ nodes,
                                                             const float4 *__restrict__ fin,
                                                             const int2 *__restrict__ tiles,
                                                             const Task *__restrict__ big,
                                                             const int32_t *__restrict__ counters,
                                                             double2 *__restrict__ part) {
    __shared__ double s_b[kTileThreads / kWave], s_s[kTileThreads / kWave];
    const int32_t ntiles = counters[kTileNext];
    for (int32_t ti = blockIdx.x; ti < ntiles; ti += gridDim.x) {
        const int2 tl = tiles[ti];
        const Node nd = nodes[big[tl.x].node];
        double bmax = 0.0, sum = 0.0;
        for (int r = 0; r < kTile / kTileThreads; r++) {
            const int32_t i = tl.y + r * kTileThreads + threadIdx.x;
            if (i >= nd.count) break;
            const double d = d2_ref(nd.com, fin[nd.first + i]);
            bmax = d > bmax ? d : bmax;
            sum += d;
        }
        bmax = wave_max(bmax);
        sum = wave_sum(sum);
        const int w = threadIdx.x / kWave;
        if (lane_id() == 0) {
            s_b[w] = bmax;
            s_s[w] = sum;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double b = s_b[0], s = s_s[0];
            for (int j = 1; j < kTileThreads / kWave; j++) {
                b = s_b[j] > b ? s_b[j] : b;
                s += s_s[j];
            }
            part[ti] = make_double2(b, s);
        }
        __syncthreads();
    }
}

// A wavefront per node, a lane per tile (one thread per node read the 2,050
// partials of a 2.1M-record call's root one after another, 282 us).
__global__ __launch_bounds__(256) void k_dmin_big(Node *__restrict__ nodes,
                                                  const Task *__restrict__ big,
                                                  const int32_t *__restrict__ counters,
                                                  const double2 *__restrict__ part) {
    const int32_t nbig = counters[kBigNext];
    const int32_t nw = (int32_t)(gridDim.x * blockDim.x / kWave);
    for (int32_t k = uniform((int32_t)((blockIdx.x * blockDim.x + threadIdx.x) / kWave)); k < nbig;
         k += nw) {
        const Task t = load_const(big + k);
        double b = 0.0, s = 0.0;
        for (int32_t j = lane_id(); j < t.ntiles; j += kWave) {
            const double2 p = part[t.tile0 + j];
            b = p.x > b ? p.x : b;
            s += p.y;
        }
        b = wave_max(b);
        s = wave_sum(s);
        if (lane_id() == 0) finish_dmin(nodes + t.node, b, s, nodes[t.node].count);
    }
}

}  // namespace hp
