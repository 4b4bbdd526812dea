// hp_props.hip -- the halo property pass that follows the bound pass
// (src/properties.c:384-510, called for bound = 0 and bound = 1 by
// src/properties.c:552-553, with the defaults BOUND_PROPS = 1 and
// LIGHTCONE = 0), for every call of a batch at once.  calc_shape,
// calc_scale_radius and _calc_pseudo_evolution_masses are not part of it.
//
// The reference walks each call's records (sorted by r2) twice:
//   1. over every kept record (bound = 0) or every bound one, !(pe < ke)
//      (bound = 1), with the running count n: the density n / r^3 against
//      five thresholds and the virial one.  Each result is "n (or the index)
//      at the last record above a threshold", and vmax is the largest n / r
//      above the virial threshold from the first record above the main
//      threshold on (the first record reaching it wins ties).
//   2. over the bound records below dens_tot (the index of the last record
//      above the main threshold): angular momentum, running means of
//      position and velocity, the velocity dispersion, the half-mass index;
//      and estimate_total_energy (src/properties.c:328-349) over the records
//      with pe > ke below dens_tot.
// Here both walks are tile passes over the same scan tiles as the bound pass
// (2048 sorted records of one call, one wavefront each, rounds of 64 carried
// from lane 63), with per-call combines:
//   k_props_counts  bound and pe > ke counts per tile
//   k_props_prefix  per call: exclusive prefix of the tile counts
//   k_props_scan    walk 1 per tile: "last above" indices and counts as
//                   max-reductions (the running count is monotone), the
//                   vmax candidates as (value, first index) argmax
//   k_props_calls   per call: combine walk 1
//   k_props_sums    walk 2 per tile: f64 sums
//   k_props_final   per call: the halo fields
// Counts, indices, masses, radii and vmax are exact (the same IEEE
// operations on the same values).  The reference's running means, Welford
// dispersion and sequential f64 sums are restated as f64 sums of exact
// differences, which agree with them to f64 rounding.

#include "hp_internal.h"

#pragma clang fp contract(off)

namespace hp {

static_assert(sizeof(hp_halo_props) == 224 && offsetof(hp_halo_props, n_mdelta) == 192,
              "hp_halo_props layout");

constexpr double kVmaxConst = 6.55833746e-5;  // src/universal_constants.h:6
constexpr double kGc = 4.30117902e-9;         // src/universal_constants.h:4

// thresholds and constants of one property pass
struct PropArgs {
    double dens_thresh;   // particle_thresh_dens[0] * 4pi/3
    double d[4];          // particle_thresh_dens[1..4] * 4pi/3
    double rvir_thresh;   // particle_rvir_dens * 4pi/3
    double thresh0;       // particle_thresh_dens[0]
    double thresh3;       // particle_thresh_dens[3] (the second shape window)
    double rvir_dens;     // particle_rvir_dens
    double rvir_dens_z0;  // particle_rvir_dens_z0
    double force_res, particle_mass;
    float scale_now;
};

struct PropCount {
    int32_t nb;  // !(pe < ke)
    int32_t ns;  // pe > ke
};

// walk 1 partial of one tile
struct PropScan {
    int32_t last_all;      // last index with (j + 1) / r^3 > dens_thresh (all records)
    int32_t first0, last0; // first / last bound index with n / r^3 > dens_thresh
    int32_t n0;            // n at last0
    int32_t alt[4];        // n at the last bound index above d[k]
    int32_t vir;           // n at the last bound index above rvir_thresh
    int32_t j_all, j_after;
    double v_all;          // best n / r above rvir_thresh in the tile
    double v_after;        // the same from the tile's first index above dens_thresh on
    double pe_b;           // max of n^2 / r^1.5 (src/properties.c:369-373)
};

// per call, walk 1 combined
struct PropCall {
    int32_t kept;
    int32_t n_all;         // part_mdelta of the bound = 0 walk
    int32_t n0;            // part_mdelta of the bound = 1 walk
    int32_t dens_tot;
    int32_t alt[4];
    int32_t vir;
    int32_t j_vmax;        // -1: vmax stays 0
    double vmax;
    double pe_b;
};

// walk 2 partial of one tile
struct PropSums {
    double L[3];
    double sx[3];          // sum of x - centre (exact differences)
    double sv[3];          // sum of v - centre velocity
    double sv2[3];         // sum of (v - centre velocity)^2
    double ke;             // pe > ke records: sum of ke
    double phi_i;          // sum of particle_mass * i / r
    double phi_c;          // sum of (particle_mass / r) * (pe > ke records before i)
    int32_t n;             // bound records
    int32_t half;          // first bound index >= 1 with 2 n >= part_mdelta, else INT32_MAX
};

// a call's kept records, clamped to its record range (the plan's tables)
__device__ __forceinline__ int32_t call_kept(const hp_halo *halos, const int64_t *hcount,
                                             int32_t h) {
    const int64_t k = halos[h].kept;
    return (int32_t)(k < 0 ? 0 : (k > hcount[h] ? hcount[h] : k));
}

__device__ __forceinline__ double prop_radius(float r2, double force_res) {
    double r = sqrt((double)r2);
    return r < force_res ? force_res : r;
}

// (value, index): larger value wins, the smaller index on ties
__device__ __forceinline__ void arg_better(double &v, int32_t &j, double v2, int32_t j2) {
    if (v2 > v || (v2 == v && j2 < j)) {
        v = v2;
        j = j2;
    }
}

__device__ __forceinline__ void wave_arg_better(double &v, int32_t &j) {
    for (int o = 32; o > 0; o >>= 1) {
        const double v2 = __shfl_xor(v, o, 64);
        const int32_t j2 = __shfl_xor(j, o, 64);
        arg_better(v, j, v2, j2);
    }
}

// words of bound flags per tile, a word per 64 records
constexpr int kTileWords = kScanTile / kWave;

// What the passes over all records read, taken from the records once: r2 (4
// bytes), the bound flags (a bit, 1: !(pe < ke)) and the float offsets from
// the centre with the flag (16 bytes, the shapes).  The passes went through
// the records' 48 bytes each for themselves, six times.
struct PropReads {
    float *r2;
    uint64_t *bound;  // kTileWords per tile
    float4 *cd;
};

__global__ __launch_bounds__(kWave) void k_props_counts(const struct potential *__restrict__ srt,
                                                        const ScanTile *__restrict__ tiles,
                                                        int32_t ntiles,
                                                        const hp_halo *__restrict__ halos,
                                                        const int64_t *__restrict__ hfirst,
                                                        const int64_t *__restrict__ hcount,
                                                        PropCount *__restrict__ cnt,
                                                        PropReads out) {
    const int32_t t = blockIdx.x;
    if (t >= ntiles) return;
    const ScanTile st = tiles[t];
    const int64_t first = hfirst[st.call];
    const int32_t end = min(st.off + kScanTile, call_kept(halos, hcount, st.call));
    const float c0 = halos[st.call].pos[0], c1 = halos[st.call].pos[1], c2 = halos[st.call].pos[2];
    int32_t nb = 0, ns = 0;
    uint64_t *word = out.bound + (int64_t)kTileWords * t;
    for (int32_t base = st.off; base < end; base += kWave, word++) {
        const int32_t j = base + lane_id();
        bool b = false, sb = false;
        if (j < end) {
            const struct potential &r = srt[first + j];
            b = !(r.pe < (double)r.ke);
            sb = r.pe > (double)r.ke;
            out.r2[first + j] = r.r2;
            out.cd[first + j] =
                make_float4(r.pos[0] - c0, r.pos[1] - c1, r.pos[2] - c2, b ? 1.0f : 0.0f);
        }
        const uint64_t m = ballot(b);
        if (lane_id() == 0) *word = m;
        nb += __popcll(m);
        ns += __popcll(ballot(sb));
    }
    if (lane_id() == 0) cnt[t] = PropCount{nb, ns};
}

// set bits of m up to this lane's
__device__ __forceinline__ int32_t count_to_lane(uint64_t m) {
    return (int32_t)__builtin_amdgcn_mbcnt_hi(
               (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0)) +
           (int32_t)((m >> lane_id()) & 1);
}

// per call: exclusive prefix of the tile counts, in tile order
__global__ __launch_bounds__(kWave) void k_props_prefix(const int32_t *__restrict__ call_tile0,
                               const int32_t *__restrict__ call_ntiles, int32_t nh,
                               PropCount *__restrict__ cnt) {
    const int32_t h = lane_call(nh, call_ntiles);
    const int32_t t0 = h < nh ? call_tile0[h] : 0, nt = h < nh ? call_ntiles[h] : 0;
    if (nt <= kFewTiles) {
        int32_t nb = 0, ns = 0;
        for (int32_t t = t0; t < t0 + nt; t++) {
            const PropCount c = cnt[t];
            cnt[t] = PropCount{nb, ns};
            nb += c.nb;
            ns += c.ns;
        }
    }
    for_large_call(t0, nt, [&](int32_t first, int32_t n, bool) {
        int32_t nb = 0, ns = 0;
        for (int32_t base = 0; base < n; base += kWave) {
            const bool in = base + lane_id() < n;
            PropCount c = {0, 0};
            if (in) c = cnt[first + base + lane_id()];
            const int32_t b = wave_scan_add(c.nb), e = wave_scan_add(c.ns);
            if (in) cnt[first + base + lane_id()] = PropCount{nb + b - c.nb, ns + e - c.ns};
            nb += read_lane(b, kWave - 1);
            ns += read_lane(e, kWave - 1);
        }
    });
}

// bound records among a call's first n, from the tile counts before each tile
// and the flags
__device__ __forceinline__ int32_t bound_before(int32_t n, int32_t tile0,
                                                const PropCount *__restrict__ pre,
                                                const uint64_t *__restrict__ bound) {
    if (n <= 0) return 0;
    const int32_t t = tile0 + (n - 1) / kScanTile, k = (n - 1) % kScanTile + 1;
    const uint64_t *w = bound + (int64_t)kTileWords * t;
    int32_t c = pre[t].nb;
    for (int32_t i = 0; i < k / kWave; i++) c += __popcll(w[i]);
    if (k % kWave) c += __popcll(w[k / kWave] & ((1ull << (k % kWave)) - 1));
    return c;
}

// walk 1 (src/properties.c:402-431), one wavefront per tile
__global__ __launch_bounds__(kWave) void k_props_scan(const PropReads in,
                                                      const ScanTile *__restrict__ tiles,
                                                      int32_t ntiles,
                                                      const hp_halo *__restrict__ halos,
                                                      const int64_t *__restrict__ hfirst,
                                                      const int64_t *__restrict__ hcount,
                                                      const PropCount *__restrict__ pre,
                                                      PropArgs pa, PropScan *__restrict__ out) {
    const int32_t t = blockIdx.x;
    if (t >= ntiles) return;
    const ScanTile st = tiles[t];
    const int64_t first = hfirst[st.call];
    const int32_t end = min(st.off + kScanTile, call_kept(halos, hcount, st.call));
    const int lane = lane_id();
    int32_t carry = pre[t].nb;
    PropScan s;
    s.last_all = -1;
    s.first0 = INT32_MAX;
    s.last0 = -1;
    s.n0 = 0;
    for (int k = 0; k < 4; k++) s.alt[k] = 0;
    s.vir = 0;
    s.v_all = s.v_after = -1.0;
    s.j_all = s.j_after = INT32_MAX;
    s.pe_b = 0.0;
    bool seen0 = false;  // an index above dens_thresh earlier in this tile
    for (int32_t base = st.off; base < end; base += kWave) {
        const int32_t j = base + lane;
        const bool v = j < end;
        float r2 = 0.0f;
        if (v) r2 = in.r2[first + j];
        const uint64_t mb = in.bound[(int64_t)kTileWords * t + (base - st.off) / kWave];
        const bool b = (mb >> lane) & 1;
        const int32_t n = count_to_lane(mb) + carry;
        carry += __popcll(mb);
        const double r = prop_radius(r2, pa.force_res);
        const double r3 = r * r * r;
        if (v && (double)(j + 1) / r3 > pa.dens_thresh) s.last_all = j;
        const double cur = (double)n / r3;
        const bool c0 = b && cur > pa.dens_thresh;
        const uint64_t m0 = ballot(c0);
        const bool after = seen0 || (m0 & (lane == 63 ? ~0ull : ((2ull << lane) - 1ull))) != 0;
        seen0 = seen0 || m0 != 0;
        if (b) {
            // src/properties.c:365-373: unclamped radius
            double r32 = sqrt(sqrt((double)r2));
            r32 = r32 * r32 * r32;
            const double q = (double)((int64_t)n * (int64_t)n) / r32;
            s.pe_b = q > s.pe_b ? q : s.pe_b;
            if (c0) {
                s.first0 = min(s.first0, j);
                s.last0 = j;
                s.n0 = n;
            }
            for (int k = 0; k < 4; k++)
                if (cur > pa.d[k]) s.alt[k] = n;
            if (cur > pa.rvir_thresh) {
                s.vir = n;
                const double circ = (double)n / r;
                arg_better(s.v_all, s.j_all, circ, j);
                if (after) arg_better(s.v_after, s.j_after, circ, j);
            }
        }
    }
    // every field is monotone in j: max (or min) over the lanes
    s.last_all = wave_max(s.last_all);
    s.first0 = wave_min(s.first0);
    s.last0 = wave_max(s.last0);
    s.n0 = wave_max(s.n0);
    for (int k = 0; k < 4; k++) s.alt[k] = wave_max(s.alt[k]);
    s.vir = wave_max(s.vir);
    wave_arg_better(s.v_all, s.j_all);
    wave_arg_better(s.v_after, s.j_after);
    s.pe_b = wave_max(s.pe_b);
    if (lane == 0) out[t] = s;
}

__global__ __launch_bounds__(kWave) void k_props_calls(const int32_t *__restrict__ call_tile0,
                              const int32_t *__restrict__ call_ntiles, int32_t nh,
                              const hp_halo *__restrict__ halos,
                              const int64_t *__restrict__ hcount,
                              const PropScan *__restrict__ ts, PropCall *__restrict__ pc) {
    const int32_t h = lane_call(nh, call_ntiles);
    const bool v = h < nh;
    const int32_t t0 = v ? call_tile0[h] : 0, nt = v ? call_ntiles[h] : 0;
    PropCall c;
    int32_t last_all = -1, last0 = -1, n0 = 0;
    for (int k = 0; k < 4; k++) c.alt[k] = 0;
    c.vir = 0;
    c.pe_b = 0.0;
    double vm = -1.0;
    int32_t jm = INT32_MAX;
    // vmax counts from the first index above dens_thresh on: the part of
    // that tile after it, then whole tiles
    if (nt <= kFewTiles) {
        for (int32_t t = t0; t < t0 + nt; t++) {
            const PropScan &s = ts[t];
            last_all = max(last_all, s.last_all);
            if (last0 >= 0) arg_better(vm, jm, s.v_all, s.j_all);
            else if (s.last0 >= 0) arg_better(vm, jm, s.v_after, s.j_after);
            if (s.last0 >= 0) {
                last0 = s.last0;
                n0 = s.n0;
            }
            for (int k = 0; k < 4; k++) c.alt[k] = max(c.alt[k], s.alt[k]);
            c.vir = max(c.vir, s.vir);
            c.pe_b = s.pe_b > c.pe_b ? s.pe_b : c.pe_b;
        }
    }
    // every field of a tile is monotone over the tiles: maxima over the lanes
    for_large_call(t0, nt, [&](int32_t a, int32_t n, bool mine) {
        int32_t all = -1, l0 = -1, n_0 = 0, vir = 0, alt[4] = {0, 0, 0, 0}, j = INT32_MAX;
        double best = -1.0, pe_b = 0.0;
        bool seen = false;
        for (int32_t base = 0; base < n; base += kWave) {
            const bool in = base + lane_id() < n;
            const PropScan &s = ts[a + base + (in ? lane_id() : 0)];
            const uint64_t above = ballot(in && s.last0 >= 0);
            if (in) {
                all = max(all, s.last_all);
                l0 = max(l0, s.last0);
                n_0 = max(n_0, s.n0);
                for (int k = 0; k < 4; k++) alt[k] = max(alt[k], s.alt[k]);
                vir = max(vir, s.vir);
                pe_b = s.pe_b > pe_b ? s.pe_b : pe_b;
                const uint64_t before = above & ((1ull << lane_id()) - 1);
                if (seen || before) arg_better(best, j, s.v_all, s.j_all);
                else if (s.last0 >= 0) arg_better(best, j, s.v_after, s.j_after);
            }
            seen = seen || above != 0;
        }
        all = wave_max(all);
        l0 = wave_max(l0);
        n_0 = wave_max(n_0);
        for (int k = 0; k < 4; k++) alt[k] = wave_max(alt[k]);
        vir = wave_max(vir);
        pe_b = wave_max(pe_b);
        wave_arg_better(best, j);
        if (mine) {
            last_all = all;
            last0 = l0;
            n0 = n_0;
            for (int k = 0; k < 4; k++) c.alt[k] = alt[k];
            c.vir = vir;
            c.pe_b = pe_b;
            vm = best;
            jm = j;
        }
    });
    if (!v) return;
    c.kept = call_kept(halos, hcount, h);
    c.n_all = last_all + 1;
    c.n0 = n0;
    c.dens_tot = last0 >= 0 ? last0 : 0;
    c.j_vmax = jm == INT32_MAX ? -1 : jm;
    c.vmax = jm == INT32_MAX ? 0.0 : vm;
    pc[h] = c;
}

// walk 2 (src/properties.c:433-450, 127-137) and estimate_total_energy
// (src/properties.c:328-349) over [0, dens_tot)
__global__ __launch_bounds__(kWave) void k_props_sums(const struct potential *__restrict__ srt,
                                                      const ScanTile *__restrict__ tiles,
                                                      int32_t ntiles,
                                                      const hp_halo *__restrict__ halos,
                                                      const int64_t *__restrict__ hfirst,
                                                      const PropCount *__restrict__ pre,
                                                      const PropCall *__restrict__ pc, PropArgs pa,
                                                      PropSums *__restrict__ out) {
    const int32_t t = blockIdx.x;
    if (t >= ntiles) return;
    const ScanTile st = tiles[t];
    const hp_halo &hh = halos[st.call];
    const PropCall c = pc[st.call];
    const int64_t first = hfirst[st.call];
    const int32_t end = min(st.off + kScanTile, c.dens_tot);
    const float cen[6] = {hh.pos[0], hh.pos[1], hh.pos[2], hh.pos[3], hh.pos[4], hh.pos[5]};
    const int lane = lane_id();
    int32_t carry_b = pre[t].nb, carry_s = pre[t].ns;
    double acc[15] = {};
    int32_t nb_tile = 0, half = INT32_MAX;
    for (int32_t base = st.off; base < end; base += kWave) {
        const int32_t j = base + lane;
        const bool v = j < end;
        struct potential rec = {};
        if (v) rec = srt[first + j];
        const bool b = v && !(rec.pe < (double)rec.ke);
        const bool sb = v && rec.pe > (double)rec.ke;
        const uint64_t mb = ballot(b), ms = ballot(sb);
        const int32_t n = count_to_lane(mb) + carry_b;
        const int32_t ns = count_to_lane(ms) + carry_s;  // inclusive
        carry_b += __popcll(mb);
        carry_s += __popcll(ms);
        nb_tile += __popcll(mb);
        if (b) {
            const float *x = rec.pos;
            // src/properties.c:127-137: float differences and products
            acc[0] += (double)((x[1] - cen[1]) * (x[5] - cen[5]));
            acc[0] -= (double)((x[2] - cen[2]) * (x[4] - cen[4]));
            acc[1] += (double)((x[2] - cen[2]) * (x[3] - cen[3]));
            acc[1] -= (double)((x[0] - cen[0]) * (x[5] - cen[5]));
            acc[2] += (double)((x[0] - cen[0]) * (x[4] - cen[4]));
            acc[2] -= (double)((x[1] - cen[1]) * (x[3] - cen[3]));
            for (int k = 0; k < 3; k++) {
                const double dx = (double)x[k] - (double)cen[k];
                const double dv = (double)x[k + 3] - (double)cen[k + 3];
                acc[3 + k] += dx;
                acc[6 + k] += dv;
                acc[9 + k] += dv * dv;
            }
            if (j >= 1 && 2 * (int64_t)n >= (int64_t)c.n0) half = min(half, j);
        }
        if (sb) {
            const double r = prop_radius(rec.r2, pa.force_res);
            acc[12] += (double)rec.ke;
            acc[13] += pa.particle_mass * (double)j / r;
            acc[14] += (pa.particle_mass / r) * (double)(ns - 1);  // pe > ke records before j
        }
    }
    PropSums s;
    for (int k = 0; k < 3; k++) {
        s.L[k] = wave_sum(acc[k]);
        s.sx[k] = wave_sum(acc[3 + k]);
        s.sv[k] = wave_sum(acc[6 + k]);
        s.sv2[k] = wave_sum(acc[9 + k]);
    }
    s.ke = wave_sum(acc[12]);
    s.phi_i = wave_sum(acc[13]);
    s.phi_c = wave_sum(acc[14]);
    s.n = nb_tile;
    s.half = wave_min(half);
    if (lane == 0) out[t] = s;
}

// ------------------------------------------------------------- shapes
//
// calc_shape (src/properties.c:216-326) twice per call: window 0 over the
// records [0, np_alt[2]) with h->r from MASS_DEFINITION4, window 1 over
// [0, dens_tot) with the final h->r.  Each iteration is a tile pass (the
// weighted second moments of the bound records inside the current
// ellipsoid) and a per-(call, window) step: normalise, Jacobi, axis ratios,
// convergence.  Windows of one tile run all of their iterations in one
// launch (k_shape_small); the others take two launches an iteration, a
// window that has stopped being skipped.  On 50,000 calls (6.7M records) ten
// tile passes over everything and their per-window steps were 1.67 ms; now
// 0.58 ms in the one launch and 0.23 in the twenty.  The records' offsets from the centre (float
// differences, as the reference takes them) and bound flags are compacted
// once into 16 bytes per record.

constexpr int kShapeIterations = 10;  // SHAPE_ITERATIONS, src/config.template.h:90

struct ShapeState {
    double orth[3][3];
    double eig[3];
    float r;           // h->r of the window, kpc/h
    float min_r;
    float b_to_a, c_to_a, A[3];
    float inertia[6];
    int32_t n;         // records [0, n)
    int32_t done;
    int32_t assigned;  // inertia written by this window
    int32_t nbound;    // bound records in [0, n)
};

struct ShapePart {
    double v[8];       // weight, xx, yy, zz, yx, zx, zy, unused
};

// the windows' first ellipsoids (spheres) and their bound records
__device__ __forceinline__ void shape_init(const PropCall &c, int32_t tile0, float r,
                                           const PropCount *__restrict__ pre,
                                           const uint64_t *__restrict__ bound,
                                           const PropArgs &pa, ShapeState *__restrict__ st) {
    for (int w = 0; w < 2; w++) {
        ShapeState &s = st[w];
        const float wr =
            w == 0 ? (float)(cbrt((3.0 / (4.0 * M_PI)) * (double)c.alt[2] / pa.thresh3) * 1e3) : r;
        s.r = wr;
        s.n = min(w == 0 ? c.alt[2] : c.dens_tot, c.kept);
        float min_r = (float)(pa.force_res * pa.force_res);
        min_r *= 1e6 / (wr * wr);
        s.min_r = min_r;
        s.b_to_a = s.c_to_a = 0.0f;
        for (int k = 0; k < 3; k++) s.A[k] = 0.0f;
        for (int k = 0; k < 6; k++) s.inertia[k] = 0.0f;
        for (int k = 0; k < 3; k++) {
            for (int l = 0; l < 3; l++) s.orth[k][l] = k == l ? 1.0 : 0.0;
            s.eig[k] = (double)(wr * wr) * 1e-6;
        }
        s.done = !(wr > 0) || s.n <= 0;
        s.assigned = 0;
        s.nbound = bound_before(s.n, tile0, pre, bound);
    }
}

// Windows summed in the reference's order, record by record (the sums of a
// window of few records decide which records the next ellipsoid holds, and
// a change in their last bit can change the result): those of at most
// kShapeExactRecords records or fewer than kShapeExactBound bound records.
constexpr int32_t kShapeExactRecords = 256;
constexpr int32_t kShapeExactBound = 64;
__device__ __forceinline__ bool shape_exact(const ShapeState &s) {
    return s.n <= kShapeExactRecords || s.nbound < kShapeExactBound;
}

// one record's terms (src/properties.c:243-268): the weight 1 / r and the
// weighted second moments, or false where the ellipsoid does not hold it
__device__ __forceinline__ bool shape_terms(double r, double min_r, const double (&d)[3],
                                            double (&v)[7]) {
    if (r < min_r) r = min_r;
    if (!(r > 0 && r <= 1)) return false;
    const double tw = 1.0 / r;  // WEIGHTED_SHAPES = 1
    v[0] = tw;
    v[1] = d[0] * d[0] * tw;
    v[2] = d[1] * d[1] * tw;
    v[3] = d[2] * d[2] * tw;
    v[4] = d[0] * d[1] * tw;
    v[5] = d[0] * d[2] * tw;
    v[6] = d[1] * d[2] * tw;
    return true;
}

// The windows too large to be summed record by record: those of one tile,
// and those of several as (tile, window) pairs 2 tile + window for
// k_shape_tiles and as windows for k_shape_large.  The lists' order does not
// reach the results: a pair's sums have a place of their own and are added
// in tile order.  A workgroup takes its places in one atomic a list (one a
// wavefront took 36 us on 50,000 calls, all on three addresses).
constexpr int kListThreads = 1024;
enum { kOneTile, kPairs, kLarge, kShapeLists };
struct ShapeLists {
    int32_t *one;      // windows
    int32_t *pairs;
    int32_t *windows;
    int32_t *counts;   // of each
};

__global__ __launch_bounds__(kListThreads) void k_shape_list(const ScanTile *__restrict__ tiles,
                                                             int32_t ntiles,
                                                             const ShapeState *__restrict__ st,
                                                             ShapeLists out) {
    __shared__ int32_t s_n[kShapeLists], s_base[kShapeLists];
    const int32_t tid = threadIdx.x, t = blockIdx.x * kListThreads + tid;
    if (tid < kShapeLists) s_n[tid] = 0;
    __syncthreads();
    const ScanTile tl = t < ntiles ? tiles[t] : ScanTile{};
    int32_t at[2][kShapeLists];  // place in the workgroup's part of each list, or -1
    for (int w = 0; w < 2; w++) {
        bool use = false, one = false;
        if (t < ntiles) {
            const ShapeState &s = st[2 * tl.call + w];
            use = !s.done && !shape_exact(s) && tl.off < s.n;
            one = use && s.n <= kScanTile;
        }
        at[w][kOneTile] = one ? atomicAdd(&s_n[kOneTile], 1) : -1;
        at[w][kPairs] = use && !one ? atomicAdd(&s_n[kPairs], 1) : -1;
        at[w][kLarge] = use && !one && tl.off == 0 ? atomicAdd(&s_n[kLarge], 1) : -1;
    }
    __syncthreads();
    if (tid < kShapeLists) s_base[tid] = s_n[tid] ? atomicAdd(&out.counts[tid], s_n[tid]) : 0;
    __syncthreads();
    for (int w = 0; w < 2; w++) {
        if (at[w][kOneTile] >= 0) out.one[s_base[kOneTile] + at[w][kOneTile]] = 2 * tl.call + w;
        if (at[w][kPairs] >= 0) out.pairs[s_base[kPairs] + at[w][kPairs]] = 2 * t + w;
        if (at[w][kLarge] >= 0) out.windows[s_base[kLarge] + at[w][kLarge]] = 2 * tl.call + w;
    }
}

// The sums of a window's records [off, end), lanes strided, in the ellipsoid
// of orth (by rows) and eig
__device__ __forceinline__ void shape_sums(const double *orth, const double *eig, double min_r,
                                           const float4 *__restrict__ rec, int32_t off,
                                           int32_t end, double (&acc)[7]) {
    double o[3][3], ie[3];
    for (int k = 0; k < 7; k++) acc[k] = 0.0;
    for (int k = 0; k < 3; k++) {
        ie[k] = 1.0 / eig[k];  // the reference divides per record; within 1 ulp
        for (int l = 0; l < 3; l++) o[k][l] = orth[3 * k + l];
    }
    for (int32_t j = off + lane_id(); j < end; j += kWave) {
        const float4 q = rec[j];
        if (q.w == 0.0f) continue;
        const double d[3] = {(double)q.x, (double)q.y, (double)q.z};
        double r = 0;
        for (int k = 0; k < 3; k++) {
            double dr = 0;
            for (int l = 0; l < 3; l++) dr += o[k][l] * d[l];
            r += dr * dr * ie[k];
        }
        double v[7];
        if (!shape_terms(r, min_r, d, v)) continue;
        for (int k = 0; k < 7; k++) acc[k] += v[k];
    }
    for (int k = 0; k < 7; k++) acc[k] = wave_sum(acc[k]);
}

// src/properties.c:243-268 for the pairs of a large window and a tile
__global__ __launch_bounds__(kWave) void k_shape_tiles(const int32_t *__restrict__ pairs,
                                                       const int32_t *__restrict__ npairs,
                                                       const ScanTile *__restrict__ tiles,
                                                       const int64_t *__restrict__ hfirst,
                                                       const ShapeState *__restrict__ st,
                                                       const float4 *__restrict__ cd,
                                                       ShapePart *__restrict__ part) {
    for (int32_t i = blockIdx.x; i < *npairs; i += gridDim.x) {
        const int32_t e = pairs[i];
        const ScanTile tl = tiles[e >> 1];
        const int64_t first = hfirst[tl.call];
        const ShapeState &s = st[2 * tl.call + (e & 1)];
        if (s.done) continue;
        double acc[7];
        shape_sums(&s.orth[0][0], s.eig, (double)s.min_r, cd + first, tl.off,
                   min(tl.off + kScanTile, s.n), acc);
        if (lane_id() == 0)
            for (int k = 0; k < 7; k++) part[e].v[k] = acc[k];
    }
}

// |a| + sqrt(x), the sum and the root taken in extended precision and
// rounded once (the reference evaluates both in x87 long double)
__device__ __forceinline__ double add_sqrt_ext(double a_abs, double x) {
    const double r = sqrt(x);
    if (!(r > 0.0)) return a_abs + r;
    const double e = fma(-r, r, x) / (2.0 * r);  // sqrt(x) = r + e to O(e^2)
    const double s = a_abs + r;
    const double bb = s - a_abs;
    const double err = (a_abs - (s - bb)) + (r - bb);
    return s + (err + e);
}

// The cyclic Jacobi eigenvalue iteration of src/jacobi.c:8-135 (largest
// off-diagonal element first, each row's largest column cached, stop when no
// eigenvalue changes by more than 1e-6 of itself) for three rows.  orth's
// rows are the eigenvectors.  The pivot (k, l) is (0, 1), (0, 2) or (1, 2),
// with n the third row: the lanes of a wavefront take different ones, so one
// rotation serves all, on operands taken and put back by selects (a branch
// per pivot ran the some 250 instructions of a rotation up to three times).
struct Jacobi3 {
    double m01, m02, m12, eig[3], orth[3][3];

    // from the matrix's diagonal in eig
    __device__ __forceinline__ void run() {
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++) orth[i][j] = i == j ? 1.0 : 0.0;
        bool col2 = fabs(m02) > fabs(m01);  // row 0's largest column: 2, else 1 (also on ties)
        // rows whose eigenvalue still changes
        bool ch[3] = {m01 != 0.0 || m02 != 0.0, m01 != 0.0 || m12 != 0.0, m02 != 0.0 || m12 != 0.0};
        for (int guard = 0; (ch[0] || ch[1] || ch[2]) && guard < 1000; guard++) {
            const bool row1 = fabs(m12) > fabs(col2 ? m02 : m01);
            const bool p02 = !row1 && col2, p01 = !row1 && !col2;
            const double v = row1 ? m12 : (p02 ? m02 : m01);
            if (v == 0.0) break;
            // k = 1 in row 1, else 0; l = 1 for (0, 1), else 2
            double ek = row1 ? eig[1] : eig[0], el = p01 ? eig[1] : eig[2];
            const double a = (el - ek) * 0.5;
            double t = add_sqrt_ext(fabs(a), v * v + a * a);
            double s = add_sqrt_ext(0.0, v * v + t * t);
            const double c = t / s;
            s = v / s;
            t = v * v / t;
            if (a < 0) {
                s = -s;
                t = -t;
            }
            ek += -t;
            el += t;
            const bool ck = changes(row1 ? ch[1] : ch[0], t, ek);
            const bool cl = changes(p01 ? ch[1] : ch[2], t, el);
            if (row1) eig[1] = ek, ch[1] = ck;
            else eig[0] = ek, ch[0] = ck;
            if (p01) eig[1] = el, ch[1] = cl;
            else eig[2] = el, ch[2] = cl;
            // src/jacobi.c:113-124: elements (k, n) and (l, n)
            const double p = p02 || row1 ? m01 : m02, q = row1 ? m02 : m12;
            const double p2 = p * c - s * q, q2 = s * p + c * q;
            m01 = p01 ? 0.0 : p2;
            m02 = p02 ? 0.0 : (row1 ? q2 : p2);
            m12 = row1 ? 0.0 : q2;
            col2 = col2 ? !(fabs(m01) > fabs(m02)) : fabs(m02) > fabs(m01);
            for (int x = 0; x < 3; x++) {
                const double ok = row1 ? orth[1][x] : orth[0][x];
                const double ol = p01 ? orth[1][x] : orth[2][x];
                const double ok2 = ok * c - s * ol, ol2 = s * ok + c * ol;
                orth[0][x] = row1 ? orth[0][x] : ok2;
                orth[1][x] = row1 ? ok2 : (p01 ? ol2 : orth[1][x]);
                orth[2][x] = p01 ? orth[2][x] : ol2;
            }
        }
    }
    // whether an eigenvalue changed by y still counts as changing
    static __device__ __forceinline__ bool changes(bool ch, double y, double e) {
        return ch ? !(fabs(y) < 1e-6 * fabs(e)) : fabs(y) > 1e-6 * fabs(e);
    }
};

// A window's running values; its other results go to its ShapeState as they
// are found.
struct ShapeRun {
    float r, b_to_a, c_to_a;
    int32_t it, limit;
};

// src/properties.c:270-325: the window's next ellipsoid (orth by rows, eig)
// from its sums (the weight and the six moments).  Returns false where the
// window stops.
__device__ __forceinline__ bool shape_step(ShapeRun &s, const double (&sum)[7],
                                           ShapeState *__restrict__ out, double *orth,
                                           double *eig) {
    const double wt = sum[0];
    const double *t6 = sum + 1;
    if (s.it >= s.limit || !(wt != 0.0)) return false;
    Jacobi3 jb;
    for (int k = 0; k < 3; k++) jb.eig[k] = t6[k] / wt;
    jb.m01 = t6[3] / wt;
    jb.m02 = t6[4] / wt;
    jb.m12 = t6[5] / wt;
    const float inert[6] = {(float)jb.eig[0], (float)jb.eig[1], (float)jb.eig[2],
                            (float)jb.m01,    (float)jb.m12,    (float)jb.m02};
    jb.run();
    const double e0 = jb.eig[0], e1 = jb.eig[1], e2 = jb.eig[2];
    auto E = [&](int q) { return q == 0 ? e0 : (q == 1 ? e1 : e2); };
    int a = 0, b = 1, c = 2;
    if (e1 > e0) {
        b = 0;
        a = 1;
    }
    if (e2 > E(b)) {
        c = b;
        b = 2;
    }
    if (E(b) > E(a)) {
        const int q = a;
        a = b;
        b = q;
    }
    const double ea = E(a), eb = E(b), ec = E(c);
    if (!(ea != 0.0) || !(eb != 0.0) || !(ec != 0.0)) return false;
    const float b_to_a = (float)sqrt(eb / ea);
    const float c_to_a = (float)sqrt(ec / ea);
    if ((fabs((double)(b_to_a - s.b_to_a)) < 0.01 * (double)s.b_to_a) &&
        (fabs((double)(c_to_a - s.c_to_a)) < 0.01 * (double)s.c_to_a))
        return false;
    s.b_to_a = b_to_a > 0 ? b_to_a : 0.0f;
    s.c_to_a = c_to_a > 0 ? c_to_a : 0.0f;
    const double r = sqrt(ea);
    const double sc = ((double)(s.r * s.r) * 1e-6) / (r * r);
    for (int k = 0; k < 3; k++) {
        const double oa = a == 0 ? jb.orth[0][k] : (a == 1 ? jb.orth[1][k] : jb.orth[2][k]);
        out->A[k] = (float)(1e3 * r * oa);
        eig[k] = jb.eig[k] * sc;
        for (int l = 0; l < 3; l++) orth[3 * k + l] = jb.orth[k][l];
    }
    for (int k = 0; k < 6; k++) out->inertia[k] = inert[k];
    out->b_to_a = s.b_to_a;
    out->c_to_a = s.c_to_a;
    out->assigned = 1;
    return ++s.it < s.limit;
}

// The windows summed in the reference's order (shape_exact), all iterations
// in one launch.  A workgroup holds 64 windows at a time of a range of its
// own; a window that stops makes room for the range's next one, so that the
// steps stay full though windows take 1 to 10 iterations.  Every iteration
//   * a thread takes a record; a round takes as many records of each window
//     that has some left as 256 threads allow (4 of 64 windows, all 256 of
//     the last one), so that in the sums all windows run at once (0.58 ms
//     against 0.61 with the windows laid end to end, some five to a round);
//   * each window's seven sums are added up in record order by four lanes,
//     from the terms in LDS (0 for a record outside the ellipsoid: the
//     running sums start at 0, so they never are -0 and keep their bits);
//   * one lane per window takes the step.
// What bounds it is the chain through the three, above all the last: some
// 2,000 dependent double instructions of the Jacobi rotations, on one of the
// four wavefronts (a vector instruction in half of the cycles, the rest in
// the tail: 10 iterations are a chain of 0.2 ms for a workgroup on its own).
// So as many workgroups as fit are kept on a compute unit: what a window
// carries from step to step is held down to a few registers, and six
// workgroups with some registers spilled are 0.58 ms against 0.65 with four.
constexpr int kShapeWindows = 64;
constexpr int kShapeThreads = 4 * kShapeWindows;
constexpr int kShapeResident = 6;                     // workgroups on a compute unit

// The first kOneTileGroups workgroups take the one-tile windows instead, 16
// each at a time: a wavefront sums a window, and the windows' steps are taken
// together as above (each on a wavefront of its own cost as much as the
// sums).  Both kinds are chains of dependent double operations and fill each
// other's waits.
constexpr int kOneTileGroups = 256;
constexpr int kOneTileSlots = 16;

__device__ __forceinline__ void shape_one_tile(const int32_t *__restrict__ list, int32_t n,
                                               const int64_t *__restrict__ hfirst,
                                               const float4 *__restrict__ cd,
                                               ShapeState *__restrict__ st, double (*s_ell)[13],
                                               double (*s_sum)[7], int64_t *s_first,
                                               int32_t *s_n) {
    const int32_t tid = threadIdx.x, wave = uniform(tid / kWave);
    for (int32_t i0 = blockIdx.x; i0 < n; i0 += kOneTileGroups * kOneTileSlots) {
        // slot k: window i0 + k kOneTileGroups of the list
        const int32_t i = i0 + tid * kOneTileGroups;
        ShapeRun run = {};
        int32_t sw = -1;
        if (tid < kOneTileSlots) {
            if (i < n) {
                sw = list[i];
                const ShapeState &s = st[sw];
                run = ShapeRun{s.r, s.b_to_a, s.c_to_a, 0, kShapeIterations};
                s_first[tid] = hfirst[sw >> 1];
                for (int k = 0; k < 9; k++) s_ell[tid][k] = s.orth[k / 3][k % 3];
                for (int k = 0; k < 3; k++) s_ell[tid][9 + k] = s.eig[k];
                s_ell[tid][12] = (double)s.min_r;
            }
            s_n[tid] = sw < 0 ? 0 : st[sw].n;
        }
        while (__syncthreads_or(tid < kOneTileSlots && sw >= 0)) {
            for (int k = wave; k < kOneTileSlots; k += kShapeThreads / kWave) {
                const int32_t nk = uniform(s_n[k]);
                if (nk == 0) continue;
                double sum[7];
                shape_sums(s_ell[k], s_ell[k] + 9, s_ell[k][12], cd + s_first[k], 0, nk, sum);
                if (lane_id() == 0)
                    for (int q = 0; q < 7; q++) s_sum[k][q] = sum[q];
            }
            __syncthreads();
            if (tid < kOneTileSlots && sw >= 0) {
                double sum[7];
                for (int q = 0; q < 7; q++) sum[q] = s_sum[tid][q];
                if (!shape_step(run, sum, st + sw, s_ell[tid], s_ell[tid] + 9)) {
                    sw = -1;
                    s_n[tid] = 0;
                }
            }
        }
    }
}

__global__ __launch_bounds__(kShapeThreads, kShapeResident) void k_shape_small(
    int32_t nh, const int64_t *__restrict__ hfirst, const float4 *__restrict__ cd,
    const int32_t *__restrict__ one, const int32_t *__restrict__ none,
    ShapeState *__restrict__ st) {
    static_assert(kShapeWindows == kWave, "a lane of the leading wavefront per window");
    __shared__ double s_term[kShapeThreads][7];
    __shared__ double s_ell[kShapeWindows][13];  // orth, eig, min_r
    __shared__ double s_sum[kShapeWindows][7];
    __shared__ int64_t s_first[kShapeWindows];
    __shared__ int32_t s_n[kShapeWindows];       // records; 0: no window
    const int32_t tid = threadIdx.x, lane = lane_id();
    if (blockIdx.x < kOneTileGroups) {
        shape_one_tile(one, *none, hfirst, cd, st, s_ell, s_sum, s_first, s_n);
        return;
    }
    const int64_t groups = gridDim.x - kOneTileGroups;
    const int64_t per = (2 * (int64_t)nh + groups - 1) / groups;
    int64_t next = (blockIdx.x - kOneTileGroups) * per;  // the range's next window
    const int64_t last = min(next + per, 2 * (int64_t)nh);
    const bool leads = tid < kWave;  // the wavefront that takes the steps
    ShapeRun run = {};    // of the window of this lane of that wavefront
    int64_t cur = -1;     // that window
    const int task = tid >> 2, comp = 2 * (tid & 3), comp2 = min(comp + 1, 6);
    if (leads) s_n[lane] = 0;
    while (true) {
        if (leads) {
            while (next < last) {
                const bool want = cur < 0;
                const uint64_t m = ballot(want);
                if (!m) break;
                const int64_t i = next + __popcll(m & ((1ull << lane) - 1));
                next += __popcll(m);
                if (want && i < last) {
                    const ShapeState &s = st[i];
                    // src/properties.c:228-236: none with fewer than 3
                    if (!s.done && shape_exact(s) && s.nbound >= 3) {
                        cur = i;
                        run = ShapeRun{s.r, s.b_to_a, s.c_to_a, 0, min(kShapeIterations, s.nbound)};
                        s_n[lane] = s.n;
                        s_first[lane] = hfirst[i >> 1];
                        for (int k = 0; k < 9; k++) s_ell[lane][k] = s.orth[k / 3][k % 3];
                        for (int k = 0; k < 3; k++) s_ell[lane][9 + k] = s.eig[k];
                        s_ell[lane][12] = (double)s.min_r;
                    }
                }
            }
        }
        __syncthreads();
        // Rounds over the windows that still have records, every one taking
        // the same number `per` of them from `pos` on: lane l of every
        // wavefront holds window l's count, and a round's k-th running
        // window has the threads and terms [k per, k per + per).
        const int32_t nl = s_n[lane], n_task = s_n[task];
        if (ballot(nl > 0) == 0) break;  // the same in every wavefront
        int32_t pos = 0, per = 0, w = 0;
        uint64_t act = 0;
        float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        // the round's record of this thread (flag 0: none), read a round ahead
        auto read = [&]() {
            act = ballot(nl > pos);
            q.w = 0.0f;
            if (act == 0) return;
            per = kShapeThreads / __popcll(act);
            // tid / per, exact for both below 256
            const int32_t k = (int32_t)((uint32_t)tid * (65536u / (uint32_t)per + 1u) >> 16);
            const int32_t i = pos + tid - k * per;
            const int32_t rank = __popcll(act & ((1ull << lane) - 1));
            const bool run_l = nl > pos;
            // window of rank k: lane k takes the lane number of the k-th one
            const int32_t kth =
                __builtin_amdgcn_ds_permute(4 * (run_l ? rank : kWave - 1), run_l ? lane : 0);
            w = __shfl(kth, k, 64);
            const int32_t n_w = __shfl(nl, w, 64);
            if (k < __popcll(act) && i < n_w) q = cd[s_first[w] + i];
        };
        read();
        double acc = 0.0, acc2 = 0.0;
        while (act != 0) {
            double v[7] = {0, 0, 0, 0, 0, 0, 0};
            if (q.w != 0.0f) {
                const double *e = s_ell[w];
                const double d[3] = {(double)q.x, (double)q.y, (double)q.z};
                double r = 0;
                for (int k = 0; k < 3; k++) {
                    double dr = 0;
                    for (int l = 0; l < 3; l++) dr += e[3 * k + l] * d[l];
                    r += dr * dr / e[9 + k];
                }
                if (!shape_terms(r, e[12], d, v))
                    for (int k = 0; k < 7; k++) v[k] = 0.0;
            }
            for (int k = 0; k < 7; k++) s_term[tid][k] = v[k];
            const int32_t a = __popcll(act & ((1ull << task) - 1)) * per;
            const int32_t b = a + min(per, n_task - pos);  // below a: not running
            pos += per;
            read();
            __syncthreads();
            int32_t i = a;
            for (; i + 4 <= b; i += 4) {
                double x[4], x2[4];
                for (int k = 0; k < 4; k++) {
                    x[k] = s_term[i + k][comp];
                    x2[k] = s_term[i + k][comp2];
                }
                for (int k = 0; k < 4; k++) {
                    acc += x[k];
                    acc2 += x2[k];
                }
            }
            for (; i < b; i++) {
                acc += s_term[i][comp];
                acc2 += s_term[i][comp2];
            }
            __syncthreads();
        }
        s_sum[task][comp] = acc;
        if (comp < 6) s_sum[task][comp2] = acc2;
        __syncthreads();
        if (cur >= 0) {
            double sum[7];
            for (int k = 0; k < 7; k++) sum[k] = s_sum[lane][k];
            if (!shape_step(run, sum, st + cur, s_ell[lane], s_ell[lane] + 9)) {
                cur = -1;
                s_n[lane] = 0;
            }
        }
    }
}

// The step of the large windows still running, a wavefront each: eight tiles'
// sums are read at a time (lane 8 i + k: sum k of tile i) and added in tile
// order, lane k holding sum k.
__global__ __launch_bounds__(kWave) void k_shape_large(
    const int32_t *__restrict__ windows, const int32_t *__restrict__ nwindows, int32_t it,
    const int32_t *__restrict__ call_tile0, const int32_t *__restrict__ call_ntiles,
    const ShapePart *__restrict__ part, ShapeState *__restrict__ st) {
    const int lane = lane_id();
    for (int32_t i = blockIdx.x; i < *nwindows; i += gridDim.x) {
        const int32_t sw = uniform(windows[i]);
        if (st[sw].done) continue;
        const int32_t h = sw >> 1, w = sw & 1;
        // the tiles that hold records of the window
        const int32_t t0 = call_tile0[h];
        const int32_t nt = min(call_ntiles[h], (st[sw].n + kScanTile - 1) / kScanTile);
        double acc = 0.0;
        for (int32_t b = 0; b < nt; b += 8) {
            const int32_t t = b + (lane >> 3);
            const double v = t < nt ? part[2 * (t0 + t) + w].v[lane & 7] : 0.0;
            for (int k = 0; k < 8; k++) acc += __shfl(v, 8 * k + (lane & 7), 64);
        }
        double sum[7];
        for (int k = 0; k < 7; k++) sum[k] = __shfl(acc, k, 64);
        ShapeState &s = st[sw];
        // at least 64 bound records, so all of the iterations
        ShapeRun run = {s.r, s.b_to_a, s.c_to_a, it, kShapeIterations};
        const bool go = shape_step(run, sum, &s, &s.orth[0][0], s.eig);
        if (lane == 0 && !go) s.done = 1;
    }
}

// ------------------------------------------- scale radius, pseudo-evolution

constexpr int kScaleBins = 50;    // MAX_SCALE_BINS, src/nfw.c:9
constexpr int kMinPerBin = 15;    // MIN_PART_PER_BIN
constexpr int kMinScale = 100;    // MIN_SCALE_PART
constexpr double kRmaxToRs = 2.1626;       // src/universal_constants.h:7
constexpr double kRsConstant = 0.216216595;  // src/universal_constants.h:8

struct ScaleCall {
    int32_t ppbin;     // bound records per bin; 0: no fit (fewer than 100)
    int32_t nbins;
    int32_t end;       // bins come from records [0, end) = [0, dens_tot - 1)
    int32_t pad;
    float bin_r[kScaleBins + 1];
    float klypin, rs, chi2;  // results for the fitted calls
};

// per call: the halo fields, and where its shape windows and its fit start
__global__ __launch_bounds__(kWave) void k_props_final(const PropReads in, const PropCount *__restrict__ pre,
                              const int32_t *__restrict__ call_tile0,
                              const int32_t *__restrict__ call_ntiles, int32_t nh,
                              const hp_halo *__restrict__ halos,
                              const int64_t *__restrict__ hfirst,
                              const PropCall *__restrict__ pc, const PropSums *__restrict__ ts,
                              PropArgs pa, hp_halo_props *__restrict__ props,
                              ShapeState *__restrict__ shapes, ScaleCall *__restrict__ scales,
                              int32_t *__restrict__ fit_list, int32_t *__restrict__ fit_n) {
    const int32_t h = lane_call(nh, call_ntiles);
    const bool v = h < nh;
    const int32_t t0 = v ? call_tile0[h] : 0, nt = v ? call_ntiles[h] : 0;
    double L[3] = {0, 0, 0}, sx[3] = {0, 0, 0}, sv[3] = {0, 0, 0}, sv2[3] = {0, 0, 0};
    double ke = 0, phi = 0;
    int32_t n = 0, half = INT32_MAX;
    auto add = [&](const PropSums &s) {
        for (int k = 0; k < 3; k++) {
            L[k] += s.L[k];
            sx[k] += s.sx[k];
            sv[k] += s.sv[k];
            sv2[k] += s.sv2[k];
        }
        ke += s.ke;
        phi += s.phi_i + s.phi_c;
        n += s.n;
        half = min(half, s.half);
    };
    if (nt <= kFewTiles)
        for (int32_t t = t0; t < t0 + nt; t++) add(ts[t]);
    for_large_call(t0, nt, [&](int32_t a, int32_t k, bool mine) {
        // lane c < 15 adds up component c, in tile order
        static_assert(offsetof(PropSums, n) == 15 * sizeof(double), "fifteen sums, then counts");
        const int c = min(lane_id(), 14);
        double x = 0.0;
        int32_t m = 0, hf = INT32_MAX;
        for (int32_t t = a; t < a + k; t++) x += reinterpret_cast<const double *>(ts + t)[c];
        for (int32_t t = a + lane_id(); t < a + k; t += kWave) {
            m += ts[t].n;
            hf = min(hf, ts[t].half);
        }
        m = wave_sum(m);
        hf = wave_min(hf);
        if (mine) {
            n = m;
            half = hf;
        }
        for (int q = 0; q < 3; q++) {
            const double l = read_lane(x, q), y = read_lane(x, 3 + q), z = read_lane(x, 6 + q),
                         z2 = read_lane(x, 9 + q);
            if (mine) {
                L[q] = l;
                sx[q] = y;
                sv[q] = z;
                sv2[q] = z2;
            }
        }
        const double e = read_lane(x, 12), p = read_lane(x, 13) + read_lane(x, 14);
        if (mine) {
            ke = e;
            phi = p;
        }
    });
    // src/nfw.c:134-152: a fit takes 100 bound records of [0, dens_tot - 1)
    const PropCall c = v ? pc[h] : PropCall{};
    int64_t nfit = 0;
    if (v) {
        const int32_t end = c.dens_tot - 1;
        nfit = n;
        if (end >= 0)
            nfit -= (in.bound[(int64_t)kTileWords * (t0 + end / kScanTile) + end % kScanTile / kWave] >>
                     (end % kWave)) & 1;
    }
    const bool fits = nfit >= kMinScale;
    const uint64_t mf = ballot(fits);  // the fits run together
    if (mf) {
        int32_t at = 0;
        if (lane_id() == 0) at = atomicAdd(fit_n, __popcll(mf));
        at = uniform(at) + __popcll(mf & ((1ull << lane_id()) - 1));
        if (fits) fit_list[at] = h;
    }
    if (!v) return;
    const hp_halo &hh = halos[h];
    const int64_t first = hfirst[h];
    const double PM = pa.particle_mass;
    const float scale_now = pa.scale_now;
    hp_halo_props o;
    const double m = (double)c.n0 * PM;
    o.m = (float)((double)c.n_all * PM);
    o.mgrav = (float)m;
    // src/properties.c:460-475: float fields accumulated from double terms
    float xoff = 0.0f, voff = 0.0f;
    double vr = 0.0;
    for (int k = 0; k < 3; k++) {
        // the reference's running means start at 0 and stay there with no
        // record averaged
        const double dsx = n > 0 ? sx[k] / (double)n : -(double)hh.pos[k];
        const double dsv = n > 0 ? sv[k] / (double)n : -(double)hh.pos[k + 3];
        xoff = (float)((double)xoff + dsx * dsx);
        voff = (float)((double)voff + dsv * dsv);
        vr += n > 0 ? (sv2[k] - sv[k] * sv[k] / (double)n) / (double)n : 0.0;
    }
    for (int k = 0; k < 4; k++) o.alt_m[k] = (float)((double)c.alt[k] * PM);
    o.Xoff = (float)(sqrt((double)xoff) * 1e3);
    o.Voff = (float)sqrt((double)voff);
    o.vrms = (float)sqrt(vr);
    o.vmax = (float)(kVmaxConst * sqrt(c.vmax * (PM / (double)scale_now)));
    o.rvmax = c.j_vmax >= 0
                  ? (float)(prop_radius(in.r2[first + c.j_vmax], pa.force_res) * 1e3)
                  : 0.0f;
    const int32_t ih = half == INT32_MAX ? 0 : half;
    o.halfmass_radius = c.kept > 0 ? (float)(sqrt((double)in.r2[first + ih]) * 1e3) : 0.0f;
    o.r = (float)(cbrt((3.0 / (4.0 * M_PI)) * (double)c.n0 / pa.thresh0) * 1e3);
    const double rvir = cbrt((3.0 / (4.0 * M_PI)) * (double)c.vir / pa.rvir_dens) * 1e3;
    const double mvir = (double)c.vir * PM;
    o.rvir = (float)rvir;
    for (int k = 0; k < 3; k++) o.J[k] = (float)(PM * (double)scale_now * L[k]);
    // src/properties.c:328-349
    const double total_phi = phi / 2.0;
    o.kin_to_pot = total_phi != 0.0 ? (float)(ke / total_phi) : 0.0f;
    o.energy = (float)((ke - total_phi) * PM * kGc / (double)scale_now);
    const double Jh = PM * (double)scale_now * sqrt(L[0] * L[0] + L[1] * L[1] + L[2] * L[2]);
    o.spin = (float)(m > 0 ? Jh * sqrt(fabs((double)o.energy)) / (kGc * pow(m, 2.5))
                           : 0.0);
    o.bullock_spin = (float)(m > 0 ? Jh / (mvir * sqrt(2.0 * kGc * mvir * rvir *
                                                        (double)scale_now / 1e3))
                                   : 0.0);
    // filled by the shape, scale-radius and pseudo-evolution kernels
    o.rs = o.klypin_rs = o.chi2 = 0.0f;
    o.b_to_a = o.c_to_a = o.b_to_a2 = o.c_to_a2 = 0.0f;
    for (int k = 0; k < 3; k++) o.A[k] = o.A2[k] = 0.0f;
    for (int k = 0; k < 6; k++) o.inertia_tensor[k] = o.inertia_tensor2[k] = 0.0f;
    o.m_pe_b = o.m_pe_d = 0.0f;
    o.n_mdelta = c.n0;
    o.dens_tot = c.dens_tot;
    o.n_vir = c.vir;
    o.n_half = ih;
    props[h] = o;
    shape_init(c, t0, o.r, pre, in.bound, pa, shapes + 2 * h);
    ScaleCall &sc = scales[h];
    sc.end = c.dens_tot - 1;
    int64_t pp = 0;
    if (fits) {
        pp = (int64_t)ceil((double)nfit / (double)kScaleBins);
        if (pp < kMinPerBin) pp = nfit / (nfit / kMinPerBin);
    }
    sc.ppbin = (int32_t)pp;
    sc.nbins = fits ? (int32_t)(nfit / pp) : 0;
    sc.bin_r[0] = 0.0f;
}

// src/nfw.c:153-162: the outer edge of bin k is between the k * ppbin-th
// bound record and the record after it
__global__ __launch_bounds__(kWave) void k_scale_bins(const PropReads in,
                                                      const ScanTile *__restrict__ tiles,
                                                      int32_t ntiles,
                                                      const int64_t *__restrict__ hfirst,
                                                      const PropCount *__restrict__ pre,
                                                      ScaleCall *__restrict__ sc) {
    const int32_t t = blockIdx.x;
    if (t >= ntiles) return;
    const ScanTile tl = tiles[t];
    const int32_t pp = sc[tl.call].ppbin, end = min(tl.off + kScanTile, sc[tl.call].end);
    if (pp == 0 || tl.off >= end) return;
    const int64_t first = hfirst[tl.call];
    int32_t carry = pre[t].nb;
    for (int32_t base = tl.off; base < end; base += kWave) {
        const int32_t j = base + lane_id();
        uint64_t mb = in.bound[(int64_t)kTileWords * t + (base - tl.off) / kWave];
        if (end - base < kWave) mb &= (1ull << (end - base)) - 1;
        const int32_t n = count_to_lane(mb) + carry;
        carry += __popcll(mb);
        if (((mb >> lane_id()) & 1) && n % pp == 0 && n / pp <= kScaleBins) {
            const float r = (float)(1e3 * 0.5 * (sqrt((double)in.r2[first + j]) +
                                                 sqrt((double)in.r2[first + j + 1])));
            sc[tl.call].bin_r[n / pp] = r;
        }
    }
}

__device__ double c_to_f(double c) {
    const double cp1 = 1.0 + c;
    return c * cp1 / (log1p(c) * cp1 - c);
}

// concentration with c_to_f(c) = f, src/nfw.c:18-33
__device__ double f_to_c(double f) {
    double c = f, tc = c_to_f(c);
    for (int guard = 0; fabs((f - tc) / f) > 1e-7 && guard < 10000; guard++) {
        const double tc2 = c_to_f(c + 0.1);
        const double slope = (tc2 - tc) / 0.1;
        const double nc = c + (f - tc) / slope;
        if (nc < 0) c /= 2;
        else c = nc;
        tc = c_to_f(c);
    }
    return c;
}

// Klypin's rs from vmax, rvmax and the virial mass and radius, src/nfw.c:35-50
__device__ float klypin_rs(float mvir, float rvir, float vmax, float rvmax, float scale) {
    if (!(mvir != 0.0f) || !(rvir != 0.0f) || !(vmax != 0.0f))
        return (float)(rvmax / kRmaxToRs);
    float vm2 = (float)(vmax / kVmaxConst);
    vm2 = vm2 * vm2 * scale;
    const float f = (float)((rvir / 1.0e3) * vm2 / (mvir * kRsConstant));
    if (f < 4.625) return (float)(rvmax / kRmaxToRs);
    const float c = (float)f_to_c(f);
    if (c <= 0) return (float)(rvmax / kRmaxToRs);
    return rvir / c;
}

__device__ __forceinline__ float nfw_menc(float r, float rs) {
    return (float)(log((double)((rs + r) / rs)) - (double)(r / (rs + r)));
}

// The bins of one fit on a row of 16 lanes: lane l holds bins l, l + 16, l + 32
// and l + 48 (50 at most).  A row takes every branch of a fit together.
constexpr int kBinLanes = 16;
constexpr int kBinSlots = (kScaleBins + kBinLanes - 1) / kBinLanes;
struct FitBins {
    float r_out[kBinSlots];   // outer edge
    float weight[kBinSlots];  // src/nfw.c:164-166: 0.1 for bins starting inside 3 FORCE_RES
    float first, last, mid;   // bin_r[0], bin_r[nb], bin_r[(nb + 1) / 2]
    int32_t nb;
};

__device__ __forceinline__ FitBins load_bins(const float *bin_r, int32_t nb, double force_res) {
    FitBins b;
    for (int k = 0; k < kBinSlots; k++) {
        const int i = kBinLanes * k + (lane_id() & (kBinLanes - 1));
        const float in = i < nb ? bin_r[i] : 0.0f;
        b.r_out[k] = i < nb ? bin_r[i + 1] : 0.0f;
        b.weight[k] = in * 1e-3 < 3 * force_res ? 0.1f : 1.0f;
    }
    b.first = bin_r[0];
    b.last = bin_r[nb];
    b.mid = bin_r[(nb + 1) / 2];
    b.nb = nb;
    return b;
}

// s plus the 16 values of the row's lanes, lane 0's first
template <int L>
__device__ __forceinline__ float row_add_in_order(float s, float v) {
    if constexpr (L == kBinLanes) return s;
    else return row_add_in_order<L + 1>(s + dpp_move<0x150 + L>(v), v);  // row_newbcast
}

// the bins' masses one bin a lane, their squares added in bin order (each sum
// takes its term from the row's lane in the same instruction)
__device__ __forceinline__ float chi2_rs(float rs, const FitBins &b) {
    const int l = lane_id() & (kBinLanes - 1);
    float menc[kBinSlots], total = 0.0f;
    for (int k = 0; k < kBinSlots; k++) {
        menc[k] = nfw_menc(b.r_out[k], rs);
        total = (b.nb - 1) / kBinLanes == k ? menc[k] : total;
    }
    const float bin_mass =
        (float)(__shfl(total, (b.nb - 1) & (kBinLanes - 1), kBinLanes) / (double)b.nb);
    float chi2 = 0.0f, wrap = 0.0f;  // wrap: the slot before's last bin
    for (int k = 0; k < kBinSlots; k++) {
        const float prev = dpp_move<0x121>(menc[k]);  // row_ror:1; lane 0 takes lane 15's
        const float last = l == 0 ? wrap : prev;
        wrap = prev;
        const float dx = b.weight[k] * ((menc[k] - last) - bin_mass) / bin_mass;
        const float sq = kBinLanes * k + l < b.nb ? dx * dx : 0.0f;
        chi2 = row_add_in_order<0>(chi2, sq);
    }
    return chi2;
}

// parabolic steps on chi2(rs), src/nfw.c:75-128
__device__ __forceinline__ float fit_rs(float rs, const FitBins &b, float *out_chi2) {
    if (!(rs > b.first) || !(rs < b.last)) rs = b.mid;
    const float initial = rs;
    float chi2 = chi2_rs(rs, b);
    float drs = (float)(rs / 10.0);
    int iter = 0;
    float last = 1e30f;
    if (!(rs > 0)) return initial;
    for (int guard = 0; fabs((double)(chi2 - last)) > 0.005 * chi2 && iter < kMinPerBin &&
                        guard < 10000; guard++) {
        last = chi2;
        if (rs + drs > b.last) drs = (float)(0.1 * (b.last - rs));
        if (rs - drs < b.first) drs = (float)(0.1 * (rs - b.first));
        const float cr = chi2_rs(rs + drs, b);
        const float cl = chi2_rs(rs - drs, b);
        const float dx = (float)(0.5 * (cr - cl) / drs);
        const float dx2 = (float)((cr + cl - 2.0 * chi2) / (drs * drs));
        float move = 0;
        if (dx2 != 0) move = -dx / dx2;
        if (!(move != 0.0f)) return rs;
        if (rs + move > 4 * rs) move = (float)(3.0 * rs);
        if (rs + move < 0.25 * rs) move = (float)(-0.75 * rs);
        float nrs = rs + move;
        if (nrs > b.last) nrs = (float)(rs + 0.8 * (b.last - rs));
        else if (nrs < b.first) nrs = (float)(rs + 0.8 * (b.first - rs));
        float nchi2 = chi2_rs(nrs, b);
        if (cr < nchi2) {
            nchi2 = cr;
            nrs = rs + drs;
        }
        if (cl < nchi2) {
            nchi2 = cl;
            nrs = rs - drs;
        }
        if (last < nchi2) {
            drs *= 0.5f;
            continue;
        }
        drs = (float)(fabs((double)(rs - nrs)) / 10.0);
        rs = nrs;
        chi2 = nchi2;
        iter++;
    }
    *out_chi2 = chi2;
    return rs;
}

// The calls with a fit, a row of 16 lanes each: Klypin's estimate, then the
// fit.  It is bound by the chain of chi2's (some four an iteration, each 50
// logarithms and a sum in bin order): with a lane a call, the fits of 50,000
// calls filled 80 wavefronts and took 0.205 ms; now 0.046.
__global__ __launch_bounds__(kWave) void k_scale_fit(const int32_t *__restrict__ fit_list,
                                                     const int32_t *__restrict__ fit_n,
                                                     const PropCall *__restrict__ pc,
                                                     const hp_halo_props *__restrict__ props,
                                                     PropArgs pa, ScaleCall *__restrict__ sc) {
    constexpr int kFits = kWave / kBinLanes;  // of a wavefront
    for (int32_t i = blockIdx.x * kFits + lane_id() / kBinLanes; i < *fit_n;
         i += gridDim.x * kFits) {
        const int32_t h = fit_list[i];
        const hp_halo_props &o = props[h];
        const double m = (double)pc[h].n0 * pa.particle_mass;
        ScaleCall &sk = sc[h];
        const FitBins bins = load_bins(sk.bin_r, sk.nbins, pa.force_res);
        const float rs0 = klypin_rs((float)m, o.r, o.vmax, o.rvmax, pa.scale_now);
        float chi2 = 0.0f;
        const float rs = fit_rs(rs0, bins, &chi2);
        if ((lane_id() & (kBinLanes - 1)) == 0) {
            sk.klypin = rs0;
            sk.rs = rs;
            sk.chi2 = chi2;
        }
    }
}

// per call: the shape fields, the scale radius (src/nfw.c:130-173), m_pe_b
// and the radius that bounds m_pe_d (src/properties.c:351-382)
__global__ void k_props_late(int32_t nh, const PropCall *__restrict__ pc,
                             const ShapeState *__restrict__ st, const ScaleCall *__restrict__ sc,
                             PropArgs pa, double *__restrict__ r_pe,
                             hp_halo_props *__restrict__ props) {
    const int32_t h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= nh) return;
    hp_halo_props o = props[h];
    const PropCall c = pc[h];
    const ShapeState &s0 = st[2 * h], &s1 = st[2 * h + 1];
    o.b_to_a2 = s0.b_to_a;
    o.c_to_a2 = s0.c_to_a;
    o.b_to_a = s1.b_to_a;
    o.c_to_a = s1.c_to_a;
    for (int k = 0; k < 3; k++) {
        o.A2[k] = s0.A[k];
        o.A[k] = s1.A[k];
    }
    // the second calc_shape keeps the first's tensor until it writes its own
    for (int k = 0; k < 6; k++) {
        o.inertia_tensor2[k] = s0.inertia[k];
        o.inertia_tensor[k] = s1.assigned ? s1.inertia[k] : s0.inertia[k];
    }
    const ScaleCall &sk = sc[h];
    float rs;
    if (sk.ppbin > 0) {  // fitted by k_scale_fit
        o.klypin_rs = sk.klypin;
        rs = sk.rs;
        o.chi2 = sk.chi2;
    } else {  // fewer than 100 bound records: Klypin's estimate
        const double m = (double)c.n0 * pa.particle_mass;
        rs = klypin_rs((float)m, o.r, o.vmax, o.rvmax, pa.scale_now);
        o.klypin_rs = rs;
    }
    o.rs = rs;
    // src/properties.c:351-382: m_pe_d counts the bound records with
    // r < r_pe_d; those come first (r2 is sorted): k_pe_tiles counts them
    double r_pe_d = rs * 4.0;
    if (r_pe_d < o.r / 5.0) r_pe_d = o.r / 5.0;
    r_pe_d *= 1e-3;
    r_pe[h] = r_pe_d;
    o.m_pe_b = (float)(pa.particle_mass * pow(c.pe_b, 2.0 / 3.0) /
                       cbrt(4.0 * M_PI * pa.rvir_dens_z0 / 3.0));
    props[h] = o;
}

// bound records with r < r_pe_d per tile
__global__ __launch_bounds__(kWave) void k_pe_tiles(const PropReads in,
                                                    const ScanTile *__restrict__ tiles,
                                                    int32_t ntiles,
                                                    const hp_halo *__restrict__ halos,
                                                    const int64_t *__restrict__ hfirst,
                                                    const int64_t *__restrict__ hcount,
                                                    const double *__restrict__ r_pe,
                                                    int32_t *__restrict__ cnt) {
    const int32_t t = blockIdx.x;
    if (t >= ntiles) return;
    const ScanTile tl = tiles[t];
    const int64_t first = hfirst[tl.call];
    const double lim = r_pe[tl.call];
    const int32_t end = min(tl.off + kScanTile, call_kept(halos, hcount, tl.call));
    int32_t n = 0;
    for (int32_t base = tl.off; base < end; base += kWave) {
        const int32_t j = base + lane_id();
        const uint64_t mb = in.bound[(int64_t)kTileWords * t + (base - tl.off) / kWave];
        n += __popcll(ballot(j < end && sqrt((double)in.r2[first + j]) < lim) & mb);
    }
    if (lane_id() == 0) cnt[t] = n;
}

__global__ __launch_bounds__(kWave) void k_pe_calls(int32_t nh, const int32_t *__restrict__ call_tile0,
                           const int32_t *__restrict__ call_ntiles,
                           const int32_t *__restrict__ cnt, PropArgs pa,
                           hp_halo_props *__restrict__ props) {
    const int32_t h = lane_call(nh, call_ntiles);
    const int32_t t0 = h < nh ? call_tile0[h] : 0, nt = h < nh ? call_ntiles[h] : 0;
    int32_t n = 0;  // a call's records are counted in 32 bits
    if (nt <= kFewTiles)
        for (int32_t t = t0; t < t0 + nt; t++) n += cnt[t];
    for_large_call(t0, nt, [&](int32_t a, int32_t k, bool mine) {
        int32_t m = 0;
        for (int32_t t = a + lane_id(); t < a + k; t += kWave) m += cnt[t];
        m = wave_sum(m);
        if (mine) n = m;
    });
    if (h < nh) props[h].m_pe_d = (float)((double)n * pa.particle_mass);
}

}  // namespace hp
