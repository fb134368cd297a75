// ecmc_chain_leg.h -- device code of the event-chain leg loop (see ecmc_chain.hip).
//
// One workgroup of NT threads (one or four wavefronts) advances one chain.  Every wavefront keeps
// the chain's state (active unit, its position, time, random cursor, estimators) in registers
// and runs the sequential part of a leg -- create lists, cell-boundary and end-of-chain events,
// selection, commit -- redundantly on the same values, so nothing of it is broadcast.  Only
// wavefront 0 writes the shared lists (cell occupants, positions, stored events) and memory.  A leg's
// barriers: after the occupancy update when the active unit changed, after the candidate tests (none
// where a single set is inverted without them), after the exact inversions, and before the thinning
// of a cell veto.  Only the third is in every leg, so what wavefronts exchange around it is kept
// twice (ChainShared::win).
//
// Bound by latency: one wavefront per SIMD issues an instruction of the leg's dependent chain about
// every seven cycles (4 to issue, the rest waits for results and LDS), whatever the chip could do
// besides; HBM and the FP64 rate are idle.  So a leg costs what its chain of instructions is long.
// Cycles per leg, one chain of 4096 Lennard-Jones units: occupancy 3400, nearby cells 2900, quick
// test of 512 candidates 6000, inversion of 5.6 contenders 6400 (beside it 1000 random words), their
// winner 1500, selection and event 2300, commit 1500, the loop 2300.  Leg times at the start of this
// form's work and now: 34.6 -> 11.9 us here, 11.7 -> 5.4 us for 256 hard disks, 66.6 -> 22.4 us for
// 256 systems of 512 charges with cell bounding, 51.7 -> 18.7 us with the cell veto, 53.6 -> 19.2 us for
// 64 systems of 1000 dipole units.
//
// The pair candidates of all taggers of a create list are evaluated together:
//   1. every candidate gets a cheap FP32 test (quick_cull) whether its factor can rise by the
//      drawn potential change within the horizon h of the leg; h is the time to the earliest
//      event already known (cell boundary, end of chain, sampling, cell veto), or a multiple of
//      the running mean of event times where that is sooner;
//   2. the few candidates left (the contenders) are inverted exactly in FP64, one per lane of a
//      wavefront, all taggers side by side, while another wavefront extends the random stream;
//   3. the earliest of them and of the stored events is committed if it lies within h (every
//      candidate left out ends later); otherwise h is widened and the step repeated.
// A tagger whose stored event outlives the commit (the committing tagger does not trash it, as a
// sampling event does not) gets its exact earliest candidate by a full evaluation first, so
// the stored events are always those of an unfiltered evaluation.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "../../include/jellyfysh_amd.h"
#include "ecmc_math.h"
#include "ecmc_potentials.h"
#include "ecmc_fp32_bounds.h"

namespace ecmc {

constexpr int AXIS_CELLS = 32;    // cells per side whose bounds are kept in LDS
constexpr int QCAP = 64;          // contenders queued per wavefront
constexpr int RING_STEP = 192;    // words one wavefront makes at a time (at most 227: see ring_make)
static_assert(ECMC_MAX_TAGGERS == 16, "the stored events are selected over one 16-lane row");

// The dynamic LDS of a leg-loop launch: a resident system's state (ChainArgs::lds_*_off).
extern __shared__ __align__(16) unsigned char chain_dyn_lds[];
// The taggers of a launch without it.
__device__ __forceinline__ ecmc_tagger_desc *static_taggers() {
    __shared__ ecmc_tagger_desc tg[ECMC_MAX_TAGGERS];
    return tg;
}

constexpr uint32_t MT_UPPER = 0x80000000u, MT_LOWER = 0x7fffffffu, MT_MATRIX = 0x9908b0dfu;

struct Slot {
    Time t;
    int64_t seq;
    int32_t valid, target;
    double apos[3];
    Time astamp;
    double tpos[3];
    double cb_boundary;
    int32_t cb_dir, adir;
    double aspeed;
    int32_t cb_cell, pad_cb;   // active cell of a cell-bounding candidate; target cell of a cell veto
    double cv_rate;            // cell veto: bounding event rate of the sampled cell
};

// One entry of Walker's table (walker.py:73-101): item0 with rate0, else the alias item1
struct CvEntry {
    double rate0;
    int32_t item0, item1;
};

struct ChainState {
    int32_t active, adir;
    double aspeed;
    Time at;
    int32_t occ_id, occ_cell;
    int32_t started, done, err, pending_creates, last_tagger, stop_reason;
    Time last;
    int64_t seq;
    Time eoc_last, samp_time;
    uint64_t cursor, produced;
    double est[8];
    int32_t ncand;
    uint32_t chash;
    int32_t nsur, pad_s;       // surplus units of a bounded occupancy
    double mean_step;          // running mean of the event times of a leg (sizes the horizon; no result depends on it)
    Slot slot[ECMC_MAX_TAGGERS];
};

// What the host reads after a launch, written by the launch's last instructions into the system's view in
// pinned host memory: the state, the committed legs and, of a launch that kept the
// positions in LDS, the positions (n x dim) behind this block.  Reading it costs no copy command:
// the four of a system (committed legs, state, positions, estimators), at 10 to 17 us each, were
// 14.1 of 40.6 ms where 256 systems of 512 units run 1000 legs and 14.6 of 26.5 ms where 256
// two-unit systems run to their next sample.
struct HostView {
    ChainState st;
    int64_t n_out;
    int32_t has_positions, pad;
};

struct ChainArgs {
    int32_t n, ncells, nb_stride, occ_cap, ring_words, n_taggers, stop_mask, leaves;   // leaves: leaf units per
                                                                                       // composite object (1: point masses)
    int32_t occupancy;         // some tagger reads the cell occupancy (else it is not kept up)
    int32_t nb_table;          // the nearby cells need the table (fewer than 2 layers + 1 cells on some axis)
    double L, half, beta;
    int32_t cps[3], cum[3];
    double side[3];
    Ewald ewald;
    double *pos;
    const double *charge;
    const double *cmin;
    const int32_t *nearby;
    const int32_t *nearby_n;
    int32_t *occ;
    int32_t *occ_n;
    uint32_t *ring;            // raw MT19937 words, word i of the run at i mod ring_words (the seed's 624 at -624 .. -1)
    ChainState *st;
    const ecmc_tagger_desc *tg;
    ecmc_event *log;
    int64_t max_events;
    HostView *host;            // device address of the system's host view (null: the host copies what it reads)
    int64_t *n_out;
    // bounded occupancy (single_active_cell_occupancy.py:62) and cell bounding
    int32_t max_occ, layers;
    int32_t *sur_cell, *sur_id;   // surplus units in the order the reference's dict yields them
    const double *cbt;            // cell-bound table: (cell offset, direction) -> upper, lower
    float cb_max[3];              // per direction the largest |entry| of the table, rounded up
    int32_t cv_m;
    // cell veto: Walker tables [direction * 2 + (0 upper, 1 lower)] of cv_m entries each
    const CvEntry *cvw;
    double cv_total[6], cv_mean[6];
    // residency (resident != 0): positions (dim x n doubles at offset 0), ring, charges, occupant counts
    // and surplus lists live in the launch's dynamic LDS at these offsets, copied in at the start of
    // a launch and back at its end, and so do the first occ_cols occupants of every cell (16-bit);
    // 0 keeps everything in global memory
    int32_t resident, lds_ring_off, lds_charge_off, lds_occ_off, lds_occn_off, lds_sur_off, lds_tg_off, occ_cols;
    int32_t ewald_ncodes, ewald_nreal;
    // the terms of the merged-image Coulomb derivative in the sequential loop's order (real-space
    // images by k, j, i, then Fourier terms by i, j, k): kind << 24 | (i + 128) << 16 |
    // (j + 128) << 8 | (k + 128), built on the host
    const int32_t *ewald_codes;
};

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)), __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
__device__ __forceinline__ uint64_t uni(uint64_t v) {
    return (uint64_t)(uint32_t)uni((int)(uint32_t)v) | ((uint64_t)(uint32_t)uni((int)(uint32_t)(v >> 32)) << 32);
}
__device__ __forceinline__ Time uni(Time t) { return Time{uni(t.q), uni(t.r)}; }
__device__ __forceinline__ double lane_d(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane), __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// A condition alike in every lane, as a scalar branch condition.  Values that went through a call
// or a lane permutation count as lane-varying to the compiler, and a branch on them would run
// through execution masks and keep everything it decides in vector registers.
__device__ __forceinline__ bool ub(bool c) { return __ballot(c) != 0ull; }
template <int NT>
__device__ __forceinline__ int wave_index() { return NT > 64 ? uni((int)(threadIdx.x >> 6)) : 0; }
// Orders a wavefront's own LDS accesses across its lanes (LDS operations of one wavefront complete
// in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The launch's constants that every leg reads, in registers (a scalar load of an argument would
// wait for it each time), and the tagger properties as bit fields.
template <int D>
struct Geo {
    unsigned char *dyn;        // the launch's dynamic LDS
    ecmc_tagger_desc *tg;      // the taggers, in LDS (a resident system's beside its state, as many as it has)
    int n, ncells, occ_cols, occ_cap, ring_mask, leaves, max_occ, o_ring, o_charge, o_occn, o_occ, o_sur;
    float inv_beta;            // 1 / beta rounded down
    double L, half, beta;
    double side[D], inv[D];    // cell side and its rounded inverse
    int cps[D], cum[D];
    float cb_max[3];           // cell bounding: the largest |rate| per direction and unit charge product
    int noff[D];               // lane k: the offset of the k-th nearby cell
    int nb_cells;              // nearby cells (0: read from the table)
    uint64_t kinds;            // 4 bits per tagger: its kind
    uint32_t tests;            // 2 bits per tagger: its quick test
    uint32_t inversions;       // 2 bits per tagger: 0 an inverse power inverted, 1 the Coulomb bound, 2 a rate or another potential
    uint32_t draws, charged;   // 1 bit per tagger
};
__device__ __forceinline__ int kind_of(uint64_t kinds, int t) { return (int)((kinds >> (4 * t)) & 15u); }

// State in LDS (RES) or in global memory.
template <bool RES, int D>
__device__ __forceinline__ int32_t occ_count(const ChainArgs &a, const Geo<D> &q, int c) {
    return RES ? reinterpret_cast<int32_t *>(q.dyn + q.o_occn)[c] : a.occ_n[c];
}
template <bool RES, int D>
__device__ __forceinline__ void set_occ_count(const ChainArgs &a, const Geo<D> &q, int c, int32_t v) {
    if (RES) reinterpret_cast<int32_t *>(q.dyn + q.o_occn)[c] = v;
    else a.occ_n[c] = v;
}
// Occupant k of cell c: the first occ_cols of a cell in LDS, those beyond in global memory.
template <bool RES, int D>
__device__ __forceinline__ int32_t occ_get(const ChainArgs &a, const Geo<D> &q, int c, int k) {
    if (RES && k < q.occ_cols) return reinterpret_cast<uint16_t *>(q.dyn + q.o_occ)[c * q.occ_cols + k];
    return a.occ[(size_t)c * q.occ_cap + k];
}
// Occupants place[u] of cells c[u]: the LDS reads together, memory only where some lane needs it.
template <bool RES, int U, int D>
__device__ __forceinline__ void occ_get_all(const ChainArgs &a, const Geo<D> &q, const int (&c)[U], const int (&place)[U], int (&v)[U]) {
    if (RES && q.occ_cols > 0) {
        const uint16_t *const lo = reinterpret_cast<const uint16_t *>(q.dyn + q.o_occ);
        bool beyond = false;
#pragma unroll
        for (int u = 0; u < U; u++) {
            v[u] = lo[c[u] * q.occ_cols + min(place[u], q.occ_cols - 1)];
            beyond |= place[u] >= q.occ_cols;
        }
        if (!ub(beyond)) return;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (place[u] >= q.occ_cols) v[u] = a.occ[(size_t)c[u] * q.occ_cap + place[u]];
    } else {
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = a.occ[(size_t)c[u] * q.occ_cap + place[u]];
    }
}
template <bool RES, int D>
__device__ __forceinline__ void occ_set(const ChainArgs &a, const Geo<D> &q, int c, int k, int32_t v) {
    if (RES && k < q.occ_cols) reinterpret_cast<uint16_t *>(q.dyn + q.o_occ)[c * q.occ_cols + k] = (uint16_t)v;
    else a.occ[(size_t)c * q.occ_cap + k] = v;
}
template <bool RES, int D>
__device__ __forceinline__ int32_t sur_cell(const ChainArgs &a, const Geo<D> &q, int i) {
    return RES ? reinterpret_cast<int32_t *>(q.dyn + q.o_sur)[i] : a.sur_cell[i];
}
template <bool RES, int D>
__device__ __forceinline__ int32_t sur_id(const ChainArgs &a, const Geo<D> &q, int i) {
    return RES ? reinterpret_cast<int32_t *>(q.dyn + q.o_sur)[q.n + i] : a.sur_id[i];
}
template <bool RES, int D>
__device__ __forceinline__ void set_sur(const ChainArgs &a, const Geo<D> &q, int i, int32_t c, int32_t id) {
    if (RES) {
        reinterpret_cast<int32_t *>(q.dyn + q.o_sur)[i] = c;
        reinterpret_cast<int32_t *>(q.dyn + q.o_sur)[q.n + i] = id;
    } else {
        a.sur_cell[i] = c;
        a.sur_id[i] = id;
    }
}
// The charge of unit id (constant over a run).
template <bool RES, int D>
__device__ __forceinline__ double charge_of(const ChainArgs &a, const Geo<D> &q, int id) {
    return RES ? reinterpret_cast<const double *>(q.dyn + q.o_charge)[id] : a.charge[id];
}
template <bool RES, int D>
__device__ __forceinline__ void load_pos(const ChainArgs &a, const Geo<D> &q, int id, double *p) {
    if (RES) {
        const double *lp = reinterpret_cast<const double *>(q.dyn) + id;
#pragma unroll
        for (int d = 0; d < D; d++) p[d] = lp[d * q.n];
    } else {
#pragma unroll
        for (int d = 0; d < D; d++) p[d] = a.pos[(size_t)d * q.n + id];
    }
}
template <bool RES, int D>
__device__ __forceinline__ void store_pos(const ChainArgs &a, const Geo<D> &q, int id, const double *p) {
    if (RES) {
        double *lp = reinterpret_cast<double *>(q.dyn) + id;
#pragma unroll
        for (int d = 0; d < D; d++) lp[d * q.n] = p[d];
    } else {
#pragma unroll
        for (int d = 0; d < D; d++) a.pos[(size_t)d * q.n + id] = p[d];
    }
}
// v[i] for a runtime index: selects of values read beforehand (a read behind the selection would
// index the array at run time and put it, and the struct around it, into private memory).
template <int D, class T>
__device__ __forceinline__ T pick_axis(const T *v, int i) {
    const T v0 = v[0], v1 = v[1], v2 = v[D - 1];
    T r = v0;
    r = i == 1 ? v1 : r;
    r = i == 2 ? v2 : r;
    return r;
}

// ---- random stream ------------------------------------------------------------------------
// The ring holds the untempered MT19937 sequence itself: word i is x_i = x_(i-227) ^
// twist(x_(i-624), x_(i-623)) for every i >= 0, the seeded state being x_(-624) .. x_(-1) (the
// generator's in-place state is the last 624 words of the sequence).  The first 227 words after
// any point depend only on words before it, so one wavefront makes RING_STEP <= 227 words with
// no wait between its lanes, and readers temper the words they read.
__device__ __forceinline__ uint32_t mt_temper(uint32_t y) {
    y ^= (y >> 11);
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= (y >> 18);
    return y;
}
__device__ __forceinline__ uint32_t mt_next(uint32_t x624, uint32_t x623, uint32_t x227) {
    const uint32_t y = (x624 & MT_UPPER) | (x623 & MT_LOWER);
    return x227 ^ (y >> 1) ^ ((y & 1u) ? MT_MATRIX : 0u);
}
// One wavefront makes words [from, from + steps * RING_STEP) of the ring (mask: its size - 1,
// at least 1023, so that a step overwrites no word it reads).
__device__ __forceinline__ void ring_make(uint32_t *ring, uint32_t mask, uint64_t from, int steps) {
    const int lane = threadIdx.x & 63;
    uint32_t b = (uint32_t)from + lane;
#pragma unroll 1
    for (int s = 0; s < steps; s++, b += RING_STEP) {
        uint32_t v[RING_STEP / 64];
#pragma unroll
        for (int u = 0; u < RING_STEP / 64; u++) {
            const uint32_t i = b + 64 * u;
            v[u] = mt_next(ring[(i - 624u) & mask], ring[(i - 623u) & mask], ring[(i - 227u) & mask]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
#pragma unroll
        for (int u = 0; u < RING_STEP / 64; u++) ring[(b + 64 * u) & mask] = v[u];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // the next step reads these words from other lanes
    }
}
// The same in LDS, where a wavefront's operations are in order: nothing waits for a step's writes, the
// words 624 and 623 back of the next step (older than this step's) are read while this one waits
// for its words 227 back, and the mask is left out where none of the four runs wraps.  575 -> 465
// cycles a step of 192 words (21 steps a leg of 1000 dipole units).
__device__ __forceinline__ void ring_make_lds(uint32_t *ring, uint32_t mask, uint64_t from, int steps) {
    constexpr int U = RING_STEP / 64;
    const uint32_t lane = threadIdx.x & 63;
    uint32_t at = (uint32_t)uni((int)(uint32_t)from);
    uint32_t x[U], y[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        x[u] = ring[(at + lane + 64u * u - 624u) & mask];
        y[u] = ring[(at + lane + 64u * u - 623u) & mask];
    }
#pragma unroll 1
    for (int s = 0; s < steps; s++, at += RING_STEP) {
        uint32_t z[U], nx[U], ny[U];
        const uint32_t o = at & mask, r = (at - 227u) & mask, n = (at + RING_STEP - 624u) & mask;
        const bool wraps = max(max(o, r), n) + RING_STEP + 1u > mask + 1u;   // (uniform)
        if (!wraps) {
            const uint32_t *const pr = ring + r + lane, *const pn = ring + n + lane;
#pragma unroll
            for (int u = 0; u < U; u++) z[u] = pr[64 * u];
#pragma unroll
            for (int u = 0; u < U; u++) {
                nx[u] = pn[64 * u];
                ny[u] = pn[64 * u + 1];
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; u++) {
                z[u] = ring[(r + lane + 64u * u) & mask];
                nx[u] = ring[(n + lane + 64u * u) & mask];
                ny[u] = ring[(n + lane + 64u * u + 1u) & mask];
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) z[u] = mt_next(x[u], y[u], z[u]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (!wraps) ring[o + lane + 64u * u] = z[u];
            else ring[(o + lane + 64u * u) & mask] = z[u];
            x[u] = nx[u];
            y[u] = ny[u];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the next step reads these words from other lanes
    }
}
template <bool RES, int D>
__device__ __forceinline__ void ring_make(const ChainArgs &a, const Geo<D> &q, uint64_t from, int steps) {
    if (RES) ring_make_lds(reinterpret_cast<uint32_t *>(q.dyn + q.o_ring), (uint32_t)q.ring_mask, from, steps);
    else ring_make(a.ring, (uint32_t)q.ring_mask, from, steps);
}
// Word `off` after the leg's first word `keep` (32-bit: the ring's mask drops the rest).
template <bool RES, int D>
__device__ __forceinline__ uint32_t ring_word(const ChainArgs &a, const Geo<D> &q, uint32_t idx) {
    const uint32_t i = idx & (uint32_t)q.ring_mask;
    return mt_temper(RES ? reinterpret_cast<const uint32_t *>(q.dyn + q.o_ring)[i] : a.ring[i]);
}

// random() from two words (genrand_res53)
__device__ __forceinline__ double words_to_random(uint32_t w0, uint32_t w1) {
    uint32_t x = w0 >> 5, y = w1 >> 6;
    return (x * 67108864.0 + y) * (1.0 / 9007199254740992.0);
}

// candidate-set hash term: order dependent, summed over the candidates of a leg
__device__ __forceinline__ uint32_t cand_mix(uint32_t j, uint32_t target) {
    uint32_t h = (j * 0x9E3779B9u) ^ target;
    h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
    return h;
}

// ---- geometry -----------------------------------------------------------------------------
// Uniform arguments: py_mod for a positive modulus, time_add, with scalar branches.
__device__ __forceinline__ double mod_u(double x, double y) {
    if (ub(x >= 0.0 && x < y)) return x + 0.0;
    if (ub(x >= 0.0 && x < 2.0 * y)) return x - y;
    return py_mod(x, y);
}
__device__ __forceinline__ Time time_add_u(Time t, double dt) {
    const double v = t.r + dt;
    if (ub(v >= 0.0 && v < 0x1p52 && dt < 0x1p52)) {
        const double f = floor(v);
        return Time{t.q + f, v - f};
    }
    return time_add(t, dt);
}
// The cell of a position, int(x / side) per axis (cuboid_cells.py), uniform.  The quotient is taken by the
// rounded inverse first: it is within 2^-51 relative of x / side, so an integer part at least
// 2^-30 away from the next integer is that of the division; else the division decides.
__device__ __forceinline__ int axis_cell(double x, double side, double inv) {
    const double q = x * inv;
    int k = (int)q;
    const double f = q - (double)k;
    if (ub(!(f > 0x1p-30 && f < 1.0 - 0x1p-30 && q < 0x1p20))) k = (int)(x / side);
    return k;
}
// The cell of a position and its coordinates; -1 outside the cell system.
template <int D>
__device__ __forceinline__ int pos_to_cell(const Geo<D> &q, const double *p, int *coord) {
    int idx = 0;
#pragma unroll
    for (int d = 0; d < D; d++) {
        coord[d] = axis_cell(p[d], q.side[d], q.inv[d]);
        idx += coord[d] * q.cum[d];
    }
    return idx < 0 || idx >= q.ncells ? -1 : idx;
}

template <int D>
__device__ __forceinline__ void separation_vector(const Geo<D> &q, const double *ap, const double *tp, double *s) {
    // within one period either way py_mod's value is x, x - L or x + L
    bool far = false;
    double x[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        x[d] = (tp[d] - ap[d]) + q.half;
        far |= !((x[d] > -q.L) & (x[d] < 2.0 * q.L));
        s[d] = (x[d] < 0.0 ? x[d] + q.L : (x[d] >= q.L ? x[d] - q.L : x[d])) - q.half;
    }
    if (!far) return;
#pragma unroll
    for (int d = 0; d < D; d++) s[d] = py_mod(x[d], q.L) - q.half;
}
template <int D>
__device__ __forceinline__ void separation_vector_u(const Geo<D> &q, const double *ap, const double *tp, double *s) {
#pragma unroll
    for (int d = 0; d < D; d++) {
        const double x = (tp[d] - ap[d]) + q.half;
        s[d] = (ub(x < 0.0 && x > -q.L) ? x + q.L : mod_u(x, q.L)) - q.half;
    }
}

// event_handler/abstracts/abstracts.py:82-95 for a velocity with one nonzero component: the other
// components are p % L, which leaves a position inside [0, L) as it is.
template <int D>
__device__ __forceinline__ void slice_pos(const Geo<D> &q, double *p, int dir, double speed, Time from, Time to) {
    const double dt = time_sub(to, from);
#pragma unroll
    for (int d = 0; d < D; d++) {
        const double x = d == dir ? p[d] + speed * dt : p[d];
        p[d] = mod_u(x, q.L);
    }
}

__device__ __forceinline__ bool pot_draws(const ecmc_tagger_desc &tg) {
    if (tg.event_handler == ECMC_EH_TWO_LEAF_BOUNDING) return true;
    return tg.potential != ECMC_POT_HARD_SPHERE && tg.potential != ECMC_POT_HARD_DIPOLE;
}
__device__ __forceinline__ bool pair_kind(int kind) {
    return kind == ECMC_TAG_PAIR_CELLS || kind == ECMC_TAG_PAIR_ALL || kind == ECMC_TAG_SURPLUS ||
           kind == ECMC_TAG_CELL_BOUNDING || kind == ECMC_TAG_FACTOR_MAP;
}

// Bounding event rate of a cell-bounding candidate: the InnerPointEstimator bound of the
// target cell's offset from the active cell along dir, upper or lower by the sign of the
// charge correction factor (cell_bounding_potential.py:161-201).
template <int D>
__device__ __forceinline__ double cell_rate_of_cells(const ChainArgs &a, const Geo<D> &q, const ecmc_tagger_desc &tg, int acell,
                                                     int tcell, int dir, double ca, double ct) {
    int rel = 0;
#pragma unroll
    for (int d = 0; d < D; d++) {
        const int off = (tcell / q.cum[d]) % q.cps[d] - (acell / q.cum[d]) % q.cps[d];
        rel += (off < 0 ? off + q.cps[d] : off) * q.cum[d];
    }
    const double *row = a.cbt + (size_t)(rel * 3 + dir) * 2;
    if (tg.use_charge) {
        const double cf = ca * ct / tg.bpar[2];
        return cf > 0.0 ? row[0] * cf : row[1] * cf;
    }
    return row[0];
}

// Kernel variants by the features of the systems they run (FM): bit p for the two-leaf pair
// potential ECMC_POT_p inverted exactly, FEAT_COULOMB for the merged-image Coulomb factors through
// the inverse-power Coulomb bound (thinning by the Ewald derivative), FEAT_FMAP for factor-type
// maps, FEAT_CELL_BOUNDING and FEAT_CELL_VETO for the two far-cell schemes.  A variant leaves the
// code of the other features out of the kernel (a smaller leg loop, fewer instruction-cache
// misses); the host launches the first variant that covers every feature of its systems.
constexpr int FEAT_COULOMB = 1 << 9, FEAT_FMAP = 1 << 10, FEAT_CELL_BOUNDING = 1 << 11, FEAT_CELL_VETO = 1 << 12;
constexpr int FEAT_ALL = (1 << 13) - 1;
constexpr int FEAT_EWALD = FEAT_COULOMB | FEAT_CELL_BOUNDING | FEAT_CELL_VETO;   // thinning by the Ewald derivative
constexpr int FEAT_IP = (1 << ECMC_POT_INVERSE_POWER) | (1 << ECMC_POT_INVERSE_POWER_TRUNC);
constexpr int VARIANT_LJ = FEAT_IP;
constexpr int VARIANT_CHARGED_CB = (1 << ECMC_POT_INVERSE_POWER) | FEAT_COULOMB | FEAT_CELL_BOUNDING;
constexpr int VARIANT_CHARGED_CV = (1 << ECMC_POT_INVERSE_POWER) | FEAT_COULOMB | FEAT_CELL_VETO;
constexpr int VARIANT_DIPOLES = (1 << ECMC_POT_INVERSE_POWER) | (1 << ECMC_POT_DISPLACED_EVEN_POWER) | FEAT_COULOMB | FEAT_FMAP;
#define POT_BUILT(p) ((FM >> (p)) & 1)

// ip_displacement and ipt_displacement (potentials) as one instruction stream with selects, so
// that lanes inverting the repulsive and the attractive factor of a Lennard-Jones pair do not
// run two paths: the same operations on the same values.  urc = U(rc) and rc2 = rc^2 of the
// truncated form, 0 and +inf without a cutoff (then current >= urc is the reference's test
// against zero).
//
// SettledPowers takes the powers through the fast paths alone, without a branch or a call between
// them (ok turns false where they do not settle a rounding, about one time in 500, by the logarithm of
// the draw): the two powers, the logarithm and the root's parts then overlap in one instruction
// stream.  1000 legs of 4096 Lennard-Jones units: 12.12 -> 11.90 ms.
struct AnyPowers {
    __device__ __forceinline__ double half(double r2, double power) { return pow_half_power(r2, power); }
    __device__ __forceinline__ double root(double x, double power) { return root_two_over_power(x, power); }
};
struct SettledPowers {   // powers 6 and 12
    bool ok = true;
    __device__ __forceinline__ double half(double r2, double power) { return pow36_settled(r2, power == 12.0, ok); }
    __device__ __forceinline__ double root(double x, double power) { return root36_settled(x, power == 12.0, ok); }
};
__device__ __forceinline__ double over_speed(double x, double speed) { return speed == 1.0 ? x : x / speed; }
// A displacement that the reference code answers with a ValueError because a root's argument rounds
// below zero (an attractive unit passed so closely that the draw is lost in the energy there): NaN, with
// the time t of the closest approach, where the event would be, as a float in the low word.
__device__ __forceinline__ double error_at(double t) {
    return __hiloint2double(0x7ff80000, __float_as_int((float)fmax(t, 0.0) * (1.f - 0x1p-22f)));
}
// The time of a NaN displacement as a positive number that is larger for earlier times (every other
// NaN: time 0), and the time of that number.
__device__ __forceinline__ int error_code(double dt) {
    const int bits = __double2loint(dt);
    return 0x7f800001 - (bits < 0 || bits > 0x7f800000 ? 0 : bits);
}
__device__ __forceinline__ float error_time(int code) { return __int_as_float(0x7f800001 - code); }
template <int D, class Powers>
__device__ __forceinline__ double ip_time(Powers &m, int dir, double speed, const double *sep, double pp, double power, double rc2,
                                          double urc, double dU) {
    const bool rep = pp > 0.0;
    const double perp2 = others_sq<D>(sep, dir);
    const double sd = dir == 0 ? sep[0] : (D == 2 || dir == 1 ? sep[1] : sep[D - 1]);
    const bool shift = !rep && sd > 0.0;      // an attractive unit ahead is first passed
    const double disp = shift ? sd : 0.0, sdd = shift ? 0.0 : sd;
    double c[D];
#pragma unroll
    for (int d = 0; d < D; d++) c[d] = d == dir ? sdd : sep[d];
    const double sn2 = norm_sq<D>(c);
    bool live = perp2 < rc2 && (rep ? sd > 0.0 : sn2 < rc2);
    const double cur = (rep && !(sn2 < rc2)) ? urc : pp / m.half(live ? sn2 : 1.0, power);
    const double maxp = pp / m.half(rep && live ? perp2 : 1.0, power);
    live = live && (rep ? dU < maxp - cur : !(cur + dU >= urc));
    const double nsq = m.root(live ? pp / (cur + dU) : 1.0, power);
    const double a = nsq - perp2;
    const double sq = sqrt(fmax(a, 0.0));
    const double t = over_speed(rep ? sdd - sq : disp + (sdd + sq), speed);
    const double res = a < 0.0 ? error_at(t) : t;
    return live ? res : INFINITY;
}

// How a candidate's time is computed: the potential inverted exactly (ECMC_POT_*), the Coulomb
// bound, or a bounding rate.
enum { TIME_COULOMB_BOUND = 16, TIME_RATE = 17 };
// Candidate time displacement (send_event_time of the pair event handlers): the potential change
// dU = -log(1 - u) / beta of the words (w0, w1), inverted for separation (s0, s1, s2), parameters
// p0 .. p2 and charges c1, c2; x is rc^p of a truncated inverse power or the box length of the
// Coulomb bound; p2, x and y are the minimum and the two factors of a Lennard-Jones potential.  A call, not inlined: everything comes in registers, and inside the leg loop the
// constants and temporaries of these chains would push the loop's own state out of them.
template <int D, int FM>
__device__ __noinline__ static double pair_time(int how, double p0, double p1, double p2, double x, double y, int dir, double speed,
                                                double s0, double s1, double s2, double c1, double c2, uint32_t w0, uint32_t w1, double beta) {
    double s[D];
    s[0] = s0;
    s[1] = s1;
    if (D > 2) s[D - 1] = s2;
    if ((FM & FEAT_IP) && (how == ECMC_POT_INVERSE_POWER || how == ECMC_POT_INVERSE_POWER_TRUNC) && (p0 == 12.0 || p0 == 6.0)) {
        const bool trunc = how == ECMC_POT_INVERSE_POWER_TRUNC;
        const double pp = (c1 * c2) * p1;
        SettledPowers m;
        const double change = -log_settled(1.0 - words_to_random(w0, w1), m.ok) / beta;
        const double dt = ip_time<D>(m, dir, speed, s, pp, p0, trunc ? p2 * p2 : INFINITY, trunc ? pp / x : 0.0, change);
        if (m.ok) return dt;
    }
    // hard potentials draw nothing (beta = 0 marks them)
    const double dU = beta != 0.0 ? -cr_log(1.0 - words_to_random(w0, w1)) / beta : 0.0;
    if ((FM & FEAT_IP) && (how == ECMC_POT_INVERSE_POWER || how == ECMC_POT_INVERSE_POWER_TRUNC)) {
        const bool trunc = how == ECMC_POT_INVERSE_POWER_TRUNC;
        const double pp = (c1 * c2) * p1;
        AnyPowers m;
        return ip_time<D>(m, dir, speed, s, pp, p0, trunc ? p2 * p2 : INFINITY, trunc ? pp / x : 0.0, dU);
    }
    if ((FM & FEAT_COULOMB) && how == TIME_COULOMB_BOUND) {
        // two_leaf_unit_bounding_potential_event_handler.py:138-143 with the Coulomb bound
        double p[3] = {0, 0, 0};
#pragma unroll
        for (int d = 0; d < D; d++) p[d] = pick_axis<D>(s, dir + d >= D ? dir + d - D : dir + d);
        return over_speed(ipcb_displacement(p0 * c1 * c2, p[0], p[1], p[2], dU, x), speed);
    }
    // two_leaf_unit_cell_bounding_potential_event_handler.py:171-177, p0 the rate
    if ((FM & FEAT_CELL_BOUNDING) && how == TIME_RATE) return over_speed(p0 > 0 ? dU / p0 : INFINITY, speed);
    if (POT_BUILT(ECMC_POT_HARD_SPHERE) && how == ECMC_POT_HARD_SPHERE) return hs_displacement<D>(dir, speed, s, p0);
    if (POT_BUILT(ECMC_POT_HARD_DIPOLE) && how == ECMC_POT_HARD_DIPOLE) return hd_displacement<D>(dir, speed, s, p0, p1);
    if (POT_BUILT(ECMC_POT_LENNARD_JONES) && how == ECMC_POT_LENNARD_JONES)
        return mh_displacement<D>(MexicanHat{1, p0, p1, p2, p2 * p2, x, y, 0.0, 0.0}, dir, speed, s, dU);
    if (POT_BUILT(ECMC_POT_DISPLACED_EVEN_POWER) && how == ECMC_POT_DISPLACED_EVEN_POWER)
        return mh_displacement<D>(mh_displaced_even_power(p0, p1, p2), dir, speed, s, dU);
    return NAN;
}
// dU of a draw, called for the same reason.
__device__ __noinline__ static double drawn_change(uint32_t w0, uint32_t w1, double beta) {
    return -cr_log(1.0 - words_to_random(w0, w1)) / beta;
}

// Candidate j of a factor-map tagger (factor_type_maps.py:325-356): a local factor's entries for
// the active leaf number k; a non-local factor's entries for every other composite object in
// identifier order, the entry's other leaf in that object (or, for numbers below P, in the
// active unit's own object).
__device__ __forceinline__ int fmap_target(const ecmc_tagger_desc &tg, int P, int m, int k, int fn, int j) {
    if (tg.fmap_local) return m * P + tg.fmap_target[k][j];
    const int o = fn == 1 ? j : (fn == 2 ? j >> 1 : (fn == 4 ? j >> 2 : j / fn)), e = j - o * fn;
    const int other = o < m ? o : o + 1;
    const int tl = tg.fmap_target[k][e];
    return tl < P ? m * P + tl : other * P + (tl - P);
}
__device__ __forceinline__ int fmap_count(const ecmc_tagger_desc &tg, int P, int n, int act) {
    const int fn = tg.fmap_n[act % P];
    return tg.fmap_local ? fn : (n / P - 1) * fn;
}

// ---- lane permutations --------------------------------------------------------------------
// Lane permutations of the 16-lane rows (CTRL: 0xB1 swaps neighbours, 0x4E pairs of neighbours,
// 0x141 mirrors each half row, 0x140 the row): after the four steps of a minimum every lane of
// a row holds the row's.
template <int CTRL>
__device__ __forceinline__ int dpp_move(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false); }
template <int CTRL>
__device__ __forceinline__ double dpp_move_d(double v) {
    return __hiloint2double(dpp_move<CTRL>(__double2hiint(v)), dpp_move<CTRL>(__double2loint(v)));
}
// Minimum of a double (no NaN) over the wavefront, uniform.
__device__ __forceinline__ double wave_min(double v) {
    v = fmin(v, dpp_move_d<0xB1>(v));
    v = fmin(v, dpp_move_d<0x4E>(v));
    v = fmin(v, dpp_move_d<0x141>(v));
    v = fmin(v, dpp_move_d<0x140>(v));
    return fmin(fmin(lane_d(v, 0), lane_d(v, 16)), fmin(lane_d(v, 32), lane_d(v, 48)));
}
__device__ __forceinline__ int wave_min(int v) {
    v = min(v, dpp_move<0xB1>(v));
    v = min(v, dpp_move<0x4E>(v));
    v = min(v, dpp_move<0x141>(v));
    v = min(v, dpp_move<0x140>(v));
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
// Inclusive sum scan over the first 32 lanes (row shifts, then row 0's total to lanes 16-31).
__device__ __forceinline__ int scan32(int v, int lane) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    const int row0 = __builtin_amdgcn_readlane(v, 15);
    return lane >= 16 ? v + row0 : v;
}

// ---- the leg's state ----------------------------------------------------------------------
// What a tagger's candidates are tested and evaluated with, per launch.
enum { QT_DIRECT = 0, QT_INVERSE_POWER = 1, QT_COULOMB_BOUND = 2, QT_CELL = 3 };
struct TaggerPlan {
    uint64_t create;     // the tagger's create list, 4 bits per entry
    uint32_t trash;      // its trash list as a bit mask
    int32_t n_create;
    int32_t p;           // integer power of the inverse-power test
    int32_t set_key;     // taggers with one key enumerate the same candidates
    float rc2_hi;        // squared cutoff rounded up (+inf: none)
    double powrc;        // rc^p of a truncated inverse power
    double r0, k6, k12;  // Lennard-Jones: the minimum and the factors of r^-6 and r^-12
};
// A candidate to invert exactly: its first random word and push rank (both from the leg's first),
// its unit, and tagger | target cell << 4 (the cell of a cell-bounding candidate).
struct Contender {
    uint32_t word;
    int32_t rank, target, tag_cell;
};
// An earliest pair candidate: its time, push rank (NO_RANK: none), tagger and unit; bad: not 0 where
// some candidate was NaN (a ValueError of the reference code), the larger the earlier (error_code).
constexpr int NO_RANK = 0x7fffffff;
struct Winner {
    Time t;
    double dt;
    int32_t rank, tag, target, bad;
};

template <int D>
struct Leg {
    int active, adir;
    double aspeed;
    Time at;
    double ap[D];                // position of the active unit at `at`
    int occ_id, occ_cell;
    int cc[D];                   // coordinates of occ_cell
    int started, done, err, pending, last_tagger, committed;
    Time last;
    int64_t seq;
    Time eoc_last, samp_time;
    uint64_t cursor, produced, keep;   // keep: the leg's first random word
    int ncand;
    uint32_t chash;
    int nsur;
    double mean_step;
    // the stored events as lane t < ECMC_MAX_TAGGERS sees tagger t's
    Time lt;
    int64_t lseq;
    int lvalid;
};

// The create list of the pair and cell-boundary events' own legs, which nearly every leg runs: pair
// taggers, at most one cell boundary and at most one cell veto, at any places.  Legs of this list take the
// short path (hot_events); the others (a sampling event's, the run's start) the general one.
constexpr int HOT_ITEMS = 4;
struct HotList {
    int32_t items;          // pair taggers (-1: no such list)
    uint32_t tags;          // 4 bits per pair tagger
    int32_t boundary, veto; // taggers, -1: none
    int32_t before;         // pair taggers created before the cell boundary
    int32_t veto_before;    // and before the cell veto
    uint32_t mask;          // all of them
    uint32_t creators;      // bit t: tagger t creates this list
    uint32_t prefixed;      // bit t: tagger t creates other taggers, then this list
    uint32_t trashers;      // bit t: tagger t trashes all of this list
    int32_t hard;           // its one pair tagger is a hard sphere's, of this radius
    double radius;
};

struct SlotTime {
    Time t;
    int64_t seq;
    int32_t valid, pad;
};
// The terms of the merged-image Coulomb derivative as the FP32 form takes them: a real-space image and
// two Fourier terms per lane, where no more are needed (ok).
struct EwaldTerms {
    int32_t code[3][64];         // image, Fourier terms (-1: none), as ChainArgs::ewald_codes
    float f[2][64];
    double L, inv_l;
    float aol, aol2, two_aol_rpi;
    int32_t ok;
};
template <int NT>
struct ChainShared {
    static constexpr int NW = NT / 64;
    Slot slot[ECMC_MAX_TAGGERS];             // payloads of the stored events, written by thread 0
    SlotTime time[NW][ECMC_MAX_TAGGERS];     // their times as every wavefront sees them, around a rare step
    TaggerPlan plan[ECMC_MAX_TAGGERS];
    Contender queue[NW][QCAP];
    // The earliest candidate of every wavefront: of the legs in turn, and of the rare steps' full
    // evaluations.  A leg may have no barrier after the one that its winners are read behind, and the
    // next leg none before it writes its own: the slowest wavefront may still be reading one copy
    // while the fastest fills the other, and the barrier of that leg lies before the first is
    // written again.
    Winner win[3][NW];
    alignas(16) int32_t nb_cell[NW][32];     // nearby cells and exclusive prefix sums of their occupants
    alignas(16) int32_t nb_pref[NW][32];
    EwaldTerms ewald;
    uint32_t far_word[NW][64], far_pref[NW][64];
    uint32_t occupied[64];       // one bit per occupied cell (cell bounding, grids of at most FAR_BLOCK cells)
    int32_t qn[NW];
    uint32_t hash[NW];
    int32_t occ_err, occ_nsur;
    double axis[3][AXIS_CELLS];  // lower bounds of the cells per axis
    double est[8];               // the estimators, summed by the first lane of wavefront 0
    Geo<3> geo;                  // the launch's constants and every wavefront's leg, for the calls of the
    Leg<3> leg[NW];              // rare steps
    ecmc_event ev;
    HotList hot;
};

// The leg to and from LDS around a rare step: uniform fields by the first lane, the stored events'
// times by their lanes.
template <int D>
__device__ __forceinline__ void leg_to(const Leg<D> &g, Leg<3> &m, SlotTime *time) {
    const int lane = threadIdx.x & 63;
    if (lane == 0) {
        m.active = g.active; m.adir = g.adir; m.aspeed = g.aspeed; m.at = g.at;
#pragma unroll
        for (int d = 0; d < D; d++) { m.ap[d] = g.ap[d]; m.cc[d] = g.cc[d]; }
        m.occ_id = g.occ_id; m.occ_cell = g.occ_cell;
        m.started = g.started; m.done = g.done; m.err = g.err; m.pending = g.pending; m.last_tagger = g.last_tagger;
        m.committed = g.committed;
        m.last = g.last; m.seq = g.seq; m.eoc_last = g.eoc_last; m.samp_time = g.samp_time;
        m.cursor = g.cursor; m.produced = g.produced; m.keep = g.keep;
        m.ncand = g.ncand; m.chash = g.chash; m.nsur = g.nsur; m.mean_step = g.mean_step;
    }
    if (lane < ECMC_MAX_TAGGERS) {
        time[lane].t = g.lt; time[lane].seq = g.lseq; time[lane].valid = g.lvalid;
    }
}
template <int D>
__device__ __forceinline__ void leg_from(const Leg<3> &m, const SlotTime *time, Leg<D> &g) {
    const int lane = threadIdx.x & 63;
    g.active = uni(m.active); g.adir = uni(m.adir); g.aspeed = uni(m.aspeed); g.at = uni(m.at);
#pragma unroll
    for (int d = 0; d < D; d++) { g.ap[d] = uni(m.ap[d]); g.cc[d] = uni(m.cc[d]); }
    g.occ_id = uni(m.occ_id); g.occ_cell = uni(m.occ_cell);
    g.started = uni(m.started); g.done = uni(m.done); g.err = uni(m.err); g.pending = uni(m.pending);
    g.last_tagger = uni(m.last_tagger); g.committed = uni(m.committed);
    g.last = uni(m.last); g.seq = (int64_t)uni((uint64_t)m.seq); g.eoc_last = uni(m.eoc_last); g.samp_time = uni(m.samp_time);
    g.cursor = uni(m.cursor); g.produced = uni(m.produced); g.keep = uni(m.keep);
    g.ncand = uni(m.ncand); g.chash = (uint32_t)uni((int)m.chash); g.nsur = uni(m.nsur); g.mean_step = uni(m.mean_step);
    const SlotTime &sl = time[lane & 15];
    g.lt = sl.t; g.lseq = sl.seq; g.lvalid = lane < ECMC_MAX_TAGGERS && sl.valid;
}
// The launch's constants: the offsets of lane k's nearby cell (the product of the offsets, the last
// axis fastest), and the rest from LDS.
template <int D>
__device__ __forceinline__ void nearby_offsets(const ChainArgs &a, Geo<D> &q) {
    const int span = 2 * a.layers + 1;
    int rem = threadIdx.x & 63;
#pragma unroll
    for (int d = D - 1; d >= 0; d--) {
        q.noff[d] = rem % span - a.layers;
        rem /= span;
    }
}
template <int D>
__device__ __forceinline__ void geo_load(const Geo<3> &m, const ChainArgs &a, Geo<D> &q) {
    q.dyn = reinterpret_cast<unsigned char *>(uni((uint64_t)m.dyn));
    q.tg = reinterpret_cast<ecmc_tagger_desc *>(uni((uint64_t)m.tg));
    q.n = uni(m.n); q.ncells = uni(m.ncells); q.occ_cols = uni(m.occ_cols); q.occ_cap = uni(m.occ_cap);
    q.ring_mask = uni(m.ring_mask); q.leaves = uni(m.leaves); q.max_occ = uni(m.max_occ);
    q.o_ring = uni(m.o_ring); q.o_charge = uni(m.o_charge); q.o_occn = uni(m.o_occn); q.o_occ = uni(m.o_occ); q.o_sur = uni(m.o_sur);
    q.L = uni(m.L); q.half = uni(m.half); q.beta = uni(m.beta); q.inv_beta = m.inv_beta;
#pragma unroll
    for (int d = 0; d < D; d++) {
        q.side[d] = uni(m.side[d]); q.inv[d] = uni(m.inv[d]);
        q.cps[d] = uni(m.cps[d]); q.cum[d] = uni(m.cum[d]);
    }
    q.nb_cells = uni(m.nb_cells); q.kinds = uni(m.kinds); q.tests = (uint32_t)uni((int)m.tests);
    q.inversions = (uint32_t)uni((int)m.inversions);
    q.draws = (uint32_t)uni((int)m.draws); q.charged = (uint32_t)uni((int)m.charged);
    nearby_offsets<D>(a, q);
}

// The pair taggers of one leg's create list, in order: item i's tagger in 4 bits of tags; lane i
// holds its first random word and push rank (from the leg's first) and the candidates before it.
struct Items {
    int count;
    uint64_t tags;
    uint32_t word;
    int32_t rank, before;
    int32_t p;           // launch constants of item i in lane i: TaggerPlan::p, rc2_hi, set_key and the
    float rc2_hi, pref;  // prefactor of the quick test
    int32_t set_key;
};
__device__ __forceinline__ float item_f(float v, int i) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i)); }
__device__ __forceinline__ int item_tag(const Items &it, int i) { return (int)((it.tags >> (4 * i)) & 15u); }
__device__ __forceinline__ uint32_t item_word(const Items &it, int i) { return (uint32_t)__builtin_amdgcn_readlane((int)it.word, i); }
__device__ __forceinline__ int item_rank(const Items &it, int i) { return __builtin_amdgcn_readlane(it.rank, i); }

// An estimator's sum, one addition a leg in leg order: by the first lane of wavefront 0, as an LDS
// operation that nothing waits for.
template <int NT>
__device__ __forceinline__ void add_est(ChainShared<NT> &sh, int k, double v) {
    if (threadIdx.x == 0) unsafeAtomicAdd(&sh.est[k], v);
}
// The stored event of tagger t as its lane sees it (its payload goes to sh.slot by thread 0).
template <int D>
__device__ __forceinline__ void lane_slot(Leg<D> &g, int t, Time time, int64_t seq, int valid) {
    if ((int)(threadIdx.x & 63) == t) {
        g.lt = time;
        g.lseq = seq;
        g.lvalid = valid;
    }
}

template <bool RES, int D>
__device__ __noinline__ static void ring_make_call(uint32_t *ring, uint32_t mask, uint64_t from, int steps) {
    ring_make(ring, mask, from, steps);
}
// Collective: every word before `upto` in the ring.  Words made ahead in the exact-inversion
// phase normally cover it, so this is the start of a run and the rare long draw.
template <bool RES, int D, int NT>
__device__ __forceinline__ void ring_ensure(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, uint64_t upto) {
    if (g.produced >= upto) return;
    const int steps = (int)((upto - g.produced + RING_STEP - 1) / RING_STEP);
    if (g.produced + (uint64_t)steps * RING_STEP > g.keep + (uint64_t)q.ring_mask + 1) {   // it would overwrite unread words
        g.err = ECMC_ERR_STATE;
        return;
    }
    __syncthreads();
    if (NT == 64 || wave_index<NT>() == 0)
        ring_make_call<RES, D>(RES ? reinterpret_cast<uint32_t *>(q.dyn + q.o_ring) : a.ring, (uint32_t)q.ring_mask, g.produced, steps);
    g.produced += (uint64_t)steps * RING_STEP;
    __syncthreads();
}

// The earliest stored event (ties: first pushed), uniform: tagger (-1: none), time, push counter.
struct Pick {
    Time t;
    int64_t seq;
    int w;
};
__device__ __forceinline__ bool pick_lt(const Pick &x, const Pick &y) {   // both hold an event
    return (x.t.q < y.t.q) | ((x.t.q == y.t.q) & ((x.t.r < y.t.r) | ((x.t.r == y.t.r) & (x.seq < y.seq))));
}
template <int CTRL>
__device__ __forceinline__ void pick_step(Pick &p) {
    Pick o;
    o.t.q = dpp_move_d<CTRL>(p.t.q);
    o.t.r = dpp_move_d<CTRL>(p.t.r);
    const uint32_t lo = (uint32_t)dpp_move<CTRL>((int)(uint32_t)p.seq), hi = (uint32_t)dpp_move<CTRL>((int)(p.seq >> 32));
    o.seq = (int64_t)(((uint64_t)hi << 32) | lo);
    o.w = dpp_move<CTRL>(p.w);
    const bool take = (o.w >= 0) & ((p.w < 0) | pick_lt(o, p));
    p.t.q = take ? o.t.q : p.t.q;
    p.t.r = take ? o.t.r : p.t.r;
    p.seq = take ? o.seq : p.seq;
    p.w = take ? o.w : p.w;
}
template <int D>
__device__ __forceinline__ Pick pick_stored(const Leg<D> &g) {
    const int lane = threadIdx.x & 63;
    Pick p;
    p.t.q = g.lvalid ? g.lt.q : 0.0;
    p.t.r = g.lvalid ? g.lt.r : 0.0;
    p.seq = g.lvalid ? g.lseq : 0;
    p.w = g.lvalid ? lane : -1;
    pick_step<0xB1>(p);
    pick_step<0x4E>(p);
    pick_step<0x141>(p);
    pick_step<0x140>(p);
    p.t = uni(p.t);
    p.seq = (int64_t)uni((uint64_t)p.seq);
    p.w = uni(p.w);
    return p;
}

// ---- cell occupancy -----------------------------------------------------------------------
// One wavefront: the first index k < count holding unit id in cell c's occupants; -1: none.
template <bool RES, int D>
__device__ __forceinline__ int find_occupant(const ChainArgs &a, const Geo<D> &q, int c, int count, int id) {
    const int lane = threadIdx.x & 63;
#pragma unroll 1
    for (int b = 0; b < count; b += 64) {
        const int k = b + lane;
        const unsigned long long m = __ballot(k < count && occ_get<RES>(a, q, c, k) == id);
        if (m) return b + __ffsll(m) - 1;
    }
    return -1;
}
// One wavefront: the last (any_id) surplus entry of cell c, or the one of unit id in it.
template <bool RES, int D>
__device__ __forceinline__ int find_surplus(const ChainArgs &a, const Geo<D> &q, int count, int c, int id, bool any_id) {
    const int lane = threadIdx.x & 63;
    int best = -1;
#pragma unroll 1
    for (int b = 0; b < count; b += 64) {
        const int i = b + lane;
        const unsigned long long m = __ballot(i < count && sur_cell<RES>(a, q, i) == c && (any_id || sur_id<RES>(a, q, i) == id));
        if (m) best = b + 63 - __clzll((long long)m);
    }
    return best;
}
// One wavefront: moves the surplus entries [from, to) one slot up (by > 0) or down, 64 at a time,
// every chunk read before it is written and the chunks ordered so that no entry is overwritten
// before it was read.
template <bool RES, int D>
__device__ __forceinline__ void shift_surplus(const ChainArgs &a, const Geo<D> &q, int from, int to, int by) {
    const int lane = threadIdx.x & 63;
    const int chunks = (to - from + 63) / 64;
#pragma unroll 1
    for (int k = 0; k < chunks; k++) {
        const int i = by > 0 ? to - 64 * k - 64 + lane : from + 64 * k + lane;
        const bool in = i >= from && i < to;
        int32_t c = 0, id = 0;
        if (in) { c = sur_cell<RES>(a, q, i); id = sur_id<RES>(a, q, i); }
        wave_sync();
        if (in) set_sur<RES>(a, q, i + by, c, id);
        wave_sync();
    }
}

// single_active_cell_occupancy.py:149-203: the unit that stops being active joins its cell's
// occupants, or the surplus when the cell is full (self._surplus.setdefault(cell, []).append(id)
// on the flat list in dict order: after the cell's last surplus entry, or at the end); the new
// active unit leaves the occupants or the surplus (the surplus never moves into the occupants:
// that branch of the reference needs an empty surplus list, which it deletes right away).
// Wavefront 0 edits the lists, the others wait for it (a barrier only where a list changes, which
// also makes the committed position of the old active unit visible).
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ void occupancy_update(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh) {
    const int id = g.active, old_id = g.occ_id, old_cell = g.occ_cell;
    int coord[D];
    const int c = uni(pos_to_cell<D>(q, g.ap, coord));
    if (c >= 0) {
#pragma unroll
        for (int d = 0; d < D; d++) g.cc[d] = uni(coord[d]);
    }
    if (id == old_id) {
        if (c < 0) g.err = ECMC_ERR_STATE;
        else g.occ_cell = c;
        return;
    }
    if (NT == 64 || wave_index<NT>() == 0) {
        const int lane = threadIdx.x & 63;
        int err = c < 0 ? ECMC_ERR_STATE : 0, nsur = g.nsur;
        int n_old = old_id >= 0 ? occ_count<RES>(a, q, old_cell) : 0, n = c >= 0 ? occ_count<RES>(a, q, c) : 0;
        n_old = uni(n_old);
        n = uni(n);
        if (old_id >= 0) {
            if (q.max_occ <= 0 || n_old < q.max_occ) {
                if (n_old >= q.occ_cap) err = ECMC_ERR_STATE;
                else {
                    if (lane == 0) {
                        occ_set<RES>(a, q, old_cell, n_old, old_id);
                        set_occ_count<RES>(a, q, old_cell, n_old + 1);
                        if (FM & FEAT_CELL_BOUNDING) sh.occupied[(old_cell >> 5) & 63] |= 1u << (old_cell & 31);
                    }
                    if (old_cell == c) n++;
                }
            } else if (nsur >= q.n) {
                err = ECMC_ERR_STATE;
            } else {
                const int last = find_surplus<RES>(a, q, nsur, old_cell, 0, true);
                const int at = last >= 0 ? last + 1 : nsur;
                shift_surplus<RES>(a, q, at, nsur, +1);
                if (lane == 0) set_sur<RES>(a, q, at, old_cell, old_id);
                nsur++;
            }
            wave_sync();
        }
        if (!err) {
            const int i = find_occupant<RES>(a, q, c, n, id);
            if (i >= 0) {
#pragma unroll 1
                for (int b = i + 1; b < n; b += 64) {   // every chunk read before it moves down
                    const int k = b + lane;
                    int32_t v = 0;
                    if (k < n) v = occ_get<RES>(a, q, c, k);
                    wave_sync();
                    if (k < n) occ_set<RES>(a, q, c, k - 1, v);
                    wave_sync();
                }
                if (lane == 0) {
                    set_occ_count<RES>(a, q, c, n - 1);
                    if ((FM & FEAT_CELL_BOUNDING) && n == 1) sh.occupied[(c >> 5) & 63] &= ~(1u << (c & 31));
                }
            } else {
                const int k = find_surplus<RES>(a, q, nsur, c, id, false);
                if (k < 0) err = ECMC_ERR_STATE;
                else {
                    shift_surplus<RES>(a, q, k + 1, nsur, -1);
                    nsur--;
                }
            }
            wave_sync();
        }
        g.nsur = nsur;
        if (err) g.err = err;
        if (NT > 64 && lane == 0) {
            sh.occ_err = err;
            sh.occ_nsur = nsur;
        }
    }
    if (NT > 64) {
        __syncthreads();
        if (int e = uni(sh.occ_err)) g.err = e;
        g.nsur = uni(sh.occ_nsur);
    }
    if (g.err) return;
    g.occ_cell = c;
    g.occ_id = id;
}

// The nearby cells of the active cell (cuboid_periodic_cells.py:91-100) and the prefix sums of
// their occupant counts, in the wavefront's own LDS arrays; returns the candidate count.
template <int D, int NT, bool RES>
__device__ __forceinline__ int nearby_cell(const ChainArgs &a, const Geo<D> &q, const Leg<D> &g, int &cnt) {
    const int lane = threadIdx.x & 63;
    int cc = 0;
    cnt = q.nb_cells;
    if (cnt == 0) {
        cnt = uni(a.nearby_n[g.occ_cell]);
        if (lane < cnt) cc = a.nearby[(size_t)g.occ_cell * a.nb_stride + lane];
    } else {
        // at least 2 layers + 1 cells on every axis: no nearby cell repeats
#pragma unroll
        for (int d = 0; d < D; d++) {
            int v = g.cc[d] + q.noff[d];
            v = v < 0 ? v + q.cps[d] : (v >= q.cps[d] ? v - q.cps[d] : v);
            cc += v * q.cum[d];
        }
    }
    return cc;
}
// Every fourth prefix sum stays uniform (group[k]: of cell 4 (k + 1)), so that a candidate's cell
// takes seven comparisons and one LDS access of the four cells left.
struct Counts {
    int nb, far;        // candidates in the nearby and the far cells (-1: not counted yet)
    int group[7];
};
template <int D, int NT, bool RES>
__device__ __forceinline__ void nearby_prefix(const ChainArgs &a, const Geo<D> &q, const Leg<D> &g, ChainShared<NT> &sh, Counts &n) {
    const int lane = threadIdx.x & 63, wave = wave_index<NT>();
    int cnt;
    const int cc = nearby_cell<D, NT, RES>(a, q, g, cnt);
    int num = 0;
    if (lane < cnt) num = occ_count<RES>(a, q, cc);
    const int incl = scan32(num, lane);
    if (lane < 32) {
        sh.nb_cell[wave][lane] = cc;
        sh.nb_pref[wave][lane] = incl - num;
    }
#pragma unroll
    for (int k = 0; k < 7; k++) n.group[k] = __builtin_amdgcn_readlane(incl, 4 * k + 3);
    n.nb = __builtin_amdgcn_readlane(incl, 31);
    wave_sync();
}

// The far cells of the active cell, cell bounding: occupied and not nearby
// (cell_bounding_potential_tagger.py:150-155), as bits per 32 cells with exclusive prefix counts
// in the wavefront's own arrays; far cell c's candidate index is the prefix count of its word
// plus the set bits below it.  One call covers FAR_BLOCK cells from `first` (a larger grid takes
// several, its words built from the counts instead of the kept bits); `before` candidates
// precede them.  Returns the block's candidates.
constexpr int FAR_BLOCK = 2048;
template <int D, int NT, bool RES>
__device__ __forceinline__ int far_prefix(const ChainArgs &a, const Geo<D> &q, const Leg<D> &g, ChainShared<NT> &sh, int first,
                                          int before) {
    const int lane = threadIdx.x & 63, wave = wave_index<NT>();
    uint32_t word = 0;
    const int c0 = first + 32 * lane;
    if (q.ncells <= FAR_BLOCK) word = sh.occupied[lane];
    else {
#pragma unroll 1
        for (int k = 0; k < 32 && c0 + k < q.ncells; k++) word |= occ_count<RES>(a, q, c0 + k) > 0 ? 1u << k : 0u;
    }
    sh.far_word[wave][lane] = word;
    int cnt;
    const int near = nearby_cell<D, NT, RES>(a, q, g, cnt) - first;
    wave_sync();
    if (lane < cnt && near >= 0 && near < FAR_BLOCK) atomicAnd(&sh.far_word[wave][near >> 5], ~(1u << (near & 31)));
    wave_sync();
    const int bits = __popc(sh.far_word[wave][lane]);
    // inclusive sums over the wavefront: within each half by row shifts, then the first half's total
    int incl = bits;
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xF, 0xF, false);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xF, 0xF, false);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xF, 0xF, false);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xF, 0xF, false);
    const int r0 = __builtin_amdgcn_readlane(incl, 15), r1 = __builtin_amdgcn_readlane(incl, 31),
              r2 = __builtin_amdgcn_readlane(incl, 47);
    incl += lane >= 48 ? r0 + r1 + r2 : (lane >= 32 ? r0 + r1 : (lane >= 16 ? r0 : 0));
    sh.far_pref[wave][lane] = (uint32_t)(before + incl - bits);
    wave_sync();
    return __builtin_amdgcn_readlane(incl, 63);
}

// ---- candidates ---------------------------------------------------------------------------
// Number of pair candidates of tagger t (kind: its kind) in this leg; the nearby and far prefixes
// are built once per leg.
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ int candidate_count(const ChainArgs &a, const Geo<D> &q, const Leg<D> &g, ChainShared<NT> &sh, int t,
                                               int kind, Counts &n) {
    if (g.active < 0) return 0;
    if ((FM & FEAT_FMAP) && kind == ECMC_TAG_FACTOR_MAP) return uni(fmap_count(q.tg[t], q.leaves, q.n, g.active));
    if (kind == ECMC_TAG_PAIR_ALL) return q.n - 1;
    if (kind == ECMC_TAG_SURPLUS) return g.nsur;
    if ((FM & FEAT_CELL_BOUNDING) && kind == ECMC_TAG_CELL_BOUNDING) {
        if (n.far < 0) {
            n.far = 0;
            for (int b = 0; b < q.ncells; b += FAR_BLOCK) n.far += far_prefix<D, NT, RES>(a, q, g, sh, b, n.far);
        }
        return n.far;
    }
    if (n.nb < 0) nearby_prefix<D, NT, RES>(a, q, g, sh, n);
    return n.nb;
}

// Enumeration of one tagger's candidates: `span` indices (in blocks of FAR_BLOCK for the far
// cells of a large grid), index idx -> candidate j, unit, far cell; false where the index holds none.
template <int D, int FM, int NT, bool RES>
struct Candidates {
    const ChainArgs &a;
    const Geo<D> &q;
    ChainShared<NT> &sh;
    const ecmc_tagger_desc &tg;
    const Counts &n;
    int kind, act, wave, M, m, k, fn, first;
    __device__ __forceinline__ Candidates(const ChainArgs &a_, const Geo<D> &q_, ChainShared<NT> &s_, int t, int kind_, int act_, int M_,
                                          const Counts &n_)
        : a(a_), q(q_), sh(s_), tg(q_.tg[t]), n(n_), kind(kind_), act(act_), wave(wave_index<NT>()), M(M_), m(0), k(0), fn(1), first(0) {
        if ((FM & FEAT_FMAP) && kind == ECMC_TAG_FACTOR_MAP) {
            m = act / q.leaves;
            k = act % q.leaves;
            fn = uni(tg.fmap_n[k]);
        }
    }
    __device__ __forceinline__ bool far() const { return (FM & FEAT_CELL_BOUNDING) && kind == ECMC_TAG_CELL_BOUNDING; }
    __device__ __forceinline__ int span() const { return far() ? min(q.ncells - first, FAR_BLOCK) : M; }
    // U indices at once, so that their loads overlap (one branch on the kind for all of them).
    template <int U>
    __device__ __forceinline__ void get(const int (&idx)[U], int (&j)[U], int (&target)[U], int (&cell)[U], bool (&live)[U]) const {
#pragma unroll
        for (int u = 0; u < U; u++) {
            j[u] = idx[u];
            cell[u] = 0;
            live[u] = true;
        }
        if (far()) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t w = sh.far_word[wave][idx[u] >> 5], bit = 1u << (idx[u] & 31);
                j[u] = (int)sh.far_pref[wave][idx[u] >> 5] + __popc(w & (bit - 1u));
                cell[u] = first + idx[u];
                live[u] = (w & bit) != 0;
            }
            int zero[U];
#pragma unroll
            for (int u = 0; u < U; u++) zero[u] = 0;
            occ_get_all<RES, U>(a, q, cell, zero, target);
#pragma unroll
            for (int u = 0; u < U; u++) target[u] = live[u] ? target[u] : act;
        } else if ((FM & FEAT_FMAP) && kind == ECMC_TAG_FACTOR_MAP) {
#pragma unroll
            for (int u = 0; u < U; u++) target[u] = fmap_target(tg, q.leaves, m, k, fn, idx[u]);
        } else if (kind == ECMC_TAG_PAIR_ALL) {
#pragma unroll
            for (int u = 0; u < U; u++) target[u] = idx[u] < act ? idx[u] : idx[u] + 1;
        } else if (kind == ECMC_TAG_SURPLUS) {
#pragma unroll
            for (int u = 0; u < U; u++) target[u] = sur_id<RES>(a, q, idx[u]);
        } else {
            // the nearby cell holding candidate idx: the largest c with pref[c] <= idx (empty cells
            // repeat a prefix, and so do the places after the last cell)
            int4 p[U], c[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                int k4 = 0;
#pragma unroll
                for (int i = 0; i < 7; i++) k4 += n.group[i] <= idx[u] ? 1 : 0;
                p[u] = *reinterpret_cast<const int4 *>(&sh.nb_pref[wave][4 * k4]);
                c[u] = *reinterpret_cast<const int4 *>(&sh.nb_cell[wave][4 * k4]);
            }
            int in[U], place[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const bool b1 = p[u].y <= idx[u], b2 = p[u].z <= idx[u], b3 = p[u].w <= idx[u];
                place[u] = idx[u] - (b3 ? p[u].w : (b2 ? p[u].z : (b1 ? p[u].y : p[u].x)));
                in[u] = b3 ? c[u].w : (b2 ? c[u].z : (b1 ? c[u].y : c[u].x));
            }
            occ_get_all<RES, U>(a, q, in, place, target);
        }
    }
    __device__ __forceinline__ bool get(int idx, int &j, int &target, int &cell) const {
        int ii[1] = {idx}, jj[1], tt[1], cc[1];
        bool ll[1];
        get<1>(ii, jj, tt, cc, ll);
        j = jj[0];
        target = tt[0];
        cell = cc[0];
        return ll[0];
    }
};

// True only if candidate (tagger plan pl) surely has no event within a displacement hf of the
// active unit (hf carries the margins below).  A rise by the drawn dU >= dU_lo needs a
// potential difference that the path [0, hf] offers: at separations of at least r = sqrt(r2)
// (r2 a lower bound over the path) an inverse power K / r^p rises by less than K / r^p in all
// and by less than p K / r^(p+1) per unit of displacement, the Coulomb bound K / r by less
// than K / r^2 per unit, and a cell bound by its rate.  A repulsive factor has no event behind the
// active unit, an attractive one none before its closest approach, a truncated one none before
// the cutoff sphere.  FP32 rounding (a few 2^-24 per operation, at most 20 of them) lies far
// inside the 2^-15 margins; hf is the horizon widened by 2^-16 relative and 2^-18 L, which covers
// the rounding of the exact inversion (a root near the closest approach is off by up to
// 2^-26 of the separation).  perp2: squared perpendicular separation, from below; sd: the component
// along the motion to 2^-23 L, which the slacks cover; behind: surely negative; edge: the sign of sd
// is not certain (at +-L / 2).
__device__ __forceinline__ bool quick_cull(int test, int p, float rc2_hi, float pp, float perp2, float sd, bool behind, bool edge,
                                           float hf, float L, float dU_lo) {
    const float K = fabsf(pp);
    const bool sure = (K >= 0x1p-100f) & (K <= 0x1p100f) & !edge;
    bool none;
    if (test == QT_INVERSE_POWER) {
        const float slack = (fabsf(sd) + hf) * 0x1p-17f + L * 0x1p-20f;
        const float e = fmaxf(fmaxf(sd - hf, -sd) - slack, 0.f);
        const float r2 = (perp2 + e * e) * (1.f - 0x1p-16f);
        none = pp > 0.f ? behind : sd - slack > hf;
        none = none | (r2 >= rc2_hi);
        // r^p for 1 <= p <= 32 by binary powering of r2 (p uniform: at most nine products)
        const float r = __builtin_amdgcn_sqrtf(r2), r4 = r2 * r2, r8 = r4 * r4, r16 = r8 * r8;
        float rp = (p & 1) ? r : 1.f;
        rp = (p & 2) ? rp * r2 : rp;
        rp = (p & 4) ? rp * r4 : rp;
        rp = (p & 8) ? rp * r8 : rp;
        rp = (p & 16) ? rp * r16 : rp;
        rp = (p & 32) ? rp * (r16 * r16) : rp;
        const float A = dU_lo * rp * (1.f - 0x1p-15f);
        none = none | (A > K) | (A * r * (1.f - 0x1p-20f) > (float)p * K * hf);
    } else {
        // the Coulomb bound runs over the periodic images along the motion: within a quarter box the
        // nearest image passed lies at |x| >= min(e, L / 4)
        const bool near = hf <= 0.25f * L;
        const float slack = (fabsf(sd) + L) * 0x1p-16f;
        const float e = near ? fminf(fmaxf(fmaxf(sd - hf, -sd) - slack, 0.f), 0.25f * L) : 0.f;
        const float r2 = (perp2 + e * e) * (1.f - 0x1p-16f);
        none = near & (pp > 0.f ? (sd < -slack) & (sd - hf > -0.5f * L + slack) : sd - hf > slack);
        none = none | (dU_lo * r2 * (1.f - 0x1p-15f) > K * hf);
    }
    return none & sure;
}

// dU_lower (ecmc_fp32_bounds.h) without its branch: u24 below 2^-10, else the hardware logarithm
// that log2f is for its normal argument, less its error bound.
__device__ __forceinline__ float draw_lower(uint32_t a, float inv_beta_lo) {
    const float u24 = (float)(a >> 8) * 0x1p-24f;
    const float ml2 = -__builtin_amdgcn_logf(1.f - u24);
    const float l = (ml2 - LOG2F_ERR * fmaxf(ml2, 1.f)) * 0x1.62e42ep-1f;
    return fmaxf((u24 < 0x1p-10f ? u24 : l) * inv_beta_lo * (1.f - 0x1p-20f), 0.f);
}

// Pass 1 of a leg: every candidate of the items tested against the horizon h (time); the
// contenders go to the wavefront's queue.  Returns their number, QCAP + 1 when they did not fit.
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ int gather_contenders(const ChainArgs &a, const Geo<D> &q, const Leg<D> &g, ChainShared<NT> &sh,
                                                 const Items &its, double h, Counts cn) {
    constexpr int U = 2;   // candidates per lane and iteration: their loads overlap
    const int lane = threadIdx.x & 63, wave = wave_index<NT>();
    const float Lf = (float)q.L;
    const float hf = (float)(h * g.aspeed) * (1.f + 0x1p-16f) + Lf * 0x1p-18f;
    const float ibf = q.inv_beta;
    const float inv_L = __builtin_amdgcn_rcpf(Lf);
    const int act = g.active, dir = g.adir;
    const float caf = (FM & FEAT_EWALD) && q.charged ? (float)charge_of<RES>(a, q, act) : 1.f;
    float cell_rate_max = 0.f;
    if (FM & FEAT_CELL_BOUNDING) cell_rate_max = pick_axis<3>(q.cb_max, dir);
    int qn = 0;
#pragma unroll 1
    for (int g0 = 0, g1; g0 < its.count; g0 = g1) {
        const int t0 = item_tag(its, g0), key = __builtin_amdgcn_readlane(its.set_key, g0);
        bool geo = false;
#pragma unroll 1
        for (g1 = g0; g1 < its.count; g1++) {
            const int t = item_tag(its, g1), test = (q.tests >> (2 * t)) & 3;
            if (g1 > g0 && __builtin_amdgcn_readlane(its.set_key, g1) != key) break;
            geo = geo || test == QT_INVERSE_POWER || test == QT_COULOMB_BOUND;
        }
        const int kind = kind_of(q.kinds, t0);
        Candidates<D, FM, NT, RES> cs(a, q, sh, t0, kind, act, candidate_count<D, FM, NT, RES>(a, q, g, sh, t0, kind, cn), cn);
        if (cs.M == 0) continue;
        int before = 0;
        for (;; cs.first += FAR_BLOCK) {   // one pass but for far cells of a large grid
            if (cs.far() && q.ncells > FAR_BLOCK) before += far_prefix<D, NT, RES>(a, q, g, sh, cs.first, before);
            const int span = cs.span();
#pragma unroll 1
            for (int base = wave * 64; base < span; base += U * NT) {
                int j[U], target[U], cell[U];
                bool live[U], edge[U], behind[U];
                float perp2[U], sd[U];
                int idx[U];
#pragma unroll
                for (int u = 0; u < U; u++) idx[u] = min(base + u * NT + lane, span - 1);
                cs.template get<U>(idx, j, target, cell, live);
#pragma unroll
                for (int u = 0; u < U; u++) {
                    live[u] = live[u] & (base + u * NT + lane < span);
                    edge[u] = behind[u] = false;
                    perp2[u] = sd[u] = 0.f;
                }
                if (geo) {
                    double tp[U][D];
#pragma unroll
                    for (int u = 0; u < U; u++) load_pos<RES>(a, q, target[u], tp[u]);
                    // minimum image in FP32: within 2^-23 L of the exact separation (the difference's
                    // conversion, the product with L), except within that of +-L / 2
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        float f[D], lo[D];
#pragma unroll
                        for (int d = 0; d < D; d++) {
                            const float v = (float)(tp[u][d] - g.ap[d]);
                            f[d] = fmaf(-Lf, rintf(v * inv_L), v);
                            lo[d] = fmaxf(fabsf(f[d]) - Lf * 0x1p-21f, 0.f);
                        }
                        sd[u] = pick_axis<D>(f, dir);
                        const float p = dir == 0 ? lo[1] : lo[0], p2 = D > 2 ? (dir == 2 ? lo[1] : lo[D - 1]) : 0.f;
                        perp2[u] = fmaf(p, p, p2 * p2);
                        edge[u] = !(fabsf(sd[u]) < (0.5f - 0x1p-20f) * Lf);
                        behind[u] = sd[u] < -0x1p-20f * Lf;
                    }
                }
#pragma unroll 1
                for (int i = g0; i < g1; i++) {
                    const int tag = item_tag(its, i);
                    const uint32_t word = item_word(its, i);
                    const int rank = item_rank(its, i);
                    const int test = (q.tests >> (2 * tag)) & 3;
                    bool keep[U];
#pragma unroll
                    for (int u = 0; u < U; u++) keep[u] = live[u];
                    if (test != QT_DIRECT) {
                        const int p = __builtin_amdgcn_readlane(its.p, i);
                        const float rc2_hi = item_f(its.rc2_hi, i);
                        float pref = item_f(its.pref, i);
                        if ((FM & FEAT_CELL_BOUNDING) && test == QT_CELL) pref = cell_rate_max;
                        float dU_lo[U], pp[U];
#pragma unroll
                        for (int u = 0; u < U; u++) {
                            dU_lo[u] = draw_lower(ring_word<RES>(a, q, (uint32_t)g.keep + word + 2u * (uint32_t)j[u]), ibf);
                            pp[u] = pref;
                        }
                        if ((q.charged >> tag) & 1u) {
                            // any pair potential may take the charges; variants without the Coulomb
                            // machinery hold no register for the active unit's
                            const float ca = FM & FEAT_EWALD ? caf : (float)charge_of<RES>(a, q, act);
#pragma unroll
                            for (int u = 0; u < U; u++) pp[u] *= ca * (float)charge_of<RES>(a, q, target[u]);
                        }
#pragma unroll
                        for (int u = 0; u < U; u++) {
                            // (a cell bound's prefactor is its largest rate per unit charge factor)
                            const bool cull = (FM & FEAT_CELL_BOUNDING) && test == QT_CELL
                                                  ? dU_lo[u] * (1.f - 0x1p-15f) > fabsf(pp[u]) * hf
                                                  : quick_cull(test, p, rc2_hi, pp[u], perp2[u], sd[u], behind[u], edge[u], hf, Lf, dU_lo[u]);
                            keep[u] = keep[u] & !cull;
                        }
                    }
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const unsigned long long m = __ballot(keep[u]);
                        const int cnt = __popcll(m);
                        if (qn + cnt > QCAP) {
                            qn = QCAP + 1;
                        } else if (cnt) {
                            if (keep[u]) {
                                Contender &c = sh.queue[wave][qn + __popcll(m & ((1ull << lane) - 1ull))];
                                c.word = word + 2u * (uint32_t)j[u];
                                c.rank = rank + j[u];
                                c.target = target[u];
                                c.tag_cell = tag | (cell[u] << 4);
                            }
                            qn += cnt;
                        }
                    }
                }
            }
            if (!cs.far() || cs.first + FAR_BLOCK >= q.ncells) break;
        }
    }
    return qn;
}

// Exact time displacement of a candidate (its tagger's event handler's send_event_time).
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ double candidate_dt(const ChainArgs &a, const Geo<D> &q, const Leg<D> &g, ChainShared<NT> &sh, int tag,
                                               uint32_t word, int target, int cell) {
    const ecmc_tagger_desc &tg = q.tg[tag];
    double tp[D], s[D];
    load_pos<RES>(a, q, target, tp);
    separation_vector<D>(q, g.ap, tp, s);
    uint32_t w0 = 0, w1 = 0;
    double beta = 0.0;
    if ((q.draws >> tag) & 1u) {
        w0 = ring_word<RES>(a, q, (uint32_t)g.keep + word);
        w1 = ring_word<RES>(a, q, (uint32_t)g.keep + word + 1u);
        beta = q.beta;
    }
    double ca = 1.0, ct = 1.0;
    if ((q.charged >> tag) & 1u) {
        ca = charge_of<RES>(a, q, g.active);
        ct = charge_of<RES>(a, q, target);
    }
    const int eh = tg.event_handler;
    int how = tg.potential;
    double p0 = tg.par[0], p1 = tg.par[1], p2 = tg.par[2], x = sh.plan[tag].powrc, y = 0.0;
    if (POT_BUILT(ECMC_POT_LENNARD_JONES) && how == ECMC_POT_LENNARD_JONES) {
        p2 = sh.plan[tag].r0;
        x = sh.plan[tag].k6;
        y = sh.plan[tag].k12;
    }
    if ((FM & FEAT_COULOMB) && eh == ECMC_EH_TWO_LEAF_BOUNDING) {
        how = TIME_COULOMB_BOUND;
        p0 = tg.bpar[0];
        x = q.L;
    }
    if ((FM & FEAT_CELL_BOUNDING) && eh == ECMC_EH_CELL_BOUNDING) {
        how = TIME_RATE;
        p0 = cell_rate_of_cells<D>(a, q, tg, g.occ_cell, cell, g.adir, ca, ct);
    }
    return pair_time<D, FM>(how, p0, p1, p2, x, y, g.adir, g.aspeed, s[0], s[1], s[D - 1], ca, ct, w0, w1, beta);
}

// Keeps the earlier of two candidates by (time, push rank).
__device__ __forceinline__ bool winner_lt(const Winner &x, const Winner &y) {
    return (x.t.q < y.t.q) | ((x.t.q == y.t.q) & ((x.t.r < y.t.r) | ((x.t.r == y.t.r) & (x.rank < y.rank))));
}
__device__ __forceinline__ Winner no_winner() {
    Winner w;
    w.t.q = w.t.r = INFINITY;
    w.dt = INFINITY;
    w.rank = NO_RANK;
    w.tag = 0;
    w.target = -1;
    w.bad = 0;
    return w;
}
// The earliest candidate over the wavefront, uniform.  The time (q, r) is monotone in the
// displacement dt, so the least dt has the least time; lanes of equal time are told apart by
// push rank.
__device__ __forceinline__ Winner wave_winner(const Winner &m) {
    Winner w = no_winner();
    if (__ballot(m.bad)) w.bad = -wave_min(-m.bad);
    const double dmin = wave_min(m.rank == NO_RANK ? INFINITY : m.dt);
    unsigned long long eq = __ballot(m.rank != NO_RANK && m.dt == dmin);
    if (!eq) return w;
    const int l0 = __ffsll(eq) - 1;
    w.t.q = lane_d(m.t.q, l0);
    w.t.r = lane_d(m.t.r, l0);
    eq = __ballot(m.rank != NO_RANK && m.t.q == w.t.q && m.t.r == w.t.r);
    int l = l0;
    if (eq & (eq - 1)) {
        const int smin = wave_min(((eq >> (threadIdx.x & 63)) & 1ull) ? m.rank : NO_RANK);
        l = __ffsll(__ballot(m.rank == smin)) - 1;
    }
    w.dt = dmin;
    w.rank = __builtin_amdgcn_readlane(m.rank, l);
    w.tag = __builtin_amdgcn_readlane(m.tag, l);
    w.target = __builtin_amdgcn_readlane(m.target, l);
    return w;
}

// Sum of the hash terms of tagger t's M candidates, over the workgroup (logged runs); `before`
// candidates of the leg precede them.
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ uint32_t candidate_hash(const ChainArgs &a, const Geo<D> &q, const Leg<D> &g, ChainShared<NT> &sh, int t,
                                                   int kind, int M, const Counts &cn, int joff) {
    const int lane = threadIdx.x & 63, wave = wave_index<NT>();
    uint32_t h = 0;
    Candidates<D, FM, NT, RES> cs(a, q, sh, t, kind, g.active, M, cn);
    int before = 0;
#pragma unroll 1
    for (;; cs.first += FAR_BLOCK) {
        if (cs.far() && q.ncells > FAR_BLOCK) before += far_prefix<D, NT, RES>(a, q, g, sh, cs.first, before);
        const int span = M ? cs.span() : 0;
#pragma unroll 1
        for (int idx = threadIdx.x; idx < span; idx += NT) {
            int j, target, cell;
            if (cs.get(idx, j, target, cell)) h += cand_mix((uint32_t)(joff + j), (uint32_t)target);
        }
        if (!cs.far() || cs.first + FAR_BLOCK >= q.ncells) break;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o, 64);
    if (NT > 64) {
        if (lane == 0) sh.hash[wave] = h;
        __syncthreads();
        h = 0;
        for (int w = 0; w < ChainShared<NT>::NW; w++) h += sh.hash[w];
        __syncthreads();
    }
    return (uint32_t)uni((int)h);
}

// ---- creates of the other taggers ---------------------------------------------------------
// A cell-boundary event, from the active unit's present state.
struct Boundary {
    Pick p;           // p.w < 0: none
    double x;         // the boundary reached
};
// cell_boundary_event_handler.py:98-156
template <int D, int NT>
__device__ __forceinline__ void create_boundary(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, int t, Boundary &b) {
    const int dir = g.adir;
    int coord[D];
    const int cell = g.occ_id == g.active ? g.occ_cell : uni(pos_to_cell<D>(q, g.ap, coord));
    if (cell < 0) { g.err = ECMC_ERR_STATE; return; }
    const int cps = pick_axis<D>(q.cps, dir), cum = pick_axis<D>(q.cum, dir);
    const int id = g.occ_id == g.active ? pick_axis<D>(g.cc, dir) : uni(pick_axis<D>(coord, dir));
    const int nid = id + 1 == cps ? 0 : id + 1;
    const double boundary = cps <= AXIS_CELLS ? sh.axis[dir][nid] : a.cmin[(size_t)(cell + (nid - id) * cum) * D + dir];
    double sep = boundary - pick_axis<D>(g.ap, dir);
    sep = sep < 0.0 ? sep + q.L : sep;
    b.p.t = time_add_u(g.at, ub(g.aspeed == 1.0) ? sep : sep / g.aspeed);
    b.p.seq = g.seq++;
    b.p.w = t;
    b.x = boundary;
}
template <int D, int NT>
__device__ __forceinline__ void store_boundary(Leg<D> &g, ChainShared<NT> &sh, const Boundary &b) {
    if (threadIdx.x == 0) {
        Slot &sl = sh.slot[b.p.w];
#pragma unroll
        for (int d = 0; d < D; d++) sl.apos[d] = g.ap[d];
        sl.astamp = g.at;
        sl.cb_boundary = b.x;
        sl.cb_dir = g.adir;
        sl.adir = g.adir;
        sl.aspeed = g.aspeed;
    }
    lane_slot(g, b.p.w, b.p.t, b.p.seq, 1);
}

// The end of chain: chain time and the randint of the next active unit
// (single_independent_active_periodic_direction_end_of_chain_event_handler.py:176-237): with
// composite objects the root's randint, then the leaf's.
template <int D, int NT, bool RES>
__device__ __forceinline__ void create_end_of_chain(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, int t) {
    const double value = q.tg[t].value;
    const double since = time_sub(g.at, g.eoc_last);
    if (ub(!(0.0 <= since && since <= value))) { g.err = ECMC_ERR_CONFIGURATION; return; }
    const double chain = time_sub(g.eoc_last, g.at) + value;
    const Time time = time_add_u(g.at, chain);
    const int P = q.leaves;
    int root = 0, v = 0;
#pragma unroll 1
    for (int phase = 0; phase < (P > 1 ? 2 : 1); phase++) {
        const uint32_t nrange = phase == 0 ? (uint32_t)(q.n / P) : (uint32_t)P;
        const int k = 32 - __clz((int)nrange);   // bit length
        // randint's rejection loop: each word is accepted with probability >= 1/2, so 40 000
        // words without success only happen after a defect
        int tries = 0;
#pragma unroll 1
        for (;; tries++) {
            ring_ensure<RES, D, NT>(a, q, g, g.cursor + 1);
            if (tries > 40000) g.err = ECMC_ERR_STATE;
            if (g.err) return;
            const uint32_t x = (uint32_t)uni((int)ring_word<RES>(a, q, (uint32_t)g.cursor)) >> (32 - k);
            g.cursor++;
            if (x < nrange) { v = (int)x; break; }
        }
        if (phase == 0) root = v;
    }
    if (threadIdx.x == 0) sh.slot[t].target = P > 1 ? root * P + v : v;
    lane_slot(g, t, time, g.seq++, 1);
}

// cell veto send_event_time (cell_veto_event_handler.py:190-238): the Walker table by the sign
// of the charge correction factor; random.choice over its entries (rejection on bit_length
// words), uniform(0, mean) for item or alias, then expovariate / (total rate * speed).
template <int D, int NT, bool RES>
__device__ __forceinline__ void create_cell_veto(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, int t) {
    const ecmc_tagger_desc &tg = q.tg[t];
    const int dir = g.adir;
    double cf = (((q.charged >> t) & 1u) ? charge_of<RES>(a, q, g.active) : 1.0) * 1.0 / tg.bpar[2];
    const int b = ub(!(cf > 0.0)) ? 1 : 0;
    if (b) cf *= -1.0;
    const int wt = dir * 2 + b;
    const uint32_t m = (uint32_t)a.cv_m;
    const int k = 32 - __clz((int)m);
    uint32_t entry = 0;
#pragma unroll 1
    for (int tries = 0;; tries++) {
        ring_ensure<RES, D, NT>(a, q, g, g.cursor + 5);
        if (tries > 40000) g.err = ECMC_ERR_STATE;
        if (g.err) return;
        entry = (uint32_t)uni((int)ring_word<RES>(a, q, (uint32_t)g.cursor)) >> (32 - k);
        g.cursor++;
        if (entry < m) break;
    }
    const uint32_t w0 = (uint32_t)g.cursor;
    const CvEntry e = a.cvw[(size_t)wt * m + entry];
    const double dU = drawn_change(ring_word<RES>(a, q, w0 + 2), ring_word<RES>(a, q, w0 + 3), a.beta);
    const double u = 0.0 + (a.cv_mean[wt] - 0.0) * words_to_random(ring_word<RES>(a, q, w0), ring_word<RES>(a, q, w0 + 1));
    const int item = u <= e.rate0 ? e.item0 : e.item1;
    const int rel = uni(item);
    g.cursor += 4;
    const double total = a.cv_total[wt] * cf;
    if (rel < 0) { g.err = ECMC_ERR_NUMERIC; return; }
    const double row = a.cbt[(size_t)(rel * 3 + dir) * 2 + b];
    const double rate = (b ? -row : row) * cf;
    if (ub(!(rate > 0.0))) { g.err = ECMC_ERR_NUMERIC; return; }
    // cuboid_periodic_cells.py:182-207: the cell centre shifted by the relative cell's lower
    // corner lies half a cell from every wall, so the per-axis identifier sum is that cell
    int tcell = 0;
#pragma unroll
    for (int d = 0; d < D; d++) {
        const int i = g.cc[d] + (rel / q.cum[d]) % q.cps[d];
        tcell += (i >= q.cps[d] ? i - q.cps[d] : i) * q.cum[d];
    }
    const double dt = dU / (total * g.aspeed);
    const Time time = time_add_u(g.at, dt);
    double ap[D];
#pragma unroll
    for (int d = 0; d < D; d++) ap[d] = g.ap[d];
    if (ub(!isinf(time.q))) slice_pos<D>(q, ap, dir, g.aspeed, g.at, time);
    if (threadIdx.x == 0) {
        Slot &sl = sh.slot[t];
        sl.target = -1;
        sl.cb_cell = tcell;
        sl.cv_rate = rate;
        sl.adir = dir;
        sl.aspeed = g.aspeed;
#pragma unroll
        for (int d = 0; d < D; d++) sl.apos[d] = ap[d];
        sl.astamp = time;
    }
    lane_slot(g, t, time, g.seq++, 1);
}

// Creates of one tagger other than the pair and cell-boundary taggers (collective for the words).
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ void create_single(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, int t, int kind) {
    const ecmc_tagger_desc &tg = q.tg[t];
    Time time = {0.0, 0.0};
    if (kind == ECMC_TAG_END_OF_CHAIN || kind == ECMC_TAG_CELL_VETO) {
        lane_slot(g, t, time, 0, 0);
        if (kind == ECMC_TAG_END_OF_CHAIN) create_end_of_chain<D, NT, RES>(a, q, g, sh, t);
        else if ((FM & FEAT_CELL_VETO) && g.active >= 0) create_cell_veto<D, NT, RES>(a, q, g, sh, t);
        return;
    }
    if (kind == ECMC_TAG_SAMPLING) {
        g.samp_time = time_add(g.samp_time, tg.value);
        time = g.samp_time;
    } else if (kind == ECMC_TAG_END_OF_RUN) {
        time = time_from_float(tg.value);
    } else if (kind != ECMC_TAG_START_OF_RUN) {
        return;
    }
    lane_slot(g, t, time, g.seq++, 1);
}

// The earliest candidate w of tagger t's M candidates as its stored event.
template <int D, int NT, bool RES>
__device__ __forceinline__ void store_winner(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, int t, int M,
                                             int64_t seq0, const Winner &w) {
    if (M == 0) {
        lane_slot(g, t, Time{0.0, 0.0}, 0, 0);
        return;
    }
    // an error counts if no event of its set comes before it (legs with a quick test see no more of
    // them); a set without a quick test is evaluated whole in every leg, and any counts
    if (w.bad && (((q.tests >> (2 * t)) & 3) == QT_DIRECT || ub((double)error_time(w.bad) <= w.dt))) {
        g.err = ECMC_ERR_NUMERIC;
        return;
    }
    double tp[D], p[D];
    load_pos<RES>(a, q, w.target, tp);
#pragma unroll
    for (int d = 0; d < D; d++) p[d] = g.ap[d];
    if (ub(!isinf(w.t.q))) slice_pos<D>(q, p, g.adir, g.aspeed, g.at, w.t);
    if (threadIdx.x == 0) {
        Slot &sl = sh.slot[t];
        sl.cb_cell = g.occ_cell;
        sl.target = w.target;
        sl.adir = g.adir;
        sl.aspeed = g.aspeed;
#pragma unroll
        for (int d = 0; d < D; d++) {
            sl.apos[d] = p[d];
            sl.tpos[d] = tp[d];
        }
        sl.astamp = w.t;
    }
    lane_slot(g, t, w.t, seq0 + w.rank, 1);
}

// ewald_derivative over one wavefront, all 64 lanes calling with the same separation.  The
// host lists the terms of the sequential loop (the real-space images by k, j, i, then the
// Fourier terms by i, j, k); term g belongs to lane g % 64, slot g / 64.  Each lane evaluates
// its terms with the sequential loop's operations (a Fourier factor by stepping the same
// cos/sin recurrence from its start as far as that term), adds its slots in order, and a
// butterfly over the lanes adds the 64 partial sums (commutative pairings, so every lane ends
// with the same sum).  The order of the additions differs from the sequential loop's, so the
// result agrees with it to rounding.  More than 256 terms fall back to the sequential function.
// The sequential form where the wave form does not apply: called, not inlined (a rare path).
__device__ __noinline__ static double ewald_derivative_call(const Ewald &e, double sx, double sy, double sz) {
    return ewald_derivative(e, sx, sy, sz);
}
__device__ __noinline__ static double ewald_derivative_wave(const Ewald &e, const int32_t *codes, int ncodes, double sx, double sy,
                                        double sz) {
    if (ncodes > 256 || !codes) return ewald_derivative_call(e, sx, sy, sz);
    const int lane = threadIdx.x & 63;
    const int n = e.fc + 1;
    const double L = e.L;
    int code[4];
#pragma unroll
    for (int s = 0; s < 4; s++) code[s] = lane + 64 * s < ncodes ? codes[lane + 64 * s] : -1;
    // cos and sin of tpol s_d on lane d (the same functions per component), broadcast
    double cd, sd;
    sincos(e.tpol * (lane == 0 ? sx : (lane == 1 ? sy : sz)), &sd, &cd);
    const double dcx = __shfl(cd, 0, 64), dsx = __shfl(sd, 0, 64);
    const double dcy = __shfl(cd, 1, 64), dsy = __shfl(sd, 1, 64);
    const double dcz = __shfl(cd, 2, 64), dsz = __shfl(sd, 2, 64);
    double sum = 0.0;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        double v = 0.0;
        const int c = code[s];
        if (c >= 0) {
            const int i = ((c >> 16) & 255) - 128, j = ((c >> 8) & 255) - 128, k = (c & 255) - 128;
            if (c >> 24) {
                double tmp, cxv = dcx, sxv = dsx, cyv = 1.0, syv = 0.0, czv = 1.0, szv = 0.0;
                for (int r = 1; r < i; r++) { tmp = cxv; cxv = tmp * dcx - sxv * dsx; sxv = sxv * dcx + tmp * dsx; }
                for (int r = 0; r < j; r++) { tmp = cyv; cyv = tmp * dcy - syv * dsy; syv = syv * dcy + tmp * dsy; }
                for (int r = 0; r < k; r++) { tmp = czv; czv = tmp * dcz - szv * dsz; szv = szv * dcz + tmp * dsz; }
                v = e.f[(i * n + j) * n + k] * sxv * cyv * czv;
            } else {
                const double vz2 = (sz + k * L) * (sz + k * L);
                const double vy2 = (sy + j * L) * (sy + j * L);
                const double vx = sx + i * L;
                const double v2 = vx * vx + vy2 + vz2;
                const double vn = sqrt(v2);
                v = vx * (e.two_aol_rpi * exp(-e.aol2 * v2) + erfc(e.aol * vn) / vn) / v2;
            }
        }
        sum += v;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    return sum;
}

// The same derivative in FP32 with a bound on its error, for the thinning of an event: the factor's
// real rate is compared with a draw, and about one comparison in 10^4 is closer than the bound (the
// FP64 sum above then decides).  Lane terms: one real-space image (creal) and two Fourier terms (cf0,
// cf1; -1: none).  Separations are reduced in FP64, then per term
//   real     exp by the hardware's exp2, erfc = exp erfcx (a polynomial of (1 + 2x) erfcx in
//            (x - 2.5) / (x + 2.5), 2.2e-7 off with its roundings), relative error below
//            2^-19 + 2^-20 z for the exponent z = a^2 v^2 (z's own relative error is 8 x 2^-24);
//   Fourier  sines of fractions of a period by the 2e-9 polynomial 4.3.97 of Abramowitz and Stegun,
//            each within 4e-7, a product of three within 2^-19;
// and the sum over the lanes adds 9 roundings of partial sums: 2^-18 + 2^-20 z of a real term and
// 2^-18 |f| of a Fourier term bound it, terms that underflow are 1e-38 of it.  The commit of a charged
// leg took 11 700 cycles with the FP64 sum (an exp, an erfc and two divisions in one chain, three
// rounds of terms) and takes 6300.
__device__ __forceinline__ float sin_turn(float f) {   // sin(2 pi f) for |f| <= 1/4
    const float y = f * 6.2831853f, y2 = y * y;
    return y * fmaf(y2, fmaf(y2, fmaf(y2, fmaf(y2, fmaf(y2, -2.39e-8f, 2.7526e-6f), -1.98409e-4f), 8.3333315e-3f), -0.1666666664f), 1.f);
}
__device__ __forceinline__ float wave_total(float v) {   // the sum over the lanes, by DPP
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xF, 0xF, true));
    const int l = __float_as_int(v);
    return (__int_as_float(__builtin_amdgcn_readlane(l, 15)) + __int_as_float(__builtin_amdgcn_readlane(l, 31))) +
           (__int_as_float(__builtin_amdgcn_readlane(l, 47)) + __int_as_float(__builtin_amdgcn_readlane(l, 63)));
}
struct EwaldBound {
    float value, error;
};
__device__ __noinline__ static EwaldBound ewald_derivative_fp32(double sx, double sy, double sz, double L, double inv_l, float aol,
                                                                float aol2, float two_aol_rpi, int creal, int cf0, int cf1, float f0,
                                                                float f1) {
    const double px = sx * inv_l, py = sy * inv_l, pz = sz * inv_l;
    auto fourier = [&](int c, float f) {
        const double i = (double)(((c >> 16) & 255) - 128), j = (double)(((c >> 8) & 255) - 128), k = (double)((c & 255) - 128);
        const double ti = i * px, tj = j * py, tk = k * pz;
        const float a = (float)(ti - rint(ti)), b = fabsf((float)(tj - rint(tj))), d = fabsf((float)(tk - rint(tk)));
        const float af = fabsf(a);
        return f * copysignf(sin_turn(af > 0.25f ? 0.5f - af : af), a) * sin_turn(0.25f - b) * sin_turn(0.25f - d);
    };
    float sum = 0.f, err = 0.f;
    if (cf0 >= 0) {
        sum += fourier(cf0, f0);
        err += fabsf(f0) * 0x1p-18f;
    }
    if (cf1 >= 0) {
        sum += fourier(cf1, f1);
        err += fabsf(f1) * 0x1p-18f;
    }
    if (creal >= 0) {
        const float vx = (float)fma((double)(((creal >> 16) & 255) - 128), L, sx), vy = (float)fma((double)(((creal >> 8) & 255) - 128), L, sy),
                    vz = (float)fma((double)((creal & 255) - 128), L, sz);
        const float v2 = fmaf(vx, vx, fmaf(vy, vy, vz * vz)), rv = __builtin_amdgcn_rsqf(v2), x = aol * (v2 * rv), z = aol2 * v2;
        const float E = __builtin_amdgcn_exp2f(-1.4426950f * z);
        const float hi = fmaf(2.f, x, 1.f), lo = x + 2.5f, r = __builtin_amdgcn_rcpf(lo * hi), t = (x - 2.5f) * hi * r;
        float p = -0x1.14e136p-14f;
        p = fmaf(p, t, 0x1.a8737ep-12f);
        p = fmaf(p, t, 0x1.eb5800p-12f);
        p = fmaf(p, t, -0x1.11da4ep-8f);
        p = fmaf(p, t, 0x1.edf72cp-11f);
        p = fmaf(p, t, 0x1.0baf52p-5f);
        p = fmaf(p, t, -0x1.a5c2b6p-4f);
        p = fmaf(p, t, 0x1.42db30p-3f);
        p = fmaf(p, t, -0x1.959aa8p-4f);
        p = fmaf(p, t, -0x1.f52d20p-4f);
        p = fmaf(p, t, 0x1.43cc70p+0f);
        const float v = vx * (E * fmaf(p * (lo * r), rv, two_aol_rpi)) * (rv * rv);
        sum += v;
        err += fabsf(v) * (0x1p-18f + 0x1p-20f * z);
    }
    return EwaldBound{wave_total(sum), wave_total(err) * (1.f + 0x1p-10f)};
}

// ---- commit -------------------------------------------------------------------------------
// The event to commit: a stored one (its payload from LDS, its time from the tagger's lane) or one of
// this leg's.
template <int D>
struct Event {
    int tagger, target, adir, cell;
    double aspeed, cv_rate, boundary;
    Time t, astamp;
    double apos[D], tpos[D];
};
template <int D, int NT>
__device__ __forceinline__ void event_of_slot(ChainShared<NT> &sh, int t, Event<D> &e) {
    const Slot &sl = sh.slot[t];
    e.tagger = t;
    e.target = uni(sl.target);
    e.adir = uni(sl.adir);
    e.aspeed = sl.aspeed;
    e.cell = uni(sl.cb_cell);
    e.astamp = sl.astamp;
    e.cv_rate = sl.cv_rate;
    e.boundary = sl.cb_boundary;
#pragma unroll
    for (int d = 0; d < D; d++) {
        e.apos[d] = sl.apos[d];
        e.tpos[d] = sl.tpos[d];
    }
}

// The out-state of the event, committed to the state: send_out_state of its event handler and
// insert_into_global_state (mediator/single_process_mediator.py:130-150), thinning included
// (event_handler_with_bounding_potential.py:75-101).  Every wavefront computes it; wavefront 0
// stores the position.  HOT: a pair, cell-veto or cell-boundary event.
template <int D, int FM, int NT, bool RES, bool HOT>
__device__ __forceinline__ void commit_event(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, const Event<D> &e,
                                             ecmc_event &ev) {
    const int kind = kind_of(q.kinds, e.tagger);
    ev.tagger = e.tagger;
    ev.flags = 0;
    ev.active = g.active;
    ev.target = -1;
    ev.tq = e.t.q;
    ev.tr = e.t.r;
    ev.ncand = g.ncand;
    ev.chash = g.chash;
    ev.pos[0] = ev.pos[1] = ev.pos[2] = 0.0;
    const int act = g.active;
    double p[D];
    int next = act;
    const bool veto = (FM & FEAT_CELL_VETO) && kind == ECMC_TAG_CELL_VETO;
    if (pair_kind(kind) || veto) {
        int target = e.target;
        double tp[D], s[D];
#pragma unroll
        for (int d = 0; d < D; d++) {
            tp[d] = e.tpos[d];
            p[d] = e.apos[d];
            s[d] = 0.0;
        }
        if (veto) {
            // mediator.py:265-292: the occupant of the sampled cell, or none
            const int no = uni(occ_count<RES>(a, q, e.cell));
            if (no > 1) { g.err = ECMC_ERR_STATE; return; }
            const int occupant = occ_get<RES>(a, q, e.cell, 0);
            target = no == 1 ? uni(occupant) : -1;
            if (NT > 64) __syncthreads();   // wavefront 0 edits the lists after the commit
            if (target >= 0) load_pos<RES>(a, q, target, tp);
        }
        if (target >= 0) separation_vector_u<D>(q, e.apos, tp, s);
        bool lift = true, thins = false;
        if (FM & FEAT_EWALD) {
            const ecmc_tagger_desc &T = q.tg[e.tagger];
            const int eh = uni(T.event_handler);
            thins = veto || eh == ECMC_EH_CELL_BOUNDING || eh == ECMC_EH_TWO_LEAF_BOUNDING;
            if (thins) {
                lift = false;
                ring_ensure<RES, D, NT>(a, q, g, g.cursor + 2);
                if (g.err) return;
                if (target >= 0) {
                    double q3[3] = {0, 0, 0};
#pragma unroll
                    for (int d = 0; d < D; d++) q3[d] = pick_axis<D>(s, e.adir + d >= D ? e.adir + d - D : e.adir + d);
                    double c1 = 1.0, c2 = 1.0;
                    if ((q.charged >> e.tagger) & 1u) {
                        c1 = charge_of<RES>(a, q, act);
                        c2 = charge_of<RES>(a, q, target);
                    }
                    double bound = e.cv_rate;   // leaf_unit_cell_veto_event_handler.py:127-149
                    if ((FM & FEAT_CELL_BOUNDING) && eh == ECMC_EH_CELL_BOUNDING) {
                        // two_leaf_unit_cell_bounding_potential_event_handler.py:181-211: the active
                        // unit is still in its cell; bound = the candidate's rate
                        int coord[D];
                        if (uni(pos_to_cell<D>(q, e.apos, coord)) != e.cell) { g.err = ECMC_ERR_STATE; return; }
                        double now[D];
                        load_pos<RES>(a, q, target, now);
                        bound = cell_rate_of_cells<D>(a, q, T, e.cell, pos_to_cell<D>(q, now, coord), e.adir, c1, c2) * e.aspeed;
                    } else if ((FM & FEAT_COULOMB) && eh == ECMC_EH_TWO_LEAF_BOUNDING) {
                        bound = ipcb_derivative(T.bpar[0] * c1 * c2, q3[0], q3[1], q3[2]) * e.aspeed;
                    }
                    // lifting with probability real / bound (two words, drawn where real > 0)
                    const uint32_t w = (uint32_t)g.cursor;
                    double u = words_to_random(ring_word<RES>(a, q, w), ring_word<RES>(a, q, w + 1));
                    u = 0 + (bound - 0) * u;
                    bool drawn = false, settled = false;
                    if (uni(sh.ewald.ok)) {
                        const EwaldTerms &x = sh.ewald;
                        const int l = threadIdx.x & 63;
                        const EwaldBound b = ewald_derivative_fp32(q3[0], q3[1], q3[2], x.L, x.inv_l, x.aol, x.aol2, x.two_aol_rpi,
                                                                   x.code[0][l], x.code[1][l], x.code[2][l], x.f[0][l], x.f[1][l]);
                        const double rate = T.par[3] * c1 * c2 * e.aspeed, real = rate * (double)b.value,
                                     off = fabs(rate) * (double)b.error;
                        drawn = ub(real - off > 0.0);
                        lift = drawn & ub(u < real - off);
                        settled = ub(real + off < 0.0) | (drawn & (lift | ub(u > real + off)));
                    }
                    if (!settled) {
                        const double der = ewald_derivative_wave(a.ewald, a.ewald_codes, a.ewald_ncodes, q3[0], q3[1], q3[2]);
                        const double real = T.par[3] * c1 * c2 * der * e.aspeed;
                        drawn = ub(real > 0);
                        lift = drawn & ub(u < real);
                    }
                    if (drawn) g.cursor += 2;
                }
                if (!lift) add_est(sh, 6, 1.0);
            }
        }
        ev.target = target;
        g.at = e.astamp;
        if (lift) {
            add_est(sh, 0, pick_axis<D>(s, e.adir));
            add_est(sh, 4, 1.0);
            next = target;
            ev.flags |= 1;
        }
        add_est(sh, 2, 1.0);
    } else {
        if (HOT || kind == ECMC_TAG_CELL_BOUNDARY) {
#pragma unroll
            for (int d = 0; d < D; d++) p[d] = e.apos[d];
            slice_pos<D>(q, p, e.adir, e.aspeed, e.astamp, e.t);
#pragma unroll
            for (int d = 0; d < D; d++) p[d] = d == e.adir ? e.boundary : p[d];
            g.at = e.t;
            add_est(sh, 3, 1.0);
        } else if (kind == ECMC_TAG_START_OF_RUN) {
            const ecmc_tagger_desc &T = q.tg[e.tagger];
            next = uni(T.ivalue2);
            g.adir = uni(T.ivalue);
            g.aspeed = T.value;
            g.at.q = 0.0;
            g.at.r = 0.0;
#pragma unroll
            for (int d = 0; d < D; d++) p[d] = g.ap[d];
        } else {
            // sampling, end of run, end of chain: the active unit moved to the event's time
#pragma unroll
            for (int d = 0; d < D; d++) p[d] = g.ap[d];
            slice_pos<D>(q, p, g.adir, g.aspeed, g.at, e.t);
            g.at = e.t;
            if (kind == ECMC_TAG_END_OF_RUN) g.done = 1;
            if (kind == ECMC_TAG_END_OF_CHAIN) {
                g.eoc_last = e.t;
                ev.target = e.target;
                add_est(sh, 1, q.tg[e.tagger].value * g.aspeed);
                add_est(sh, 5, 1.0);
                g.adir = g.adir + 1 == D ? 0 : g.adir + 1;
                if (e.target != act) ev.flags |= 1;
                next = e.target;
            }
        }
    }
    if (act >= 0) {
        if (threadIdx.x == 0) store_pos<RES>(a, q, act, p);
#pragma unroll
        for (int d = 0; d < D; d++) ev.pos[d] = p[d];
    }
    g.active = next;
    if (next == act) {
#pragma unroll
        for (int d = 0; d < D; d++) g.ap[d] = p[d];
    } else {
        load_pos<RES>(a, q, next, g.ap);
    }
}

// ---- launch ---------------------------------------------------------------------------------
// The hot list: the create list of the first pair tagger, if it has the form (one thread).
template <int NT>
__device__ __forceinline__ HotList hot_list(const ChainShared<NT> &sh, const ecmc_tagger_desc *tg, uint64_t kinds, int n_taggers) {
    HotList l;
    l.hard = 0;
    l.radius = 0.0;
    l.items = -1;
    l.tags = l.mask = l.creators = l.prefixed = l.trashers = 0;
    l.boundary = l.veto = -1;
    l.before = l.veto_before = 0;
    int first = 0;
    while (first < n_taggers && !pair_kind(kind_of(kinds, first))) first++;
    if (first == n_taggers) return l;
    const uint64_t create = sh.plan[first].create;
    const int n = sh.plan[first].n_create;
    int items = 0;
    for (int i = 0; i < n; i++) {
        const int t = (int)((create >> (4 * i)) & 15u), kind = kind_of(kinds, t);
        if ((l.mask >> t) & 1u) return l;
        l.mask |= 1u << t;
        if (pair_kind(kind)) {
            if (items == HOT_ITEMS) return l;
            l.tags |= (uint32_t)t << (4 * items++);
        } else if (kind == ECMC_TAG_CELL_BOUNDARY && l.boundary < 0) {
            l.boundary = t;
            l.before = items;
        } else if (kind == ECMC_TAG_CELL_VETO && l.veto < 0) {
            l.veto = t;
            l.veto_before = items;
        } else {
            return l;
        }
    }
    if (items == 0) return l;
    for (int t = 0; t < n_taggers; t++) {
        const TaggerPlan &p = sh.plan[t];
        if ((p.trash & l.mask) == l.mask) l.trashers |= 1u << t;
        const int extra = p.n_create - n;
        if (extra < 0 || (n < 16 && (p.create >> (4 * extra)) != create)) continue;
        bool apart = true;
        for (int i = 0; i < extra; i++) {
            const int o = (int)((p.create >> (4 * i)) & 15u);
            apart = apart && !((l.mask >> o) & 1u) && !pair_kind(kind_of(kinds, o));
        }
        if (!apart) continue;
        if (extra == 0) l.creators |= 1u << t;
        else l.prefixed |= 1u << t;
    }
    l.items = items;
    const ecmc_tagger_desc &pair = tg[l.tags & 15u];
    l.hard = items == 1 && pair.event_handler == ECMC_EH_TWO_LEAF && pair.potential == ECMC_POT_HARD_SPHERE;
    l.radius = pair.par[0];
    return l;
}

// Copies a system's launch state into LDS and registers: the stored events' payloads once into LDS, their
// times into the lanes of every wavefront.
template <int D, int NT, bool RES>
__device__ __forceinline__ void launch_load(const ChainArgs &a, Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh) {
    const int tid = threadIdx.x, lane = tid & 63;
    q.dyn = chain_dyn_lds;
    q.tg = RES ? reinterpret_cast<ecmc_tagger_desc *>(chain_dyn_lds + a.lds_tg_off) : static_taggers();
    q.n = a.n; q.ncells = a.ncells; q.occ_cols = a.occ_cols; q.occ_cap = a.occ_cap; q.ring_mask = a.ring_words - 1;
    q.leaves = a.leaves; q.max_occ = a.max_occ;
    q.o_ring = a.lds_ring_off; q.o_charge = a.lds_charge_off; q.o_occn = a.lds_occn_off; q.o_occ = a.lds_occ_off;
    q.o_sur = a.lds_sur_off;
    {
        EwaldTerms &x = sh.ewald;
        const int nr = a.ewald_nreal, nf = a.ewald_ncodes - nr, nn = a.ewald.fc + 1;
        const bool ok = a.ewald_ncodes > 0 && nr <= 64 && nf <= 128 && a.L > 1e-6 && a.L < 1e6;
        for (int i = threadIdx.x; ok && i < 192; i += NT) {
            const int t = i < 64 ? (i < nr ? i : -1) : (i - 64 < nf ? nr + i - 64 : -1), c = t >= 0 ? a.ewald_codes[t] : -1;
            x.code[i >> 6][i & 63] = c;
            if (i >= 64)
                x.f[(i >> 6) - 1][i & 63] =
                    c >= 0 ? (float)a.ewald.f[((((c >> 16) & 255) - 128) * nn + ((c >> 8) & 255) - 128) * nn + (c & 255) - 128] : 0.f;
        }
        if (threadIdx.x == 0) {
            x.L = a.L;
            x.inv_l = 1.0 / a.L;
            x.aol = (float)a.ewald.aol;
            x.aol2 = (float)a.ewald.aol2;
            x.two_aol_rpi = (float)a.ewald.two_aol_rpi;
            x.ok = ok;
        }
    }
    q.L = a.L; q.half = a.half; q.beta = a.beta;
    q.inv_beta = (float)(1.0 / a.beta) * (1.f - 0x1p-20f);
    q.nb_cells = a.nb_table ? 0 : a.nb_stride;
#pragma unroll
    for (int d = 0; d < 3; d++) q.cb_max[d] = a.cb_max[d];
    nearby_offsets<D>(a, q);
#pragma unroll
    for (int d = 0; d < D; d++) {
        q.side[d] = a.side[d];
        q.inv[d] = 1.0 / a.side[d];
        q.cps[d] = a.cps[d];
        q.cum[d] = a.cum[d];
    }
    const ChainState &s = *a.st;
    // (loads through pointers from memory count as lane-varying)
    g.active = uni(s.active); g.adir = uni(s.adir); g.aspeed = uni(s.aspeed); g.at = uni(s.at);
    g.occ_id = uni(s.occ_id); g.occ_cell = uni(s.occ_cell);
    g.started = uni(s.started); g.done = uni(s.done); g.err = uni(s.err); g.pending = uni(s.pending_creates);
    g.last_tagger = uni(s.last_tagger); g.committed = 0;
    g.last = uni(s.last); g.seq = (int64_t)uni((uint64_t)s.seq); g.eoc_last = uni(s.eoc_last); g.samp_time = uni(s.samp_time);
    g.cursor = uni(s.cursor); g.produced = uni(s.produced); g.keep = g.cursor;
    if (tid < 8) sh.est[tid] = s.est[tid];
    g.ncand = uni(s.ncand); g.chash = (uint32_t)uni((int)s.chash); g.nsur = uni(s.nsur); g.mean_step = uni(s.mean_step);
    const Slot &sl = s.slot[lane < ECMC_MAX_TAGGERS ? lane : 0];
    g.lt = sl.t; g.lseq = sl.seq; g.lvalid = lane < ECMC_MAX_TAGGERS && sl.valid;
#pragma unroll
    for (int d = 0; d < D; d++) {
        g.ap[d] = 0.0;
        g.cc[d] = g.occ_cell >= 0 ? (g.occ_cell / q.cum[d]) % q.cps[d] : 0;
    }
    if (RES) {
        double *lp = reinterpret_cast<double *>(q.dyn);
        for (int i = tid; i < D * q.n; i += NT) lp[i] = a.pos[i];
        uint32_t *lr = reinterpret_cast<uint32_t *>(q.dyn + q.o_ring);
        for (int i = tid; i <= q.ring_mask; i += NT) lr[i] = a.ring[i];
        if (q.o_charge >= 0)
            for (int i = tid; i < q.n; i += NT) reinterpret_cast<double *>(q.dyn + q.o_charge)[i] = a.charge[i];
        if (a.occupancy) {
            for (int i = tid; i < q.ncells; i += NT) reinterpret_cast<int32_t *>(q.dyn + q.o_occn)[i] = a.occ_n[i];
            uint16_t *lo = reinterpret_cast<uint16_t *>(q.dyn + q.o_occ);
            for (int i = tid; i < q.ncells * q.occ_cols; i += NT)
                lo[i] = (uint16_t)a.occ[(size_t)(i / q.occ_cols) * q.occ_cap + i % q.occ_cols];
            if (q.max_occ > 0)
                for (int i = tid; i < g.nsur; i += NT) set_sur<true>(a, q, i, a.sur_cell[i], a.sur_id[i]);
        }
    }
    {
        const uint32_t *src = reinterpret_cast<const uint32_t *>(a.tg);
        uint32_t *dst = reinterpret_cast<uint32_t *>(q.tg);
        for (int i = tid; i < (int)(sizeof(ecmc_tagger_desc) / 4) * a.n_taggers; i += NT) dst[i] = src[i];
        const uint32_t *ss = reinterpret_cast<const uint32_t *>(s.slot);
        const int words = (int)sizeof(Slot) / 4 * ECMC_MAX_TAGGERS;
        uint32_t *ds = reinterpret_cast<uint32_t *>(sh.slot);
        for (int i = tid; i < words; i += NT) ds[i] = ss[i];
    }
    for (int i = tid; i < 3 * AXIS_CELLS; i += NT) {
        const int d = i / AXIS_CELLS, c = i % AXIS_CELLS;
        if (d < D && c < a.cps[d]) sh.axis[d][c] = a.cmin[(size_t)(c * a.cum[d]) * D + d];
    }
    __syncthreads();
    // one bit per occupied cell (grids of at most FAR_BLOCK cells; larger ones read the counts)
    if (tid < 64 && a.occupancy) {
        uint32_t w = 0;
#pragma unroll 1
        for (int k = 0; k < 32; k++)
            if (tid * 32 + k < q.ncells && occ_count<RES>(a, q, tid * 32 + k) > 0) w |= 1u << k;
        sh.occupied[tid] = w;
    }
    // every wavefront derives the bit fields of its own; wavefront 0 writes the plans
    int kind = 0, test = QT_DIRECT, draws = 0, charged = 0, inversion = 0;
    if (lane < a.n_taggers) {
        const ecmc_tagger_desc &tg = q.tg[lane];
        kind = tg.kind;
        draws = pair_kind(kind) && pot_draws(tg);
        charged = tg.use_charge != 0;
        TaggerPlan pl;
        pl.create = 0;
        pl.trash = 0;
        pl.n_create = tg.n_create;
        for (int i = 0; i < tg.n_create; i++) pl.create |= (uint64_t)tg.create[i] << (4 * i);
        for (int i = 0; i < tg.n_trash; i++) pl.trash |= 1u << tg.trash[i];
        pl.p = 1;
        pl.rc2_hi = INFINITY;
        pl.powrc = 1.0;
        pl.r0 = pl.k6 = pl.k12 = 0.0;
        if (pair_kind(kind) && tg.potential == ECMC_POT_LENNARD_JONES) {
            const MexicanHat h = mh_lennard_jones(tg.par[0], tg.par[1]);
            pl.r0 = h.r0;
            pl.k6 = h.k6;
            pl.k12 = h.k12;
        }
        pl.set_key = 16 + lane;
        if (pair_kind(kind)) {
            inversion = tg.event_handler == ECMC_EH_TWO_LEAF_BOUNDING                                                          ? 1
                        : tg.event_handler == ECMC_EH_CELL_BOUNDING                                                            ? 2
                        : tg.potential == ECMC_POT_INVERSE_POWER || tg.potential == ECMC_POT_INVERSE_POWER_TRUNC               ? 0
                                                                                                                               : 2;
            if (tg.event_handler == ECMC_EH_TWO_LEAF_BOUNDING) test = QT_COULOMB_BOUND;
            else if (tg.event_handler == ECMC_EH_CELL_BOUNDING) test = QT_CELL;
            else if (tg.potential == ECMC_POT_INVERSE_POWER || tg.potential == ECMC_POT_INVERSE_POWER_TRUNC) {
                const double p = tg.par[0];
                const bool trunc = tg.potential == ECMC_POT_INVERSE_POWER_TRUNC;
                if (p >= 1.0 && p <= 32.0 && p == floor(p)) {
                    test = QT_INVERSE_POWER;
                    pl.p = (int)p;
                    if (trunc) pl.rc2_hi = (float)(tg.par[2] * tg.par[2]) * (1.f + 0x1p-22f);
                }
                if (trunc) pl.powrc = pow_half_power(tg.par[2] * tg.par[2], p);
            }
            pl.set_key = kind;
            if (kind == ECMC_TAG_FACTOR_MAP) {
                // the first tagger with the same map stands for all of them
                pl.set_key = 16 + lane;
                for (int o = lane - 1; o >= 0; o--) {
                    const ecmc_tagger_desc &og = q.tg[o];
                    bool same = og.kind == ECMC_TAG_FACTOR_MAP && og.fmap_local == tg.fmap_local;
                    for (int k = 0; same && k < ECMC_MAX_LEAVES; k++) {
                        same = og.fmap_n[k] == tg.fmap_n[k];
                        for (int e = 0; same && e < tg.fmap_n[k]; e++) same = og.fmap_target[k][e] == tg.fmap_target[k][e];
                    }
                    if (same) pl.set_key = 16 + o;
                }
            }
        }
        if (tid < 64) sh.plan[lane] = pl;
    }
    q.kinds = 0;
    q.tests = q.draws = q.charged = q.inversions = 0;
#pragma unroll
    for (int t = 0; t < ECMC_MAX_TAGGERS; t++) {
        q.kinds |= (uint64_t)(uint32_t)__builtin_amdgcn_readlane(kind, t) << (4 * t);
        q.tests |= (uint32_t)__builtin_amdgcn_readlane(test, t) << (2 * t);
        q.inversions |= (uint32_t)__builtin_amdgcn_readlane(inversion, t) << (2 * t);
    }
    q.draws = (uint32_t)__ballot(draws) & 0xffffu;
    q.charged = (uint32_t)__ballot(charged) & 0xffffu;
    __syncthreads();
    if (tid == 0) {
        Geo<3> &m = sh.geo;
        m.dyn = q.dyn;
        m.tg = q.tg;
        m.n = q.n; m.ncells = q.ncells; m.occ_cols = q.occ_cols; m.occ_cap = q.occ_cap; m.ring_mask = q.ring_mask;
        m.leaves = q.leaves; m.max_occ = q.max_occ;
        m.o_ring = q.o_ring; m.o_charge = q.o_charge; m.o_occn = q.o_occn; m.o_occ = q.o_occ; m.o_sur = q.o_sur;
        m.L = q.L; m.half = q.half; m.beta = q.beta; m.inv_beta = q.inv_beta;
#pragma unroll
        for (int d = 0; d < D; d++) { m.side[d] = q.side[d]; m.inv[d] = q.inv[d]; m.cps[d] = q.cps[d]; m.cum[d] = q.cum[d]; }
        m.nb_cells = q.nb_cells; m.kinds = q.kinds; m.tests = q.tests; m.inversions = q.inversions; m.draws = q.draws; m.charged = q.charged;
        sh.hot = hot_list<NT>(sh, q.tg, q.kinds, a.n_taggers);
    }
    __syncthreads();
    if (g.active >= 0) load_pos<RES>(a, q, g.active, g.ap);
}

// Writes the launch state back (lane t of wavefront 0 the stored event of tagger t).
template <int D, int NT, bool RES>
__device__ __forceinline__ void launch_store(const ChainArgs &a, const Geo<D> &q, const Leg<D> &g, ChainShared<NT> &sh) {
    const int tid = threadIdx.x;
    __syncthreads();
    ChainState &s = *a.st;
    if (tid < ECMC_MAX_TAGGERS) {
        Slot sl = sh.slot[tid];
        sl.t = g.lt; sl.seq = g.lseq; sl.valid = g.lvalid;
        s.slot[tid] = sl;
    }
    if (tid == 0) {
        s.active = g.active; s.adir = g.adir; s.aspeed = g.aspeed; s.at = g.at;
        s.occ_id = g.occ_id; s.occ_cell = g.occ_cell;
        s.started = g.started; s.done = g.done; s.err = g.err; s.pending_creates = g.pending;
        s.last_tagger = g.last_tagger; s.stop_reason = 0;
        s.last = g.last; s.seq = g.seq; s.eoc_last = g.eoc_last; s.samp_time = g.samp_time;
        s.cursor = g.cursor; s.produced = g.produced;
        for (int k = 0; k < 7; k++) s.est[k] = sh.est[k];
        s.ncand = g.ncand; s.chash = g.chash; s.nsur = g.nsur; s.mean_step = g.mean_step;
    }
    if (RES) {
        const double *lp = reinterpret_cast<const double *>(q.dyn);
        for (int i = tid; i < D * q.n; i += NT) a.pos[i] = lp[i];
        const uint32_t *lr = reinterpret_cast<const uint32_t *>(q.dyn + q.o_ring);
        for (int i = tid; i <= q.ring_mask; i += NT) a.ring[i] = lr[i];
        if (a.occupancy) {
            for (int i = tid; i < q.ncells; i += NT) a.occ_n[i] = occ_count<true>(a, q, i);
            const uint16_t *lo = reinterpret_cast<const uint16_t *>(q.dyn + q.o_occ);
            for (int i = tid; i < q.ncells * q.occ_cols; i += NT)
                a.occ[(size_t)(i / q.occ_cols) * q.occ_cap + i % q.occ_cols] = lo[i];
            if (q.max_occ > 0)
                for (int i = tid; i < g.nsur; i += NT) {
                    a.sur_cell[i] = sur_cell<true>(a, q, i);
                    a.sur_id[i] = sur_id<true>(a, q, i);
                }
        }
    }
    if (a.host) {
        __syncthreads();   // the state is thread 0's and the first lanes'
        const uint64_t *from = reinterpret_cast<const uint64_t *>(a.st);
        uint64_t *to = reinterpret_cast<uint64_t *>(&a.host->st);
        for (int i = tid; i < (int)(sizeof(ChainState) / 8); i += NT) to[i] = from[i];
        if (tid == 0) {
            a.host->n_out = *a.n_out;
            a.host->has_positions = RES ? 1 : 0;
        }
        if (RES) {
            const double *lp = reinterpret_cast<const double *>(q.dyn);
            double *out = reinterpret_cast<double *>(a.host + 1);
            for (int i = tid; i < D * q.n; i += NT) out[i] = lp[(i % D) * q.n + i / D];
        }
    }
}

// The earliest candidate among the work of all wavefronts (each with its lanes' best in m), after
// one barrier; `win`: a copy of ChainShared::win that no wavefront reads any more.  The rare steps
// evaluate several sets one after the other into one copy: `again` ends with a second barrier.
template <int NT>
__device__ __forceinline__ Winner group_winner(Winner *win, const Winner &m, bool again) {
    constexpr int NW = NT / 64;
    Winner w = wave_winner(m);
    if (NW > 1) {
        if ((threadIdx.x & 63) == 0) win[wave_index<NT>()] = w;
        __syncthreads();
        w = no_winner();
#pragma unroll
        for (int v = 0; v < NW; v++) {
            // read as uniform values: the comparison is then a scalar branch
            Winner o;
            o.rank = uni(win[v].rank);
            w.bad = max(w.bad, uni(win[v].bad));
            if (o.rank == NO_RANK) continue;
            o.t.q = uni(win[v].t.q);
            o.t.r = uni(win[v].t.r);
            if (w.rank != NO_RANK && !ub(winner_lt(o, w))) continue;
            w.t = o.t;
            w.rank = o.rank;
            w.dt = uni(win[v].dt);
            w.tag = uni(win[v].tag);
            w.target = uni(win[v].target);
        }
        if (again) __syncthreads();
    }
    return w;
}

// Evaluates every candidate of tagger t exactly, over the workgroup, and keeps the earliest as its
// stored event; a set whose words do not fit in the ring goes in segments.
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ void create_pair_full(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, int t, int kind,
                                                 Counts &cn, bool hashed) {
    const int lane = threadIdx.x & 63, wave = wave_index<NT>();
    const int M = candidate_count<D, FM, NT, RES>(a, q, g, sh, t, kind, cn);
    const bool draws = (q.draws >> t) & 1u;
    if (hashed) g.chash += candidate_hash<D, FM, NT, RES>(a, q, g, sh, t, kind, M, cn, g.ncand);
    const uint64_t first = g.cursor;
    const int64_t seq0 = g.seq;
    if (draws) g.cursor += 2ull * (uint64_t)M;
    g.seq += M;
    g.ncand += M;
    lane_slot(g, t, Time{0.0, 0.0}, 0, 0);
    const int seg_cap = (q.ring_mask + 1 - 512 - 2 * RING_STEP) / 2;
    Winner acc = no_winner();
#pragma unroll 1
    for (int lo = 0; lo < M; lo += seg_cap) {
        const int hi = min(M, lo + seg_cap);
        g.keep = draws ? first + 2ull * (uint64_t)lo : g.cursor;
        if (draws) ring_ensure<RES, D, NT>(a, q, g, g.keep + 2ull * (uint64_t)(hi - lo));
        if (g.err) return;
        Winner m = no_winner();
        Candidates<D, FM, NT, RES> cs(a, q, sh, t, kind, g.active, M, cn);
        int before = 0;
#pragma unroll 1
        for (;; cs.first += FAR_BLOCK) {
            if (cs.far() && q.ncells > FAR_BLOCK) before += far_prefix<D, NT, RES>(a, q, g, sh, cs.first, before);
            const int count = cs.span();
#pragma unroll 1
            for (int b = wave * 64; b < count; b += NT) {
                const int idx = b + lane;
                int j, target, cell;
                bool live = cs.get(min(idx, count - 1), j, target, cell) && idx < count;
                live = live && j >= lo && j < hi;
                if (live) {
                    const double dt = candidate_dt<D, FM, NT, RES>(a, q, g, sh, t, 2u * (uint32_t)(j - lo), target, cell);
                    Winner c;
                    c.t = time_add(g.at, dt);
                    c.dt = dt;
                    c.rank = j;
                    c.tag = t;
                    c.target = target;
                    c.bad = m.bad;
                    if (isnan(dt)) m.bad = max(m.bad, error_code(dt));
                    else if (winner_lt(c, m)) m = c;
                }
            }
            if (!cs.far() || cs.first + FAR_BLOCK >= q.ncells) break;
        }
        const Winner w = group_winner<NT>(sh.win[2], m, true);
        const int bad = max(w.bad, acc.bad);
        if (w.rank != NO_RANK && (acc.rank == NO_RANK || ub(winner_lt(w, acc)))) acc = w;
        acc.bad = bad;
    }
    store_winner<D, NT, RES>(a, q, g, sh, t, M, seq0, acc);
}

// The create list of tagger `creator` from its entry ci on, up to entry `end`, every tagger's event
// stored.
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ void general_creates(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, int creator, int ci,
                                                int end, bool hashed) {
    const uint64_t create = uni(sh.plan[creator].create);
    Counts cn;
    cn.nb = cn.far = -1;
#pragma unroll 1
    for (; ci < end && !g.err; ci++) {
        const int t = (int)((create >> (4 * ci)) & 15u), kind = kind_of(q.kinds, t);
        g.keep = g.cursor;
        if (kind == ECMC_TAG_CELL_BOUNDARY) {
            Boundary b;
            b.p.w = -1;
            create_boundary<D, NT>(a, q, g, sh, t, b);
            if (!g.err) store_boundary<D, NT>(g, sh, b);
        } else if (pair_kind(kind)) {
            create_pair_full<D, FM, NT, RES>(a, q, g, sh, t, kind, cn, hashed);
        } else {
            create_single<D, FM, NT, RES>(a, q, g, sh, t, kind);
        }
    }
}

// The rare steps of a chain, called from the leg loop with the leg in LDS (sh.leg, every wavefront
// its own) so that their code takes no registers from it:
//   STEP_LEG     the create list of `arg` from entry `from` on in the general form, the earliest stored event and its commit;
//   STEP_START   the start of run's event and its commit;
//   STEP_CREATE  the first `from` entries of the create list of `arg`;
//   STEP_COMMIT  the commit of tagger `arg`'s stored event.
enum { STEP_LEG = 0, STEP_START = 1, STEP_CREATE = 2, STEP_COMMIT = 3 };
template <int D, int FM, int NT, bool RES>
__device__ __noinline__ static void rare_step(const ChainArgs *args, ChainShared<NT> *shared, int step, int arg, int from) {
    const ChainArgs &a = *reinterpret_cast<const ChainArgs *>(uni((uint64_t)args));
    ChainShared<NT> &sh = *reinterpret_cast<ChainShared<NT> *>(uni((uint64_t)shared));
    step = uni(step);
    arg = uni(arg);
    from = uni(from);
    const int wave = wave_index<NT>();
    wave_sync();
    Geo<D> q;
    geo_load<D>(sh.geo, a, q);
    Leg<D> g;
    leg_from<D>(sh.leg[wave], sh.time[wave], g);
    const bool hashed = a.log != nullptr;
    if (step == STEP_CREATE) {
        general_creates<D, FM, NT, RES>(a, q, g, sh, arg, 0, from, hashed);
    } else {
        int chosen = arg;
        if (step == STEP_START) {
            int sor = -1;
#pragma unroll 1
            for (int t = 0; t < a.n_taggers; t++)
                if (kind_of(q.kinds, t) == ECMC_TAG_START_OF_RUN) sor = t;
            if (sor < 0) g.err = ECMC_ERR_CONFIGURATION;
            else create_single<D, FM, NT, RES>(a, q, g, sh, sor, ECMC_TAG_START_OF_RUN);
            g.started = 1;
        } else if (step == STEP_LEG && arg >= 0) {
            general_creates<D, FM, NT, RES>(a, q, g, sh, arg, from, uni(sh.plan[arg].n_create), hashed);
        }
        g.keep = g.cursor;
        if (!g.err && step != STEP_COMMIT) {
            g.pending = 0;
            const Pick s = pick_stored(g);
            chosen = s.w;
            if (chosen < 0) g.err = ECMC_ERR_SCHEDULER;
        }
        if (!g.err) {
            if (NT > 64) __syncthreads();   // the payloads are thread 0's
            else wave_sync();
            Event<D> e;
            event_of_slot<D, NT>(sh, chosen, e);
            e.t.q = lane_d(g.lt.q, chosen);
            e.t.r = lane_d(g.lt.r, chosen);
            if (ub(time_lt(e.t, g.last))) {
                g.err = ECMC_ERR_SCHEDULER;
            } else {
                g.last = e.t;
                g.pending = 0;
                ecmc_event ev;
                commit_event<D, FM, NT, RES, false>(a, q, g, sh, e, ev);
                if (threadIdx.x == 0) sh.ev = ev;
                g.last_tagger = chosen;
                g.committed = 1;
                if ((uni((int)sh.plan[chosen].trash) >> (threadIdx.x & 15)) & 1) g.lvalid = 0;
            }
        }
    }
    if (NT > 64) __syncthreads();   // lists that other wavefronts read are edited by the next leg
    leg_to<D>(g, sh.leg[wave], sh.time[wave]);
    wave_sync();
}

// A leg of the hot list: its creates and the choice of its event, in `e`.  Returns the outcome:
// HOT_EVENT (commit e), HOT_STORED (the earliest stored event `stored` comes first and trashes the
// list) or HOT_GENERAL (the general form has to run the leg: the leg's state is as before).  `turn`: the
// leg's parity, which copy of the winners it uses.
enum { HOT_EVENT = 0, HOT_STORED = 1, HOT_GENERAL = 2 };
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ int hot_events(const ChainArgs &a, const Geo<D> &q, Leg<D> &g, ChainShared<NT> &sh, const HotList &hot,
                                          const Items &constants, const Pick &stored, bool hashed, int turn, Event<D> &e) {
    constexpr int NW = NT / 64;
    const int lane = threadIdx.x & 63, wave = wave_index<NT>();
    const uint64_t cursor0 = g.cursor;
    const int64_t seq0 = g.seq;
    g.keep = cursor0;
    auto general = [&]() {
        g.cursor = cursor0;
        g.seq = seq0;
        g.ncand = 0;
        g.chash = 0;
        return HOT_GENERAL;
    };
    // ---- creates: the earliest event known before the pairs is S
    Pick S = stored;
    Boundary B;
    B.p.w = -1;
    B.x = 0.0;
    if (hot.boundary >= 0) {
        create_boundary<D, NT>(a, q, g, sh, hot.boundary, B);
        if (g.err) { g.err = 0; return general(); }
        if (S.w < 0 || ub(time_lt(B.p.t, S.t))) S = B.p;
        else if (ub(time_eq(B.p.t, S.t))) return general();
    }
    Counts cn;
    cn.nb = cn.far = -1;
    Items its = constants;
    its.word = 0;
    its.rank = its.before = 0;
    uint32_t word = 0, veto_word = 0;
    int M0 = 0, ncand = 0;
#pragma unroll
    for (int i = 0; i < HOT_ITEMS; i++) {
        if (i >= hot.items) break;
        const int t = (int)((hot.tags >> (4 * i)) & 15u);
        const int M = candidate_count<D, FM, NT, RES>(a, q, g, sh, t, kind_of(q.kinds, t), cn);
        if (i == 0) M0 = M;
        its.word = lane == i ? word : its.word;
        its.rank = lane == i ? ncand + (hot.boundary >= 0 && i >= hot.before ? 1 : 0) : its.rank;
        its.before = lane == i ? ncand : its.before;
        if ((q.draws >> t) & 1u) word += 2u * (uint32_t)M;
        ncand += M;
        if (i + 1 == hot.veto_before) veto_word = word;
    }
    if ((int)word + 512 + 2 * RING_STEP > q.ring_mask + 1) return general();   // more words than the ring holds
    if ((FM & FEAT_CELL_VETO) && hot.veto >= 0) {
        // the veto draws its words between the pair taggers' created before and after it
        g.cursor = cursor0 + veto_word;
        create_cell_veto<D, NT, RES>(a, q, g, sh, hot.veto);
        if (g.err) { g.err = 0; return general(); }
        const uint32_t took = (uint32_t)(g.cursor - cursor0) - veto_word;
        word += took;
        its.word += lane >= hot.veto_before ? took : 0u;
        its.rank += lane >= hot.veto_before ? 1 : 0;
        Pick v;
        v.t.q = lane_d(g.lt.q, hot.veto);
        v.t.r = lane_d(g.lt.r, hot.veto);
        v.w = hot.veto;
        if (S.w < 0 || ub(time_lt(v.t, S.t))) S = v;
        else if (ub(time_eq(v.t, S.t))) return general();
        lane_slot(g, hot.veto, v.t, 0, 0);   // its payload stays in LDS; only this leg may commit it
    }
    g.cursor = cursor0 + word;
    g.seq += ncand;
    g.ncand = ncand;
    ring_ensure<RES, D, NT>(a, q, g, g.cursor);
    if (hashed) {
        g.chash = 0;
#pragma unroll 1
        for (int i = 0; i < hot.items; i++) {
            const int t = (int)((hot.tags >> (4 * i)) & 15u), kind = kind_of(q.kinds, t);
            g.chash += candidate_hash<D, FM, NT, RES>(a, q, g, sh, t, kind, candidate_count<D, FM, NT, RES>(a, q, g, sh, t, kind, cn), cn,
                                                      __builtin_amdgcn_readlane(its.before, i));
        }
    }
    // ---- the horizon: the time of S, or sooner
    const double dS = S.w >= 0 ? fmax(time_sub(S.t, g.at), 0.0) : INFINITY;
    double h = fmin(dS, g.mean_step > 0.0 ? 3.0 * g.mean_step : 0.125 * q.L / g.aspeed);
    const int tag0 = (int)(hot.tags & 15u);
    // a single set without a quick test is evaluated over all wavefronts at once
    const bool direct = hot.items == 1 && ((q.tests >> (2 * tag0)) & 3) == QT_DIRECT;
    Winner P = no_winner();
#pragma unroll 1
    for (int narrowed = 0;;) {
        int total = 0, q0 = 0, q1 = 0, q2 = 0;
        if (!direct) {
            const int qn = gather_contenders<D, FM, NT, RES>(a, q, g, sh, its, h, cn);
            total = q0 = qn;
            bool overflow = qn > QCAP;
            if (NW > 1) {
                if (lane == 0) sh.qn[wave] = qn;
                __syncthreads();
                q0 = uni(sh.qn[0]);
                q1 = uni(sh.qn[1]);
                q2 = uni(sh.qn[2]);
                const int q3 = uni(sh.qn[3]);
                total = q0 + q1 + q2 + q3;
                overflow = max(max(q0, q1), max(q2, q3)) > QCAP;
            } else {
                wave_sync();
            }
            if (overflow) {
                // a narrower horizon, else the general form
                if (NW > 1) __syncthreads();   // the counts are read before they are written again
                if (++narrowed > 2) return general();
                h *= 0.25;
                continue;
            }
        }
        // Words ahead of the stream, made by the wavefront that inverts no contenders: as many as
        // this leg drew and some more, as far as the ring holds them beside this leg's and the two
        // before it (a direct leg has no barrier up to here, and a slower wavefront may still be
        // taking the last leg's thinning draw).
        const int drawn = (int)word, ready = (int)(g.produced - cursor0);
        const int want = min(2 * drawn + drawn / 4 + 640, q.ring_mask + 1 - 2) - ready;
        constexpr int maker = NW > 1 ? 1 : 0;
        int steps = 0;
        if (want >= RING_STEP) {
            steps = want / RING_STEP;
            if (wave == maker) ring_make<RES>(a, q, g.produced, steps);
        }
        Winner m = no_winner();
        const int workers = NW > 1 && !direct ? NW - 1 : NW;
        // few contenders: each kind of inversion on a wavefront of its own, so that they run side by
        // side and not one after the other in one wavefront (12 000 -> 9000 cycles for the 33
        // contenders of three kinds of a charged leg)
        const bool by_kind = NW > 1 && !direct && total <= 64;
        const int kind_here = wave == 0 ? 0 : wave - 1;
        int b = by_kind ? (wave == maker ? total : 0) : direct ? wave * 64 : (NW > 1 ? (wave == 0 ? 0 : (wave == maker ? total : (wave - 1) * 64)) : 0);
        const int count = direct ? M0 : total;
        Candidates<D, FM, NT, RES> cs(a, q, sh, tag0, kind_of(q.kinds, tag0), g.active, M0, cn);
        const uint32_t word0 = item_word(its, 0);
        const int rank0 = item_rank(its, 0);
#pragma unroll 1
        for (; b < count; b += workers * 64) {
            const int idx = b + lane;
            bool here = idx < count;
            if (by_kind && here) {
                const bool b0 = idx >= q0, b1 = idx >= q0 + q1, b2 = idx >= q0 + q1 + q2;
                const int w = (int)b0 + (int)b1 + (int)b2, k = idx - (b2 ? q0 + q1 + q2 : (b1 ? q0 + q1 : (b0 ? q0 : 0)));
                here = (int)((q.inversions >> (2 * (sh.queue[w][k].tag_cell & 15))) & 3u) == kind_here;
            }
            if (here) {
                Contender c;
                if (direct) {
                    int j, cell;
                    cs.get(idx, j, c.target, cell);
                    c.word = word0 + 2u * (uint32_t)j;
                    c.rank = rank0 + j;
                    c.tag_cell = tag0;
                } else {
                    int w = 0, k = idx;
                    if (NW > 1) {
                        const bool b0 = k >= q0, b1 = k >= q0 + q1, b2 = k >= q0 + q1 + q2;
                        w = (int)b0 + (int)b1 + (int)b2;
                        k -= b2 ? q0 + q1 + q2 : (b1 ? q0 + q1 : (b0 ? q0 : 0));
                    }
                    c = sh.queue[w][k];
                }
                double dt;
                if (POT_BUILT(ECMC_POT_HARD_SPHERE) && hot.hard) {
                    // nothing is drawn or looked up: the call's generality costs more than the root
                    double tp[D], s[D];
                    load_pos<RES>(a, q, c.target, tp);
                    separation_vector<D>(q, g.ap, tp, s);
                    dt = hs_displacement<D>(g.adir, g.aspeed, s, hot.radius);
                } else {
                    dt = candidate_dt<D, FM, NT, RES>(a, q, g, sh, c.tag_cell & 15, c.word, c.target, c.tag_cell >> 4);
                }
                Winner v;
                v.t = time_add(g.at, dt);
                v.dt = dt;
                v.rank = c.rank;
                v.tag = c.tag_cell & 15;
                v.target = c.target;
                v.bad = m.bad;
                if (isnan(dt)) m.bad = max(m.bad, error_code(dt));
                else if (winner_lt(v, m)) m = v;
            }
        }
        P = group_winner<NT>(sh.win[turn], m, false);
        g.produced += (uint64_t)steps * RING_STEP;
        if (P.bad) return general();   // which reports it, unless its set has an earlier event or another set errs first
        const bool any = P.rank != NO_RANK;
        if (direct || (any && ub(P.dt <= h)) || (S.w >= 0 && ub(dS <= h))) break;
        // nothing within the horizon: a wider one
        if (narrowed || ub(!(h < 0x1p60))) return general();
        h = h > 0.0 ? h * 4.0 : 0x1p-10 * q.L / g.aspeed;
        h = fmin(fmin(h, dS), 0x1p60);
    }
    const bool any = P.rank != NO_RANK;
    const bool fresh = any && (S.w < 0 || ub(time_lt(P.t, S.t)));
    if ((!fresh && (S.w < 0 || (any && ub(time_eq(P.t, S.t))))) || ub(isinf(fresh ? P.t.q : S.t.q))) return general();
    const int chosen = fresh ? P.tag : S.w;
    if (!((hot.trashers >> chosen) & 1u)) return general();   // some event of this list outlives the commit
    if (ub(time_lt(fresh ? P.t : S.t, g.last))) {
        g.err = ECMC_ERR_SCHEDULER;
        return HOT_EVENT;
    }
    e.tagger = chosen;
    if (fresh || chosen == hot.boundary) {
        e.t = fresh ? P.t : B.p.t;
        e.target = P.target;
        e.adir = g.adir;
        e.aspeed = g.aspeed;
        e.cell = g.occ_cell;
        e.astamp = fresh ? P.t : g.at;
        e.cv_rate = 0.0;
        e.boundary = B.x;
#pragma unroll
        for (int d = 0; d < D; d++) e.tpos[d] = e.apos[d] = g.ap[d];
        if (fresh) {
            slice_pos<D>(q, e.apos, g.adir, g.aspeed, g.at, P.t);
            load_pos<RES>(a, q, P.target, e.tpos);
        }
    } else if ((FM & FEAT_CELL_VETO) && chosen == hot.veto) {
        wave_sync();
        event_of_slot<D, NT>(sh, chosen, e);
        e.t = S.t;
    } else {
        return HOT_STORED;
    }
    g.last = e.t;
    return HOT_EVENT;
}

// One workgroup runs one system's legs (the whole leg loop of the reference's mediator).
template <int D, int FM, int NT, bool RES>
__device__ __forceinline__ void chain_body(const ChainArgs &a) {
    __shared__ ChainShared<NT> sh;
    Geo<D> q;
    Leg<D> g;
    launch_load<D, NT, RES>(a, q, g, sh);
    const int wave = wave_index<NT>();
    HotList hot;
    hot.items = uni(sh.hot.items);
    hot.tags = (uint32_t)uni((int)sh.hot.tags);
    hot.boundary = uni(sh.hot.boundary);
    hot.veto = uni(sh.hot.veto);
    hot.before = uni(sh.hot.before);
    hot.veto_before = uni(sh.hot.veto_before);
    hot.hard = uni(sh.hot.hard);
    hot.radius = uni(sh.hot.radius);
    hot.mask = (uint32_t)uni((int)sh.hot.mask);
    hot.creators = (uint32_t)uni((int)sh.hot.creators);
    hot.prefixed = (uint32_t)uni((int)sh.hot.prefixed);
    hot.trashers = (uint32_t)uni((int)sh.hot.trashers);
    Items its;
    its.count = hot.items;
    its.tags = hot.tags;
    its.word = 0;
    its.rank = its.before = 0;
    {
        const int i = min((int)(threadIdx.x & 63), HOT_ITEMS - 1), t = item_tag(its, i);
        const ecmc_tagger_desc &tg = q.tg[t];
        const int test = (q.tests >> (2 * t)) & 3;
        its.p = sh.plan[t].p;
        its.rc2_hi = sh.plan[t].rc2_hi;
        its.set_key = sh.plan[t].set_key;
        its.pref = test == QT_INVERSE_POWER ? (float)tg.par[1] : (float)tg.bpar[0];
    }
    const int64_t max_events = a.max_events;
    ecmc_event *const log = a.log;
    const int stop_mask = a.stop_mask, occupancy = a.occupancy;
    auto rare = [&](int step, int arg, int from) {
        leg_to<D>(g, sh.leg[wave], sh.time[wave]);
        rare_step<D, FM, NT, RES>(&a, &sh, step, arg, from);
        leg_from<D>(sh.leg[wave], sh.time[wave], g);
    };
    Pick stored = pick_stored(g);
    int64_t k = 0;
#pragma unroll 1
    while (k < max_events) {
        if (g.done | g.err) break;
        const Time before = g.at;
        const int creator = g.last_tagger;
        g.committed = 0;
        int done = HOT_GENERAL, from = 0;
        Event<D> e;
        if (g.started && g.pending) {
            if (occupancy) occupancy_update<D, FM, NT, RES>(a, q, g, sh);
            else if (NT > 64) __syncthreads();   // the committed position, before others read it as a target
            if (g.err) break;
            g.ncand = 0;
            g.chash = 0;
            const bool prefixed = (hot.prefixed >> creator) & 1u;
            if (prefixed | ((hot.creators >> creator) & 1u)) {
                if (prefixed) {
                    from = uni(sh.plan[creator].n_create) - __popc(hot.mask);
                    rare(STEP_CREATE, creator, from);
                    if (g.err) break;
                }
                if (prefixed | (stored.w >= 0 && ((hot.mask >> stored.w) & 1u))) {
                    if ((hot.mask >> (threadIdx.x & 15)) & 1u) g.lvalid = 0;   // created anew
                    stored = pick_stored(g);
                }
                done = hot_events<D, FM, NT, RES>(a, q, g, sh, hot, its, stored, log != nullptr, (int)(k & 1), e);
            }
        }
        int w;
        if (done == HOT_EVENT) {
            if (g.err) break;
            w = e.tagger;
            g.pending = 0;
            ecmc_event ev;
            commit_event<D, FM, NT, RES, true>(a, q, g, sh, e, ev);
            if (log && threadIdx.x == 0) log[k] = ev;
            g.last_tagger = w;
            const uint32_t trash = (uint32_t)uni((int)sh.plan[w].trash);
            if (stored.w >= 0 && ((trash >> stored.w) & 1u)) {
                if ((trash >> (threadIdx.x & 15)) & 1u) g.lvalid = 0;
                stored = pick_stored(g);
            } else if (trash & ~hot.mask) {
                if ((trash >> (threadIdx.x & 15)) & 1u) g.lvalid = 0;
            }
        } else {
            if (done == HOT_STORED) rare(STEP_COMMIT, e.tagger, 0);
            else if (!g.started) rare(STEP_START, 0, 0);
            else rare(STEP_LEG, g.pending ? creator : -1, from);
            if (!g.committed) break;
            w = g.last_tagger;
            if (log && threadIdx.x == 0) log[k] = sh.ev;
            stored = pick_stored(g);
        }
        // the mean over about 16 legs of the time a leg takes
        const double step = time_sub(g.last, before);
        const double mean = g.mean_step > 0.0 ? g.mean_step + (step - g.mean_step) * 0.0625 : step;
        g.mean_step = step >= 0.0 && step < 0x1p60 ? mean : g.mean_step;
        g.pending = 1;
        k++;
        if (stop_mask & (1 << w)) break;
    }
    if (threadIdx.x == 0) *a.n_out = k;
    launch_store<D, NT, RES>(a, q, g, sh);
}

// Independent systems: workgroup b runs system b (its own positions, cell occupancy, random stream
// and state), its arguments read in place from device memory.  The full kernel of two
// dimensions leaves out what only three-dimensional systems have (the Coulomb machinery).
template <int D, int FM, int NT, bool RES>
__global__ __launch_bounds__(NT) void chain_kernel(const ChainArgs *__restrict__ args) {
    chain_body<D, D == 2 ? FM & ~FEAT_EWALD : FM, NT, RES>(args[blockIdx.x]);
}

// One step of a leg driven from the host, for the set-level event handler (the mediator and
// its scheduler stay on the host, the state and the candidate sets on the device):
//   op 0  the start of a leg: the cell occupancy follows the active unit and the candidate
//         statistics restart (the activator's internal-state update, tag_activator.py:205-226);
//   op 1  send_event_time of tagger t's handlers: its candidates' times, the earliest kept in
//         slot t (time, target, in-state copies);
//   op 2  send_out_state of tagger t's stored event, committed to the state; *out receives it.
template <int D, int FM, int NT>
__global__ __launch_bounds__(NT) void chain_step_kernel(const ChainArgs *__restrict__ args, int op, int t, ecmc_event *out) {
    constexpr int F = D == 2 ? FM & ~FEAT_EWALD : FM;
    const ChainArgs &a = *args;
    __shared__ ChainShared<NT> sh;
    Geo<D> q;
    Leg<D> g;
    launch_load<D, NT, false>(a, q, g, sh);
    if (op <= 1) {
        // the occupancy follows the active unit in op 1 too (a no-op after op 0 in the same leg), so
        // that a cell tagger never reads the cell of a unit that stopped being active
        if (a.occupancy && g.active >= 0) occupancy_update<D, F, NT, false>(a, q, g, sh);
        if (op == 0) {
            g.ncand = 0;
            g.chash = 0;
        } else if (!g.err) {
            const int kind = kind_of(q.kinds, t);
            Counts cn;
            cn.nb = cn.far = -1;
            if (kind == ECMC_TAG_CELL_BOUNDARY) {
                Boundary b;
                b.p.w = -1;
                create_boundary<D, NT>(a, q, g, sh, t, b);
                if (!g.err) store_boundary<D, NT>(g, sh, b);
            } else if (pair_kind(kind)) {
                create_pair_full<D, F, NT, false>(a, q, g, sh, t, kind, cn, true);
            } else {
                create_single<D, F, NT, false>(a, q, g, sh, t, kind);
            }
        }
    } else {
        Event<D> e;
        event_of_slot<D, NT>(sh, t, e);
        e.t = uni(sh.slot[t].t);
        ecmc_event ev;
        commit_event<D, F, NT, false, false>(a, q, g, sh, e, ev);
        g.last = e.t;
        if (threadIdx.x == 0) *out = ev;
    }
    launch_store<D, NT, false>(a, q, g, sh);
}

}  // namespace ecmc
