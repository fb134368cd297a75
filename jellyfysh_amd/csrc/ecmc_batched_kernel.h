// ecmc_batched_kernel.h -- device code of the batched replicas (see ecmc_batched.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/jellyfysh_amd.h"
#include "ecmc_math.h"
#include "ecmc_potentials.h"
#include "ecmc_fp32_bounds.h"

namespace ecmc {

constexpr int B_MAX_WPR = 8;
constexpr int B_CONTENDERS = 48;     // contenders per leg (about 7 typical; beyond, all candidates go exact)
constexpr int B_QUEUE = 256;         // per-wavefront queue of candidates past the capsule test (63 left + 3 x 64)
constexpr int B_MAX_CPS = 8;         // cells per side handled in LDS (512 cells)
// the chunk start counts units per cell in the (then idle) contender and queue area
static_assert(36 * B_CONTENDERS + 2 * B_QUEUE >= 4 * B_MAX_CPS * B_MAX_CPS * B_MAX_CPS, "cell counts do not fit");

struct ReplicaDev {
    int32_t n, cps;
    int64_t off;           // offset of the replica's SoA rows in pos64 (3 * n doubles)
    double L, cutoff, side;
    int32_t bound_off, pad;
    // state
    int32_t active, direction;
    double chain_left;
    uint64_t leg;
    double est[8];
    int32_t err, pad2;
    int64_t stats[4];      // candidates, geometric survivors, contenders, exact evaluations
};

struct FactorDev {
    int32_t n_factors, pad;
    double power[2], prefactor[2];
};

struct BatchArgs {
    ReplicaDev *rep;
    double *pos64;
    const double *bounds;        // cell lower bounds, per replica cps+1 entries
    const int32_t *order;        // replica indices of this class, largest first
    int32_t *state;              // per class member: (chunks done << 1) | held
    int32_t count;               // replicas in this class
    int32_t nmax, cellmax;       // LDS sizing of this class
    int32_t legs;                // legs per replica of this step
    int32_t chunk_legs, nchunks; // a work item is one chunk of legs of one replica
    int32_t mode;                // 0 filtered, 1 all candidates exact, 2 filtered + audit
    int32_t log_legs;            // legs logged per replica (0 = none)
    uint32_t seed_lo, pad;
    double beta, chain_length;
    FactorDev fac;
    int32_t *queue;              // [0] claim cursor
    ecmc_batch_event *log;       // n_replicas x log_legs
    unsigned long long *audit;   // bound violations
};

// ---- Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) --------------------------------
__device__ __forceinline__ void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                                              uint32_t k1, uint32_t out[4]) {
#pragma unroll
    for (int r = 0; r < 10; r++) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0, n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c0 = n0; c1 = (uint32_t)p1; c2 = n2; c3 = (uint32_t)p0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

__device__ __forceinline__ double unit53(uint32_t a, uint32_t b) {
    return ((a >> 5) * 67108864.0 + (b >> 6)) * (1.0 / 9007199254740992.0);
}

__device__ __forceinline__ double bmin_image(double s, double L) {
    if (s >= 0.5 * L) return s - L;
    if (s < -0.5 * L) return s + L;
    return s;
}

__device__ __forceinline__ int bcell1(double x, double side, int cps) {
    int c = (int)(x / side);
    return c < cps ? c : cps - 1;
}

// ---- FP32 lower bound of the truncated inverse-power event displacement ------------------
// (the bracketing helpers up, dn, rcp1, sqrt_up, sqrt_dn and dU_lower are in ecmc_fp32_bounds.h)

// 1 / r2^(p/2) with p in {6, 12} (integer powers by multiplication), bounded up (hi) or down for
// an r2 that is itself a lower/upper bound.  At most four products (2^-24 each), K's conversion
// and K * rcp(rp) (3 x 2^-24) stay inside an 8 x 2^-24 allowance, to which ETA is added; the two
// factors are one constant, (1 +- 2^-21)(1 +- 2^-17) without its 2^-38 term (the side that
// widens the bound), applied with one more rounding.
__device__ __forceinline__ float vpow_bound(float K, float r2, bool twelve, bool hi) {
    float r3 = r2 * r2 * r2;
    float rp = twelve ? r3 * r3 : r3;
    float v = K * rcp1(rp);
    return v * (hi ? 1.f + 0x1p-17f + 0x1p-21f : 1.f - 0x1p-17f - 0x1p-21f);
}

// A candidate's separation as pass 1 bounds it: along the motion (sd_lo <= sd <= sd_hi), squared
// across it, squared in all.
struct Reach {
    float sd_lo, sd_hi, perp2_lo, perp2_hi;
};

// True when the factor surely has no event within the displacement hf, given the exponential
// draw's lower bound dU_lo.  An event within hf means that the truncated energy rises by the draw
// on the way there, and the energy rises on one stretch only:
//   repulsive (k > 0)  a unit ahead, from the start (or the cutoff sphere) to the closest approach
//                      or hf: rise = V(nearest) - max(V(start), V(rc)), V = k / r^p;
//   attractive         from the closest approach (or the start, for a unit behind) to hf or the
//                      cutoff: rise = V(nearest) - max(V(at hf), V(rc)), V = |k| / r^p.
// Bounded up with the nearest distance from below and the farther one from above; no power or
// logarithm has to be inverted for it (a bound on the displacement itself takes two exp2/log2
// pairs and a root per factor).  Infinite or
// NaN bounds (a nearest distance of zero) keep the candidate.
__device__ __forceinline__ bool factor_surely_later(const Reach &g, float k, bool twelve, float rc2_hi, float vrc_lo, float hf,
                                                    float dU_lo) {
    const bool rep = k > 0.f;
    const float K = fabsf(k);
    const float x_near = fmaxf(rep ? g.sd_lo - hf : -g.sd_hi, 0.f);
    const float x_far = rep ? fmaxf(fabsf(g.sd_lo), fabsf(g.sd_hi)) : hf - g.sd_lo;
    const float near2 = dn(fmaf(x_near, x_near, g.perp2_lo)), far2 = up(fmaf(x_far, x_far, g.perp2_hi));
    const float low = fmaxf(vpow_bound(K, far2, twelve, false), vrc_lo);
    const float rise = vpow_bound(K, near2, twelve, true) - low;
    return (near2 >= rc2_hi) | (rep ? g.sd_hi <= 0.f : g.sd_lo > hf) | (up(rise) < dU_lo);
}

// dU_lower (ecmc_fp32_bounds.h) without its branch: u24 below 2^-10, else the hardware logarithm
// that log2f is for a normal argument (1 - u24 >= 2^-24), less its error bound.
__device__ __forceinline__ float dU_lower_flat(uint32_t a, float inv_beta_lo) {
    const float u24 = (float)(a >> 8) * 0x1p-24f;
    const float ml2 = -__builtin_amdgcn_logf(1.f - u24);
    const float l = (ml2 - LOG2F_ERR * fmaxf(ml2, 1.f)) * 0x1.62e42ep-1f;
    return fmaxf((u24 < 0x1p-10f ? u24 : l) * inv_beta_lo * (1.f - 0x1p-20f), 0.f);
}

// A value that is alike in all lanes, as a scalar.
__device__ __forceinline__ int buni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t buni(uint64_t v) {
    return (uint64_t)(uint32_t)buni((int)(uint32_t)v) | ((uint64_t)(uint32_t)buni((int)(uint32_t)(v >> 32)) << 32);
}

// The launch arguments, read again from the kernel's argument segment: what a leg needs of them
// seldom is then not held in scalar registers (or spilled to lanes) through the leg.
typedef double __attribute__((address_space(1))) gdouble;   // global memory
typedef const BatchArgs __attribute__((address_space(4))) BatchArgsRef;
__device__ __forceinline__ BatchArgsRef &again() {
    uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(BatchArgsRef *)p;
}

struct BKey {
    double d;
    int32_t rank, j, f;
};
__device__ __forceinline__ bool bkey_lt(const BKey &a, const BKey &b) {
    if (a.d != b.d) return a.d < b.d;
    if (a.rank != b.rank) return a.rank < b.rank;
    if (a.j != b.j) return a.j < b.j;
    return a.f < b.f;
}
__device__ __forceinline__ bool bkey_eq(const BKey &a, const BKey &b) {
    return a.d == b.d && a.rank == b.rank && a.j == b.j && a.f == b.f;
}

// One step of the (displacement, key) minimum across lanes with a DPP lane permutation of
// the 16-lane row (CTRL: 0xB1 swaps neighbours, 0x4E pairs of neighbours, 0x141 mirrors each
// half row, 0x140 the row), in registers.
template <int CTRL>
__device__ __forceinline__ void dpp_min_step(double &d, int &k) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(d), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(d), CTRL, 0xF, 0xF, false);
    const int ok = __builtin_amdgcn_update_dpp(0, k, CTRL, 0xF, 0xF, false);
    const double od = __hiloint2double(hi, lo);
    if (od < d || (od == d && ok < k)) { d = od; k = ok; }
}

// The leg's event over the workgroup: the minimum over lanes of (displacement, packed (kind,
// target, factor)), then LDS across wavefronts (one barrier).  With one wavefront per replica
// the first 16 lanes reduce by DPP and the other rows join only when more than 16 lanes hold
// keys (nlive: lanes beyond hold +inf), the result taken from lane 0, and the returned index
// is the lane holding the winning key (keys are unique; 0 unless a pair wins), from which the
// caller reads the candidate's position; with several, a shuffle butterfly, the winning lane
// of each wavefront leaves that candidate's FP64 position in newpos[3 * wave] and its slot in
// newslot[wave], and the returned index is the winning wavefront.
template <int WPR>
__device__ int block_min(BKey &b, const BKey &mine, const double *pos, int slot, BKey *sk, double *newpos, int *newslot, int nlive) {
    // (rank, j, f) packed into one word orders like the triple (rank < 4, j < 2^27, f < 2)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double d = b.d;
    int k = (b.rank << 28) | (b.j << 1) | b.f;
    if (WPR == 1) {
        dpp_min_step<0xB1>(d, k);
        dpp_min_step<0x4E>(d, k);
        dpp_min_step<0x141>(d, k);
        dpp_min_step<0x140>(d, k);
        if (nlive > 16) {
#pragma unroll
            for (int off = 16; off <= 32; off <<= 1) {
                const double od = __shfl_xor(d, off, 64);
                const int ok = __shfl_xor(k, off, 64);
                if (od < d || (od == d && ok < k)) { d = od; k = ok; }
            }
        }
        d = __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(d)),
                             __builtin_amdgcn_readfirstlane(__double2loint(d)));
        k = __builtin_amdgcn_readfirstlane(k);
        b.d = d;
        b.rank = k >> 28;
        b.j = (k >> 1) & 0x7ffffff;
        b.f = k & 1;
        const unsigned long long wm = __ballot(b.rank == 0 && bkey_eq(mine, b));
        return wm ? __ffsll((long long)wm) - 1 : 0;
    } else {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const double od = __shfl_xor(d, off, 64);
            const int ok = __shfl_xor(k, off, 64);
            if (od < d || (od == d && ok < k)) { d = od; k = ok; }
        }
    }
    b.d = d;
    b.rank = k >> 28;
    b.j = (k >> 1) & 0x7ffffff;
    b.f = k & 1;
    if (b.rank == 0 && bkey_eq(mine, b)) {
        newpos[3 * wave] = pos[0];
        newpos[3 * wave + 1] = pos[1];
        newpos[3 * wave + 2] = pos[2];
        newslot[wave] = slot;
    }
    int wb = 0;
    if (WPR > 1) {
        if (lane == 0) sk[wave] = b;
        __syncthreads();
        b = sk[0];
#pragma unroll
        for (int w = 1; w < WPR; w++)
            if (bkey_lt(sk[w], b)) {
                b = sk[w];
                wb = w;
            }
    }
    return wb;
}

__device__ __forceinline__ void bsync() { __syncthreads(); }

// Factor-indexed values held in registers (a runtime index into a private array would put
// the array in scratch memory).
template <class T>
__device__ __forceinline__ T pick(int f, T v0, T v1) { return f ? v1 : v0; }

// Exact FP64 event displacement of one truncated-and-shifted inverse-power factor
// (k / r^p - k / rc^p inside rc), p = 12 (six: r^p = (r^2)^6) or 6, for separation s (target
// minus active, minimum image) along +d with unit speed: the values of ipt_displacement (and
// so of the oracle), each pow correctly rounded.  The repulsive (k > 0) and attractive forms
// run as one instruction stream with selects, so lanes of a wavefront evaluating different
// factors do not diverge; sum(v ** 2 for v in others) is also the maximum potential's
// squared distance (the d component set to zero adds an exact 0).  urc = k / rc^p.
#ifndef ECMC_BATCHED_WAVES_PER_SIMD
#define ECMC_BATCHED_WAVES_PER_SIMD 2   // waves per SIMD the register allocation must allow (VGPRs <= 256)
#endif
struct SlowMath {   // correctly rounded for every argument
    __device__ __forceinline__ double pow36(double x, bool six) { return ecmc::pow36(x, six); }
    __device__ __forceinline__ double root36(double x, bool six) { return ecmc::root36(x, six); }
};
struct FastMath {   // the fast paths alone: ok turns false where they do not settle the rounding
    bool ok = true;
    __device__ __forceinline__ double pow36(double x, bool six) { return pow36_settled(x, six, ok); }
    __device__ __forceinline__ double root36(double x, bool six) { return root36_settled(x, six, ok); }
};
template <class Math>
__device__ __forceinline__ double exact_ipt(Math &m, double s0, double s1, double s2, int d, bool six, double prefactor,
                                            double rc2, double urc, double dU) {
    const double perp2 = d == 0 ? s1 * s1 + s2 * s2 : (d == 1 ? s0 * s0 + s2 * s2 : s0 * s0 + s1 * s1);
    const bool rep = prefactor > 0.0;
    const double sd = d == 0 ? s0 : (d == 1 ? s1 : s2);
    // attractive: a unit ahead is first passed (its closest approach is at s[d] = 0)
    const bool shift = !rep && sd > 0.0;
    const double disp = shift ? sd : 0.0;
    const double sdd = shift ? 0.0 : sd;
    const double c0 = d == 0 ? sdd : s0, c1 = d == 1 ? sdd : s1, c2 = d == 2 ? sdd : s2;
    const double sn2 = (0.0 + c0 * c0 + c1 * c1) + c2 * c2;
    bool live = perp2 < rc2 && (rep ? sd > 0.0 : sn2 < rc2);
    const double cur = (rep && !(sn2 < rc2)) ? urc : prefactor / m.pow36(live ? sn2 : 1.0, six);
    const double maxp = prefactor / m.pow36(rep && live ? perp2 : 1.0, six);
    live = live && (rep ? dU < maxp - cur : !(cur + dU >= urc));
    const double nsq = m.root36(live ? prefactor / (cur + dU) : 1.0, six);
    const double a = nsq - perp2;
    const double sq = sqrt(fmax(a, 0.0));
    const double res = a < 0.0 ? NAN : (rep ? sdd - sq : disp + (sdd + sq));
    return live ? res : INFINITY;
}

// The exact FP64 event displacement of one contender: the exponential draw dU = -log(1 - u) /
// beta from its two words (correctly rounded log), then exact_ipt.  The fast paths of the
// correctly rounded functions run inlined; the few arguments that they leave open (about one in
// 500, by the logarithm) take the call, whose registers the leg loop does not hold.
__device__ __noinline__ double exact_event_slow(uint32_t wa, uint32_t wb, double beta, double s0, double s1, double s2, int d,
                                                bool six, double prefactor, double rc2, double urc) {
    const double dU = -cr_log(1.0 - unit53(wa, wb)) / beta;
    SlowMath m;
    return exact_ipt(m, s0, s1, s2, d, six, prefactor, rc2, urc, dU);
}
__device__ __forceinline__ double exact_event(uint32_t wa, uint32_t wb, double beta, double s0, double s1, double s2, int d,
                                              bool six, double prefactor, double rc2, double urc) {
    FastMath m;
    const double dU = -log_settled(1.0 - unit53(wa, wb), m.ok) / beta;
    double dx = exact_ipt(m, s0, s1, s2, d, six, prefactor, rc2, urc, dU);
    if (__builtin_expect(!m.ok, 0)) dx = exact_event_slow(wa, wb, beta, s0, s1, s2, d, six, prefactor, rc2, urc);
    return dx;
}

// Positions in LDS: 16-bit fixed point per coordinate, q = round(x 2^16 / L) mod 2^16 (x in
// [0, L)), with the unit's number in one 8-byte record (x | y << 16, z | unit << 16), the records
// sorted by cell.  The separation q_j - q_a wrapped into [-2^15, 2^15) is the minimum image
// exactly in integers (the wrap is that of 16-bit subtraction); times L 2^-16 it is within
// L 2^-16 (two roundings of L 2^-17) plus L 2^-25 (the float product) of the true minimum-image
// separation, unless that is within the same distance of +-L/2.  The slack E = L 2^-15 (two
// steps) covers both.  One read of a record follows the candidate's place directly; three arrays
// by unit behind a list of units by cell cost four reads in two dependent steps.
__device__ __forceinline__ uint32_t quant1(double x, double inv_step) { return (uint32_t)(x * inv_step + 0.5) & 0xFFFFu; }
typedef unsigned short bushort2 __attribute__((ext_vector_type(2)));
typedef short bshort2 __attribute__((ext_vector_type(2)));
struct Sep {
    float x, y, z;   // in steps of L 2^-16, exact
};
__device__ __forceinline__ Sep qsep(uint2 rec, uint32_t qa01, uint32_t qa2) {
    const bshort2 xy = __builtin_bit_cast(bshort2, __builtin_bit_cast(bushort2, rec.x) - __builtin_bit_cast(bushort2, qa01));
    const short z = (short)(rec.y - qa2);
    return Sep{(float)xy.x, (float)xy.y, (float)z};
}
__device__ __forceinline__ bool qsep_ambiguous(const Sep &s) {   // within 2E of +-L/2 on some axis
    return fmaxf(fmaxf(fabsf(s.x), fabsf(s.y)), fabsf(s.z)) >= 32764.f;
}

// The separation's bounds with the position slack E.
__device__ __forceinline__ Reach cand_reach(const Sep &s, int d, float step, float E) {
    Reach g;
    const float sd = (d == 0 ? s.x : (d == 1 ? s.y : s.z)) * step;
    g.sd_lo = sd - E;
    g.sd_hi = sd + E;
    const float u = fabsf(d == 0 ? s.y : s.x) * step, v = fabsf(d == 2 ? s.y : s.z) * step;
    const float ul = fmaxf(u - E, 0.f), vl = fmaxf(v - E, 0.f), uh = u + E, vh = v + E;
    g.perp2_lo = dn(fmaf(ul, ul, vl * vl));
    g.perp2_hi = up(fmaf(uh, uh, vh * vh));
    return g;
}

// Pre-filter of pass 1 on the fixed-point separation (dx, dy, dz): false only for a candidate
// that no factor can reach within the horizon h.  Every candidate with an event at most h
// away lies within rc of the segment [0, h] along the axis of motion: a repulsive factor has
// no event before its unit enters the cutoff sphere (ahead), an attractive one none for a
// unit behind beyond the cutoff (its distance only grows) and none ahead before the closest
// approach (at s_d <= h).  The fixed-point separation is within E of the true one on each
// axis, so within sqrt(3) E < 2E of it; hq >= h and RQ2 >= (rc + 2E)^2, both in steps.  The
// squared distance is taken as |s|^2 - s_d^2 + e^2, exact but for float roundings of terms below
// 3 x 2^30: RQ2 holds 2^11 for them.  A separation within 2E of +-L/2 on any axis (minimum image
// not certain) always passes; check_amb false (uniform) skips that test where no such separation
// can lie in the capsule.
__device__ __forceinline__ bool cand_near(const Sep &s, int d, float RQ2, float hq, bool check_amb) {
    const float sd = d == 0 ? s.x : (d == 1 ? s.y : s.z);
    const float e = sd - fminf(fmaxf(sd, 0.f), hq);
    const float r2 = fmaf(s.x, s.x, fmaf(s.y, s.y, s.z * s.z));
    const bool near = fmaf(e, e, r2 - sd * sd) < RQ2;
    return check_amb ? near | qsep_ambiguous(s) : near;
}

// Records sorted by cell: move record x, at slot p of cell X's segment, to cell Y != X
// (one wavefront, uniform arguments).  Going up (Y > X), x leaves through X's last slot (X's
// last unit fills p), every non-empty cell between passes its last unit to the slot before its
// first, and x becomes Y's first; going down is the mirror image.  Starts of the cells
// between, and of the far end, shift by one.  Each pass reads all its slots before it writes.
__device__ void csr_move(uint2 *cu, int16_t *cs, int p, int X, int Y, uint2 x, int lane) {
    if (Y > X) {
        const int eX = cs[X + 1] - 1;
        const uint2 vX = cu[eX];
        if (lane == 0 && p != eX) cu[p] = vX;
        for (int c0 = X + 1; c0 < Y; c0 += 64) {
            const int c = c0 + lane;
            uint2 v = {0u, 0u};
            int dst = -1;
            if (c < Y) {
                const int b = cs[c], e = cs[c + 1];
                if (e > b) {
                    v = cu[e - 1];
                    dst = b - 1;
                }
            }
            __builtin_amdgcn_wave_barrier();
            if (dst >= 0) cu[dst] = v;
        }
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) cu[cs[Y] - 1] = x;
        __builtin_amdgcn_wave_barrier();
        for (int c = X + 1 + lane; c <= Y; c += 64) cs[c] = (int16_t)(cs[c] - 1);
    } else {
        const int fX = cs[X];
        const uint2 vX = cu[fX];
        if (lane == 0 && p != fX) cu[p] = vX;
        // downwards, chunks from the top so that a chunk reads its slots before the chunk below
        // writes into them
        for (int c0 = X - 1; c0 > Y; c0 -= 64) {
            const int c = c0 - lane;
            uint2 v = {0u, 0u};
            int dst = -1;
            if (c > Y) {
                const int b = cs[c], e = cs[c + 1];
                if (e > b) {
                    v = cu[b];
                    dst = e;
                }
            }
            __builtin_amdgcn_wave_barrier();
            if (dst >= 0) cu[dst] = v;
        }
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) cu[cs[Y + 1]] = x;
        __builtin_amdgcn_wave_barrier();
        for (int c = Y + 1 + lane; c <= X; c += 64) cs[c] = (int16_t)(cs[c] + 1);
    }
}

// candidate idx -> slot (binary search over the 27 prefix sums; without cells the slots themselves)
__device__ __forceinline__ int candidate_slot(int idx, bool whole_box, const int *pref, const int *start) {
    if (whole_box) return idx;
    int lo = 0, hi = 27;  // pref[lo] <= idx < pref[hi]
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (pref[mid] <= idx) lo = mid;
        else hi = mid;
    }
    return start[lo] + (idx - pref[lo]);
}

// The nearby cells as runs of slots.  Cells are numbered along x first, so the three nearby cells
// of a row (one y and z) are one run of slots where the row does not wrap and two where it does:
// 9 or 18 runs, run k holding candidates first[k] <= idx < first[k + 1] at slots idx + shift[k].
// (Culled cells count as empty; a row's live cells always include its middle one or none, so the
// run's shift is the middle cell's.)  A candidate's run is found by comparing with every first
// in order: eight comparisons and selects without memory, against five dependent LDS reads of a
// binary search over 27 cells.
struct Runs {
    alignas(16) int first[20];
    alignas(16) int shift[20];
};
// Slots of the candidates idx[0 .. C) over R runs, in place.  (Every run is read once, before its
// compare: arrays of registers indexed by a select would end in scratch memory.)
template <int R, int C>
__device__ __forceinline__ void run_slots(const Runs &s, int (&idx)[C]) {
    int v[C];
    const int v0 = s.shift[0];
#pragma unroll
    for (int c = 0; c < C; c++) v[c] = v0;
#pragma unroll
    for (int k = 1; k < R; k++) {
        const int first = s.first[k], shift = s.shift[k];
#pragma unroll
        for (int c = 0; c < C; c++) v[c] = idx[c] >= first ? shift : v[c];
    }
#pragma unroll
    for (int c = 0; c < C; c++) idx[c] += v[c];
}

// LDS bytes of the dynamic part for a class (fixed-point positions, cell lists, contenders and
// the per-wavefront candidate queues); the host sizes launches with the same function.
__host__ __device__ inline size_t batched_lds_bytes(int nmax, int cellmax, int wpr) {
    size_t b = 8ull * nmax + 2ull * (cellmax + 1);
    b = (b + 7) & ~7ull;
    b += (24ull + 8ull + 4ull) * B_CONTENDERS;     // positions, random words, identifiers
    b += 2ull * B_QUEUE * wpr;
    return (b + 15) & ~15ull;
}

// One leg of a replica, for the workgroup that owns it:
//   1. horizon h = min(distance to the next cell wall, rest of the chain) (FP64);
//   2. pass 1a over every candidate: the fixed-point separation against the capsule of
//      radius rc about the segment of motion (cand_near); candidates outside are done, the
//      others are appended to the wavefront's queue (ballot compaction);
//   3. pass 1b over each full queue: FP32 geometry with the position slack, Philox draws (FP32
//      bound of dU from the draw's leading bits); a factor whose energy may rise by the draw
//      within h (factor_surely_later) is a contender;
//   4. pass 2, one contender per thread: its FP64 position from global memory, exact FP64
//      inversion with correctly rounded pow/log, workgroup min-reduce over (displacement,
//      kind, target, factor);
//   5. wavefront 0 commits.
// Bound by the instructions it issues: with two wavefronts per SIMD (LDS for the largest replica
// and 256 VGPRs) the VALU is busy 72% of the time.  1697 vector instructions a leg before the
// cell-sorted records, the runs, the energy test, the division-free cells and the inlined
// inversion, 1267 with them; 4096 replicas of 64 to 2048 units, 20 000 legs each: 343 -> 270 ms.
//
// CHECK: modes 1 and 2 (their own instance, so that the filtered mode's registers hold nothing of
// them).
template <int WPR, bool CHECK>
__global__ __launch_bounds__(64 * WPR, ECMC_BATCHED_WAVES_PER_SIMD) void batched_kernel(BatchArgs A) {
    const int mode = CHECK ? A.mode : 0;
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NTH = 64 * WPR;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint2 *cu = (uint2 *)smem;                    // records sorted by cell, the active unit left out
    int16_t *cs = (int16_t *)(cu + A.nmax);       // cell c holds cu[cs[c] .. cs[c + 1])
    size_t off = (8ull * A.nmax + 2ull * (A.cellmax + 1) + 7) & ~7ull;
    int32_t *ccount = (int32_t *)(smem + off);                        // 24 B x B_CONTENDERS: chunk-start cell counts
    uint32_t *cont_w = (uint32_t *)(smem + off + 24 * B_CONTENDERS);  // B_CONTENDERS x 2
    int32_t *cont_id = (int32_t *)(cont_w + 2 * B_CONTENDERS);       // (slot << 1) | f
    uint16_t *queue = (uint16_t *)(cont_id + B_CONTENDERS) + wave * B_QUEUE;   // slots
    __shared__ BKey sk[B_MAX_WPR];
    __shared__ int s_item, s_chunk, s_nc, s_overflow, s_nearby[27], s_pref[28], s_M, s_Mfull;
    __shared__ int s_preff[28];   // audit mode: prefix sums over every unit of the 27 cells (none culled)
    __shared__ double s_ap[3], s_newpos[3 * B_MAX_WPR], s_h, s_cb, s_bounds[B_MAX_CPS + 1];
    __shared__ int s_newslot[B_MAX_WPR];
    __shared__ Runs s_runs;
    __shared__ ReplicaDev R;
    __shared__ unsigned long long s_geo;   // geometric survivors of the other wavefronts (several per replica)

    for (;;) {
        // Claim a work item: a class member that no block holds and that has chunks left.  Wave
        // 0 probes the members 64 at a time from a rotating cursor and takes one with a
        // compare-and-swap; when none is free the block ends (the members left are held by
        // running blocks, which take them on).  Every probe is bounded, so the grid drains.
        if (wave == 0) {
            int got = -1, chunk = 0;
            const uint32_t start = (uint32_t)__shfl(lane == 0 ? atomicAdd(A.queue, 1) : 0, 0);
            for (int base = 0; base < A.count && got < 0; base += 64) {
                const int m = (int)((start + (uint32_t)(base + lane)) % (uint32_t)A.count);
                const bool in = base + lane < A.count;
                const int st = in ? __hip_atomic_load(A.state + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 1;
                uint64_t free_mask = __ballot(in && !(st & 1) && (st >> 1) < A.nchunks);
                while (free_mask && got < 0) {
                    const int l = __ffsll((unsigned long long)free_mask) - 1;
                    int won = 0;
                    if (lane == l) {
                        int expect = st;
                        won = __hip_atomic_compare_exchange_strong(A.state + m, &expect, st | 1, __ATOMIC_RELAXED,
                                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    if (__shfl(won, l)) {
                        got = __shfl(m, l);
                        chunk = __shfl(st >> 1, l);
                    }
                    free_mask &= free_mask - 1;
                }
            }
            if (lane == 0) {
                s_item = got;
                s_chunk = chunk;
                // acquire: the previous holder's stores (any XCD) are visible from here on
                if (got >= 0) __threadfence();
            }
        }
        bsync();
        const int member = buni(s_item);
        if (member < 0) break;
        const int r = buni(A.order[member]);
        if (tid == 0) {
            R = A.rep[r];
            s_geo = 0;
        }
        bsync();
        const int chunk = buni(s_chunk);
        const int legs_now = min(A.chunk_legs, A.legs - chunk * A.chunk_legs);
        const int n = buni(R.n), cps = buni(R.cps);
        const double L = R.L, side = R.side;
        gdouble *P = (gdouble *)buni((uint64_t)(A.pos64 + R.off));
        const double inv_step = 0x1p16 / L;
        auto record = [&](int i, double x, double y, double z) {
            return make_uint2(quant1(x, inv_step) | (quant1(y, inv_step) << 16), quant1(z, inv_step) | ((uint32_t)i << 16));
        };
        const int ncell = cps ? cps * cps * cps : 0;
        // counting sort of the units by cell; the counts and cursors live in the contender
        // area, which is idle here (4 * 512 bytes fit in it)
        for (int c = tid; c < ncell; c += NTH) ccount[c] = 0;
        if (tid < 3) s_ap[tid] = P[(size_t)tid * n + R.active];
        if (cps && tid <= cps) s_bounds[tid] = A.bounds[R.bound_off + tid];
        bsync();
        if (cps) {
            auto unit_cell = [&](int i) {
                return bcell1(P[i], R.side, cps) +
                       cps * (bcell1(P[(size_t)n + i], R.side, cps) + cps * bcell1(P[2 * (size_t)n + i], R.side, cps));
            };
            for (int i = tid; i < n; i += NTH)
                if (i != R.active) atomicAdd(&ccount[unit_cell(i)], 1);
            bsync();
            if (wave == 0) {
                // exclusive scan over the cells: each lane a run of up to 8, then across lanes
                const int per = (ncell + 63) / 64;
                int sum = 0;
                for (int k = 0; k < per; k++) {
                    const int c = lane * per + k;
                    if (c < ncell) sum += ccount[c];
                }
                int incl = sum;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int v = __shfl_up(incl, o, 64);
                    if (lane >= o) incl += v;
                }
                int run = incl - sum;
                for (int k = 0; k < per; k++) {
                    const int c = lane * per + k;
                    if (c < ncell) {
                        const int t = ccount[c];
                        cs[c] = (int16_t)run;
                        ccount[c] = run;
                        run += t;
                    }
                }
                if (lane == 63) cs[ncell] = (int16_t)incl;
            }
            bsync();
            for (int i = tid; i < n; i += NTH)
                if (i != R.active) cu[atomicAdd(&ccount[unit_cell(i)], 1)] = record(i, P[i], P[(size_t)n + i], P[2 * (size_t)n + i]);
        } else {
            for (int i = tid; i < n; i += NTH)
                if (i != R.active) cu[i < R.active ? i : i - 1] = record(i, P[i], P[(size_t)n + i], P[2 * (size_t)n + i]);
        }
        const float Lf = (float)L;
        const float step = (float)(L * 0x1p-16);
        const float E = Lf * 0x1p-15f;
        const double rc2 = R.cutoff * R.cutoff;
        const float rc2_hi = (float)rc2 * (1.f + 0x1p-22f);
        const int nf = A.fac.n_factors;
        // per-factor constants (the second factor's equal the first's when there is one factor)
        const double pw0 = A.fac.power[0], pw1 = nf > 1 ? A.fac.power[1] : pw0;
        const double pk0 = A.fac.prefactor[0], pk1 = nf > 1 ? A.fac.prefactor[1] : pk0;
        const double urc0 = pk0 / cr_pow(rc2, pw0 / 2.0), urc1 = pk1 / cr_pow(rc2, pw1 / 2.0);
        const float vrc0 = (float)fabs(urc0) * (1.f - 0x1p-20f), vrc1 = (float)fabs(urc1) * (1.f - 0x1p-20f);
        const float kf0 = (float)pk0, kf1 = (float)pk1;
        const int pf0 = (int)pw0, pf1 = (int)pw1;
        const float inv_beta_lo = (float)(1.0 / A.beta) * (1.f - 0x1p-22f);
        // pre-filter constants (cand_near), in steps: (rc + 2E)^2 rounded up
        const float RB = ((float)R.cutoff * (1.f + 0x1p-22f) + 2.f * E) * (1.f + 0x1p-20f);
        const float inv_stepf = (float)inv_step * (1.f + 0x1p-22f);
        const float RQ = RB * inv_stepf * (1.f + 0x1p-20f);
        const float RQ2 = RQ * RQ * (1.f + 0x1p-20f) + 0x1p11f;
        const float halfL = 0.5f * Lf, E2 = 2.f * E;
        // A separation within 2E of +-L/2 on some axis has |s_q| >= L/2 - 2E.  When that exceeds
        // the capsule's reach rc + 2E ahead of the largest horizon (the chain length, rounded
        // up as hf is), such a candidate fails the capsule test on either image, so neither
        // pass needs the ambiguity test.
        const float hf_max = (float)A.chain_length * (1.f + 0x1p-22f) + 0x1p-60f;
        const bool check_amb = !(halfL - E2 > (hf_max + RB) * (1.f + 0x1p-20f));
        // with 3 cells per side the 27 nearby cells are the whole box: candidate idx is slot idx
        const bool whole_box = cps == 0 || cps == 3;
        // Replica state through the chunk, in registers (with one wavefront per replica the LDS
        // copy R is only read at the start and written at the end; with several, wavefront 0
        // publishes it to LDS after each commit and every wavefront reloads it)
        int st_a = buni(R.active), st_d = buni(R.direction), st_err = buni(R.err);
        uint64_t st_leg = buni(R.leg);
        double st_cl = R.chain_left;
        double st_ap[3] = {s_ap[0], s_ap[1], s_ap[2]};
        double st_h = 0.0, st_cb = 0.0;
        int st_M = 0, st_pc[3] = {0, 0, 0};
        bool st_wrap = false;           // the rows of nearby cells wrap (18 runs)
        int ncell_at = 0, ncell_n = 0;  // lane k < 27: first slot and units of nearby cell k, its coordinates
        int ncell_c = 0;
        const int off0 = lane % 3 - 1, off1 = (lane / 3) % 3 - 1, off2 = lane / 9 - 1;
        if (cps && wave == 0) {
#pragma unroll
            for (int q = 0; q < 3; q++) st_pc[q] = buni(bcell1(st_ap[q], side, cps));
        }
        // Nearby cells that cannot meet the capsule of the next leg are left out of its candidate
        // list (their count is taken as zero): the box distance from the segment [0, h] (h
        // widened to cover hf) must be at least rc + 2E rounded up, plus 2E for the position
        // slack of the fixed-point test and L 2^-18 for the FP32 box bounds (each rounded once
        // from an FP64 difference below L, then a few FP32 operations).  Not in the all-FP64
        // mode (which inverts every candidate of the 27 cells) nor where the ambiguity tests
        // are on; the audit mode keeps it and checks every candidate of the 27 cells, culled
        // or not.  (The radius is recomputed in each call from the cutoff in LDS, so that it
        // does not hold a register through the leg.)
        const bool cull = mode != 1 && !check_amb;
        // the estimators, summed leg by leg in the oracle's order (wavefront 0)
        double dest[6] = {R.est[0], R.est[1], R.est[2], R.est[3], R.est[4], R.est[5]};
        unsigned long long dst[4] = {0ull, 0ull, 0ull, 0ull};  // statistics increments (wavefront 0)
        // The next leg's 27 nearby cells with an inclusive scan of their counts (not needed when
        // they are the whole box), its cell, horizon and candidate count, and cleared contender
        // counters: wavefront 0, before the first leg and right after each commit (so that no
        // separate barrier precedes pass 1)
        auto prepare_leg = [&](double pa0, double pa1, double pa2, int pc0, int pc1, int pc2, int dn_, double cl) {
            double hh = cl, cb = INFINITY;
            if (cps) {
                const int pcd = dn_ == 0 ? pc0 : (dn_ == 1 ? pc1 : pc2);
                cb = s_bounds[pcd + 1] - (dn_ == 0 ? pa0 : (dn_ == 1 ? pa1 : pa2));
                if (cb < hh) hh = cb;
            }
            int Mv = n - 1, Mf = n - 1;
            bool wrap = false;
            if (cps) {
                const int lim = lane < 27 ? 1 : 0;
                const int u0 = pc0 + off0, u1 = pc1 + off1, u2 = pc2 + (lane < 27 ? off2 : 0);
                const int c0 = u0 < 0 ? u0 + cps : (u0 >= cps ? u0 - cps : u0), c1 = u1 < 0 ? u1 + cps : (u1 >= cps ? u1 - cps : u1),
                          c2 = u2 < 0 ? u2 + cps : (u2 >= cps ? u2 - cps : u2);
                const int c = c0 + cps * (c1 + cps * c2);
                ncell_at = cs[c];
                ncell_n = (cs[c + 1] - ncell_at) * lim;
                ncell_c = c0 | (c1 << 4) | (c2 << 8);
            }
            if (cps && !whole_box) {
                bool live = true;
                if (cull) {
                    const float rb = ((float)R.cutoff * (1.f + 0x1p-22f) + 2.f * E) * (1.f + 0x1p-20f);
                    const float cull_r = (rb * (1.f + 0x1p-20f) + 2.f * E + Lf * 0x1p-18f) * (1.f + 0x1p-20f);
                    const float cull_r2 = cull_r * cull_r * (1.f + 0x1p-20f);
                    // the cell's box relative to the active unit (not wrapped: its image on that
                    // side), against the point 0 across the motion and the segment [0, h] along it
                    const float top = (float)hh * (1.f + 0x1p-20f) + 0x1p-50f, sidef = (float)side;
                    float g2 = 0.f;
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        const float lo = fmaf((float)(q == 0 ? pc0 + off0 : (q == 1 ? pc1 + off1 : pc2 + off2)), sidef,
                                              -(float)(q == 0 ? pa0 : (q == 1 ? pa1 : pa2)));
                        float gap = fmaxf(fmaxf(lo - (q == dn_ ? top : 0.f), -(lo + sidef)), 0.f);
                        // (a row's middle cell never is farther than its neighbours, see Runs)
                        if (q == 0) gap = off0 == 0 ? 0.f : gap;
                        g2 = fmaf(gap, gap, g2);
                    }
                    live = g2 < cull_r2;
                }
                // inclusive scans of the counts kept (low half) and of all (high half) in one word,
                // each sum below 2^15: within each 16-lane row by DPP row shifts (a lane whose
                // source is outside the row adds 0), then lanes 16-26 add row 0's sum
                const uint32_t own = (live ? (uint32_t)ncell_n : 0u) | ((uint32_t)ncell_n << 16);
                uint32_t incl = own;
                incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x111, 0xF, 0xF, false);
                incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x112, 0xF, 0xF, false);
                incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x114, 0xF, 0xF, false);
                incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x118, 0xF, 0xF, false);
                const uint32_t row0 = (uint32_t)__builtin_amdgcn_readlane((int)incl, 15);
                incl += lane >= 16 ? row0 : 0u;
                const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)incl, 26);
                Mv = (int)(all & 0xFFFFu);
                Mf = (int)(all >> 16);
                const int first = (int)((incl - own) & 0xFFFFu), shift = ncell_at - first;
                // the runs: column 0 of a row begins one, and so does a column after a wrap
                const bool wrap_lo = pc0 == 0, wrap_hi = pc0 == cps - 1;
                wrap = wrap_lo || wrap_hi;
                if (lane < 27) {
                    s_nearby[lane] = ncell_at;
                    s_pref[lane + 1] = (int)(incl & 0xFFFFu);
                    if (mode == 2) s_preff[lane + 1] = (int)(incl >> 16);
                    const int row = lane / 3, col = off0 + 1;
                    const int run = wrap ? 2 * row + (wrap_lo ? (col > 0) : (col > 1)) : row;
                    const bool begins = col == 0 || (wrap_lo && col == 1) || (wrap_hi && col == 2);
                    const bool speaks = col == 1 || (wrap_lo && col == 0) || (wrap_hi && col == 2);
                    if (begins) s_runs.first[run] = first;
                    if (speaks) s_runs.shift[run] = shift;
                }
            }
            st_h = hh;
            st_cb = cb;
            st_M = Mv;
            st_wrap = wrap;
            if (lane == 0) {
                s_nc = 0;
                s_overflow = 0;
                s_Mfull = Mf;   // the statistics count every candidate of the 27 cells
                if (WPR > 1) {
                    s_h = hh;
                    s_cb = cb;
                    s_M = Mv | (wrap ? 1 << 20 : 0);
                }
            }
        };
        if (tid == 0) s_pref[0] = s_preff[0] = 0;
        if (wave == 0) prepare_leg(st_ap[0], st_ap[1], st_ap[2], st_pc[0], st_pc[1], st_pc[2], st_d, st_cl);
        bsync();
        if (WPR > 1) {
            st_h = s_h;
            st_cb = s_cb;
            st_M = buni(s_M) & 0xFFFFF;
            st_wrap = buni(s_M) >> 20;
        }
        for (int leg_i = 0; leg_i < legs_now && !st_err; leg_i++) {
            const int a = st_a, d = st_d;
            const uint64_t leg = st_leg;
            const double ap[3] = {st_ap[0], st_ap[1], st_ap[2]};
            const int M = st_M;
            const double h = st_h;
            const uint32_t qa01 = quant1(ap[0], inv_step) | (quant1(ap[1], inv_step) << 16), qa2 = quant1(ap[2], inv_step);
            const float hf = (float)h * (1.f + 0x1p-22f) + 0x1p-60f;
            const float hq = hf * inv_stepf * (1.f + 0x1p-22f);
            BKey best = {INFINITY, 3, 0x7ffffff, 0};   // j < 2^27: the reduction packs (rank, j, f)
            double bestpos[3] = {0.0, 0.0, 0.0};
            int bestslot = 0;
            unsigned geo_pass = 0;   // geometric survivors of this wavefront (uniform)
            if (mode != 1) {
                // ---- pass 1b: bounds of the queued candidates of this wavefront
                int nc = 0;   // contenders so far (one wavefront per replica: uniform register)
                auto bound_queue = [&](const uint16_t *from, int cnt) {
                    const bool act = lane < cnt;
                    int j = 0;
                    uint32_t w[4] = {0u, 0u, 0u, 0u};
                    bool con[2] = {false, false};
                    if (act) {
                        j = from[lane];
                        const uint2 rec = cu[j];
                        const Sep s = qsep(rec, qa01, qa2);
                        const bool amb = check_amb && qsep_ambiguous(s);
                        const Reach g = cand_reach(s, d, step, E);
                        philox4x32_10((uint32_t)leg, (uint32_t)(leg >> 32), rec.y >> 16, 0u, (uint32_t)r, again().seed_lo, w);
#pragma unroll
                        for (int f = 0; f < 2; f++) {
                            if (f >= nf) break;
                            con[f] = amb | !factor_surely_later(g, pick(f, kf0, kf1), pick(f, pf0, pf1) == 12, rc2_hi, pick(f, vrc0, vrc1),
                                                                hf, dU_lower_flat(pick(f, w[0], w[2]), inv_beta_lo));
                        }
                    }
                    // contender slots: with one wavefront per replica from ballots over the whole
                    // (converged) wavefront, else from the workgroup's LDS counter
#pragma unroll
                    for (int f = 0; f < 2; f++) {
                        int slot;
                        if (WPR == 1) {
                            const unsigned long long m = __ballot(con[f]);
                            slot = nc + __popcll(m & ((1ull << lane) - 1ull));
                            nc += __popcll(m);
                            if (!con[f]) continue;
                        } else {
                            if (!con[f]) continue;
                            slot = atomicAdd(&s_nc, 1);
                        }
                        if (slot >= B_CONTENDERS) {
                            s_overflow = 1;
                            continue;
                        }
                        cont_id[slot] = (j << 1) | f;
                        cont_w[2 * slot] = pick(f, w[0], w[2]);
                        cont_w[2 * slot + 1] = pick(f, w[1], w[3]);
                    }
                };
                // ---- pass 1a: every candidate against the capsule, survivors queued; three
                // chunks of 64 per wavefront and iteration, so that their LDS reads (cell search,
                // unit, position) overlap
                int qn = 0;
                // C chunks of 64 candidates (a place past the end reads the last candidate again)
                auto near_chunks = [&](int base, auto chunks) {
                    constexpr int C = decltype(chunks)::value;
                    int j[C];
                    bool s[C];
#pragma unroll
                    for (int k = 0; k < C; k++) j[k] = min(base + k * NTH + lane, M - 1);
                    if (!whole_box) {
                        if (!st_wrap) run_slots<9, C>(s_runs, j);
                        else run_slots<18, C>(s_runs, j);
                    }
#pragma unroll
                    for (int k = 0; k < C; k++)
                        s[k] = cand_near(qsep(cu[j[k]], qa01, qa2), d, RQ2, hq, check_amb) & (base + k * NTH + lane < M);
#pragma unroll
                    for (int k = 0; k < C; k++) {
                        const unsigned long long m = __ballot(s[k]);
                        const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                        if (s[k]) queue[qn + before] = (uint16_t)j[k];
                        qn += __popcll(m);
                        geo_pass += (unsigned)__popcll(m);
                    }
                };
                for (int base = wave * 64;;) {
                    if (base + 2 * NTH < M) near_chunks(base, std::integral_constant<int, 3>{});
                    else if (base + NTH < M) near_chunks(base, std::integral_constant<int, 2>{});
                    else if (base < M) near_chunks(base, std::integral_constant<int, 1>{});
                    base += 3 * NTH;
                    const bool last = base >= M;
                    int done = 0;
                    for (; qn - done >= (last ? 1 : 64); done += 64) bound_queue(queue + done, min(qn - done, 64));
                    if (last) break;
                    const int rem = max(qn - done, 0);
                    const uint16_t v = queue[done + min(lane, 63)];
                    if (lane < rem) queue[lane] = v;
                    qn = rem;
                }
                if (WPR == 1 && lane == 0) s_nc = nc;
                bsync();
            }
            const int listed = buni(s_nc);
            const bool all_exact = mode == 1 || buni(s_overflow);
            // ---- pass 2: exact FP64 inversion of the contenders (or of every candidate)
            const int nwork = all_exact ? M * nf : min(listed, B_CONTENDERS);
            for (int w = tid; w < nwork; w += NTH) {
                int j, f, slot;
                double pj[3];
                uint32_t wa, wb;
                if (all_exact) {
                    f = w % nf;
                    const int idx = w / nf;
                    slot = candidate_slot(idx, whole_box, s_pref, s_nearby);
                    j = (int)(cu[slot].y >> 16);
                    pj[0] = P[j]; pj[1] = P[(size_t)n + j]; pj[2] = P[2 * (size_t)n + j];
                    uint32_t ww[4];
                    philox4x32_10((uint32_t)leg, (uint32_t)(leg >> 32), (uint32_t)j, 0u, (uint32_t)r, again().seed_lo, ww);
                    wa = pick(f, ww[0], ww[2]);
                    wb = pick(f, ww[1], ww[3]);
                } else {
                    slot = cont_id[w] >> 1;
                    f = cont_id[w] & 1;
                    j = (int)(cu[slot].y >> 16);
                    // the FP64 position from global memory (its latency overlaps the log of
                    // the draw inside exact_event)
                    pj[0] = P[j]; pj[1] = P[(size_t)n + j]; pj[2] = P[2 * (size_t)n + j];
                    wa = cont_w[2 * w];
                    wb = cont_w[2 * w + 1];
                }
                const double dx = exact_event(wa, wb, again().beta, bmin_image(pj[0] - ap[0], L), bmin_image(pj[1] - ap[1], L),
                                              bmin_image(pj[2] - ap[2], L), d, pick(f, pf0, pf1) == 12, pick(f, pk0, pk1),
                                              rc2, pick(f, urc0, urc1));
                BKey c = {dx, 0, j, f};
                if (bkey_lt(c, best)) {
                    best = c;
                    bestpos[0] = pj[0]; bestpos[1] = pj[1]; bestpos[2] = pj[2];
                    bestslot = slot;
                }
            }
            if (mode == 2) {
                // audit: every candidate of the 27 cells (or of the whole box), including those in
                // cells culled from the leg's list, whose exact displacement is <= h must be a
                // contender (before the selection's barrier: after it, wavefront 0 already
                // prepares the next leg)
                const int Ma = whole_box ? M : s_Mfull;
                for (int idx = tid; idx < Ma * nf; idx += NTH) {
                    const int f = idx % nf;
                    const int ci = idx / nf;
                    const int slot = candidate_slot(ci, whole_box, s_preff, s_nearby), j = (int)(cu[slot].y >> 16);
                    uint32_t ww[4];
                    philox4x32_10((uint32_t)leg, (uint32_t)(leg >> 32), (uint32_t)j, 0u, (uint32_t)r, again().seed_lo, ww);
                    const double dx = exact_event_slow(pick(f, ww[0], ww[2]), pick(f, ww[1], ww[3]), again().beta,
                                                  bmin_image(P[j] - ap[0], L), bmin_image(P[(size_t)n + j] - ap[1], L),
                                                  bmin_image(P[2 * (size_t)n + j] - ap[2], L), d, pick(f, pf0, pf1) == 12,
                                                  pick(f, pk0, pk1), rc2, pick(f, urc0, urc1));
                    if (dx <= h) {
                        bool found = false;
                        for (int q = 0; q < min(s_nc, B_CONTENDERS); q++)
                            if (cont_id[q] == ((slot << 1) | f)) found = true;
                        if (!found && !s_overflow) atomicAdd(again().audit, 1ull);
                    }
                }
            }
            BKey mine = best;
            if (tid == 0) {
                BKey c1k = {st_cb, 1, 0, 0};
                if (bkey_lt(c1k, best)) best = c1k;
                BKey c2k = {st_cl, 2, 0, 0};
                if (bkey_lt(c2k, best)) best = c2k;
            }
            const int wbest = block_min<WPR>(best, mine, bestpos, bestslot, sk, s_newpos, s_newslot, nwork);
            if (wave == 0) {
                dst[0] += (unsigned long long)buni(s_Mfull);   // every candidate of the 27 cells
                dst[2] += (unsigned long long)min(listed, B_CONTENDERS);
                dst[3] += (unsigned long long)nwork;
            }
            if (WPR == 1) dst[1] += geo_pass;
            else if (lane == 0 && geo_pass) atomicAdd(&s_geo, (unsigned long long)geo_pass);
            // ---- commit (wavefront 0; the winner's position is in the winning lane's registers
            // or, with several wavefronts, in s_newpos): the values below are uniform across the
            // wavefront, a ballot finds the new active unit's slot in its cell list, lane 0 writes
            if (wave == 0) {
                gdouble *Pw = P;
                // the cell on axis d after the move, from the cell's upper bound (the least double
                // whose quotient by the side lies in the next cell)
                double x;
                const int pc0 = st_pc[0], pc1 = st_pc[1], pc2 = st_pc[2];
                const double ap0 = ap[0], ap1 = ap[1], ap2 = ap[2], apd = d == 0 ? ap0 : (d == 1 ? ap1 : ap2);
                int pcd = d == 0 ? pc0 : (d == 1 ? pc1 : pc2);
                if (best.rank == 1) {
                    x = pcd + 1 < cps ? s_bounds[pcd + 1] : 0.0;
                    pcd = pcd + 1 < cps ? pcd + 1 : 0;
                } else {
                    x = apd + best.d;
                    const bool round = x >= L;
                    if (round) x -= L;
                    if (cps) pcd = round ? 0 : (x >= s_bounds[pcd + 1] ? pcd + 1 : pcd);
                }
                int newa = a;
                double np[3] = {d == 0 ? x : ap0, d == 1 ? x : ap1, d == 2 ? x : ap2};
                int pc[3] = {d == 0 ? pcd : pc0, d == 1 ? pcd : pc1, d == 2 ? pcd : pc2};
                const double pold[3] = {np[0], np[1], np[2]};
                const int ca = pc[0] + cps * (pc[1] + cps * pc[2]);
                int cn = 0, q = -1;
                if (best.rank == 0) {
                    newa = best.j;
                    if (WPR == 1) {
#pragma unroll
                        for (int k = 0; k < 3; k++)
                            np[k] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(bestpos[k]), wbest),
                                                     __builtin_amdgcn_readlane(__double2loint(bestpos[k]), wbest));
                        q = __builtin_amdgcn_readlane(bestslot, wbest);
                    } else {
                        np[0] = s_newpos[3 * wbest]; np[1] = s_newpos[3 * wbest + 1]; np[2] = s_newpos[3 * wbest + 2];
                        q = __builtin_amdgcn_readfirstlane(s_newslot[wbest]);
                    }
                    if (cps) {
                        // the nearby cell whose slots hold the new active unit
                        const unsigned long long in = __ballot((unsigned)(q - ncell_at) < (unsigned)ncell_n);
                        const int k = in ? __ffsll((long long)in) - 1 : 0;
                        const int c = __builtin_amdgcn_readlane(ncell_c, k);
                        pc[0] = c & 15; pc[1] = (c >> 4) & 15; pc[2] = c >> 8;
                        if (!in) q = -1;
                    }
                } else if (best.rank == 2) {
                    uint32_t w[4];
                    philox4x32_10((uint32_t)leg, (uint32_t)(leg >> 32), 0xFFFFFFFFu, 1u, (uint32_t)r, again().seed_lo, w);
                    newa = (int)(((uint64_t)w[0] * (uint64_t)n) >> 32);
                    if (newa != a) {
                        np[0] = Pw[newa]; np[1] = Pw[(size_t)n + newa]; np[2] = Pw[2 * (size_t)n + newa];
                        int from = 0, to = n - 1;
                        if (cps) {
#pragma unroll
                            for (int k = 0; k < 3; k++) pc[k] = __builtin_amdgcn_readfirstlane(bcell1(np[k], side, cps));
                            const int c = pc[0] + cps * (pc[1] + cps * pc[2]);
                            from = cs[c];
                            to = cs[c + 1];
                        }
                        for (int base = from; base < to && q < 0; base += 64) {
                            const unsigned long long mask = __ballot(base + lane < to && (int)(cu[min(base + lane, to - 1)].y >> 16) == newa);
                            if (mask) q = base + __ffsll((long long)mask) - 1;
                        }
                    }
                }
                cn = pc[0] + cps * (pc[1] + cps * pc[2]);
                // the replica's state, alike in every lane of wavefront 0
                const double np0 = np[0], np1 = np[1], np2 = np[2], npd = d == 0 ? np0 : (d == 1 ? np1 : np2);
                dest[1] += best.d;
                if (best.rank == 0) {
                    dest[0] += bmin_image(npd - apd, L) - best.d;
                    dest[2] += 1.0;
                    dest[4] += 1.0;
                    st_cl -= best.d;
                } else if (best.rank == 1) {
                    dest[3] += 1.0;
                    st_cl -= best.d;
                } else {
                    dest[5] += 1.0;
                    st_cl = again().chain_length;
                    st_d = (d + 1) % 3;
                }
                if (newa != a && q < 0) st_err = 2;
                st_a = newa;
                st_leg = leg + 1;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    st_ap[k] = np[k];
                    st_pc[k] = buni(pc[k]);
                }
                const uint2 old = record(a, pold[0], pold[1], pold[2]);
                if (lane == 0) {
                    Pw[(size_t)d * n + a] = x;
                    // the old active unit takes the new one's slot (and is moved to the cell it
                    // ended in below)
                    if (newa != a && q >= 0) cu[q] = old;
                    if (leg < (uint64_t)again().log_legs) {
                        ecmc_batch_event ev;
                        ev.kind = best.rank;
                        ev.active = a;
                        ev.target = best.rank == 0 ? best.j : (best.rank == 2 ? newa : -1);
                        ev.factor = best.rank == 0 ? best.f : 0;
                        ev.displacement = best.d;
                        ev.x = x;
                        again().log[(size_t)r * again().log_legs + leg] = ev;
                    }
                    if (WPR > 1) {
                        R.active = st_a;
                        R.direction = st_d;
                        R.leg = st_leg;
                        R.chain_left = st_cl;
                        R.err = st_err;
                        s_ap[0] = np[0]; s_ap[1] = np[1]; s_ap[2] = np[2];
                    }
                }
                // lane 0's LDS writes above precede the other lanes' reads below (one wavefront,
                // LDS operations in order; the fence keeps the compiler from reordering them)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (newa != a && cps && q >= 0 && ca != cn) {
                    csr_move(cu, cs, q, cn, ca, old, lane);
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                }
                prepare_leg(st_ap[0], st_ap[1], st_ap[2], st_pc[0], st_pc[1], st_pc[2], st_d, st_cl);
            }
            bsync();
            if (WPR > 1) {
                st_a = buni(R.active);
                st_d = buni(R.direction);
                st_leg = buni(R.leg);
                st_cl = R.chain_left;
                st_err = buni(R.err);
                st_ap[0] = s_ap[0]; st_ap[1] = s_ap[1]; st_ap[2] = s_ap[2];
                st_h = s_h;
                st_cb = s_cb;
                st_M = buni(s_M) & 0xFFFFF;
                st_wrap = buni(s_M) >> 20;
            }
        }
        if (tid == 0) {
            R.active = st_a;
            R.direction = st_d;
            R.leg = st_leg;
            R.chain_left = st_cl;
            R.err = st_err;
            for (int q = 0; q < 6; q++) R.est[q] = dest[q];
            R.stats[0] += (int64_t)dst[0];
            R.stats[1] += (int64_t)(dst[1] + s_geo);
            R.stats[2] += (int64_t)dst[2];
            R.stats[3] += (int64_t)dst[3];
            again().rep[r] = R;
        }
        bsync();   // every store of this chunk (positions, log, state) has completed
        if (tid == 0) {
            // release: make this block's stores visible device-wide, then free the member with
            // one more chunk done
            // (an exchange, whose return is awaited, so this block's next probe sees the update)
            __threadfence();
            const int prev = __hip_atomic_exchange(again().state + member, (chunk + 1) << 1, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
            if (prev != ((chunk << 1) | 1)) again().rep[r].err = 3;   // the claim protocol was broken
        }
    }
}

}  // namespace ecmc
