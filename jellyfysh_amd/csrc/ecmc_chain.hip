// ecmc_chain.hip -- event chains advanced on the GPU, leg after leg, one persistent workgroup per
// chain (the plain form): host side, kernel variants and table kernels; the leg loop itself is in
// ecmc_chain_leg.h.
//
// A leg follows the reference mediator (mediator/single_process_mediator.py:84-156):
//   update the cell occupancy for the active unit, run the event handlers of the taggers in
//   the `create` list of the tagger that committed last (tag_activator.py:228-289), take the
//   earliest stored candidate, build and commit its out-state, and trash by tag
//   (tag_activator.py:291-316).
//
// Mapping to the hardware:
//   * the candidates of a create list's pair taggers are spread over the workgroup in canonical
//     order (nearby cells in itertools.product order, occupants in list order; excluded_cells_
//     tagger.py:129-132); positions, the random ring, charges and cell lists are read from LDS
//     where the launch placed them, else from HBM;
//   * each candidate's exponential draw is the 2 MT19937 words at its rank in the stream; the
//     ring holds the MT19937 sequence itself, extended by one wavefront 192 words at a time, so the
//     draws are those of CPython's random in the reference's call order;
//   * an FP32 test leaves the few candidates that can decide the leg, which are inverted exactly
//     in FP64, one per lane;
//   * the scheduler keeps, per tagger, the earliest of its pushed events (all events of one
//     tagger are trashed together), and ties go to the first pushed event as in
//     list_scheduler.py:129-156;
//   * the sequential bookkeeping runs redundantly in every wavefront;
//   * the leg loop is compiled once per feature set (FEAT_*) and workgroup size, and each launch
//     runs the smallest variant that covers its systems.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <math.h>
#include <vector>
#include <string>
#include <atomic>
#include <mutex>
#include <utility>
#include <cmath>

#include "../../include/jellyfysh_amd.h"
#include "ecmc_math.h"
#include "ecmc_potentials.h"
#include "ecmc_fp32_bounds.h"
#include "ecmc_chain_leg.h"
#include "ecmc_common.h"

namespace ecmc {

constexpr int NT = 256;   // workgroup size of the table kernels
constexpr double ONE_WAVE_CANDIDATES = 96.0;   // pair candidates of a leg up to which one wavefront runs a system

// The terms of ewald_derivative in its loop order, as the codes of ewald_derivative_wave.
static std::vector<int32_t> ewald_term_codes(int fc, int pc) {
    std::vector<int32_t> out;
    for (int k = -pc; k < pc + 1; k++) {
        const int cy = (int)sqrt((double)(pc * pc - k * k));
        for (int j = -cy; j < cy + 1; j++) {
            const int cx = (int)sqrt((double)(pc * pc - j * j - k * k));
            for (int i = -cx; i < cx + 1; i++) out.push_back(((i + 128) << 16) | ((j + 128) << 8) | (k + 128));
        }
    }
    for (int i = 1; i < fc + 1; i++) {
        const int cy = (int)sqrt((double)(fc * fc - i * i));
        for (int j = 0; j < cy + 1; j++) {
            const int cx = (int)sqrt((double)(fc * fc - i * i - j * j));
            for (int k = 0; k < cx + 1; k++) out.push_back((1 << 24) | ((i + 128) << 16) | ((j + 128) << 8) | (k + 128));
        }
    }
    return out;
}

// InnerPointEstimator.derivative_bound (inner_point_estimator.py:108-171) for the cell
// separations of cell_bounding_potential.py:100-126: one workgroup per (cell, direction)
// evaluates the merged-image Coulomb derivative on the (pps + 1)^3 grid spanning the corners
// (corners[6c .. 6c+6] = lower[3], upper[3]; NaN marks a nearby separation).
__global__ __launch_bounds__(NT) void cell_bound_kernel(Ewald ew, const double *corners, double L, double pot_pref,
                                                        double target_charge, int pps, double est_pref, double emp,
                                                        double *out) {
    __shared__ double smax[NT], smin[NT];
    const int c = blockIdx.x / 3, dir = blockIdx.x % 3, t = threadIdx.x;
    const double *cr = corners + (size_t)c * 6;
    double *o = out + (size_t)blockIdx.x * 2;
    if (isnan(cr[0])) {
        if (t == 0) { o[0] = NAN; o[1] = NAN; }
        return;
    }
    const int np = pps + 1, total = np * np * np;
    const double half = L / 2.0;
    double mx = -INFINITY, mn = INFINITY;
    for (int k = t; k < total; k += NT) {
        const int ix = k / (np * np), iy = (k / np) % np, iz = k % np;
        double sep[3];
        sep[0] = cr[0] + (cr[3] - cr[0]) * ix / pps;
        sep[1] = cr[1] + (cr[4] - cr[1]) * iy / pps;
        sep[2] = cr[2] + (cr[5] - cr[2]) * iz / pps;
#pragma unroll
        for (int d = 0; d < 3; d++) sep[d] = py_mod(sep[d] + half, L) - half;   // correct_separation
        double der = pot_pref * 1.0 * target_charge * ewald_derivative(ew, sep[dir], sep[(dir + 1) % 3], sep[(dir + 2) % 3]);
        der = der * 1.0;
        if (der > mx) mx = der;
        if (der < mn) mn = der;
    }
    smax[t] = mx;
    smin[t] = mn;
    __syncthreads();
    for (int w = NT / 2; w > 0; w >>= 1) {
        if (t < w) {
            if (smax[t + w] > smax[t]) smax[t] = smax[t + w];
            if (smin[t + w] < smin[t]) smin[t] = smin[t + w];
        }
        __syncthreads();
    }
    if (t == 0) {
        double upper = smax[0], lower = smin[0];
        upper = upper > 0.0 ? upper * est_pref : upper / est_pref;
        lower = lower > 0.0 ? lower / est_pref : lower * est_pref;
        o[0] = upper < emp ? upper : emp;
        o[1] = lower > -emp ? lower : -emp;
    }
}

// ---- host side --------------------------------------------------------------------------
static void mt_seed_host(uint64_t seed, uint32_t *mt) {
    uint32_t key[2] = {(uint32_t)(seed & 0xffffffffu), (uint32_t)(seed >> 32)};
    int klen = key[1] ? 2 : 1;
    mt[0] = 19650218u;
    for (int i = 1; i < 624; i++) mt[i] = 1812433253u * (mt[i - 1] ^ (mt[i - 1] >> 30)) + (uint32_t)i;
    int i = 1, j = 0;
    for (int k = 624 > klen ? 624 : klen; k; k--) {
        mt[i] = (mt[i] ^ ((mt[i - 1] ^ (mt[i - 1] >> 30)) * 1664525u)) + key[j] + (uint32_t)j;
        i++; j++;
        if (i >= 624) { mt[0] = mt[623]; i = 1; }
        if (j >= klen) j = 0;
    }
    for (int k = 623; k; k--) {
        mt[i] = (mt[i] ^ ((mt[i - 1] ^ (mt[i - 1] >> 30)) * 1566083941u)) - (uint32_t)i;
        i++;
        if (i >= 624) { mt[0] = mt[623]; i = 1; }
    }
    mt[0] = 0x80000000u;
}

}  // namespace ecmc

using namespace ecmc;

// Walker's table (walker.py:73-101): small and large stacks split at the mean (sequential sum
// of the rates), one (small, alias large) entry per step with the large item's residual pushed
// back by comparison with the mean; the leftovers must lie within 1e-6 of the mean.
static bool walker_table(const std::vector<int32_t> &items, const std::vector<double> &rates, CvEntry *out,
                         double &total_out, double &mean_out) {
    const int m = (int)items.size();
    double total = 0.0;
    for (int i = 0; i < m; i++) total += rates[i];
    const double mean = total / m;
    std::vector<std::pair<int32_t, double>> small, large;
    for (int i = 0; i < m; i++) {
        if (!(rates[i] >= 0.0)) return false;
        if (rates[i] > mean) large.emplace_back(items[i], rates[i]);
        else small.emplace_back(items[i], rates[i]);
    }
    int k = 0;
    while (!small.empty() && !large.empty()) {
        const std::pair<int32_t, double> sm = small.back();
        small.pop_back();
        std::pair<int32_t, double> lg = large.back();
        large.pop_back();
        out[k++] = CvEntry{sm.second, sm.first, lg.first};
        lg.second -= mean - sm.second;
        if (lg.second < mean) small.push_back(lg);
        else large.push_back(lg);
    }
    for (std::vector<std::pair<int32_t, double>> *rest : {&small, &large}) {
        while (!rest->empty()) {
            const std::pair<int32_t, double> it = rest->back();
            rest->pop_back();
            const double q = it.second / mean;
            if (!(1 - 1e-6 < q && q < 1 + 1e-6)) return false;
            out[k++] = CvEntry{mean, it.first, -1};
        }
    }
    total_out = total;
    mean_out = mean;
    return k == m;
}

struct ecmc_system {
    ecmc_system_desc desc;
    int dim, n, ncells, nb_stride, occ_cap, ring_words;
    std::vector<double> cmin;
    double *d_pos = nullptr, *d_charge = nullptr, *d_cmin = nullptr, *d_ewald = nullptr;
    int32_t *d_ewald_codes = nullptr;
    int32_t *d_nearby = nullptr, *d_nearby_n = nullptr, *d_occ = nullptr, *d_occ_n = nullptr;
    int32_t *d_sur_cell = nullptr, *d_sur_id = nullptr;
    double *d_cbt = nullptr, *d_corners = nullptr;
    CvEntry *d_cvw = nullptr;
    uint32_t *d_ring = nullptr;
    ChainState *d_st = nullptr;
    ecmc_tagger_desc *d_tg = nullptr;
    ecmc_event *d_log = nullptr;
    int64_t log_cap = 0;
    int64_t *d_nout = nullptr;
    HostView *host = nullptr;          // pinned: what the last launch left for the host to read
    std::atomic<uint32_t> began{0}, ended{0};   // calls that launch: begun and ended (see read_host)
    ecmc_event *d_step_ev = nullptr;   // the event of the last host-driven commit
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_ms = 0.0;
    int32_t stop_mask = 0;
    int device = 0;          // the device current at creation, which holds its memory
    size_t lds_bytes = 0;    // dynamic LDS of a launch (positions and ring resident there)
    bool one_wave = false;   // few candidates a leg: workgroups of one wavefront
    int features = FEAT_ALL; // the kernel features the system uses (FEAT_*, potential bits)
    ChainArgs args;
    ChainArgs *d_args = nullptr;   // the arguments of the system's own launches, in device memory
};

// The kernel features a system's taggers use.
static int system_features(const ecmc_system_desc &d) {
    int f = 0;
    for (int t = 0; t < d.n_taggers; t++) {
        const ecmc_tagger_desc &tg = d.taggers[t];
        const bool pair = tg.kind == ECMC_TAG_PAIR_CELLS || tg.kind == ECMC_TAG_PAIR_ALL || tg.kind == ECMC_TAG_SURPLUS ||
                          tg.kind == ECMC_TAG_CELL_BOUNDING || tg.kind == ECMC_TAG_FACTOR_MAP;
        if (pair) {
            if (tg.event_handler == ECMC_EH_TWO_LEAF && tg.potential >= 0 && tg.potential < 9) f |= 1 << tg.potential;
            else if (tg.event_handler == ECMC_EH_TWO_LEAF_BOUNDING) f |= FEAT_COULOMB;
            else if (tg.event_handler == ECMC_EH_CELL_BOUNDING) f |= FEAT_CELL_BOUNDING;
            else f |= FEAT_ALL;
            if (tg.kind == ECMC_TAG_FACTOR_MAP) f |= FEAT_FMAP;
            if (tg.kind == ECMC_TAG_CELL_BOUNDING) f |= FEAT_CELL_BOUNDING;
        }
        if (tg.kind == ECMC_TAG_CELL_VETO) f |= FEAT_CELL_VETO;
    }
    return f;
}

// The kernel variants of the leg loop, in the order the host tries them (three dimensions; two
// dimensions run the full kernel): the first whose features cover a launch's runs it.
struct ChainVariant {
    int features;
    const void *one_wave, *four_waves, *global;   // resident systems with 64 and 256 threads, others
};
#define ECMC_VARIANT(D, FM) \
    {FM, reinterpret_cast<const void *>(&chain_kernel<D, FM, 64, true>), \
     reinterpret_cast<const void *>(&chain_kernel<D, FM, 256, true>), reinterpret_cast<const void *>(&chain_kernel<D, FM, 256, false>)}
static const ChainVariant CHAIN_VARIANTS_3D[] = {ECMC_VARIANT(3, VARIANT_LJ), ECMC_VARIANT(3, VARIANT_CHARGED_CB),
                                                 ECMC_VARIANT(3, VARIANT_CHARGED_CV), ECMC_VARIANT(3, VARIANT_DIPOLES),
                                                 ECMC_VARIANT(3, FEAT_ALL)};
static const ChainVariant CHAIN_VARIANTS_2D[] = {ECMC_VARIANT(2, FEAT_ALL)};
#undef ECMC_VARIANT
static const ChainVariant &chain_variant(int dim, int features) {
    if (dim == 2) return CHAIN_VARIANTS_2D[0];
    for (const ChainVariant &v : CHAIN_VARIANTS_3D)
        if ((features & ~v.features) == 0) return v;
    return CHAIN_VARIANTS_3D[sizeof(CHAIN_VARIANTS_3D) / sizeof(CHAIN_VARIANTS_3D[0]) - 1];
}

// Residency of a system: its positions, random ring, charges, occupant counts and surplus lists in
// the launch's dynamic LDS when they fit next to the kernel's static LDS within the device's
// per-workgroup limit, with as many occupants of every cell (16-bit) as fit after them; else
// everything stays in global memory.
static void plan_lds(ecmc_system *s) {
    int dev_max = 0;
    hipDeviceGetAttribute(&dev_max, hipDeviceAttributeMaxSharedMemoryPerBlock, s->device);
    const size_t stat = sizeof(ChainShared<256>) + 256;
    const size_t budget = dev_max > (int)stat ? (size_t)dev_max - stat : 0;
    bool charged = false;
    for (int t = 0; t < s->desc.n_taggers; t++) charged = charged || s->desc.taggers[t].use_charge;
    ChainArgs &a = s->args;
    a.resident = 0;
    a.lds_ring_off = a.lds_charge_off = a.lds_occ_off = a.lds_occn_off = a.lds_sur_off = -1;
    a.occ_cols = 0;
    s->lds_bytes = 0;
    if (s->n > 65536) return;   // the occupants are kept as 16-bit numbers
    size_t used = 0;
    auto place = [&](size_t bytes) -> int32_t {
        const size_t at = used;
        used += (bytes + 15) & ~(size_t)15;
        return (int32_t)at;
    };
    place((size_t)s->dim * s->n * sizeof(double));
    a.lds_ring_off = place((size_t)s->ring_words * sizeof(uint32_t));
    a.lds_tg_off = place((size_t)s->desc.n_taggers * sizeof(ecmc_tagger_desc));
    if (charged) a.lds_charge_off = place((size_t)s->n * sizeof(double));
    if (a.occupancy) {
        a.lds_occn_off = place((size_t)s->ncells * sizeof(int32_t));
        if (a.max_occ > 0) a.lds_sur_off = place((size_t)s->n * 2 * sizeof(int32_t));
    }
    if (used > budget) return;
    if (a.occupancy) {
        a.occ_cols = (int32_t)std::min<size_t>((size_t)s->occ_cap, (budget - used) / (2 * (size_t)s->ncells));
        if (a.occ_cols * 2 * (size_t)s->ncells + used + 16 > budget && a.occ_cols > 0) a.occ_cols--;
        a.lds_occ_off = place((size_t)s->ncells * a.occ_cols * sizeof(uint16_t));
    }
    if (used > 65536) {
        // every variant may run the system (a launch of several systems takes the variant that
        // covers all of them)
        const ChainVariant *vs = s->dim == 2 ? CHAIN_VARIANTS_2D : CHAIN_VARIANTS_3D;
        const size_t nv = s->dim == 2 ? sizeof(CHAIN_VARIANTS_2D) / sizeof(ChainVariant) : sizeof(CHAIN_VARIANTS_3D) / sizeof(ChainVariant);
        for (size_t i = 0; i < nv; i++)
            for (const void *f : {vs[i].one_wave, vs[i].four_waves})
                if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)used) != hipSuccess) {
                    (void)hipGetLastError();
                    return;
                }
    }
    a.resident = 1;
    s->lds_bytes = used;
}

// The kernel and workgroup size of a launch.
static const void *chain_launch(int dim, int features, bool resident, bool one_wave, dim3 &block) {
    const ChainVariant &v = chain_variant(dim, features);
    block = dim3(resident && one_wave ? 64 : 256);
    return !resident ? v.global : (one_wave ? v.one_wave : v.four_waves);
}

extern "C" int ecmc_system_set_stop_mask(ecmc_system *sys, int32_t mask) {
    if (!sys) return ecmc_fail(ECMC_ERR_ARGUMENT, "null system");
    sys->stop_mask = mask;
    return ECMC_OK;
}

// Cell-bound tables already built in this process, per device, keyed by everything they
// depend on (cell corners, box, potential and estimator parameters); the last eight are kept.
struct CellBoundCacheEntry {
    int device;
    std::vector<double> key, table;
};
static std::mutex g_cb_mutex;
static std::vector<CellBoundCacheEntry> g_cb_cache;

static bool cell_bound_cache_find(const std::vector<double> &key, std::vector<double> &table) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    std::lock_guard<std::mutex> lock(g_cb_mutex);
    for (const CellBoundCacheEntry &e : g_cb_cache)
        if (e.device == dev && e.key.size() == key.size() &&
            memcmp(e.key.data(), key.data(), sizeof(double) * key.size()) == 0) {
            table = e.table;
            return true;
        }
    return false;
}

static void cell_bound_cache_store(const std::vector<double> &key, const std::vector<double> &table) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    std::lock_guard<std::mutex> lock(g_cb_mutex);
    if (g_cb_cache.size() >= 8) g_cb_cache.erase(g_cb_cache.begin());
    g_cb_cache.push_back({dev, key, table});
}

// The host views of the live systems, in slabs of pinned memory: one device's views of one size, as many
// slots in a new slab as the slabs of that size already have (at most VIEW_SLAB bytes), so that a lone
// system takes one view and 256 of them ten allocations, of 50 to 130 us each, instead of 256.  A slab
// goes back to the system with its last view.
struct ViewSlab {
    int device;
    size_t bytes;                 // of one view
    int32_t slots;
    unsigned char *base, *seen;   // host address, and the device's
    std::vector<int32_t> free;
};
static std::mutex g_view_mutex;
static std::vector<ViewSlab> g_view_slabs;
constexpr size_t VIEW_SLAB = 1 << 20;

// A view of `bytes` for the current device, its device address in `seen`; null: pinned memory exhausted.
static HostView *take_view(int device, size_t bytes, HostView **seen) {
    bytes = (bytes + 255) & ~(size_t)255;
    std::lock_guard<std::mutex> lock(g_view_mutex);
    size_t at = g_view_slabs.size();
    int64_t have = 0;
    for (size_t k = 0; k < g_view_slabs.size(); k++) {
        const ViewSlab &v = g_view_slabs[k];
        if (v.device != device || v.bytes != bytes) continue;
        have += v.slots;
        if (!v.free.empty()) at = k;
    }
    if (at == g_view_slabs.size()) {
        ViewSlab v = {device, bytes, 0, nullptr, nullptr, {}};
        const int64_t most = std::max<int64_t>(1, (int64_t)(VIEW_SLAB / bytes));
        void *base = nullptr, *dev = nullptr;
        for (int64_t slots = std::min(std::max<int64_t>(1, have), most); slots > 0 && !base; slots = slots > 1 ? 1 : 0) {
            v.slots = (int32_t)slots;
            if (hipHostMalloc(&base, bytes * slots, hipHostMallocPortable | hipHostMallocMapped) != hipSuccess) {
                base = nullptr;
                (void)hipGetLastError();
            }
        }
        if (!base) return nullptr;
        if (hipHostGetDevicePointer(&dev, base, 0) != hipSuccess) {
            (void)hipGetLastError();
            hipHostFree(base);
            return nullptr;
        }
        v.base = (unsigned char *)base;
        v.seen = (unsigned char *)dev;
        for (int32_t i = v.slots; i-- > 0;) v.free.push_back(i);
        g_view_slabs.push_back(v);
    }
    ViewSlab &v = g_view_slabs[at];
    const size_t off = (size_t)v.free.back() * v.bytes;
    v.free.pop_back();
    *seen = (HostView *)(v.seen + off);
    return (HostView *)(v.base + off);
}

// Returns a view that no launch writes any more.
static void release_view(HostView *view) {
    unsigned char *const p = (unsigned char *)view, *empty = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_view_mutex);
        for (size_t k = 0; k < g_view_slabs.size(); k++) {
            ViewSlab &v = g_view_slabs[k];
            if (p < v.base || p >= v.base + v.bytes * v.slots) continue;
            v.free.push_back((int32_t)((p - v.base) / v.bytes));
            if ((int32_t)v.free.size() == v.slots) {
                empty = v.base;
                g_view_slabs.erase(g_view_slabs.begin() + k);
            }
            break;
        }
    }
    if (empty) hipHostFree(empty);
}

extern "C" int ecmc_system_create(const ecmc_system_desc *desc, const double *positions, const double *charges,
                                  ecmc_system **out) {
    if (!desc || !positions || !out) return ecmc_fail(ECMC_ERR_ARGUMENT, "null argument");
    *out = nullptr;
    const int dim = desc->dim, n = desc->n;
    if (dim != 2 && dim != 3) return ecmc_fail(ECMC_ERR_CONFIGURATION, "dimension must be 2 or 3");
    if (desc->rng_skip < 0) return ecmc_fail(ECMC_ERR_CONFIGURATION, "rng_skip must be >= 0");
    if (n < 2) return ecmc_fail(ECMC_ERR_CONFIGURATION, "at least two units are required");
    if (desc->n_taggers < 1 || desc->n_taggers > ECMC_MAX_TAGGERS)
        return ecmc_fail(ECMC_ERR_CONFIGURATION, "number of taggers out of range");
    if (desc->neighbor_layers < 0 || desc->neighbor_layers > 1)
        return ecmc_fail(ECMC_ERR_CONFIGURATION, "neighbor_layers must be 0 or 1");
    const int P = desc->leaves_per_root > 1 ? desc->leaves_per_root : 1;
    if (P > ECMC_MAX_LEAVES) return ecmc_fail(ECMC_ERR_CONFIGURATION, "more leaf units per composite object than ECMC_MAX_LEAVES");
    if (n % P != 0) return ecmc_fail(ECMC_ERR_CONFIGURATION, "the number of units is not a multiple of leaves_per_root");
    int ewald_tagger = -1, cb_tagger = -1;
    for (int t = 0; t < desc->n_taggers; t++) {
        const ecmc_tagger_desc &tg = desc->taggers[t];
        if (tg.kind < 0 || tg.kind > ECMC_TAG_FACTOR_MAP) return ecmc_fail(ECMC_ERR_CONFIGURATION, "unknown tagger kind");
        // with composite objects the cells hold leaf units (cell_level 2): the excluded-cells and
        // cell-boundary taggers work on leaf units as on point masses; the others are not built
        if (P > 1 && (tg.kind == ECMC_TAG_PAIR_ALL || tg.kind == ECMC_TAG_SURPLUS || tg.kind == ECMC_TAG_CELL_BOUNDING ||
                      tg.kind == ECMC_TAG_CELL_VETO))
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "with composite objects the pair taggers are factor-type-map and excluded-cells taggers");
        if (tg.kind == ECMC_TAG_FACTOR_MAP) {
            int fmax = 0;
            for (int k = 0; k < P; k++) {
                if (tg.fmap_n[k] < 0 || tg.fmap_n[k] > ECMC_MAX_FACTOR_MAP)
                    return ecmc_fail(ECMC_ERR_CONFIGURATION, "factor type map entries out of range");
                fmax = tg.fmap_n[k] > fmax ? tg.fmap_n[k] : fmax;
                for (int e = 0; e < tg.fmap_n[k]; e++) {
                    const int tl = tg.fmap_target[k][e];
                    const bool ok = tg.fmap_local ? (tl >= 0 && tl < P && tl != k) : (tl >= P && tl < 2 * P);
                    if (!ok) return ecmc_fail(ECMC_ERR_CONFIGURATION, "factor type map leaf number out of range");
                }
            }
            const int64_t m = tg.fmap_local ? fmax : (int64_t)(n / P - 1) * fmax;
            if (!tg.fmap_local && n / P < 2) return ecmc_fail(ECMC_ERR_CONFIGURATION, "a non-local factor needs two composite objects");
            if (tg.n_handlers > 0 && tg.n_handlers < m)
                return ecmc_fail(ECMC_ERR_TAG_ACTIVATOR, "not-running event handler list would run empty");
        }
        if ((tg.kind == ECMC_TAG_CELL_VETO) != (tg.event_handler == ECMC_EH_CELL_VETO))
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "the cell-veto handler runs under the cell-veto tagger only");
        if (tg.kind == ECMC_TAG_SURPLUS && desc->max_occupants <= 0)
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "the surplus tagger needs a bounded cell occupancy");
        if ((tg.kind == ECMC_TAG_CELL_BOUNDING) != (tg.event_handler == ECMC_EH_CELL_BOUNDING))
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "the cell-bounding handler runs under the cell-bounding tagger only");
        if (tg.kind == ECMC_TAG_CELL_BOUNDING || tg.kind == ECMC_TAG_CELL_VETO) {
            if (tg.potential != ECMC_POT_MERGED_IMAGE_COULOMB || tg.bounding_potential != ECMC_POT_CELL_BOUNDING || dim != 3)
                return ecmc_fail(ECMC_ERR_CONFIGURATION, "cell bounding needs merged-image Coulomb with the cell bounding potential in 3D");
            if (desc->max_occupants != 1)
                return ecmc_fail(ECMC_ERR_CONFIGURATION, "cell bounding needs maximum_number_occupants = 1");
            if (!(tg.bpar[0] > 0.0) || tg.bpar[1] < 1.0 || tg.bpar[1] > 64.0 || (tg.use_charge && tg.bpar[2] == 0.0))
                return ecmc_fail(ECMC_ERR_CONFIGURATION, "estimator prefactor, points_per_side or target_charge out of range");
            if (cb_tagger >= 0) {
                const ecmc_tagger_desc &o = desc->taggers[cb_tagger];
                for (int q = 0; q < 4; q++)
                    if (o.bpar[q] != tg.bpar[q] || o.par[q] != tg.par[q])
                        return ecmc_fail(ECMC_ERR_CONFIGURATION, "one cell-bounding parameter set per system");
            }
            cb_tagger = t;
            if (ewald_tagger >= 0) {
                const ecmc_tagger_desc &o = desc->taggers[ewald_tagger];
                if (o.par[0] != tg.par[0] || o.par[1] != tg.par[1] || o.par[2] != tg.par[2])
                    return ecmc_fail(ECMC_ERR_CONFIGURATION, "one merged-image Coulomb parameter set per system");
            }
            ewald_tagger = t;
        }
        if (tg.n_create < 0 || tg.n_create > ECMC_MAX_TAGGERS || tg.n_trash < 0 || tg.n_trash > ECMC_MAX_TAGGERS)
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "create/trash list length out of range");
        if (tg.kind == ECMC_TAG_START_OF_RUN &&
            (tg.ivalue < 0 || tg.ivalue >= dim || tg.ivalue2 < 0 || tg.ivalue2 >= n || !(tg.value > 0.0)))
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "initial direction, active identifier or speed out of range");
        if (tg.kind == ECMC_TAG_END_OF_CHAIN && !(tg.value > 0.0))
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "chain_time must be > 0.0");
        if (tg.kind == ECMC_TAG_SAMPLING && !(tg.value > 0.0))
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "sampling_interval must be > 0.0");
        for (int i = 0; i < tg.n_create; i++)
            if (tg.create[i] < 0 || tg.create[i] >= desc->n_taggers) return ecmc_fail(ECMC_ERR_CONFIGURATION, "create tag out of range");
        for (int i = 0; i < tg.n_trash; i++)
            if (tg.trash[i] < 0 || tg.trash[i] >= desc->n_taggers) return ecmc_fail(ECMC_ERR_CONFIGURATION, "trash tag out of range");
        if (tg.kind == ECMC_TAG_PAIR_CELLS || tg.kind == ECMC_TAG_PAIR_ALL || tg.kind == ECMC_TAG_SURPLUS ||
            tg.kind == ECMC_TAG_FACTOR_MAP) {
            if (tg.event_handler == ECMC_EH_TWO_LEAF_BOUNDING) {
                if (tg.potential != ECMC_POT_MERGED_IMAGE_COULOMB || tg.bounding_potential != ECMC_POT_INVERSE_POWER_COULOMB_BOUND || dim != 3)
                    return ecmc_fail(ECMC_ERR_CONFIGURATION, "bounding handler needs merged-image Coulomb with the inverse-power Coulomb bound in 3D");
                if (ewald_tagger >= 0) {
                    const ecmc_tagger_desc &o = desc->taggers[ewald_tagger];
                    if (o.par[0] != tg.par[0] || o.par[1] != tg.par[1] || o.par[2] != tg.par[2])
                        return ecmc_fail(ECMC_ERR_CONFIGURATION, "one merged-image Coulomb parameter set per system");
                }
                ewald_tagger = t;
            } else if (tg.potential == ECMC_POT_MERGED_IMAGE_COULOMB || tg.potential == ECMC_POT_INVERSE_POWER_COULOMB_BOUND) {
                return ecmc_fail(ECMC_ERR_CONFIGURATION, "the Coulomb potentials are not invertible here");
            }
            if (tg.n_handlers > 0 && tg.n_handlers < n - 1 && tg.kind == ECMC_TAG_PAIR_ALL)
                return ecmc_fail(ECMC_ERR_TAG_ACTIVATOR, "not-running event handler list would run empty");
        }
    }
    ecmc_system *s = new ecmc_system();
    s->desc = *desc;
    s->features = system_features(*desc);
    if (hipGetDevice(&s->device) != hipSuccess) {
        delete s;
        return ecmc_fail(ECMC_ERR_HIP, "no current HIP device");
    }
    s->dim = dim;
    s->n = n;
    CellGrid grid;
    std::string err;
    if (!build_cell_grid(dim, desc->system_length, desc->cells_per_side, desc->neighbor_layers, grid, err)) {
        delete s;
        return ecmc_fail(ECMC_ERR_CONFIGURATION, err.c_str());
    }
    s->ncells = grid.count;
    s->nb_stride = grid.nb_stride;
    // initial occupancy in global-state order (single_active_cell_occupancy.py:111-121)
    std::vector<std::vector<int32_t>> lists(grid.count);
    std::vector<int32_t> sur_cell, sur_id;     // the surplus dict, flattened in its yield order
    for (int i = 0; i < n; i++) {
        int c = grid.position_to_cell(positions + (size_t)i * dim);
        if (c < 0) { delete s; return ecmc_fail(ECMC_ERR_STATE, "initial position outside of the cell system"); }
        if (desc->max_occupants <= 0 || (int)lists[c].size() < desc->max_occupants) {
            lists[c].push_back(i);
        } else {
            size_t at = sur_cell.size();
            for (size_t k = sur_cell.size(); k-- > 0;)
                if (sur_cell[k] == c) { at = k + 1; break; }
            sur_cell.insert(sur_cell.begin() + at, c);
            sur_id.insert(sur_id.begin() + at, i);
        }
    }
    size_t maxocc = 0;
    for (auto &l : lists) maxocc = l.size() > maxocc ? l.size() : maxocc;
    int cap = (int)(maxocc * 4 + 32);
    if (cap > n) cap = n;
    s->occ_cap = cap;
    std::vector<int32_t> occ((size_t)grid.count * cap, -1), occ_n(grid.count);
    for (int c = 0; c < grid.count; c++) {
        occ_n[c] = (int32_t)lists[c].size();
        for (size_t i = 0; i < lists[c].size(); i++) occ[(size_t)c * cap + i] = lists[c][i];
    }
    std::vector<double> pos_soa((size_t)dim * n);
    for (int i = 0; i < n; i++)
        for (int d = 0; d < dim; d++) pos_soa[(size_t)d * n + i] = positions[(size_t)i * dim + d];
    std::vector<double> ch(n, 1.0);
    if (charges) for (int i = 0; i < n; i++) ch[i] = charges[i];
    // the pair candidates of a leg, about: all other units, the surplus, the occupants of the nearby
    // cells, the occupied far cells, the entries of a factor type map
    double words = 0.0, typical = 0.0;
    for (int t = 0; t < desc->n_taggers; t++) {
        const ecmc_tagger_desc &tg = desc->taggers[t];
        double m = 0.0;
        if (tg.kind == ECMC_TAG_PAIR_ALL) m = n;
        else if (tg.kind == ECMC_TAG_SURPLUS) m = (double)sur_id.size();
        else if (tg.kind == ECMC_TAG_PAIR_CELLS) m = std::min((double)n, (double)grid.nb_stride * (n - (double)sur_id.size()) / grid.count);
        else if (tg.kind == ECMC_TAG_CELL_BOUNDING) m = (double)n - (double)sur_id.size();
        else if (tg.kind == ECMC_TAG_FACTOR_MAP) {
            int fmax = 0;
            for (int k = 0; k < P; k++) fmax = std::max(fmax, tg.fmap_n[k]);
            m = tg.fmap_local ? fmax : (double)(n / P - 1) * fmax;
        }
        typical += m;
        if (tg.event_handler == ECMC_EH_TWO_LEAF_BOUNDING ||
            (tg.potential != ECMC_POT_HARD_SPHERE && tg.potential != ECMC_POT_HARD_DIPOLE)) words += 2.0 * m;
    }
    s->one_wave = typical <= ONE_WAVE_CANDIDATES;
    // the ring: the words of two legs and the generator's 624 (a leg that needs more evaluates its
    // candidates in segments), a power of two so that indices wrap with a mask, at most 16384 words
    // (8192 beside large position arrays, so that both fit into LDS)
    s->ring_words = 2048;
    const int ring_max = (size_t)dim * n * sizeof(double) > 65536 ? 8192 : 16384;
    while (s->ring_words < ring_max && (double)s->ring_words < 2.0 * words + 1600.0) s->ring_words <<= 1;
    uint32_t mt[624];
    mt_seed_host(desc->seed, mt);
    ChainState st;
    memset(&st, 0, sizeof(st));
    st.cursor = (uint64_t)desc->rng_skip;   // words drawn before the run (random input handler)
    st.active = -1;
    st.aspeed = 1.0;
    st.occ_id = -1;
    st.occ_cell = -1;
    st.last.q = -INFINITY;
    st.last.r = -INFINITY;
    st.nsur = (int32_t)sur_cell.size();
    for (int t = 0; t < desc->n_taggers; t++) {
        st.slot[t].valid = 0;
        const ecmc_tagger_desc &tg = desc->taggers[t];
        if (tg.kind == ECMC_TAG_SAMPLING && tg.ivalue) {
            Time z = time_from_float(-tg.value);
            st.samp_time = z;
        }
    }
    std::vector<double> ewald;
    std::vector<int32_t> ewald_codes;
    ChainArgs &a = s->args;
    memset(&a, 0, sizeof(a));
    if (ewald_tagger >= 0) {
        const ecmc_tagger_desc &tg = desc->taggers[ewald_tagger];
        int fc = (int)tg.par[1], pc = (int)tg.par[2];
        double alpha = tg.par[0], L = desc->system_length;
        build_ewald_table(fc, alpha, L, ewald);
        ewald_codes = ewald_term_codes(fc, pc);
        a.ewald.fc = fc;
        a.ewald.pc = pc;
        a.ewald.L = L;
        a.ewald.aol = alpha / L;
        a.ewald.aol2 = alpha * alpha / (L * L);
        a.ewald.two_aol_rpi = 2.0 * alpha / (L * sqrt(M_PI));
        a.ewald.tpol = 2.0 * M_PI / L;
    }
#define ECMC_ALLOC(ptr, bytes) \
    if (hipMalloc((void **)&(ptr), (bytes)) != hipSuccess) { ecmc_system_destroy(s); return ecmc_fail(ECMC_ERR_HIP, "hipMalloc failed"); }
#define ECMC_UP(dst, src, bytes) \
    if (hipMemcpy((dst), (src), (bytes), hipMemcpyHostToDevice) != hipSuccess) { ecmc_system_destroy(s); return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy failed"); }
    ECMC_ALLOC(s->d_pos, sizeof(double) * dim * n);
    ECMC_ALLOC(s->d_args, sizeof(ChainArgs));
    ECMC_ALLOC(s->d_charge, sizeof(double) * n);
    ECMC_ALLOC(s->d_cmin, sizeof(double) * grid.cmin.size());
    ECMC_ALLOC(s->d_nearby, sizeof(int32_t) * grid.nearby.size());
    ECMC_ALLOC(s->d_nearby_n, sizeof(int32_t) * grid.nearby_n.size());
    ECMC_ALLOC(s->d_occ, sizeof(int32_t) * occ.size());
    ECMC_ALLOC(s->d_occ_n, sizeof(int32_t) * occ_n.size());
    ECMC_ALLOC(s->d_ring, sizeof(uint32_t) * s->ring_words);
    ECMC_ALLOC(s->d_st, sizeof(ChainState));
    ECMC_ALLOC(s->d_tg, sizeof(ecmc_tagger_desc) * ECMC_MAX_TAGGERS);
    ECMC_ALLOC(s->d_nout, sizeof(int64_t));
    ECMC_ALLOC(s->d_step_ev, sizeof(ecmc_event));
    if (!ewald.empty()) { ECMC_ALLOC(s->d_ewald, sizeof(double) * ewald.size()); }
    if (!ewald_codes.empty()) { ECMC_ALLOC(s->d_ewald_codes, sizeof(int32_t) * ewald_codes.size()); }
    ECMC_ALLOC(s->d_sur_cell, sizeof(int32_t) * n);
    ECMC_ALLOC(s->d_sur_id, sizeof(int32_t) * n);
    if (!sur_cell.empty()) {
        ECMC_UP(s->d_sur_cell, sur_cell.data(), sizeof(int32_t) * sur_cell.size());
        ECMC_UP(s->d_sur_id, sur_id.data(), sizeof(int32_t) * sur_id.size());
    }
    ECMC_UP(s->d_pos, pos_soa.data(), sizeof(double) * dim * n);
    ECMC_UP(s->d_charge, ch.data(), sizeof(double) * n);
    ECMC_UP(s->d_cmin, grid.cmin.data(), sizeof(double) * grid.cmin.size());
    ECMC_UP(s->d_nearby, grid.nearby.data(), sizeof(int32_t) * grid.nearby.size());
    ECMC_UP(s->d_nearby_n, grid.nearby_n.data(), sizeof(int32_t) * grid.nearby_n.size());
    ECMC_UP(s->d_occ, occ.data(), sizeof(int32_t) * occ.size());
    ECMC_UP(s->d_occ_n, occ_n.data(), sizeof(int32_t) * occ_n.size());
    // the seeded state is words -624 .. -1 of the sequence
    std::vector<uint32_t> ring((size_t)s->ring_words, 0u);
    for (int i = 0; i < 624; i++) ring[s->ring_words - 624 + i] = mt[i];
    ECMC_UP(s->d_ring, ring.data(), sizeof(uint32_t) * ring.size());
    ECMC_UP(s->d_st, &st, sizeof(ChainState));
    ECMC_UP(s->d_tg, desc->taggers, sizeof(ecmc_tagger_desc) * ECMC_MAX_TAGGERS);
    if (!ewald.empty()) { ECMC_UP(s->d_ewald, ewald.data(), sizeof(double) * ewald.size()); }
    if (!ewald_codes.empty()) { ECMC_UP(s->d_ewald_codes, ewald_codes.data(), sizeof(int32_t) * ewald_codes.size()); }
#undef ECMC_ALLOC
#undef ECMC_UP
    if (hipStreamCreate(&s->stream) != hipSuccess || hipEventCreate(&s->ev0) != hipSuccess ||
        hipEventCreate(&s->ev1) != hipSuccess) {
        ecmc_system_destroy(s);
        return ecmc_fail(ECMC_ERR_HIP, "stream/event creation failed");
    }
    a.n = n;
    a.leaves = P;
    for (int t = 0; t < desc->n_taggers; t++) {
        const int k = desc->taggers[t].kind;
        if (k == ECMC_TAG_PAIR_CELLS || k == ECMC_TAG_SURPLUS || k == ECMC_TAG_CELL_BOUNDING || k == ECMC_TAG_CELL_VETO)
            a.occupancy = 1;
    }
    a.ncells = grid.count;
    a.nb_stride = grid.nb_stride;
    for (int d = 0; d < dim; d++)
        if (grid.cps[d] < 2 * desc->neighbor_layers + 1) a.nb_table = 1;
    a.occ_cap = cap;
    a.ring_words = s->ring_words;
    a.n_taggers = desc->n_taggers;
    a.L = desc->system_length;
    a.half = desc->system_length / 2.0;
    a.beta = desc->beta;
    for (int d = 0; d < 3; d++) {
        a.cps[d] = d < dim ? grid.cps[d] : 1;
        a.cum[d] = d < dim ? (int32_t)grid.cum[d] : 0;
        a.side[d] = d < dim ? grid.side[d] : 1.0;
    }
    a.pos = s->d_pos;
    a.charge = s->d_charge;
    a.cmin = s->d_cmin;
    a.nearby = s->d_nearby;
    a.nearby_n = s->d_nearby_n;
    a.occ = s->d_occ;
    a.occ_n = s->d_occ_n;
    a.ring = s->d_ring;
    a.st = s->d_st;
    a.tg = s->d_tg;
    a.ewald.f = s->d_ewald;
    a.ewald_codes = s->d_ewald_codes;
    a.ewald_ncodes = (int32_t)ewald_codes.size();
    for (int32_t c : ewald_codes) a.ewald_nreal += (c >> 24) == 0;
    a.n_out = s->d_nout;
    a.max_occ = desc->max_occupants;
    a.layers = desc->neighbor_layers;
    a.sur_cell = s->d_sur_cell;
    a.sur_id = s->d_sur_id;
    if (cb_tagger >= 0) {
        // cell-bound tables on the device (cell_bounding_potential.py:100-126)
        const ecmc_tagger_desc &tg = desc->taggers[cb_tagger];
        std::vector<double> corners((size_t)grid.count * 6);
        const int32_t *near0 = grid.nearby.data();
        for (int c = 0; c < grid.count; c++) {
            bool is_near = false;
            for (int k = 0; k < grid.nearby_n[0]; k++) if (near0[k] == c) is_near = true;
            for (int d = 0; d < 3; d++) {
                corners[(size_t)c * 6 + d] = is_near ? NAN : grid.cmin[(size_t)c * dim + d] - grid.cmax[d];
                corners[(size_t)c * 6 + 3 + d] = is_near ? NAN : grid.cmax[(size_t)c * dim + d] - grid.cmin[d];
            }
        }
        if (hipMalloc((void **)&s->d_cbt, sizeof(double) * grid.count * 6) != hipSuccess) {
            ecmc_system_destroy(s);
            return ecmc_fail(ECMC_ERR_HIP, "cell-bound table allocation failed");
        }
        // the table depends only on the cell geometry, the box, the potential and the
        // estimator: replicas of one system take it from the cache instead of rebuilding it
        std::vector<double> key(corners);
        key.push_back(desc->system_length);
        for (int q = 0; q < 4; q++) key.push_back(tg.par[q]);
        for (int q = 0; q < 4; q++) key.push_back(tg.bpar[q]);
        std::vector<double> table;
        if (cell_bound_cache_find(key, table)) {
            if (hipMemcpy(s->d_cbt, table.data(), sizeof(double) * table.size(), hipMemcpyHostToDevice) != hipSuccess) {
                ecmc_system_destroy(s);
                return ecmc_fail(ECMC_ERR_HIP, "cell-bound table upload failed");
            }
        } else {
            if (hipMalloc((void **)&s->d_corners, sizeof(double) * corners.size()) != hipSuccess ||
                hipMemcpy(s->d_corners, corners.data(), sizeof(double) * corners.size(), hipMemcpyHostToDevice) != hipSuccess) {
                ecmc_system_destroy(s);
                return ecmc_fail(ECMC_ERR_HIP, "cell-bound table allocation failed");
            }
            hipLaunchKernelGGL(cell_bound_kernel, dim3(grid.count * 3), dim3(NT), 0, s->stream, a.ewald, s->d_corners,
                               desc->system_length, tg.par[3], tg.bpar[2], (int)tg.bpar[1], tg.bpar[0], tg.bpar[3],
                               s->d_cbt);
            table.resize((size_t)grid.count * 6);
            if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s->stream) != hipSuccess ||
                hipMemcpy(table.data(), s->d_cbt, sizeof(double) * table.size(), hipMemcpyDeviceToHost) != hipSuccess) {
                ecmc_system_destroy(s);
                return ecmc_fail(ECMC_ERR_HIP, "cell-bound table kernel failed");
            }
            cell_bound_cache_store(key, table);
        }
        a.cbt = s->d_cbt;
        for (int d = 0; d < 3; d++) {
            double m = 0.0;
            for (int c = 0; c < grid.count; c++)
                for (int b = 0; b < 2; b++) {
                    const double v = fabs(table[(size_t)(c * 3 + d) * 2 + b]);
                    if (v > m) m = v;   // NaN marks a nearby separation
                }
            // per unit of the charge product: bounds use it divided by the target charge
            a.cb_max[d] = nextafterf((float)(tg.use_charge ? m / fabs(tg.bpar[2]) : m), INFINITY) * (1.f + 0x1p-20f);
        }
        bool veto = false;
        for (int t = 0; t < desc->n_taggers; t++) veto = veto || desc->taggers[t].kind == ECMC_TAG_CELL_VETO;
        if (veto) {
            // cell_veto_event_handler.py:147-159: per direction, the non-nearby cells in
            // yield_cells() order with rates max(upper, 0) and max(-lower, 0)
            std::vector<int32_t> items;
            for (int c = 0; c < grid.count; c++)
                if (!std::isnan(table[(size_t)c * 6])) items.push_back(c);
            const int m = (int)items.size();
            std::vector<CvEntry> all((size_t)6 * m);
            std::vector<double> rates(m);
            for (int wt = 0; wt < 6 && m > 0; wt++) {
                const int d = wt / 2, b = wt % 2;
                for (int i = 0; i < m; i++) {
                    const double v = table[(size_t)(items[i] * 3 + d) * 2 + b];
                    const double r = b ? -v : v;
                    rates[i] = 0.0 > r ? 0.0 : r;
                }
                if (!walker_table(items, rates, &all[(size_t)wt * m], a.cv_total[wt], a.cv_mean[wt])) {
                    ecmc_system_destroy(s);
                    return ecmc_fail(ECMC_ERR_CONFIGURATION, "cell veto: Walker table failed (negative rate or leftover check)");
                }
            }
            if (m == 0) {
                ecmc_system_destroy(s);
                return ecmc_fail(ECMC_ERR_CONFIGURATION, "cell veto: no cell lies outside the nearby cells");
            }
            if (hipMalloc((void **)&s->d_cvw, sizeof(CvEntry) * all.size()) != hipSuccess ||
                hipMemcpy(s->d_cvw, all.data(), sizeof(CvEntry) * all.size(), hipMemcpyHostToDevice) != hipSuccess) {
                ecmc_system_destroy(s);
                return ecmc_fail(ECMC_ERR_HIP, "cell veto table upload failed");
            }
            a.cvw = s->d_cvw;
            a.cv_m = m;
        }
    }
    plan_lds(s);
    // the host view; a system without one (pinned memory exhausted) copies what it reads
    const bool res_positions = s->args.resident != 0;
    s->host = take_view(s->device, sizeof(HostView) + (res_positions ? sizeof(double) * dim * n : 0), &a.host);
    if (s->host) {
        s->host->st = st;
        s->host->n_out = 0;
        s->host->has_positions = 0;
    }
    *out = s;
    return ECMC_OK;
}

extern "C" void ecmc_system_destroy(ecmc_system *s) {
    if (!s) return;
    hipFree(s->d_pos); hipFree(s->d_charge); hipFree(s->d_cmin); hipFree(s->d_nearby); hipFree(s->d_nearby_n);
    hipFree(s->d_occ); hipFree(s->d_occ_n); hipFree(s->d_ring); hipFree(s->d_st);
    hipFree(s->d_sur_cell); hipFree(s->d_sur_id); hipFree(s->d_cbt); hipFree(s->d_corners);
    hipFree(s->d_cvw);
    hipFree(s->d_tg); hipFree(s->d_nout); hipFree(s->d_log); hipFree(s->d_ewald); hipFree(s->d_ewald_codes); hipFree(s->d_step_ev); hipFree(s->d_args);
    if (s->ev0) hipEventDestroy(s->ev0);
    if (s->ev1) hipEventDestroy(s->ev1);
    if (s->stream) hipStreamDestroy(s->stream);
    if (s->host) release_view(s->host);   // (freeing device memory has waited for the launches)
    delete s;
}

static int status_of_state(int err) {
    switch (err) {
    case 0: return ECMC_OK;
    case ECMC_ERR_SCHEDULER: return ecmc_fail(ECMC_ERR_SCHEDULER, "SchedulerError: no event or decreasing event time");
    case ECMC_ERR_STATE: return ecmc_fail(ECMC_ERR_STATE, "a position left the cell system or an occupancy list overflowed");
    case ECMC_ERR_NUMERIC: return ecmc_fail(ECMC_ERR_NUMERIC, "ValueError: math domain error in a displacement");
    case ECMC_ERR_CONFIGURATION: return ecmc_fail(ECMC_ERR_CONFIGURATION, "end-of-chain time assertion or missing start of run");
    default: return ecmc_fail(err, "device error");
    }
}

// A call that launches work of these systems, from before the launch to its end.
struct InFlight {
    ecmc_system *const *systems;
    int32_t count;
    InFlight(ecmc_system *const *systems_, int32_t count_) : systems(systems_), count(count_) {
        for (int i = 0; i < count; i++) systems[i]->began++;
    }
    ~InFlight() {
        for (int i = 0; i < count; i++) systems[i]->ended++;
    }
};

// Copies from the host view, false if a launch may write it meanwhile: another thread's call is
// under way (`own`: the caller's own, 1 within its InFlight) or began during the copy.  The reader
// then takes a copy command, which waits for the launches before it.
static bool read_host(const ecmc_system *s, void *to, const void *from, size_t bytes, uint32_t own) {
    const uint32_t ended = s->ended.load(), began = s->began.load();
    if (began - ended != own) return false;
    memcpy(to, from, bytes);
    std::atomic_thread_fence(std::memory_order_seq_cst);
    return s->began.load() == began;
}

// The state that the last launch left (or the initial one): from the host view, else copied.
static int read_state(const ecmc_system *s, ChainState &st, uint32_t own = 0) {
    if (s->host && read_host(s, &st, &s->host->st, sizeof(st), own)) return ECMC_OK;
    if (hipMemcpy(&st, s->d_st, sizeof(ChainState), hipMemcpyDeviceToHost) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy failed");
    return ECMC_OK;
}

// The committed legs of the launch that just ended and its error code.
static int read_launch(const ecmc_system *s, int64_t &k, int &err) {
    if (s->host && read_host(s, &k, &s->host->n_out, sizeof(k), 1) &&
        read_host(s, &err, &s->host->st.err, sizeof(err), 1))
        return ECMC_OK;
    if (hipMemcpy(&k, s->d_nout, sizeof(int64_t), hipMemcpyDeviceToHost) != hipSuccess ||
               hipMemcpy(&err, (const char *)s->d_st + offsetof(ChainState, err), sizeof(int), hipMemcpyDeviceToHost) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy failed");
    return ECMC_OK;
}

extern "C" int ecmc_system_run(ecmc_system *s, int64_t max_events, ecmc_event *host_log, int64_t *n_committed) {
    if (!s || max_events < 0) return ecmc_fail(ECMC_ERR_ARGUMENT, "bad argument");
    if (n_committed) *n_committed = 0;
    if (max_events == 0) return ECMC_OK;
    if (host_log && s->log_cap < max_events) {
        hipFree(s->d_log);
        s->d_log = nullptr;
        if (hipMalloc((void **)&s->d_log, sizeof(ecmc_event) * max_events) != hipSuccess)
            return ecmc_fail(ECMC_ERR_HIP, "hipMalloc of the event log failed");
        s->log_cap = max_events;
    }
    ChainArgs a = s->args;
    a.log = host_log ? s->d_log : nullptr;
    a.max_events = max_events;
    a.stop_mask = s->stop_mask;
    const InFlight flight(&s, 1);
    hipEventRecord(s->ev0, s->stream);
    if (hipMemcpyAsync(s->d_args, &a, sizeof(ChainArgs), hipMemcpyHostToDevice, s->stream) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy of the launch arguments failed");
    {
        void *kargs[] = {&s->d_args};
        dim3 block;
        const void *kernel = chain_launch(s->dim, s->features, s->args.resident, s->one_wave, block);
        hipLaunchKernel(kernel, dim3(1), block, kargs, s->lds_bytes, s->stream);
    }
    hipEventRecord(s->ev1, s->stream);
    if (hipGetLastError() != hipSuccess) return ecmc_fail(ECMC_ERR_HIP, "kernel launch failed");
    if (hipStreamSynchronize(s->stream) != hipSuccess) return ecmc_fail(ECMC_ERR_HIP, "kernel execution failed");
    float ms = 0.f;
    hipEventElapsedTime(&ms, s->ev0, s->ev1);
    s->last_ms = ms;
    int64_t k = 0;
    int err = 0, rc = read_launch(s, k, err);
    if (rc) return rc;
    if (host_log && k > 0 &&
        hipMemcpy(host_log, s->d_log, sizeof(ecmc_event) * k, hipMemcpyDeviceToHost) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy of the event log failed");
    if (n_committed) *n_committed = k;
    return status_of_state(err);
}

// The launch of independent systems with their arguments staged in `host_args` (count
// entries, filled here) and copied to the device array `d_args`: one workgroup per system on the
// first system's stream, then every system's committed legs and state are read back.
static int systems_run_staged(ecmc_system *const *systems, int32_t count, int64_t max_events, int64_t *n_committed,
                              ChainArgs *host_args, ChainArgs *d_args) {
    const int dim = systems[0]->dim;
    size_t lds = 0;
    for (int i = 0; i < count; i++) {
        ecmc_system *s = systems[i];
        if (s->lds_bytes > lds) lds = s->lds_bytes;
        host_args[i] = s->args;
        host_args[i].log = nullptr;
        host_args[i].max_events = max_events;
        host_args[i].stop_mask = s->stop_mask;
        if (n_committed) n_committed[i] = 0;
    }
    if (max_events == 0) return ECMC_OK;
    const InFlight flight(systems, count);
    ecmc_system *s0 = systems[0];
    if (hipMemcpyAsync(d_args, host_args, sizeof(ChainArgs) * count, hipMemcpyHostToDevice, s0->stream) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy of the launch arguments failed");
    hipEventRecord(s0->ev0, s0->stream);
    int features = 0;
    bool one_wave = true, resident = true;
    for (int i = 0; i < count; i++) {
        features |= systems[i]->features;
        one_wave = one_wave && systems[i]->one_wave;
        resident = resident && systems[i]->args.resident;
    }
    void *kargs[] = {&d_args};
    dim3 block;
    const void *kernel = chain_launch(dim, features, resident, one_wave, block);
    hipLaunchKernel(kernel, dim3(count), block, kargs, resident ? lds : 0, s0->stream);
    hipEventRecord(s0->ev1, s0->stream);
    const bool launched = hipGetLastError() == hipSuccess;
    const bool ran = hipStreamSynchronize(s0->stream) == hipSuccess;
    if (!launched) return ecmc_fail(ECMC_ERR_HIP, "kernel launch failed");
    if (!ran) return ecmc_fail(ECMC_ERR_HIP, "kernel execution failed");
    float ms = 0.f;
    hipEventElapsedTime(&ms, s0->ev0, s0->ev1);
    int rc = ECMC_OK;
    for (int i = 0; i < count; i++) {
        ecmc_system *s = systems[i];
        s->last_ms = ms;
        int64_t k = 0;
        int err = 0, read = read_launch(s, k, err);
        if (read) return read;
        if (n_committed) n_committed[i] = k;
        if (rc == ECMC_OK) rc = status_of_state(err);
    }
    return rc;
}

static int check_systems(ecmc_system *const *systems, int32_t count, int64_t max_events) {
    if (!systems || count < 1 || max_events < 0) return ecmc_fail(ECMC_ERR_ARGUMENT, "bad argument");
    if (!systems[0]) return ecmc_fail(ECMC_ERR_ARGUMENT, "null system");
    const int dim = systems[0]->dim;
    for (int i = 0; i < count; i++) {
        ecmc_system *s = systems[i];
        if (!s) return ecmc_fail(ECMC_ERR_ARGUMENT, "null system");
        if (s->dim != dim) return ecmc_fail(ECMC_ERR_ARGUMENT, "all systems of one launch must have one dimension");
        if (s->device != systems[0]->device)
            return ecmc_fail(ECMC_ERR_ARGUMENT, "all systems of one launch must live on one device");
        for (int k = 0; k < i; k++)
            if (systems[k] == s) return ecmc_fail(ECMC_ERR_ARGUMENT, "a system appears twice in one launch");
    }
    return ECMC_OK;
}

extern "C" int ecmc_systems_run(ecmc_system *const *systems, int32_t count, int64_t max_events,
                                int64_t *n_committed) {
    int rc = check_systems(systems, count, max_events);
    if (rc) return rc;
    std::vector<ChainArgs> args((size_t)count);
    ChainArgs *d_args = nullptr;
    if (hipMalloc((void **)&d_args, sizeof(ChainArgs) * count) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMalloc of the launch arguments failed");
    rc = systems_run_staged(systems, count, max_events, n_committed, args.data(), d_args);
    hipFree(d_args);
    return rc;
}

// ---- independent systems without allocation -------------------------------------------------
// The launch arguments of ecmc_systems_run_noalloc live in a fixed device array of the library
// (each GPU the library runs on holds its own copy until the process ends) and are staged in a
// fixed host array; one process-wide lock serialises the calls, so calls from one process never
// share the arrays at the same time.  The array's device address comes from
// hipGetSymbolAddress once per device (the name itself is not a device address in host code).
static_assert(sizeof(ChainArgs) <= 512, "the no-allocation argument array is sized for 512 B per system");
static __device__ __align__(256) ChainArgs scratch[ECMC_SYSTEMS_NOALLOC_MAX];
static ChainArgs g_noalloc_host[ECMC_SYSTEMS_NOALLOC_MAX];
constexpr int NOALLOC_DEVICES = 64;
static void *g_scratch_ptr[NOALLOC_DEVICES];
static std::mutex g_noalloc_mutex;

extern "C" int ecmc_systems_run_noalloc(ecmc_system *const *systems, int32_t count, int64_t max_events,
                                        int64_t *n_committed) {
    if (count > ECMC_SYSTEMS_NOALLOC_MAX)
        return ecmc_fail(ECMC_ERR_ARGUMENT, "more systems than ECMC_SYSTEMS_NOALLOC_MAX in one no-allocation launch");
    int rc = check_systems(systems, count, max_events);
    if (rc) return rc;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return ecmc_fail(ECMC_ERR_HIP, "no current HIP device");
    if (dev != systems[0]->device)
        return ecmc_fail(ECMC_ERR_ARGUMENT, "the systems' device must be the current device");
    if (dev < 0 || dev >= NOALLOC_DEVICES) return ecmc_fail(ECMC_ERR_HIP, "device index out of range");
    std::lock_guard<std::mutex> lock(g_noalloc_mutex);
    if (!g_scratch_ptr[dev]) {
        // set-up on the first call on this device, with the device current
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p)
            return ecmc_fail(ECMC_ERR_HIP, "hipGetSymbolAddress of the argument array failed");
        g_scratch_ptr[dev] = p;
    }
    return systems_run_staged(systems, count, max_events, n_committed, g_noalloc_host,
                              (ChainArgs *)g_scratch_ptr[dev]);
}

// ---- the leg driven step by step from the host (set-level event handler) -------------------
static int system_step(ecmc_system *s, int op, int tagger, ChainState &st) {
    if (!s) return ecmc_fail(ECMC_ERR_ARGUMENT, "null system");
    if (op != 0 && (tagger < 0 || tagger >= s->desc.n_taggers)) return ecmc_fail(ECMC_ERR_ARGUMENT, "no such tagger");
    const InFlight flight(&s, 1);
    const ChainArgs &sa = s->args;   // one step works on global memory
    if (hipMemcpyAsync(s->d_args, &sa, sizeof(ChainArgs), hipMemcpyHostToDevice, s->stream) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy of the launch arguments failed");
    if (s->dim == 2) hipLaunchKernelGGL((chain_step_kernel<2, FEAT_ALL, 256>), dim3(1), dim3(256), 0, s->stream, s->d_args, op, tagger, s->d_step_ev);
    else hipLaunchKernelGGL((chain_step_kernel<3, FEAT_ALL, 256>), dim3(1), dim3(256), 0, s->stream, s->d_args, op, tagger, s->d_step_ev);
    if (hipGetLastError() != hipSuccess) return ecmc_fail(ECMC_ERR_HIP, "kernel launch failed");
    if (hipStreamSynchronize(s->stream) != hipSuccess) return ecmc_fail(ECMC_ERR_HIP, "kernel execution failed");
    const int rc = read_state(s, st, 1);
    if (rc) return rc;
    return status_of_state(st.err);
}

extern "C" int ecmc_system_begin_leg(ecmc_system *s) {
    ChainState st;
    return system_step(s, 0, 0, st);
}

extern "C" int ecmc_system_send_event_time(ecmc_system *s, int32_t tagger, double *tq, double *tr, int32_t *target,
                                           int32_t *valid) {
    ChainState st;
    const int rc = system_step(s, 1, tagger, st);
    if (rc) return rc;
    const Slot &sl = st.slot[tagger];
    if (tq) *tq = sl.valid ? sl.t.q : INFINITY;
    if (tr) *tr = sl.valid ? sl.t.r : INFINITY;
    if (target) *target = sl.valid ? sl.target : -1;
    if (valid) *valid = sl.valid;
    return ECMC_OK;
}

extern "C" int ecmc_system_send_out_state(ecmc_system *s, int32_t tagger, ecmc_event *event) {
    ChainState st;
    if (s && tagger >= 0 && tagger < s->desc.n_taggers) {
        // the handler must hold an event (the host's scheduler never returns one without)
        const int read = read_state(s, st);
        if (read) return read;
        if (!st.slot[tagger].valid) return ecmc_fail(ECMC_ERR_SCHEDULER, "the event handler holds no event");
    }
    const int rc = system_step(s, 2, tagger, st);
    if (rc) return rc;
    if (event && hipMemcpy(event, s->d_step_ev, sizeof(ecmc_event), hipMemcpyDeviceToHost) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy failed");
    return ECMC_OK;
}

extern "C" int ecmc_system_positions(const ecmc_system *s, double *out) {
    if (!s || !out) return ecmc_fail(ECMC_ERR_ARGUMENT, "null argument");
    if (s->host) {
        int32_t filled = 0;
        const uint32_t began = s->began.load();   // one launch's flag and positions
        if (read_host(s, &filled, &s->host->has_positions, sizeof(filled), 0) && filled &&
            read_host(s, out, s->host + 1, sizeof(double) * s->dim * s->n, 0) && s->began.load() == began)
            return ECMC_OK;
    }
    std::vector<double> soa((size_t)s->dim * s->n);
    if (hipMemcpy(soa.data(), s->d_pos, sizeof(double) * soa.size(), hipMemcpyDeviceToHost) != hipSuccess)
        return ecmc_fail(ECMC_ERR_HIP, "hipMemcpy failed");
    for (int i = 0; i < s->n; i++)
        for (int d = 0; d < s->dim; d++) out[(size_t)i * s->dim + d] = soa[(size_t)d * s->n + i];
    return ECMC_OK;
}

extern "C" int ecmc_system_active(const ecmc_system *s, int32_t *active, int32_t *direction, double *tq, double *tr,
                                  int32_t *done) {
    if (!s) return ecmc_fail(ECMC_ERR_ARGUMENT, "null system");
    ChainState st;
    int rc = read_state(s, st);
    if (rc) return rc;
    if (active) *active = st.active;
    if (direction) *direction = st.adir;
    if (tq) *tq = st.at.q;
    if (tr) *tr = st.at.r;
    if (done) *done = st.done;
    return ECMC_OK;
}

extern "C" int ecmc_system_estimators(const ecmc_system *s, double *est8) {
    if (!s || !est8) return ecmc_fail(ECMC_ERR_ARGUMENT, "null argument");
    ChainState st;
    int rc = read_state(s, st);
    if (rc) return rc;
    memcpy(est8, st.est, sizeof(st.est));
    return ECMC_OK;
}

extern "C" int ecmc_system_rng_words(const ecmc_system *s, int64_t *words) {
    if (!s || !words) return ecmc_fail(ECMC_ERR_ARGUMENT, "null argument");
    ChainState st;
    int rc = read_state(s, st);
    if (rc) return rc;
    *words = (int64_t)st.cursor;
    return ECMC_OK;
}

extern "C" int ecmc_system_launch_lds(const ecmc_system *s, int64_t *bytes, int32_t *positions, int32_t *ring) {
    if (!s) return ecmc_fail(ECMC_ERR_ARGUMENT, "null system");
    if (bytes) *bytes = (int64_t)s->lds_bytes;
    if (positions) *positions = s->args.resident;
    if (ring) *ring = s->args.resident;
    return ECMC_OK;
}

extern "C" int ecmc_system_kernel_variant(const ecmc_system *s, int32_t *features, int32_t *variant) {
    if (!s) return ecmc_fail(ECMC_ERR_ARGUMENT, "null system");
    if (features) *features = s->features;
    if (variant) *variant = chain_variant(s->dim, s->features).features;
    return ECMC_OK;
}

extern "C" int ecmc_desc_kernel_variant(const ecmc_system_desc *desc, int32_t *features, int32_t *variant) {
    if (!desc) return ecmc_fail(ECMC_ERR_ARGUMENT, "null descriptor");
    if (desc->dim != 2 && desc->dim != 3) return ecmc_fail(ECMC_ERR_CONFIGURATION, "dimension must be 2 or 3");
    if (desc->n_taggers < 0 || desc->n_taggers > ECMC_MAX_TAGGERS)
        return ecmc_fail(ECMC_ERR_CONFIGURATION, "number of taggers out of range");
    const int f = system_features(*desc);
    if (features) *features = f;
    if (variant) *variant = chain_variant(desc->dim, f).features;
    return ECMC_OK;
}

extern "C" int ecmc_system_last_kernel_ms(const ecmc_system *s, double *ms) {
    if (!s || !ms) return ecmc_fail(ECMC_ERR_ARGUMENT, "null argument");
    *ms = s->last_ms;
    return ECMC_OK;
}

// ---- MT19937 words on the device (testing the ring against CPython) ----------------------
__global__ __launch_bounds__(64) void mt_words_kernel(const uint32_t *state, uint32_t *out, int64_t n) {
    __shared__ uint32_t ring[2048];
    for (int i = threadIdx.x; i < 624; i += 64) ring[2048 - 624 + i] = state[i];
    __syncthreads();
    for (int64_t from = 0; from < n; from += RING_STEP) {
        ring_make(ring, 2047u, (uint64_t)from, 1);
        for (int i = threadIdx.x; i < RING_STEP && from + i < n; i += 64) out[from + i] = mt_temper(ring[(from + i) & 2047]);
        __syncthreads();
    }
}

extern "C" int ecmc_mt_words(uint64_t seed, int64_t n, uint32_t *d_out, void *stream) {
    if (n < 0 || (n > 0 && !d_out)) return ecmc_fail(ECMC_ERR_ARGUMENT, "bad argument");
    if (n % 624 != 0) return ecmc_fail(ECMC_ERR_ARGUMENT, "n must be a multiple of 624");
    if (n == 0) return ECMC_OK;
    uint32_t mt[624];
    mt_seed_host(seed, mt);
    uint32_t *d_state = nullptr;
    if (hipMalloc((void **)&d_state, sizeof(mt)) != hipSuccess) return ecmc_fail(ECMC_ERR_HIP, "hipMalloc failed");
    hipStream_t st = (hipStream_t)stream;
    hipMemcpyAsync(d_state, mt, sizeof(mt), hipMemcpyHostToDevice, st);
    hipLaunchKernelGGL(mt_words_kernel, dim3(1), dim3(64), 0, st, d_state, d_out, n);
    hipError_t e = hipStreamSynchronize(st);
    hipFree(d_state);
    if (e != hipSuccess) return ecmc_fail(ECMC_ERR_HIP, "mt kernel failed");
    return ECMC_OK;
}
