// Derived compile-time constants of the active model directory (the -I path selects
// gamedev_amd/mod/<model>/const_defs.h) and the shared plain records of the collision library.
#ifndef GDX_MODEL_H
#define GDX_MODEL_H

#include <cstdint>

#include "const_defs.h"

namespace gdx {

constexpr double PI = 3.14159265358979323846;
constexpr int DIM = (N_Z > 1) ? 3 : 2;
// an azimuthal wedge needs periodic images (inc/swarm/const_defs.cuh:56-57): records near either seam
// get a rotated ghost whose code 3*i + image keeps the physical identifier (inc/swarm/_col_image.cuh:11-26)
constexpr bool X_WEDGE = N_X > 1
    && static_cast<float>(X_MAX) - static_cast<float>(X_MIN) < 6.28318530717958647692f - 1.0e-06f;
// spatial controller groups (inc/swarm/_col_types.cuh:123-125)
constexpr int LOCAL_GROUPS = ((N_X > 1) ? COL_BIN_X : 1)*COL_BIN_Y*((N_Z > 1) ? COL_BIN_Z : 1);
constexpr int LOCAL_WORDS = (LOCAL_GROUPS + 31) / 32;
constexpr int RAW_BINS = LOCAL_GROUPS*COL_BIN_S;
static_assert(LOCAL_GROUPS <= 64, "one 64-bit dependency mask per group");
static_assert(COL_BIN_S <= 8, "per-block controller accumulators hold 8 size bins");
// one wavefront holds 64/N_K owners, one neighbour slot per lane
static_assert(N_K == 16 || N_K == 32 || N_K == 64, "N_K must be 16, 32 or 64");
constexpr int SEG = N_K;
constexpr int NSEG = 64 / N_K;
constexpr int LOG2K = (N_K == 16) ? 4 : (N_K == 32) ? 5 : 6;
// neighbour rows are stored in bit-reversed slot order: position t holds slot bitrev(t), so that
// streaming positions 0..K-1 pairs slots exactly as the upper-half fold does (j with j + K/2, ...)
constexpr int bitrev_slot(int t)
{
    return static_cast<int>(__builtin_bitreverse32(static_cast<unsigned>(t)) >> (32 - LOG2K));
}
static_assert(bitrev_slot(1) == N_K / 2 && bitrev_slot(N_K - 2) == N_K / 2 - 1, "bit-reversed slot order");
// pairs at or above the fragmentation speed exist only for the physical kernel (other kernels carry
// vrel = 0 into the outcome test)
constexpr bool CAN_FRAGMENT = (COAG_KERNEL == 3) ? (V_FRAG < 1.0e300) : (V_FRAG <= 0.0);
// the physical kernel evaluated in a vertically integrated disk needs each partner's gas scale height
constexpr bool PARTNER_HG = (COAG_KERNEL == 3 && N_Z == 1);

}  // namespace gdx

// owner-position gas coefficients, computed once per geometry epoch with the exact operation sequence
// of the per-pair reference evaluation (inc/swarm/_col_types.cuh:15-18, _col_rates.cuh:13-24)
struct gdx_env
{
    double Z, omega, vn, radial, strat, cs, re_inv_sqrt, vg_sq;
};

// Morton hierarchy node; children occupy [first_child, first_child + child_count) in code order
struct gdx_node
{
    float lx, ly, lz, width;
    int begin, count, first_child, child_count;
};

// axis-aligned box as the neighbour search reads it, 32 bytes. Of a node: first = its first child and
// info = its child count, or first = its first record and info = minus its record count (a leaf)
struct gdx_box
{
    float lx, ly, lz;
    int first;
    float hx, hy, hz;
    int info;
};

// per raw controller bin (spatial group x size bin) sums of one bath-start rating pass
struct gdx_raw_rate
{
    double mass, weighted_rate, weighted_change, weighted_second;
    int count, owner_count, invalid_count, pad;
};

// per raw controller bin sums of one post-bath audit pass (col_audit_accum field order)
struct gdx_raw_audit
{
    double mass, predicted_f, predicted_e, predicted_var_f, predicted_var_e, predicted_g, predicted_var_g;
    unsigned long long maximum_weight_bits, maximum_g_jump_bits;
    double touched, event_weight, growth, end_mass;
    int owner_count, invalid_count;
};

// per-slot event statistics of one operator call (_col_types.cuh:32-33): four sticking mass-ratio
// bins, catastrophic fragmentation, remnant erosion, debris
constexpr int GDX_EVENT_CATEGORIES = 7;
struct gdx_event_work
{
    unsigned long long count[GDX_EVENT_CATEGORIES];
    double log_mass[GDX_EVENT_CATEGORIES];
};

// one controller group of one swarm among the swarms an operator run advances together: where the
// group's owner arrays live and its per-group scalars (pointers already offset to the group)
struct gdx_gref
{
    double2 *st, *res;
    const int *nbr;
    const double *measure;
    const gdx_env *env;
    const double *hgs;
    double4 *cached;
    uint64_t *rng;
    const int *slot_pidx;
    int *queue;
    double4 *qsum;
    int *qevents;
    gdx_event_work *evw;                      // null without diagnostics
    gdx_raw_rate *raw_rate;                   // the group's COL_BIN_S raw bins
    gdx_raw_audit *raw_audit;
    int *qcount;                              // the group's light queue length (from the region's end down)
    int *hcount;                              // the group's heavy queue length (from the region's start up)
    unsigned long long *scr_min, *scr_max;    // the group's size extrema scratch
    double *lower, *upper;                    // the group's moving size bounds
    unsigned long long *counters;             // the swarm's operator counters (GDX_CTR_*)
    unsigned long long *wave_ctr;             // the swarm's per-wave counters (GDX_WAVE_*)
    int *err;                                 // the swarm's chain error
    double lambda_0;
    uint64_t seed;
    // learned majorant (mlp null: the plain method)
    const void *mlp;                          // packed network of the swarm's majorant
    double safety;                            // bound = safety * S * softplus(net)
    int thin_stride;                          // exact subsample: one run of THIN_RUN slots in thin_stride
    double *lam;                              // per slot: S * softplus(net) of the owner's last evaluation
                                              // (the bound before the safety factors)
    double *lam_add;                          // per slot: exact increases of the owner's pair rates from
                                              // partner changes since that evaluation (added after the
                                              // safety factors: bound = safety * lam + lam_add)
    unsigned char *dirty;                     // per slot: state changed since the slot's last publish
    unsigned char *stale;                     // per slot: bound inputs changed since its last evaluation
                                              // (null: not tracked, the swarm has no majorant)
    const unsigned *rev_beg, *rev_end;        // per slot: its range in rev
    const int *rev;                           // the owners whose partner rows hold each slot
    int bound_reuse;                          // keep the bounds of owners whose inputs are unchanged
    int exact_walk;                           // chain partner walk from sequential partials only (test access)
    float2 *res32;                            // per slot: published {size, number} in FP32 (feature gathers)
    double2 *qstart;                          // per queue position: {start time, 1 = event at the start}
    int *cqueue;                              // thinning candidates of the bath, in the group's slot range
    double2 *cstart;                          // per candidate: {candidate time, bound}
    int *ccount;                              // the group's candidate count
};

// a slot whose published record changed: its table entry, slot and the record it replaced
struct gdx_changed
{
    int ref, slot;
    double size, numr;
};

// changed-slot lists of one publish: block b appends to list b % CHANGED_LISTS, so that the lists of
// the blocks on one XCD (blocks are dealt to the XCDs in turn) are that XCD's own and each list counter
// takes the returning atomics of a few hundred blocks, not thousands; each list holds up to its blocks'
// owners
constexpr int CHANGED_LISTS = 32;

// due slots per block of the majorant kernel (host block starts and device share it)
constexpr int MAJ_SLOTS = 4096;

// operator counters per swarm; the bound-evaluation count is spread over GDX_CTR_SPREAD slots (one per
// block index modulo the spread, summed on the host) so that the majorant's blocks do not all add to one
// address
constexpr int GDX_CTR_SPREAD = 32;
enum
{
    GDX_CTR_EVENTS, GDX_CTR_CHAINED, GDX_CTR_PAIRS, GDX_CTR_LONGEST, GDX_CTR_THINNED, GDX_CTR_CANDIDATES,
    GDX_CTR_ACCEPTED, GDX_CTR_CHECKS, GDX_CTR_VIOLATIONS, GDX_CTR_CAND_PAIRS, GDX_CTR_BOUND_EVALS,
    GDX_CTRS = GDX_CTR_BOUND_EVALS + GDX_CTR_SPREAD
};
// per-wave counters per swarm
enum
{
    GDX_WAVE_LONGEST, GDX_WAVE_BLOCKS, GDX_WAVE_CHAINED, GDX_WAVE_CHECKS, GDX_WAVE_VIOLATIONS,
    GDX_WAVE_RATE_CHECKS, GDX_WAVE_RATE_VIOLATIONS, GDX_WAVE_CTRS
};
// learned swarms rate one run of THIN_RUN consecutive slots in every `stride` runs exactly per bath (the
// controller and audit subsample; consecutive slots keep the accesses coalesced): a stride of
// THIN_STRIDE (1/16 of the owners), or THIN_STRIDE_LARGE (1/32) for swarms of at least THIN_LARGE_OWNERS
// active owners, whose subsample still holds ~10^4 owners per controller group
constexpr int THIN_STRIDE = 16;
constexpr int THIN_STRIDE_LARGE = 32;
constexpr int THIN_LARGE_OWNERS = 1 << 21;
constexpr int THIN_RUN = 32;
// owners of a group of cnt slots rated exactly in subsample phase sub
constexpr int thin_rated(int cnt, int sub, int stride)
{
    return (cnt / (THIN_RUN*stride))*THIN_RUN
        + (cnt % (THIN_RUN*stride) - sub*THIN_RUN < 0 ? 0
           : (cnt % (THIN_RUN*stride) - sub*THIN_RUN > THIN_RUN ? THIN_RUN
              : cnt % (THIN_RUN*stride) - sub*THIN_RUN));
}

// the due groups of one phase of a run, in device memory: group-table index, owner slot range in the
// group's swarm, first block of each group for the launching kernel's owners per block, bath end
struct gdx_wave
{
    int n;                       // due groups with active owners
    int total;                   // their owners
    const gdx_gref *table;
    const int *ref;
    const int *beg;
    const int *cnt;
    const int *bstart;           // n + 1 entries
    const double *dt;
    const int *qprefix;          // chain: exclusive prefixes of the groups' heavy queue lengths (n + 1),
                                 // then of their light queue lengths (n + 1)
    const int *sub;              // per group: exact-rate subsample phase of a learned swarm, -1 plain
    int learned;                 // some group belongs to a learned swarm
};

// waiting intervals {size, length} of the heavy owners that one chain launch ran alone on a wavefront each,
// in chunks of CHAIN_CHUNK intervals of one owner: chunk h is heavy owner h's first, the `extra` chunks
// from `owners` on go to the owners that need more, in order of `next`. An owner's chunks are linked from its
// last one back, and each gets the jump-moment sums {j1, j2, jmax} of its intervals.
constexpr int CHAIN_CHUNK = 64;
constexpr int CHAIN_EXTRA = 8192;   // extra chunks reserved
struct gdx_chain_log
{
    double2 *entry;              // CHAIN_CHUNK per chunk
    double4 *part;
    int4 *use;                   // per chunk: its owner's group-table entry and slot, its intervals
    int *prev;                   // per chunk: the owner's chunk before, -1 none
    int *last;                   // per heavy owner: its last chunk, -1 none logged
    int *next;                   // extra chunks asked for
    int owners;                  // heavy owners that run alone at most; with more there are no logs
    int extra;                   // at most CHAIN_EXTRA
    int enabled;                 // 0: no logs, owners that need jump moments take the general loop
    const int *hcount, *qcount;  // heavy and light queue lengths by group-table entry
};

#endif  // GDX_MODEL_H
