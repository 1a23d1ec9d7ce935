// Kernels of the GODAR step pipeline (one launch sequence per step):
//
//   [steps with the build kernels: k_begin -> radix sort -> k_ranges -> k_sup ...]
//    -> k_cand -> k_events (contacts, bonds, walls) -> k_repair -> k_fixup
//    -> k_final (which also gathers the bond terms)
//
// Sequential semantics of the reference (stepper.f90:71-280 visits floes i
// in index order and, for each, its candidates j > i in ascending distance;
// ridging reshapes floes in place, so later pairs see the new radius and
// thickness) are reproduced as follows:
//   * The event kernels evaluate every pair event with the start-of-step
//     floe properties.  Contact, bond and sheltering terms feed disjoint
//     accumulators, so each kind has code of its own: the candidate
//     search k_cand also computes every floe's sheltering minima and queues
//     the floes that have contact, bond or wall work.  One thread per
//     floe gathers its own contributions in the reference's per-floe order:
//     first the pairs where it is the inner index (ascending outer index),
//     then its own candidates in distance order.  Contact and sheltering
//     terms are evaluated by both floes of a pair; a bond is evaluated once,
//     by its owner, which stores the terms; k_final gathers them.  No atomics,
//     and FP64 sums stay identical to the reference.
//   * An event's speculative result is exact unless one of its floes was
//     reshaped earlier in the sequence.  Events that ridge are seeds; the
//     per-member k_repair settles which events reshape which floe, and to
//     what, in the order of the sequence, and lists the floes whose terms
//     that changes.
//   * k_fixup evaluates those floes' events again, each with the properties
//     its floes have at its place in the sequence, k_final applies the final
//     floe properties, forcing, Coriolis, totals and integration.
//
// Layout: the per-step kernels run over floes in cell order ("pos"), reading
// a sorted copy of the 96-byte floe records, so that a floe's neighbours sit
// close in memory.  Pair state persists per floe id.  List entries pack the
// partner as (id << 32 | pos).  The lists hold the candidates that can matter
// (sup_bound_of).
#include "godar_engine.h"
#include "godar_physics.h"
#include <type_traits>

namespace godar {

__device__ __forceinline__ void set_err(const DS& S, uint32_t bit) { atomicOr(S.err, bit); }

// LDS written by some lanes of a one-wavefront block, then read by others:
// the wavefront's LDS operations complete in order, so waiting for its own
// outstanding ones (and keeping the compiler from moving accesses across)
// is enough; no block barrier, which would also wait for global stores.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0); vmcnt, expcnt unchanged (gfx9 encoding)
    __builtin_amdgcn_wave_barrier();
}

// Inclusive scans over the wavefront's lanes (all of them active) by DPP moves,
// which stay in the vector registers: within each row of 16 lanes, then the
// last lane of rows 0 and 2 to rows 1 and 3, then lane 31 to the upper half.
// (Six shuffles one behind the other go through LDS: about a tenth of the
// latency of each.)  `none` stands in for lanes that have no source.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_move(int none, int v) {
    return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ int wave_scan(int v) {
    v += dpp_move<0x111, 0xF>(0, v);     // row_shr:1, 2, 4, 8
    v += dpp_move<0x112, 0xF>(0, v);
    v += dpp_move<0x114, 0xF>(0, v);
    v += dpp_move<0x118, 0xF>(0, v);
    v += dpp_move<0x142, 0xA>(0, v);     // row_bcast:15
    v += dpp_move<0x143, 0xC>(0, v);     // row_bcast:31
    return v;
}
__device__ __forceinline__ int wave_scan_max(int v) {   // of values >= 0
    v = max(v, dpp_move<0x111, 0xF>(0, v));
    v = max(v, dpp_move<0x112, 0xF>(0, v));
    v = max(v, dpp_move<0x114, 0xF>(0, v));
    v = max(v, dpp_move<0x118, 0xF>(0, v));
    v = max(v, dpp_move<0x142, 0xA>(0, v));
    v = max(v, dpp_move<0x143, 0xC>(0, v));
    return v;
}
__device__ __forceinline__ int wave_last(int v) { return __builtin_amdgcn_readlane(v, 63); }

// Workgroups are dispatched to the 8 XCDs round-robin, and each XCD has its
// own L2.  Kernels that read their neighbours' rows take this logical block
// index instead of blockIdx.x, so that each XCD works on one contiguous eighth
// of the floes (whose neighbours then sit in the same L2).  The grid must be a
// multiple of XCD_COUNT blocks (launch_grid on the host).
__device__ __forceinline__ int xcd_block() {
    const int per = (int)(gridDim.x / XCD_COUNT);
    return (int)(blockIdx.x % XCD_COUNT) * per + (int)(blockIdx.x / XCD_COUNT);
}

// The blocks a queue's kernel runs: this block's XCD, its index among the
// XCD's blocks of the same work and their number.  Each XCD takes one
// contiguous share of the queue, so that short queues still spread over all
// XCDs and each XCD's share sits together in its L2.
struct QueueBlocks { int xcd, block, blocks; };
__device__ __forceinline__ QueueBlocks queue_blocks() {
    QueueBlocks b;
    b.xcd = (int)(blockIdx.x % XCD_COUNT);
    b.block = (int)(blockIdx.x / XCD_COUNT);
    b.blocks = (int)(gridDim.x / XCD_COUNT);
    return b;
}

__device__ __forceinline__ int32_t* qcount(const DS& S, int c, int x) {
    return S.qn + (c * XCD_COUNT + x) * QN_STRIDE;
}

// Queue c read as one sequence (its segments in XCD order): the segment
// counts and the total.
struct QueueView {
    int cnt[XCD_COUNT];
    int total;
};
__device__ __forceinline__ QueueView queue_view(const DS& S, int c) {
    QueueView v;
    v.total = 0;
#pragma unroll
    for (int x = 0; x < XCD_COUNT; ++x) {
        v.cnt[x] = *qcount(S, c, x);
        v.total += v.cnt[x];
    }
    return v;
}
// position held by entry t (0 <= t < total) of the sequence
__device__ __forceinline__ int queue_at(const DS& S, int c, const QueueView& v, int t) {
    int idx = 0;
#pragma unroll
    for (int x = 0; x < XCD_COUNT; ++x) {
        idx = (t >= 0 && t < v.cnt[x]) ? x * S.qseg + t : idx;
        t -= v.cnt[x];
    }
    return S.qlist[(int64_t)c * S.S + idx];
}
// Slot of this thread's it-th entry of a queue of length qn, or -1: there may
// be fewer blocks than the queue fills (the host caps them at
// QUEUE_GRID_WAVES wavefronts), so each thread takes every (threads per
// XCD)-th entry of its XCD's share.
__device__ __forceinline__ int queue_slot_it(const QueueBlocks& b, int qn, int it) {
    const int per = (qn + XCD_COUNT - 1) / XCD_COUNT;
    const int local = (b.block + it * b.blocks) * (int)blockDim.x + (int)threadIdx.x;
    if (local >= per) return -1;
    const int t = b.xcd * per + local;
    return t < qn ? t : -1;
}
// Entries of a queue of length qn taken by this wavefront when a wavefront
// evaluates its floes' pairs together: `floes` consecutive entries of its
// XCD's share at begin, begin + stride, ... below end.  Just enough floes for
// one full pass of 64 pairs (by the mean number of superset entries the search
// reads), more only if the queue has more for every wavefront of the grid: with 64
// floes of tens of candidates each, a wavefront works through all their pairs
// one pass after the other while the rest of the GPU has nothing to do (one
// MI355X, contact kernel: 320,000 floes in 24 members with about 43
// candidates a floe, 2,100 of them queued, 0.45 -> 0.03 ms), while one floe
// of two pairs per wavefront only spreads the same chain over more compute
// units (2,501 floes, 130 queued: 0.029 ms with full passes, 0.037 without).
// Queues with more than 16 floes for every wavefront keep 64: all wavefronts
// are busy then, and full passes count for more (the 512-field ensemble's
// 157,000 queued floes lost 0.03 ms per step with 39).
struct QueueShare { int begin, end, stride, floes; };
__device__ __forceinline__ QueueShare queue_share(const DS& S, const QueueBlocks& b, int qn) {
    const int per = (qn + XCD_COUNT - 1) / XCD_COUNT;
    const int wpb = (int)(blockDim.x >> 6);
    const int nw = b.blocks * wpb;
    const int w = b.block * wpb + (int)(threadIdx.x >> 6);
    const int lo = b.xcd * per;
    QueueShare q;
    const int f = (per + nw - 1) / nw;
    const int64_t entries = *S.nearsum;     // entries the search reads
    // (a floe in contact has about 1.6 listed pairs for each entry of the mean)
    const int full = (int)min((int64_t)64, 40 * (int64_t)S.N / max(entries, (int64_t)1));
    q.floes = f > 16 ? 64 : max(1, max(f, full));
    q.begin = lo + w * q.floes;
    q.end = min(qn, lo + per);
    q.stride = nw * q.floes;
    return q;
}
// The bond queue's: a wavefront evaluates its owners' records (1.2 each) 64 a
// round, so half as many owners while the wavefronts are not all taken keeps
// most of them to one round.
__device__ __forceinline__ QueueShare bond_share(const QueueBlocks& b, int qn) {
    const int per = (qn + XCD_COUNT - 1) / XCD_COUNT;
    const int wpb = (int)(blockDim.x >> 6);
    const int nw = b.blocks * wpb;
    const int lo = b.xcd * per;
    QueueShare q;
    q.floes = per > 32 * nw ? 64 : 32;
    q.begin = lo + (b.block * wpb + (int)(threadIdx.x >> 6)) * q.floes;
    q.end = min(qn, lo + per);
    q.stride = nw * q.floes;
    return q;
}
// appends position k to queue c from a single lane
__device__ __forceinline__ void enqueue_one(const DS& S, int c, int k) {
    const int x = k / S.qseg;
    S.qlist[(int64_t)c * S.S + x * S.qseg + atomicAdd(qcount(S, c, x), 1)] = k;
}

__device__ __forceinline__ int ent_id(int64_t e) { return (int)(e >> 32); }
__device__ __forceinline__ int ent_pos(int64_t e) { return (int)(uint32_t)(e & 0xffffffffll); }
__device__ __forceinline__ int64_t ent(int id, int pos) {
    return ((int64_t)id << 32) | (int64_t)(uint32_t)pos;
}

// Superset entries: the partner's position and, in the high half, the bound
// (a float): the pair is listed only while its floes are no further apart
// than that (sup_bound_of).
constexpr float SUP_KEEP = __builtin_inff();
__device__ __forceinline__ int64_t sup_ent(float bound, int pos) {
    return ((int64_t)__float_as_int(bound) << 32) | (int64_t)(uint32_t)pos;
}
__device__ __forceinline__ double sup_bound(int64_t e) { return (double)__int_as_float((int)(e >> 32)); }
// The pair at positions a and b is listed from now on whatever its distance
// (it has a contact history or a bond): its entries of both supersets.
__device__ __forceinline__ void sup_keep(const DS& S, int a, int b) {
    int64_t *sa = S.sup + S.soff[a], *sb = S.sup + S.soff[b];
    const int na = S.snear[a], nb = S.snear[b];
    for (int i0 = 0; i0 < max(na, nb); i0 += 4) {
        int64_t ea[4], eb[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ea[u] = sa[min(i0 + u, max(na - 1, 0))];
            eb[u] = sb[min(i0 + u, max(nb - 1, 0))];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (i0 + u < na && ent_pos(ea[u]) == b) sa[i0 + u] = sup_ent(SUP_KEEP, b);
            if (i0 + u < nb && ent_pos(eb[u]) == a) sb[i0 + u] = sup_ent(SUP_KEEP, a);
        }
    }
}

// floe at position k of this step's cell order
__device__ __forceinline__ Floe floe_at(const DS& S, int k) {
    const GeoRec g = S.geo[k];
    const ShelRec h = S.shel[k];
    const KinRec q = S.kin[k];
    Floe F;
    F.x = g.x; F.y = g.y; F.u = q.u; F.v = q.v; F.omega = q.omega;
    F.r = g.r; F.h = q.h; F.mass = q.mass; F.inertia = q.inertia; F.hfa = h.hfa; F.hfw = h.hfw;
    return F;
}

__device__ __forceinline__ double2 wind_at(const DS& S, int k) {
    const ShelRec h = S.shel[k];
    return make_double2(h.wx, h.wy);
}

__device__ __forceinline__ void take_shape(const Reshape& w, Floe& F) {
    F.r = w.r; F.h = w.h; F.mass = w.mass; F.inertia = w.inertia; F.hfa = w.hfa; F.hfw = w.hfw;
}

// Properties of a floe during the step's ordered sequence of events: F, the
// properties it starts the step with, unless a reshape of it (list `head` of
// the member's records) comes before event `key`; then those the last such
// reshape left.
__device__ __forceinline__ void floe_at_event(const Reshape* rec, int head, int64_t key, Floe& F) {
    int best = -1;
    int64_t bk = -1;
    for (int p = head; p >= 0; p = rec[p].next)
        if (rec[p].live && rec[p].key < key && rec[p].key > bk) { bk = rec[p].key; best = p; }
    if (best >= 0) take_shape(rec[best], F);
}
// (the record of the list's first reshape, -1 if none; its key, INT64_MAX)
__device__ __forceinline__ int first_record(const Reshape* rec, int head) {
    int best = -1;
    int64_t k = INT64_MAX;
    for (int p = head; p >= 0; p = rec[p].next)
        if (rec[p].live && rec[p].key < k) { k = rec[p].key; best = p; }
    return best;
}
__device__ __forceinline__ int64_t first_reshape(const Reshape* rec, int head) {
    const int p = first_record(rec, head);
    return p >= 0 ? rec[p].key : INT64_MAX;
}
// Records the reshape event `key` of the floes at kf (outer) and kj (-1: a
// wall) gives the floe at kg, as record p of the member, and links it to the
// floe's list.
__device__ __forceinline__ void add_reshape(const DS& S, Reshape* rec, int p, int64_t key, int kg,
                                            int kf, int kj, double r, double h, double mass,
                                            double inertia, double hfa, double hfw) {
    Reshape& w = rec[p];
    w.key = key; w.r = r; w.h = h; w.mass = mass; w.inertia = inertia; w.hfa = hfa; w.hfw = hfw;
    w.pos = kg; w.kf = kf; w.kj = kj; w.live = 1;
    w.next = atomicExch(&S.rhead[kg], p);
}

__device__ __forceinline__ int cell_coord(double p, double cell, int g) {
    double q = floor(p / cell);
    if (!(q >= 0.0)) return 0;          // also catches NaN
    if (q >= (double)(g - 1)) return g - 1;
    return (int)q;
}

// Old pair state of (i, j): owner i by storage slot, partner j by identity.
// Lists are searched with their first LIST_PEEK entries read at once (a
// floe's lists are short): one round of loads instead of one per entry.  Two:
// with four, most loads of a sparse field repeat a list's last entry, 64
// scattered lines each (512 members of 2,700 floes: events 190 -> 181 us).
constexpr int LIST_PEEK = 2;
// The bond gather reads both sides' words of a floe: with two, k_final waits
// for a second round in most wavefronts (114 -> 118 us there).
constexpr int GATHER_PEEK = 4;

// Index of the first of owner i's n records (slot-major rows of stride SS)
// whose partner is j (j >= 0; empty records hold -1), or -1.
// The first PEEK rows are requested together (one test of n, no test per
// row; rows past n stand in for the last one, so no other line is read).
template <int PEEK = LIST_PEEK, typename Rec>
__device__ __forceinline__ int find_partner(const Rec* list, int64_t SS, int i, int n, int j) {
    int id[PEEK];
#pragma unroll
    for (int p = 0; p < PEEK; ++p) id[p] = -1;
    if (n > 0) {
#pragma unroll
        for (int p = 0; p < PEEK; ++p) id[p] = list[(int64_t)min(p, n - 1) * SS + i].j;
    }
    int q = -1;
#pragma unroll
    for (int p = PEEK - 1; p >= 0; --p) q = (p < n && id[p] == j) ? p : q;
    for (int p = PEEK; q < 0 && p < n; ++p)
        if (list[(int64_t)p * SS + i].j == j) q = p;
    return q;
}

// The first LIST_PEEK of n entries of the slot-major list row kp (outer oj or
// inner ik), requested together (entries past n stand in for the last one).
struct Peek { int64_t e[LIST_PEEK]; };
__device__ __forceinline__ Peek peek_entries(const int64_t* list, int64_t SS, int kp, int n) {
    Peek p;
#pragma unroll
    for (int s = 0; s < LIST_PEEK; ++s) p.e[s] = -1;
    if (n > 0) {
#pragma unroll
        for (int s = 0; s < LIST_PEEK; ++s) p.e[s] = list[(int64_t)min(s, n - 1) * SS + kp];
    }
    return p;
}
// Slot of partner g among the n entries, or -1, and its entry; the rest of a
// long list LIST_PEEK entries a round.
__device__ __forceinline__ int find_peeked(const Peek& p, const int64_t* list, int64_t SS, int kp,
                                           int n, int g, int64_t& e) {
    int r = -1;
    e = -1;
#pragma unroll
    for (int s = LIST_PEEK - 1; s >= 0; --s) {
        const bool is = s < n && ent_id(p.e[s]) == g;
        r = is ? s : r;
        e = is ? p.e[s] : e;
    }
    for (int s0 = LIST_PEEK; r < 0 && s0 < n; s0 += LIST_PEEK) {
        Peek q;
#pragma unroll
        for (int s = 0; s < LIST_PEEK; ++s) q.e[s] = list[(int64_t)min(s0 + s, n - 1) * SS + kp];
#pragma unroll
        for (int s = LIST_PEEK - 1; s >= 0; --s) {
            const bool is = s0 + s < n && ent_id(q.e[s]) == g;
            r = is ? s0 + s : r;
            e = is ? q.e[s] : e;
        }
    }
    return r;
}
__device__ __forceinline__ int find_entry(const int64_t* list, int64_t SS, int kp, int n, int g) {
    int64_t e;
    return find_peeked(peek_entries(list, SS, kp, n), list, SS, kp, n, g, e);
}

// Old contact history and bond records of the floe at position k (what its
// storage slot's counts say, which are one load further away).
__device__ __forceinline__ int2 record_counts(uint32_t w) { return make_int2((int)(w & 0xFFFF), (int)(w >> 16)); }

__device__ __forceinline__ BondRec bond_from(const PairState& ps, int j) {
    BondRec b;
    b.j = j; b.bond = ps.bond; b.damage = ps.damage; b.deltanb = ps.deltanb; b.deltatb = ps.deltatb;
    b.trb_ji = ps.trb_ji; b.trb_ij = ps.trb_ij; b.rb = ps.rb; b.hb = ps.hb; b.lb = ps.lb;
    b.sb = ps.sb; b.ib = ps.ib;
    return b;
}

// Gather of one event into floe i's accumulators (stepper.f90:113-146,
// 165-198, 215-223), operand order kept; one helper per accumulator kind.
__device__ __forceinline__ void apply_contact_i(double* a, const EventOut& o) {
    if (o.flags & EV_CONTACT) {
        a[A_FCX] = a[A_FCX] - o.fcn_c + o.fcr_s;
        a[A_FCY] = a[A_FCY] - o.fcn_s - o.fcr_c;
        a[A_MC] = a[A_MC] - o.ri_fct - o.mcc;
        a[A_TAC] = a[A_TAC] + o.ac;
        a[A_PC] = a[A_PC] - o.fcn_ac;
    }
}
template <typename E>   // EventOut or BondTerms
__device__ __forceinline__ void add_bond_i(double* a, const E& o) {
    a[A_FBX] = a[A_FBX] + o.fbn_c - o.fbt_s;
    a[A_FBY] = a[A_FBY] + o.fbn_s + o.fbt_c;
    a[A_MB] = a[A_MB] - o.lri_fbt - o.mbb_ji;
    a[A_TAB] = a[A_TAB] + o.sb;
    a[A_PB] = a[A_PB] - o.fbn_sb;
}
__device__ __forceinline__ void apply_bond_i(double* a, const EventOut& o) {
    if (o.flags & EV_BONDED) add_bond_i(a, o);
}
__device__ __forceinline__ void apply_i(double* a, const EventOut& o) {
    apply_contact_i(a, o);
    apply_bond_i(a, o);
    if (o.flags & EV_SHELTER) {
        a[A_SHA] = fmin(a[A_SHA], o.hsfa_ji);
        a[A_SHW] = fmin(a[A_SHW], o.hsfw_ji);
    }
}

// ... and into floe j's.
__device__ __forceinline__ void apply_contact_j(double* a, const EventOut& o) {
    if (o.flags & EV_CONTACT) {
        a[A_FCX] = a[A_FCX] + o.fcn_c - o.fcr_s;
        a[A_FCY] = a[A_FCY] + o.fcn_s + o.fcr_c;
        a[A_MC] = a[A_MC] - o.rj_fct + o.mcc;
        a[A_TAC] = a[A_TAC] + o.ac;
        a[A_PC] = a[A_PC] - o.fcn_ac;
    }
}
template <typename E>
__device__ __forceinline__ void add_bond_j(double* a, const E& o) {
    a[A_FBX] = a[A_FBX] - o.fbn_c + o.fbt_s;
    a[A_FBY] = a[A_FBY] - o.fbn_s - o.fbt_c;
    a[A_MB] = a[A_MB] - o.lrj_fbt - o.mbb_ij;
    a[A_TAB] = a[A_TAB] + o.sb;
    a[A_PB] = a[A_PB] - o.fbn_sb;
}
__device__ __forceinline__ void apply_bond_j(double* a, const EventOut& o) {
    if (o.flags & EV_BONDED) add_bond_j(a, o);
}
__device__ __forceinline__ void apply_j(double* a, const EventOut& o) {
    apply_contact_j(a, o);
    apply_bond_j(a, o);
    if (o.flags & EV_SHELTER) {
        a[A_SHA] = fmin(a[A_SHA], o.hsfa_ij);
        a[A_SHW] = fmin(a[A_SHW], o.hsfw_ij);
    }
}

__device__ __forceinline__ void acc_init(double* a) {
#pragma unroll
    for (int k = 0; k < NACC; ++k) a[k] = 0.0;
    a[A_SHA] = 1.0;
    a[A_SHW] = 1.0;
}

// ---------------------------------------------------------------------
// 1. cell keys (one per floe id)
// ---------------------------------------------------------------------
// rec from the ordered copies (k_final's state) where they are newer, for
// the host (`host`, which clears the flag itself) before it reads or writes
// floe records or changes the floe count; k_begin does the same at the start
// of build and refresh steps.  Positions whose copy is of no live member are
// skipped: their records are current.
__global__ void k_spill(DS S, int host) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= S.N || !S.rebuild[2] || (!host && !S.rebuild[0] && !S.rebuild[1])) return;
    const GeoRec g = S.geo[k];
    const uint32_t f = S.cval[k];
    if (g.member < 0 || f >= (uint32_t)S.N) return;
    const KinRec q = S.kin[k];
    const ShelRec h = S.shel[k];
    FloeRec r;
    r.x = g.x; r.y = g.y; r.u = q.u; r.v = q.v; r.omega = q.omega;
    r.r = g.r; r.h = q.h; r.mass = q.mass; r.inertia = q.inertia; r.hfa = h.hfa; r.hfw = h.hfw;
    r.theta = q.theta;
    S.rec[f] = r;
}

// The per-member resets of a step (thread i of `threads` takes members i,
// i + threads, ...).
__device__ __forceinline__ void member_resets(const DS& S, int i, int threads, int nmembers) {
    for (; i < nmembers; i += threads) {
        if (!member_live(S.members[i])) continue;
        S.nseeds[i] = 0;
        S.stats[4 * i + 2] = 0; S.stats[4 * i + 3] = 0;
        S.tcur[i] = S.members[i].tstep;
    }
}

// First kernel of a step with the build kernels, over max(N, cells) threads
// (a step without them, lean, starts with k_cand).  BUILD_SOON alone is
// enough to build.
//  * the queue counters (k_final clears the next step's, which a failed step
//    leaves as they are) and, on build steps, the cell ranges;
//  * thread i as position: rec from the ordered copies where they are newer,
//    on build and refresh steps (k_spill's work; k_ranges clears the flag);
//  * thread i as storage slot: the per-member resets of the step and, on
//    build steps, the floe's cell key for the sort, written to the sort's
//    input buffers (bkey, bval).  The position is read from the ordered copy
//    where that is newer than rec (it is the same value the spill writes),
//    so the spill and the keys need no order between them.
__global__ void k_begin(DS S, int nmembers) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (*S.err) return;
    const bool build = S.rebuild[0] != 0, refresh = S.rebuild[1] != 0;
    const bool newer = S.rebuild[2] != 0;
    if (i < NQUEUE * XCD_COUNT) S.qn[i * QN_STRIDE] = 0;
    if (build && i <= S.ncells) S.crange[i] = make_int2(0, 0);
    if (build && i == 0) {
        *S.nearsum = 0;
        ++S.rebuild[3];
    }
    member_resets(S, i, (int)(gridDim.x * blockDim.x), nmembers);
    if (i >= S.N) return;
    if (newer && (build || refresh)) {
        const GeoRec g = S.geo[i];
        const uint32_t fs = S.cval[i];
        if (g.member >= 0 && fs < (uint32_t)S.N) {
            const KinRec q = S.kin[i];
            const ShelRec h = S.shel[i];
            FloeRec r;
            r.x = g.x; r.y = g.y; r.u = q.u; r.v = q.v; r.omega = q.omega;
            r.r = g.r; r.h = q.h; r.mass = q.mass; r.inertia = q.inertia; r.hfa = h.hfa; r.hfw = h.hfw;
            r.theta = q.theta;
            S.rec[fs] = r;
        }
    }
    const int f = i;
    if (!build) return;           // the cell order of the last build stands
    const int m = S.member_of[f];
    const bool live = m >= 0 && member_live(S.members[m]);
    S.bval[f] = (uint32_t)f;
    // floes of free slots and of members past their stop step sort last and
    // take no part in the step
    if (!live) { S.bkey[f] = (uint32_t)S.ncells; return; }
    const DevParams& P = S.params[m];
    double x, y;
    const int pos = newer ? S.pos_of[f] : -1;
    const GeoRec g = pos >= 0 ? S.geo[pos] : GeoRec{};
    if (pos >= 0 && g.member >= 0) { x = g.x; y = g.y; }
    else { x = S.rec[f].x; y = S.rec[f].y; }
    int cx = cell_coord(x, P.cell, P.gx), cy = cell_coord(y, P.cell, P.gy);
    S.bkey[f] = (uint32_t)(P.cell_base + cy * P.gx + cx);
}

// Distance beyond which a floe's sheltering terms are exactly 1 (shelter_min;
// lim: 20 in FP32, 40 in FP64), from its own drafts; the room kept for the
// drafts to grow before the next build.
constexpr double NEAR_ROOM = 1.25;
__device__ __forceinline__ double near_reach(double lim, double hfa, double hfw) {
    return lim * fmax(hfa, hfw) / (double)0.18f;
}

// The floe records in the current order and the wind at each floe
// (winds_currents, forcing.f90:1-29); on build steps the cell ranges over the
// sorted keys.  Between builds the order stands and k_final writes these
// copies for the next step itself, so this runs only on build steps and after
// the copies went stale (a member stopped, the host changed the wind).
__global__ void k_ranges(DS S) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    // k_begin has brought rec up to date where this step reads it
    if (k == 0 && !*S.err && (S.rebuild[0] || S.rebuild[1])) S.rebuild[2] = 0;
    if (k >= S.N || *S.err || (!S.rebuild[0] && !S.rebuild[1])) return;
    int f = (int)S.cval[k];
    int m = S.member_of[f];
    if (m >= 0 && !member_live(S.members[m])) {
        // The first step after a member stopped (and every build): its pair
        // state into the other buffers too, which no step of its own writes
        // any more while they go on changing place.
        m = -1;
        const int nh = S.hcnt_old[f], nb = S.bcnt_old[f];
        for (int q = 0; q < nh; ++q) S.hist_new[(int64_t)q * S.S + f] = S.hist_old[(int64_t)q * S.S + f];
        for (int q = 0; q < nb; ++q) S.bond_new[(int64_t)q * S.S + f] = S.bond_old[(int64_t)q * S.S + f];
        S.hcnt_new[f] = nh;
        S.bcnt_new[f] = nb;
    }
    const FloeRec fr = S.rec[f];
    GeoRec g;
    g.x = fr.x; g.y = fr.y; g.r = fr.r; g.id = S.gid_of[f]; g.member = m;
    S.geo[k] = g;
    KinRec q;
    q.u = fr.u; q.v = fr.v; q.omega = fr.omega; q.h = fr.h; q.mass = fr.mass; q.inertia = fr.inertia;
    q.theta = fr.theta;
    S.kin[k] = q;
    S.pos_of[f] = k;
    double ua = 0.0, va = 0.0;
    if (m >= 0) {
        S.pos_id[g.id] = k;
        if (*S.rebuild) {
            // how far apart a pair of this floe may be and still matter to it
            const DevParams& P = S.params[m];
            double nb = P.shelter ? NEAR_ROOM * near_reach(S.near_lim, fr.hfa, fr.hfw) : 0.0;
            if (P.cohesion) nb = fmax(nb, P.bond_lim);
            nb = fmax(nb, (double)S.nbmin[f]) * (1.0 + 1e-6);
            S.nb[k] = nb < 1e30 ? (float)nb : SUP_KEEP;
            S.rcnt[k] = (uint32_t)S.hcnt_old[f] | ((uint32_t)S.bcnt_old[f] << 16);
            const uint32_t key = S.ckey[k];
            if (k == 0 || S.ckey[k - 1] != key) S.crange[key].x = k;
            if (k == S.N - 1 || S.ckey[k + 1] != key) S.crange[key].y = k + 1;
        }
        const DevParams& P = S.params[m];
        ua = P.ua; va = P.va;
        // the wind at the start of step tcur: model time (tcur - 1) dt
        if (P.wind_grid >= 0)
            sample_wind(S.wgrids[P.wind_grid], S.wpool, fr.x, fr.y, fr.r,
                        (double)(S.tcur[m] - 1) * P.dt, ua, va);
    }
    ShelRec h;
    h.hfa = fr.hfa; h.hfw = fr.hfw; h.wx = ua; h.wy = va;
    S.shel[k] = h;
}

// Appends position k to work queue c, one atomic per wavefront.  Every lane
// of the wavefront must call it; the wavefront's positions lie in one XCD
// share of the candidate search.
__device__ __forceinline__ void enqueue(const DS& S, bool want, int c, int k) {
    uint64_t mask = __ballot(want);
    const int lane = threadIdx.x & 63;
    // (once, unless the wavefront's positions lie on either side of a segment
    // boundary, which the candidate search's never do)
    while (mask) {
        const int leader = __ffsll((long long)mask) - 1;
        const int x = __builtin_amdgcn_readlane(k, leader) / S.qseg;
        const uint64_t mine = __ballot(want && k < (x + 1) * S.qseg);
        int base = 0;
        if (lane == leader) base = atomicAdd(qcount(S, c, x), __popcll(mine));
        base = __builtin_amdgcn_readlane(base, leader);
        if (mine >> lane & 1) {
            const uint64_t below = lane ? mine & ((~0ull) >> (64 - lane)) : 0ull;
            S.qlist[(int64_t)c * S.S + x * S.qseg + base + __popcll(below)] = k;
            want = false;
        }
        mask &= ~mine;
    }
}

// ---------------------------------------------------------------------
// 2. candidate lists (replaces coretran kNearest, stepper.f90:77-87)
//    outer(f) = { j > f : dist <= r(f) + rtree } by (dist, j)
//    inner(f) = { k < f : dist <= r(k) + rtree } by k
//    fused with each floe's sheltering minima (forcing.f90:162-186; a
//    minimum does not depend on the order its terms come in, and every term
//    is computed from exactly the operands the pair event would use) and the
//    work classification: a floe joins the contact queue if it overlaps a
//    candidate partner or holds contact histories, the bond queue if it owns
//    bond records (or a bond of its own forms this step), the wall queue if
//    it crosses the box.
// ---------------------------------------------------------------------
constexpr int SCAN_BATCH = 4;

// The query radius r + rtree holds many floes that are far away: no contact,
// no bond, and a sheltering term that is exactly 1 (with power-law radii on
// [200, 5000] m, nearly all of a floe's 43 candidates).  A pair can only matter
// while its floes are no further apart than the larger of their two bounds nb
// (the reach of their own sheltering, with room for the drafts to grow, and
// the distance bonds form at), or if it has a contact history or a bond.  So
// a superset puts the entries that can come within their bound before the
// next build first (snear of them), each entry with its bound (SUP_KEEP for
// pairs with a history or a bond; k_contact and k_bond set it on the entries
// of new ones), and the step's search reads those alone and lists the pairs
// within their bound: 9-11 of 59 entries and 2.4-4.2 of 43 candidates a floe
// at packing 0.7 of the power-law radii, 2.2-2.5 of 3.6 and 1.5-1.7 of 2.6
// with radii on [500, 2000] m at 0.55.  (One MI355X, against a search and
// lists of all candidates: 320,000 power-law floes mixed, search 0.39 -> 0.11
// ms, integration 0.088 -> 0.034, bonds 0.034 -> 0.016; 262,144 FP64, search
// 0.38 -> 0.16; 1,000 floes 0.114 -> 0.041; the 512-field ensemble of radii on
// [500, 2000] m, search 0.136 -> 0.115.)
// The other entries only answer which pairs were candidates (k_pairs) and how
// many events a reshape came before (k_repair).  A reshape whose drafts
// outgrow their room ends the step, which is run again with a build and more
// room (k_fixup).
__device__ __forceinline__ bool has_records(const DS& S, int i, uint32_t rc, int j) {
    const int2 n = record_counts(rc);
    return find_partner(S.hist_old, S.S, i, n.x, j) >= 0 || find_partner(S.bond_old, S.S, i, n.y, j) >= 0;
}
// bound of the pair of floe f (storage slot fs, bound nbf, record counts rcf)
// and floe j at q (bound nbq, record counts rcq)
__device__ __forceinline__ float sup_bound_of(const DS& S, int f, int fs, float nbf, uint32_t rcf, int j,
                                              int q, float nbq, uint32_t rcq) {
    const bool keep = j > f ? rcf != 0 && has_records(S, fs, rcf, j)
                            : rcq != 0 && has_records(S, S.cval[q], rcq, f);
    return keep ? SUP_KEEP : fmaxf(nbf, nbq);
}

// Candidate superset of one floe by one thread over its (2 SPAN + 1)^2 cell
// block: every floe j within (j > f ? r(f) : r(j)) + rtree + skin.  The cells
// of one row of the block are consecutive in the cell order, so each row is
// one contiguous range of positions; every cell range is read at once
// (indices clamped into the grid, cells outside it masked out afterwards) and
// the rows, taken as one sequence, SCAN_BATCH records at a time.  Returns the
// counts of all entries and of those that can come within their bound
// (sup_bound_of); FILL writes the entries at `out`, the latter (`snear`)
// first.
template <int SPAN, bool FILL>
__device__ __forceinline__ int2 sup_thread(const DS& S, int k, const GeoRec& me, const DevParams& P,
                                           int64_t* out, int snear) {
    constexpr int R = 2 * SPAN + 1;
    const int cx = cell_coord(me.x, P.cell, P.gx), cy = cell_coord(me.y, P.cell, P.gy);
    int2 rg[R][R];
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const int b = min(max(cy - SPAN + t, 0), P.gy - 1);
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int a = min(max(cx - SPAN + u, 0), P.gx - 1);
            rg[t][u] = S.crange[P.cell_base + b * P.gx + a];
        }
    }
    int rlo[R], rlen[R];
    int L = 0;
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const int b = cy - SPAN + t;
        int lo = INT_MAX, hi = 0;
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int a = cx - SPAN + u;
            const bool in = b >= 0 && b < P.gy && a >= 0 && a < P.gx && rg[t][u].y > rg[t][u].x;
            lo = in ? min(lo, rg[t][u].x) : lo;
            hi = in ? max(hi, rg[t][u].y) : hi;
        }
        rlo[t] = lo;
        rlen[t] = lo < hi ? hi - lo : 0;
        L += rlen[t];
    }
    const int f = me.id;
    const double rad = me.r + P.rtree + P.skin, reach = P.rtree + P.skin;
    const int fs = S.cval[k];
    const float nbme = S.nb[k];
    const uint32_t rcme = S.rcnt[k];
    int n = 0, nn = 0;
    for (int v0 = 0; v0 < L; v0 += SCAN_BATCH) {
        GeoRec g[SCAN_BATCH];
        int qq[SCAN_BATCH];
#pragma unroll
        for (int u = 0; u < SCAN_BATCH; ++u) {
            // position of entry v of the concatenated rows (the last entry
            // stands in past the end; it is not tested twice)
            int rem = min(v0 + u, L - 1), q = 0;
#pragma unroll
            for (int t = 0; t < R; ++t) {
                q = (rem >= 0 && rem < rlen[t]) ? rlo[t] + rem : q;
                rem -= rlen[t];
            }
            qq[u] = q;
            g[u] = S.geo[q];
        }
#pragma unroll
        for (int u = 0; u < SCAN_BATCH; ++u) {
            const int q = qq[u];
            if (v0 + u >= L || q == k) continue;
            const double dx = me.x - g[u].x, dy = me.y - g[u].y;
            const double thr = g[u].id > f ? rad : g[u].r + reach;
            // a superset: the margin only adds entries
            const double d2 = dx * dx + dy * dy;
            if (d2 <= thr * thr * (1.0 + 1e-12)) {
                const float bound = sup_bound_of(S, f, fs, nbme, rcme, g[u].id, q, S.nb[q], S.rcnt[q]);
                const double w = me.r + g[u].r + (double)bound + P.skin;
                const bool near = d2 <= w * w * (1.0 + 1e-12);
                if (FILL) out[near ? nn : snear + n - nn] = sup_ent(bound, q);
                ++n;
                nn += near ? 1 : 0;
            }
        }
    }
    return make_int2(n, nn);
}

// (floe, candidate) pairs of one wavefront in LDS: entry, distance (inner: -1 -
// identity) and owner lane, the per-lane pair counts and the pairs whose terms are
// evaluated
constexpr int CAND_TCAP = 512;
constexpr int CAND_LDS_PER_WAVE = CAND_TCAP * (8 + 8 + 1) + 64 * 4 + CAND_TCAP * 2 + 64;
static_assert(CAND_TCAP < 1 << 10, "the per-lane counts are packed 10 bits each");

// Neighbour search of one floe by one thread: its candidate lists are the
// entries of its superset within the query radius, in the slot-major rows
// (the outer ones by distance and identity, the inner ones by identity), then
// sheltering minima, classification and the per-step resets of the floe's
// rows.
//
// Every lane of the wavefront calls it (act: the lane has a floe).  The
// wavefront's supersets lie one after the other in the pool; they are tested
// together, 64 consecutive entries a round (each lane finds the entry's
// owner among the lanes), and the entries within the query radius are listed
// in LDS (`lds`, CAND_LDS_PER_WAVE bytes for this wavefront) in superset
// order, so each owner's are contiguous.  Then one lane per listed pair
// counts how many of its owner's come before it and writes the entry to that
// place (inserting them one after the other, a lane per floe, held the
// wavefront for its longest list, whose part past a few entries in registers
// went through memory: 320,000 power-law floes mixed 109 -> 60 us, 40,015 57
// -> 33, 262,144 FP64 164 -> 76; with one comparison for both lists and the
// equal distances apart, of 320,000 51 -> 46, 262,144 FP64 72 -> 61, 1.38 M on
// [500, 2000] m 111 -> 105), and the
// sheltering and classification terms of the pairs that need them are
// evaluated together, 64 at a time; each floe then takes the minimum of its
// own terms (a minimum of fmin terms does not depend on which lane computed
// them).  Floes whose pairs outnumber CAND_TCAP together are taken in smaller
// groups; one that does by itself inserts its entries in memory.
// The rows of position k (and its storage slot's counts) that the search
// reads first, loaded at once as soon as k is known.
struct CandPre {
    ShelRec msh;
    int64_t soff;
    int fs, L, hc, bc;
};
__device__ __forceinline__ CandPre cand_pre(const DS& S, int k) {
    CandPre c;
    c.msh = S.shel[k];
    c.fs = S.cval[k];
    c.L = S.snear[k];
    c.soff = S.soff[k];
    c.hc = S.hcnt_old[c.fs];
    c.bc = S.bcnt_old[c.fs];
    return c;
}

// The lists, minima and flags of one floe with more pairs than the
// wavefront's LDS holds, by its lane alone: insertion in memory (the outer
// list's distances in S.od), the terms as they come.
template <bool MIXED>
__device__ __forceinline__ void cand_single(const DS& S, int k, int m, bool bond_step, int& no, int& ni,
                                            typename Prec<MIXED>::T& sha, typename Prec<MIXED>::T& shw,
                                            bool& qc, bool& qb) {
    using T = typename Prec<MIXED>::T;
    const GeoRec me = S.geo[k];
    const CandPre pre = cand_pre(S, k);
    const DevParams& P = S.params[m];
    const int first = S.members[m].first;
    const int64_t SS = S.S;
    const int f = me.id;
    const double rad = me.r + P.rtree;
    const int64_t* se = S.sup + pre.soff;
    for (int v = 0; v < pre.L; ++v) {
        const int64_t e0 = se[v];
        const int q = ent_pos(e0);
        const GeoRec o = S.geo[q];
        const int j = o.id;
        const bool outer = j > f;
        const double dx = me.x - o.x, dy = me.y - o.y;
        const double dist2 = dx * dx + dy * dy;
        const double thr = outer ? rad : o.r + P.rtree;
        if (dist2 > thr * thr * (1.0 + 1e-12)) continue;
        const double d = sqrt(dist2);
        if (!(d <= thr) || !(me.r + o.r - d >= -sup_bound(e0))) continue;
        const int64_t e = ent(j, q);
        if (outer && no < S.CO) {
            int p = no;
            for (; p > 0; --p) {
                const double dp = S.od[(p - 1) * SS + k];
                const int64_t ep = S.oj[(p - 1) * SS + k];
                if (dp < d || (dp == d && ent_id(ep) < j)) break;
                S.od[p * SS + k] = dp;
                S.oj[p * SS + k] = ep;
            }
            S.od[p * SS + k] = d;
            S.oj[p * SS + k] = e;
            S.evf[no * SS + k] = P.shelter ? EV_SHELTER : 0u;
            if (S.record_forces) { S.ssc[no * SS + k] = 0.0; S.ssb[no * SS + k] = 0.0; }
        } else if (!outer && ni < S.CI) {
            int p = ni;
            for (; p > 0; --p) {
                const int64_t ep = S.ik[(p - 1) * SS + k];
                if (ep < e) break;
                S.ik[p * SS + k] = ep;
            }
            S.ik[p * SS + k] = e;
            S.ibond[ni * SS + k] = 0;
        }
        ++(outer ? no : ni);
        // outer: pair (f, j), f the outer floe i of the event, which takes
        // hsf*(j,f) evaluated with -cosa, -sina; inner: pair (j, f), cosa/sina
        // point from j to f, which takes hsf*(j,f) with j's wind
        const double deltan = outer ? me.r + o.r - d : o.r + me.r - d;
        if (deltan > 0) qc = true;
        if (outer && bond_step && deltan >= -P.bond_lim &&
            bond_keep(f - first, j - first, P.bond_seed, P.bond_thr24))
            qb = true;
        if (P.shelter) {
            const double nx = outer ? o.x - me.x : me.x - o.x;
            const double ny = outer ? o.y - me.y : me.y - o.y;
            const double cosa = nx / d, sina = ny / d;
            const ShelRec oh = S.shel[q];
            const T dn = T(deltan), c0t = T(cosa), s0t = T(sina);
            const T c = outer ? -c0t : c0t, sn = outer ? -s0t : s0t;
            const T ux = outer ? T(pre.msh.wx) : T(oh.wx), uy = outer ? T(pre.msh.wy) : T(oh.wy);
            sha = shelter_min(sha, T(oh.hfa), T(pre.msh.hfa), dn, c, sn, ux, uy);
            shw = shelter_min(shw, T(oh.hfw), T(pre.msh.hfw), dn, c, sn, T(P.uw), T(P.vw));
        }
    }
}

template <bool MIXED>
__device__ __forceinline__ void cand_thread(const DS& S, int k0, int k, const GeoRec& me, const CandPre& pre,
                                            int m, bool act, bool& qc, bool& qb, bool& qw,
                                            unsigned char* lds) {
    using T = typename Prec<MIXED>::T;
    // member m's parameters and step, read at once (m is a valid member
    // index whether or not the lane has a floe); no short-circuit tests
    // between them, which would turn into a chain of single loads
    const DevParams& P = S.params[m];
    const Member Mb = S.members[m];
    const double rtree = P.rtree, pnx = P.nx, pny = P.ny;
    const int coh = P.cohesion, rst = P.restart, shl = P.shelter;
    const double mx = act ? me.x : 0.0, my = act ? me.y : 0.0, mr = act ? me.r : 0.0;
    const int f = act ? me.id : 0;
    const bool bond_step = act & (Mb.tstep == 1) & (rst != 1) & (coh != 0);
    T sha = T(1), shw = T(1);
    double hfa = 0.0, hfw = 0.0;
    int fs = 0;
    int no = 0, ni = 0;
    const int64_t SS = S.S;
    int L = 0;
    int64_t soff = 0;
    if (act) {
        hfa = pre.msh.hfa; hfw = pre.msh.hfw;
        fs = pre.fs;
        qc = pre.hc > 0;
        qb = pre.bc > 0;
        qw = (me.y - me.r < 0) | (me.y + me.r > pny) | (me.x - me.r < 0) | (me.x + me.r > pnx);
        L = pre.L;
        soff = pre.soff;
    }
    int64_t* te = reinterpret_cast<int64_t*>(lds);                      // entry, then the water term
    double* td = reinterpret_cast<double*>(lds + 8 * CAND_TCAP);         // distance (inner: -1 - identity), then the air term
    uint8_t* to = lds + 16 * CAND_TCAP;                                   // owner lane, then flags
    // per lane: pairs, outer ones << 10, pairs whose terms are needed << 20
    int32_t* tn = reinterpret_cast<int32_t*>(lds + 17 * CAND_TCAP);
    // the pairs whose terms the last pass evaluates (indices into the above)
    uint16_t* tx = reinterpret_cast<uint16_t*>(lds + 17 * CAND_TCAP + 64 * 4);
    const int lane = (int)(threadIdx.x & 63);
    const uint64_t lt = lane ? ((~0ull) >> (64 - lane)) : 0ull;
    const int incl = wave_scan(L);
    const int start = incl - L, totalL = wave_last(incl);
    // the floe's switches for the other passes: sheltering on (bit 0), bonds
    // may form this step (bit 1)
    const int pflags = (shl != 0 ? 1 : 0) | (bond_step ? 2 : 0);
    // the owners of entries c0 .. c0 + 63, a lane each: every lane marks where
    // its superset starts, if that is among them, and the marks are scanned
    // (`before`: the owner of entry c0 - 1; lanes past the group's entries get
    // the last one's).  (A search over the lanes' starts was six shuffles one
    // behind the other, each through LDS: with the scans, 320,000 power-law
    // floes mixed 59 -> 56 us, 262,144 FP64 74 -> 72.)
    uint8_t* mk = lds + CAND_LDS_PER_WAVE - 64;
    auto owners = [&](int c0, int before, int g1) {
        mk[lane] = 0;
        if (L > 0 && lane < g1 && start >= c0 && start < c0 + 64) mk[start - c0] = (uint8_t)lane;
        wave_lds_sync();
        return max(wave_scan_max((int)mk[lane]), before);
    };
    auto entry_at = [&](int idx, int own) -> int64_t {
        return S.sup[__shfl(soff, own) + (idx - __shfl(start, own))];
    };
    // the floes [g0, g1) of the wavefront at a time: all of them, as a rule
    uint64_t alone = 0;         // lanes of floes that list their pairs by themselves
    for (int g0 = 0, gs = 64; g0 < 64;) {
        const int g1 = min(g0 + gs, 64);
        const int lo = __builtin_amdgcn_readlane(start, g0);
        const int hi = g1 < 64 ? __builtin_amdgcn_readlane(start, g1 & 63) : totalL;
        int atotal = 0, nneed = 0;
        tn[lane] = 0;
        wave_lds_sync();
        bool ovf = false;
        // each round's superset entries are requested two rounds before and
        // their floes one round before (a lane past the end reads the last
        // entry again)
        int own = 0, own_nxt = 0;
        int64_t e = 0, e_nxt = 0;
        GeoRec o = {};
        if (lo < hi) {
            own = owners(lo, 0, g1);
            e = entry_at(min(lo + lane, hi - 1), own);
            own_nxt = owners(lo + 64, wave_last(own), g1);
            e_nxt = entry_at(min(lo + 64 + lane, hi - 1), own_nxt);
            o = S.geo[ent_pos(e)];
        }
        for (int c0 = lo; c0 < hi; c0 += 64) {
            const int idx = c0 + lane;
            int own_2 = 0;
            int64_t e_2 = 0;
            GeoRec o_nxt = o;
            if (c0 + 64 < hi) {
                o_nxt = S.geo[ent_pos(e_nxt)];
                own_2 = owners(c0 + 128, wave_last(own_nxt), g1);
                e_2 = entry_at(min(idx + 128, hi - 1), own_2);
            }
            const double ox = __shfl(mx, own), oy = __shfl(my, own);
            const double ort = __shfl(rtree, own), orr = __shfl(mr, own);
            const double ohfa = __shfl(hfa, own), ohfw = __shfl(hfw, own);
            const int of = __shfl(f, own), ofl = __shfl(pflags, own);
            bool hit = false, need = false;
            double d = 0.0;
            const int j = o.id, q = ent_pos(e);
            if (idx < hi) {
                const double dx = ox - o.x, dy = oy - o.y;
                const double dist2 = dx * dx + dy * dy;
                const double thr = j > of ? orr + ort : o.r + ort;
                // far beyond the radius: no square root needed (sqrt is
                // correctly rounded, so it cannot cross a margin of 1e-12)
                if (dist2 <= thr * thr * (1.0 + 1e-12)) {
                    d = sqrt(dist2);
                    // (the same overlap on either side of the pair, so both
                    // floes list it or neither does)
                    hit = d <= thr && orr + o.r - d >= -sup_bound(e);
                }
                if (hit) {
                    // The last pass changes nothing for a pair out of
                    // contact, with no bond forming this step, whose two
                    // sheltering terms are exactly 1: the test shelter_min
                    // makes (the same overlap, the floe's own drafts, type T).
                    const double dn = j > of ? orr + o.r - d : o.r + orr - d;
                    const T dnt = T(dn);
                    const T lim = sizeof(T) == 4 ? T(20) : T(40);
                    const bool one_a = dnt < T(0) && T((double)0.18f) * -dnt >= lim * T(ohfa);
                    const bool one_w = dnt < T(0) && T((double)0.18f) * -dnt >= lim * T(ohfw);
                    need = dn > 0 || (ofl & 2) || ((ofl & 1) && !(one_a && one_w));
                }
            }
            const uint64_t mh = __ballot(hit);
            if (atotal + __popcll(mh) > CAND_TCAP) { ovf = true; break; }
            const uint64_t mn = __ballot(need);
            if (hit) {
                const int at = atotal + __popcll(mh & lt);
                te[at] = ent(j, q);
                td[at] = j > of ? d : -(double)j - 1.0;
                to[at] = (uint8_t)own;
                atomicAdd(&tn[own], 1 + (j > of ? 1 << 10 : 0) + (need ? 1 << 20 : 0));
                if (need) tx[nneed + __popcll(mn & lt)] = (uint16_t)at;
            }
            atotal += __popcll(mh);
            nneed += __popcll(mn);
            own = own_nxt; e = e_nxt; o = o_nxt;
            own_nxt = own_2; e_nxt = e_2;
        }
        wave_lds_sync();
        if (ovf) {
            if (g1 - g0 > 1) { gs = (g1 - g0) / 2; continue; }
            alone |= 1ull << g0;
            g0 = g1;
            continue;
        }
        const int mine = tn[lane];
        const int acount = mine & 1023;
        const int ai = wave_scan(mine);                        // (no field carries: at most CAND_TCAP in all)
        const int bases = ai - mine;
        const int abase = bases & 1023, nbase = bases >> 20, ncount = mine >> 20;
        if (lane >= g0 && lane < g1) {
            no = (mine >> 10) & 1023;
            ni = acount - no;
        }
        // every listed pair to its place in its owner's list, with the
        // per-step resets of its rows
        for (int c0 = 0; c0 < atotal; c0 += 64) {
            const int idx = min(c0 + lane, atotal - 1);
            const int ow = to[idx];
            const int b = __shfl(abase, ow), n = __shfl(acount, ow), fl_o = __shfl(pflags, ow);
            const int64_t en = te[idx];
            const double d = td[idx];
            const int id = ent_id(en);
            // outer entries below the distance, inner ones with a smaller
            // identity; equal distances, which next to never meet, by identity
            const double above = d >= 0.0 ? -0.5 : d, below = d >= 0.0 ? d : -0.5;
            int before = 0, same = 0;
            for (int t = b; t < b + n; ++t) {
                const double dt = td[t];
                before += (dt > above) & (dt < below);
                same += dt == d;
            }
            if (same > 1)
                for (int t = b; t < b + n; ++t) before += td[t] == d && ent_id(te[t]) < id;
            if (c0 + lane < atotal) {
                const int64_t at = before * SS + (k0 + ow);
                if (d >= 0.0) {
                    if (before < S.CO) {
                        S.oj[at] = en;
                        S.evf[at] = (fl_o & 1) ? EV_SHELTER : 0u;
                        if (S.record_forces) { S.ssc[at] = 0.0; S.ssb[at] = 0.0; }
                    }
                } else if (before < S.CI) {
                    S.ik[at] = en;
                    S.ibond[at] = 0;
                }
            }
        }
        // sheltering and classification over the pairs that need it.  A
        // minimum and an "any" do not depend on the order of their terms.
        // (A pair's terms replace the entry of the pair whose number among
        // all listed equals its own among those that need them: no later one
        // still to be read.)
        for (int c0 = 0; c0 < nneed; c0 += 64) {
            const bool valid = c0 + lane < nneed;
            const int idx = valid ? (int)tx[c0 + lane] : 0;
            int64_t en = 0;
            double d = -1.0;
            int ow = lane;
            if (valid) { en = te[idx]; d = td[idx]; ow = to[idx]; }
            // (the member parameters are read again: kept for this pass they
            // cost the search its fourth wavefront per SIMD)
            const int ko = k0 + ow;
            const int om = __shfl(m, ow), fl_o = __shfl(pflags, ow);
            T ta = T(1), tw = T(1);
            uint32_t fl = 0;
            if (valid) {
                const int q = ent_pos(en);
                const GeoRec mo = S.geo[ko];
                const GeoRec go = S.geo[q];
                const ShelRec oh = S.shel[q];
                const ShelRec mh = S.shel[ko];
                const bool outer = d >= 0.0;
                double dd = d;
                if (!outer) {
                    const double dx = mo.x - go.x, dy = mo.y - go.y;
                    dd = sqrt(dx * dx + dy * dy);
                }
                // outer: pair (f, j), f the outer floe i of the event; inner:
                // pair (j, f), f the inner floe j
                const double deltan = outer ? mo.r + go.r - dd : go.r + mo.r - dd;
                if (deltan > 0) fl |= 1u;
                const DevParams& Po = S.params[om];
                if (outer && (fl_o & 2) && deltan >= -Po.bond_lim) {
                    const int first = S.members[om].first;
                    if (bond_keep(mo.id - first, ent_id(en) - first, Po.bond_seed, Po.bond_thr24)) fl |= 2u;
                }
                if (fl_o & 1) {
                    // outer: floe f takes hsf*(j,f), evaluated with -cosa,
                    // -sina of the direction f -> j; inner: cosa/sina point
                    // from j to f and f takes hsf*(j,f) with j's wind
                    const double nx = outer ? go.x - mo.x : mo.x - go.x;
                    const double ny = outer ? go.y - mo.y : mo.y - go.y;
                    const double cosa = nx / dd, sina = ny / dd;
                    const T dn = T(deltan), c0t = T(cosa), s0t = T(sina);
                    const T c = outer ? -c0t : c0t, sn = outer ? -s0t : s0t;
                    const T ux = outer ? T(mh.wx) : T(oh.wx), uy = outer ? T(mh.wy) : T(oh.wy);
                    ta = shelter_min(T(1), T(oh.hfa), T(mh.hfa), dn, c, sn, ux, uy);
                    tw = shelter_min(T(1), T(oh.hfw), T(mh.hfw), dn, c, sn, T(Po.uw), T(Po.vw));
                }
            }
            wave_lds_sync();
            if (valid) {
                td[c0 + lane] = (double)ta;
                te[c0 + lane] = __double_as_longlong((double)tw);
                to[c0 + lane] = (uint8_t)fl;
            }
        }
        wave_lds_sync();
        if (lane >= g0 && lane < g1) {
            for (int i = nbase; i < nbase + ncount; ++i) {
                sha = dmin(sha, T(td[i]));
                shw = dmin(shw, T(__longlong_as_double(te[i])));
                qc = qc || (to[i] & 1u);
                qb = qb || (to[i] & 2u);
            }
        }
        wave_lds_sync();
        g0 = g1;
    }
    if (!act) return;
    if (alone >> lane & 1) cand_single<MIXED>(S, k, m, bond_step, no, ni, sha, shw, qc, qb);
    const uint32_t over = (no > S.CO ? ERR_OUTER_CAP : 0u) | (ni > S.CI ? ERR_INNER_CAP : 0u);
    if (over) set_err(S, over);
    S.ocnt[k] = min(no, S.CO);
    S.icnt[k] = min(ni, S.CI);
    S.acc[A_SHA * SS + k] = double(sha);
    S.acc[A_SHW * SS + k] = double(shw);
    if (!qc) S.hcnt_new[fs] = 0;
    if (!qb) S.bcnt_new[fs] = 0;
    S.wflag[k] = 0;
    S.bgat[k] = 0;
    S.rhead[k] = -1;
    S.cls[k] = qc ? CLS_CONTACT : 0;   // the fix-up sets CLS_BOND
    S.rcnt[k] = (uint32_t)pre.hc | ((uint32_t)pre.bc << 16);
}

// Superset build, thread per floe (members that are not dense; span 1 or
// 2 cells on each side): counts (FILL false) or entries and the build
// positions x0 (FILL true).  The count pass lists the dense members' floes in
// queue 3 for k_sup_dense.  Only on build steps.
template <bool FILL>
__global__ __launch_bounds__(FLOE_BLOCK) void k_sup(DS S) {
    if (!*S.rebuild || *S.err) return;
    const int k = xcd_block() * blockDim.x + threadIdx.x;
    bool qd = false;
    if (k < S.N) {
        const GeoRec me = S.geo[k];
        if (me.member < 0) {
            if (!FILL) S.scnt[k] = S.snear[k] = 0;
        } else {
            const DevParams& P = S.params[me.member];
            if (P.dense) {
                qd = !FILL;
            } else if (FILL) {
                int64_t* out = S.sup + S.soff[k];
                if (P.span == 2) sup_thread<2, true>(S, k, me, P, out, S.snear[k]);
                else sup_thread<1, true>(S, k, me, P, out, S.snear[k]);
                S.x0[k] = make_double2(me.x, me.y);
            } else {
                const int2 c = P.span == 2 ? sup_thread<2, false>(S, k, me, P, nullptr, 0)
                                           : sup_thread<1, false>(S, k, me, P, nullptr, 0);
                S.scnt[k] = c.x;
                S.snear[k] = c.y;
            }
        }
    }
    if (!FILL) enqueue(S, qd, 3, k);
}

// Superset offsets: per-tile totals, their exclusive scan (one workgroup;
// the total must fit the superset pool), then offsets within each tile.
__device__ __forceinline__ int64_t block_exclusive_scan(int64_t v, int64_t* tmp, int64_t& total) {
    const int t = (int)threadIdx.x, n = (int)blockDim.x;
    tmp[t] = v;
    __syncthreads();
    for (int off = 1; off < n; off <<= 1) {
        const int64_t add = t >= off ? tmp[t - off] : 0;
        __syncthreads();
        tmp[t] += add;
        __syncthreads();
    }
    total = tmp[n - 1];
    const int64_t incl = tmp[t];
    __syncthreads();
    return incl - v;
}

__global__ __launch_bounds__(SCAN_TILE) void k_scan_tiles(DS S) {
    __shared__ int64_t tmp[SCAN_TILE];
    __shared__ int near;
    if (!*S.rebuild || *S.err) return;
    const int k = blockIdx.x * SCAN_TILE + threadIdx.x;
    if (threadIdx.x == 0) near = 0;
    int64_t tot;
    block_exclusive_scan(k < S.N ? S.scnt[k] : 0, tmp, tot);
    // the near entries' sum: one global atomic per tile (one per wavefront of
    // the counting kernels, 8,192 on one word, took 60 us by themselves)
    const int sum = wave_last(wave_scan(k < S.N ? S.snear[k] : 0));
    if ((threadIdx.x & 63) == 0) atomicAdd(&near, sum);
    __syncthreads();
    if (threadIdx.x == 0) {
        S.sblk[blockIdx.x] = tot;
        atomicAdd((unsigned long long*)S.nearsum, (unsigned long long)near);
    }
}

__global__ __launch_bounds__(SCAN_TILE) void k_scan_total(DS S, int ntiles) {
    __shared__ int64_t tmp[SCAN_TILE];
    if (!*S.rebuild || *S.err) return;
    int64_t base = 0;
    for (int t0 = 0; t0 < ntiles; t0 += SCAN_TILE) {
        const int t = t0 + (int)threadIdx.x;
        const int64_t v = t < ntiles ? S.sblk[t] : 0;
        int64_t tot;
        const int64_t ex = block_exclusive_scan(v, tmp, tot);
        if (t < ntiles) S.sblk[t] = base + ex;
        base += tot;
    }
    if (threadIdx.x == 0) {
        S.sblk[ntiles] = base;
        if (base > S.sup_cap) set_err(S, ERR_SUP_CAP);
    }
}

__global__ __launch_bounds__(SCAN_TILE) void k_scan_offsets(DS S) {
    __shared__ int64_t tmp[SCAN_TILE];
    if (!*S.rebuild || *S.err) return;
    const int k = blockIdx.x * SCAN_TILE + threadIdx.x;
    int64_t tot;
    const int64_t ex = block_exclusive_scan(k < S.N ? S.scnt[k] : 0, tmp, tot);
    if (k < S.N) S.soff[k] = S.sblk[blockIdx.x] + ex;
}

// (lean: the step has no build kernels.  It then starts here, with the
// per-member resets; if a build or a refresh is due it sets ERR_NEED_BUILD and
// does nothing else: every later kernel of the step returns at once and the
// host runs the step again with them.)
template <bool MIXED>
__global__ __launch_bounds__(FLOE_BLOCK) void k_cand(DS S, int lean, int nmembers, int floes) {
    // (the wavefront's floes: lanes past them only help with the pairs)
    const int lane = (int)(threadIdx.x & 63);
    const int k0 = (xcd_block() * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6)) * floes;
    const int k = k0 + lane;
    bool qc = false, qb = false, qw = false;
    // every row the search starts from is requested before anything is
    // tested (reads only: harmless for free slots and failed steps)
    const bool inr = lane < floes && k < S.N;
    GeoRec me;
    CandPre pre;
    if (inr) {
        me = S.geo[k];
        pre = cand_pre(S, k);
    }
    const bool slot_used = inr && me.member >= 0;
    const int m = slot_used ? me.member : 0;
    // (the build flags stand while this kernel runs)
    const bool due = lean && ((S.rebuild[0] & BUILD_DUE) | S.rebuild[1]) != 0;
    const bool ok = !*S.err && !due;
    if (lean) {
        if (due && blockIdx.x == 0 && threadIdx.x == 0) atomicOr(S.err, ERR_NEED_BUILD);
        // (by every block: one alone held the launch for 0.1 ms at 16,384
        // members)
        if (ok) member_resets(S, (int)(blockIdx.x * blockDim.x + threadIdx.x), (int)(gridDim.x * blockDim.x), nmembers);
    }
    extern __shared__ unsigned char cand_lds[];
    const bool act = slot_used & ok;
    cand_thread<MIXED>(S, k0, k, me, pre, m, act, qc, qb, qw,
                       cand_lds + (threadIdx.x >> 6) * CAND_LDS_PER_WAVE);
    if (inr && ok && !slot_used) {
        S.ocnt[k] = 0;
        S.icnt[k] = 0;
    }
    enqueue(S, qc, 0, k);
    enqueue(S, qb, 1, k);
    enqueue(S, qw, 2, k);
}

// Superset build of the dense members' floes (queue 3), one wavefront per
// floe over its (2 span + 1)^2 cell block: counts, or the entries and the build
// positions.  Only on build steps.  A lane per cell reads the ranges at once,
// and the rows of the block, each one range of positions (the cells of a row
// are consecutive in the cell order), are taken as one sequence, SUP_AHEAD
// rounds of 64 positions requested together: the kernel is bound by its chain
// of loads, six of them instead of about 25 with the rows one after the other
// and the record counts behind the storage slots (count + fill of a build:
// 320,000 power-law floes 0.79 + 0.87 -> 0.40 + 0.44 ms, 106,000 0.29 + 0.27 ->
// 0.14 + 0.15, 262,144 in FP64 0.67 + 0.74 -> 0.33 + 0.38; the next floe's rows
// requested ahead as well: the same).
constexpr int SUP_AHEAD = 2;
template <bool FILL>
__global__ __launch_bounds__(64) void k_sup_dense(DS S) {
    if (!*S.rebuild || *S.err) return;
    const int lane = threadIdx.x;
    const QueueView qv = queue_view(S, 3);
    const int nq = qv.total;
    const int nb = (int)(gridDim.x / XCD_COUNT);
    const int xcd = (int)(blockIdx.x % XCD_COUNT), bi = (int)(blockIdx.x / XCD_COUNT);
    const int per = (nq + XCD_COUNT - 1) / XCD_COUNT;
    const int t1 = min(nq, xcd * per + per);
    const uint64_t lt = lane ? ((~0ull) >> (64 - lane)) : 0ull;
    for (int t = xcd * per + bi; t < t1; t += nb) {
        const int k = queue_at(S, 3, qv, t);
        const GeoRec me = S.geo[k];
        const int f = me.id, fs = S.cval[k];
        const float nbme = S.nb[k];
        const uint32_t rcme = S.rcnt[k];
        const int64_t soff = FILL ? S.soff[k] : 0;
        const int snear = FILL ? S.snear[k] : 0;
        const DevParams& P = S.params[me.member];
        const double skin = P.skin, rad = me.r + P.rtree + skin, reach = P.rtree + skin;
        const int sp = P.span, gx = P.gx, gy = P.gy, cell_base = P.cell_base;
        const int cx = cell_coord(me.x, P.cell, gx), cy = cell_coord(me.y, P.cell, gy);
        // the block's cells by row, a lane each (span 1 or 2: at most 25)
        const int R = 2 * sp + 1;
        const int lr = R == 3 ? lane / 3 : lane / 5;
        const int ca = cx - sp + (lane - lr * R), cb = cy - sp + lr;
        int2 rg = make_int2(0, 0);
        if (lane < R * R && ca >= 0 && ca < gx && cb >= 0 && cb < gy) rg = S.crange[cell_base + cb * gx + ca];
        const uint64_t cells = __ballot(rg.y > rg.x);
        int lo[5], end[5], L = 0;       // row r holds the sequence's entries up to end[r]
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            const uint32_t row = r < R ? (uint32_t)(cells >> (r * R)) & ((1u << R) - 1) : 0u;
            lo[r] = row ? __builtin_amdgcn_readlane(rg.x, r * R + __ffs((int)row) - 1) : 0;
            if (row) L += __builtin_amdgcn_readlane(rg.y, r * R + 31 - __clz((int)row)) - lo[r];
            end[r] = L;
        }
        int64_t* out = FILL ? S.sup + soff : nullptr;
        int n = 0, nn = 0;
        for (int c0 = 0; c0 < L; c0 += 64 * SUP_AHEAD) {
            GeoRec o[SUP_AHEAD];
            int qq[SUP_AHEAD];
            float nbq[SUP_AHEAD];
            uint32_t rcq[SUP_AHEAD];
#pragma unroll
            for (int u = 0; u < SUP_AHEAD; ++u) {
                const int v = min(c0 + 64 * u + lane, L - 1);    // (the last entry stands in past the end)
                int q = lo[0] + v;
#pragma unroll
                for (int r = 1; r < 5; ++r) q = v >= end[r - 1] ? lo[r] + v - end[r - 1] : q;
                qq[u] = q;
                o[u] = S.geo[q];
                nbq[u] = S.nb[q];
                rcq[u] = S.rcnt[q];
            }
#pragma unroll
            for (int u = 0; u < SUP_AHEAD; ++u) {
                const int q = qq[u];
                bool in = false, near = false;
                float bound = 0.0f;
                if (c0 + 64 * u + lane < L && q != k) {
                    const double dx = me.x - o[u].x, dy = me.y - o[u].y, d2 = dx * dx + dy * dy;
                    const double thr = o[u].id > f ? rad : o[u].r + reach;
                    in = d2 <= thr * thr * (1.0 + 1e-12);
                    if (in) {
                        bound = sup_bound_of(S, f, fs, nbme, rcme, o[u].id, q, nbq[u], rcq[u]);
                        const double w = me.r + o[u].r + (double)bound + skin;
                        near = d2 <= w * w * (1.0 + 1e-12);
                    }
                }
                const uint64_t mi = __ballot(in), mn = __ballot(near);
                if (FILL && in)
                    out[near ? nn + (int)__popcll(mn & lt) : snear + (n - nn) + (int)__popcll(mi & ~mn & lt)] =
                        sup_ent(bound, q);
                n += (int)__popcll(mi);
                nn += (int)__popcll(mn);
            }
        }
        if (lane == 0) {
            if (FILL) {
                S.x0[k] = make_double2(me.x, me.y);
            } else {
                S.scnt[k] = n;
                S.snear[k] = nn;
            }
        }
    }
}

// ---------------------------------------------------------------------
// 3. speculative events + per-floe gather + owner state writes
// ---------------------------------------------------------------------
// Contact state of pair (i, j), owner i by storage slot, partner j by
// identity: history, last contact forces and whether it is bonded.  Returns
// whether it has a history.
__device__ __forceinline__ bool load_contact_state(const DS& S, int i, int j, int2 counts, PairState& ps) {
    ps.deltat = 0.0; ps.thetarelc = 0.0; ps.fcn = 0.0; ps.fct = 0.0;
    ps.bond = 0; ps.has_bond_rec = false;
    ps.damage = ps.deltanb = ps.deltatb = ps.trb_ji = ps.trb_ij = 0.0;
    ps.rb = ps.hb = ps.lb = ps.sb = ps.ib = 0.0;
    // both lists are searched at once, the first two records of each
    // requested together
    const int hq = find_partner<2>(S.hist_old, S.S, i, counts.x, j);
    const int bq = find_partner<2>(S.bond_old, S.S, i, counts.y, j);
    if (hq >= 0) {
        const HistRec& hr = S.hist_old[(int64_t)hq * S.S + i];
        ps.deltat = hr.deltat; ps.thetarelc = hr.thetarelc; ps.fcn = hr.fcn; ps.fct = hr.fct;
    }
    if (bq >= 0) {
        ps.has_bond_rec = true;
        ps.bond = S.bond_old[(int64_t)bq * S.S + i].bond;
    }
    return hq >= 0;
}

// Contact terms of the queued floes (contact_forces, plastic_contact,
// update_shape, coulomb; stepper.f90:103-146) + the owner's new histories.
// The (floe, candidate) pairs of a wavefront's floes are evaluated together,
// 64 a pass, one per lane (each lane finds its pair's floe among the lanes
// by a binary search over their offsets): a floe's inner pairs (ascending
// outer index) first, then its own candidates in distance order.  Each pass
// leaves every pair's contact terms and history outcome in LDS, and every
// floe then adds its own, in order: the same additions in the same order as
// a floe's own walk, without one lane holding the wavefront through a long
// list.
struct ContactOut {
    double fcn_c, fcr_s, fcn_s, fcr_c, r_fct, mcc, ac, fcn_ac;   // the floe's side of the terms
    double deltat, thetarelc, fcn, fct;                           // history to append (owner side)
    int32_t j;
    uint32_t kind;     // bit 0: contact terms, bit 1: history record to append
};
constexpr int CONTACT_LDS_PER_WAVE = 64 * (int)sizeof(ContactOut);

template <bool MIXED>
__device__ __forceinline__ void contacts(const DS& S, const QueueBlocks& qb, ContactOut* co) {
    const int lane = (int)(threadIdx.x & 63);
    const QueueView qv = queue_view(S, 0);
    // (the wavefront's lanes share LDS and shuffles: every lane runs each
    // round, whether or not it has an entry)
    const QueueShare qs = queue_share(S, qb, qv.total);
    for (int t0 = qs.begin; t0 < qs.end; t0 += qs.stride) {
        const int qt = t0 + lane;
        const int k = lane < qs.floes && qt < qs.end ? queue_at(S, 0, qv, qt) : -1;
        const bool act = k >= 0;
        const int64_t SS = S.S;
        int m = 0, f = 0, fs = 0, ni = 0, no = 0;
        uint32_t rc = 0;
        if (act) {
            const GeoRec me = S.geo[k];
            m = me.member;
            f = me.id;                  // identity (ordering, bond mask)
            fs = S.cval[k];             // storage slot of the floe's pair state
            ni = S.icnt[k];
            no = S.ocnt[k];
            rc = S.rcnt[k];
        }
        const int cnt = ni + no;
        const int incl = wave_scan(cnt);
        const int start = incl - cnt, total = wave_last(incl);
        double afx = 0.0, afy = 0.0, amc = 0.0, atac = 0.0, apc = 0.0;
        int nh = 0;
        uint32_t over = 0;
        for (int c0 = 0; c0 < total; c0 += 64) {
            const int idx = c0 + lane;
            int own = 0;
#pragma unroll
            for (int step = 32; step > 0; step >>= 1)
                if (__shfl(start, own + step) <= idx) own += step;
            const int ko = __shfl(k, own), om = __shfl(m, own), of = __shfl(f, own);
            const int ofs = __shfl(fs, own), oni = __shfl(ni, own), ostart = __shfl(start, own);
            const uint32_t orc = (uint32_t)__shfl((int)rc, own);
            ContactOut r;
            r.kind = 0;
            if (idx < total) {
                const DevParams& P = S.params[om];
                const int tstep = S.members[om].tstep;
                const int first = S.members[om].first;
                const int local = idx - ostart;
                // overlap first from the position rows alone (the expression
                // kinematics evaluates, so the same decision); the full rows
                // only for contacts
                const GeoRec gf = S.geo[ko];
                if (local < oni) {
                    // pair (i, f), f the inner floe: only overlapping pairs contribute
                    const int64_t e = S.ik[(int64_t)local * SS + ko];
                    const int i = ent_id(e), qi = ent_pos(e);
                    const GeoRec gi = S.geo[qi];
                    const int si = S.cval[qi];
                    const uint32_t irc = S.rcnt[qi];
                    const double dx = gi.x - gf.x, dy = gi.y - gf.y;
                    const double dn = gi.r + gf.r - sqrt(dx * dx + dy * dy);
                    if (dn > 0) {
                        Floe Fi = floe_at(S, qi);
                        Floe Fj = floe_at(S, ko);
                        Kin kn;
                        kinematics(Fi, Fj, kn);
                        PairState ps;
                        load_contact_state(S, si, of, record_counts(irc), ps);
                        bond_create(P, tstep, i - first, of - first, Fi, Fj, kn, ps);
                        EventOut o;
                        o.flags = 0;
                        o.ridged = -1;
                        contact_part<MIXED>(P, Fi, Fj, kn, ps, o);
                        r.kind = 1;
                        r.fcn_c = o.fcn_c; r.fcr_s = o.fcr_s; r.fcn_s = o.fcn_s; r.fcr_c = o.fcr_c;
                        r.r_fct = o.rj_fct; r.mcc = o.mcc; r.ac = o.ac; r.fcn_ac = o.fcn_ac;
                    }
                } else {
                    // pair (f, j), f the outer floe (the owner)
                    const int s = local - oni;
                    const int64_t e = S.oj[(int64_t)s * SS + ko];
                    const int j = ent_id(e), qj = ent_pos(e);
                    const GeoRec gj = S.geo[qj];
                    const double dx = gf.x - gj.x, dy = gf.y - gj.y;
                    const double dn = gf.r + gj.r - sqrt(dx * dx + dy * dy);
                    r.j = j;
                    if (!(dn > 0)) {
                        // reset_contact (reset.f90:1-15): the history goes, the
                        // last contact forces stay
                        const int q = find_partner<2>(S.hist_old, SS, ofs, record_counts(orc).x, j);
                        if (q >= 0) {
                            const HistRec& h0 = S.hist_old[(int64_t)q * SS + ofs];
                            if (h0.fcn != 0.0 || h0.fct != 0.0) {
                                r.kind = 2;
                                r.deltat = 0.0; r.thetarelc = 0.0; r.fcn = h0.fcn; r.fct = h0.fct;
                                if (S.record_forces) {
                                    PairState pz;
                                    pz.fcn = h0.fcn; pz.fct = h0.fct;
                                    S.ssc[(int64_t)s * SS + ko] = stale_contact_magnitude<MIXED>(pz);
                                }
                            }
                        }
                    } else {
                        Floe Fi = floe_at(S, ko);
                        Floe Fj = floe_at(S, qj);
                        Kin kn;
                        kinematics(Fi, Fj, kn);
                        PairState ps;
                        const bool had = load_contact_state(S, ofs, j, record_counts(orc), ps);
                        bond_create(P, tstep, of - first, j - first, Fi, Fj, kn, ps);
                        EventOut o;
                        o.flags = 0;
                        o.ridged = -1;
                        contact_part<MIXED>(P, Fi, Fj, kn, ps, o);
                        atomicOr(&S.evf[(int64_t)s * SS + ko], o.flags);   // (k_bond sets bits too)
                        if (S.record_forces) S.ssc[(int64_t)s * SS + ko] = o.sc;
                        r.kind = 1;
                        r.fcn_c = o.fcn_c; r.fcr_s = o.fcr_s; r.fcn_s = o.fcn_s; r.fcr_c = o.fcr_c;
                        r.r_fct = o.ri_fct; r.mcc = o.mcc; r.ac = o.ac; r.fcn_ac = o.fcn_ac;
                        if (ps.deltat != 0.0 || ps.thetarelc != 0.0 || ps.fcn != 0.0 || ps.fct != 0.0) {
                            r.kind |= 2;
                            r.deltat = ps.deltat; r.thetarelc = ps.thetarelc; r.fcn = ps.fcn; r.fct = ps.fct;
                            if (!had) sup_keep(S, ko, qj);
                        }
                        if (o.flags & EV_RIDGED) {
                            const int p = atomicAdd(&S.nseeds[om], 1);
                            if (p < S.SEEDK * S.members[om].n)
                                add_reshape(S, S.shape + (int64_t)S.SEEDK * first, p,
                                            ((int64_t)(of - first) << 16) | s, o.ridged == 0 ? ko : qj,
                                            ko, qj, o.nr, o.nh, o.nmass, o.ninertia, o.nhfa, o.nhfw);
                            else
                                over |= ERR_SEED_CAP;
                        }
                    }
                }
            }
            co[lane] = r;
            wave_lds_sync();
            // every floe adds this pass's terms of its own, in order
            if (act) {
                const int lo = max(start, c0), hi = min(start + cnt, c0 + 64);
                for (int i2 = lo; i2 < hi; ++i2) {
                    const ContactOut& t = co[i2 - c0];
                    if (t.kind & 1) {
                        if (i2 - start < ni) {
                            afx = afx + t.fcn_c - t.fcr_s;
                            afy = afy + t.fcn_s + t.fcr_c;
                            amc = amc - t.r_fct + t.mcc;
                        } else {
                            afx = afx - t.fcn_c + t.fcr_s;
                            afy = afy - t.fcn_s - t.fcr_c;
                            amc = amc - t.r_fct - t.mcc;
                        }
                        atac = atac + t.ac;
                        apc = apc - t.fcn_ac;
                    }
                    if (t.kind & 2) {
                        if (nh < S.HC) {
                            HistRec hr; hr.j = t.j; hr.pad_ = 0; hr.deltat = t.deltat; hr.thetarelc = t.thetarelc;
                            hr.fcn = t.fcn; hr.fct = t.fct;
                            S.hist_new[(int64_t)nh * SS + fs] = hr;
                            ++nh;
                        } else {
                            over |= ERR_HIST_CAP;
                        }
                    }
                }
            }
            wave_lds_sync();
        }
        if (act) {
            // contact histories of pairs that are not candidates this step
            // persist (the reference only resets a candidate pair, reset_contact)
            const int hco = record_counts(rc).x;
            const Peek po = peek_entries(S.oj, SS, k, hco > 0 ? no : 0);
            for (int q = 0; q < hco; ++q) {
                HistRec hr = S.hist_old[(int64_t)q * SS + fs];
                if (hr.j < 0) continue;
                int64_t e;
                const bool cand = find_peeked(po, S.oj, SS, k, no, hr.j, e) >= 0;
                if (!cand) {
                    if (nh < S.HC) S.hist_new[(int64_t)nh * SS + fs] = hr, ++nh;
                    else over |= ERR_HIST_CAP;
                }
            }
            S.hcnt_new[fs] = nh;
            S.acc[A_FCX * SS + k] = afx;
            S.acc[A_FCY * SS + k] = afy;
            S.acc[A_MC * SS + k] = amc;
            S.acc[A_TAC * SS + k] = atac;
            S.acc[A_PC * SS + k] = apc;
        }
        if (over) set_err(S, over);
    }
}

// One bond event of owner f (position k, storage slot fs, floe F0): pair
// (f, j) at outer slot s, written to record rq (new records: rq < 0, appended
// at nb if the event leaves one).  Returns whether the pair is bonded after
// it (the floes then have bond terms to gather).
template <bool MIXED>
__device__ __forceinline__ bool bond_event(const DS& S, const DevParams& P, int tstep, int first,
                                           int f, int k, int fs, const Floe& F0, int s, int64_t e,
                                           int rq, int& nb, PairState& ps, uint32_t& over) {
    const int64_t SS = S.S;
    const int j = ent_id(e), qj = ent_pos(e);
    Floe Fi = F0;
    Floe Fj = floe_at(S, qj);
    const int nij = S.icnt[qj];
    Kin kn;
    kinematics(Fi, Fj, kn);
    // (the partner's inner list, searched at the end, arrives meanwhile)
    const Peek pij = peek_entries(S.ik, SS, qj, nij);
    bond_create(P, tstep, f - first, j - first, Fi, Fj, kn, ps);
    if (!ps.has_bond_rec) return false;
    EventOut o;
    o.flags = 0;
    o.ridged = -1;
    o.sbd = 0.0;
    bond_part<MIXED>(P, Fi, Fj, kn, ps, o);
    if (S.record_forces) S.ssb[s * SS + k] = o.sbd;
    if (rq < 0) {
        if (nb < S.BC) rq = nb++;
        else { over |= ERR_BOND_CAP; return false; }
        sup_keep(S, k, qj);
    }
    S.bond_new[(int64_t)rq * SS + fs] = bond_from(ps, j);
    if (!(o.flags & EV_BONDED)) return false;
    BondTerms bt;
    bt.fbn_c = o.fbn_c; bt.fbt_s = o.fbt_s; bt.fbn_s = o.fbn_s; bt.fbt_c = o.fbt_c;
    bt.lri_fbt = o.lri_fbt; bt.lrj_fbt = o.lrj_fbt; bt.mbb_ji = o.mbb_ji; bt.mbb_ij = o.mbb_ij;
    bt.sb = o.sb; bt.fbn_sb = o.fbn_sb;
    S.bterm[(int64_t)rq * SS + k] = bt;          // (by the owner's position)
    atomicOr(&S.evf[s * SS + k], EV_BONDED | ((uint32_t)(rq + 1) << 16));   // (as k_contact)
    // tell the partner where its terms are: its inner slot of f
    int64_t eij;
    const int qi = find_peeked(pij, S.ik, SS, qj, nij, f, eij);
    if (qi >= 0) S.ibond[(int64_t)qi * SS + qj] = rq + 1;
    S.bgat[qj] = 1;
    return true;
}

// Old record b of the owner at record index rq of the new list: a record
// whose partner is a candidate this step takes part in an event (its new
// values replace it), the others carry over unchanged.
template <bool MIXED>
__device__ __forceinline__ bool bond_record(const DS& S, const DevParams& P, int tstep, int first,
                                            int f, int k, int fs, const Floe& F0, int no,
                                            const Peek& po, const BondRec& b, int rq, int& nb,
                                            uint32_t& over) {
    int64_t e;
    const int s = find_peeked(po, S.oj, S.S, k, no, b.j, e);
    if (s < 0) {
        S.bond_new[(int64_t)rq * S.S + fs] = b;
        return false;
    }
    PairState ps;
    ps.deltat = 0.0; ps.thetarelc = 0.0; ps.fcn = 0.0; ps.fct = 0.0;
    ps.has_bond_rec = true; ps.bond = b.bond; ps.damage = b.damage;
    ps.deltanb = b.deltanb; ps.deltatb = b.deltatb; ps.trb_ji = b.trb_ji; ps.trb_ij = b.trb_ij;
    ps.rb = b.rb; ps.hb = b.hb; ps.lb = b.lb; ps.sb = b.sb; ps.ib = b.ib;
    return bond_event<MIXED>(S, P, tstep, first, f, k, fs, F0, s, e, rq, nb, ps, over);
}

// (owner lane, record, new record index) triples of one wavefront, evaluated
// one per lane
constexpr int BOND_TCAP = 256;

// Bond events of the queued owners (bond_forces_euler, bond_breaking;
// stepper.f90:148-198): each bond is evaluated once, by its owner (the lower
// index), which writes the new record and the event's terms for both floes;
// k_final then sums every floe's terms in the reference's order.  An
// owner's records keep their order, cleared ones dropped: record q goes to
// the new index rq = the number of live records before it.  The wavefront's
// records are listed in LDS and evaluated one per lane, so that an owner with
// several bonds does not hold its lane through all of them; owners whose
// bonds form this step (step 1) append new records in candidate order and
// walk their own lists.
template <bool MIXED>
__device__ __forceinline__ void bonds(const DS& S, const QueueBlocks& qb, uint32_t* rl) {
    const QueueView qv = queue_view(S, 1);
    // (the wavefront loops while any lane has an entry: its lanes share LDS
    // and shuffles)
    const QueueShare qs = bond_share(qb, qv.total);
    for (int t0 = qs.begin; t0 < qs.end; t0 += qs.stride) {
        const int qt = t0 + (int)(threadIdx.x & 63);
        const int k = qt < min(t0 + qs.floes, qs.end) ? queue_at(S, 1, qv, qt) : -1;
        const bool act = k >= 0;
        const int lane = (int)(threadIdx.x & 63);
        const int64_t SS = S.S;
        int m = 0, fs = 0, no = 0, bco = 0, fid = 0, tstep = 0, first = 0;
        bool bond_step = false;
        // partners of the first LIST_PEEK records, requested together
        int id[LIST_PEEK];
        if (act) {
            const GeoRec g = S.geo[k];
            fs = S.cval[k];
            no = S.ocnt[k];
            bco = record_counts(S.rcnt[k]).y;
            // (a queued owner has at least one record)
#pragma unroll
            for (int q = 0; q < LIST_PEEK; ++q) id[q] = S.bond_old[(int64_t)min(q, max(bco - 1, 0)) * SS + fs].j;
            m = g.member;
            fid = g.id;
            // (no short-circuit tests: the loads go out together)
            const DevParams& P = S.params[m];
            const Member Mb = S.members[m];
            const int rst = P.restart, coh = P.cohesion;
            tstep = Mb.tstep;
            first = Mb.first;
            bond_step = (tstep == 1) & (rst != 1) & (coh != 0);
#pragma unroll
            for (int q = 0; q < LIST_PEEK; ++q) id[q] = q < bco ? id[q] : -1;
        }
        // the live records of the owners that form no bonds this step
        int nlive = 0;
        uint32_t over = 0;
        const bool listed = act && !bond_step;
        if (listed) {
#pragma unroll
            for (int q = 0; q < LIST_PEEK; ++q) nlive += id[q] >= 0;
            for (int q = LIST_PEEK; q < bco; ++q) nlive += S.bond_old[(int64_t)q * SS + fs].j >= 0;
        }
        const int incl = wave_scan(nlive);
        const int total = wave_last(incl);
        const bool fits = total <= BOND_TCAP;
        if (fits) {
            if (listed) {
                int at = incl - nlive, rq = 0;
                auto list_rec = [&](int q) {
                    rl[at++] = (uint32_t)lane | ((uint32_t)q << 6) | ((uint32_t)rq << 19);
                    ++rq;
                };
#pragma unroll
                for (int q = 0; q < LIST_PEEK; ++q)
                    if (id[q] >= 0) list_rec(q);    // (-1 past the count)
                for (int q = LIST_PEEK; q < bco; ++q)
                    if (S.bond_old[(int64_t)q * SS + fs].j >= 0) list_rec(q);
                S.bcnt_new[fs] = nlive;
            }
            wave_lds_sync();
            for (int c0 = 0; c0 < total; c0 += 64) {
                const int idx = c0 + lane;
                const uint32_t w = idx < total ? rl[idx] : (uint32_t)lane;
                const int own = (int)(w & 63);
                // the owner's member, step and identity, from its lane
                const int ko = __shfl(k, own), mo = __shfl(m, own), fso = __shfl(fs, own);
                const int noo = __shfl(no, own), fo = __shfl(fid, own);
                const int tso = __shfl(tstep, own), fro = __shfl(first, own);
                if (idx < total) {
                    const int q = (int)((w >> 6) & 0x1FFF), rq = (int)(w >> 19);
                    const DevParams& P = S.params[mo];
                    const Floe F0 = floe_at(S, ko);
                    const BondRec b = S.bond_old[(int64_t)q * SS + fso];
                    const Peek po = peek_entries(S.oj, SS, ko, noo);
                    int nb = 0;
                    if (bond_record<MIXED>(S, P, tso, fro, fo, ko, fso, F0, noo, po, b, rq, nb, over))
                        S.bgat[ko] = 1;
                }
            }
        }
        if (act && (bond_step || !fits)) {
            const GeoRec me = S.geo[k];
            const DevParams& P = S.params[m];
            const int tstep = S.members[m].tstep;
            const int first = S.members[m].first;
            const int f = me.id;
            const Floe F0 = floe_at(S, k);
            const Peek po = peek_entries(S.oj, SS, k, no);
            bool any = false;
            int nb = 0;                     // records written so far
            for (int q = 0; q < bco; ++q) {
                const BondRec b = S.bond_old[q * SS + fs];
                if (b.j < 0) continue;
                const int rq = nb++;
                any |= bond_record<MIXED>(S, P, tstep, first, f, k, fs, F0, no, po, b, rq, nb, over);
            }
            // bonds that form this step (bond_create), in candidate order, appended
            if (bond_step) {
                const int nb_old = nb;
                for (int s = 0; s < no; ++s) {
                    const int64_t e = S.oj[s * SS + k];
                    const int j = ent_id(e);
                    bool has = false;
                    for (int q = 0; q < nb_old; ++q)
                        if (S.bond_new[(int64_t)q * SS + fs].j == j) { has = true; break; }
                    if (has) continue;
                    PairState ps;
                    ps.deltat = 0.0; ps.thetarelc = 0.0; ps.fcn = 0.0; ps.fct = 0.0;
                    ps.bond = 0; ps.has_bond_rec = false;
                    ps.damage = ps.deltanb = ps.deltatb = ps.trb_ji = ps.trb_ij = 0.0;
                    ps.rb = ps.hb = ps.lb = ps.sb = ps.ib = 0.0;
                    any |= bond_event<MIXED>(S, P, tstep, first, f, k, fs, F0, s, e, -1, nb, ps, over);
                }
            }
            if (any) S.bgat[k] = 1;
            S.bcnt_new[fs] = nb;
        }
        if (over) set_err(S, over);
    }
}

// Bond rows of a floe with a bonded event (position k), added to a[] (rows
// at zero): the terms its owners wrote, first the pairs
// where it is the inner index (ascending outer index), then its own, in
// distance order (stepper.f90:165-198).  k_final calls it for the floes the
// repair left alone: their flags and terms are k_bond's.
__device__ __forceinline__ void gather_bonds(const DS& S, int k, int ni, int no, double* a) {
    const int64_t SS = S.S;
    // the first GATHER_PEEK slots' bond words and inner partners of both sides
    // are requested together (slots past a count stand in for its last one)
    int rqi[GATHER_PEEK], rqo[GATHER_PEEK], pki[GATHER_PEEK];
#pragma unroll
    for (int q = 0; q < GATHER_PEEK; ++q) rqi[q] = rqo[q] = pki[q] = 0;
    if (ni > 0) {
#pragma unroll
        for (int q = 0; q < GATHER_PEEK; ++q) {
            const int64_t r = (int64_t)min(q, ni - 1) * SS + k;
            rqi[q] = S.ibond[r];
            pki[q] = ent_pos(S.ik[r]);
        }
    }
    if (no > 0) {
#pragma unroll
        for (int q = 0; q < GATHER_PEEK; ++q) rqo[q] = (int)S.evf[(int64_t)min(q, no - 1) * SS + k];
    }
#pragma unroll
    for (int q = 0; q < GATHER_PEEK; ++q) {
        rqi[q] = q < ni ? rqi[q] : 0;
        rqo[q] = q < no ? rqo[q] : 0;
    }
    auto inner = [&](int pk, int rq) {
        if (rq) add_bond_j(a, S.bterm[(int64_t)(rq - 1) * SS + pk]);
    };
    auto outer = [&](uint32_t fl) {
        const int rq = (int)(fl >> 16);
        if ((fl & EV_BONDED) && rq >= 1 && rq <= S.BC) add_bond_i(a, S.bterm[(int64_t)(rq - 1) * SS + k]);
    };
#pragma unroll
    for (int q = 0; q < GATHER_PEEK; ++q) inner(pki[q], rqi[q]);
    for (int q = GATHER_PEEK; q < ni; ++q) inner(ent_pos(S.ik[q * SS + k]), S.ibond[q * SS + k]);
#pragma unroll
    for (int s = 0; s < GATHER_PEEK; ++s) outer((uint32_t)rqo[s]);
    for (int s = GATHER_PEEK; s < no; ++s) outer(S.evf[s * SS + k]);
}

// Walls of the queued floes (verify_bc, boundaries.f90:1-97).
template <bool MIXED>
__device__ __forceinline__ void wall_contacts(const DS& S, const QueueBlocks& qb) {
    // no later kernel of the step reads the build flag; k_final raises it
    // again when a floe has moved too far for the supersets
    if (qb.xcd == 0 && qb.block == 0 && threadIdx.x == 0) { S.rebuild[0] = 0; S.rebuild[1] = 0; }
    const QueueView qv = queue_view(S, 2);
    for (int it = 0;; ++it) {
        const int t = queue_slot_it(qb, qv.total, it);
        if (t < 0) break;
        const int k = queue_at(S, 2, qv, t);
        const GeoRec me = S.geo[k];
        const int m = me.member;
        const DevParams& P = S.params[m];
        const int first = S.members[m].first;
        const int f = me.id;
        const int fs = S.cval[k];
        const int64_t SS = S.S;
        Floe Fw = floe_at(S, k);
        double hist[4] = {S.wbc[0 * SS + fs], S.wbc[1 * SS + fs], S.wbc[2 * SS + fs], S.wbc[3 * SS + fs]};
        WallOut W;
        walls<MIXED>(P, Fw, hist, W);
        S.wflag[k] = (uint8_t)((W.flags & 1u) ? WF_WALL : 0u);
        if (W.flags & 1u) S.wout[k] = W;
        if (W.flags & 4u) {
            int p = atomicAdd(&S.nseeds[m], 1);
            if (p < S.SEEDK * S.members[m].n)
                add_reshape(S, S.shape + (int64_t)S.SEEDK * first, p,
                            ((int64_t)(f - first) << 16) | WALL_SLOT, k, k, -1, W.nr, W.nh, W.nmass,
                            W.ninertia, W.nhfa, W.nhfw);
            else
                set_err(S, ERR_SEED_CAP);
        }
    }
}

// The three kinds of events of a step: they touch disjoint state (the flag
// words that both contacts and bonds set are set with atomicOr), so they run
// in one launch, single-wavefront blocks of contacts and bonds alternating so
// that both are under way from the start, the few of the walls first.  (One
// launch instead of three on two streams takes the fork, the join and two
// kernel starts out of the step: with the steps' k_begin gone as well, 94 ->
// 76 us a step at 1,000 floes in mixed precision and 145 -> 126 us at 24
// members of 2,700; at 512 members, where each kind fills the chip by itself,
// it is the same to 1%.)  Steps timed stage by stage run
// them one after another, in the kernels below.
template <bool MIXED>
__global__ __launch_bounds__(64, 3) void k_events(DS S, int nwall, int ncontact, int nbond) {
    extern __shared__ __align__(16) unsigned char ev_lds[];
    if (*S.err) return;
    QueueBlocks qb;
    qb.xcd = (int)(blockIdx.x % XCD_COUNT);
    int b = (int)(blockIdx.x / XCD_COUNT);
    if (b < nwall) {
        qb.block = b;
        qb.blocks = nwall;
        wall_contacts<MIXED>(S, qb);
        return;
    }
    b -= nwall;
    const int both = 2 * min(ncontact, nbond);
    const bool contact = b < both ? (b & 1) == 0 : ncontact > nbond;
    qb.block = b < both ? b >> 1 : b - both / 2;
    if (contact) {
        qb.blocks = ncontact;
        contacts<MIXED>(S, qb, reinterpret_cast<ContactOut*>(ev_lds));
    } else {
        qb.blocks = nbond;
        bonds<MIXED>(S, qb, reinterpret_cast<uint32_t*>(ev_lds));
    }
}
static_assert(BOND_TCAP * 4 <= CONTACT_LDS_PER_WAVE, "k_events' LDS holds either list");

template <bool MIXED>
__global__ __launch_bounds__(FLOE_BLOCK, 3) void k_contact(DS S) {
    extern __shared__ unsigned char contact_lds[];
    if (*S.err) return;
    contacts<MIXED>(S, queue_blocks(), reinterpret_cast<ContactOut*>(contact_lds + (threadIdx.x >> 6) * CONTACT_LDS_PER_WAVE));
}
template <bool MIXED>
__global__ __launch_bounds__(FLOE_BLOCK, 3) void k_bond(DS S) {
    __shared__ uint32_t recs[FLOE_BLOCK / 64][BOND_TCAP];
    if (*S.err) return;
    bonds<MIXED>(S, queue_blocks(), recs[threadIdx.x >> 6]);
}
template <bool MIXED>
__global__ __launch_bounds__(FLOE_BLOCK) void k_walls(DS S) {
    if (*S.err) return;
    wall_contacts<MIXED>(S, queue_blocks());
}

// ---------------------------------------------------------------------
// 4. ordered repair, one member per block
//
// An event reads the radius, thickness, mass and drafts of its two floes and
// only a reshape changes those, so the result of the reference's sequence is
// fixed by the reshapes alone: for every event that ridges, which floe it
// reshapes and to what.  Events are named by their place in the sequence, key
// (outer local index << 16 | slot), and each floe has a list of its reshape
// records; an event takes the properties of the last record before its key.
// Only a floe's contacts and walls can reshape it, and radii only shrink, so
// the events that can ridge are the contacts and walls the event kernels
// found at the start-of-step radii.
//
// The records start as the seeds (what ridges with the start-of-step
// properties).  Round by round, every contact and wall event that comes after
// a record that changed, on the same floe, is evaluated again, all of a
// member's at once; one whose outcome differs from its record updates it,
// which is a change for the next round.  When nothing changes, each event's
// outcome follows from the records before it, and by induction over the keys
// that is the sequence's own outcome, whatever order the rounds took.  The
// rounds a member needs are the longest chain of reshapes that act on each
// other, not the number of events behind them.
//
// What it costs is the chain of dependent loads of a round (event -> rows ->
// records), about 8 us; most members have a handful of seeds, one round that
// finds no later contact, and the closing pass that queues the floes whose
// terms change.  (One MI355X, against committing the events in key order 64
// at a time, which also took every candidate after a reshape through the
// rounds and went on one event at a time past 1,024 pending: 262,144 floes of
// one field with 43 candidates a floe and 80 seeds, FP64, 20 -> 0.043 ms per
// step; 24 such fields, 320,000 floes, mixed, 0.23-0.9 -> 0.023; 2,501 floes
// with 50 seeds 0.26 -> 0.027; the 512-field ensemble 0.064 -> 0.026.)
// ---------------------------------------------------------------------
constexpr int REPAIR_ROUNDS = 1 << 20;   // (never reached: every round settles one more key)

// slot of partner id g in the outer list of the floe at position kp
__device__ __forceinline__ int slot_of(const DS& S, int kp, int g) {
    return find_entry(S.oj, S.S, kp, S.ocnt[kp], g);
}

// Sets bits of position k's wflag byte; returns the byte as it was.
__device__ __forceinline__ uint32_t wflag_fetch_set(const DS& S, int k, uint32_t bits) {
    const int sh = 8 * (k & 3);
    return (atomicOr(reinterpret_cast<uint32_t*>(S.wflag + (k & ~3)), bits << sh) >> sh) & 255u;
}
__device__ __forceinline__ void wflag_clear(const DS& S, int k, uint32_t bits) {
    atomicAnd(reinterpret_cast<uint32_t*>(S.wflag + (k & ~3)), ~(bits << (8 * (k & 3))));
}
// a record list's head, changed by other wavefronts of the block
__device__ __forceinline__ int rhead_at(const DS& S, int k) {
    return __hip_atomic_load(S.rhead + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The floe at position k joins the fix-up queue (once).
__device__ __forceinline__ void touch_floe(const DS& S, int k) {
    if (!(wflag_fetch_set(S, k, WF_FIXUP) & WF_FIXUP)) enqueue_one(S, 4, k);
}

// The events after a record of the floe at kg: its inner pairs of later outer
// floes, its own candidates from slot s0 on, its walls.  A wavefront takes
// the records of its lanes together, 64 events at a time.
struct LaterEvents {
    int ni, s0, no;        // inner entries (0: none is later), own slots [s0, s0 + no)
    int f;                 // local index of the record's outer floe
};
__device__ __forceinline__ LaterEvents later_events(const DS& S, int64_t key, int kg, int gid, int first) {
    LaterEvents l;
    const int s = (int)(key & 0xFFFF);
    l.f = (int)(key >> 16);
    const bool own = gid - first == l.f;          // the record's event is one of the floe's own
    const int ni = S.icnt[kg], no = S.ocnt[kg];
    l.ni = own ? 0 : ni;
    l.s0 = own ? s + 1 : 0;
    l.no = s == WALL_SLOT ? 0 : max(no - l.s0, 0);
    if (s == WALL_SLOT) l.ni = 0;                 // (a floe's walls are its last event)
    return l;
}

template <bool MIXED>
__global__ __launch_bounds__(REPAIR_THREADS) void k_repair(DS S, int nmembers, int list) {
    // events to evaluate (outer position << 16 | slot) and records that
    // changed, `list` entries of each
    extern __shared__ __align__(16) unsigned char repair_lds[];
    uint64_t* wl = reinterpret_cast<uint64_t*>(repair_lds);
    int* cl = reinterpret_cast<int*>(repair_lds + 8 * (size_t)list);
    __shared__ int nw_, nc_, nn_, rep_, ns_, nt_, first_, nmem_, tstep_;
    __shared__ int64_t mean_;
    __shared__ uint32_t over_;
    // the member's parameters: the physics reads them at LDS latency
    __shared__ uint64_t pbuf[sizeof(DevParams) / 8];
    static_assert(sizeof(DevParams) % 8 == 0 && sizeof(DevParams) / 8 <= 64, "DevParams copied by lane");
    const int m = blockIdx.x;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    if (m >= nmembers) return;
    // (the parameters and the mean superset length of the last build are
    // requested beside the seed count, by other wavefronts where the block has
    // some: by the first one, a microsecond later)
    const int lastw = (int)(blockDim.x >> 6) - 1;
    if ((tid >> 6) == min(1, lastw) && lane < (int)(sizeof(DevParams) / 8))
        pbuf[lane] = reinterpret_cast<const uint64_t*>(S.params + m)[lane];
    if (tid == 64 * min(2, lastw)) mean_ = 1 + S.sblk[(S.N + SCAN_TILE - 1) / SCAN_TILE] / S.N;
    // (the error word is read once for the block: all its wavefronts take the
    // barriers below or none does)
    if (tid == 0) {
        const uint32_t err = *S.err;
        const int n = S.nseeds[m];
        const Member M = S.members[m];
        ns_ = err || !member_live(M) ? 0 : min(n, S.SEEDK * M.n);
        nn_ = ns_;
        nw_ = nc_ = rep_ = nt_ = 0;
        over_ = 0;
        first_ = M.first; nmem_ = M.n; tstep_ = M.tstep;
    }
    __syncthreads();
    const int ns = ns_;
    if (ns == 0) return;
    // as many of the block's wavefronts as the events after the seeds fill (by
    // the mean superset length of the last build); where the caller allows fewer than
    // 64 lanes, the first wavefront with those
    const int lanes = min(max(S.repair_lanes, 1), 64);
    int waves = 1;
    if (lanes == 64) {
        waves = (int)min((int64_t)(blockDim.x / 64), ((int64_t)ns * mean_ + 63) / 64);
    }
    const int width = lanes < 64 ? lanes : waves * 64;
    if (tid >= waves * 64) return;
    // records a wavefront takes at once from a list of n
    auto share = [&](int n) { return min(lanes, (n + waves - 1) / waves); };
    const DevParams& P = *reinterpret_cast<const DevParams*>(pbuf);
    const int first = first_, nmem = nmem_, tstep = tstep_;
    const int64_t SS = S.S;
    Reshape* rec = S.shape + (int64_t)S.SEEDK * first;
    const int reccap = S.SEEDK * nmem;
    // lists beyond LDS: the member's share of `heap`, half for each
    const int cap = min(max(S.repair_cap, 1), list);
    uint64_t* whbm = S.heap + (int64_t)S.HEAPK * first;
    const int hcap = S.HEAPK / 2 * nmem;
    uint64_t* chbm = whbm + hcap;
    uint32_t over = 0;
    auto put_event = [&](int k, int s) {
        const uint64_t w = ((uint64_t)(uint32_t)k << 16) | (uint32_t)s;
        const int at = atomicAdd(&nw_, 1);
        if (at < cap) wl[at] = w;
        else if (at - cap < hcap) whbm[at - cap] = w;
        else over |= ERR_REPAIR_CAP;
    };
    // floes for the fix-up queue: listed in LDS (the event list's room, which
    // the rounds have done with) and queued together at the end, two atomics
    // one behind the other once instead of for every floe
    auto touch = [&](int k) {
        const int at = atomicAdd(&nt_, 1);
        if (at < list) wl[at] = (uint64_t)(uint32_t)k;
        else touch_floe(S, k);
    };
    auto put_change = [&](int p) {
        const int at = atomicAdd(&nc_, 1);
        if (at < cap) cl[at] = p;
        else if (at - cap < hcap) chbm[at - cap] = (uint64_t)p;
        else over |= ERR_REPAIR_CAP;
    };
    // the records c0 .. of a list of n (at(i): record index), a lane each, and
    // every event after them, fn(record lane's values, event)
    auto each_later = [&](int cnt, auto&& fn) {
        const int incl = wave_scan(cnt);
        const int start = incl - cnt, total = wave_last(incl);
        for (int c0 = 0; c0 < total; c0 += 64) {
            const int idx = c0 + lane;
            int own = 0;
#pragma unroll
            for (int step = 32; step > 0; step >>= 1)
                if (__shfl(start, own + step) <= idx) own += step;
            const int at = idx - __shfl(start, own);
            fn(own, idx < total ? at : -1);
        }
    };
    int nchg = ns;
    bool seeds = true;       // (the first round's changes: the seeds, records 0 .. ns - 1)
    for (int round = 0;; ++round) {
        // ---- the contact and wall events after the changed records
        const int rpw = share(nchg);
        for (int c0 = 0; c0 < nchg; c0 += waves * rpw) {
            const int ci = c0 + (tid >> 6) * rpw + lane;
            const bool act = lane < rpw && ci < nchg;
            int kg = 0, gid = 0, wl1 = 0;
            LaterEvents l{0, 0, 0, 0};
            GeoRec gg;
            gg.x = gg.y = gg.r = 0.0;
            if (act) {
                const int p = seeds ? ci : ci < cap ? cl[ci] : (int)chbm[ci - cap];
                const int64_t key = rec[p].key;
                kg = rec[p].pos;
                gg = S.geo[kg];
                gid = gg.id;
                l = later_events(S, key, kg, gid, first);
                wl1 = (key & 0xFFFF) != WALL_SLOT && (S.wflag[kg] & WF_WALL) ? 1 : 0;
            }
            each_later(l.ni + l.no + wl1, [&](int own, int local) {
                const int ko = __shfl(kg, own), go = __shfl(gid, own), fo = __shfl(l.f, own);
                const int nio = __shfl(l.ni, own), s0 = __shfl(l.s0, own), noo = __shfl(l.no, own);
                const double ox = __shfl(gg.x, own), oy = __shfl(gg.y, own), orr = __shfl(gg.r, own);
                if (local < 0) return;
                int ke = ko, s = WALL_SLOT;
                bool want = true;
                if (local < nio + noo) {
                    const bool inner = local < nio;
                    const int64_t e = inner ? S.ik[(int64_t)local * SS + ko]
                                            : S.oj[(int64_t)(s0 + local - nio) * SS + ko];
                    const int q = ent_pos(e);
                    const GeoRec o = S.geo[q];
                    // the pair's overlap as k_contact evaluates it
                    const double dx = inner ? o.x - ox : ox - o.x, dy = inner ? o.y - oy : oy - o.y;
                    const double dn = (inner ? o.r + orr : orr + o.r) - sqrt(dx * dx + dy * dy);
                    want = dn > 0 && (!inner || ent_id(e) - first > fo);
                    ke = inner ? q : ko;
                    s = inner ? (want ? slot_of(S, q, go) : -1) : s0 + local - nio;
                    want = want && s >= 0;
                }
                if (!want) return;
                const bool listed = s == WALL_SLOT ? (wflag_fetch_set(S, ke, WF_PENDING) & WF_PENDING) != 0
                                                   : (atomicOr(&S.evf[(int64_t)s * SS + ke], EV_PENDING) & EV_PENDING) != 0;
                if (!listed) put_event(ke, s);
            });
        }
        if (over) atomicOr(&over_, over);
        __syncthreads();
        const int nw = min(nw_, cap + hcap);
        const bool stop = nw == 0 || over_ != 0 || round >= REPAIR_ROUNDS;
        __syncthreads();
        if (stop) {
            if (round >= REPAIR_ROUNDS) over |= ERR_REPAIR_CAP;
            break;
        }
        if (tid == 0) { nw_ = 0; nc_ = 0; }
        // ---- their outcome, from the records before them
        for (int w0 = 0; w0 < nw; w0 += width) {
            const bool act = tid < width && w0 + tid < nw;
            int kf = 0, kj = -1, s = WALL_SLOT, who = -1, hf = -1, hj = -1;
            int64_t key = 0;
            double nr = 0.0, nh = 0.0, nmass = 0.0, ninertia = 0.0, nhfa = 0.0, nhfw = 0.0;
            if (act) {
                const int wi = w0 + tid;
                const uint64_t w = wi < cap ? wl[wi] : whbm[wi - cap];
                kf = (int)(w >> 16);
                s = (int)(w & 0xFFFF);
                const int f = S.geo[kf].id;
                key = ((int64_t)(f - first) << 16) | s;
                hf = rhead_at(S, kf);
                Floe Fi = floe_at(S, kf);
                if (s == WALL_SLOT) {
                    floe_at_event(rec, hf, key, Fi);
                    double hist[4] = {0.0, 0.0, 0.0, 0.0};   // (no part in a reshape)
                    WallOut W;
                    walls<MIXED>(P, Fi, hist, W);
                    who = (W.flags & 4u) ? 0 : -1;
                    nr = W.nr; nh = W.nh; nmass = W.nmass; ninertia = W.ninertia; nhfa = W.nhfa; nhfw = W.nhfw;
                } else {
                    kj = ent_pos(S.oj[(int64_t)s * SS + kf]);
                    hj = rhead_at(S, kj);
                    Floe Fj = floe_at(S, kj);
                    // the query radius: the outer floe's at the top of its iteration
                    Floe Fq = Fi;
                    floe_at_event(rec, hf, key & ~0xFFFFll, Fq);
                    floe_at_event(rec, hf, key, Fi);
                    floe_at_event(rec, hj, key, Fj);
                    Kin kn;
                    kinematics(Fi, Fj, kn);
                    if (kn.dist <= Fq.r + P.rtree && kn.deltan > 0) {
                        PairState ps{};                      // (no part in a reshape)
                        EventOut o;
                        o.flags = 0;
                        o.ridged = -1;
                        contact_part<MIXED>(P, Fi, Fj, kn, ps, o);
                        if (o.flags & EV_RIDGED) {
                            who = o.ridged;
                            nr = o.nr; nh = o.nh; nmass = o.nmass; ninertia = o.ninertia; nhfa = o.nhfa; nhfw = o.nhfw;
                        }
                    }
                }
            }
            __syncthreads();        // every outcome is known before a record changes
            if (act) {
                int xf = -1, xj = -1;      // the event's records, of either floe
                for (int p = hf; p >= 0; p = rec[p].next)
                    if (rec[p].key == key) xf = p;
                for (int p = hj; p >= 0; p = rec[p].next)
                    if (rec[p].key == key) xj = p;
                if (xf >= 0 && who != 0 && rec[xf].live) { rec[xf].live = 0; put_change(xf); }
                if (xj >= 0 && who != 1 && rec[xj].live) { rec[xj].live = 0; put_change(xj); }
                if (who >= 0) {
                    const int x = who == 0 ? xf : xj;
                    if (x < 0) {
                        const int p = atomicAdd(&nn_, 1);
                        if (p < reccap) {
                            add_reshape(S, rec, p, key, who == 0 ? kf : kj, kf, kj, nr, nh, nmass, ninertia, nhfa, nhfw);
                            put_change(p);
                        } else {
                            over |= ERR_SEED_CAP;
                        }
                    } else if (!rec[x].live || rec[x].r != nr || rec[x].h != nh) {
                        Reshape& w = rec[x];
                        w.r = nr; w.h = nh; w.mass = nmass; w.inertia = ninertia; w.hfa = nhfa; w.hfw = nhfw;
                        w.live = 1;
                        put_change(x);
                    }
                }
                if (s == WALL_SLOT) wflag_clear(S, kf, WF_PENDING);
                else atomicAnd(&S.evf[(int64_t)s * SS + kf], ~EV_PENDING);
            }
            __syncthreads();
        }
        nchg = min(nc_, cap + hcap);
        seeds = false;
        if (nchg == 0) break;
    }
    if (over) atomicOr(&over_, over);
    __syncthreads();
    if (over_) {
        if (tid == 0) set_err(S, over_);
        return;
    }
    // ---- the floes whose terms change: those of every event with a record,
    // every reshaped floe, and the partners of its later events that can
    // notice (in contact, bonded, or near enough for their own sheltering).
    // Counted on the way: the seeds and the events after a reshape of one of
    // their floes (each once), over all candidates, listed or not, so from
    // the supersets.
    const int nn = nn_;
    const bool bond_step = tstep == 1 && P.restart != 1 && P.cohesion;
    const double rtree = P.rtree;
    int counted = 0;
    const int rpw = share(nn);
    for (int c0 = 0; c0 < nn; c0 += waves * rpw) {
        const int p = c0 + (tid >> 6) * rpw + lane;
        const bool act = lane < rpw && p < nn;
        int kg = 0, gid = 0, bown = 0, cnt = 0, fr = 0, idr = 0;
        int64_t soff = 0;
        double dr = -1.0;           // the record's pair, if it is one of the floe's own
        GeoRec gg;
        gg.x = gg.y = gg.r = 0.0;
        if (act) {
            const int64_t key = rec[p].key;
            kg = rec[p].pos;
            const int kf = rec[p].kf, kj = rec[p].kj;
            const bool live = rec[p].live != 0;
            const int ko = kg == kf ? kj : kf;
            // (what follows reads, requested at once)
            gg = S.geo[kg];
            const int h0 = rhead_at(S, kg), h1 = ko >= 0 ? rhead_at(S, ko) : -1;
            const GeoRec gj = S.geo[max(kj, 0)];
            const int scnt = S.scnt[kg];
            soff = S.soff[kg];
            bown = record_counts(S.rcnt[kg]).y;
            touch(kf);
            if (kj >= 0) touch(kj);
            gid = gg.id;
            const int64_t k0 = first_reshape(rec, h0);
            // a seed that is not after a reshape of either floe
            if (p < ns && !(k0 < key) && !(first_reshape(rec, h1) < key)) ++counted;
            // (a floe's walls are its last event)
            if (live && k0 == key && (key & 0xFFFF) != WALL_SLOT) {
                ++counted;           // its walls come after
                cnt = scnt;
                fr = (int)(key >> 16);
                if (kg == kf) {
                    const double dx = gg.x - gj.x, dy = gg.y - gj.y;
                    dr = sqrt(dx * dx + dy * dy);
                    idr = gj.id;
                }
            }
        }
        each_later(cnt, [&](int own, int local) {
            const int go = __shfl(gid, own), fo = __shfl(fr, own), bo = __shfl(bown, own), ido = __shfl(idr, own);
            const int64_t so = __shfl(soff, own);
            const double dro = __shfl(dr, own);
            const double ox = __shfl(gg.x, own), oy = __shfl(gg.y, own), orr = __shfl(gg.r, own);
            if (local < 0) return;
            const int q = ent_pos(S.sup[so + local]);
            const GeoRec o = S.geo[q];
            const bool inner = o.id < go;                 // the floe is the pair's inner one
            const double dx = ox - o.x, dy = oy - o.y;
            const double d = sqrt(dx * dx + dy * dy);
            if (!(d <= (inner ? o.r : orr) + rtree)) return;        // not a candidate
            // after the record: in a later iteration, or later in the same one
            const bool later = dro >= 0.0 ? !inner && (d > dro || (d == dro && o.id > ido))
                                          : !inner || o.id - first > fo;
            if (!later) return;
            const ShelRec sh = S.shel[q];
            const int hq = rhead_at(S, q);
            const int bc = inner ? record_counts(S.rcnt[q]).y : bo;
            // the partner's own reshape may come before the event too: counted
            // from the outer floe's side
            bool both = false;
            if (hq >= 0) {
                const int pq = first_record(rec, hq);
                if (pq >= 0) {
                    const Reshape& w = rec[pq];
                    const int al = (inner ? o.id : go) - first, wf = (int)(w.key >> 16);
                    if (wf != al) {
                        both = wf < al;
                    } else if ((w.key & 0xFFFF) != WALL_SLOT) {
                        const GeoRec a = S.geo[w.kf], b = S.geo[w.kj];
                        const double ex = a.x - b.x, ey = a.y - b.y;
                        const double de = sqrt(ex * ex + ey * ey);
                        both = de < d || (de == d && b.id < (inner ? go : o.id));
                    }
                }
            }
            if (!(both && inner)) ++counted;
            const double dn = orr + o.r - d;
            // (radii only shrink: a term that is exactly 1 stays so)
            using T = typename Prec<MIXED>::T;
            const T lim = sizeof(T) == 4 ? T(20) : T(40), dnt = T(dn);
            const bool far = dnt < T(0) && T((double)0.18f) * -dnt >= lim * T(sh.hfa) &&
                             T((double)0.18f) * -dnt >= lim * T(sh.hfw);
            if (dn > 0 || bc > 0 || (bond_step && dn >= -P.bond_lim) || (P.shelter && !far)) touch(q);
        });
    }
    atomicAdd(&rep_, counted);
    __syncthreads();
    for (int t = tid; t < min(nt_, list); t += waves * 64) touch_floe(S, (int)wl[t]);
    if (tid == 0) {
        S.stats[4 * m + 2] = ns;
        S.stats[4 * m + 3] = rep_;
    }
}

// ---------------------------------------------------------------------
// 5. re-gather floes touched by the repair
// ---------------------------------------------------------------------
// Events of one wavefront's touched floes evaluated together (LDS per
// wavefront: one pass of 64 results).
constexpr int FIX_LDS_PER_WAVE = 64 * (int)sizeof(EventOut);
static_assert(sizeof(EventOut) % 8 == 0, "EventOut is copied in 8-byte words");
// (LDS copies only) the event's new contact history, in nr, nh, nmass,
// ninertia, is to be appended to the owner's list for partner `ridged`
constexpr uint32_t EV_PUT_HIST = 1u << 15;

__device__ __forceinline__ void copy_event(EventOut* dst, const EventOut* src) {
    const uint64_t* s = reinterpret_cast<const uint64_t*>(src);
    uint64_t* d = reinterpret_cast<uint64_t*>(dst);
#pragma unroll
    for (int w = 0; w < (int)(sizeof(EventOut) / 8); ++w) d[w] = s[w];
}

// Where the records of pair (i, j), owner i by storage slot and partner j by
// identity, are in the owner's lists, old and new (-1: none).  The counts and
// the first two partners of all four lists are requested together.
struct PairRefs { int hist, bond, hist_new, bond_new; };
__device__ __forceinline__ PairRefs find_pair(const DS& S, int i, int j) {
    const int64_t SS = S.S;
    const int64_t h1 = (int64_t)min(1, S.HC - 1) * SS + i, b1 = (int64_t)min(1, S.BC - 1) * SS + i;
    const int n[4] = {S.hcnt_old[i], S.bcnt_old[i], S.hcnt_new[i], S.bcnt_new[i]};
    const int j0[4] = {S.hist_old[i].j, S.bond_old[i].j, S.hist_new[i].j, S.bond_new[i].j};
    const int j1[4] = {S.hist_old[h1].j, S.bond_old[b1].j, S.hist_new[h1].j, S.bond_new[b1].j};
    int q[4];
#pragma unroll
    for (int l = 0; l < 4; ++l) q[l] = (n[l] > 0 && j0[l] == j) ? 0 : (n[l] > 1 && j1[l] == j) ? 1 : -1;
    for (int p = 2; q[0] < 0 && p < n[0]; ++p) if (S.hist_old[(int64_t)p * SS + i].j == j) q[0] = p;
    for (int p = 2; q[1] < 0 && p < n[1]; ++p) if (S.bond_old[(int64_t)p * SS + i].j == j) q[1] = p;
    for (int p = 2; q[2] < 0 && p < n[2]; ++p) if (S.hist_new[(int64_t)p * SS + i].j == j) q[2] = p;
    for (int p = 2; q[3] < 0 && p < n[3]; ++p) if (S.bond_new[(int64_t)p * SS + i].j == j) q[3] = p;
    PairRefs r;
    r.hist = q[0]; r.bond = q[1]; r.hist_new = q[2]; r.bond_new = q[3];
    return r;
}
// The pair's old state (contact history, bond record) at those places.
__device__ __forceinline__ void pair_state_at(const DS& S, int i, const PairRefs& r, PairState& ps) {
    ps.deltat = 0.0; ps.thetarelc = 0.0; ps.fcn = 0.0; ps.fct = 0.0;
    ps.bond = 0; ps.has_bond_rec = false;
    ps.damage = ps.deltanb = ps.deltatb = ps.trb_ji = ps.trb_ij = 0.0;
    ps.rb = ps.hb = ps.lb = ps.sb = ps.ib = 0.0;
    if (r.hist >= 0) {
        const HistRec& hr = S.hist_old[(int64_t)r.hist * S.S + i];
        ps.deltat = hr.deltat; ps.thetarelc = hr.thetarelc; ps.fcn = hr.fcn; ps.fct = hr.fct;
    }
    if (r.bond >= 0) {
        const BondRec& b = S.bond_old[(int64_t)r.bond * S.S + i];
        ps.has_bond_rec = true; ps.bond = b.bond; ps.damage = b.damage;
        ps.deltanb = b.deltanb; ps.deltatb = b.deltatb; ps.trb_ji = b.trb_ji; ps.trb_ij = b.trb_ij;
        ps.rb = b.rb; ps.hb = b.hb; ps.lb = b.lb; ps.sb = b.sb; ps.ib = b.ib;
    }
}

// The touched floes that a reshape changed, one per lane: their walls, with
// the properties they have when their turn comes, and the properties the step
// leaves them with.  Wavefront w of nw takes every nw-th share of the queue.
template <bool MIXED>
__device__ __forceinline__ void reshaped_floes(const DS& S, const QueueView& qv, int w, int nw) {
    const int F = min(64, max(1, (qv.total + nw - 1) / nw));
    for (int t0 = w * F; t0 < qv.total; t0 += nw * F) {
        const int lane = (int)(threadIdx.x & 63), t = t0 + lane;
        if (lane >= F || t >= qv.total || *S.err) continue;
        const int k = queue_at(S, 4, qv, t);
        const GeoRec me = S.geo[k];
        const int hk = S.rhead[k], fs = S.cval[k];
        const uint8_t wf = S.wflag[k];
        const float nb = S.nb[k];
        const int m = me.member;
        if (m < 0 || hk < 0) continue;
        const int first = S.members[m].first;
        const Reshape* rec = S.shape + (int64_t)S.SEEDK * first;
        const DevParams& P = S.params[m];
        if (wf & WF_WALL) {
            Floe Fw = floe_at(S, k);
            floe_at_event(rec, hk, ((int64_t)(me.id - first) << 16) | WALL_SLOT, Fw);
            double hist[4] = {S.wbc[0 * S.S + fs], S.wbc[1 * S.S + fs], S.wbc[2 * S.S + fs], S.wbc[3 * S.S + fs]};
            WallOut W;
            walls<MIXED>(P, Fw, hist, W);
            if (W.flags & 1u) S.wout[k] = W;
            else wflag_clear(S, k, WF_WALL);
        }
        if (first_reshape(rec, hk) == INT64_MAX) continue;
        Floe Fn;
        floe_at_event(rec, hk, INT64_MAX, Fn);
        S.cur[0 * S.S + fs] = Fn.r; S.cur[1 * S.S + fs] = Fn.h; S.cur[2 * S.S + fs] = Fn.mass;
        S.cur[3 * S.S + fs] = Fn.inertia; S.cur[4 * S.S + fs] = Fn.hfa; S.cur[5 * S.S + fs] = Fn.hfw;
        S.dirty[fs] = 1;
        // drafts that outgrew the floe's bound: its lists may lack a
        // pair, so the step runs again with a build and more room
        const double reach = P.shelter ? near_reach(S.near_lim, Fn.hfa, Fn.hfw) : 0.0;
        if (1.01 * reach > (double)nb) {
            S.nbmin[fs] = (float)fmin(NEAR_ROOM * reach, 1e30);
            atomicOr(S.rebuild, BUILD_DUE);
            set_err(S, ERR_NEED_BUILD);
        }
    }
}

// The floes the repair touched re-gather every event of theirs, in the
// reference's order (inner pairs by ascending outer index, then their own
// candidates in distance order), each event with the properties its floes
// have at its place in the sequence (their reshape records).  The owner's new
// pair state and flags are written again from these results; a pair that is
// no longer a candidate when its outer floe's turn comes (the query radius
// shrank) keeps its old state.  Pairs that add nothing (apart, not bonded,
// too far to shelter) are passed over after their distance.  All the
// wavefront's events are evaluated together, 64 a pass (each lane finds its
// event's floe among the lanes), and after each pass every floe adds its own
// in order, so that a floe with many candidates does not hold one lane
// through all of them.  It is bound by the chain of loads of one event (queue
// -> list entry -> rows -> the owner's lists -> records), so each round of
// that chain requests all it can at once.  (One MI355X: 0.016 ms for 1,000
// sparse floes, 0.021 for a few thousand touched ones, 0.017 for 24 dense
// fields; 0.10 when every partner of a reshaped floe was gathered again.)
template <bool MIXED>
__global__ __launch_bounds__(FLOE_BLOCK, 2) void k_fixup(DS S) {
    using T = typename Prec<MIXED>::T;
    extern __shared__ unsigned char fix_lds[];
    EventOut* ev = reinterpret_cast<EventOut*>(fix_lds + (threadIdx.x >> 6) * FIX_LDS_PER_WAVE);
    // The touched floes (the fixup queue, filled by k_repair), a few per
    // wavefront: every wavefront of the grid (about one resident round)
    // takes F consecutive entries, F as small as the queue allows, so that
    // the floes' re-gathers run side by side rather than in a few long
    // wavefronts.
    const int lane = (int)(threadIdx.x & 63);
    const QueueView qv = queue_view(S, 4);
    const int waves = (int)(gridDim.x * blockDim.x) >> 6;
    const int wave = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    // every eighth wavefront leaves the reshaped floes with their final
    // properties instead, beside the events (behind them it was a fifth of a
    // small field's chain of loads)
    if ((wave & 7) == 7) {
        reshaped_floes<MIXED>(S, qv, wave >> 3, waves >> 3);
        return;
    }
    const int nw = waves - (waves >> 3), w = wave - (wave >> 3);
    const int F = min(64, max(1, (qv.total + nw - 1) / nw));
    for (int t0 = w * F; t0 < qv.total; t0 += nw * F) {     // (the same for all lanes)
        const int t = t0 + lane;
        bool act = lane < F && t < qv.total && !*S.err;
        const int k = act ? queue_at(S, 4, qv, t) : 0;
        int m = 0;
        if (act) {
            m = S.geo[k].member;
            act = m >= 0;
        }
        if (!__ballot(act)) continue;
        if (!act) m = 0;
        const int f = act ? S.geo[k].id : 0;
        const int fs = act ? (int)S.cval[k] : 0;
        const int ni = act ? S.icnt[k] : 0, no = act ? S.ocnt[k] : 0;
        const int hk = act ? S.rhead[k] : -1;
        const int cnt = ni + no;
        const int incl = wave_scan(cnt);
        const int start = incl - cnt, total = wave_last(incl);
        const int64_t SS = S.S;
        double acc[NACC];
        acc_init(acc);
        uint32_t over = 0;
        for (int c0 = 0; c0 < total; c0 += 64) {
            const int idx = c0 + lane;
            int own = 0;
#pragma unroll
            for (int step = 32; step > 0; step >>= 1)
                if (__shfl(start, own + step) <= idx) own += step;
            const int ko = __shfl(k, own), om = __shfl(m, own), of = __shfl(f, own);
            const int ofs = __shfl(fs, own), oni = __shfl(ni, own), ostart = __shfl(start, own);
            const int oh = __shfl(hk, own);
            bool adds = false;
            if (idx < total) {
                const DevParams& P = S.params[om];
                const Member Mb = S.members[om];
                const int rst = P.restart, coh = P.cohesion, shl = P.shelter;
                const double rtree = P.rtree, blim = P.bond_lim;
                const int tstep = Mb.tstep, first = Mb.first;
                const Reshape* rec = S.shape + (int64_t)S.SEEDK * first;
                const int local = idx - ostart;
                const bool inner = local < oni;
                const int64_t e = inner ? S.ik[(int64_t)local * SS + ko] : S.oj[(int64_t)(local - oni) * SS + ko];
                const int pid = ent_id(e), qp = ent_pos(e);
                // outer floe a, inner floe b; their rows, requested at once
                const int ka = inner ? qp : ko, kb = inner ? ko : qp;
                const int ia = inner ? pid : of, ib = inner ? of : pid;
                const int hq = S.rhead[qp];
                const int sq = S.cval[qp];
                Floe Fa = floe_at(S, ka), Fb = floe_at(S, kb);
                const double2 wa = wind_at(S, ka);
                const int sa = inner ? sq : ofs;
                // the owner's lists, old and new
                const PairRefs pr = find_pair(S, sa, ib);
                const double dx = Fa.x - Fb.x, dy = Fa.y - Fb.y;
                const double d = sqrt(dx * dx + dy * dy);
                const double dn = Fa.r + Fb.r - d;
                // the properties at the event, the outer floe's radius at the
                // top of its iteration
                bool removed = false;
                EventOut o;
                o.ridged = -1;
                // the event's own record: the floe it reshapes, and to what
                auto own_record = [&](const Reshape& w, int side) {
                    if (w.kf != ka || w.kj != kb) return;
                    o.ridged = side;
                    o.nr = w.r; o.nh = w.h; o.nmass = w.mass;
                    o.ninertia = w.inertia; o.nhfa = w.hfa; o.nhfw = w.hfw;
                };
                if ((oh >= 0) | (hq >= 0)) {
                    const int al = ia - first;
                    // last record before the event: of a, of b; of a before its
                    // iteration
                    int wa_ = -1, wb_ = -1, wq_ = -1;
                    int64_t ka_ = -1, kb_ = -1, kq_ = -1;
                    auto before = [&](const Reshape& w) {
                        const int rf = (int)(w.key >> 16);
                        if (rf != al) return rf < al;
                        const int ws = (int)(w.key & 0xFFFF);
                        if (!inner) return ws < local - oni;
                        // the same outer floe's event with another partner, or its
                        // walls: by distance, as its list is
                        if (ws == WALL_SLOT || w.kj == kb) return false;
                        const GeoRec wf = S.geo[w.kf], wj = S.geo[w.kj];
                        const double ex = wf.x - wj.x, ey = wf.y - wj.y;
                        const double de = sqrt(ex * ex + ey * ey);
                        return de < d || (de == d && wj.id < ib);
                    };
                    for (int p = inner ? hq : oh; p >= 0; p = rec[p].next) {
                        const Reshape& w = rec[p];
                        if (!w.live) continue;
                        own_record(w, 0);
                        if ((int)(w.key >> 16) < al && w.key > kq_) { kq_ = w.key; wq_ = p; }
                        if (w.key > ka_ && before(w)) { ka_ = w.key; wa_ = p; }
                    }
                    for (int p = inner ? oh : hq; p >= 0; p = rec[p].next) {
                        const Reshape& w = rec[p];
                        if (!w.live) continue;
                        own_record(w, 1);
                        if (w.key > kb_ && before(w)) { kb_ = w.key; wb_ = p; }
                    }
                    const double rq = wq_ >= 0 ? rec[wq_].r : Fa.r;
                    removed = !(d <= rq + rtree);
                    if (wa_ >= 0) take_shape(rec[wa_], Fa);
                    if (wb_ >= 0) take_shape(rec[wb_], Fb);
                }
                // (the start-of-step overlap is the largest the pair can have)
                const T lim = sizeof(T) == 4 ? T(20) : T(40), dnt = T(dn);
                const bool far = dnt < T(0) && T((double)0.18f) * -dnt >= lim * T(inner ? Fb.hfa : Fa.hfa) &&
                                 T((double)0.18f) * -dnt >= lim * T(inner ? Fb.hfw : Fa.hfw);
                const bool bond_step = (tstep == 1) & (rst != 1) & (coh != 0);
                adds = dn > 0 || pr.bond >= 0 || (bond_step && dn >= -blim) || (shl && !far) || removed ||
                       (S.record_forces && !inner && oh >= 0);
                if (adds) {
                    PairState ps;
                    pair_state_at(S, sa, pr, ps);
                    if (removed) {
                        // no longer a candidate: the pair keeps its old state
                        o.flags = EV_REMOVED;
                        o.sc = o.sbd = o.sri = 0.0;
                    } else {
                        pair_event<MIXED>(P, tstep, ia - first, ib - first, Fa, Fb, wa.x, wa.y, P.uw, P.vw,
                                          ps, o, inner ? 2 : 1);
                    }
                    if (!inner) {
                        const int64_t at = (int64_t)(local - oni) * SS + ko;
                        S.evf[at] = (S.evf[at] & 0xffff0000u) | o.flags | (S.record_forces ? EV_SRI : 0u);
                        if (S.record_forces) { S.ssc[at] = o.sc; S.ssb[at] = o.sbd; S.od[at] = o.sri; }
                        // the pair's new records, each in its place; a history
                        // with no place yet is the owner's lane's to append
                        if (pr.bond_new >= 0) {
                            if (ps.has_bond_rec) S.bond_new[(int64_t)pr.bond_new * SS + ofs] = bond_from(ps, pid);
                            else S.bond_new[(int64_t)pr.bond_new * SS + ofs].j = -1;
                        } else if (ps.has_bond_rec) {
                            const int p = atomicAdd(&S.bcnt_new[ofs], 1);
                            if (p < S.BC) S.bond_new[(int64_t)p * SS + ofs] = bond_from(ps, pid);
                            else over |= ERR_BOND_CAP;
                            sup_keep(S, ko, qp);
                        }
                        const bool hist = ps.deltat != 0.0 || ps.thetarelc != 0.0 || ps.fcn != 0.0 || ps.fct != 0.0;
                        HistRec hr;
                        hr.j = hist ? pid : -1; hr.pad_ = 0;
                        hr.deltat = ps.deltat; hr.thetarelc = ps.thetarelc; hr.fcn = ps.fcn; hr.fct = ps.fct;
                        if (pr.hist_new >= 0) {
                            S.hist_new[(int64_t)pr.hist_new * SS + ofs] = hr;
                        } else if (hist) {
                            o.nr = hr.deltat; o.nh = hr.thetarelc; o.nmass = hr.fcn; o.ninertia = hr.fct;
                            o.ridged = pid;
                            sup_keep(S, ko, qp);
                            o.flags |= EV_PUT_HIST;
                        }
                    }
                    copy_event(&ev[lane], &o);
                }
            }
            const uint64_t am = __ballot(adds);
            wave_lds_sync();
            // every floe adds this pass's events of its own, in order
            if (act) {
                const int lo = max(start, c0) - c0, hi = min(start + cnt, c0 + 64) - c0;
                uint64_t mine = hi > lo ? am & (~0ull >> (64 - hi)) & (~0ull << lo) : 0ull;
                for (; mine; mine &= mine - 1) {
                    const int i2 = __ffsll((long long)mine) - 1;
                    const EventOut& o = ev[i2];
                    if (c0 + i2 - start < ni) {
                        apply_j(acc, o);
                    } else {
                        apply_i(acc, o);
                        if (o.flags & EV_PUT_HIST) {
                            const int n = S.hcnt_new[fs];
                            if (n < S.HC) {
                                HistRec hr;
                                hr.j = o.ridged; hr.pad_ = 0;
                                hr.deltat = o.nr; hr.thetarelc = o.nh; hr.fcn = o.nmass; hr.fct = o.ninertia;
                                S.hist_new[(int64_t)n * SS + fs] = hr;
                                S.hcnt_new[fs] = n + 1;
                            } else {
                                over |= ERR_HIST_CAP;
                            }
                        }
                    }
                }
            }
            wave_lds_sync();
        }
        if (act) {
#pragma unroll
            for (int a = 0; a < NACC; ++a) S.acc[a * SS + k] = acc[a];
            S.cls[k] = CLS_CONTACT | CLS_BOND;
        }
        if (over) set_err(S, over);
    }
}

// ---------------------------------------------------------------------
// 5b. stress diagnostics (stepper.f90:238-271), only when forces are
//     recorded: for every candidate pair (j,i), both floes take
//     sig -= S * (direction terms) * r(i) with S = |(fcn,fct)| + |(fbn,fbt)|,
//     the pair's current or last contact forces and current bond forces, in
//     the reference's per-floe order.
// ---------------------------------------------------------------------
__device__ __forceinline__ void stress_terms(double Sv, double c, double sn, double ri, double* a) {
    a[A_SXX] = a[A_SXX] - Sv * c * ri * c;
    a[A_SYY] = a[A_SYY] - Sv * sn * ri * sn;
    a[A_SXY] = a[A_SXY] - Sv * sn * ri * c;
    a[A_SYX] = a[A_SYX] - Sv * c * ri * sn;
}

__global__ __launch_bounds__(FLOE_BLOCK) void k_stress(DS S) {
    const int k = xcd_block() * blockDim.x + threadIdx.x;
    if (k >= S.N || *S.err) return;
    const GeoRec me = S.geo[k];
    const int m = me.member;
    if (m < 0) return;
    const int f = me.id;
    const int64_t SS = S.S;
    double a[NACC];
    a[A_SXX] = a[A_SYY] = a[A_SXY] = a[A_SYX] = 0.0;
    // pairs (i, f), f inner, ascending i
    const int ni = S.icnt[k];
    for (int q = 0; q < ni; ++q) {
        const int64_t e = S.ik[q * SS + k];
        const int qi = ent_pos(e);
        const int s = slot_of(S, qi, f);
        if (s < 0) continue;
        const int64_t at = (int64_t)s * SS + qi;
        const uint32_t fl = S.evf[at];
        if (fl & EV_REMOVED) continue;
        const GeoRec gi = S.geo[qi];
        const double sc = S.ssc[at], sb = S.ssb[at];
        const double ri = (fl & EV_SRI) ? S.od[at] : gi.r;
        const double dx = gi.x - me.x, dy = gi.y - me.y;
        const double dist = sqrt(dx * dx + dy * dy);
        const double c = (me.x - gi.x) / dist, sn = (me.y - gi.y) / dist;
        stress_terms(sc + sb, c, sn, ri, a);
    }
    // pairs (f, j), f outer, distance order
    const int no = S.ocnt[k];
    for (int s = 0; s < no; ++s) {
        const int64_t e = S.oj[s * SS + k];
        const int qj = ent_pos(e);
        const int64_t at = (int64_t)s * SS + k;
        const uint32_t fl = S.evf[at];
        if (fl & EV_REMOVED) continue;
        const double sc = S.ssc[at], sb = S.ssb[at];
        const double ri = (fl & EV_SRI) ? S.od[at] : me.r;
        const GeoRec gj = S.geo[qj];
        const double dx = me.x - gj.x, dy = me.y - gj.y;
        const double dist = sqrt(dx * dx + dy * dy);
        const double c = (gj.x - me.x) / dist, sn = (gj.y - me.y) / dist;
        stress_terms(sc + sb, c, sn, ri, a);
    }
    S.acc[A_SXX * SS + k] = a[A_SXX];
    S.acc[A_SYY * SS + k] = a[A_SYY];
    S.acc[A_SXY * SS + k] = a[A_SXY];
    S.acc[A_SYX * SS + k] = a[A_SYX];
}

// ---------------------------------------------------------------------
// 6. final properties, forcing + coriolis, totals, integration
//    (stepper.f90:295-343, integration.f90:1-38)
// ---------------------------------------------------------------------
// (REC: forces are recorded; the other instance carries no code for the
// recorded columns and stress rows.  The mixed-precision instance without
// them fits 5 wavefronts per SIMD in 96 VGPRs, one value kept in scratch
// from the first loads to the writes: its chains of dependent loads, the
// gridded wind's among them, gain more from the extra wavefront)
template <bool MIXED, bool REC>
__global__ __launch_bounds__(FLOE_BLOCK, (MIXED && !REC) ? 5 : 4) void k_final(DS S) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    // the next step's queue counters
    if (k < NQUEUE * XCD_COUNT && !*S.err) S.qn_next[k * QN_STRIDE] = 0;
    if (k >= S.N) return;
    // the position's rows are requested at once, before anything is tested
    const GeoRec me = S.geo[k];
    const int f = S.cval[k];        // storage slot
    Floe F = floe_at(S, k);
    const uint8_t wf = S.wflag[k], cl = S.cls[k], bg = S.bgat[k];
    const int ni = S.icnt[k], no = S.ocnt[k];
    if (*S.err) return;
    // every earlier kernel of the step has finished: the step is complete
    if (k == 0) *S.steps_done += 1;
    const int m = me.member;
    if (m < 0) {
        // (only the member is read of such a row)
        S.geo_new[k].member = m;
        return;
    }
    const DevParams& P = S.params[m];
    const int64_t SS = S.S;
    const uint8_t dflags = S.dirty[f];
    const bool dirty = dflags != 0;
    if (dirty) {
        F.r = S.cur[0 * SS + f]; F.h = S.cur[1 * SS + f]; F.mass = S.cur[2 * SS + f];
        F.inertia = S.cur[3 * SS + f]; F.hfa = S.cur[4 * SS + f]; F.hfw = S.cur[5 * SS + f];
    }
    WallOut W;
    if (wf & WF_WALL) {
        W = S.wout[k];
    } else {
        // no wall touched: reset_boundary(i, 0) cleared every wall history
        W.fx_bc = W.fy_bc = W.m_bc = W.ta_bc = W.p_bc = 0.0;
        W.deltat_bc1 = W.deltat_bc2 = W.theta_bc1 = W.theta_bc2 = 0.0;
        W.sxx_bc = W.syy_bc = W.sxy_bc = W.syx_bc = 0.0;
    }
    {
        // wall histories: rows that are all +0.0 and stay so are not rewritten
        const bool had = S.wnz[f] != 0;
        const bool now = (__double_as_longlong(W.deltat_bc1) | __double_as_longlong(W.deltat_bc2) |
                          __double_as_longlong(W.theta_bc1) | __double_as_longlong(W.theta_bc2)) != 0;
        if (had || now) {
            S.wbc[0 * SS + f] = W.deltat_bc1; S.wbc[1 * SS + f] = W.deltat_bc2;
            S.wbc[2 * SS + f] = W.theta_bc1; S.wbc[3 * SS + f] = W.theta_bc2;
        }
        if (had != now) S.wnz[f] = now;
    }
    double a[NACC];
#pragma unroll
    for (int c = 0; c < NACC; ++c) {
        const bool bond_row = c == A_FBX || c == A_FBY || c == A_MB || c == A_TAB || c == A_PB;
        const bool shel_row = c == A_SHA || c == A_SHW;
        const bool stress_row = c >= A_SXX;
        const bool valid = stress_row ? REC
                         : shel_row || (bond_row ? (cl & CLS_BOND) : (cl & CLS_CONTACT));
        a[c] = valid ? S.acc[c * SS + k] : 0.0;
    }
    // bond terms: rows the fix-up wrote (CLS_BOND), else gathered here
    if (!(cl & CLS_BOND) && bg) gather_bonds(S, k, ni, no, a);
    // shelter minima (reset_shelter + thread reduction); with shelter off
    // the reference's minima stay at their zero initial value
    double sha = P.shelter ? a[A_SHA] : 0.0;
    double shw = P.shelter ? a[A_SHW] : 0.0;
    const double2 w = wind_at(S, k);
    Forcing Fo;
    forcing<MIXED>(P, F, w.x, w.y, P.uw, P.vw, sha, shw, Fo);
    double tfx = a[A_FCX] + a[A_FBX] + Fo.fax + Fo.fwx + Fo.fcorx + W.fx_bc;
    double tfy = a[A_FCY] + a[A_FBY] + Fo.fay + Fo.fwy + Fo.fcory + W.fy_bc;
    double mt = a[A_MC] + a[A_MB] + Fo.ma + Fo.mw + W.m_bc;
    double u = F.u + (tfx / F.mass) * P.dt;
    double v = F.v + (tfy / F.mass) * P.dt;
    double om = F.omega + (mt / F.inertia) * P.dt;
    FloeRec out;
    out.x = F.x + u * P.dt;
    out.y = F.y + v * P.dt;
    out.u = u; out.v = v; out.omega = om;
    out.r = F.r; out.h = F.h; out.mass = F.mass; out.inertia = F.inertia; out.hfa = F.hfa; out.hfw = F.hfw;
    out.theta = S.kin[k].theta + om * P.dt;
    {
        // next step builds the supersets anew if this floe has moved more
        // than 0.45 skin since the last build (a pair not in a superset was
        // more than its query radius + skin apart then, so it stays outside
        // the query radius while both floes stay within half the skin);
        // beyond 0.3 skin the next step with the build kernels builds early
        const double2 p0 = S.x0[k];
        const double ex = out.x - p0.x, ey = out.y - p0.y, e2 = ex * ex + ey * ey;
        const double lim = 0.45 * P.skin, soon = 0.3 * P.skin;
        // one atomic per wavefront (every such floe writing the one word
        // would queue the writes behind each other)
        const uint64_t md = __ballot(e2 > lim * lim), ms = __ballot(e2 > soon * soon);
        const int bits = (md ? BUILD_DUE : 0) | (ms ? BUILD_SOON : 0);
        const int leader = __ffsll((long long)(md | ms)) - 1;
        if (bits && (int)(threadIdx.x & 63) == leader) atomicOr(S.rebuild, bits);
    }
    if (REC) {
        double tp = (a[A_TAC] != 0.0 ? a[A_PC] / a[A_TAC] : 0.0)
                  + (a[A_TAB] != 0.0 ? a[A_PB] / a[A_TAB] : 0.0)
                  + (W.ta_bc != 0.0 ? W.p_bc / W.ta_bc : 0.0);
        // total stress: pairs + last wall + drag (forcing.f90 sig*_aw)
        const double sxx_aw = (Fo.fax + Fo.fwx) * F.r, syy_aw = (Fo.fay + Fo.fwy) * F.r;
        const double tsxx = a[A_SXX] + W.sxx_bc + sxx_aw;
        const double tsyy = a[A_SYY] + W.syy_bc + syy_aw;
        const double tsxy = a[A_SXY] + W.sxy_bc + 0.0;
        const double tsyx = a[A_SYX] + W.syx_bc + 0.0;
        double cols[33] = {tfx, tfy, mt, a[A_FCX], a[A_FCY], a[A_MC], a[A_FBX], a[A_FBY], a[A_MB],
                           Fo.fax, Fo.fay, Fo.ma, Fo.fwx, Fo.fwy, Fo.mw, Fo.fcorx, Fo.fcory,
                           W.fx_bc, W.fy_bc, W.m_bc, sha, shw, tp, tsxx, tsyy, tsxy, tsyx,
                           a[A_TAC], a[A_PC], a[A_TAB], a[A_PB], W.ta_bc, W.p_bc};
        for (int c = 0; c < 33; ++c) S.fout[c * SS + f] = cols[c];
    }
    // flags set by the repair are cleared (most floes have none: no write)
    if (dflags) S.dirty[f] = 0;
    // the new state, in the current order (the next step's copies unless it
    // rebuilds them from rec): position, kinematics, the wind at the new
    // position
    {
        GeoRec g;
        g.x = out.x; g.y = out.y; g.r = out.r; g.id = me.id; g.member = m;
        S.geo_new[k] = g;
        KinRec q;
        q.u = out.u; q.v = out.v; q.omega = out.omega; q.h = out.h; q.mass = out.mass;
        q.inertia = out.inertia; q.theta = out.theta;
        S.kin[k] = q;
        // the sheltering copy changes only with a reshape or a gridded wind
        // (the uniform wind stands until the host changes it, which
        // refreshes the copies)
        if (dirty || P.wind_grid >= 0) {
            double ua = P.ua, va = P.va;
            // at the start of the next step: model time tcur dt
            if (P.wind_grid >= 0)
                sample_wind(S.wgrids[P.wind_grid], S.wpool, out.x, out.y, out.r,
                            (double)S.tcur[m] * P.dt, ua, va);
            ShelRec h;
            h.hfa = out.hfa; h.hfw = out.hfw; h.wx = ua; h.wy = va;
            S.shel[k] = h;
        }
    }
    if (f == S.members[m].first) {   // once per member
        S.rebuild[2] = 1;                // the copies hold the new state
        S.members[m].tstep += 1;
        if (!member_live(S.members[m])) S.rebuild[1] = 1;   // its floes leave the next step
    }
}

// Whether the row at position k of the last step's order is a floe that is
// still there.  Positions, and with them the lists and the reshape records,
// stand until the next build while members leave and others take their slots
// and storage: rows of a member that left have no member at their storage slot
// any more, and floes added since the step have no position (k_admit).  Lists
// are walked for such rows only: a new member in an old one's slot has another
// first floe, and the old one's record indices lead anywhere from there.
__device__ __forceinline__ bool still_there(const DS& S, const GeoRec& g, int k) {
    if (g.member < 0) return false;
    const int f = S.sid_of[g.id];
    return S.member_of[f] == g.member && S.pos_of[f] == k;
}

// The candidate pairs of the last step (the reference's kNearest within
// r(i) + rtree) of a wavefront's floes, a lane each (act: the lane has one, at
// position k, still_there): those of their supersets within the query radius, by
// the positions the step started from (the other of the two position buffers)
// and the floe's radius at the top of its iteration.  The supersets' entries
// are tested together, PAIR_AHEAD rounds of 64 requested at once, each lane
// finding its entry's owner among the lanes: a lane per floe reading its own
// superset took a line per lane and entry (the totals' call on the host: 1.45 M
// power-law floes 1.30 -> 0.66 ms, 320,000 0.43 -> 0.22, 1,000 0.098 -> 0.075;
// 1.4 M on [500, 2000] m 0.87 -> 0.61, most of it their bond records).
// fn(listed, identity, partner's identity) is called by every lane, once a
// round.
constexpr int PAIR_AHEAD = 4;
template <typename F>
__device__ __forceinline__ void each_candidate(const DS& S, int k, const GeoRec& me, bool act, F&& fn) {
    const int lane = (int)(threadIdx.x & 63);
    double rq = 0.0;
    int n = 0;
    int64_t at0 = 0;
    if (act) {
        const int first = S.members[me.member].first;
        Floe Fq;
        Fq.r = me.r;
        floe_at_event(S.shape + (int64_t)S.SEEDK * first, S.rhead[k], (int64_t)(me.id - first) << 16, Fq);
        rq = Fq.r + S.params[me.member].rtree;
        n = S.scnt[k];
        at0 = S.soff[k];
    }
    const int incl = wave_scan(n), start = incl - n, total = wave_last(incl);
    at0 -= start;
    for (int c0 = 0; c0 < total; c0 += 64 * PAIR_AHEAD) {
        int own[PAIR_AHEAD];
        int64_t e[PAIR_AHEAD];
        GeoRec o[PAIR_AHEAD];
#pragma unroll
        for (int u = 0; u < PAIR_AHEAD; ++u) {
            const int idx = min(c0 + 64 * u + lane, total - 1);      // (the last entry stands in past the end)
            own[u] = 0;
#pragma unroll
            for (int step = 32; step > 0; step >>= 1)
                if (__shfl(start, own[u] + step) <= idx) own[u] += step;
            e[u] = S.sup[__shfl(at0, own[u]) + idx];
        }
#pragma unroll
        for (int u = 0; u < PAIR_AHEAD; ++u) o[u] = S.geo_new[ent_pos(e[u])];
#pragma unroll
        for (int u = 0; u < PAIR_AHEAD; ++u) {
            const double dx = __shfl(me.x, own[u]) - o[u].x, dy = __shfl(me.y, own[u]) - o[u].y;
            const double r = __shfl(rq, own[u]), d2 = dx * dx + dy * dy;
            const int id = __shfl(me.id, own[u]);
            // (k_cand's test: far beyond the radius no square root is taken)
            const bool in = c0 + 64 * u + lane < total && o[u].id > id && d2 <= r * r * (1.0 + 1e-12);
            fn(in && sqrt(d2) <= r, id, o[u].id);
        }
    }
}

// totals of the last step: candidates, contacts (evf flags) and current bonds,
// of the members that take steps; diagnostics only.  A wavefront takes `floes`
// positions' lists (of the step's np positions; 0: there are no lists to read)
// and as many storage slots' bonds, a lane each.
__global__ __launch_bounds__(64) void k_totals(DS S, int np, int floes, int64_t* out) {
    const int lane = (int)threadIdx.x;
    const int k = blockIdx.x * floes + lane;
    const bool mine = lane < floes;
    int64_t c = 0, ct = 0, bd = 0;
    const GeoRec me = mine && k < np ? S.geo_new[k] : GeoRec{0.0, 0.0, 0.0, 0, -1};
    const bool act = still_there(S, me, k);
    each_candidate(S, k, me, act, [&](bool listed, int, int) { c += listed; });
    if (act) {
        const int no = S.ocnt[k];
        for (int s = 0; s < no; ++s) {
            uint32_t fl = S.evf[(int64_t)s * S.S + k];
            if (fl & EV_REMOVED) continue;
            if (fl & EV_CONTACT) ++ct;
        }
    }
    if (mine && k < S.N && S.member_of[k] >= 0 && S.pos_of[k] >= 0 && S.geo[S.pos_of[k]].member == S.member_of[k]) {
        int nb = S.bcnt_old[k];
        for (int q = 0; q < nb; ++q) {
            const BondRec& b = S.bond_old[(int64_t)q * S.S + k];
            if (b.j >= 0 && b.bond == 1) ++bd;
        }
    }
    // wavefront reduction, one atomic per wave
    for (int off = 32; off > 0; off >>= 1) {
        c += __shfl_down(c, off);
        ct += __shfl_down(ct, off);
        bd += __shfl_down(bd, off);
    }
    if (lane == 0) {
        if (c) atomicAdd((unsigned long long*)&out[0], (unsigned long long)c);
        if (ct) atomicAdd((unsigned long long*)&out[1], (unsigned long long)ct);
        if (bd) atomicAdd((unsigned long long*)&out[2], (unsigned long long)bd);
    }
}

// Storage slot's position in the current order, or -1 where the ordered
// copies do not hold the floe's state: rec does then.
__device__ __forceinline__ int newer_pos(const DS& S, int m, int slot) {
    if (!S.rebuild[2]) return -1;
    const int k = S.pos_of[slot];
    if ((uint32_t)k >= (uint32_t)S.N || S.cval[k] != (uint32_t)slot || S.geo[k].member != m) return -1;
    return k;
}

// Rows of member m's floes [begin, begin + count) in the caller's order, one
// thread per floe, to `out` ([rows][count], pinned host memory): the floe
// state from the ordered copies where they are newer than rec (no spill of
// every member's records first), or the recorded columns, or the wall
// histories.  The stores go over the bus coalesced, a row of 64 floes each,
// and the host copies plain rows: 512 reads of 2,700 floes 51 -> 30 ms, one
// of 262,144 floes 6.1 -> 1.0 ms.
template <int W>
__global__ __launch_bounds__(64) void k_read(DS S, int m, int begin, int count, double* out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const int f = S.sid_of[S.members[m].first + begin + t];
    double* o = out + t;
    if (W == READ_FLOES) {
        FloeRec r;
        const int k = newer_pos(S, m, f);
        if (k >= 0) {
            const GeoRec g = S.geo[k];
            const KinRec q = S.kin[k];
            const ShelRec h = S.shel[k];
            r.x = g.x; r.y = g.y; r.u = q.u; r.v = q.v; r.omega = q.omega;
            r.r = g.r; r.h = q.h; r.mass = q.mass; r.inertia = q.inertia; r.hfa = h.hfa; r.hfw = h.hfw;
            r.theta = q.theta;
        } else {
            r = S.rec[f];
        }
        const double v[12] = {r.x, r.y, r.u, r.v, r.theta, r.omega, r.r, r.h, r.mass, r.inertia, r.hfa, r.hfw};
#pragma unroll
        for (int c = 0; c < 12; ++c) o[(int64_t)c * count] = v[c];
    } else {
        const double* src = W == READ_FORCES ? S.fout : S.wbc;
        constexpr int ROWS = W == READ_FORCES ? NFORCE : 4;
#pragma unroll
        for (int c = 0; c < ROWS; ++c) o[(int64_t)c * count] = src[c * S.S + f];
    }
}

// Member m's pairs of the last step, in the caller's indices, in no order:
// counted in *S.npairs, those from number `skip` on, up to `cap`, written to
// `out`.  Candidates come from the supersets (a wavefront takes `floes` of the
// step's positions [b, e), which may be more than the floe slots in use now),
// contacts from the step's lists and bonds from the owners' records (a thread
// for each of the member's floes [b, e)).
template <int K>
__global__ __launch_bounds__(64) void k_pairs(DS S, int m, int b, int e, int floes, int skip,
                                              typename PairKind<K>::Out* out, int cap) {
    const int lane = (int)threadIdx.x;
    const int k = b + (int)blockIdx.x * floes + lane;
    const bool mine = lane < floes && k < e;
    const Member mb = S.members[m];
    if constexpr (K == PAIRS_CANDIDATE) {
        GeoRec me = mine ? S.geo_new[k] : GeoRec{0.0, 0.0, 0.0, 0, -1};
        const bool act = me.member == m && still_there(S, me, k);
        each_candidate(S, k, me, act, [&](bool listed, int i, int j) {
            const uint64_t mask = __ballot(listed);
            if (!mask) return;
            int at = 0;
            if (lane == 0) at = atomicAdd(S.npairs, (int)__popcll(mask)) - skip;
            at = __builtin_amdgcn_readlane(at, 0) + (int)__popcll(lane ? mask & (~0ull >> (64 - lane)) : 0ull);
            if (listed && at >= 0 && at < cap) { out[at].i = i - mb.first; out[at].j = j - mb.first; }
        });
        return;
    }
    if (!mine) return;
    const int f = mb.first + k, i = S.gid_of[f] - mb.first;
    if (K == PAIRS_CONTACT) {
        const int q = S.pos_of[f];
        if (q < 0) return;                                  // (the member's first step is to come)
        const int no = min(S.ocnt[q], S.CO);
        for (int s = 0; s < no; ++s) {
            const int64_t at0 = (int64_t)s * S.S + q;
            const uint32_t fl = S.evf[at0];
            if ((fl & EV_REMOVED) || !(fl & EV_CONTACT)) continue;
            const int at = atomicAdd(S.npairs, 1) - skip;
            if (at >= 0 && at < cap) { out[at].i = i; out[at].j = ent_id(S.oj[at0]) - mb.first; }
        }
    }
    if constexpr (K == PAIRS_BOND) {
        const int nb = min(S.bcnt_old[f], S.BC);
        for (int q = 0; q < nb; ++q) {
            const BondRec b = S.bond_old[(int64_t)q * S.S + f];
            if (b.j < 0 || b.bond != 1) continue;
            const int at = atomicAdd(S.npairs, 1) - skip;
            if (at < 0 || at >= cap) continue;
            BondOut p;
            p.i = i; p.j = b.j - mb.first;
            const double v[11] = {(double)b.bond, b.damage, b.deltanb, b.deltatb, b.trb_ji, b.trb_ij, b.rb, b.hb,
                                  b.lb, b.sb, b.ib};
#pragma unroll
            for (int c = 0; c < 11; ++c) p.v[c] = v[c];
            out[at] = p;
        }
    }
}

// Floes [b, b + count) in storage order of a new member m from storage slot
// `first` on: their records and their indices in the caller's arrays, from
// pinned host memory, and empty pair and wall state (one launch for eleven
// clears and four copies, each of which waited: adding 5,000 floes 0.70 ->
// 0.15 ms).
__global__ __launch_bounds__(64) void k_admit(DS S, int m, int first, int b, int count, const FloeRec* recs,
                                              const int32_t* order) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const int f = first + b + t, id = first + order[t];
    S.rec[f] = recs[t];
    S.gid_of[f] = id;
    S.sid_of[id] = f;
    S.pos_of[f] = -1;              // (none before the next build)
    S.member_of[f] = m;
#pragma unroll
    for (int k = 0; k < 4; ++k) S.wbc[k * S.S + f] = 0.0;
    S.hcnt_old[f] = S.hcnt_new[f] = S.bcnt_old[f] = S.bcnt_new[f] = 0;
    S.nbmin[f] = 0.0f;
    S.dirty[f] = 0;
    S.wnz[f] = 0;                  // (the wall history rows are all +0.0)
    if (b + t == 0)                // (those of the slot's last member)
        for (int k = 0; k < 4; ++k) S.stats[4 * m + k] = 0;
}

// The pair count to the host, and back to 0 for the next list.
__global__ void k_take_count(int32_t* n, int32_t* out) {
    *out = *n;
    *n = 0;
}

// The step status and the members' first `words` words to the host.
__global__ void k_status(DS S, int words, HostStatus* out) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        out->steps_done = *S.steps_done;
        out->err = *S.err;
        out->due = S.rebuild[0] | S.rebuild[1];
        out->builds = S.rebuild[3];
    }
    const int32_t* src = reinterpret_cast<const int32_t*>(S.members);
    int32_t* dst = reinterpret_cast<int32_t*>(out->members());
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x) dst[i] = src[i];
}

// explicit instantiations used by the host launcher
template __global__ void k_read<READ_FLOES>(DS, int, int, int, double*);
template __global__ void k_read<READ_FORCES>(DS, int, int, int, double*);
template __global__ void k_read<READ_WALLS>(DS, int, int, int, double*);
template __global__ void k_pairs<PAIRS_CANDIDATE>(DS, int, int, int, int, int, PairOut*, int);
template __global__ void k_pairs<PAIRS_CONTACT>(DS, int, int, int, int, int, PairOut*, int);
template __global__ void k_pairs<PAIRS_BOND>(DS, int, int, int, int, int, BondOut*, int);
template __global__ void k_sup<false>(DS);
template __global__ void k_sup<true>(DS);
template __global__ void k_sup_dense<false>(DS);
template __global__ void k_sup_dense<true>(DS);
template __global__ void k_cand<false>(DS, int, int, int);
template __global__ void k_cand<true>(DS, int, int, int);
template __global__ void k_events<false>(DS, int, int, int);
template __global__ void k_events<true>(DS, int, int, int);
template __global__ void k_contact<false>(DS);
template __global__ void k_contact<true>(DS);
template __global__ void k_bond<false>(DS);
template __global__ void k_bond<true>(DS);
template __global__ void k_walls<false>(DS);
template __global__ void k_walls<true>(DS);
template __global__ void k_repair<false>(DS, int, int);
template __global__ void k_repair<true>(DS, int, int);
template __global__ void k_fixup<false>(DS);
template __global__ void k_fixup<true>(DS);
template __global__ void k_final<false, false>(DS);
template __global__ void k_final<true, false>(DS);
template __global__ void k_final<false, true>(DS);
template __global__ void k_final<true, true>(DS);

}  // namespace godar
