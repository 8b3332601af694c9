// The fused simulation step: one stencil walk per step.
//
// SimulationLoop.h:280-300 runs integrate -> NL -> reactions -> NL -> forces, and the forces of the
// post-reaction state drive the next integration.  Here the state between two walks is x'(t), the
// positions after step t's integration and before its reactions, and a step is
//   (bonded terms)  on x'(t); topology particles are never moved by reactions
//   k_brick_step    one LDS-staged stencil walk over x'(t): the pair forces G (fixed point), the
//                   reaction candidates of step t, and, optimistically, step t+1's Euler-Maruyama
//                   move with G, re-binned into the next buffer; it also clears the cell counters
//                   of the buffer after that
//   k_resolve_step  the replicas' step counters; step t's reactions on x'(t) (in place), listing every
//                   record they change (k_step_book does the counters when there are no reactions)
//   k_fix_sites     per changed record: withdraws moved copies from the next buffer (of killed and
//                   retyped records, and of every surviving neighbour whose pair force with it
//                   changed) and lists the records to move again (those neighbours, inserted and
//                   retyped records)
//   k_fix_advance   forms each listed record's pair force afresh on the post-reaction state and
//                   moves it again
// A kernel boundary costs about 4.5 us whatever the kernel does, which is most of a small system's step:
// hence the counters cleared two buffers ahead (four sets of counters take turns), the bookkeeping in the
// resolve and the withdrawals in k_fix_sites.
// A reaction changes the pair set only around the records it changes; every other record's G is
// already the force of the post-reaction state, bit for bit (an integer sum of per-pair integers,
// pair_fixed, over the same pairs), so its optimistic move stands, as the reference's order needs.
// The first walk of a run (k_brick_step with prologue set) forms the forces of the current state
// and makes step 1's move; the last step of a run (and of a replica's budget) copies instead of
// moving, so that a run ends on the post-reaction state of its last step.
#pragma once

#include "rdy_bricks.hip"

namespace rdy {

// Moves a record one Euler-Maruyama step (CPUEulerBDIntegrator.cpp:63-73) with the pair force
// (fx, fy, fz, 2^-32 fixed point) plus its bonded force, Philox counter `step`, or copies it
// (integ false), and re-bins it into nxt.  Returns the new slot (UINT32_MAX on a full pool).
__device__ __forceinline__ uint32_t advance_particle(const Grid &nxt, const ReplicaDev &R, const RepGeom &geo,
                                                     const Tables &T, const Topo &topo, uint32_t cap, double dt,
                                                     uint32_t step, bool integ, State me, long long fx, long long fy,
                                                     long long fz, uint32_t *err) {
    State nw = me;
    nw.tw &= ~TW_NEW;
    if (integ) {
        if ((me.tw & TW_TOPO) && topo.fb) {
            const long long *fb = topo.fb + 3ull * (R.topo_base + me.h);
            fx += fb[0];
            fy += fb[1];
            fz += fb[2];
        }
        if (fixed_saturated(fx) || fixed_saturated(fy) || fixed_saturated(fz)) atomicAdd(&err[ERR_FORCE_RANGE], 1u);
        const double Fv[3] = {(double)fx * FORCE_INV, (double)fy * FORCE_INV, (double)fz * FORCE_INV};
        double xi[3];
        bd_noise(nullptr, me.h, step, R.seed, xi);
        double p[3] = {me.x, me.y, me.z};
        em_move(T, tw_type(me.tw), dt, Fv, xi, geo.box, geo.pbc, p, err);
        nw.x = p[0];
        nw.y = p[1];
        nw.z = p[2];
    }
    const uint32_t slot = bin_insert(nxt, geo, cap, nw, err, false, 0);
    if (slot != 0xFFFFFFFFu && (me.tw & TW_TOPO) && topo.loc) topo.loc[R.topo_base + me.h] = slot;
    return slot;
}

// What step t's walk makes of a replica, from its counters before the step: take the step (active) with Philox
// step R.step + 1, and integrate step t+1 in the same walk unless this is its last step or the launch's.  The
// prologue takes no step and makes step 1's move.
struct StepPlan {
    bool active, integ;
    uint32_t step, step_next;
};
constexpr int WALK_PROLOGUE = 1, WALK_LAST = 2;  // flags of a walk

__device__ __forceinline__ StepPlan plan_step(const ReplicaDev &R, int flags) {
    StepPlan p;
    const uint64_t left = R.in_use ? R.steps_left : 0ull;
    p.active = !(flags & WALK_PROLOGUE) && left > 0;
    p.integ = (flags & WALK_PROLOGUE) ? left > 0 : (left > 1 && !(flags & WALK_LAST));
    p.step = R.step + (p.active ? 1u : 0u);
    p.step_next = p.step + 1u;
    return p;
}

// the replica's counters after its walk of step t (one thread)
__device__ __forceinline__ void book_step(ReplicaDev &R, int last) {
    if (R.in_use && R.steps_left > 0) {
        R.active = 1u;
        R.step += 1u;
        R.steps_left -= 1u;
        R.steps_done += 1u;
        R.integ = (R.steps_left > 0 && !last) ? 1u : 0u;
    } else {
        R.active = 0u;
        R.integ = 0u;
    }
}

__global__ void k_step_book(ReplicaDev *reps, uint32_t n_reps, int last) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_reps) book_step(reps[i], last);
}

// Engines with topologies only, before the bonded terms: clears the bonded forces and, with topology reactions
// on, keeps each topology particle's slot in the buffer the walk reads (loc_cur): the walk's moves point loc at
// the next buffer, and the topology reactions run after it.
__global__ void k_topo_begin(long long *fb, uint32_t n_fb, const uint32_t *loc, uint32_t *loc_cur, uint32_t n_loc) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_fb) fb[i] = 0;
    if (i < n_loc) loc_cur[i] = loc[i];
}

// The type tables of the walk, read into registers before the brick and its replica are known (one
// entry per thread: n_types <= MAX_STAGED_TYPES gives n_types^2 <= BRICK_THREADS), so that their loads
// overlap the brick's, then placed in LDS with the thresholds of the brick's frame: the force tables
// (ft) and the order-2 reaction index (st.o2); st.thr / st.reach hold the larger of the force and
// reaction thresholds / reaches.  Every entry is formed from the placing thread's own words (the
// reaches from the per-type row maxima), so the placement needs no barrier of its own: the staging
// that follows has barriers before anything reads the tables.
struct TablePrefetch {  // raw words (registers, not a stack object)
    uint4 pi;
    uint2 ri;
    uint4 pot0, pot1, pot2;
    float2 rm;
    uint32_t o1a, o1b;
};
static_assert(sizeof(PairIdx) == 16 && sizeof(RxPairIdx) == 8 && sizeof(PotDev) == 48, "table entry sizes");

__device__ __forceinline__ TablePrefetch prefetch_tables(const Tables &T) {
    TablePrefetch f{};
    const uint32_t k = threadIdx.x, n2 = T.n_types * T.n_types;
    if (k < n2) {
        f.pi = reinterpret_cast<const uint4 *>(T.pidx)[k];
        f.ri = reinterpret_cast<const uint2 *>(T.o2idx)[k];
    }
    if (k < T.n_pots) {
        const uint4 *q = reinterpret_cast<const uint4 *>(T.pots) + 3ull * k;
        f.pot0 = q[0];
        f.pot1 = q[1];
        f.pot2 = q[2];
    }
    if (k < T.n_types) {
        f.rm = T.rowmax[k];
        f.o1a = T.o1idx[k];
        f.o1b = T.o1idx[k + 1];
    }
    return f;
}

__device__ __forceinline__ void place_tables(char *base, const Tables &T, const TablePrefetch &f, float margin,
                                             ForceTables &ft, SearchTables &st) {
    const uint32_t nt = T.n_types, n2 = nt * nt, k = threadIdx.x;
    char *p = base;
    ft.pidx = (PairIdx *)p;
    p += align16(sizeof(PairIdx) * n2);
    ft.pots = (PotDev *)p;
    p += align16(sizeof(PotDev) * T.n_pots);
    ft.thr = (float *)p;
    p += align16(4 * n2);
    ft.reach = (float *)p;
    p = base + force_table_bytes(nt, T.n_pots);
    st.o2 = (RxPairIdx *)p;
    p += align16(sizeof(RxPairIdx) * n2);
    st.thr = (float *)p;
    p += align16(4 * n2);
    st.reach = (float *)p;
    p += align16(4 * nt);
    st.o1 = (uint32_t *)p;
    if (k < n2) {
        reinterpret_cast<uint4 *>(ft.pidx)[k] = f.pi;
        reinterpret_cast<uint2 *>(st.o2)[k] = f.ri;
        const PairIdx pi = ft.pidx[k];
        const RxPairIdx ri = st.o2[k];
        const float tf = prefilter_thr(pi.maxcut2_f, pi.count != 0, margin);
        ft.thr[k] = tf;
        st.thr[k] = fmaxf(tf, prefilter_thr(ri.maxr2_f, ri.count != 0, margin));
    }
    if (k < T.n_pots) {
        uint4 *q = reinterpret_cast<uint4 *>(ft.pots) + 3ull * k;
        q[0] = f.pot0;
        q[1] = f.pot1;
        q[2] = f.pot2;
    }
    for (uint32_t q = k + BRICK_THREADS; q < T.n_pots; q += BRICK_THREADS) ft.pots[q] = T.pots[q];
    if (k < nt) {
        const float rf = reach_of(f.rm.x, f.rm.x >= 0.f, margin);
        ft.reach[k] = rf;
        st.reach[k] = fmaxf(rf, reach_of(f.rm.y, f.rm.y >= 0.f, margin));
        st.o1[k] = f.o1a | ((f.o1b - f.o1a) << 16);
    }
}

// The walk of one brick over cur = x'(t): the pair forces of the brick's own records (2^-32 fixed
// point, summed in LDS per wave), step t's reaction candidates (order 1 and 2, the draws of
// k_brick_search), and each particle moved to step t+1 (or copied) into nxt as soon as its force is
// complete.  flags: WALK_PROLOGUE, the first walk of a run (no candidates; moves replicas with steps
// left, Philox step R.step + 1); WALK_LAST, the launch's last step.  Replicas neither searching nor moving are copied without a walk.  Five waves per
// SIMD are asked of the register allocator (the move inside the walk loop would otherwise take the
// kernel to three).
struct WalkArgs {
    Grid cur, nxt;
    uint32_t *clear_counts, *clear_ovf;
    const ReplicaDev *reps;
    Tables T;
    Topo topo;
    const BrickDev *bricks;
    Event *events;
    uint32_t *ev_count, *slow, *change_counts, *err;
    double dt;
    uint32_t brick0, cap, max_states, max_halo, smem_bytes;
    int32_t flags, radius, handler;
};

template <bool AH>
__global__ __launch_bounds__(BRICK_THREADS) __attribute__((amdgpu_waves_per_eu(5))) void k_brick_step(WalkArgs) {
    extern __shared__ __align__(16) char smem[];
    __shared__ StepWave wave_lds[BRICK_WAVES];
    BrickSmem m;
    ForceTables ft;
    SearchTables st;
    WalkCtx wc;
    float expand;
    uint32_t r, nt, bidx;
    const float *thr_tab, *reach_tab;
    bool rx_on, o2_on;
    bool inside;           // no halo cell across a boundary, and the brick with its halo spans less than half of
                           // every axis: raw differences are minimum images
    float lbox[3];         // FP32 box and axis modes for the general walk
    {  // staging, and the bricks that are only copied
        const WalkArgs &a = kernel_args<WalkArgs>();
        nt = a.T.n_types;
        const bool staged_types = nt <= MAX_STAGED_TYPES;
        TablePrefetch tpf;
        if (staged_types) tpf = prefetch_tables(a.T);
        bidx = a.brick0 + xcd_block(blockIdx.x, gridDim.x);
        const BrickDev &B = read_only(a.bricks + bidx);
        // the halo counters load from the brick record alone, alongside the replica's record
        const Halo Hs = make_halo(B);
        const uint32_t per = cells_per_thread(Hs);
        const HaloCells hcn = load_halo_cells(a.cur.counts, a.clear_counts, B, Hs, threadIdx.x * per, min(per, STAGE_CELLS));
        for (uint32_t u = STAGE_CELLS; u < per; u += STAGE_CELLS)  // a large halo's further cells: cleared here
            (void)load_halo_cells(a.cur.counts, a.clear_counts, B, Hs, threadIdx.x * per + u, min(per - u, STAGE_CELLS));
        r = B.r;
        const ReplicaDev &R = read_only(a.reps + r);
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *a.nxt.wl_count = 0u;
            *a.clear_ovf = 0u;
            a.change_counts[0] = 0u;  // changed records
            a.change_counts[1] = 0u;  // records to move again
        }
        if (!R.in_use) return;
        const RepGeom geo = load_geom(R);
        const StepPlan plan = plan_step(R, a.flags);  // block-uniform
        if (!plan.active && !plan.integ) {  // copy only: no forces needed
            for_each_own_record(a.cur, B, a.cap, [&](uint32_t s, const State &me) {
                if (!(me.tw & TW_DEAD))
                    advance_particle(a.nxt, R, geo, a.T, a.topo, a.cap, a.dt, plan.step_next, false, me, 0, 0, 0, a.err);
            });
            return;
        }
        rx_on = plan.active && replica_handler(R, a.handler) <= 1 && a.T.n_rx > 0;  // block-uniform
        o2_on = rx_on && a.T.has_o2;
        inside = true;
        for (int k = 0; k < 3; ++k)
            inside = inside && B.o[k] >= B.h[k] && B.o[k] + B.e[k] + B.h[k] <= B.dims[k] &&
                     2 * (B.e[k] + 2 * B.h[k]) < B.dims[k];
        const Frame F = make_frame(B, geo);
        expand = F.expand;
        for (int k = 0; k < 3; ++k) lbox[k] = F.L[k];
        uint32_t total = 0xFFFFFFFFu;
        if (staged_types) {
            if (table_bytes(nt, a.T.n_pots) + brick_smem_bytes(a.max_states, a.max_halo) > a.smem_bytes) {  // block-uniform
                if (threadIdx.x == 0) atomicAdd(&a.err[ERR_LDS_LAYOUT], 1u);
                return;
            }
            // with reactions on, the walk reaches the larger of the force and reaction cutoffs
            place_tables(smem, a.T, tpf, F.margin, ft, st);
            m = carve(smem + table_bytes(nt, a.T.n_pots), a.max_states, a.max_halo);
            total = stage_brick(a.cur, B, geo, F, a.cap, m, a.max_states, Hs, hcn);
        }
        if (total == 0xFFFFFFFFu) {
            list_slow_brick(a.slow, bidx, a.err);
            return;
        }
        wc = make_walk(B, geo, Hs, a.radius);
        if (AH != (wc.whole == 0)) {  // launch and brick disagree (host invariant): refuse the brick
            if (threadIdx.x == 0) atomicAdd(&a.err[ERR_LDS_LAYOUT], 1u);
            return;
        }
        thr_tab = o2_on ? st.thr : ft.thr;
        reach_tab = o2_on ? st.reach : ft.reach;
    }
    StepWave &W = wave_lds[threadIdx.x / 64];
    const uint32_t lane = __lane_id();
    // a surviving pair (entry = owner lane << 16 | staged neighbour): the exact FP64 gates, the
    // pair force on the owner, and (each unordered pair once) the order-2 draws
    State me{};  // this lane's own record in the current round (the walk's owner records)
    // The draws of the wave's reaction candidates: entries as the pairs', with NO_PARTNER for an order-1
    // candidate.  Almost every batch of pairs holds a candidate or two, and a wave a dozen: one batch of draws
    // for all of them costs the wave one Philox block instead of one a batch.
    uint32_t n_draw = 0;  // wave-uniform
    auto draw = [&]() {   // makes the last 64 listed draws
        wave_lds_sync();
        const uint32_t first = n_draw > 64u ? n_draw - 64u : 0u;
        const uint32_t ent = first + lane < n_draw ? W.draw[first + lane] : NO_ENTRY;
        const uint32_t ol = ent == NO_ENTRY ? 0u : ent >> 16, q = ent & 0xFFFFu;
        State own;
        own.x = __shfl(me.x, (int)ol);
        own.y = __shfl(me.y, (int)ol);
        own.z = __shfl(me.z, (int)ol);
        own.tw = __shfl(me.tw, (int)ol);
        own.h = __shfl(me.h, (int)ol);
        n_draw = first;
        if (ent == NO_ENTRY) return;
        const WalkArgs &a = kernel_args<WalkArgs>();
        const ReplicaDev &R = read_only(a.reps + r);
        const uint32_t s1 = m.slot[W.j[ol]], t1 = tw_type(own.tw), step = plan_step(R, a.flags).step;
        const bool pair = q != NO_PARTNER;
        uint32_t s2 = s1, h2 = own.h, t2 = t1;
        double d2 = 0.0;
        if (pair) {
            s2 = m.slot[q];
            const State o = a.cur.bins[s2];
            h2 = o.h;
            t2 = tw_type(o.tw);
            // distSquared(neighbor.pos, entry.pos) (CPUUncontrolledApproximation.cpp:108)
            d2 = dist2(min_image(o.x - own.x, R.box[0], R.pbc[0]), min_image(o.y - own.y, R.box[1], R.pbc[1]),
                       min_image(o.z - own.z, R.box[2], R.pbc[2]));
        }
        const RxPairIdx ri = st.o2[t1 * nt + t2];
        const uint32_t o1 = st.o1[t1];
        uint32_t k = pair ? ri.start : (o1 & 0xFFFFu);
        const uint32_t ke = k + (pair ? ri.count : (o1 >> 16));
        for (; k < ke; ++k) {
            const uint32_t rx = pair ? a.T.o2list[k] : a.T.o1list[k];
            const RxDev X = a.T.rx[rx];
            if (!(X.rate > 0) || (pair && !(d2 < X.educt_dist2))) continue;
            uint32_t x4[4];
            philox(min(own.h, h2), step, (pair ? 2u : 1u) | (rx << 8), pair ? max(own.h, h2) : 0u, R.seed, x4);
            if (!(u53(x4[0], x4[1]) < X.p_accept)) continue;
            // entry1: the educt of type educts[0]; equal educt types: the lower handle
            const bool me_first =
                !pair || ((X.educts[0] != X.educts[1]) ? (t1 == X.educts[0]) : (own.h < h2));
            const uint32_t p = atomicAdd(&a.ev_count[r], 1u);
            if (p < R.ev_cap) {
                Event ev;
                ev.key = event_words(x4);
                ev.s1 = me_first ? s1 : s2;
                ev.s2 = me_first ? s2 : s1;
                ev.h1 = me_first ? own.h : h2;
                ev.h2 = me_first ? h2 : own.h;
                ev.rx = rx;
                ev.pad = 0;
                a.events[R.ev_base + p] = ev;
            } else {
                atomicAdd(&a.err[ERR_EVENT_OVERFLOW], 1u);
            }
        }
    };
    auto list_draw = [&](bool want, uint32_t ent) {  // every lane of the wave comes along
        const unsigned long long mk = __ballot(want);
        if (want) W.draw[n_draw + rank_in_mask(mk)] = ent;
        n_draw += (uint32_t)__popcll(mk);
    };
    auto eval = [&](uint32_t ent) {
        // the owner's record from the owner lane's registers (every lane takes part in the shuffles)
        const uint32_t ol = ent == NO_ENTRY ? 0u : ent >> 16, q = ent & 0xFFFFu;
        State me_o;
        me_o.x = __shfl(me.x, (int)ol);
        me_o.y = __shfl(me.y, (int)ol);
        me_o.z = __shfl(me.z, (int)ol);
        me_o.tw = __shfl(me.tw, (int)ol);
        me_o.h = __shfl(me.h, (int)ol);
        bool react = false;
        if (ent != NO_ENTRY) {
            const WalkArgs &a = kernel_args<WalkArgs>();
            const ReplicaDev &R = read_only(a.reps + r);
            const State &me = me_o;
            const uint32_t s2 = m.slot[q];
            const State o = a.cur.bins[s2];
            const uint32_t t1 = tw_type(me.tw), t2 = tw_type(o.tw);
            // CPUCalculateForces.cpp:226-259: x_ij = shortestDifference(x_i, x_j), gate d2 < rc^2.
            // The reaction gate measures distSquared(x_j, x_i) (CPUUncontrolledApproximation.cpp:108):
            // the same square, since a - b = -(b - a) and the minimum image is symmetric in magnitude.
            double ddx = o.x - me.x, ddy = o.y - me.y, ddz = o.z - me.z;
            if (!inside) {
                ddx = min_image(ddx, R.box[0], R.pbc[0]);
                ddy = min_image(ddy, R.box[1], R.pbc[1]);
                ddz = min_image(ddz, R.box[2], R.pbc[2]);
            }
            const double d2 = dist2(ddx, ddy, ddz);
            long long px, py, pz, pe;
            bool saturated;
            if (pair_fixed<false>(ft.pots, ft.pidx[t1 * nt + t2], ddx, ddy, ddz, d2, px, py, pz, pe, &saturated)) {
                if (saturated) atomicAdd(&a.err[ERR_FORCE_RANGE], 1u);
                atomicAdd(&W.acc[0][ol], (unsigned long long)px);
                atomicAdd(&W.acc[1][ol], (unsigned long long)py);
                atomicAdd(&W.acc[2][ol], (unsigned long long)pz);
            }
            // order-2 candidates, each unordered pair once: the lower type finds it; equal types: the lower bin
            // slot.  Their draws wait in a list of the wave (list_draw), with those of order 1
            if (o2_on && ((t2 > t1) || (t2 == t1 && s2 > m.slot[W.j[ol]]))) {
                const RxPairIdx ri = st.o2[t1 * nt + t2];
                react = ri.count != 0 && d2 < (double)ri.maxr2_f * (1.0 + 1.0e-6);
            }
        }
        if (__ballot(react)) list_draw(react, ent);
    };
    for (uint32_t q0 = threadIdx.x / 64 * 16;; q0 += BRICK_THREADS / 4) {  // wave-uniform
        uint32_t n_quads;
        {
            const BrickDev &B = read_only(kernel_args<WalkArgs>().bricks + bidx);
            n_quads = wave_quads(m, B, make_halo(B), W.quads, q0);
        }
        if (q0 >= n_quads) break;
        wave_lds_sync();
        const OwnerLane ow = owner_lane(m, W.quads, q0, n_quads);
        const uint32_t j = ow.j;
        const bool valid = ow.valid;
        me = State{};
        uint32_t sj = 0;
        {
            const WalkArgs &a = kernel_args<WalkArgs>();
            if (valid) {
                sj = m.slot[j];
                me = a.cur.bins[sj];  // (first needed by the first batch of pairs)
            }
            W.j[lane] = (uint16_t)j;
            W.acc[0][lane] = 0ull;
            W.acc[1][lane] = 0ull;
            W.acc[2][lane] = 0ull;
            wave_lds_sync();
        }
        const uint32_t t = ow.t & TYP_MASK;
        // order 1 (CPUUncontrolledApproximation.cpp:81-95)
        if (rx_on) list_draw(valid && (st.o1[t] >> 16) != 0u, (lane << 16) | NO_PARTNER);
        const float reach = reach_tab[t];
        const bool active = valid && !(ow.t & TYP_OUTSIDE) && reach >= 0.f;
        const float4 pj = m.P[j];
        char *wave_ring = m.rings + (threadIdx.x / 64) * WAVE_RING_BYTES;
        if constexpr (AH) {
            auto filter = [&](uint32_t ent) -> bool {
                const uint32_t q = ent & 0xFFFFu, jo = W.j[ent >> 16];
                const float4 a = m.P[jo], b = m.P[q];
                return (q != jo) & (prefilter_d2(b.x - a.x, b.y - a.y, b.z - a.z) < thr_tab[m.typ[jo] * nt + m.typ[q]]);
            };
            // draws a full list as it comes, and the rest when the pairs are done
            auto after = [&](bool done) -> bool {
                if (n_draw >= 64 || (done && n_draw)) draw();
                return n_draw != 0;
            };
            mfma_pipeline(wc, m.hstart, m.P, m.far, wave_ring, active, m.hc_of[j], pj, reach, expand, filter, eval, after);
        } else {
            const float *thr_row = thr_tab + t * nt;
            // prefilter, branch-free: one LDS read of the candidate, one of the threshold
            auto keep = [&](uint32_t q, const float4 &pq) -> bool {
                const uint32_t tq = m.typ[q];
                float dx = pq.x - pj.x, dy = pq.y - pj.y, dz = pq.z - pj.z;
                frame_min_image(wc.whole, lbox, dx, dy, dz);
                return (q != j) & (tq < TYP_OUTSIDE) & (prefilter_d2(dx, dy, dz) < thr_row[tq & TYP_MASK]);
            };
            auto eval_draw = [&](uint32_t ent) {
                eval(ent);
                if (n_draw >= 64) draw();
            };
            if (n_draw >= 64) draw();
            pair_pipeline(wc, m.hstart, m.P, (uint32_t *)wave_ring, active, m.hc_of[j], keep, eval_draw);
            if (n_draw) draw();
        }
        wave_lds_sync();
        // the move with the finished pair force, from the owner's registers
        const long long fx = (long long)W.acc[0][lane], fy = (long long)W.acc[1][lane], fz = (long long)W.acc[2][lane];
        wave_lds_sync();
        if (valid) {
            const WalkArgs &a = kernel_args<WalkArgs>();
            const ReplicaDev &R = read_only(a.reps + r);
            const StepPlan plan = plan_step(R, a.flags);
            advance_particle(a.nxt, R, load_geom(R), a.T, a.topo, a.cap, a.dt, plan.step_next, plan.integ, me, fx, fy, fz,
                             a.err);
        }
    }
}

// the listed bricks of a k_brick_step without candidates (a prologue, or a step without reactions), neighbours
// read straight from the bins
__global__ __launch_bounds__(BRICK_THREADS) void k_brick_step_slow(Grid cur, Grid nxt, int flags, ReplicaDev *reps,
                                                                   Tables T, Topo topo, const BrickDev *bricks,
                                                                   uint32_t cap, int radius, double dt, uint32_t *slow,
                                                                   uint32_t *err) {
    const uint32_t n = slow_count(slow);
    if (n == 0) return;  // grid-uniform
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {  // block-uniform
        const BrickDev B = bricks[slow[2 + i]];
        const ReplicaDev &R = reps[B.r];
        const RepGeom geo = load_geom(R);
        const StepPlan plan = plan_step(R, flags);
        for_each_own_record(cur, B, cap, [&](uint32_t s, const State &me) {
            if (me.tw & TW_DEAD) return;
            long long fx = 0, fy = 0, fz = 0, e = 0;
            if (!(me.tw & TW_OUTSIDE)) global_forces(cur, geo, cap, radius, T, s, me, fx, fy, fz, e);
            advance_particle(nxt, R, geo, T, topo, cap, dt, plan.step_next, plan.integ, me, fx, fy, fz, err);
        });
    }
    release_slow_list(slow);
}

// A fused step's counters and reactions (resolve_replica, one workgroup per replica), preceded by the replica's
// bricks that k_brick_step listed for the bin-reading path (their candidates join the replica's list
// first).  The walk then needs no follow-up launch, which costs as much as a short kernel's work.
__global__ __launch_bounds__(RESOLVE_THREADS) void k_resolve_step(Grid cur, Grid nxt, ReplicaDev *reps, Tables T,
                                                                  Topo topo, const BrickDev *bricks, uint32_t cap,
                                                                  int radius, int handler, double dt, int last,
                                                                  Event *events, uint32_t *ev_count, uint32_t *slow,
                                                                  unsigned long long *rx_step,
                                                                  unsigned long long *rx_total, uint32_t max_wl,
                                                                  Edit *edits, uint32_t *edit_count,
                                                                  uint32_t edit_cap, RxRecord *recs,
                                                                  uint32_t *rec_count, uint32_t *err) {
    const uint32_t n = slow_count(slow);  // the same for every block: the walk has ended
    if (threadIdx.x == 0) book_step(reps[blockIdx.x], last);
    __syncthreads();
    for (uint32_t i = 0; i < n; ++i) {    // block-uniform
        const BrickDev B = bricks[slow[2 + i]];
        if (B.r != blockIdx.x) continue;
        const ReplicaDev &R = reps[B.r];
        const RepGeom geo = load_geom(R);
        const bool integ = R.integ != 0u;
        const uint32_t step_next = R.step + 1u;
        for_each_own_record(cur, B, cap, [&](uint32_t s, const State &me) {
            if (me.tw & TW_DEAD) return;
            long long fx = 0, fy = 0, fz = 0, e = 0;
            if (!(me.tw & TW_OUTSIDE)) global_forces(cur, geo, cap, radius, T, s, me, fx, fy, fz, e);
            if (R.active && replica_handler(R, handler) <= 1)  // as the staged walk's rx_on
                search_one(cur, reps, T, cap, radius, 0, events, ev_count, nullptr, 0, s, me, err);
            advance_particle(nxt, R, geo, T, topo, cap, dt, step_next, integ, me, fx, fy, fz, err);
        });
    }
    if (n) {
        __syncthreads();
        __threadfence();  // the listed bricks' candidates before the replica's list is read
    }
    resolve_replica(cur, reps, T, cap, events, ev_count, rx_step, rx_total, handler, 1, max_wl, edits, edit_count, edit_cap,
                    recs, rec_count, err);
    if (n) release_slow_list(slow);
}

// the cells of the (2r+1)^3 stencil of local cell cl, de-duplicated as axis_cells does
struct StencilDims {
    int i[3], na[3];
    uint32_t n;
};

__device__ __forceinline__ StencilDims stencil_dims(const RepGeom &geo, uint32_t cl, int radius) {
    const uint32_t nz = (uint32_t)geo.dims[2], ny = (uint32_t)geo.dims[1];
    StencilDims d;
    d.i[2] = (int)(cl % nz);
    d.i[1] = (int)((cl / nz) % ny);
    d.i[0] = (int)(cl / (nz * ny));
    d.n = 1;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        d.na[a] = axis_count(d.i[a], geo.dims[a], geo.pbc[a], radius);
        d.n *= (uint32_t)d.na[a];
    }
    return d;
}

__device__ __forceinline__ uint32_t stencil_cell(const RepGeom &geo, const StencilDims &d, uint32_t c, int radius) {
    const int yz = d.na[1] * d.na[2], a = (int)c / yz, rem = (int)c % yz, b = rem / d.na[2], k = rem % d.na[2];
    return geo.cell_base + ((uint32_t)axis_elem(a, d.i[0], geo.dims[0], geo.pbc[0], radius) * (uint32_t)geo.dims[1] +
                            (uint32_t)axis_elem(b, d.i[1], geo.dims[1], geo.pbc[1], radius)) *
                               (uint32_t)geo.dims[2] +
           (uint32_t)axis_elem(k, d.i[2], geo.dims[2], geo.pbc[2], radius);
}

// fn(cell) for every `lanes`-th cell of the stencil from cell `first` on
template <class Fn>
__device__ __forceinline__ void stencil_cells(const RepGeom &geo, uint32_t cl, int radius, uint32_t first,
                                              uint32_t lanes, Fn &&fn) {
    const StencilDims d = stencil_dims(geo, cl, radius);
    for (uint32_t c = first; c < d.n; c += lanes) fn(stencil_cell(geo, d, c, radius));
}

// fn(slot) for every record of one cell of buffer g (overflow records included)
template <class Fn>
__device__ __forceinline__ void cell_records(const Grid &g, uint32_t cap, uint32_t cell, Fn &&fn) {
    const uint32_t cnt = g.counts[cell];
    const uint32_t mm = cnt < cap ? cnt : cap;
    for (uint32_t q = 0; q < mm; ++q) fn(cell * cap + q);
    if (cnt > cap) {  // rare: a crowded cell spilled into the overflow region
        uint32_t no = *g.ovf_count;
        no = no < g.ovf_cap ? no : g.ovf_cap;
        for (uint32_t o = 0; o < no; ++o)
            if (g.ovf_cell[o] == cell) fn(g.nbin + o);
    }
}

// fn(slot, record) for every record of one cell, four records loaded together (a cell's records are one
// round trip instead of one each)
template <class Fn>
__device__ __forceinline__ void cell_records4(const Grid &g, uint32_t cap, uint32_t cell, Fn &&fn) {
    const uint32_t cnt = g.counts[cell];
    const uint32_t mm = cnt < cap ? cnt : cap;
    for (uint32_t q = 0; q < mm; q += 4) {
        State o[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            if (q + u < mm) o[u] = g.bins[cell * cap + q + u];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            if (q + u < mm) fn(cell * cap + q + u, o[u]);
    }
    if (cnt > cap) {  // rare: a crowded cell spilled into the overflow region
        uint32_t no = *g.ovf_count;
        no = no < g.ovf_cap ? no : g.ovf_cap;
        for (uint32_t o = 0; o < no; ++o)
            if (g.ovf_cell[o] == cell) fn(g.nbin + o, g.bins[g.nbin + o]);
    }
}

// Withdraws the moved copies of the wave's pending records from nxt: lanes with `has` name a record (its slot in
// cur and the handle its copy carries).  Two records at a time, half a wave each, its lanes spread over the
// cells around the record's cell; a copy that moved further than one cell is searched by the whole wave, at
// last in the replica's whole grid.
__device__ __forceinline__ void withdraw_copies(const Grid &cur, const Grid &nxt, const ReplicaDev &R,
                                                const RepGeom &geo, uint32_t cap, bool has, uint32_t slot,
                                                uint32_t handle) {
    const uint32_t lane = __lane_id();
    unsigned long long pending = __ballot(has);
    while (pending) {
        const int l0 = __ffsll((long long)pending) - 1;
        pending &= pending - 1ull;
        const int l1 = pending ? __ffsll((long long)pending) - 1 : -1;
        if (pending) pending &= pending - 1ull;
        const int src = lane < 32 ? l0 : l1;
        const uint32_t s = (uint32_t)__shfl((int)slot, src < 0 ? l0 : src);
        const uint32_t h = (uint32_t)__shfl((int)handle, src < 0 ? l0 : src);
        const uint32_t cl = cell_of_slot(cur, s, cap) - geo.cell_base;
        bool found = false;
        auto probe = [&](uint32_t cell) {
            cell_records4(nxt, cap, cell, [&](uint32_t s2, const State &o) {
                if (o.h == h && !(o.tw & TW_DEAD)) {
                    nxt.bins[s2].tw = o.tw | TW_DEAD;
                    found = true;
                }
            });
        };
        if (src >= 0) stencil_cells(geo, cl, 1, lane & 31u, 32u, probe);
        const unsigned long long f = __ballot(found);
        for (int half = 0; half < 2; ++half) {  // wave-uniform
            if ((f >> (32 * half)) & 0xFFFFFFFFull) continue;
            const int l = half ? l1 : l0;
            if (l < 0) continue;
            const uint32_t sw = (uint32_t)__shfl((int)slot, l), hw = (uint32_t)__shfl((int)handle, l);
            bool hit = false;
            auto far = [&](uint32_t cell) {
                cell_records4(nxt, cap, cell, [&](uint32_t s2, const State &o) {
                    if (o.h == hw && !(o.tw & TW_DEAD)) {
                        nxt.bins[s2].tw = o.tw | TW_DEAD;
                        hit = true;
                    }
                });
            };
            stencil_cells(geo, cell_of_slot(cur, sw, cap) - geo.cell_base, 2, lane, 64u, far);
            if (__ballot(hit)) continue;
            for (uint32_t c = lane; c < R.n_cells; c += 64) far(geo.cell_base + c);
        }
    }
}

// Per changed record of step t's reactions, one wave each, its lanes spread over the record's
// stencil cells; cur is x'(t) with the reactions applied, nxt holds the walk's optimistic moves.
//   killed k:   its moved copy is withdrawn;
//   inserted p: p is listed for a move;
//   retyped r:  its moved copy (under its old handle) is withdrawn and r is listed;
// and, when the replica moves this step, every surviving old neighbour n (a live record without
// TW_NEW) whose pair force from the changed record differs between before and after is listed
// once (bit in aff_bits) for a fresh force and a new move, its moved copy withdrawn.  Nothing is
// inserted into nxt before every withdrawal is done (k_fix_advance), so the records below each
// cell's count are stable while they are searched.
__global__ __launch_bounds__(256) void k_fix_sites(Grid cur, Grid nxt, const ReplicaDev *reps, Tables T, uint32_t cap,
                                                   int radius, const Edit *edits, const uint32_t *edit_count,
                                                   uint32_t edit_cap, uint32_t *aff_bits, uint32_t *aff_list,
                                                   uint32_t *aff_count, uint32_t aff_cap, uint32_t *err) {
    const uint32_t lane = __lane_id();
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const uint32_t n_waves = (gridDim.x * blockDim.x) >> 6;
    uint32_t n_edit = *edit_count;
    n_edit = n_edit < edit_cap ? n_edit : edit_cap;
    const uint32_t nt = T.n_types;
    auto list = [&](uint32_t s) {
        const uint32_t p = atomicAdd(aff_count, 1u);
        if (p < aff_cap) aff_list[p] = s;
        else atomicAdd(&err[ERR_EDIT_OVERFLOW], 1u);
    };
    for (uint32_t k = wave; k < n_edit; k += n_waves) {  // wave-uniform
        const Edit ed = edits[k];
        const uint32_t kind = ed.info & 3u, t_old = ed.info >> 2;
        const uint32_t slot = ed.slot;
        const ReplicaDev &R = reps[ed.r];
        const State st = cur.bins[slot];
        const RepGeom geo = load_geom(R);
        if (lane == 0 && kind != EDIT_KILLED) list(slot);
        // the copy carries the handle the record had
        withdraw_copies(cur, nxt, R, geo, cap, lane == 0 && kind != EDIT_INSERTED, slot,
                        kind == EDIT_RETYPED ? ed.pad : st.h);
        if (!R.integ || (st.tw & TW_OUTSIDE)) continue;  // copies only, or no neighbours
        const uint32_t ts = tw_type(st.tw);
        // true when n's pair force changed and no other site has listed it
        auto affected = [&](uint32_t s2, const State &n) -> bool {
            if (s2 == slot || (n.tw & (TW_DEAD | TW_OUTSIDE | TW_NEW))) return false;
            const uint32_t tn = tw_type(n.tw);
            // the pair seen from n: x = site - n
            const double dx = min_image(st.x - n.x, geo.box[0], geo.pbc[0]);
            const double dy = min_image(st.y - n.y, geo.box[1], geo.pbc[1]);
            const double dz = min_image(st.z - n.z, geo.box[2], geo.pbc[2]);
            const double d2 = dist2(dx, dy, dz);
            long long ax, ay, az, bx = 0, by = 0, bz = 0, pe;
            pair_fixed<false>(T.pots, T.pidx[tn * nt + ts], dx, dy, dz, d2, ax, ay, az, pe);
            if (kind == EDIT_RETYPED)
                pair_fixed<false>(T.pots, T.pidx[tn * nt + t_old], dx, dy, dz, d2, bx, by, bz, pe);
            if (((ax - bx) | (ay - by) | (az - bz)) == 0) return false;  // n's sum is unchanged
            const uint32_t bit = 1u << (s2 & 31u);
            return !(atomicOr(&aff_bits[s2 >> 5], bit) & bit);
        };
        const uint32_t cl = cell_of_slot(cur, slot, cap) - geo.cell_base;
        const StencilDims sd = stencil_dims(geo, cl, radius);
        for (uint32_t c0 = 0; c0 < sd.n; c0 += 64) {  // wave-uniform
            const bool mine = c0 + lane < sd.n;
            const uint32_t cell = mine ? stencil_cell(geo, sd, c0 + lane, radius) : 0u;
            const uint32_t cnt = mine ? cur.counts[cell] : 0u, mm = cnt < cap ? cnt : cap;
            for (uint32_t q = 0; __ballot(q < mm); q += 4) {
                State o[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u)
                    if (q + u < mm) o[u] = cur.bins[cell * cap + q + u];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) {
                    const uint32_t s2 = cell * cap + q + u;
                    const bool hit = q + u < mm && affected(s2, o[u]);
                    if (hit) list(s2);
                    withdraw_copies(cur, nxt, R, geo, cap, hit, s2, hit ? o[u].h : 0u);
                }
            }
            if (__ballot(cnt > cap)) {  // rare: crowded cells spilled into the overflow region
                uint32_t no = *cur.ovf_count;
                no = no < cur.ovf_cap ? no : cur.ovf_cap;
                for (uint32_t v = 0; v < no; ++v) {
                    const uint32_t s2 = cur.nbin + v;
                    const bool in = cnt > cap && cur.ovf_cell[v] == cell;
                    State n{};
                    if (in) n = cur.bins[s2];
                    const bool hit = in && affected(s2, n);
                    if (hit) list(s2);
                    withdraw_copies(cur, nxt, R, geo, cap, hit, s2, n.h);
                }
            }
        }
    }
}

// Moves each listed record again (one wave each): its pair force formed afresh over the live
// records of its stencil in the post-reaction state cur (pair_fixed, the sum a walk forms), then
// the move (or the copy) into nxt; an old record's bit in aff_bits is cleared for the next step
__global__ __launch_bounds__(256) void k_fix_advance(Grid cur, Grid nxt, const ReplicaDev *reps, Tables T, Topo topo,
                                                     uint32_t cap, int radius, double dt, uint32_t *aff_bits,
                                                     const uint32_t *aff_list, const uint32_t *aff_count,
                                                     uint32_t aff_cap, uint32_t *err) {
    const uint32_t lane = __lane_id();
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const uint32_t n_waves = (gridDim.x * blockDim.x) >> 6;
    uint32_t n = *aff_count;
    n = n < aff_cap ? n : aff_cap;
    const uint32_t nt = T.n_types;
    for (uint32_t k = wave; k < n; k += n_waves) {  // wave-uniform
        const uint32_t s = aff_list[k];
        const State me = cur.bins[s];
        const ReplicaDev &R = reps[tw_replica(me.tw)];
        const RepGeom geo = load_geom(R);
        const bool integ = R.integ != 0u;
        long long fx = 0, fy = 0, fz = 0;
        if (integ && !(me.tw & TW_OUTSIDE)) {
            const uint32_t t = tw_type(me.tw);
            stencil_cells(geo, cell_of_slot(cur, s, cap) - geo.cell_base, radius, lane, 64u, [&](uint32_t cell) {
                cell_records4(cur, cap, cell, [&](uint32_t s2, const State &o) {
                    if (s2 == s) return;
                    if (o.tw & (TW_DEAD | TW_OUTSIDE)) return;
                    // CPUCalculateForces.cpp:226-259: x = shortestDifference(x_i, x_j)
                    const double dx = min_image(o.x - me.x, geo.box[0], geo.pbc[0]);
                    const double dy = min_image(o.y - me.y, geo.box[1], geo.pbc[1]);
                    const double dz = min_image(o.z - me.z, geo.box[2], geo.pbc[2]);
                    long long px, py, pz, pe;
                    if (pair_fixed<false>(T.pots, T.pidx[t * nt + tw_type(o.tw)], dx, dy, dz, dist2(dx, dy, dz), px,
                                          py, pz, pe)) {
                        fx += px;
                        fy += py;
                        fz += pz;
                    }
                });
            });
            for (int off = 32; off > 0; off >>= 1) {
                fx += __shfl_xor(fx, off);
                fy += __shfl_xor(fy, off);
                fz += __shfl_xor(fz, off);
            }
        }
        if (lane == 0) {
            if (!(me.tw & TW_NEW)) atomicAnd(&aff_bits[s >> 5], ~(1u << (s & 31u)));
            advance_particle(nxt, R, geo, T, topo, cap, dt, R.step + 1u, integ, me, fx, fy, fz, err);
        }
    }
}

}  // namespace rdy
