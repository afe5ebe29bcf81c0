// VolPathTracerAD samples in stages: the paths of a batch of samples advance one bounce
// per launch, with their state in HBM between launches.
//
//  k_ad_bounce<N>   one bounce (ad_bounce.inc) of every path still alive, the continuation
//                   walk that the last bounce handed over first; the first launch of a
//                   batch starts the samples at their camera rays
//  k_ad_edges<N>    the edge term (edgeTerm) of the bounces that have one
//  k_ad_finish<N>   the samples' radiance into the accumulators, the samples whose pushes
//                   overflowed the queue into the replay list
//
// Included by kernels.hip.
#pragma once

// Path state of one batch: structure of arrays over the batch's slots (slot i is the
// batch's sample i). Reals: ro, rd, beta, L with their tangents, the walk's MIS partner
// pdf, and what the edge term needs of its bounce. Words: see Word.
template <int N> struct AdSlots {
    real *f;
    uint32_t *w;
    size_t n;   // slots
    enum Real { RO = 0, RD = 3 * (N + 1), BETA = 6 * (N + 1), L = 9 * (N + 1), CPDF = 12 * (N + 1), ETHR, EBETA = ETHR + 3,
                EWI = EBETA + 3, EGN = EWI + 3, ESN = EGN + 3, REALS = ESN + 3 };
    enum Word { PIX = 0, VIEW, FLAGS, FACE, RBLK, RPOS, RB0, RB1, RB2, RB3, CHILD, SKIP, FAILED, EFLAGS, EFACE, WORDS };
    static_assert(REALS == adSlotReals(N) && WORDS == AD_SLOT_WORDS, "adSlotBytes sizes this layout");
    static constexpr uint32_t RD_CONST = 1u << 31;   // FLAGS: rd has no tangents (none are stored)
    DI real &r(int k, uint32_t slot) const { return f[(size_t)k * n + slot]; }
    DI uint32_t &u(int k, uint32_t slot) const { return w[(size_t)k * n + slot]; }
    DI f3 ld(int k, uint32_t s) const { return f3{r(k, s), r(k + 1, s), r(k + 2, s)}; }
    DI void st(int k, uint32_t s, f3 v) const { r(k, s) = v.x; r(k + 1, s) = v.y; r(k + 2, s) = v.z; }
    DI Dv<N> ldv(int k, uint32_t s) const {
        Dv<N> v(ld(k, s));
#pragma unroll
        for (int j = 0; j < N; ++j) v.setGrad(j, ld(k + 3 + 3 * j, s));
        return v;
    }
    DI void stv(int k, uint32_t s, const Dv<N> &v) const {
        st(k, s, v.val());
#pragma unroll
        for (int j = 0; j < N; ++j) st(k + 3 + 3 * j, s, v.grad(j));
    }
    DI Ds<N> lds(int k, uint32_t s) const {
        Ds<N> v(ld(k, s));
#pragma unroll
        for (int j = 0; j < N; ++j)
            for (int c = 0; c < 3; ++c) v.c[c].d[j] = r(k + 3 + 3 * j + c, s);
        return v;
    }
    DI void sts(int k, uint32_t s, const Ds<N> &v) const {
        st(k, s, v.val());
#pragma unroll
        for (int j = 0; j < N; ++j)
            for (int c = 0; c < 3; ++c) r(k + 3 + 3 * j + c, s) = v.c[c].d[j];
    }
    // the random stream of slot s's sample: keyed by its view's seed and index ls
    DI void ldRng(uint32_t s, uint64_t seed, uint64_t ls, Rng &g) const {
        g.init(seed, ls);
        g.blk = u(RBLK, s);
        g.pos = (int)u(RPOS, s);
        g.b0 = u(RB0, s); g.b1 = u(RB1, s); g.b2 = u(RB2, s); g.b3 = u(RB3, s);
    }
    DI void stRng(uint32_t s, const Rng &g) const {
        u(RBLK, s) = g.blk;
        u(RPOS, s) = (uint32_t)g.pos;
        if (g.pos < 4) { u(RB0, s) = g.b0; u(RB1, s) = g.b1; u(RB2, s) = g.b2; u(RB3, s) = g.b3; }
    }
};

// A batch: its samples, its slots, and the lists and counters of one bounce.
struct AdBatch {
    char *state;                 // AdSlots: REALS * n reals, then WORDS * n words
    uint32_t n;                  // slots
    uint32_t m;                  // samples of the batch, <= n
    uint64_t s0;                 // first sample (replay == nullptr)
    const uint4 *replay;         // or the batch's entries {sid lo, sid hi, children delivered, 0}
    const uint32_t *in;          // slots alive at the start of the bounce (nullptr: all m, started here)
    uint32_t *out, *edges;       // slots alive after it; slots with an edge term
    uint32_t *cnt;               // [0] length of in, [1] consumed, [2] length of edges, [3] consumed, [4] length of out
};
template <int N> DI AdSlots<N> slotsOf(const AdBatch &B) {
    AdSlots<N> a;
    a.n = B.n;
    a.f = reinterpret_cast<real *>(B.state);
    a.w = reinterpret_cast<uint32_t *>(a.f + (size_t)AdSlots<N>::REALS * B.n);
    return a;
}

// Where a bounce's edge term is written for k_ad_edges (AD_EDGE_DEFERRED of ad_bounce.inc).
template <int N> struct AdEdgeOut {
    const AdSlots<N> &a;
    uint32_t slot;
    bool set;
    DI void put(bool vol, const Dv<N> &x, const Hit &its0, f3 rdin, f3 thrv, f3 betav, int med, int depth) {
        using A = AdSlots<N>;
        set = true;
        a.stv(A::RO, slot, x);   // also the next ray's origin
        a.st(A::ETHR, slot, thrv);
        a.st(A::EBETA, slot, betav);
        a.u(A::EFLAGS, slot) = (vol ? 1u : 0u) | (uint32_t)depth << 1 | (uint32_t)(med + 1) << 9;
        if (vol) {
            a.st(A::EWI, slot, rdin);
        } else {
            a.u(A::EFACE, slot) = (uint32_t)its0.face;
            a.st(A::EWI, slot, its0.wi);
            a.st(A::EGN, slot, its0.gn);
            a.st(A::ESN, slot, its0.sn);
        }
    }
};

// A wave's share of a list of `n` items. It takes a full wave's at a time while there are
// more than the launch's waves can hold, else an even share, so that a short list (a small
// image, the last bounces) spreads over the whole chip: a wave's time grows with the lanes
// that diverge in it. The first share is fixed, dealt to one wave of each block before the
// next one's; the others come from the counter.
struct ListShare {
    uint32_t *consumed;
    uint32_t n, per, waves, base;
    DI ListShare(uint32_t *consumed_, uint32_t n_) : consumed(consumed_), n(n_) {
        waves = gridDim.x * (blockDim.x / 64);
        const uint32_t even = (n + waves - 1) / waves;
        per = even >= 64 ? 64 : even < 4 ? 4 : even;
        base = (threadIdx.x / 64 * gridDim.x + blockIdx.x) * per;
    }
    DI bool idleBlock() const { return blockIdx.x * per >= n; }   // nothing for any wave of the block
    DI bool more() const { return base < n; }
    DI bool item(uint32_t &i) const {
        i = base + (threadIdx.x & 63);
        return (threadIdx.x & 63) < per && i < n;
    }
    DI void next() {
        uint32_t k = 0;
        if ((threadIdx.x & 63) == 0) k = atomicAdd(consumed, per);
        base = waves * per + __shfl(k, 0);
    }
};
// Appends the slots of the lanes with `put` to a list, in lane order.
DI void appendSlots(bool put, uint32_t slot, uint32_t *list, uint32_t *len) {
    const uint64_t m = __ballot(put);
    if (!m) return;
    const int lead = __ffsll((unsigned long long)m) - 1;
    uint32_t base = 0;
    if ((int)(threadIdx.x & 63) == lead) base = atomicAdd(len, (uint32_t)__popcll(m));
    base = __shfl(base, lead);
    if (put) list[base + (uint32_t)__popcll(m & __lanemask_lt())] = slot;
}

template <int N>
__global__ __launch_bounds__(AD_STAGE_BLOCK, AD_BOUNCE_WAVES) void k_ad_bounce(DScene S, RenderParams P, AdBatch B, char *q,
                                                                             unsigned *qcount, unsigned *stats,
                                                                             unsigned long long *work) {
    using A = AdSlots<N>;
    const A a = slotsOf<N>(B);
    const bool first = B.in == nullptr;
    ListShare share(B.cnt + 1, first ? B.m : B.cnt[0]);
    if (share.idleBlock()) return;
    Tracer<N> T(S);
    T.useLdsTree(P);
    uint32_t nlk = 0;
    for (; share.more(); share.next()) {
        uint32_t li;
        const bool active = share.item(li);
        bool alive = false, edge = false;
        uint32_t slot = 0;
        if (active) {
            slot = first ? li : B.in[li];
            AdState<N> st;
            Rng r;
            Pusher u{q, qcount, 0, 0, 0, 0, 0, Pusher::NO_FAIL};
            uint64_t sid = B.s0 + slot;
            if (B.replay) {
                const uint4 e = B.replay[slot];
                sid = (uint64_t)e.x | ((uint64_t)e.y << 32);
                u.skip = e.z;
            }
            if (first) {
                u.view = viewOf(S, sid);
                const DView &vw = S.views[u.view];
                const uint64_t ls = sid - vw.s0;   // sample index within the view: keys its random stream
                const int pixel = (int)(ls / (uint64_t)vw.spp);
                u.gpix = vw.pix0 + pixel;
                u.key = (ls + 1) << 20;
                r.init(vw.seed, ls);
                alive = adBegin<N>(P, vw, r, pixel, st);
                a.u(A::PIX, slot) = (uint32_t)u.gpix;
                a.u(A::VIEW, slot) = (uint32_t)u.view;
                a.u(A::SKIP, slot) = u.skip;
            } else {
                u.gpix = (int)a.u(A::PIX, slot);
                u.view = (int)a.u(A::VIEW, slot);
                const DView &vw = S.views[u.view];
                const uint64_t ls = sid - vw.s0;
                u.key = (ls + 1) << 20;
                u.child = a.u(A::CHILD, slot);
                u.failed_at = a.u(A::FAILED, slot);
                a.ldRng(slot, vw.seed, ls, r);
                const uint32_t fl = a.u(A::FLAGS, slot);
                st.med = (int)(fl & 255u) - 1;
                st.depth = (int)(fl >> 8 & 255u);
                st.mode = (int)(fl >> 16 & 63u);
                st.walk = (int)(fl >> 22 & 3u);
                st.walk_surf = (fl >> 24 & 1u) != 0;
                st.walk_add = (fl >> 25 & 1u) != 0;
                st.walk_cpdf = a.r(A::CPDF, slot);
                st.hface = -1;
                st.ro = a.ldv(A::RO, slot);
                st.rd = fl & A::RD_CONST ? Dv<N>(a.ld(A::RD, slot)) : a.ldv(A::RD, slot);
                st.beta = a.lds(A::BETA, slot);
                alive = true;
            }
            Ds<N> L;
            if (alive) {
                AdEdgeOut<N> eo{a, slot, false};
                alive = adBounce<N>(T, P, r, st, L, u, stats, eo);
                edge = eo.set;
            }
            nlk += r.nlk;
            a.u(A::CHILD, slot) = u.child;
            a.u(A::FAILED, slot) = u.failed_at;
            if (alive || edge) a.stRng(slot, r);
            if (alive) {
                const bool rdc = st.rd.gradZero(0._r);
                a.u(A::FLAGS, slot) = (uint32_t)(st.med + 1) | (uint32_t)st.depth << 8 | (uint32_t)st.mode << 16 |
                                      (uint32_t)st.walk << 22 | (st.walk_surf ? 1u << 24 : 0u) | (st.walk_add ? 1u << 25 : 0u) |
                                      (rdc ? A::RD_CONST : 0u);
                a.r(A::CPDF, slot) = st.walk_cpdf;
                if (rdc) a.st(A::RD, slot, st.rd.val());
                else a.stv(A::RD, slot, st.rd);
                a.sts(A::BETA, slot, st.beta);
            }
            if (alive && !edge) a.stv(A::RO, slot, st.ro);   // an edge term has stored its vertex, the next ray's origin
            if (first) a.sts(A::L, slot, L);
            else a.sts(A::L, slot, a.lds(A::L, slot) + L);
        }
        appendSlots(alive, slot, B.out, B.cnt + 4);
        appendSlots(edge, slot, B.edges, B.cnt + 2);
    }
    flushWork(work, 0, T.nbox, T.ntri, nlk, T.nseg);
}

// The edge terms of one bounce. The random stream and the child count continue from the
// bounce's and are handed on to the next one.
template <int N>
__global__ __launch_bounds__(AD_STAGE_BLOCK, AD_EDGE_WAVES) void k_ad_edges(DScene S, RenderParams P, AdBatch B, char *q,
                                                                          unsigned *qcount, unsigned *stats,
                                                                          unsigned long long *work) {
    using A = AdSlots<N>;
    const A a = slotsOf<N>(B);
    ListShare share(B.cnt + 3, B.cnt[2]);
    if (share.idleBlock()) return;
    Tracer<N> T(S);
    T.useLdsTree(P);
    uint32_t nlk = 0;
    for (; share.more(); share.next()) {
        uint32_t li;
        if (share.item(li)) {
        const uint32_t slot = B.edges[li];
        uint64_t sid = B.s0 + slot;
        if (B.replay) {
            const uint4 e = B.replay[slot];
            sid = (uint64_t)e.x | ((uint64_t)e.y << 32);
        }
        const int view = (int)a.u(A::VIEW, slot);
        const DView &vw = S.views[view];
        const uint64_t ls = sid - vw.s0;
        Pusher u{q, qcount, (int)a.u(A::PIX, slot), view, (ls + 1) << 20, a.u(A::CHILD, slot), a.u(A::SKIP, slot),
                 a.u(A::FAILED, slot)};
        Rng r;
        a.ldRng(slot, vw.seed, ls, r);
        const uint32_t fl = a.u(A::EFLAGS, slot);
        const bool vol = (fl & 1u) != 0;
        const int depth = (int)(fl >> 1 & 255u), med = (int)(fl >> 9 & 255u) - 1;
        const Dv<N> x = a.ldv(A::RO, slot);
        Hit its0;
        const DBsdf *bp = nullptr;
        const DPhase *ph = nullptr;
        f3 rdin{0, 0, 0};
        if (vol) {
            ph = &S.phases[S.media[med].phase_id];
            rdin = a.ld(A::EWI, slot);
        } else {
            its0.face = (int)a.u(A::EFACE, slot);
            its0.p = x.val();
            its0.wi = a.ld(A::EWI, slot);
            its0.gn = a.ld(A::EGN, slot);
            its0.sn = a.ld(A::ESN, slot);
            bp = &bsdfOf(S, shapeOf(S, its0.face));
        }
        edgeTerm<N>(T, P, r, vol, x, &its0, bp, ph, rdin, a.ld(A::ETHR, slot), a.ld(A::EBETA, slot), med, depth, u, stats);
        nlk += r.nlk;
        a.stRng(slot, r);
        a.u(A::CHILD, slot) = u.child;
        a.u(A::FAILED, slot) = u.failed_at;
        }
    }
    flushWork(work, 0, T.nbox, T.ntri, nlk, T.nseg);
}

// The batch's radiance into acc: block row y = channel (value, then the lanes, of each
// colour), one thread per sample. A wave's runs of samples of one pixel are summed by
// shuffles and added with one atomic each (with one atomic per sample, 1M samples of
// 16 per pixel took 480 us instead of 40). Row 0 also lists the samples whose pushes
// overflowed the queue, which contribute nothing in this launch, in ovf.
template <int N>
__global__ __launch_bounds__(256) void k_ad_finish(RenderParams P, AdBatch B, real *acc, uint4 *ovf, unsigned *ovf_count) {
    using A = AdSlots<N>;
    const A a = slotsOf<N>(B);
    const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
    const int lane = threadIdx.x & 63;
    const bool active = slot < B.m;
    const int gpix = active ? (int)a.u(A::PIX, slot) : -1;
    const uint32_t failed_at = active ? a.u(A::FAILED, slot) : Pusher::NO_FAIL;
    const bool put = active && failed_at == Pusher::NO_FAIL;
    if (k == 0 && active && !put) {
        uint64_t sid = B.s0 + slot;
        if (B.replay) {
            const uint4 e = B.replay[slot];
            sid = (uint64_t)e.x | ((uint64_t)e.y << 32);
        }
        ovf[atomicAdd(ovf_count, 1u)] = make_uint4((uint32_t)sid, (uint32_t)(sid >> 32), failed_at, 0u);
    }
    real x = put ? a.r(A::L + k, slot) : 0._r;
    // head: the first lane of a run of equal pixels; after the loop it holds the run's sum
    const int before = __shfl_up(gpix, 1);
    const bool head = lane == 0 || before != gpix;
    const uint64_t heads = __ballot(head);
    const uint64_t above = lane == 63 ? 0 : heads >> (lane + 1);
    const int len = above ? __ffsll((unsigned long long)above) : 64 - lane;   // lanes to the run's end
    for (int off = 1; off < 64; off <<= 1) {
        const real y = __shfl_down(x, off);
        if (off < len) x += y;
    }
    if (head && active && x != 0._r) unsafeAtomicAdd(acc + ((size_t)(k / 3) * P.npix + gpix) * 3 + k % 3, x);
}
