// VolPathTracerAD samples in stages: the paths of a batch of samples advance one bounce
// per launch, with their state in HBM between launches.
//
//  k_ad_bounce<N>   one bounce (adBounce) of every path still alive, the continuation walk
//                   that the last bounce handed over first; the first launch of a batch
//                   starts the samples at their camera rays
//  k_ad_edges<N>    the edge term (edgeTerm) of the bounces that have one
//  k_ad_tail<N>     the paths of a list too short to fill the chip, from where they are to
//                   their ends
//  k_ad_finish<N>   the samples' radiance into the accumulators, the samples whose pushes
//                   overflowed the queue into the replay list
//  k_adj_list<1>, k_adj_bounce<1>
//                   the density adjoint: which samples take part, and the bounces of the
//                   replay that scatters the derivative of every contribution
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
    enum Word { PIX = 0, VIEW, FLAGS, MED, RBLK, RPOS, RB0, RB1, RB2, RB3, CHILD, SKIP, FAILED, EFLAGS, EFACE, WORDS };
    static constexpr size_t BYTES = REALS * sizeof(real) + WORDS * 4;
    static_assert(REALS == adSlotReals(N) && WORDS == AD_SLOT_WORDS, "adSlotBytes sizes this layout");
    // FLAGS: depth | mode << 8 | walk << 16, then these; rd has no tangents (none are stored)
    static constexpr uint32_t SURF = 1u << 18, ADD = 1u << 19, RD_CONST = 1u << 20;
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
    int start;                   // the bounce starts its paths at their camera rays
    const uint32_t *in;          // slots alive at the start of the bounce (nullptr: all m)
    uint32_t *out, *edges;       // slots alive after it; slots with an edge term
    uint32_t *cnt;               // AD_CNT words apart: length of in, consumed, length of edges, consumed, length of out
    uint32_t tail;               // lists of at most so many paths are k_ad_tail's
};
template <int N> DI AdSlots<N> slotsOf(const AdBatch &B) {
    AdSlots<N> a;
    a.n = B.n;
    a.f = reinterpret_cast<real *>(B.state);
    a.w = reinterpret_cast<uint32_t *>(a.f + (size_t)AdSlots<N>::REALS * B.n);
    return a;
}

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

// State of one AD path between bounces, but for its throughput and radiance, which stay in
// its slot until they are needed.
template <int N> struct AdState {
    Dv<N> ro, rd;
    int med, depth, mode;
    // The walk along (ro, rd) to run first: 1 first hit only from a surface, 2 emitter walk,
    // 3 the camera ray's first hit (from 0); walk_add: its emitter term counts, with MIS
    // partner pdf walk_cpdf.
    int walk;
    bool walk_surf, walk_add;
    real walk_cpdf;
};
// Passes over a path: FORWARD adds its radiance with tangents into its slot; SCATTER replays
// it from the same stream and adds the reverse-mode density derivative of every
// contribution into grad (AdjCtx).
enum class AdPass { FORWARD, SCATTER };
struct AdjCtx {
    double *grad;        // d loss / d node density of the grid of *pm (accumulated)
    const DMedium *pm;
    f3 adj;              // d loss / d pixel value of this sample (already / spp)
    f3 Ltot;             // the sample's radiance
};

// One bounce of the dual-number estimator LiAD (volpathAD.cpp:145-620) for the path of `slot`.
// alive, edge: what follows.
//
// The path carries only the face its ray (ro, rd) hits: the hit record with its tangents is
// recomputed from the face and the dual ray, by the same refinement that produced it
// (shape.cpp:210-252). The two kinds of event, a scattering in the medium
// (volpathAD.cpp:171-305) and a surface hit (:306-616), run the same steps in the same
// order: the light sample (NEE), the edge term, the continuation's walk to the next hit.
// Each is set up per kind and then runs once for both, so the lanes of a wave on either kind
// of event share one shadow walk, one edge term and one continuation walk. The edge term
// is left to k_ad_edges and the continuation's walk to the next launch.
//
// What bounds it is the size of a dual-number path, which spills. The draws of the light
// sample and of the continuation all come before the shadow walk's, so the continuation
// is sampled and stored before that walk, and throughput and radiance are read and
// written where they are used: the hit record, the throughput and the radiance are not
// live across it.
template <int N, AdPass A>
DI void adBounce(Tracer<N> &T, const RenderParams &P, const AdSlots<N> &a, uint32_t slot, Rng &r, AdState<N> &st, Pusher &u,
                 unsigned *stats, const AdjCtx *ac, bool &alive, bool &edge) {
    using AS = AdSlots<N>;
    const DScene &S = T.S;
    alive = edge = false;
    Dv<N> ro = st.ro;
    const Dv<N> &rd = st.rd;
    const int med = st.med, depth = st.depth, mode = st.mode;
    auto addL = [&](const Ds<N> &c) {
        if constexpr (A == AdPass::FORWARD) a.sts(AS::L, slot, a.lds(AS::L, slot) + c);
        else a.st(AS::L, slot, a.ld(AS::L, slot) + c.val());
    };
    int hface = -1;
    {   // the walk the last bounce handed over, or the camera ray's first hit
        real pdf_nee = 0._r;
        Rng rs;   // stream position before the walk (scatter pass only)
        if constexpr (A == AdPass::SCATTER) rs = r;
        const Ds<N> att = T.lookForEmitterAD(ro, rd, st.walk_surf, r, med, depth, hface, pdf_nee, nullptr, nullptr, nullptr,
                                             st.walk != 2);
        if (st.walk_add && !att.isZero(EPS)) {
            const Ds<N> c = a.lds(AS::BETA, slot) * (att * misPower(st.walk_cpdf, pdf_nee));
            addL(c);
            if constexpr (A == AdPass::SCATTER) {
                ScatterCtx sc{ac->grad, ac->pm, dot(ac->adj, c.val())};
                Rng r2 = rs;
                int f2;
                real pdf2;
                T.lookForEmitterAD(ro, rd, st.walk_surf, r2, med, depth, f2, pdf2, nullptr, nullptr, &sc);
            }
        }
        if (st.walk == 3 && hface < 0) return;
    }
    HitAD<N> its;
    if (hface >= 0) refineHitAD<N>(S, hface, ro, rd, its);
    else its.t = Df<N>(FINF);
    const real r1a = r.next(), r1b = r.next();
    const real r2[4] = {r.next(), r.next(), r.next(), r.next()};
    const real r3[3] = {r.next(), r.next(), r.next()};
    Ds<N> thr(f3{1, 1, 1});
    bool vol = false;
    if (med >= 0) {
        Dv<N> ps;
        ScatterCtx fs{nullptr, nullptr, 0._r};
        const ScatterCtx *fsp = nullptr;
        if constexpr (A == AdPass::SCATTER) {   // free flight weighs everything from here on
            fs = ScatterCtx{ac->grad, ac->pm, dot(ac->adj, ac->Ltot - a.ld(AS::L, slot))};
            fsp = &fs;
        }
        vol = sampleDistanceAD<N>(S.media[med], ro, rd, its.t, r1a, r1b, r, ps, thr, fsp);
        if (vol) ro = ps;
    }
    const f3 rdin = rd.val();
    typename Tracer<N>::ShadowAD q;
    q.live = false;
    Ds<N> f;                          // the light sample's weight but for its radiance and MIS weight
    real fpdf = 0._r;                 // its MIS partner pdf
    bool fadd = true, cont = false, first_only = false;
    f3 nd{0, 0, 0};                   // the continuation's direction (through a null surface: rd)
    real cpdf = 1._r;
    int med1 = med;
    Ds<N> beta = a.lds(AS::BETA, slot);
    if (vol) {
        if (depth == 0 || thr.isZero(EPS)) return;
        const DPhase &ph = S.phases[S.media[med].phase_id];
        if (mode & 8) T.neePointADSetup(ro, r2, med, depth - 1, q);   // volume NEE with tangents
        const Ds<N> bt = beta * thr;
        if (q.live) {
            const Df<N> pv = phaseEvalAD<N>(ph, -rd, q.d);
            fadd = pv.v > EPS;
            f = bt * pv;
            fpdf = phaseEval(ph, -rdin, q.d);
        }
        if (P.sppse > 0 && (mode & 32) && S.edges_valid) {   // volume edges (volpathAD.cpp:207-305)
            edge = true;
            a.st(AS::ETHR, slot, thr.val());
            a.st(AS::EBETA, slot, beta.val());
            a.st(AS::EWI, slot, rdin);
        }
        nd = phaseSample(ph, -rdin, r3[0], r3[1]);   // volpathAD.cpp:250-268
        const Df<N> pv = phaseSampleWeightAD<N>(ph, -rd, nd);
        cont = pv.v > EPS;
        if (cont) a.sts(AS::BETA, slot, bt * pv);
        cpdf = phaseEval(ph, -nd, nd);
    } else {
        if (its.face < 0 || thr.isZero(EPS)) return;
        const DShape &sh = shapeOf(S, its.face);
        if (isTransition(sh) && targetMedium(sh, its.gn.val(), -rdin) != med) {
            atomicAdd(stats + STAT_MED_INCONSISTENT, 1u);
            return;
        }
        if (sh.light_id >= 0 && (mode & 1)) addL(beta * (thr * emitterEvalAD<N>(S.emitters[sh.light_id], its, -rd)));
        if (depth == 0) return;
        const DBsdf &b = bsdfOf(S, sh);
        const bool isnull = b.type == BSDF_NULL;
        const Hit its0 = its.val();
        // Lins boundary term (volpathAD.cpp:321-467): queued as primal sub-paths
        if (A == AdPass::FORWARD && med >= 0 && !its.t.gradZero(EPS) && (mode & 16)) {
            int ns = min(max((int)(P.ddist * its.t.gradAbsMax()), 1), 100);
            f3 n = dot(its0.gn, rdin) < 0._r ? -its0.gn : its0.gn;
            f3 sgs = sigS(S.media[med], its0.p - n * SHADOW_EPS);
            f3 base = beta.val() * thr.val() * sgs * (1.0_r / ns);
            real W[N * 3];
#pragma unroll
            for (int j = 0; j < N; ++j) { W[3 * j] = base.x * its.t.d[j]; W[3 * j + 1] = base.y * its.t.d[j]; W[3 * j + 2] = base.z * its.t.d[j]; }
            ChildHdr h;
            h.org[0] = its0.p.x; h.org[1] = its0.p.y; h.org[2] = its0.p.z;
            h.dir[0] = rdin.x; h.dir[1] = rdin.y; h.dir[2] = rdin.z;
            h.meta = (isnull ? CHILD_LINS_NULL : CHILD_LINS_SURF) | (depth << 4) | ((med + 1) << 12);
            h.face = its0.face;
            h.gn[0] = its0.gn.x; h.gn[1] = its0.gn.y; h.gn[2] = its0.gn.z;
            h.sn[0] = its0.sn.x; h.sn[1] = its0.sn.y; h.sn[2] = its0.sn.z;
            for (int s = 0; s < ns; ++s) push(P, u, h, W, N * 3);
        }
        if (isBlackAD<N>(b)) return;   // no light or edge sample counts and no direction follows
        ro = its.p;
        if (isnull) {
            nd = rdin;   // toWorld(-wi) == incoming direction, tangents included (rd)
            cont = first_only = true;
            a.sts(AS::BETA, slot, beta * thr);
        } else {
            if (mode & 2) T.neeSurfaceADSetup(its, r2, med, depth - 1, q);   // surface NEE with tangents
            const Ds<N> bt = beta * thr;
            const FrameAD<N> shf(its.sn);
            if (q.live) {
                const Dv<N> woL = shf.toLocal(Dv<N>(q.d));
                f = bt * bsdfEvalAD<N>(b, its.wi, woL);
                fpdf = bsdfPdf(b, its0.wi, woL.val());
            }
            if (P.sppse > 0 && (mode & 4) && S.edges_valid) {   // interface edges (volpathAD.cpp:513-616)
                edge = true;
                a.st(AS::ETHR, slot, thr.val());
                a.st(AS::EBETA, slot, beta.val());
                a.u(AS::EFACE, slot) = (uint32_t)its0.face;
                a.st(AS::EWI, slot, its0.wi);
                a.st(AS::EGN, slot, its0.gn);
                a.st(AS::ESN, slot, its0.sn);
            }
            f3 wo0;   // bsdf.cpp:11-21; null.cpp:18-23
            const f3 w0 = bsdfSample(b, its0.wi, r3[0], r3[1], r3[2], wo0, cpdf);
            if (!allZero(w0, EPS) && cpdf > EPS) {
                nd = shf.val().toWorld(wo0);
                const Ds<N> bw = bsdfEvalAD<N>(b, its.wi, shf.toLocal(Dv<N>(nd))) * (1.0_r / cpdf);
                cont = !bw.isZero(EPS);
                if (cont) a.sts(AS::BETA, slot, bt * bw);
            }
        }
        if (cont) med1 = isTransition(sh) ? targetMedium(sh, its0.gn, nd) : med;
    }
    if (edge) a.u(AS::EFLAGS, slot) = (vol ? 1u : 0u) | (uint32_t)depth << 1 | (uint32_t)(med + 1) << 9;
    if (edge || cont) a.stv(AS::RO, slot, ro);   // the edge term's vertex and the next ray's origin
    if (cont) {
        const int mode1 = first_only ? mode : mode & ~1;
        const bool addc = !first_only && (mode & (vol ? 8 : 2)) != 0;
        const bool keep = first_only && !rd.gradZero(0._r);   // the direction's tangents go on
        if (keep) a.stv(AS::RD, slot, rd);
        else a.st(AS::RD, slot, nd);
        a.r(AS::CPDF, slot) = cpdf;
        a.u(AS::MED, slot) = (uint32_t)med1;
        a.u(AS::FLAGS, slot) = (uint32_t)(depth - 1) | (uint32_t)mode1 << 8 | (first_only ? 1u : 2u) << 16 |
                               (vol ? 0u : AS::SURF) | (addc ? AS::ADD : 0u) | (keep ? 0u : AS::RD_CONST);
        alive = mode1 != 0;
    }
    if (q.live) {   // one shadow walk for both kinds of event
        real pdf_nee = 0._r;
        Rng rs;   // stream position before the walk (scatter pass only)
        if constexpr (A == AdPass::SCATTER) rs = r;
        const Ds<N> value = T.neeWalkAD(q, r, pdf_nee);
        if (fadd && !value.isZero(EPS)) {
            const Ds<N> c = f * value * misPower(pdf_nee, fpdf);
            addL(c);
            if constexpr (A == AdPass::SCATTER) {   // the shadow walk weighs this term only
                ScatterCtx sc{ac->grad, ac->pm, dot(ac->adj, c.val())};
                Rng r2w = rs;
                real pdf2;
                T.neeWalkAD(q, r2w, pdf2, &sc);
            }
        }
    }
}

// The path of `slot` at the start of a bounce: its camera ray (start) or its stored state.
// False when it has nothing to do.
template <int N>
DI bool adLoad(const DScene &S, const RenderParams &P, const AdBatch &B, const AdSlots<N> &a, uint32_t slot, bool start, Rng &r,
               AdState<N> &st, Pusher &u) {
    using A = AdSlots<N>;
    uint64_t sid = B.s0 + slot;
    if (B.replay) {
        const uint4 e = B.replay[slot];
        sid = (uint64_t)e.x | ((uint64_t)e.y << 32);
        u.skip = e.z;
    }
    u.view = start ? viewOf(S, sid) : (int)a.u(A::VIEW, slot);
    const DView &vw = S.views[u.view];
    const uint64_t ls = sid - vw.s0;   // sample index within the view: keys its random stream
    u.key = (ls + 1) << 20;
    if (start) {
        const int pixel = (int)(ls / (uint64_t)vw.spp);
        u.gpix = vw.pix0 + pixel;
        a.u(A::PIX, slot) = (uint32_t)u.gpix;
        a.u(A::VIEW, slot) = (uint32_t)u.view;
        a.u(A::SKIP, slot) = u.skip;
        a.sts(A::BETA, slot, Ds<N>(f3{1, 1, 1}));
        a.sts(A::L, slot, Ds<N>());
        r.init(vw.seed, ls);
        adCameraRay<N>(vw, r, pixel, st.ro, st.rd);
        st.walk = 3;
        st.walk_surf = st.walk_add = false;
        st.walk_cpdf = 0._r;
        st.med = vw.cam.med_id;
        st.depth = P.max_bounces;
        st.mode = P.mode;
        return st.mode != 0;
    }
    u.gpix = (int)a.u(A::PIX, slot);
    u.child = a.u(A::CHILD, slot);
    u.failed_at = a.u(A::FAILED, slot);
    a.ldRng(slot, vw.seed, ls, r);
    const uint32_t fl = a.u(A::FLAGS, slot);
    st.med = (int)a.u(A::MED, slot);
    st.depth = (int)(fl & 255u);
    st.mode = (int)(fl >> 8 & (uint32_t)AD_MODES);
    st.walk = (int)(fl >> 16 & 3u);
    st.walk_surf = (fl & A::SURF) != 0;
    st.walk_add = (fl & A::ADD) != 0;
    st.walk_cpdf = a.r(A::CPDF, slot);
    st.ro = a.ldv(A::RO, slot);
    st.rd = fl & A::RD_CONST ? Dv<N>(a.ld(A::RD, slot)) : a.ldv(A::RD, slot);
    return true;
}

template <int N>
__global__ __launch_bounds__(AD_STAGE_BLOCK, AD_BOUNCE_WAVES) void k_ad_bounce(DScene S, RenderParams P, AdBatch B, char *q,
                                                                             unsigned *qcount, unsigned *stats,
                                                                             unsigned long long *work) {
    using A = AdSlots<N>;
    const A a = slotsOf<N>(B);
    const uint32_t n = B.in ? B.cnt[0] : B.m;
    if (n <= B.tail) return;
    ListShare share(B.cnt + AD_CNT, n);
    if (share.idleBlock()) return;
    Tracer<N> T(S);
    T.useLdsTree(P);
    uint32_t nlk = 0;
    for (; share.more(); share.next()) {
        uint32_t li, slot = 0;
        bool alive = false, edge = false;
        if (share.item(li)) {
            slot = B.in ? B.in[li] : li;
            AdState<N> st;
            Rng r;
            Pusher u{q, qcount, 0, 0, 0, 0, 0, Pusher::NO_FAIL};
            if (adLoad<N>(S, P, B, a, slot, B.start, r, st, u))
                adBounce<N, AdPass::FORWARD>(T, P, a, slot, r, st, u, stats, nullptr, alive, edge);
            nlk += r.nlk;
            a.u(A::CHILD, slot) = u.child;
            a.u(A::FAILED, slot) = u.failed_at;
            if (alive || edge) a.stRng(slot, r);
        }
        appendSlots(alive, slot, B.out, B.cnt + 4 * AD_CNT);
        appendSlots(edge, slot, B.edges, B.cnt + 2 * AD_CNT);
    }
    flushWork(work, 0, T.nbox, T.ntri, nlk, T.nseg);
}

// Path-replay adjoint of the density derivative of the interior terms: the host restricts the
// terms to emission, surface and volume interior (no edge or Lins sub-paths), so nothing is
// pushed. Pass 0 lists the samples whose pixel has a loss gradient (dimg, into EBETA as
// gradient / spp), pass 1 those of them that have radiance (L, into ETHR).
template <int N> __global__ __launch_bounds__(256) void k_adj_list(DScene S, AdBatch B, const float *dimg, int pass) {
    using A = AdSlots<N>;
    const A a = slotsOf<N>(B);
    const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
    bool put = false;
    if (slot < B.m) {
        if (pass == 0) {
            const uint64_t sid = B.s0 + slot;
            const DView &vw = S.views[viewOf(S, sid)];
            const size_t gp = (size_t)vw.pix0 + (size_t)((sid - vw.s0) / (uint64_t)vw.spp);   // pixel of the concatenated gradient images
            const f3 adj = ld3(dimg + 3 * gp) * (1.0_r / vw.spp);
            put = !allZero(adj, 0._r);
            a.st(A::EBETA, slot, adj);
        } else if (!allZero(a.ld(A::EBETA, slot), 0._r)) {
            const f3 Lt = a.ld(A::L, slot);
            put = !allZero(Lt, 0._r);
            a.st(A::ETHR, slot, Lt);
        }
    }
    // one append per block: waves' appends to one counter take about 11 ns each
    __shared__ uint32_t len[4], base;
    const uint64_t m = __ballot(put);
    if ((threadIdx.x & 63) == 0) len[threadIdx.x / 64] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) base = atomicAdd(B.cnt, len[0] + len[1] + len[2] + len[3]);
    __syncthreads();
    if (put) {
        uint32_t at = base + (uint32_t)__popcll(m & __lanemask_lt());
        for (unsigned k = 0; k < threadIdx.x / 64; ++k) at += len[k];
        B.out[at] = slot;
    }
}
// One bounce of the replay: like k_ad_bounce, adding d loss / d node density of medium pmed's
// grid into grad.
template <int N>
__global__ __launch_bounds__(AD_STAGE_BLOCK, AD_BOUNCE_WAVES) void k_adj_bounce(DScene S, RenderParams P, AdBatch B, double *grad,
                                                                              int pmed, unsigned *stats,
                                                                              unsigned long long *work) {
    using A = AdSlots<N>;
    const A a = slotsOf<N>(B);
    const uint32_t n = B.cnt[0];
    if (n <= B.tail) return;
    ListShare share(B.cnt + AD_CNT, n);
    if (share.idleBlock()) return;
    Tracer<N> T(S);
    T.useLdsTree(P);
    uint32_t nlk = 0;
    for (; share.more(); share.next()) {
        uint32_t li, slot = 0;
        bool alive = false, edge = false;
        if (share.item(li)) {
            slot = B.in[li];
            AdState<N> st;
            Rng r;
            Pusher u{nullptr, nullptr, 0, 0, 0, 0, 0, Pusher::NO_FAIL};
            const AdjCtx ac{grad, S.media + pmed, a.ld(A::EBETA, slot), a.ld(A::ETHR, slot)};
            if (adLoad<N>(S, P, B, a, slot, B.start, r, st, u))
                adBounce<N, AdPass::SCATTER>(T, P, a, slot, r, st, u, stats, &ac, alive, edge);
            nlk += r.nlk;
            if (alive) a.stRng(slot, r);
        }
        appendSlots(alive, slot, B.out, B.cnt + 4 * AD_CNT);
    }
    flushWork(work, 0, T.nbox, T.ntri, nlk, T.nseg);
}

// The edge term of the bounce that the path of `slot` has just made. The random stream and
// the child count continue from the bounce's and are handed on to the next one.
template <int N>
DI void adEdge(Tracer<N> &T, const RenderParams &P, const AdBatch &B, const AdSlots<N> &a, uint32_t slot, char *q, unsigned *qcount,
               unsigned *stats, uint32_t &nlk) {
    using A = AdSlots<N>;
    const DScene &S = T.S;
    uint64_t sid = B.s0 + slot;
    if (B.replay) {
        const uint4 e = B.replay[slot];
        sid = (uint64_t)e.x | ((uint64_t)e.y << 32);
    }
    const int view = (int)a.u(A::VIEW, slot);
    const DView &vw = S.views[view];
    const uint64_t ls = sid - vw.s0;
    Pusher u{q, qcount, (int)a.u(A::PIX, slot), view, (ls + 1) << 20, a.u(A::CHILD, slot), a.u(A::SKIP, slot), a.u(A::FAILED, slot)};
    Rng r;
    a.ldRng(slot, vw.seed, ls, r);
    const uint32_t fl = a.u(A::EFLAGS, slot);
    const bool vol = (fl & 1u) != 0;
    const int depth = (int)(fl >> 1 & 255u), med = (int)(fl >> 9) - 1;
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
// The edge terms of one bounce.
template <int N>
__global__ __launch_bounds__(AD_STAGE_BLOCK, AD_EDGE_WAVES) void k_ad_edges(DScene S, RenderParams P, AdBatch B, char *q,
                                                                          unsigned *qcount, unsigned *stats,
                                                                          unsigned long long *work) {
    const AdSlots<N> a = slotsOf<N>(B);
    ListShare share(B.cnt + 3 * AD_CNT, B.cnt[2 * AD_CNT]);
    if (share.idleBlock()) return;
    Tracer<N> T(S);
    T.useLdsTree(P);
    uint32_t nlk = 0;
    for (; share.more(); share.next()) {
        uint32_t li;
        if (share.item(li)) adEdge<N>(T, P, B, a, B.edges[li], q, qcount, stats, nlk);
    }
    flushWork(work, 0, T.nbox, T.ntri, nlk, T.nseg);
}

// The paths of the batch's short list, if it has one (at most B.tail paths), to their ends: a
// launch per bounce waits for the slowest path of every bounce, one launch for the slowest
// path. A bounce that finds its list so short leaves it, and all later lists are empty: it is the
// last one with any path. B.in, B.out: the lists of even and odd bounces; B.cnt: the
// counters of bounce 0; B.start: the list is the whole batch, and no bounce has run.
template <int N, AdPass A, bool EDGES>
__global__ __launch_bounds__(AD_STAGE_BLOCK, AD_TAIL_WAVES) void k_ad_tail(DScene S, RenderParams P, AdBatch B, char *q,
                                                                         unsigned *qcount, double *grad, int pmed,
                                                                         unsigned *stats, unsigned long long *work) {
    using AS = AdSlots<N>;
    const AS a = slotsOf<N>(B);
    uint32_t n = B.m;
    int at = 0;   // the list's bounce
    if (!B.start) {
        n = 0;
        const int lane = threadIdx.x & 63;
        for (int k0 = 0; k0 <= P.max_bounces; k0 += 64) {
            const uint32_t c = k0 + lane <= P.max_bounces ? B.cnt[4 * (k0 + lane) * AD_CNT] : 0;
            const uint64_t some = __ballot(c > 0);
            if (!some) continue;
            const int last = 63 - __clzll(some);
            at = k0 + last;
            n = __shfl(c, last);
        }
    }
    if (n > B.tail) return;
    ListShare share(B.cnt + 4 * (P.max_bounces + 2) * AD_CNT, n);
    if (share.idleBlock()) return;
    const uint32_t *list = B.start ? nullptr : at & 1 ? B.out : B.in;
    Tracer<N> T(S);
    T.useLdsTree(P);
    uint32_t nlk = 0;
    for (; share.more(); share.next()) {
        uint32_t li;
        if (!share.item(li)) continue;
        const uint32_t slot = list ? list[li] : li;
        bool alive = true, edge;
        for (bool start = at == 0; alive; start = false) {
            alive = edge = false;
            AdState<N> st;
            Rng r;
            Pusher u{q, qcount, 0, 0, 0, 0, 0, Pusher::NO_FAIL};
            const bool go = adLoad<N>(S, P, B, a, slot, start, r, st, u);
            if constexpr (A == AdPass::FORWARD) {
                if (go) adBounce<N, A>(T, P, a, slot, r, st, u, stats, nullptr, alive, edge);
                a.u(AS::CHILD, slot) = u.child;
                a.u(AS::FAILED, slot) = u.failed_at;
            } else {
                const AdjCtx ac{grad, S.media + pmed, a.ld(AS::EBETA, slot), a.ld(AS::ETHR, slot)};
                if (go) adBounce<N, A>(T, P, a, slot, r, st, u, stats, &ac, alive, edge);
            }
            nlk += r.nlk;
            if (alive || edge) a.stRng(slot, r);
            if constexpr (EDGES)
                if (edge) adEdge<N>(T, P, B, a, slot, q, qcount, stats, nlk);
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
