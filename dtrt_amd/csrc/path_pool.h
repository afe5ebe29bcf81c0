// The primal volumetric path estimator (volpathAD.cpp:50-142; the Lins boundary samples of
// :338-441) over pools of paths: the sub-paths of the boundary terms, the samples of
// VolPathTracer, and single rays.
//
// Each wave owns POOL_PATHS paths, whose state lies in HBM, and runs one stage of the
// estimator at a time for up to 64 of the paths that wait for it:
//
//   FETCH   new paths from the source into free slots
//   TRACE   the closest hits of the waiting rays (all of them, a lane takes the next ray
//           as soon as it is done with one)
//   HIT     what a segment's hit means: blocked, a null crossing, a light, an end
//   TRACK   ratio tracking of a segment that lies in a medium
//   EVENT   free flight and the scattering event at its end: emission, light sample, next
//           direction
//   LINS1-3 the steps of a Lins sample before its primal continuation
//   DONE    the estimate to where it belongs, the slot free
//
// What bounds the estimator is the divergence of its paths: with one path per lane from
// bounce to bounce, 12 of 64 lanes were active in the average traversal step and 12 in a
// tracking loop. Here every stage starts with its lanes full as long as enough paths wait
// for it, at the price of reading and writing the part of the path state that it uses.
// Included by kernels.hip.
#pragma once

#ifndef POOL_PATHS
#define POOL_PATHS 128
#endif
constexpr int POOL_GROUPS = POOL_PATHS / 64;
static_assert(POOL_PATHS == POOL_SLOTS && POOL_GROUPS * 64 == POOL_PATHS && POOL_GROUPS <= 4, "a byte of a word per group");

enum PoolStage : uint32_t { PS_FREE = 0, PS_TRACE, PS_HIT, PS_TRACK, PS_EVENT, PS_LINS1, PS_LINS2, PS_LINS3, PS_DONE, PS_COUNT };

// State of the wave's paths, one row of POOL_PATHS values per field.
struct PoolState {
    real *f;
    uint32_t *w;
    // CO, CD: the ray being walked. P, RD: the event's position and its continuation. C, VMAX:
    // what the walk adds if it ends on its light with transmittance TT: TT * C, unless TT *
    // VMAX is below the walk's threshold. REM: distance left to a light sample.
    enum Real { CO = 0, CD = 3, P = 6, RD = 9, THR = 12, RET = 15, C = 18, VMAX = 21, TT, REM, CPDF, TMAX, REALS };
    enum Word { FLAGS = 0, WALK, NEXT, FACE, FIRST, K0, K1, S0, S1, BLK, POS, B0, B1, B2, B3, ITEM, WORDS };
    // FLAGS: 0 emitter walk (else shadow walk), 1 first hit only, 2 the segment starts
    // ShadowEpsilon off a surface, 3 contribution threshold 1e-12 (else Epsilon), 4 emission
    // at the next hit counts, 5-6 what follows the shadow walk (After), 7 the estimate is
    // weighted by the record's cw, 8-15 depth, 16-23 maximum depth, 24-25 Fate, 26 bit 2 of the
    // emitter walk that follows. WALK: 0-7 medium + 1, 8-15 medium + 1 after the event, 16-23
    // interfaces crossed, 24-31 the most allowed. NEXT: medium + 1 beyond the segment.
    enum : uint32_t { EMIT = 1, FIRST_ONLY = 2, OFF = 4, TINY = 8, INC = 16, AFTER = 5, CW = 128, OFF_NEXT = 1u << 26 };
    enum After : uint32_t { WALK_ON = 0, END = 1, TO_LINS2 = 2, TO_LINS3 = 3 };
    enum Fate : uint32_t { CROSS = 0, ADD = 1, NONE = 2 };
    DI real &r(int k, uint32_t s) const { return f[k * POOL_PATHS + s]; }
    DI uint32_t &u(int k, uint32_t s) const { return w[k * POOL_PATHS + s]; }
    DI f3 ld(int k, uint32_t s) const { return f3{r(k, s), r(k + 1, s), r(k + 2, s)}; }
    DI void st(int k, uint32_t s, f3 v) const { r(k, s) = v.x; r(k + 1, s) = v.y; r(k + 2, s) = v.z; }
    DI void initRng(uint32_t s, const Rng &g) const {
        u(K0, s) = g.k0; u(K1, s) = g.k1; u(S0, s) = g.s0; u(S1, s) = g.s1;
        stRng(s, g);
    }
    DI void ldRng(uint32_t s, Rng &g) const {
        g.nlk = 0;
        g.k0 = u(K0, s); g.k1 = u(K1, s); g.s0 = u(S0, s); g.s1 = u(S1, s);
        g.blk = u(BLK, s);
        g.pos = (int)u(POS, s);
        g.b0 = u(B0, s); g.b1 = u(B1, s); g.b2 = u(B2, s); g.b3 = u(B3, s);
    }
    DI void stRng(uint32_t s, const Rng &g) const {
        u(BLK, s) = g.blk;
        u(POS, s) = (uint32_t)g.pos;
        if (g.pos < 4) { u(B0, s) = g.b0; u(B1, s) = g.b1; u(B2, s) = g.b2; u(B3, s) = g.b3; }
    }
};
static_assert(PoolState::REALS == POOL_REALS && PoolState::WORDS == POOL_WORDS, "poolWaveBytes sizes this layout");

// One wave's pool. SRC: where paths come from and where their estimates go (see ChildSource).
template <int N, class SRC> struct PathPool {
    using PS = PoolState;
    Tracer<N> &T;
    const DScene &S;
    SRC &src;
    PoolState ps;
    uint16_t *list;    // LDS: slots of the stage being run
    uint8_t *stages;   // LDS: stage of every slot
    uint32_t nlk = 0;

    DI PathPool(Tracer<N> &T_, SRC &src_, char *state, uint16_t *list_, uint8_t *stages_)
        : T(T_), S(T_.S), src(src_), list(list_), stages(stages_) {
        ps.f = reinterpret_cast<real *>(state);
        ps.w = reinterpret_cast<uint32_t *>(ps.f + PS::REALS * POOL_PATHS);
    }
    DI static int lane() { return threadIdx.x & 63; }
    DI static void waveSync() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    DI static real maxAbs(f3 v) { return fmax(fabs(v.x), fmax(fabs(v.y), fabs(v.z))); }
    DI static uint32_t walkWord(int med, int pmed, int inter, int max_inter) {
        return (uint32_t)(med + 1) | (uint32_t)(pmed + 1) << 8 | (uint32_t)inter << 16 | (uint32_t)max_inter << 24;
    }

    // The emitter walk along (P, RD) that FLAGS describes.
    DI uint32_t startWalk(uint32_t s, uint32_t fl, uint32_t wk, f3 p, f3 rd) {
        ps.st(PS::CO, s, p);
        ps.st(PS::CD, s, rd);
        ps.r(PS::TT, s) = 1._r;
        ps.u(PS::FLAGS, s) = (fl & ~PS::OFF) | PS::EMIT | (fl & PS::OFF_NEXT ? PS::OFF : 0u);
        const uint32_t pm = wk >> 8 & 255u;
        ps.u(PS::WALK, s) = pm | pm << 8 | (wk & 0xFF000000u);
        return PS_TRACE;
    }
    // The walk has ended: what comes next.
    DI uint32_t endWalk(uint32_t s, uint32_t fl, uint32_t wk) {
        if (fl & PS::EMIT) return PS_EVENT;
        switch (fl >> PS::AFTER & 3u) {
            case PS::WALK_ON: return startWalk(s, fl, wk, ps.ld(PS::P, s), ps.ld(PS::RD, s));
            case PS::END: return PS_DONE;
            case PS::TO_LINS2: return PS_LINS2;
            default: return PS_LINS3;
        }
    }
    // A segment of length tmax is done with transmittance Tt: the walk goes on beyond its
    // null interface, or ends.
    DI uint32_t afterSegment(uint32_t s, uint32_t fl, uint32_t wk, uint32_t fate, f3 o, f3 d, real tmax, real Tt, uint32_t next) {
        if (fate == PS::CROSS) {
            bool on = true;
            if (!(fl & PS::EMIT)) {
                const real rem = ps.r(PS::REM, s) - tmax;
                ps.r(PS::REM, s) = rem;
                on = rem > 0._r;   // else the walk has reached its light
            }
            if (on) {
                ps.st(PS::CO, s, o + d * tmax);
                ps.r(PS::TT, s) = Tt;
                ps.u(PS::FLAGS, s) = fl | PS::OFF;
                ps.u(PS::WALK, s) = (wk & 0xFF00FF00u) | next | ((wk >> 16 & 255u) + 1u) << 16;
                return PS_TRACE;
            }
            fate = PS::ADD;
        }
        if (fate == PS::ADD && ps.r(PS::VMAX, s) * Tt > ((fl & PS::EMIT) && (fl & PS::TINY) ? 1e-12_r : EPS))
            ps.st(PS::RET, s, ps.ld(PS::RET, s) + ps.ld(PS::C, s) * Tt);
        return endWalk(s, fl, wk);
    }

    // TRACE: every listed ray (`count` of them). A lane that is done takes the next ray once
    // a quarter of the wave is idle, so that the setup runs for several lanes at a time.
    DI void trace(uint32_t count) {
        BvhWalk<treePrefixInLds<N>()> b(S.nodes, S.tris, S.nnodes, T.lds_nodes, T.lds_tris, S.stack_depth);
        uint32_t taken = 0, slot = 0;
        bool have = false;
        while (true) {
            const bool idle = !have || b.done();
            if (have && idle) {
                ps.u(PS::FACE, slot) = (uint32_t)b.face;
                stages[slot] = PS_HIT;
                have = false;
                T.nseg++;
            }
            const uint64_t im = __ballot(idle);
            if (taken < count) {
                if (im == ~0ull || __popcll(im) >= 16) {
                    const uint32_t k = taken + (uint32_t)__popcll(im & __lanemask_lt());
                    if (idle && k < count) {
                        slot = list[k];
                        const uint32_t fl = ps.u(PS::FLAGS, slot);
                        real tfar = FINF;
                        if (!(fl & PS::EMIT)) tfar = (1.0_r - SHADOW_EPS) * ps.r(PS::REM, slot);
                        b.start(ps.ld(PS::CO, slot), ps.ld(PS::CD, slot), fl & PS::OFF ? SHADOW_EPS : 0._r, tfar);
                        have = true;
                    }
                    taken += (uint32_t)__popcll(im);
                }
            } else if (im == ~0ull) {
                break;
            }
            if (have && !b.done()) b.advance();
        }
        T.nbox += b.nbox;
        T.ntri += b.ntri;
    }

    // HIT (scene.cpp:177-237 for shadow walks, :617-701 for emitter walks)
    DI uint32_t hit(uint32_t s) {
        const uint32_t fl = ps.u(PS::FLAGS, s), wk = ps.u(PS::WALK, s);
        const int face = (int)ps.u(PS::FACE, s), med = (int)(wk & 255u) - 1;
        const uint32_t inter = wk >> 16 & 255u, max_inter = wk >> 24;
        const bool emit = (fl & PS::EMIT) != 0;
        if (emit && inter == 0) ps.u(PS::FIRST, s) = (uint32_t)face;
        if (emit && (face < 0 || (fl & PS::FIRST_ONLY))) return endWalk(s, fl, wk);
        const f3 o = ps.ld(PS::CO, s), d = ps.ld(PS::CD, s);
        real tmax = emit ? 0._r : ps.r(PS::REM, s);
        uint32_t fate = PS::ADD, next = wk & 255u;
        if (face >= 0) {
            const DShape &sh = shapeOf(S, face);
            const bool pass = inter != max_inter && bsdfOf(S, sh).type == BSDF_NULL;
            if (!emit && !pass) return endWalk(s, fl, wk);   // blocked
            Hit nh;
            refineHit(S, face, o, d, nh);
            if (emit || nh.t < tmax) tmax = nh.t;
            if (emit && sh.light_id >= 0) {
                const f3 dv = nh.p - ps.ld(PS::P, s);
                const real G = nh.wi.z / dot(dv, dv);
                const real pdf = S.light_pmf[sh.light_id] / (S.light_areas[sh.light_id] * G);
                const f3 le = emitterEval(S.emitters[sh.light_id], nh.gn, nh.sn, -d);
                ps.st(PS::C, s, ps.ld(PS::THR, s) * le * misPower(ps.r(PS::CPDF, s), pdf));
                ps.r(PS::VMAX, s) = maxAbs(le);
            } else {
                fate = pass ? PS::CROSS : PS::NONE;
                if (pass && isTransition(sh)) next = (uint32_t)(targetMedium(sh, nh.gn, d) + 1);
            }
        }
        if (med >= 0) {
            ps.r(PS::TMAX, s) = tmax;
            ps.u(PS::NEXT, s) = next;
            ps.u(PS::FLAGS, s) = (fl & ~(3u << 24)) | fate << 24;
            return PS_TRACK;
        }
        return afterSegment(s, fl, wk, fate, o, d, tmax, ps.r(PS::TT, s), next);
    }

    // TRACK
    DI uint32_t track(uint32_t s) {
        const uint32_t fl = ps.u(PS::FLAGS, s), wk = ps.u(PS::WALK, s);
        const f3 o = ps.ld(PS::CO, s), d = ps.ld(PS::CD, s);
        const real tmax = ps.r(PS::TMAX, s);
        Rng r;
        ps.ldRng(s, r);
        const real Tt = ps.r(PS::TT, s) *
                        mediumTransmittance(S.media[(int)(wk & 255u) - 1], o, d, fl & PS::OFF ? SHADOW_EPS : 0._r, tmax, r);
        nlk += r.nlk;
        ps.stRng(s, r);
        return afterSegment(s, fl, wk, fl >> 24 & 3u, o, d, tmax, Tt, ps.u(PS::NEXT, s));
    }

    // The shadow walk of a light sample whose contribution is c, le / pdf at most vmax.
    DI uint32_t startShadow(uint32_t s, uint32_t fl, uint32_t wk, const typename Tracer<N>::Shadow &q, f3 c, real vmax) {
        ps.st(PS::CO, s, q.o);
        ps.st(PS::CD, s, q.d);
        ps.st(PS::C, s, c);
        ps.r(PS::VMAX, s) = vmax;
        ps.r(PS::REM, s) = q.dist;
        ps.r(PS::TT, s) = 1._r;
        ps.u(PS::FLAGS, s) = (fl & ~(PS::EMIT | PS::OFF)) | (q.on_surface ? PS::OFF : 0u);
        ps.u(PS::WALK, s) = (wk & 0x0000FF00u) | (uint32_t)(q.med + 1) | (uint32_t)q.max_inter << 24;
        return PS_TRACE;
    }

    // EVENT: one bounce of volpathAD.cpp:50-142 from the hit that the walk found
    DI uint32_t event(uint32_t s) {
        uint32_t fl = ps.u(PS::FLAGS, s);
        const int depth = (int)(fl >> 8 & 255u), max_depth = (int)(fl >> 16 & 255u), max_inter = max_depth - depth - 1;
        if (depth > max_depth) return PS_DONE;
        int med = (int)(ps.u(PS::WALK, s) >> 8 & 255u) - 1;
        f3 ro = ps.ld(PS::P, s);
        const f3 rd = ps.ld(PS::RD, s);
        f3 thr = ps.ld(PS::THR, s);
        Hit its;
        const int face = (int)ps.u(PS::FIRST, s);
        if (face >= 0) refineHit(S, face, ro, rd, its);
        Rng r;
        ps.ldRng(s, r);
        const real r1a = r.next(), r1b = r.next();
        const real r2[4] = {r.next(), r.next(), r.next(), r.next()};
        const real r3[3] = {r.next(), r.next(), r.next()};
        bool inside = false;
        if (med >= 0) {
            f3 pos;
            inside = sampleDistance(S.media[med], ro, rd, its.t, r1a, r1b, r, pos, thr);
            if (inside) ro = pos;
        }
        nlk += r.nlk;
        typename Tracer<N>::Shadow q;
        q.live = false;
        f3 wo, c{0, 0, 0};
        real cpdf = 0._r, pdf = 0._r;
        bool cont = true, first_only = false;
        const DPhase *ph = nullptr;
        if (inside) {
            if (depth >= max_depth || allZero(thr, EPS)) return PS_DONE;
            ph = &S.phases[S.media[med].phase_id];
            T.neePointSetup(ro, r2, med, max_inter, q);
        } else {
            if (its.face < 0) return PS_DONE;
            const DShape &sh = shapeOf(S, its.face);
            if (sh.light_id >= 0 && (fl & PS::INC))
                ps.st(PS::RET, s, ps.ld(PS::RET, s) + thr * emitterEval(S.emitters[sh.light_id], its.gn, its.sn, -rd));
            if (depth >= max_depth) return PS_DONE;
            first_only = bsdfOf(S, sh).type == BSDF_NULL;
            if (!first_only) T.neeSurfaceSetup(its, r2, med, max_inter, q);
        }
        const f3 le = T.neeFinish(q, 1._r, pdf);   // over its pdf
        if (inside) {
            if (q.live) {
                const real pv = phaseEval(*ph, -rd, q.d);
                if (pv > EPS) c = thr * le * (misPower(pdf, pv) * pv);
            }
            wo = phaseSample(*ph, -rd, r3[0], r3[1]);
            cpdf = phaseEval(*ph, -wo, wo);
        } else {
            const DShape &sh = shapeOf(S, its.face);
            const DBsdf &b = bsdfOf(S, sh);
            const Frame shf(its.sn);
            if (q.live) {
                const f3 wl = shf.toLocal(q.d);
                c = thr * le * bsdfEval(b, its.wi, wl) * misPower(pdf, bsdfPdf(b, its.wi, wl));
            }
            const f3 bw = bsdfSample(b, its.wi, r3[0], r3[1], r3[2], wo, cpdf);
            cont = !allZero(bw, EPS);
            if (cont) {
                wo = shf.toWorld(wo);
                ro = its.p;
                if (isTransition(sh)) med = targetMedium(sh, its.gn, wo);
                if (!first_only) thr = thr * bw;
            }
        }
        ps.stRng(s, r);
        if (!cont && !q.live) return PS_DONE;
        fl &= ~(PS::FIRST_ONLY | PS::TINY | PS::OFF_NEXT | 3u << PS::AFTER | 0xFF00u);
        fl |= (uint32_t)(depth + 1) << 8 | (first_only ? PS::FIRST_ONLY : 0u) | (inside ? 0u : PS::TINY | PS::OFF_NEXT) |
              (cont ? PS::WALK_ON : PS::END) << PS::AFTER;
        if (!first_only) fl &= ~PS::INC;
        const uint32_t wk = walkWord(-1, med, 0, max_inter);
        if (cont) {
            ps.st(PS::P, s, ro);
            ps.st(PS::RD, s, wo);
            ps.st(PS::THR, s, thr);
            ps.r(PS::CPDF, s) = cpdf;
        }
        if (q.live) return startShadow(s, fl, wk, q, c, maxAbs(le));
        return startWalk(s, fl, wk, ro, wo);
    }

    // The light sample at a Lins boundary hit (scene.cpp:456-491). flag: a sample on the other
    // side of the surface takes one interaction more.
    DI void linsLight(const Hit &its, const Frame &shf, const real *r4, int med, int max_inter, bool flag,
                      typename Tracer<N>::Shadow &q) {
        T.neeSurfaceSetup(its, r4, med, max_inter < 0 ? -1 : max_inter, q);
        if (q.live && flag && signum(its.wi.z) != signum(shf.toLocal(q.d).z) && --q.max_inter < 0) q.live = false;
    }
    // The boundary hit, the incoming direction and the medium of a Lins record.
    DI Hit linsHit(const ChildHdr &h, f3 &rdv) const {
        Hit its;
        its.face = h.face;
        its.p = f3{h.org[0], h.org[1], h.org[2]};
        its.gn = f3{h.gn[0], h.gn[1], h.gn[2]};
        its.sn = f3{h.sn[0], h.sn[1], h.sn[2]};
        rdv = f3{h.dir[0], h.dir[1], h.dir[2]};
        return its;
    }
    // LINS1 (volpathAD.cpp:338-370): the light sample at the boundary
    DI uint32_t lins1(uint32_t s) {
        const ChildHdr &h = src.record(ps.u(PS::ITEM, s));
        const bool null_bsdf = (h.meta & 3) == CHILD_LINS_NULL;
        const int max_depth = (h.meta >> 4) & 255, med = ((h.meta >> 12) & 255) - 1;
        f3 rdv;
        Hit its = linsHit(h, rdv);
        const Frame shf(its.sn);
        its.wi = shf.toLocal(-rdv);
        Rng r;
        ps.ldRng(s, r);
        const real r4[4] = {r.next(), r.next(), r.next(), r.next()};
        ps.stRng(s, r);
        typename Tracer<N>::Shadow q;
        linsLight(its, shf, r4, med, max_depth - 1, null_bsdf, q);
        if (!q.live) return PS_LINS2;
        real pdf = 0._r;
        const f3 le = T.neeFinish(q, 1._r, pdf), wo = shf.toWorld(shf.toLocal(q.d));
        const f3 n = dot(its.gn, rdv) < 0._r ? -its.gn : its.gn;
        const real pv = phaseEval(S.phases[S.media[med].phase_id], -rdv, wo);
        f3 c{0, 0, 0};
        if (pv > EPS && (null_bsdf || dot(wo, n) < -EPS)) c = le * (pv * misPower(pdf, pv));
        return startShadow(s, PS::TO_LINS2 << PS::AFTER, walkWord(-1, med, 0, 0), q, c, maxAbs(le));
    }
    // The primal continuation of a Lins sample along (p, wo).
    DI uint32_t linsContinue(uint32_t s, uint32_t fl, f3 p, f3 wo, int med, int max_depth, real cpdf) {
        ps.st(PS::P, s, p);
        ps.st(PS::RD, s, wo);
        ps.st(PS::THR, s, f3{1, 1, 1});
        ps.r(PS::CPDF, s) = cpdf;
        return startWalk(s, fl | PS::OFF_NEXT | (uint32_t)max_depth << 16, walkWord(med, med, 0, max_depth), p, wo);
    }
    // LINS2 (volpathAD.cpp:371-420): a direction from the phase function
    DI uint32_t lins2(uint32_t s) {
        const ChildHdr &h = src.record(ps.u(PS::ITEM, s));
        const bool null_bsdf = (h.meta & 3) == CHILD_LINS_NULL;
        const int max_depth = (h.meta >> 4) & 255, med = ((h.meta >> 12) & 255) - 1;
        f3 rdv;
        const Hit its = linsHit(h, rdv);
        const DShape &sh = shapeOf(S, its.face);
        const DPhase &ph = S.phases[S.media[med].phase_id];
        const f3 n = dot(its.gn, rdv) < 0._r ? -its.gn : its.gn;
        Rng r;
        ps.ldRng(s, r);
        const real u1 = r.next(), u2 = r.next();
        const f3 wo = phaseSample(ph, -rdv, u1, u2);
        const real wdn = dot(wo, n);
        const bool back = wdn > EPS;
        if (back && sh.light_id >= 0)
            ps.st(PS::RET, s, ps.ld(PS::RET, s) + emitterEval(S.emitters[sh.light_id], its.gn, its.sn, -wo));
        uint32_t to = PS_DONE;
        if (null_bsdf) {
            const int md1 = max_depth - (back ? 2 : 1);
            if (md1 > 0)
                to = linsContinue(s, 0u, its.p, wo, isTransition(sh) ? targetMedium(sh, its.gn, wo) : med, md1, phaseEval(ph, -rdv, wo));
        } else if (wdn < -EPS) {
            to = linsContinue(s, 0u, its.p, wo, med, max_depth - 1, phaseEval(ph, -rdv, wo));
        } else if (back && max_depth > 1) {
            const Frame shf(its.sn);
            Hit itsb = its;
            itsb.wi = shf.toLocal(-wo);
            const real r4[4] = {r.next(), r.next(), r.next(), r.next()};
            ps.st(PS::RD, s, wo);
            typename Tracer<N>::Shadow q;
            linsLight(itsb, shf, r4, med, max_depth - 2, false, q);
            to = PS_LINS3;
            if (q.live) {
                real pdf = 0._r;
                const f3 le = T.neeFinish(q, 1._r, pdf), wl = shf.toLocal(q.d);
                const DBsdf &b = bsdfOf(S, sh);
                const f3 c = bsdfEval(b, itsb.wi, wl) * le * misPower(pdf, bsdfPdf(b, itsb.wi, wl));
                to = startShadow(s, PS::TO_LINS3 << PS::AFTER, walkWord(-1, med, 0, 0), q, c, maxAbs(le));
            }
        }
        ps.stRng(s, r);
        return to;
    }
    // LINS3 (volpathAD.cpp:421-441): a direction from the BSDF at the boundary. The record
    // keeps what was added so far and the weight of the continuation (SRC::weigh).
    DI uint32_t lins3(uint32_t s) {
        ChildHdr &h = src.record(ps.u(PS::ITEM, s));
        const int max_depth = (h.meta >> 4) & 255, med = ((h.meta >> 12) & 255) - 1;
        f3 rdv, wl;
        Hit its = linsHit(h, rdv);
        const DShape &sh = shapeOf(S, its.face);
        const DBsdf &b = bsdfOf(S, sh);
        const Frame shf(its.sn);
        its.wi = shf.toLocal(-ps.ld(PS::RD, s));
        Rng r;
        ps.ldRng(s, r);
        const real q0 = r.next(), q1 = r.next(), q2 = r.next();
        ps.stRng(s, r);
        real bpdf = 0._r;
        const f3 bv = bsdfSample(b, its.wi, q0, q1, q2, wl, bpdf);
        if (allZero(bv, EPS)) return PS_DONE;
        const f3 wo = shf.toWorld(wl), pre = ps.ld(PS::RET, s);
        h.org[0] = pre.x; h.org[1] = pre.y; h.org[2] = pre.z;
        h.dir[0] = bv.x; h.dir[1] = bv.y; h.dir[2] = bv.z;
        ps.st(PS::RET, s, f3{0, 0, 0});
        return linsContinue(s, PS::CW | PS::TINY, its.p, wo, isTransition(sh) ? targetMedium(sh, its.gn, wo) : med, max_depth - 2, bpdf);
    }

    // Runs the pool until the source is used up and every path has ended.
    DI void run(uint32_t waves) {
        // paths in flight: fewer than the pool holds when the source has fewer for every wave
        const uint32_t share = (src.n + waves - 1) / waves;
        const uint32_t limit = share >= POOL_PATHS ? POOL_PATHS : share < 4 ? 4 : share, fetch = limit < 64 ? limit : 64;
        for (int g = 0; g < POOL_GROUPS; ++g) stages[lane() + 64 * g] = PS_FREE;
        waveSync();
        bool more = true;   // the source may have paths
        while (true) {
            uint32_t mine[POOL_GROUPS];
            for (int g = 0; g < POOL_GROUPS; ++g) mine[g] = stages[lane() + 64 * g];
            // the stage to run: one with a full wave of paths waiting, else rays, else new
            // paths, else whatever most paths wait for
            uint32_t cnt[PS_COUNT];
#pragma unroll
            for (uint32_t k = 0; k < PS_COUNT; ++k) {
                cnt[k] = 0;
                for (int g = 0; g < POOL_GROUPS; ++g) cnt[k] += (uint32_t)__popcll(__ballot(mine[g] == k));
            }
            uint32_t pick = PS_FREE, best = 0;
#pragma unroll
            for (uint32_t k = PS_HIT; k < PS_COUNT; ++k)
                if (cnt[k] > best) { best = cnt[k]; pick = k; }
            if (best < 64) {
                if (more && POOL_PATHS - cnt[PS_FREE] + fetch <= limit) pick = PS_FREE;
                else if (cnt[PS_TRACE] >= best) pick = PS_TRACE;
                if (pick == PS_TRACE && cnt[PS_TRACE] == 0) pick = PS_FREE;
                if (pick == PS_FREE && !more) break;   // nothing waits and nothing comes
            }
            // list the slots that wait for it
            uint32_t at = 0;
            for (int g = 0; g < POOL_GROUPS; ++g) {
                const uint64_t m = __ballot(mine[g] == pick);
                if (mine[g] == pick) list[at + (uint32_t)__popcll(m & __lanemask_lt())] = (uint16_t)(lane() + 64 * g);
                at += (uint32_t)__popcll(m);
            }
            waveSync();
            if (pick == PS_TRACE) {
                trace(at);
            } else {
                const uint32_t most = pick == PS_FREE ? fetch : 64, n = at < most ? at : most;
                bool on = lane() < (int)n;
                uint32_t slot = on ? list[lane()] : 0, to = PS_FREE;
                if (pick == PS_FREE) {
                    uint32_t item = 0;
                    more = src.take(on, item);
                    if (on) to = src.start(*this, slot, item);
                } else if (pick == PS_DONE) {
                    src.finish(*this, on, slot);
                } else if (on) {
                    switch (pick) {
                        case PS_HIT: to = hit(slot); break;
                        case PS_TRACK: to = track(slot); break;
                        case PS_EVENT: to = event(slot); break;
                        case PS_LINS1: if constexpr (SRC::LINS) to = lins1(slot); break;
                        case PS_LINS2: if constexpr (SRC::LINS) to = lins2(slot); break;
                        case PS_LINS3: if constexpr (SRC::LINS) to = lins3(slot); break;
                        default: break;
                    }
                }
                if (on) stages[slot] = (uint8_t)to;
            }
            waveSync();
        }
    }
    // A new path: ray, random stream, depth, medium; off: the ray starts on a surface.
    DI uint32_t begin(uint32_t s, uint32_t item, const Rng &r, f3 o, f3 d, int max_depth, int med, bool off) {
        ps.initRng(s, r);
        ps.u(PS::ITEM, s) = item;
        ps.st(PS::P, s, o);
        ps.st(PS::RD, s, d);
        ps.st(PS::THR, s, f3{1, 1, 1});
        ps.st(PS::RET, s, f3{0, 0, 0});
        return startWalk(s, PS::FIRST_ONLY | PS::INC | (uint32_t)max_depth << 16 | (off ? PS::OFF_NEXT : 0u), walkWord(med, med, 0, 0),
                         o, d);
    }
    DI f3 estimate(uint32_t s) const { return ps.ld(PS::RET, s); }
    DI bool weighted(uint32_t s) const { return (ps.u(PS::FLAGS, s) & PS::CW) != 0; }
};

// Takes the next item of a list of n for every lane with `on` (one atomic per wave); clears
// `on` where there is none. False once the list is used up.
DI bool takeItems(uint32_t *next, uint32_t n, bool &on, uint32_t &item) {
    const uint64_t m = __ballot(on);
    uint32_t base = 0;
    if ((threadIdx.x & 63) == 0) base = atomicAdd(next, (uint32_t)__popcll(m));
    base = __shfl(base, 0);
    item = base + (uint32_t)__popcll(m & __lanemask_lt());
    on = on && item < n;
    return base + (uint32_t)__popcll(m) < n;
}

// The child records of the queue; estimates go, with the records' weights, into acc.
template <int N> struct ChildSource {
    static constexpr bool LINS = true;
    const DScene &S;
    const RenderParams &P;
    char *q;
    uint32_t n;
    uint32_t *next;
    real *acc, *acc_pe;
    DI ChildHdr &record(uint32_t item) const { return *reinterpret_cast<ChildHdr *>(q + (size_t)item * P.rec_stride); }
    DI bool take(bool &on, uint32_t &item) { return takeItems(next, n, on, item); }
    template <class POOL> DI uint32_t start(POOL &p, uint32_t s, uint32_t item) {
        const ChildHdr h = record(item);
        Rng r;
        r.init(S.views[h.view].seed ^ 0x6a09e667f3bcc909ull, ((uint64_t)h.key_hi << 32) | h.key_lo);
        const uint32_t to = p.begin(s, item, r, f3{h.org[0], h.org[1], h.org[2]}, f3{h.dir[0], h.dir[1], h.dir[2]}, (h.meta >> 4) & 255,
                                    ((h.meta >> 12) & 255) - 1, true);
        if ((h.meta & 3) == CHILD_LI) return to;
        p.ps.u(PoolState::FLAGS, s) = 0u;
        return PS_LINS1;
    }
    template <class POOL> DI void finish(POOL &p, bool on, uint32_t s) {
        f3 L{0, 0, 0};
        uint32_t item = 0;
        if (on) {
            item = p.ps.u(PoolState::ITEM, s);
            L = p.estimate(s);
            if (p.weighted(s)) {
                const ChildHdr &h = record(item);
                L = f3{h.org[0], h.org[1], h.org[2]} + f3{h.dir[0], h.dir[1], h.dir[2]} * L;
            }
        }
        scatterFinished<N>(P, q, acc, acc_pe, on, item, L);
    }
};

// VolPathTracer's samples s0 .. s0+n-1 of view 0: sums into acc[pixel][3].
struct PrimalSource {
    static constexpr bool LINS = false;
    const DScene &S;
    const RenderParams &P;
    uint64_t s0;
    uint32_t n;
    uint32_t *next;
    real *acc;
    DI ChildHdr &record(uint32_t) const { return *(ChildHdr *)nullptr; }   // never asked for
    DI bool take(bool &on, uint32_t &item) { return takeItems(next, n, on, item); }
    template <class POOL> DI uint32_t start(POOL &p, uint32_t s, uint32_t item) {
        const DView &vw = S.views[0];
        const DCamera &cam = vw.cam;
        const uint64_t ls = s0 + item;
        const int pixel = (int)(ls / (uint64_t)vw.spp);
        Rng r;
        r.init(vw.seed, ls);
        const int ix = cam.cropped ? cam.ox + pixel % cam.cw : pixel % cam.width;
        const int iy = cam.cropped ? cam.oy + pixel / cam.cw : pixel / cam.width;
        const real jx = r.next(), jy = r.next();
        f3 ro, rd;
        cameraRay(cam, ix + jx, iy + jy, ro, rd);
        return p.begin(s, (uint32_t)pixel, r, ro, rd, P.max_bounces, cam.med_id, false);
    }
    template <class POOL> DI void finish(POOL &p, bool on, uint32_t s) {
        // runs of one pixel in lane order (slots are listed in order, samples start in order)
        const int lane = threadIdx.x & 63;
        const int pixel = on ? (int)p.ps.u(PoolState::ITEM, s) : -1;
        f3 L = on ? p.estimate(s) : f3{0, 0, 0};
        const int before = __shfl_up(pixel, 1);
        const bool head = lane == 0 || before != pixel;
        const uint64_t heads = __ballot(head), above = lane == 63 ? 0 : heads >> (lane + 1);
        const int len = above ? __ffsll((unsigned long long)above) : 64 - lane;
        for (int off = 1; off < 64; off <<= 1) {
            const f3 y{__shfl_down(L.x, off), __shfl_down(L.y, off), __shfl_down(L.z, off)};
            if (off < len) L = L + y;
        }
        if (head && on) {
            if (L.x != 0._r) unsafeAtomicAdd(acc + (size_t)pixel * 3, L.x);
            if (L.y != 0._r) unsafeAtomicAdd(acc + (size_t)pixel * 3 + 1, L.y);
            if (L.z != 0._r) unsafeAtomicAdd(acc + (size_t)pixel * 3 + 2, L.z);
        }
    }
};

// Rays {o, d}, stream = ray index: estimates into out[ray][3] (a test hook).
struct RaySource {
    static constexpr bool LINS = false;
    const float *rays;
    uint32_t n;
    uint32_t *next;
    int depth, med;
    uint64_t seed;
    float *out;
    DI ChildHdr &record(uint32_t) const { return *(ChildHdr *)nullptr; }   // never asked for
    DI bool take(bool &on, uint32_t &item) { return takeItems(next, n, on, item); }
    template <class POOL> DI uint32_t start(POOL &p, uint32_t s, uint32_t item) {
        const float *r6 = rays + (size_t)item * 6;
        Rng r;
        r.init(seed, (uint64_t)item);
        return p.begin(s, item, r, f3{r6[0], r6[1], r6[2]}, f3{r6[3], r6[4], r6[5]}, depth, med, true);
    }
    template <class POOL> DI void finish(POOL &p, bool on, uint32_t s) {
        if (!on) return;
        const f3 L = p.estimate(s);
        float *o = out + 3 * (size_t)p.ps.u(PoolState::ITEM, s);
        o[0] = (float)L.x; o[1] = (float)L.y; o[2] = (float)L.z;
    }
};

// The wave's share of the pool memory and its lists, then the pool until it is empty.
template <int N, class SRC>
DI void runPool(Tracer<N> &T, const RenderParams &P, SRC &src, uint32_t &nlk) {
    __shared__ uint16_t lists[POOL_BLOCK / 64][POOL_PATHS];
    __shared__ uint8_t stages[POOL_BLOCK / 64][POOL_PATHS];
    const int wv = threadIdx.x / 64;
    const size_t wave = (size_t)blockIdx.x * (POOL_BLOCK / 64) + wv;
    PathPool<N, SRC> pool(T, src, P.pool + wave * poolWaveBytes(kF64), lists[wv], stages[wv]);
    pool.run(gridDim.x * (POOL_BLOCK / 64));
    nlk += pool.nlk;
}

template <int N>
__global__ __launch_bounds__(POOL_BLOCK, POOL_WAVES) void k_children(DScene S, RenderParams P, char *q, const unsigned *qcount,
                                                                    unsigned *qnext, real *acc, real *acc_pe,
                                                                    unsigned long long *work) {
    Tracer<N> T(S);
    T.useLdsTree(P);
    uint32_t nlk = 0;
    ChildSource<N> src{S, P, q, min(*qcount, P.qcap), qnext, acc, acc_pe};
    runPool<N>(T, P, src, nlk);
    flushWork(work, 4, T.nbox, T.ntri, nlk, T.nseg);
}
