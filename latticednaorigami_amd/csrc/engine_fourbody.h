// engine_fourbody.h - FourBody binding potential on slot-indexed domains.
//
// JunctionBindingPotential (origami_potential.cpp:158-934): binding a
// complementary pair is scored by walking the chain neighbours of both
// partners, their partners and the crossover junctions they form.  The walk
// is the same sequence of checks as the reference, so the FP64 energy is
// accumulated in the same order.
//
// Three forms of it:
//   FbChecks   the wavefront engine's: the checks side by side, one per lane
//   FourBody   the walk itself for that engine, where a violation has ended
//              the sum early
//   Eng::fb_*  the general engine's walk
//
// FourBody<A> is a leaf evaluated on an access object A (a replica block in a
// workgroup's LDS), which provides
//   rec(s)      position, orientation, state and partner of domain slot s
//   stk(a, b)   stacking energy of the pair
//   ns, lmask, cyc, dtype
// Neighbour slots past a staple's end are slots of the chain's stride that
// hold no domain: their state is never OCC_BOUND, so eb() is false on them.
// Written as loops over candidate lists with one copy of every check: 30 KB of
// code in the sweep kernel, where inlining each check at its uses gave 195 KB,
// three times the instruction cache two CUs share.
#ifndef LDO_ENGINE_FOURBODY_H
#define LDO_ENGINE_FOURBODY_H

#include "engine.h"

// A domain as the walk reads it: position and the packed orientation (byte
// 0), state (byte 1) and partner (upper half) of DomRec.
struct FbRec {
    int x, y, z;
    uint32_t w;
    DEV int ore() const { return (int)(w & 0xFFu); }
    DEV int state() const { return (int)((w >> 8) & 0xFFu); }
    DEV int bound() const { return (int)w >> 16; }
};

// index of the unit vector (dx, dy, dz), 7 for any other vector
DEV int fb_dir(int dx, int dy, int dz) {
    int ax = dx < 0 ? -dx : dx, ay = dy < 0 ? -dy : dy, az = dz < 0 ? -dz : dz;
    int i = ay * 2 + az * 4 + (dx + dy + dz < 0 ? 1 : 0);
    return ax + ay + az == 1 ? i : 7;
}

// VectorThree::rotate_half (utility.cpp:68-85) on vector indices; an axis
// that is no unit vector leaves v as it is
DEV int fb_half_turn(int v, int axis) {
    return (axis == 7 || (v >> 1) == (axis >> 1)) ? v : (v ^ 1);
}

// VectorThree::rotate(axis, -1) (utility.cpp:102-142) on vector indices: the
// six images of each axis, three bits each
DEV int fb_minus_quarter_turn(int v, int axis) {
    if (axis == 7) {
        return v;
    }
    // about +x: y -> -z, z -> y; about +y: x -> -z, z -> x; about +z: x -> -y, y -> x
    constexpr uint32_t rows[3] = {
        0u | 1u << 3 | 5u << 6 | 4u << 9 | 2u << 12 | 3u << 15,
        5u | 4u << 3 | 2u << 6 | 3u << 9 | 0u << 12 | 1u << 15,
        3u | 2u << 3 | 0u << 6 | 1u << 9 | 4u << 12 | 5u << 15,
    };
    int a = axis >> 1;
    uint32_t row = a == 0 ? rows[0] : (a == 1 ? rows[1] : rows[2]);
    int r = (int)((row >> (3 * v)) & 7u);
    // the opposite axis turns the other way: the image is negated unless v
    // lies along the axis
    return ((axis & 1) && (v >> 1) != a) ? (r ^ 1) : r;
}

template <class A>
struct FourBody {
    const A& a;
    double e;
    int st;
    bool viol;

    DEV explicit FourBody(const A& acc) : a(acc), e(0), st(0), viol(false) {}

    // ------------------------------------------------------- chain walks
    DEV int cs(int s) const { return s < a.ns ? -1 : (s - a.ns) & ~a.lmask; }
    DEV int dom_of(int s) const { return s < a.ns ? s : ((s - a.ns) & a.lmask); }
    DEV int fwd(int s) const {
        if (s < 0) {
            return -1;
        }
        if (s < a.ns) {
            return s + 1 < a.ns ? s + 1 : (a.cyc ? 0 : -1);
        }
        return ((s - a.ns) & a.lmask) != a.lmask ? s + 1 : -1;
    }
    DEV int bwd(int s) const {
        if (s < 0) {
            return -1;
        }
        if (s < a.ns) {
            return s > 0 ? s - 1 : (a.cyc ? a.ns - 1 : -1);
        }
        return ((s - a.ns) & a.lmask) != 0 ? s - 1 : -1;
    }
    DEV int next(int s, int step) const { return step > 0 ? fwd(s) : bwd(s); }
    // the domain as far from v as v is from its chain neighbour u, on the
    // other side (Domain::operator+ with the difference of their indices,
    // which on a ring may be a whole turn less one)
    DEV int beyond(int v, int u) const {
        int n = dom_of(v) - dom_of(u);
        if (v < a.ns) {
            int t = v + n;
            if (a.cyc) {
                return t >= a.ns ? t - a.ns : (t < 0 ? t + a.ns : t);
            }
            return t >= 0 && t < a.ns ? t : -1;
        }
        return n > 0 ? fwd(v) : bwd(v);
    }
    DEV bool bound(const FbRec& r, int s) const { return s >= 0 && r.state() == OCC_BOUND; }
    // record of slot s (slot 0's where there is none; see bound())
    DEV FbRec rec(int s) const { return a.rec(s < 0 ? 0 : s); }
    DEV bool eb(int s) const { return s >= 0 && a.rec(s).state() == OCC_BOUND; }
    DEV int bd(int s) const { return a.rec(s).bound(); }

    // ------------------------------------------------------------ rules
    static DEV int dir(const FbRec& p, const FbRec& q) {
        return fb_dir(q.x - p.x, q.y - p.y, q.z - p.z);
    }
    // q - p equals r - q
    static DEV bool straight(const FbRec& p, const FbRec& q, const FbRec& r) {
        return q.x - p.x == r.x - q.x && q.y - p.y == r.y - q.y && q.z - p.z == r.z - q.z;
    }
    // check_twist_constraint (domain.cpp:33-40, 69-78)
    DEV bool twist_ok(const FbRec& p, int ndr, const FbRec& q) const {
        int r = a.dtype == 0 ? fb_half_turn(p.ore(), ndr) : fb_minus_quarter_turn(p.ore(), ndr);
        return r == q.ore();
    }
    // check_kink_constraint (domain.cpp:42-57, 80-97)
    DEV bool kink_ok(const FbRec& p, int ndr, const FbRec& q) const {
        int oa = p.ore(), ob = q.ore();
        if (ndr == (oa ^ 1)) {
            return false;
        }
        if (ndr == oa) {
            return a.dtype == 0 ? ob != (oa ^ 1) : (oa >> 1) != (ob >> 1);
        }
        return (ndr >> 1) != (ob >> 1);
    }
    // check_pair_stacked (origami_potential.cpp:70-83)
    DEV bool stacked(int s, const FbRec& rs, int t, const FbRec& rt) const {
        bool swap = dom_of(s) > dom_of(t);
        const FbRec& p = swap ? rt : rs;
        const FbRec& q = swap ? rs : rt;
        int ndr = dir(p, q);
        return (ndr >> 1) != (p.ore() >> 1) && twist_ok(p, ndr, q);
    }
    // doubly_contiguous (origami_potential.cpp:51-68)
    DEV bool doubly_contig(int s, const FbRec& rs, int t, const FbRec& rt) const {
        if (cs(s) != cs(t) || dom_of(t) != dom_of(s) + 1) {
            return false;
        }
        int bs = rs.bound(), bt = rt.bound();
        if (cs(bs) != cs(bt)) {
            return false;
        }
        int dd = dom_of(bt) - dom_of(bs);
        return dd == 1 || dd == -1;
    }

    // ------------------------------------------------------ energy terms
    DEV void single(int h2, int h3, const FbRec& r1, const FbRec& r2, const FbRec& r3) {
        if (dir(r1, r2) != r1.ore() && !straight(r1, r2, r3)) {
            e -= a.stk(h2, h3);
            st -= 1;
        }
    }
    DEV void twice(int h1, int h2, int h3, const FbRec& r1, const FbRec& r2, const FbRec& r3) {
        if (!straight(r1, r2, r3)) {
            e -= a.stk(h1, h2) / 2;
            e -= a.stk(h2, h3) / 2;
            st -= 1;
        }
    }

    // check_junction (origami_potential.cpp:419-462) with the stacking
    // penalty of check_junction_stacking_penalty (:85-127)
    DEV void junction(int j1, int j2, int j3, int j4, int k1, int k2) {
        if (dom_of(k1) > dom_of(k2)) {
            int t = k1;
            k1 = k2;
            k2 = t;
            t = j1;
            j1 = j4;
            j4 = t;
            t = j2;
            j2 = j3;
            j3 = t;
        }
        FbRec r1 = rec(j1), r2 = rec(j2), r3 = rec(j3), r4 = rec(j4);
        FbRec s1 = rec(k1), s2 = rec(k2);
        if (!(stacked(j1, r1, j2, r2) && stacked(j3, r3, j4, r4))) {
            return;
        }
        if (dir(s1, s2) != s1.ore()) {
            return; // no junction rule and no penalty away from the orientation
        }
        int n1 = dir(r1, r2), n3 = dir(r3, r4);
        // directions along increasing domain index
        n1 = n1 < 7 && dom_of(j1) > dom_of(j2) ? n1 ^ 1 : n1;
        n3 = n3 < 7 && dom_of(j3) > dom_of(j4) ? n3 ^ 1 : n3;
        // check_junction_constraint (domain.cpp:59-67, 99-118)
        if (a.dtype != 0 && !twist_ok(s1, n1, s2)) {
            viol = true;
            return;
        }
        if (n1 == n3) {
            e -= a.stk(j1, j2);
            e -= a.stk(j3, j4);
            st -= 2;
        }
        else if ((n1 >> 1) != (n3 >> 1)) {
            e -= a.stk(j1, j2) / 2;
            e -= a.stk(j3, j4) / 2;
            st -= 1;
        }
    }

    // The junction walks.  Each forms pairs (u, v) out of the pair's one end
    // and pairs (x, y) out of the other, at most three each, and checks the
    // junction of every combination in order; a candidate the reference does
    // not add is -1.
    //   BACKWARD  check_backward_single_junction (:654-748)
    //   FORWARD   check_forward_single_junction (:750-844)
    //   CENTRAL   check_central_single_junction (:846-934)
    //   CONTIG    check_doubly_contig_junction_pair (:359-417)
    enum { BACKWARD, FORWARD, CENTRAL, CONTIG };
    DEV void junctions(int mode, int p, int q) {
        int u0, v0, u1, v1, v2, x0 = 0, y0 = -1, x1 = 0, y1 = -1, y2 = -1;
        if (mode <= FORWARD) {
            // n: the end the walk leaves from, f: the other end
            int step = mode == BACKWARD ? -1 : 1;
            int n = mode == BACKWARD ? p : q, f = mode == BACKWARD ? q : p;
            int nb = bd(n), fb = bd(f);
            int out = next(n, step);
            FbRec ro = rec(out);
            int nf = fwd(nb), nr = bwd(nb);
            u0 = n;
            v0 = out;
            u1 = nb;
            v2 = -1;
            bool eo = bound(ro, out);
            if (mode == BACKWARD ? nf == fb : nr == fb) {
                v1 = mode == BACKWARD ? nr : nf;
            }
            else if (eo && ro.bound() == nr && eb(nr)) {
                v1 = nf;
            }
            else if (eo && ro.bound() == nf && eb(nf)) {
                v1 = nr;
            }
            else {
                v1 = nf;
                v2 = nr;
            }
        }
        else if (mode == CENTRAL) {
            int pb = bd(p), qb = bd(q);
            if (cs(pb) == cs(qb)) {
                int dd = dom_of(pb) - dom_of(qb);
                if (dd == 1 || dd == -1) {
                    return;
                }
            }
            u0 = p;
            v0 = bwd(p);
            u1 = pb;
            v1 = fwd(pb);
            v2 = bwd(pb);
            x0 = q;
            y0 = fwd(q);
            x1 = qb;
            y1 = fwd(qb);
            y2 = bwd(qb);
            FbRec r = rec(v0);
            if (bound(r, v0)) {
                v1 = v1 == r.bound() ? -1 : v1;
                v2 = v2 == r.bound() ? -1 : v2;
            }
            r = rec(y0);
            if (bound(r, y0)) {
                y1 = y1 == r.bound() ? -1 : y1;
                y2 = y2 == r.bound() ? -1 : y2;
            }
        }
        else {
            u0 = p;
            v0 = bwd(p);
            u1 = bd(p);
            v1 = fwd(u1);
            v2 = -1;
            x0 = q;
            y0 = fwd(q);
            x1 = bd(q);
            y1 = bwd(x1);
        }
#pragma unroll 1
        for (int i = 0; i < 3; i++) {
            int u = i == 0 ? u0 : u1;
            int v = i == 0 ? v0 : (i == 1 ? v1 : v2);
            FbRec rv = rec(v);
            if (!bound(rv, v)) {
                continue;
            }
            if (mode <= FORWARD) {
                if (stacked(v, rv, u, rec(u))) {
                    continue;
                }
                x0 = v;
                y0 = beyond(v, u);
                x1 = rv.bound();
                y1 = fwd(x1);
                y2 = bwd(x1);
                FbRec r = rec(y0);
                if (bound(r, y0)) {
                    y1 = y1 == r.bound() ? -1 : y1;
                    y2 = y2 == r.bound() ? -1 : y2;
                }
            }
#pragma unroll 1
            for (int j = 0; j < 3; j++) {
                int x = j == 0 ? x0 : x1;
                int y = j == 0 ? y0 : (j == 1 ? y1 : y2);
                if (!eb(y)) {
                    continue;
                }
                // BACKWARD: (y, x, p, q) over the kink (v, u); FORWARD:
                // (p, q, x, y) over (u, v); else (v, u, x, y) over (p, q)
                bool bk = mode == BACKWARD, fw = mode == FORWARD;
                junction(bk ? y : (fw ? p : v), bk ? x : (fw ? q : u), bk ? p : x, bk ? q : y,
                         bk ? v : (fw ? u : p), bk ? u : (fw ? v : q));
            }
        }
    }

    // check_backward_triplet_stacking_combos (:464-519)
    DEV void backward_triplets(int p, const FbRec& rp, int q, const FbRec& rq) {
        if (!stacked(p, rp, q, rq)) {
            return;
        }
        int h1 = bwd(p);
        FbRec r1 = rec(h1);
        if (bound(r1, h1)) {
            if (stacked(h1, r1, p, rp)) {
                if (doubly_contig(p, rp, q, rq) && doubly_contig(h1, r1, p, rp)) {
                    viol = viol || !straight(r1, rp, rq);
                    if (viol) {
                        return;
                    }
                }
                twice(h1, p, q, r1, rp, rq);
            }
            else {
                single(p, q, r1, rp, rq);
            }
        }
        int prev = h1;
        int pb = rp.bound();
        FbRec rb = rec(pb);
        h1 = fwd(pb);
        r1 = rec(h1);
        if (bound(r1, h1) && r1.bound() != prev && r1.bound() != q && stacked(pb, rb, h1, r1)) {
            twice(h1, p, q, r1, rp, rq);
        }
        h1 = bwd(pb);
        r1 = rec(h1);
        if (bound(r1, h1) && r1.bound() != prev && r1.bound() != q) {
            if (stacked(h1, r1, pb, rb)) {
                twice(h1, p, q, r1, rp, rq);
            }
            else {
                single(pb, q, r1, rb, rq);
            }
        }
    }

    // check_forward_triplet_stacking_combos (:521-585)
    DEV void forward_triplets(int p, const FbRec& rp, int q, const FbRec& rq) {
        bool first = stacked(p, rp, q, rq);
        int h3 = fwd(q);
        FbRec r3 = rec(h3);
        if (bound(r3, h3)) {
            bool second = stacked(q, rq, h3, r3);
            if (first && second) {
                if (doubly_contig(p, rp, q, rq) && doubly_contig(q, rq, h3, r3)) {
                    viol = viol || !straight(rp, rq, r3);
                    if (viol) {
                        return;
                    }
                }
                twice(p, q, h3, rp, rq, r3);
            }
            else if (second) {
                single(q, h3, rp, rq, r3);
            }
        }
        int nxt = h3;
        int qb = rq.bound();
        FbRec rb = rec(qb);
        h3 = fwd(qb);
        r3 = rec(h3);
        if (bound(r3, h3) && r3.bound() != nxt && r3.bound() != p && stacked(qb, rb, h3, r3)) {
            if (first) {
                twice(p, q, h3, rp, rq, r3);
            }
            else {
                single(q, h3, rp, rq, r3);
            }
        }
        h3 = bwd(qb);
        r3 = rec(h3);
        if (bound(r3, h3) && r3.bound() != nxt && r3.bound() != p) {
            if (stacked(h3, r3, qb, rb)) {
                if (first) {
                    twice(p, q, h3, rp, rq, r3);
                }
                else {
                    single(q, h3, rp, rq, r3);
                }
            }
            else if (first) {
                single(qb, p, r3, rb, rp);
            }
        }
    }

    // check_central_triplet_stacking_combos (:587-652); ip, in, jp and jn
    // are the chain neighbours of di and dj
    DEV void central_triplets(int di, int dj, const FbRec& ri, const FbRec& rj, int ip,
                              const FbRec& rip, int in, const FbRec& rin, int jp,
                              const FbRec& rjp, int jn, const FbRec& rjn) {
        bool eip = bound(rip, ip), ein = bound(rin, in), ejp = bound(rjp, jp), ejn = bound(rjn, jn);
        if (!(eip || ein) || !(ejp || ejn)) {
            return;
        }
        // the stacking of each neighbouring pair; every use below sits
        // behind the same eb() tests
        bool s_ip = eip && stacked(ip, rip, di, ri);
        bool s_in = ein && stacked(di, ri, in, rin);
        bool s_jp = ejp && stacked(jp, rjp, dj, rj);
        bool s_jn = ejn && stacked(dj, rj, jn, rjn);
        if (eip && !doubly_contig(ip, rip, di, ri)) {
            if (ejn && rjn.bound() != in && s_jn) {
                if (s_ip) {
                    twice(ip, di, jn, rip, ri, rjn);
                }
                else {
                    single(di, jn, rip, ri, rjn);
                }
            }
            if (ejp && rjp.bound() != ip) {
                if (s_ip) {
                    if (s_jp) {
                        twice(ip, di, jp, rip, ri, rjp);
                    }
                    else {
                        single(dj, ip, rjp, rj, rip);
                    }
                }
                else if (s_jp) {
                    single(di, jp, rip, ri, rjp);
                }
            }
        }
        if (ein && s_in && !doubly_contig(di, ri, in, rin)) {
            if (ejn && rjn.bound() != in && s_jn) {
                twice(jn, di, in, rjn, ri, rin);
            }
            if (ejp && rjp.bound() != ip) {
                if (s_jp) {
                    twice(jp, di, in, rjp, ri, rin);
                }
                else {
                    single(dj, in, rjp, rj, rin);
                }
            }
        }
    }

    // One pair (p, q) of contiguous bound domains around a domain of the new
    // pair: check_regular_pair_constraints (:288-320),
    // check_doubly_contig_helix_pair (:322-357) or
    // check_doubly_contig_junction_pair (:359-417).  i: the pair ends (-1)
    // or starts (0) at that domain; second: it is the second partner, whose
    // doubly contiguous pairs the first has scored.
    DEV void pair(int p, const FbRec& rp, int q, const FbRec& rq, int i, bool second) {
        int pb = rp.bound(), qb = rq.bound();
        int dd = cs(pb) == cs(qb) ? dom_of(qb) - dom_of(pb) : 0;
        bool helix = dd == 1, contig = dd == -1;
        int ndr = dir(rp, rq);
        if (contig) {
            if (ndr != rp.ore()) {
                viol = true;
                return;
            }
            if (second) {
                return;
            }
            junctions(CONTIG, p, q);
            return;
        }
        int mode = i == -1 ? BACKWARD : FORWARD;
        if (helix) {
            if (second) {
                return;
            }
            if ((ndr >> 1) == (rp.ore() >> 1) || !twist_ok(rp, ndr, rq)) {
                viol = true;
                return;
            }
        }
        else {
            if (!kink_ok(rp, ndr, rq)) {
                viol = true;
                return;
            }
            if (!stacked(p, rp, q, rq)) {
                mode = CENTRAL;
            }
        }
        if (mode != CENTRAL) {
            e += a.stk(p, q);
            st += 1;
        }
        // a regular pair's junctions come before its triplets, a helix
        // pair's after
#pragma unroll 1
        for (int k = 0; k < 2; k++) {
            if ((k == 0) != helix) {
                junctions(mode, p, q);
            }
            else if (i == -1) {
                backward_triplets(p, rp, q, rq);
            }
            else {
                forward_triplets(p, rp, q, rq);
            }
        }
    }

    // calc_stacking_and_steric_terms (:212-229) with check_constraints
    // (:231-286) around each of the two domains
    DEV void terms(int di, int dj) {
        int ip = bwd(di), in = fwd(di), jp = bwd(dj), jn = fwd(dj);
        FbRec ri = rec(di), rj = rec(dj);
        FbRec rip = rec(ip), rin = rec(in), rjp = rec(jp), rjn = rec(jn);
#pragma unroll 1
        for (int j = 0; j < 2; j++) {
            int cd = j ? dj : di, pv = j ? jp : ip, nx = j ? jn : in;
            FbRec rc = j ? rj : ri, rpv = j ? rjp : rip, rnx = j ? rjn : rin;
            bool epv = bound(rpv, pv), enx = bound(rnx, nx);
#pragma unroll 1
            for (int i = -1; i <= 0; i++) {
                if (i == -1 ? epv : enx) {
                    bool b = i == -1;
                    pair(b ? pv : cd, b ? rpv : rc, b ? cd : nx, b ? rc : rnx, i, j == 1);
                    if (viol) {
                        return;
                    }
                }
            }
            if (epv && enx && stacked(cd, rc, nx, rnx)) {
                if (stacked(pv, rpv, cd, rc)) {
                    if (doubly_contig(pv, rpv, cd, rc) && doubly_contig(cd, rc, nx, rnx) &&
                        !straight(rpv, rc, rnx)) {
                        viol = true;
                        return;
                    }
                    twice(pv, cd, nx, rpv, rc, rnx);
                }
                else {
                    single(cd, nx, rpv, rc, rnx);
                }
            }
        }
        central_triplets(di, dj, ri, rj, ip, rip, in, rin, jp, rjp, jn, rjn);
    }
};

// The walk as 60 independent checks, one per lane of a wavefront.  The walk's
// checks read records and add to a sum; none depends on another's result, so
// they can be made side by side and their terms added in the walk's order
// (in_order).  Check c = 16 b + t belongs to pair b of contiguous domains (the
// pair ending at di, the pair starting at di, then dj's):
//   t = 0       the pair itself
//   t = 1..9    its junctions, outer candidate (t - 1) / 3, inner (t - 1) % 3
//   t = 10..12  its triplets
//   t = 13      (pairs ending at a domain) the triplet around the domain
//   t = 14      central triplet b
// A violated check ends the walk early; its partial sum then is the walk's
// alone (FourBody::terms), and only the violation is told here.
//
// Lanes of every kind run the same instructions with their results selected,
// so a check has no branch of its own; the wavefront leaves out the junctions
// when no lane has a candidate for one.  Positions are folded into one word
// (x + 2^10 y + 2^20 z, modulo 2^32): the difference of two folded positions is
// the folded unit vector between chain neighbours that lie side by side.  Placed
// neighbours always do.  A trial may put a domain at a site that is not next to
// its placed neighbour; its differences are no folded unit vectors (or look like
// other ones, more than 1000 sites away), and its verdict and energy mean
// nothing: the caller takes no such site, because no walk remains from it.  HALF: HalfTurn domains, whose twist rule is that contiguous
// domains off the orientation's axis point in opposite directions.  ONE: every
// pair has the same stacking energy, so a term's pairs are not told.
struct FbTerm {
    int op;         // 0 none; 1 + s1; 2 - s1; 3 - s1/2 - s2/2; 4 - s1 - s2
    int viol;
    int helix;      // (t = 0) a helix pair: triplets come before junctions
    int a1, b1, a2, b2; // s1 and s2 are the stacking energies of these pairs
};

// a domain as a check reads it: folded position, DomRec's packed word
struct FbWord {
    uint32_t c;
    uint32_t w;
    DEV int ore() const { return (int)(w & 0xFFu); }
    DEV int partner() const { return (int)w >> 16; }
    DEV bool is_bound() const { return (w & 0xFF00u) == (uint32_t)OCC_BOUND << 8; }
};
DEV uint32_t fb_fold(int x, int y, int z) {
    return (uint32_t)x + ((uint32_t)y << 10) + ((uint32_t)z << 20);
}
// from p to q
DEV int fb_diff(const FbWord& q, const FbWord& p) { return (int)(q.c - p.c); }
DEV int fb_neg(int d) { return (int)(0u - (uint32_t)d); }
// the axis of vector index o as a folded unit vector, and the vector itself
DEV int fb_axis(int o) { return 1 << (5 * (o & 6)); }
DEV int fb_vector(int o) { return (o & 1) ? -fb_axis(o) : fb_axis(o); }
// index of a folded unit vector
DEV int fb_index(int d) {
    int m = d < 0 ? fb_neg(d) : d;
    return 2 * (m > 1) + 2 * (m > 1024) + (d < 0);
}

template <class A, bool HALF, bool ONE>
struct FbChecks {
    const A& a; // rec(s) as a record, ns, lmask, cyc
    DEV explicit FbChecks(const A& acc) : a(acc) {}

    // chain neighbour of s, after it (up = 1) or before it (0); -1 for none
    DEV int step(int s, int up) const {
        int r = s - a.ns;
        bool sc = r < 0;
        // the last slot of the chain that way, as an offset from ns
        int end = sc ? (up ? -1 : -a.ns) : (up ? r | a.lmask : r & ~a.lmask);
        int ring = a.cyc ? (up ? 0 : a.ns - 1) : -1;
        int past = sc ? ring : -1;
        int next = s + 2 * up - 1;
        return (r == end ? past : next) | (s >> 31);
    }
    DEV int fwd(int s) const { return step(s, 1); }
    DEV int bwd(int s) const { return step(s, 0); }
    // slots a and b are neighbours of one chain, b = a +- 1
    DEV bool adjacent(int x, int y) const {
        int d = x - y, hi = x > y ? x : y;
        return ((d == 1) | (d == -1)) & ((hi < a.ns) | (((hi - a.ns) & a.lmask) != 0));
    }
    DEV FbWord rec(int s) const {
        FbRec r = a.rec(s < 0 ? 0 : s);
        return FbWord {fb_fold(r.x, r.y, r.z), r.w};
    }
    static DEV bool bound(const FbWord& r, int s) { return (s >= 0) & r.is_bound(); }
    static DEV FbWord pick(bool c, const FbWord& x, const FbWord& y) {
        return FbWord {c ? x.c : y.c, c ? x.w : y.w};
    }
    // check_twist_constraint along d off p's axis
    static DEV bool twist_ok(const FbWord& p, int d, const FbWord& q) {
        if (HALF) {
            return (p.ore() ^ q.ore()) == 1;
        }
        return fb_minus_quarter_turn(p.ore(), fb_index(d)) == q.ore();
    }
    // check_pair_stacked of chain neighbours s and t
    static DEV bool stacked(int s, const FbWord& rs, int t, const FbWord& rt) {
        bool up = s < t;
        FbWord p = HALF ? rs : pick(up, rs, rt), q = HALF ? rt : pick(up, rt, rs);
        int d = fb_diff(q, p), m = d < 0 ? fb_neg(d) : d;
        return (m != fb_axis(p.ore())) & twist_ok(p, d, q);
    }

    // `any(b)`: whether b holds for any check of the wavefront
    template <class Any>
    DEV FbTerm check(int c, int di, int dj, Any any) const {
        FbTerm out {0, 0, 0, 0, 0, 0, 0};
        int b = c >> 4, t = c & 15;
        int back = 1 - (b & 1), second = b >> 1;
        bool is_j = (unsigned)(t - 1) < 9u, is_t = (unsigned)(t - 10) < 3u;
        bool is_tail = (t == 13) & (back != 0), is_c = t == 14;
        int cd = second ? dj : di;
        // a central triplet's neighbours of di and dj stand for p and q
        int near = step(is_c ? di : cd, is_c ? second : 1 - back);
        int cb = step(dj, back);
        int p = is_c | (back != 0) ? near : cd;
        int q = is_c ? cb : (back ? cd : near);
        FbWord rp = rec(p), rq = rec(q);
        bool live = bound(rp, p) & bound(rq, q) & ((t <= 12) | is_tail | is_c);
        if (!any(live)) {
            return out;
        }
        // the pair: its kind, its own rules
        int pb = rp.partner(), qb = rq.partner();
        bool next_to = adjacent(pb, qb);
        bool helix = next_to & (qb > pb), contig = next_to & (qb < pb);
        int d = fb_diff(rq, rp), m = d < 0 ? fb_neg(d) : d;
        int po = rp.ore(), qo = rq.ore();
        bool along = m == fb_axis(po);  // the pair lies on p's axis
        bool ahead = d == fb_vector(po); // q is where p points
        bool spq = stacked(p, rp, q, rq);
        bool central = !next_to & !spq; // a regular pair off the stack
        bool pair_on = live & !((second != 0) & next_to);
        {
            // check_kink_constraint (domain.cpp:42-57, 80-97)
            bool flat = HALF ? qo != (po ^ 1) : (po >> 1) != (qo >> 1);
            bool kink = (ahead & flat) | (!along & (m != fb_axis(qo)));
            bool turn = (second == 0) & (along | !twist_ok(rp, d, rq));
            bool is_p = t == 0;
            out.helix = is_p & live & helix;
            out.viol = is_p & live & ((contig & !ahead) | (helix & turn) | (!next_to & !kink));
            out.op = is_p & pair_on & !contig & !central;
            if (!ONE) {
                out.a1 = p;
                out.b1 = q;
            }
        }
        // what is kept of it: one word instead of a lane mask each
        enum { ON = 1, CONTIG_PAIR = 2, OFF_STACK = 4, NEXT_TO = 8, STACKED = 16, LIVE = 32 };
        int kind = keep((int)pair_on * ON | (int)contig * CONTIG_PAIR | (int)central * OFF_STACK |
                        (int)next_to * NEXT_TO | (int)spq * STACKED | (int)live * LIVE);
        t = keep(t); // the kinds of check below are worked out again from it
        back = keep(back);
        is_j = (unsigned)(t - 1) < 9u;
        is_t = (unsigned)(t - 10) < 3u;
        is_c = t == 14;
        is_tail = (t == 13) & (back != 0);
        // n: the end the check leaves from; f: the other
        bool leave = (is_j & ((kind & (CONTIG_PAIR | OFF_STACK)) == 0)) | is_t;
        bool fw = is_tail | (leave & (back == 0));
        int n = fw ? q : p, f = fw ? p : q;
        FbWord rn = pick(fw, rq, rp), rf = pick(fw, rp, rq);
        int far = step(n, fw), nb = rn.partner();
        far = is_c ? di : far;
        nb = is_c ? dj : nb;
        int nf = fwd(nb), nr = bwd(nb);
        FbWord ro = rec(far), rnb = rec(nb), rnf = rec(nf), rnr = rec(nr);
        int i = keep(is_j ? (t >= 4) + (t >= 7) : (is_t ? t - 10 : 0));
        int v;
        {
            // the outer candidates after far, which a junction restricts
            int ob = bound(ro, far) ? ro.partner() : -2;
            bool to_r = ob == nr, to_f = ob == nf;
            bool single = (back ? nf : nr) == rf.partner();
            bool r_out = !single & to_r & bound(rnr, nr);
            bool f_out = !single & !r_out & to_f & bound(rnf, nf);
            bool off = (kind & OFF_STACK) != 0, ct = (kind & CONTIG_PAIR) != 0;
            bool use_r = (f_out | ((back != 0) & single)) & !ct;
            int k1 = off ? (to_f ? -1 : nf) : (use_r ? nr : nf);
            bool no2 = off ? to_r : (single | r_out | f_out | ct);
            int k2 = no2 ? -1 : nr;
            int v1 = is_j ? k1 : nf, v2 = is_j ? k2 : nr;
            v = i == 0 ? far : (i == 1 ? v1 : v2);
        }
        FbWord rv = pick(i == 0, ro, pick(v == nf, rnf, rnr));
        int u = i == 0 ? n : nb;
        FbWord ru = pick(i == 0, rn, rnb);
        bool sf = (kind & STACKED) != 0;
        {
            // central: candidate ip or in, centre di, the other end jp or jn
            bool sc = stacked(q, rq, dj, rnb);
            sf = is_c ? sc : sf;
            n = is_c ? di : n;
            u = is_c ? di : u;
            f = is_c ? q : f;
            v = is_c ? p : v;
            rn = pick(is_c, ro, rn);
            ru = pick(is_c, ro, ru);
            rf = pick(is_c, rq, rf);
            rv = pick(is_c, rp, rv);
        }
        bool bv = bound(rv, v);
        bool sv = stacked(u, ru, v, rv);
        t = keep(t);
        back = keep(back);
        is_t = (unsigned)(t - 10) < 3u;
        is_c = t == 14;
        is_tail = (t == 13) & (back != 0);
        {
            // ---- triplets (v, n, f)
            bool bk = (is_t & (back != 0)) | (is_c & (second == 0));
            int other = step(di, back);
            int dn = fb_diff(rn, rv);
            bool str = dn == fb_diff(rf, rn);
            bool dcv = ((bk ? n - v : v - n) == 1) & adjacent(rv.partner(), rn.partner());
            int vb = rv.partner();
            bool on = (is_t & ((kind & (ON | CONTIG_PAIR)) == ON)) |
                      ((is_tail | (is_c & !dcv & (rf.partner() != other))) & ((kind & LIVE) != 0));
            bool again = is_t & (i > 0) & ((vb == far) | (vb == f));
            bool trip = on & bv & !str & !again;
            bool off_v = dn != fb_vector(rv.ore());
            bool off_f = fb_diff(rn, rf) != fb_vector(rf.ore());
            bool may_v = fw | (is_c & (back == 0));
            bool may_f = is_c ? second == 0 : is_t & ((i == 2) | ((back != 0) & (i == 0)));
            bool both = trip & sv & sf;
            bool lone_v = trip & sv & !sf & off_f & may_v;
            bool lone_f = trip & !sv & sf & off_v & may_f;
            bool chain = both & (i == 0) & !is_c & dcv & ((kind & NEXT_TO) != 0) & (q == p + 1);
            int nv = is_c ? dj : n, nl = is_t & (i == 2) ? nb : n;
            bool any_t = trip & (t != 0);
            out.op = any_t ? (both ? 3 : (lone_v | lone_f ? 2 : 0)) : out.op;
            if (!ONE) {
                out.a1 = any_t ? (both ? (bk ? v : f) : (lone_v ? nv : nl)) : out.a1;
                out.b1 = any_t ? (both ? n : (lone_v ? v : f)) : out.b1;
                out.a2 = n;
                out.b2 = bk ? f : v;
            }
            out.viol = out.viol | (int)chain;
        }
        // ---- junctions
        is_j = (unsigned)(keep(t) - 1) < 9u;
        bool off = (kind & (CONTIG_PAIR | OFF_STACK)) == 0; // out of a stacked pair's end
        bool ct = (kind & CONTIG_PAIR) != 0;
        bool jn_ok = is_j & ((kind & ON) != 0) & bv & !(off & sv);
        if (!any(jn_ok)) {
            return out;
        }
        int j = t - 1 - 3 * i;
        // the next domain past v, going on from u (on a ring the difference
        // of their indices may be a whole turn less one)
        int gap = v - u;
        int up = (gap > 0) != (a.cyc && v < a.ns && gap * gap != 1);
        int y0 = step(off ? v : q, off ? up : 1);
        int x1 = off ? rv.partner() : qb;
        int y1 = step(x1, (j == 1) != ct);
        int y = j == 0 ? y0 : (ct & (j == 2) ? -1 : y1);
        FbWord ry0 = rec(y0), rx1 = rec(x1), ry = rec(y);
        jn_ok = jn_ok & bound(ry, y) & !((j > 0) & !ct & bound(ry0, y0) & (ry0.partner() == y));
        int x = j == 0 ? (off ? v : q) : x1;
        FbWord rx = pick(j == 0, pick(off, rv, rq), rx1);
        // the junction (j1, j2, x, y) over (s1, s2): (f, n, x, y) over (u,
        // v), or (v, u, x, y) over (p, q)
        int j1 = off ? f : v, j2 = off ? n : u, c1 = off ? u : p, c2 = off ? v : q;
        FbWord r1 = pick(off, rf, rv), r2 = pick(off, rn, ru);
        FbWord s1 = pick(off, ru, rp), s2 = pick(off, rv, rq);
        bool flip = c1 > c2;
        FbWord lo = pick(flip, s2, s1), hi = pick(flip, s1, s2);
        jn_ok = jn_ok & stacked(j1, r1, j2, r2) & stacked(x, rx, y, ry) &
                (fb_diff(hi, lo) == fb_vector(lo.ore()));
        // directions along increasing domain index
        int n1 = j1 < j2 ? fb_diff(r2, r1) : fb_diff(r1, r2);
        int n3 = x < y ? fb_diff(ry, rx) : fb_diff(rx, ry);
        // check_junction_constraint (domain.cpp:59-67, 99-118)
        bool jv = !HALF && !twist_off_axis(lo, flip ? n3 : n1, hi);
        int jop = n1 == n3 ? 4 : (n1 == fb_neg(n3) ? 0 : 3);
        out.viol = jn_ok ? (int)jv : out.viol;
        out.op = jn_ok ? (jv ? 0 : jop) : out.op;
        if (!ONE) {
            out.a1 = jn_ok ? (flip ? y : j1) : out.a1;
            out.b1 = jn_ok ? (flip ? x : j2) : out.b1;
            out.a2 = jn_ok ? (flip ? j2 : x) : out.a2;
            out.b2 = jn_ok ? (flip ? j1 : y) : out.b2;
        }
        return out;
    }
    // v as one register (a wavefront's conditions are pairs of scalar
    // registers, and the call would have to save them)
    static DEV int keep(int v) {
#ifdef __HIP_DEVICE_COMPILE__
        asm("" : "+v"(v));
#endif
        return v;
    }
    // check_twist_constraint along any d
    static DEV bool twist_off_axis(const FbWord& p, int d, const FbWord& q) {
        return fb_minus_quarter_turn(p.ore(), fb_index(d)) == q.ore();
    }

    // The order of the walk: for each pair its own term, then its junctions
    // and triplets (a helix pair's triplets first), after the pairs around a
    // domain the triplet around it, and the central triplets last.  `ops`:
    // checks with a term; `helix`: helix pairs (bit 16 b); add(c) adds check
    // c's term.
    template <class F>
    static DEV void in_order(uint64_t ops, uint64_t helix, F add) {
        constexpr uint64_t junctions = 0x3FEull, triplets = 0x1C00ull;
        // two passes per pair and one per domain, and the central triplets
#pragma unroll 1
        for (int k = 0; ops != 0 && k < 11; k++) {
            uint64_t m;
            if (k == 10) {
                m = ops;
            }
            else {
                int side = k >= 5 ? 1 : 0, r = k - 5 * side;
                int b = 2 * side + (r >> 1);
                bool hx = (helix >> (16 * (b & 3))) & 1;
                if (r == 4) {
                    m = ops & (1ull << (32 * side + 13));
                }
                else {
                    bool j = ((r & 1) == 0) != hx;
                    m = (j ? junctions : triplets) | ((r & 1) == 0 ? 1ull : 0ull);
                    m = ops & (m << (16 * b));
                }
            }
            ops &= ~m;
            for (; m; m &= m - 1) {
                add(__builtin_ctzll(m));
            }
        }
    }
};

// ------------------------------------------------ the general engine's walk
// One function per check of the reference, inlined into fb_terms but for the
// junction.  A block in device memory makes the walk wait for the memory side,
// which the call frames stream through too, so what counts is a small frame
// and few bytes read.  FourBody on such a block needs 2028 bytes of frame per
// lane (this form 1712) and reads every neighbour's whole record: 100 steps of
// 4096 chains take 32.3 ms with it and 28.1 with this form.
DEVIN void Eng::fb_single(int h1, int h2, int h3) {
    I3 n1 = sub3(pos(h2), pos(h1));
    if (eq3(n1, ore(h1))) {
        return;
    }
    I3 n2 = sub3(pos(h3), pos(h2));
    if (!eq3(n1, n2)) {
        dc_e -= stk(h2, h3);
        dc_st -= 1;
    }
}

DEVIN void Eng::fb_double(int h1, int h2, int h3) {
    I3 n1 = sub3(pos(h2), pos(h1));
    I3 n2 = sub3(pos(h3), pos(h2));
    if (!eq3(n1, n2)) {
        dc_e -= stk(h1, h2) / 2;
        dc_e -= stk(h2, h3) / 2;
        dc_st -= 1;
    }
}

DEVIN void Eng::fb_triply(int h1, int h2, int h3) {
    I3 n1 = sub3(pos(h2), pos(h1));
    I3 n2 = sub3(pos(h3), pos(h2));
    if (!eq3(n1, n2)) {
        fb_viol = true;
    }
}

// check_junction (origami_potential.cpp:419-462) with the stacking penalty
// of check_junction_stacking_penalty (:85-127)
DEVNI void Eng::fb_junction(int j1, int j2, int j3, int j4, int k1, int k2) {
    if (d_of(k1) > d_of(k2)) {
        int t = k1;
        k1 = k2;
        k2 = t;
        t = j1;
        j1 = j4;
        j4 = t;
        t = j2;
        j2 = j3;
        j3 = t;
    }
    if (!(pair_stacked(j1, j2) && pair_stacked(j3, j4))) {
        return;
    }
    if (!junction_ok(j1, j2, k1, k2)) {
        fb_viol = true;
        return;
    }
    int pen = 0;
    I3 nk = sub3(pos(k2), pos(k1));
    if (eq3(nk, ore(k1))) {
        I3 n1 = sub3(pos(j2), pos(j1));
        if (d_of(j1) > d_of(j2)) {
            n1 = neg3(n1);
        }
        I3 n3 = sub3(pos(j4), pos(j3));
        if (d_of(j3) > d_of(j4)) {
            n3 = neg3(n3);
        }
        pen = eq3(n1, n3) ? 2 : (eq3(n1, neg3(n3)) ? 0 : 1);
    }
    if (pen == 1) {
        dc_e -= stk(j1, j2) / 2;
        dc_e -= stk(j3, j4) / 2;
        dc_st -= 1;
    }
    else if (pen == 2) {
        dc_e -= stk(j1, j2);
        dc_e -= stk(j3, j4);
        dc_st -= 2;
    }
}

// check_doubly_contig_junction_pair (:359-417)
DEVIN void Eng::fb_junction_pair(int a, int b, int j) {
    int k1 = a, k2 = b;
    I3 ndr = sub3(pos(k2), pos(k1));
    if (!eq3(ore(k1), ndr)) {
        fb_viol = true;
        return;
    }
    if (j == 1) {
        return;
    }
    int sel_j1[2] = {walk(a, -1), walk(bd(a), 1)};
    int sel_j2[2] = {a, bd(a)};
    for (int q = 0; q < 2; q++) {
        int j1 = sel_j1[q], j2 = sel_j2[q];
        int j3 = k2;
        int j4 = walk(k2, 1);
        if (eb(j4) && eb(j1)) {
            fb_junction(j1, j2, j3, j4, k1, k2);
        }
        j3 = bd(k2);
        j4 = walk(j3, -1);
        if (eb(j4) && eb(j1)) {
            fb_junction(j1, j2, j3, j4, k1, k2);
        }
    }
}

// check_backward_triplet_stacking_combos (:464-519)
DEVIN void Eng::fb_backward_triplets(int a, int b) {
    int h2 = a, h3 = b;
    if (!pair_stacked(h2, h3)) {
        return;
    }
    int h1 = walk(a, -1);
    bool dc23 = doubly_contig(h2, h3);
    if (eb(h1)) {
        bool dc12 = doubly_contig(h1, h2);
        if (pair_stacked(h1, h2)) {
            if (dc12 && dc23) {
                fb_triply(h1, h2, h3);
                if (fb_viol) {
                    return;
                }
            }
            fb_double(h1, h2, h3);
        }
        else {
            fb_single(h1, h2, h3);
        }
    }
    int h2_prev = h1;
    int ba = bd(a);
    h1 = walk(ba, 1);
    if (eb(h1) && bd(h1) != h2_prev && bd(h1) != h3) {
        if (pair_stacked(ba, h1)) {
            fb_double(h1, h2, h3);
        }
    }
    h1 = walk(ba, -1);
    if (eb(h1) && bd(h1) != h2_prev && bd(h1) != h3) {
        if (pair_stacked(h1, ba)) {
            fb_double(h1, h2, h3);
        }
        else {
            fb_single(h1, ba, h3);
        }
    }
}

// check_forward_triplet_stacking_combos (:521-585)
DEVIN void Eng::fb_forward_triplets(int a, int b) {
    int h2 = b, h1 = a;
    bool first = pair_stacked(h1, h2);
    int h3 = walk(b, 1);
    bool dc12 = doubly_contig(h1, h2);
    if (eb(h3)) {
        bool second = pair_stacked(h2, h3);
        if (first && second) {
            bool dc23 = doubly_contig(h2, h3);
            if (dc12 && dc23) {
                fb_triply(h1, h2, h3);
                if (fb_viol) {
                    return;
                }
            }
            fb_double(h1, h2, h3);
        }
        else if (second) {
            fb_single(h1, h2, h3);
        }
    }
    int h2_next = h3;
    int bb = bd(b);
    h3 = walk(bb, 1);
    if (eb(h3) && bd(h3) != h2_next && bd(h3) != h1) {
        if (pair_stacked(bb, h3)) {
            if (first) {
                fb_double(h1, h2, h3);
            }
            else {
                fb_single(h1, h2, h3);
            }
        }
    }
    h3 = walk(bb, -1);
    if (eb(h3) && bd(h3) != h2_next && bd(h3) != h1) {
        if (pair_stacked(h3, bb)) {
            if (first) {
                fb_double(h1, h2, h3);
            }
            else {
                fb_single(h1, h2, h3);
            }
        }
        else if (first) {
            fb_single(h3, bb, h1);
        }
    }
}

// check_central_triplet_stacking_combos (:587-652)
DEVIN void Eng::fb_central_triplets(int di, int dj) {
    int h1 = walk(di, -1);
    int h2 = di;
    int h3 = walk(dj, 1);
    int h2_next = walk(di, 1);
    if (eb(h1) && eb(h3) && bd(h3) != h2_next && !doubly_contig(h1, h2)) {
        if (pair_stacked(dj, h3)) {
            if (pair_stacked(h1, h2)) {
                fb_double(h1, h2, h3);
            }
            else {
                fb_single(h1, h2, h3);
            }
        }
    }
    h3 = walk(dj, -1);
    if (eb(h1) && eb(h3) && bd(h3) != h1 && !doubly_contig(h1, h2)) {
        if (pair_stacked(h1, h2)) {
            if (pair_stacked(h3, dj)) {
                fb_double(h1, h2, h3);
            }
            else {
                fb_single(h3, dj, h1);
            }
        }
        else if (pair_stacked(h3, dj)) {
            fb_single(h1, h2, h3);
        }
    }
    h2 = di;
    h3 = walk(di, 1);
    h1 = walk(dj, 1);
    int h2_prev = walk(di, -1);
    if (eb(h1) && eb(h3) && bd(h1) != h3 && !doubly_contig(h2, h3)) {
        if (pair_stacked(dj, h1) && pair_stacked(h2, h3)) {
            fb_double(h1, h2, h3);
        }
    }
    h1 = walk(dj, -1);
    if (eb(h1) && eb(h3) && bd(h1) != h2_prev && !doubly_contig(h2, h3)) {
        if (pair_stacked(h2, h3)) {
            if (pair_stacked(h1, dj)) {
                fb_double(h1, h2, h3);
            }
            else {
                fb_single(h1, dj, h3);
            }
        }
    }
}

// The single-junction checks below enumerate up to three outer candidate
// pairs and, for each, up to three inner ones.  The lists are kept in scalar
// variables (LDO_NONE for an entry the reference does not add; eb() is false
// on it), each outer candidate in a function of its own, and no list lives in
// a local array: gfx950 code for a small stack array filled on divergent
// branches was found to store the last entry at the wrong index and leave the
// next one unwritten, which the loop then used as a domain slot.  The order
// of the fb_junction calls, and of every read before them, is the reference's.

// inner candidates of one outer pair (k2, k1) of check_backward_single_junction
DEVIN void Eng::fb_backward_outer(int j3, int j4, int k2, int k1) {
    if (!eb(k1) || pair_stacked(k1, k2)) {
        return;
    }
    int k1_next = walk(k1, d_of(k1) - d_of(k2));
    int k1b = bd(k1);
    int k1b_for = fwd(k1b);
    int k1b_bac = bwd(k1b);
    int e1 = k1b_for, e2 = k1b_bac;
    if (eb(k1_next)) {
        int k1nb = bd(k1_next);
        if (k1b_for == k1nb) {
            e1 = LDO_NONE;
        }
        if (k1b_bac == k1nb) {
            e2 = LDO_NONE;
        }
    }
    if (eb(k1_next)) {
        fb_junction(k1_next, k1, j3, j4, k1, k2);
    }
    if (eb(e1)) {
        fb_junction(e1, k1b, j3, j4, k1, k2);
    }
    if (eb(e2)) {
        fb_junction(e2, k1b, j3, j4, k1, k2);
    }
}

// check_backward_single_junction (:654-748)
DEVIN void Eng::fb_backward_single_junction(int a, int b) {
    int j3 = a, j4 = b;
    int j3_bac = bwd(j3);
    int j3b = bd(j3);
    int j3b_for = fwd(j3b);
    int j3b_bac = bwd(j3b);
    int c1, c2 = LDO_NONE; // outer candidates (j3b, c) after (j3, j3_bac)
    if (j3b_for == bd(j4)) {
        c1 = j3b_bac;
    }
    else if (eb(j3_bac) && eb(j3b_bac) && bd(j3_bac) == j3b_bac) {
        c1 = j3b_for;
    }
    else if (eb(j3_bac) && eb(j3b_for) && bd(j3_bac) == j3b_for) {
        c1 = j3b_bac;
    }
    else {
        c1 = j3b_for;
        c2 = j3b_bac;
    }
    fb_backward_outer(j3, j4, j3, j3_bac);
    fb_backward_outer(j3, j4, j3b, c1);
    fb_backward_outer(j3, j4, j3b, c2);
}

// inner candidates of one outer pair (k1, k2) of check_forward_single_junction
DEVIN void Eng::fb_forward_outer(int j1, int j2, int k1, int k2) {
    if (!eb(k2) || pair_stacked(k1, k2)) {
        return;
    }
    int k2_next = walk(k2, d_of(k2) - d_of(k1));
    int k2b = bd(k2);
    int k2b_for = fwd(k2b);
    int k2b_bac = bwd(k2b);
    int e1 = k2b_for, e2 = k2b_bac;
    if (eb(k2_next)) {
        int k2nb = bd(k2_next);
        if (k2b_for == k2nb) {
            e1 = LDO_NONE;
        }
        if (k2b_bac == k2nb) {
            e2 = LDO_NONE;
        }
    }
    if (eb(k2_next)) {
        fb_junction(j1, j2, k2, k2_next, k1, k2);
    }
    if (eb(e1)) {
        fb_junction(j1, j2, k2b, e1, k1, k2);
    }
    if (eb(e2)) {
        fb_junction(j1, j2, k2b, e2, k1, k2);
    }
}

// check_forward_single_junction (:750-844)
DEVIN void Eng::fb_forward_single_junction(int a, int b) {
    int j1 = a, j2 = b;
    int j2_for = fwd(j2);
    int j1b = bd(j1);
    int j2b = bd(j2);
    int j2b_for = fwd(j2b);
    int j2b_bac = bwd(j2b);
    int c1, c2 = LDO_NONE; // outer candidates (j2b, c) after (j2, j2_for)
    if (walk(j1b, 1) == j2b) {
        c1 = j2b_for;
    }
    else if (eb(j2_for) && eb(j2b_bac) && bd(j2_for) == j2b_bac) {
        c1 = j2b_for;
    }
    else if (eb(j2_for) && eb(j2b_for) && bd(j2_for) == j2b_for) {
        c1 = j2b_bac;
    }
    else {
        c1 = j2b_for;
        c2 = j2b_bac;
    }
    fb_forward_outer(j1, j2, j2, j2_for);
    fb_forward_outer(j1, j2, j2b, c1);
    fb_forward_outer(j1, j2, j2b, c2);
}

// inner candidates of one outer pair (j2, j1) of check_central_single_junction
DEVIN void Eng::fb_central_outer(int j1, int j2, int k1, int k2, int k2b) {
    if (!eb(j1)) {
        return;
    }
    int k2_for = fwd(k2);
    int k2b_for = fwd(k2b);
    int k2b_bac = bwd(k2b);
    int e1 = k2b_for, e2 = k2b_bac;
    if (eb(k2_for)) {
        int k2fb = bd(k2_for);
        if (k2b_for == k2fb) {
            e1 = LDO_NONE;
        }
        if (k2b_bac == k2fb) {
            e2 = LDO_NONE;
        }
    }
    if (eb(k2_for)) {
        fb_junction(j1, j2, k2, k2_for, k1, k2);
    }
    if (eb(e1)) {
        fb_junction(j1, j2, k2b, e1, k1, k2);
    }
    if (eb(e2)) {
        fb_junction(j1, j2, k2b, e2, k1, k2);
    }
}

// check_central_single_junction (:846-934)
DEVIN void Eng::fb_central_single_junction(int a, int b) {
    int k1 = a, k2 = b;
    int k1b = bd(k1), k2b = bd(k2);
    if (cslot_of(k1b) == cslot_of(k2b)) {
        int dd = d_of(k1b) - d_of(k2b);
        if (dd == 1 || dd == -1) {
            return;
        }
    }
    int k1_bac = bwd(k1);
    int k1b_for = fwd(k1b);
    int k1b_bac = bwd(k1b);
    int e1 = k1b_for, e2 = k1b_bac; // outer candidates (k1b, e) after (k1, k1_bac)
    if (eb(k1_bac)) {
        int k1bacb = bd(k1_bac);
        if (k1b_for == k1bacb) {
            e1 = LDO_NONE;
        }
        if (k1b_bac == k1bacb) {
            e2 = LDO_NONE;
        }
    }
    fb_central_outer(k1_bac, k1, k1, k2, k2b);
    fb_central_outer(e1, k1b, k1, k2, k2b);
    fb_central_outer(e2, k1b, k1, k2, k2b);
}

// check_regular_pair_constraints (:288-320)
DEVIN void Eng::fb_regular_pair(int a, int b, int i) {
    I3 ndr = sub3(pos(b), pos(a));
    if (!kink_ok(a, ndr, b)) {
        fb_viol = true;
        return;
    }
    if (pair_stacked(a, b)) {
        dc_e += stk(a, b);
        dc_st += 1;
        if (i == -1) {
            fb_backward_single_junction(a, b);
        }
        else {
            fb_forward_single_junction(a, b);
        }
    }
    else {
        fb_central_single_junction(a, b);
    }
    if (i == -1) {
        fb_backward_triplets(a, b);
    }
    else {
        fb_forward_triplets(a, b);
    }
}

// check_doubly_contig_helix_pair (:322-357)
DEVIN void Eng::fb_helix_pair(int a, int b, int i, int j) {
    if (j == 1) {
        return;
    }
    I3 ndr = sub3(pos(b), pos(a));
    I3 oa = ore(a);
    if (eq3(ndr, oa) || eq3(ndr, neg3(oa))) {
        fb_viol = true;
        return;
    }
    if (twist_ok(a, ndr, b)) {
        dc_e += stk(a, b);
        dc_st += 1;
    }
    else {
        fb_viol = true;
        return;
    }
    if (i == -1) {
        fb_backward_triplets(a, b);
        fb_backward_single_junction(a, b);
    }
    else {
        fb_forward_triplets(a, b);
        fb_forward_single_junction(a, b);
    }
}

// JunctionBindingPotential::check_constraints (:231-286)
DEVIN void Eng::fb_around(int cd, int j) {
    for (int i = -1; i <= 0; i++) {
        int a = walk(cd, i);
        int b = walk(cd, i + 1);
        if (!(eb(a) && eb(b))) {
            continue;
        }
        int ba = bd(a), bb = bd(b);
        if (cslot_of(ba) == cslot_of(bb)) {
            if (d_of(ba) == d_of(bb) - 1) {
                fb_helix_pair(a, b, i, j);
            }
            else if (d_of(ba) == d_of(bb) + 1) {
                fb_junction_pair(a, b, j);
            }
            else {
                fb_regular_pair(a, b, i);
            }
        }
        else {
            fb_regular_pair(a, b, i);
        }
        if (fb_viol) {
            return;
        }
    }
    int pv = walk(cd, -1);
    int nx = walk(cd, 1);
    if (eb(pv) && eb(nx)) {
        if (pair_stacked(cd, nx)) {
            if (pair_stacked(pv, cd)) {
                if (doubly_contig(pv, cd) && doubly_contig(cd, nx)) {
                    fb_triply(pv, cd, nx);
                    if (fb_viol) {
                        return;
                    }
                }
                fb_double(pv, cd, nx);
            }
            else {
                fb_single(pv, cd, nx);
            }
        }
    }
}

// calc_stacking_and_steric_terms (:212-229)
DEVNI void Eng::fb_terms(int di, int dj) {
    fb_around(di, 0);
    if (fb_viol) {
        return;
    }
    fb_around(dj, 1);
    if (fb_viol) {
        return;
    }
    fb_central_triplets(di, dj);
}

// OrigamiPotential::bind_domain (:1282-1312), BindingPotential::bind_domains
// (:131-147) and OpposingMisbindingPotential / Disallowed (:938-950)
DEVIN Delta Eng::bind_domain(int di) {
    Delta r;
    r.e = 0;
    r.st = 0;
    pot_viol = false;
    int dj = bd(di);
    S->site_bind++;
    if (ident_of(di) == -ident_of(dj)) {
        dc_e = 0;
        dc_st = 0;
        fb_viol = false;
        if (dom[di].ore != (dom[dj].ore ^ 1)) {
            fb_viol = true;
        }
        else {
            fb_terms(di, dj);
            if (!fb_viol) {
                dc_e += hyb(di, dj);
                r.e = dc_e;
                r.st = dc_st;
            }
        }
        pot_viol = fb_viol;
    }
    else if (mispot == 0) {
        if (dom[di].ore != (dom[dj].ore ^ 1)) {
            pot_viol = true;
        }
        else {
            r.e += hyb(di, dj);
        }
    }
    else {
        pot_viol = true;
    }
    return r;
}

#endif
