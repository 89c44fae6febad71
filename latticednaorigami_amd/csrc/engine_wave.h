// engine_wave.h - the replica engine of the sweep kernels: one wavefront per
// replica, its block in the workgroup's LDS.
//
// A Markov chain is serial, so the time of a step is the sum of the latencies
// along it.  Eng, run by a wavefront, spent 13 000 instructions and 2 000
// dependent memory accesses on a step of the 64-domain raster workload: every
// field read went through the engine object and a flat pointer, and every
// branch was an exec-mask branch on values the compiler could not know to be
// equal on all lanes.  WEng keeps the chain's scalars in registers, addresses
// LDS directly, makes every value read from it uniform (v_readfirstlane), so
// control flow and index arithmetic run on the scalar unit, and uses the 64
// lanes where a step has independent work:
//   random draws      64 of a step's Philox draws in one evaluation
//   site hash         64 entries of a probe run per read; the six trial sites
//                     of a growth step at once (eight lanes each)
//   trial weights     table reads, exp and division of all sites at once
//   endpoints         64 active endpoints per read
//   chain lists       searches and deletions by ballot
// All functions but the FourBody walk are inlined into the kernel: a call
// would spill the registers it exists to keep.
//
// Measured (MI355X, general engine in LDS -> this one): 64-domain raster, 32
// replicas, a 1000-step interval and its observables 84.5 -> 22.4 ms; recoil
// growth on it, 16 replicas 106.2 -> 36.6 ms; 4-domain system, one replica 80
// -> 26 us per step; 200-domain umbrella windows, 64 replicas 22.7 -> 7.5 ms.
// What is left is instruction latency of one wavefront: a FourBody walk
// (4 600 cycles) per binding evaluation, an unassignment 1 100, a choice among
// six sites 5 000, and the scalar registers the inlined moves spill to vector
// lanes (a fifth of the instructions).
//
// The move types are engine_moves.h's, compiled again for this class; what is
// redefined here computes the same values in the same order.
#ifndef LDO_ENGINE_WAVE_H
#define LDO_ENGINE_WAVE_H

#include "engine.h"
#include "engine_fourbody.h"
#include "engine_system.h"
#include "engine_moves.h"

#ifdef __HIP_DEVICE_COMPILE__
#define LDO_LDS __attribute__((address_space(3)))
#else
#define LDO_LDS
#endif
typedef LDO_LDS char* lds_t;

// ------------------------------------------------- uniform values, lanes
DEV int32_t uni(int32_t v) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_readfirstlane(v);
#else
    return v;
#endif
}
DEV uint32_t uni(uint32_t v) { return (uint32_t)uni((int32_t)v); }
DEV int16_t uni(int16_t v) { return (int16_t)uni((int32_t)v); }
DEV int8_t uni(int8_t v) { return (int8_t)uni((int32_t)v); }
DEV uint64_t uni(uint64_t v) {
    return (uint64_t)uni((uint32_t)v) | (uint64_t)uni((uint32_t)(v >> 32)) << 32;
}
DEV int64_t uni(int64_t v) { return (int64_t)uni((uint64_t)v); }
// FP64 values stay in vector registers (there is no scalar FP64 unit)
DEV double uni(double v) { return v; }
// a condition that is the same on every lane
DEV bool all_lanes(bool b) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_ballot_w64(b) != 0;
#else
    return b;
#endif
}
#ifdef __HIP_DEVICE_COMPILE__
__device__ __forceinline__ double lane_double(double v, int src) {
    uint64_t b = __builtin_bit_cast(uint64_t, v);
    uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, src);
    uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), src);
    return __builtin_bit_cast(double, (uint64_t)lo | (uint64_t)hi << 32);
}
#endif

// one value in LDS: reads are uniform, writes store the same value from all
// lanes
template <class T>
struct LRef {
    lds_t p;
    DEV operator T() const { return uni(*(LDO_LDS const T*)p); }
    DEV T operator=(T v) const {
        *(LDO_LDS T*)p = v;
        return v;
    }
    DEV T operator=(const LRef& o) const { return *this = (T)o; }
    DEV void operator+=(T v) const { *this = (T)((T)*this + v); }
    DEV T operator++(int) const {
        T v = *this;
        *this = (T)(v + 1);
        return v;
    }
};

template <class T>
struct LArr {
    lds_t p;
    DEV LRef<T> operator[](int i) const { return LRef<T> {p + i * (int)sizeof(T)}; }
    DEV LArr operator+(int n) const { return LArr {p + n * (int)sizeof(T)}; }
    // this lane's own element
    DEV T lane(int i) const { return *(LDO_LDS const T*)(p + i * (int)sizeof(T)); }
};

// records in LDS (the structs of layout.h, field by field)
template <class R, int SIZE>
struct LRecs {
    lds_t p;
    DEV R operator[](int i) const { return R(p + i * SIZE); }
};
struct LDom {
    LRef<int32_t> x, y, z;
    LRef<int8_t> ore, state;
    LRef<int16_t> bound;
    DEV explicit LDom(lds_t p) : x {p}, y {p + 4}, z {p + 8}, ore {p + 12}, state {p + 13},
                                 bound {p + 14} {}
};
struct LPosOre {
    lds_t p;
    LRef<int32_t> x, y, z, ore;
    DEV explicit LPosOre(lds_t q) : p(q), x {q}, y {q + 4}, z {q + 8}, ore {q + 12} {}
    DEV void operator=(const LPosOre& o) const {
        *(LDO_LDS Quad*)p = *(LDO_LDS const Quad*)o.p;
    }
};
struct LChain {
    LRef<int32_t> uid;
    LRef<int16_t> ident, len;
    DEV explicit LChain(lds_t p) : uid {p}, ident {p + 4}, len {p + 6} {}
};
struct LNetFrame {
    LRef<int16_t> growth, idx;
    DEV explicit LNetFrame(lds_t p) : growth {p}, idx {p + 2} {}
};
struct LGrowFrame {
    LRef<int16_t> first, count, i, prev, gold, gnew;
    LRef<int8_t> dir, kind, phase;
    DEV explicit LGrowFrame(lds_t p) : first {p}, count {p + 2}, i {p + 4}, prev {p + 6},
                                       gold {p + 8}, gnew {p + 10}, dir {p + 12}, kind {p + 13},
                                       phase {p + 14} {}
    DEV void operator=(const GrowFrame& f) const {
        first = f.first;
        count = f.count;
        i = f.i;
        prev = f.prev;
        gold = f.gold;
        gnew = f.gnew;
        dir = f.dir;
        kind = f.kind;
        phase = f.phase;
    }
};
struct LJumpSeg {
    LRef<int16_t> first, count, last;
    LRef<int8_t> dir;
    DEV explicit LJumpSeg(lds_t p) : first {p}, count {p + 2}, last {p + 4}, dir {p + 6} {}
    DEV void operator=(const JumpSeg& s) const {
        first = s.first;
        count = s.count;
        last = s.last;
        dir = s.dir;
    }
};
struct LEndpoint {
    LRef<int16_t> cslot, d;
    LRef<int32_t> seg, x, y, z;
    DEV explicit LEndpoint(lds_t p) : cslot {p}, d {p + 2}, seg {p + 4}, x {p + 8}, y {p + 12},
                                      z {p + 16} {}
};
static_assert(sizeof(DomRec) == 16 && sizeof(PosOre) == 16 && sizeof(ChainRec) == 8 &&
                  sizeof(NetFrame) == 4 && sizeof(GrowFrame) == 16 && sizeof(JumpSeg) == 8 &&
                  sizeof(Endpoint) == 20,
              "LDS records follow layout.h");

// The chain's scalars in registers: RepScalars without the arrays indexed at
// run time, which stay in the block's head.
struct WScal : RepScalars {
    LArr<int64_t> attempts, accepts;
    LArr<int32_t> added;
};

// ------------------------------------------------------------- FourBody
// the walk's access to a replica block in LDS
struct FbLds {
    lds_t dom, dident;
    const double* t_stack;
    double stack_all; // every pair's stacking energy, when it is one value
    int stack_one;
    int ns, lmask, cyc, dtype, n_ident;
    DEV FbRec rec(int s) const {
        Quad v = *(LDO_LDS const Quad*)(dom + s * 16);
        return FbRec {uni((int32_t)v.x), uni((int32_t)v.y), uni((int32_t)v.z), uni(v.w)};
    }
    DEV double stk(int p, int q) const {
        if (stack_one) {
            return stack_all;
        }
        int a = uni(*(LDO_LDS const int16_t*)(dident + 2 * p));
        int b = uni(*(LDO_LDS const int16_t*)(dident + 2 * q));
        return t_stack[(size_t)a * n_ident + b];
    }
};

struct FbOut {
    double e;
    int st, viol;
};

// the same for one lane's own record
struct FbLane {
    lds_t dom;
    int ns, lmask, cyc, dtype;
    DEV FbRec rec(int s) const {
        Quad v = *(LDO_LDS const Quad*)(dom + s * 16);
        return FbRec {(int32_t)v.x, (int32_t)v.y, (int32_t)v.z, v.w};
    }
    DEV double stk(int, int) const { return 0; }
};

// What a FourBody evaluation reads besides the pair: passed by value, since
// the evaluation is a call.  `flags`: lmask | cyc << 8 | dtype << 9 |
// stack_one << 10.
struct FbArgs {
    lds_t dom, dident;
    const double* t_stack;
    double stack_all; // every pair's stacking energy, when it is one value
    int flags, ns, n_ident;
};
DEV FbArgs fb_uniform(FbArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
    a.dom = (lds_t)(uint32_t)uni((int32_t)(uint32_t)a.dom);
    a.dident = (lds_t)(uint32_t)uni((int32_t)(uint32_t)a.dident);
#endif
    a.flags = uni(a.flags);
    a.ns = uni(a.ns);
    a.n_ident = uni(a.n_ident);
    return a;
}

// The walk itself: for a sum that a violation has ended early.
static __host__ __device__ __noinline__ FbOut wave_fb_walk(FbArgs g, int di, int dj) {
    g = fb_uniform(g);
    FbLds a {g.dom, g.dident, g.t_stack, g.stack_all, (g.flags >> 10) & 1, g.ns, g.flags & 255,
             (g.flags >> 8) & 1, (g.flags >> 9) & 1, g.n_ident};
    FourBody<FbLds> f(a);
    f.terms(uni(di), uni(dj));
    return FbOut {f.e, f.st, f.viol ? 1 : 0};
}

// The walk's checks side by side (FbChecks).  On a violation e and st are not
// set.
template <bool HALF, bool ONE>
static __host__ __device__ __noinline__ FbOut wave_fb_terms(FbArgs g, int di, int dj) {
    g = fb_uniform(g);
    FbLane a {g.dom, g.ns, g.flags & 255, (g.flags >> 8) & 1, (g.flags >> 9) & 1};
    typedef FbChecks<FbLane, HALF, ONE> Checks;
    Checks f(a);
    di = uni(di);
    dj = uni(dj);
    FbOut out {0.0, 0, 0};
    constexpr bool one = ONE;
#ifdef __HIP_DEVICE_COMPILE__
    int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    FbTerm t = f.check(lane, di, dj,
                       [](bool b) { return __builtin_amdgcn_ballot_w64(b) != 0; });
    if (__builtin_amdgcn_ballot_w64(t.viol != 0)) {
        out.viol = 1;
        return out;
    }
    uint64_t ops = __builtin_amdgcn_ballot_w64(t.op != 0);
    if (ops == 0) {
        return out;
    }
    double s1 = g.stack_all, s2 = g.stack_all;
    if (!one) {
        LDO_LDS const int16_t* id = (LDO_LDS const int16_t*)g.dident;
        if (t.op != 0) {
            s1 = g.t_stack[(size_t)id[t.a1] * g.n_ident + id[t.b1]];
        }
        if (t.op > 2) {
            s2 = g.t_stack[(size_t)id[t.a2] * g.n_ident + id[t.b2]];
        }
    }
    double e = 0;
    Checks::in_order(ops, __builtin_amdgcn_ballot_w64(t.helix != 0), [&](int c) {
        int op = __builtin_amdgcn_readlane(t.op, c);
        double x = one ? s1 : lane_double(s1, c);
        if (op == 1) {
            e += x;
        }
        else if (op == 3) {
            double y = one ? s2 : lane_double(s2, c);
            e -= x / 2;
            e -= y / 2;
        }
        else {
            e -= x;
            if (op == 4) {
                e -= one ? s2 : lane_double(s2, c);
            }
        }
    });
    out.e = e;
    out.st = __builtin_popcountll(__builtin_amdgcn_ballot_w64(t.op == 1)) -
             __builtin_popcountll(__builtin_amdgcn_ballot_w64(t.op == 2 || t.op == 3)) -
             2 * __builtin_popcountll(__builtin_amdgcn_ballot_w64(t.op == 4));
    return out;
#else
    FbTerm t[64];
    uint64_t ops = 0, helix = 0;
    for (int c = 0; c < 64; c++) {
        t[c] = f.check(c, di, dj, [](bool) { return true; });
        out.viol |= t[c].viol;
        ops |= t[c].op != 0 ? 1ull << c : 0;
        helix |= t[c].helix != 0 ? 1ull << c : 0;
    }
    if (out.viol) {
        return out;
    }
    const int16_t* id = (const int16_t*)g.dident;
    Checks::in_order(ops, helix, [&](int c) {
        double x = one ? g.stack_all : g.t_stack[(size_t)id[t[c].a1] * g.n_ident + id[t[c].b1]];
        double y = one || t[c].op < 3
                       ? g.stack_all
                       : g.t_stack[(size_t)id[t[c].a2] * g.n_ident + id[t[c].b2]];
        switch (t[c].op) {
        case 1:
            out.e += x;
            out.st += 1;
            break;
        case 2:
            out.e -= x;
            out.st -= 1;
            break;
        case 3:
            out.e -= x / 2;
            out.e -= y / 2;
            out.st -= 1;
            break;
        case 4:
            out.e -= x;
            out.e -= y;
            out.st -= 2;
            break;
        }
    });
    return out;
#endif
}

// a lattice site as a lookup finds it: its occupancy, its occupant (the
// domain placed last) and the index of its hash entry, or of the free entry a
// domain placed there takes
struct Site {
    int occ, s, home, at;
    uint32_t w; // the occupant's packed orientation, state and partner
};

// endpoints held in LDS; a longer list goes on in the block in device memory
#define LDO_WAVE_EP 64

// LDS bytes of a replica: the staged part of its block, the two endpoint
// lists and the binding energies of complementary pairs
LDO_HD int64_t wave_lds_bytes(const Params& p) {
    int64_t b = p.L.stage + 2 * LDO_WAVE_EP * (int64_t)sizeof(Endpoint) + 8 * (int64_t)p.n_ident;
    return (b + 255) / 256 * 256;
}

#define S (&sc)
struct WEng {
    const Params* P;
    char* gblk; // the block in device memory (sections past Layout::stage)
    int rep;
    WScal sc;
    lds_t blk;
    LRecs<LDom, 16> dom;
    LArr<int16_t> dident;
    LRecs<LChain, 8> ch;
    LArr<int16_t> order, freel, tlist, tcount;
    LArr<uint32_t> hash;
    LArr<int16_t> modified, assigned;
    LRecs<LPosOre, 16> prev, old;
    LArr<int8_t> seg;
    LArr<int16_t> gp, stem, inact;
    LArr<int8_t> netseg, netds_flag, checked, netcs, regrow, dir0, dir1;
    LArr<int16_t> gps, iaes, netds;
    LRecs<LNetFrame, 4> frames, sframes;
    LArr<int8_t> part;
    LRecs<LGrowFrame, 16> gstack;
    LArr<int16_t> gpl, rgs;
    LArr<int8_t> rgatt, rgwatt;
    LArr<uint64_t> rgavail, rgwavail;
    LArr<double> rgopen;
    LRecs<LEndpoint, 20> erstk;
    LArr<int16_t> ercnt;
    LArr<int8_t> jdom;
    LArr<int16_t> jps;
    LRecs<LJumpSeg, 8> jseg;
    LArr<int16_t> jstem;
    LArr<int8_t> stemseg, sdir;
    lds_t ep, ep0;        // active endpoints and their initial copy
    LArr<double> full;    // binding energy of identity i and its complement
    const double* t_hyb;
    const double* t_stack;
    double stack_all;
    double init_e;
    int fb_flags;
    int ns, lshift, lmask, nslots, nchain, hmask, hbits, n_ident, ident_lo, ecap;
    int cyc, dtype, mispot, rngmode;
    uint64_t seed;
    int n_gps, n_iaes, n_netds;
    bool net_external;
    int rg_max_recoils, rg_max_att, rg_max_segreg;
    int64_t rg_dup;
    int seg_first, seg_count, seg_dir;
    // this replica's umbrella window
    int w_on, w_op, w_min, w_max, w_last;
    double w_well, w_minb, w_slope, w_off, w_mult, w_st0, w_st1, w_grid;
    // The six sites around a domain's chain neighbour, eight lanes each; the
    // first of the eight (lane 8 v) holds site v's lookup.  six_d: the domain
    // they were looked up for while they stand, -1 once a domain or an
    // endpoint has changed.
    int six_d;
    I3 six_p;                 // this lane's site
    int six_s, six_h, six_at; // occupant, home, entry
    uint32_t six_w;
    uint64_t six_empty, six_unb, six_full;
    uint64_t six_walk;        // sites d's walks remain possible from
    uint64_t six_ends;        // sites that are an endpoint of d
    // lane m: kind, max_regrowth and first tracking counters of move m, its
    // attempts and accepts since the launch
    int mv_kind, mv_maxreg, mv_track, mv_width, mv_att, mv_acc;
    // random draws of the current block of 64 (this lane's)
    uint64_t rng_draw;
    int rng_block;

    // ------------------------------------------------------------ lanes
    DEV int plane() const {
#ifdef __HIP_DEVICE_COMPILE__
        return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
#else
        return 0;
#endif
    }
#ifdef __HIP_DEVICE_COMPILE__
    static constexpr int width = 64;
    static __device__ __forceinline__ uint64_t ballot(bool b) {
        return __builtin_amdgcn_ballot_w64(b);
    }
    static __device__ __forceinline__ int lane_int(int v, int src) {
        return __builtin_amdgcn_readlane(v, src);
    }
    // lanes of m below this one
    static __device__ __forceinline__ int below(uint64_t m) {
        return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                              __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    }
#else
    static constexpr int width = 1;
#endif
    DEV int pwidth() const { return width; }

    template <class T>
    DEV void fill_section(LArr<T> a, int64_t bytes, uint32_t pattern) {
        Quad q {pattern, pattern, pattern, pattern};
        for (int i = plane(), n = (int)((bytes + 15) / 16); i < n; i += width) {
            *(LDO_LDS Quad*)(a.p + 16 * i) = q;
        }
    }

    // ----------------------------------------------------------- wiring
    // Takes over a replica whose block's staged part has been copied to
    // `lds` (wave_lds_bytes); `g` is the block itself.
    DEV void attach(const Params* p, char* g, lds_t lds, int r) {
        P = p;
        gblk = g;
        rep = r;
        blk = lds;
        const Layout& L = p->L;
        dom.p = lds + L.off_dom;
        dident.p = lds + L.off_dident;
        ch.p = lds + L.off_chain;
        order.p = lds + L.off_order;
        freel.p = lds + L.off_free;
        tlist.p = lds + L.off_tlist;
        tcount.p = lds + L.off_tcount;
        hash.p = lds + L.off_hash;
        modified.p = lds + L.off_modified;
        assigned.p = lds + L.off_assigned;
        prev.p = lds + L.off_prev;
        old.p = lds + L.off_old;
        seg.p = lds + L.off_seg;
        gp.p = lds + L.off_gp;
        stem.p = lds + L.off_stem;
        inact.p = lds + L.off_inact;
        netseg.p = lds + L.off_netseg;
        netds_flag.p = lds + L.off_netds_flag;
        checked.p = lds + L.off_checked;
        netcs.p = lds + L.off_netcs;
        regrow.p = lds + L.off_regrow;
        dir0.p = lds + L.off_dir0;
        dir1.p = lds + L.off_dir1;
        gps.p = lds + L.off_gps;
        iaes.p = lds + L.off_iaes;
        netds.p = lds + L.off_netds;
        frames.p = lds + L.off_frames;
        part.p = lds + L.off_part;
        sframes.p = lds + L.off_sframes;
        gstack.p = lds + L.off_gstack;
        gpl.p = lds + L.off_gpl;
        rgs.p = lds + L.off_rgs;
        rgatt.p = lds + L.off_rgatt;
        rgwatt.p = lds + L.off_rgwatt;
        rgavail.p = lds + L.off_rgavail;
        rgwavail.p = lds + L.off_rgwavail;
        rgopen.p = lds + L.off_rgopen;
        erstk.p = lds + L.off_erstk;
        ercnt.p = lds + L.off_ercnt;
        jdom.p = lds + L.off_jdom;
        jps.p = lds + L.off_jps;
        jseg.p = lds + L.off_jseg;
        jstem.p = lds + L.off_jstem;
        stemseg.p = lds + L.off_stemseg;
        sdir.p = lds + L.off_sdir;
        ep = lds + L.stage;
        ep0 = ep + LDO_WAVE_EP * (int)sizeof(Endpoint);
        full.p = ep0 + LDO_WAVE_EP * (int)sizeof(Endpoint);
        ns = L.ns;
        lshift = L.lshift;
        lmask = (1 << L.lshift) - 1;
        nslots = L.nslots;
        nchain = L.nchain;
        hbits = L.hbits;
        hmask = L.hcap - 1;
        ecap = L.ecap;
        n_ident = p->n_ident;
        ident_lo = p->ident_lo;
        cyc = p->cyclic;
        dtype = p->domain_type;
        mispot = p->misbinding_pot;
        rngmode = p->rng_mode;
        seed = p->seed;
        fb_flags = lmask | (cyc ? 1 : 0) << 8 | (dtype ? 1 : 0) << 9 | (p->stack_one ? 1 : 0) << 10;
        load_scalars();
        select_tables();
        rng_block = -1;
        six_d = -1;
    }

#define LDO_WAVE_SCALARS(F) \
    F(step) F(energy) F(hyb_h) F(hyb_s) F(stack_e) F(modifier) F(delta_e) F(bias) F(new_bias) \
    F(new_modifier) F(tape_pos) F(visited) F(site_empty) F(site_bind) F(commits) \
    F(learned_step) F(num_domains) F(num_staples) F(num_bound) F(num_fully) F(num_self) \
    F(num_unassigned) F(num_stacked) F(current_c_i) F(n_chains) F(status) F(violated) \
    F(temp_slot) F(init_slot) F(n_free) F(n_modified) F(n_assigned) F(n_added) F(rejected) \
    F(regrow_old) F(insertion_sites) F(kind) F(n_active) F(n_active0) F(rng_idx) F(rng_sub) \
    F(trk_type) F(trk_ins) F(trk_nost) F(trk_len) F(trk_nst) F(last_move) F(last_acc) F(n_rgs) \
    F(er_top) F(er_depth) F(n_jsegs) F(n_jstems) F(n_jdom)
    DEV void load_scalars() {
        LDO_LDS const RepScalars* s = (LDO_LDS const RepScalars*)blk;
#define LDO_LOAD(f) sc.f = uni(s->f);
        LDO_WAVE_SCALARS(LDO_LOAD)
#undef LDO_LOAD
        sc.attempts.p = blk + offsetof(RepScalars, attempts);
        sc.accepts.p = blk + offsetof(RepScalars, accepts);
        sc.added.p = blk + offsetof(RepScalars, added);
    }
    // back to the block's head (in LDS), and the window's stored biases
    DEV void store_scalars() {
        LDO_LDS RepScalars* s = (LDO_LDS RepScalars*)blk;
#define LDO_STORE(f) s->f = sc.f;
        LDO_WAVE_SCALARS(LDO_STORE)
#undef LDO_STORE
        if (w_on && plane() == 0) {
            double* st = P->win_stored + 2 * S->temp_slot;
            st[0] = w_st0;
            st[1] = w_st1;
        }
    }

    // tables, initiation energy and window of the replica's ladder slot
    DEV void select_tables() {
        size_t n2 = (size_t)n_ident * n_ident;
        t_hyb = P->hyb_e + (size_t)S->temp_slot * n2;
        t_stack = P->stack + (size_t)S->temp_slot * n2;
        init_e = P->init_e[S->init_slot];
        // the scaffold's first domain stands for every identity
        size_t i0 = (size_t)(int16_t)dident[0];
        stack_all = t_stack[i0 * n_ident + i0];
        for (int i = plane(); i < n_ident; i += width) {
            int c = -(i + ident_lo) - ident_lo; // index of identity -(i + lo)
            double e = (c >= 0 && c < n_ident) ? t_hyb[(size_t)i * n_ident + c] : 0.0;
            *(LDO_LDS double*)(full.p + 8 * i) = e;
        }
        w_on = P->windows != nullptr ? 1 : 0;
        w_last = -1;
        w_grid = 0;
        if (w_on) {
            const ldo_window& w = P->windows[S->temp_slot];
            w_op = uni(w.op);
            w_min = uni(w.min_op);
            w_max = uni(w.max_op);
            w_well = w.well_bias;
            w_minb = w.min_bias;
            w_slope = w.slope;
            w_off = w.off_grid_bias;
            w_mult = w.bias_mult;
            w_st0 = P->win_stored[2 * S->temp_slot];
            w_st1 = P->win_stored[2 * S->temp_slot + 1];
        }
    }

    DEV void push_modified(int s) {
        if (S->n_modified >= 2 * nslots) {
            fail(ST_CAPACITY);
            return;
        }
        modified[S->n_modified++] = (int16_t)s;
    }
    DEV void push_assigned(int s) {
        if (S->n_assigned >= 2 * nslots) {
            fail(ST_CAPACITY);
            return;
        }
        assigned[S->n_assigned++] = (int16_t)s;
    }
    DEV void fail(int code) {
        if (S->status == ST_OK) {
            S->status = code;
        }
    }

    // ------------------------------------------------------------ rng
    // Eng::philox64's draws of one step, 64 at a time: lane l holds draw
    // 64 rng_block + l.  A step takes some ten draws one after the other; one
    // evaluation gives them all for the time of one.
    DEV uint64_t philox_draw(uint32_t idx) const {
        uint64_t ctr = S->rng_sub ? (uint64_t)S->learned_step : (uint64_t)S->step;
        uint32_t c0 = idx, c1 = (uint32_t)S->rng_sub;
        uint32_t c2 = (uint32_t)ctr, c3 = (uint32_t)(ctr >> 32);
        uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)rep;
#pragma unroll
        for (int r = 0; r < 10; r++) {
            uint64_t p0 = (uint64_t)0xD2511F53u * c0;
            uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
            uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
            uint32_t n1 = (uint32_t)p1;
            uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
            uint32_t n3 = (uint32_t)p0;
            c0 = n0;
            c1 = n1;
            c2 = n2;
            c3 = n3;
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        return (uint64_t)c0 | ((uint64_t)c1 << 32);
    }
    DEV void rng_begin() {
        S->rng_idx = 0;
        rng_block = -1;
        six_d = -1; // a new move's segments and endpoints
    }
    DEV uint64_t philox64() {
        int i = S->rng_idx++;
#ifdef __HIP_DEVICE_COMPILE__
        if ((i >> 6) != rng_block) {
            rng_block = i >> 6;
            rng_draw = philox_draw((uint32_t)(i & ~63) + (uint32_t)plane());
        }
        uint32_t lo = (uint32_t)lane_int((int)(uint32_t)rng_draw, i & 63);
        uint32_t hi = (uint32_t)lane_int((int)(uint32_t)(rng_draw >> 32), i & 63);
        return (uint64_t)lo | (uint64_t)hi << 32;
#else
        return philox_draw((uint32_t)i);
#endif
    }
    DEV uint64_t tape_next() {
        int64_t pos = S->tape_pos;
        if (pos >= P->tape_len[rep]) {
            fail(ST_TAPE);
            return 0;
        }
        S->tape_pos = pos + 1;
        return uni(P->tapes[P->tape_off[rep] + pos]);
    }
    DEV double uniform_real() {
        if (rngmode == 1) {
            return bits_to_double(tape_next());
        }
        return (double)(philox64() >> 11) * 0x1.0p-53;
    }
    DEV int uniform_int(int lo, int hi) {
        if (rngmode == 1) {
            return (int)(int64_t)tape_next();
        }
        uint32_t x = (uint32_t)(philox64() >> 32);
        uint32_t n = (uint32_t)(hi - lo + 1);
        return lo + (int)(uint32_t)(((uint64_t)x * n) >> 32);
    }

    // ------------------------------------------------------------ slots
    DEV int cslot_of(int s) const { return s < ns ? 0 : 1 + ((s - ns) >> lshift); }
    DEV int d_of(int s) const { return s < ns ? s : ((s - ns) & lmask); }
    DEV int slot(int cs, int d) const { return cs == 0 ? d : ns + ((cs - 1) << lshift) + d; }
    DEV int fwd(int s) const {
        if (s < 0) {
            return LDO_NONE;
        }
        if (s < ns) {
            return s + 1 < ns ? s + 1 : (cyc ? 0 : LDO_NONE);
        }
        return d_of(s) + 1 < ch[cslot_of(s)].len ? s + 1 : LDO_NONE;
    }
    DEV int bwd(int s) const {
        if (s < 0) {
            return LDO_NONE;
        }
        if (s < ns) {
            return s > 0 ? s - 1 : (cyc ? ns - 1 : LDO_NONE);
        }
        return d_of(s) > 0 ? s - 1 : LDO_NONE;
    }
    // Domain::operator+ (domain.cpp:9-31), one step
    DEV int walk(int s, int incr) const { return incr > 0 ? fwd(s) : bwd(s); }

    // a domain's record in one read
    DEV FbRec rec(int s) const {
        Quad v = *(LDO_LDS const Quad*)(dom.p + s * 16);
        return FbRec {uni((int32_t)v.x), uni((int32_t)v.y), uni((int32_t)v.z), uni(v.w)};
    }
    DEV void put_rec(int s, I3 p, uint32_t w) const {
        *(LDO_LDS Quad*)(dom.p + s * 16) =
            Quad {(uint32_t)p.x, (uint32_t)p.y, (uint32_t)p.z, w};
    }
    static DEV uint32_t pack(int ore, int state, int bound) {
        return (uint32_t)ore | (uint32_t)state << 8 | (uint32_t)(uint16_t)bound << 16;
    }
    // state and partner of slot s, the orientation left as it is
    DEV void put_state(int s, int state, int bound) const {
        *(LDO_LDS int8_t*)(dom.p + s * 16 + 13) = (int8_t)state;
        *(LDO_LDS int16_t*)(dom.p + s * 16 + 14) = (int16_t)bound;
    }
    DEV I3 pos(int s) const {
        FbRec r = rec(s);
        return i3(r.x, r.y, r.z);
    }
    DEV int ident_of(int s) const { return dident[s] + ident_lo; }
    // prev[s] = the domain's position and orientation
    DEV void save_prev(int s) const {
        Quad v = *(LDO_LDS const Quad*)(dom.p + s * 16);
        v.w &= 0xFFu;
        *(LDO_LDS Quad*)(prev.p + s * 16) = v;
    }
    // binding energy of s and t; `comp`: their identities are complementary
    DEV double hyb(int s, int t, bool comp) const {
        int a = dident[s];
        return comp ? (double)full[a] : t_hyb[(size_t)a * n_ident + (int)dident[t]];
    }

    // FourBody terms of the bound pair (di, dj).  Without a bound chain
    // neighbour of either there is none, which four lanes see in one read.
    // `trial`: the sum does not matter when a constraint is violated.
    DEV FbOut fb_terms(int di, int dj, bool trial = false) const {
#ifdef __HIP_DEVICE_COMPILE__
        // lanes 0, 1: the slots before and after di; 2, 3: dj's
        int l = plane();
        int base = l < 2 ? di : dj;
        int n = base + ((l & 1) ? 1 : -1);
        bool has;
        if (base < ns) {
            has = (n >= 0 && n < ns) || cyc;
            n = n < 0 ? ns - 1 : (n >= ns ? 0 : n);
        }
        else {
            has = ((base - ns) & lmask) != ((l & 1) ? lmask : 0);
        }
        n = has && l < 4 ? n : 0;
        int st = *(LDO_LDS const int8_t*)(dom.p + n * 16 + 13);
        if (ballot(has && l < 4 && st == OCC_BOUND) == 0) {
            return FbOut {0.0, 0, 0};
        }
#endif
        FbArgs g {dom.p, dident.p, t_stack, stack_all, fb_flags, ns, n_ident};
        FbOut o = (fb_flags >> 10) & 1
                      ? (dtype == 0 ? wave_fb_terms<true, true>(g, di, dj)
                                    : wave_fb_terms<false, true>(g, di, dj))
                      : (dtype == 0 ? wave_fb_terms<true, false>(g, di, dj)
                                    : wave_fb_terms<false, false>(g, di, dj));
        o.st = uni(o.st);
        o.viol = uni(o.viol);
        if (o.viol && !trial) {
            o = wave_fb_walk(g, di, dj);
            o.st = uni(o.st);
        }
        return o;
    }

    // ------------------------------------------------------------ site hash
    // The site's entry, found by 64 lanes reading 64 entries from its home on.
    DEV Site find(I3 p) {
        Site t;
        t.occ = OCC_UNASSIGNED;
        t.s = -1;
        t.at = -1;
        t.w = 0;
        int h = t.home = site_home(p.x, p.y, p.z, hbits);
#ifdef __HIP_DEVICE_COMPILE__
        for (int base = 0; base <= hmask; base += 64) {
            uint32_t v = hash.lane((h + base + plane()) & hmask);
            uint64_t free = ballot(v == LDO_HASH_EMPTY);
            uint64_t m = ballot((int)(v >> 16) == h);
            if (free) {
                m &= (free & -free) - 1;
            }
            for (; m; m &= m - 1) {
                int l = __builtin_ctzll(m);
                int s = lane_int((int)v, l) & 0xFFFF;
                FbRec r = rec(s);
                if (r.x == p.x && r.y == p.y && r.z == p.z) {
                    t.occ = r.state();
                    t.s = s;
                    t.at = (h + base + l) & hmask;
                    t.w = r.w;
                    return t;
                }
            }
            if (free) {
                t.at = (h + base + __builtin_ctzll(free)) & hmask;
                return t;
            }
        }
        return t;
#else
        for (int n = 0; n <= hmask; n++) {
            int i = (h + n) & hmask;
            uint32_t v = hash[i];
            if (v == LDO_HASH_EMPTY) {
                t.at = i;
                return t;
            }
            if ((int)(v >> 16) == h) {
                FbRec r = rec((int)(v & 0xFFFFu));
                if (r.x == p.x && r.y == p.y && r.z == p.z) {
                    t.occ = r.state();
                    t.s = (int)(v & 0xFFFFu);
                    t.at = i;
                    t.w = r.w;
                    return t;
                }
            }
        }
        return t;
#endif
    }
    DEV int occupancy(I3 p) { return find(p).occ; }
    DEV int unbound_at(I3 p) {
        Site t = find(p);
        if (t.s < 0) {
            fail(ST_CONSTRAINT);
            return 0;
        }
        return t.s;
    }
    // index of the entry of domain s (home h), or of its partner's; -1: none
    DEV int entry_of(int h, int s, int t) const {
        uint32_t a = (uint32_t)h << 16 | (uint32_t)s, b = (uint32_t)h << 16 | (uint32_t)(t & 0xFFFF);
#ifdef __HIP_DEVICE_COMPILE__
        for (int base = 0; base <= hmask; base += 64) {
            uint32_t v = hash.lane((h + base + plane()) & hmask);
            uint64_t m = ballot(v == a || v == b);
            if (m) {
                return (h + base + __builtin_ctzll(m)) & hmask;
            }
            if (ballot(v == LDO_HASH_EMPTY)) {
                return -1;
            }
        }
#else
        for (int n = 0; n <= hmask; n++) {
            uint32_t v = hash[(h + n) & hmask];
            if (v == a || v == b) {
                return (h + n) & hmask;
            }
            if (v == LDO_HASH_EMPTY) {
                return -1;
            }
        }
#endif
        return -1;
    }
    // takes the entry of domain s (home h) out: linear probing with backward
    // shift (Knuth, TAOCP 6.4 Alg. R).  The window that finds the entry mostly
    // shows that the next one is free.
    DEV void erase(int h, int s) {
        int i = -1;
#ifdef __HIP_DEVICE_COMPILE__
        uint32_t a = (uint32_t)h << 16 | (uint32_t)s;
        for (int base = 0; base <= hmask; base += 64) {
            uint32_t v = hash.lane((h + base + plane()) & hmask);
            uint64_t m = ballot(v == a), free = ballot(v == LDO_HASH_EMPTY);
            if (m) {
                i = (h + base + __builtin_ctzll(m)) & hmask;
                if (free & (m << 1)) {
                    hash[i] = LDO_HASH_EMPTY;
                    return;
                }
                break;
            }
            if (free) {
                break;
            }
        }
#else
        i = entry_of(h, s, s);
#endif
        if (i < 0) {
            return;
        }
        int j = i;
        for (int n = 0; n <= hmask; n++) {
            j = (j + 1) & hmask;
            uint32_t v = hash[j];
            if (v == LDO_HASH_EMPTY) {
                break;
            }
            int k = (int)(v >> 16);
            if (((k - i - 1) & hmask) < ((j - i) & hmask)) {
                continue; // its home lies past i
            }
            hash[i] = v;
            i = j;
        }
        hash[i] = LDO_HASH_EMPTY;
    }
    DEV void check_coord(I3 p) {
        constexpr uint32_t lim = 2 * LDO_COORD_OFFSET - 5;
        uint32_t x = (uint32_t)(p.x + LDO_COORD_OFFSET - 3), y = (uint32_t)(p.y + LDO_COORD_OFFSET - 3),
                 z = (uint32_t)(p.z + LDO_COORD_OFFSET - 3);
        if (x >= lim || y >= lim || z >= lim) {
            fail(ST_COORD);
        }
    }

    // ------------------------------------------------- domain operations
    // The domain operations of engine_system.h on one lookup and one record
    // read each.
    // update_occupancies of s at site t (origami_system.cpp:770-806) with its
    // record; returns its state, UNASSIGNED where the site is full
    DEV int occupy(int s, I3 p, int o, const Site& t, bool comp) {
        six_d = -1;
        check_coord(p);
        if (t.occ == OCC_UNASSIGNED) {
            if (t.at < 0) {
                fail(ST_CAPACITY);
                return OCC_UNASSIGNED;
            }
            put_rec(s, p, pack(o, OCC_UNBOUND, LDO_NONE));
            hash[t.at] = (uint32_t)t.home << 16 | (uint32_t)s;
            return OCC_UNBOUND;
        }
        if (t.occ != OCC_UNBOUND) {
            dom[s].x = p.x;
            dom[s].y = p.y;
            dom[s].z = p.z;
            dom[s].ore = (int8_t)o;
            fail(ST_CONSTRAINT);
            return OCC_UNASSIGNED;
        }
        int st = comp ? OCC_BOUND : OCC_MISBOUND;
        put_rec(s, p, pack(o, st, t.s));
        put_state(t.s, st, s);
        hash[t.at] = (uint32_t)t.home << 16 | (uint32_t)s;
        return st;
    }
    DEV void count_bound(int s, int t, bool comp, int n) {
        S->num_bound += n;
        if (comp) {
            S->num_fully += n;
        }
        else if (cslot_of(s) == cslot_of(t)) {
            S->num_self += n;
        }
    }
    // OrigamiSystem::set_checked_domain_config (:478-515) at a site looked
    // up before.  `scored`: de and st are the site's energy and stacked pairs
    // as a trial of this configuration found them.
    DEV double set_checked_at(int s, I3 p, int o, const Site& t, bool scored, double de, int st) {
        bool comp = t.occ == OCC_UNBOUND && ident_of(s) == -ident_of(t.s);
        int now = occupy(s, p, o, t, comp);
        if (now == OCC_UNBOUND || now == OCC_UNASSIGNED) {
            de = 0;
        }
        else {
            count_bound(s, t.s, comp, 1);
            if (!scored) {
                de = hyb(s, t.s, comp);
                st = 0;
                if (comp) {
                    FbOut f = fb_terms(s, t.s);
                    de += f.e;
                    st = f.st;
                }
            }
            if (comp) {
                S->site_bind++;
                S->num_stacked += st;
            }
        }
        S->energy += de;
        S->num_unassigned--;
        S->commits++;
        return de;
    }
    DEV double set_checked_domain_config(int s, I3 p, int o) {
        return set_checked_at(s, p, o, find(p), false, 0.0, 0);
    }
    // bind_domain (:1282-1312) of an unassigned domain s on the unbound
    // occupant of site t: whether it may bind, its energy and stacked pairs.
    // The pair's records are left as they were but for s's position and
    // orientation.
    DEV bool try_bind(int s, I3 p, int o, const Site& t, bool comp, double& de, int& st) {
        S->site_bind++;
        de = 0;
        st = 0;
        bool opposed = o == (int)((t.w & 0xFFu) ^ 1u);
        if (!comp || !opposed) {
            put_rec(s, p, pack(o, OCC_UNASSIGNED, LDO_NONE));
        }
        if (!comp) {
            if (mispot == 0 && opposed) {
                de = hyb(s, t.s, false);
                return true;
            }
            return false;
        }
        if (!opposed) {
            return false;
        }
        put_rec(s, p, pack(o, OCC_BOUND, t.s));
        put_state(t.s, OCC_BOUND, s);
        FbOut f = fb_terms(s, t.s, true);
        put_state(s, OCC_UNASSIGNED, LDO_NONE);
        put_state(t.s, OCC_UNBOUND, LDO_NONE);
        if (f.viol) {
            return false;
        }
        de = f.e + hyb(s, t.s, true);
        st = f.st;
        return true;
    }
    // OrigamiSystem::check_domain_constraints (:343-355) of an unassigned
    // domain
    DEV double check_domain_constraints(int s, I3 p, int o) {
        Site t = find(p);
        if (t.occ == OCC_UNASSIGNED) {
            // a trial leaves its position on the unassigned domain
            put_rec(s, p, pack(o, OCC_UNASSIGNED, LDO_NONE));
            S->site_empty++;
            return 0;
        }
        if (t.occ != OCC_UNBOUND) {
            S->violated = 1;
            return 0;
        }
        double de;
        int st;
        bool ok = try_bind(s, p, o, t, ident_of(s) == -ident_of(t.s), de, st);
        S->violated = ok ? 0 : 1;
        return de;
    }
    // OrigamiSystem::set_domain_config (:517-541)
    DEV double set_domain_config(int s, I3 p, int o) {
        if (dom[s].state != OCC_UNASSIGNED) {
            fail(ST_CONSTRAINT);
            return 0;
        }
        Site t = find(p);
        double de = 0;
        int st = 0;
        bool comp = false;
        if (t.occ == OCC_UNBOUND) {
            comp = ident_of(s) == -ident_of(t.s);
            if (!try_bind(s, p, o, t, comp, de, st)) {
                S->violated = 1;
                return 0;
            }
            S->violated = 0;
            count_bound(s, t.s, comp, 1);
        }
        else if (t.occ == OCC_UNASSIGNED) {
            S->site_empty++;
            if (S->violated) {
                // placed and taken off again
                put_rec(s, p, pack(o, OCC_UNASSIGNED, LDO_NONE));
                check_coord(p);
                return 0;
            }
        }
        else {
            S->violated = 1;
            return 0;
        }
        occupy(s, p, o, t, comp);
        S->energy += de;
        S->num_stacked += st;
        S->num_unassigned--;
        S->commits++;
        return de;
    }
    // OrigamiSystem::unassign_domain (:375-385, 695-760)
    DEV double unassign_domain(int s) {
        six_d = -1;
        FbRec r = rec(s);
        int st = r.state();
        double de = 0;
        if (st == OCC_UNBOUND) {
            erase(site_home(r.x, r.y, r.z, hbits), s);
            put_state(s, OCC_UNASSIGNED, r.bound());
            S->num_unassigned++;
        }
        else if (st != OCC_UNASSIGNED) {
            int t = r.bound();
            bool comp = st == OCC_BOUND;
            count_bound(s, t, comp, -1);
            if (comp) {
                S->site_bind++;
                FbOut f = fb_terms(s, t);
                de = f.e * -1;
                S->num_stacked += f.st * -1;
            }
            de += -hyb(s, t, comp);
            int h = site_home(r.x, r.y, r.z, hbits);
            int i = entry_of(h, s, t);
            if (i >= 0) {
                hash[i] = (uint32_t)h << 16 | (uint32_t)t;
            }
            put_state(s, OCC_UNASSIGNED, LDO_NONE);
            put_state(t, OCC_UNBOUND, LDO_NONE);
            S->energy += de;
            S->num_unassigned++;
        }
        S->commits++;
        return de;
    }
    DEV void set_domain_orientation(int s, int o) {
        if (dom[s].state == OCC_BOUND) {
            S->violated = 1;
        }
        else {
            dom[s].ore = (int8_t)o;
        }
    }

    typedef LRecs<LPosOre, 16> PosList;
#define LDO_WAVE
#undef DEVNI
#define DEVNI __host__ __device__ __forceinline__
#include "engine_decl.h"

#ifdef __HIP_DEVICE_COMPILE__
    __device__ __forceinline__ void count_moves();
    __device__ __forceinline__ void look_six(int d, I3 pp);
    // sg, std_: seg[d] and stem[d]
    __device__ __forceinline__ void walk_six(int d, int sg, int std_);
#endif
    DEV bool agreed(bool b) const { return all_lanes(b); }
    // whether the moveset holds a recoil-growth or jump move: a constant of
    // the kernel, so that the kernels of the standard moveset leave their code out
    bool kinds;
#ifdef __HIP_DEVICE_COMPILE__
    __device__ __forceinline__ int kind_of(int m) const { return lane_int(mv_kind, m); }
    __device__ __forceinline__ int maxreg_of(int m) const { return lane_int(mv_maxreg, m); }
#else
    DEV int kind_of(int m) const { return P->move_kind[m]; }
    DEV int maxreg_of(int m) const { return P->move_maxreg[m]; }
#endif
    DEVIN void rg_look(const RgCur& c);
    DEV bool all_kinds() const { return kinds; }
    DEV int staple_of(int k) const { return LArr<int16_t> {sframes.p}[k]; }
    // enters domain s as the occupant of site p
    DEV void hput(I3 p, int s) {
        check_coord(p);
        Site t = find(p);
        if (t.at < 0) {
            fail(ST_CAPACITY);
            return;
        }
        hash[t.at] = (uint32_t)t.home << 16 | (uint32_t)s;
    }
    // Endpoint i of a list: lane by lane, or one for all lanes
    DEV Endpoint ep_read(lds_t l, int64_t off, int i) const {
        Endpoint e;
        if (i < LDO_WAVE_EP) {
            LDO_LDS const Endpoint* q = (LDO_LDS const Endpoint*)(l + i * (int)sizeof(Endpoint));
            e.cslot = q->cslot;
            e.d = q->d;
            e.seg = q->seg;
            e.x = q->x;
            e.y = q->y;
            e.z = q->z;
        }
        else {
            e = ((const Endpoint*)(gblk + off))[i];
        }
        return e;
    }
    DEV void ep_write(lds_t l, int64_t off, int i, const Endpoint& e) const {
        if (i < LDO_WAVE_EP) {
            LDO_LDS Endpoint* q = (LDO_LDS Endpoint*)(l + i * (int)sizeof(Endpoint));
            q->cslot = e.cslot;
            q->d = e.d;
            q->seg = e.seg;
            q->x = e.x;
            q->y = e.y;
            q->z = e.z;
        }
        else {
            ((Endpoint*)(gblk + off))[i] = e;
        }
    }
    DEV Endpoint active_at(int i) const { return ep_read(ep, P->L.off_active, i); }
    DEV void active_put(int i, const Endpoint& e) const { ep_write(ep, P->L.off_active, i, e); }
    DEV Endpoint active0_at(int i) const { return ep_read(ep0, P->L.off_active0, i); }
    DEV void active0_put(int i, const Endpoint& e) const { ep_write(ep0, P->L.off_active0, i, e); }
};

#undef LDO_ENG
#define LDO_ENG WEng
#include "engine_system.h"
#include "engine_moves.h"

// ------------------------------------------------------------ chain lists
// OrigamiSystem::add_chain(ident, index) (:402-443) for a staple
DEVNI int WEng::add_chain_with(int ident, int uid) {
    if (S->n_free == 0) {
        fail(ST_CAPACITY);
        return -1;
    }
    int cs = freel[--S->n_free];
    int tc = tcount[ident];
    if (tc >= P->L.tcap) {
        fail(ST_CAPACITY);
        return -1;
    }
    int len = uni(P->type_len[ident]);
    // one domain per lane
    int s0 = slot(cs, 0);
    for (int d = plane(); d < len; d += width) {
        *(LDO_LDS int16_t*)(dident.p + 2 * (s0 + d)) =
            P->type_ident[ident * P->type_ident_stride + d];
        put_rec(s0 + d, i3(0, 0, 0), pack(0, OCC_UNASSIGNED, LDO_NONE));
    }
    tlist[ident * P->L.tcap + tc] = (int16_t)cs;
    tcount[ident] = (int16_t)(tc + 1);
    ch[cs].uid = uid;
    ch[cs].ident = (int16_t)ident;
    ch[cs].len = (int16_t)len;
    order[S->n_chains++] = (int16_t)cs;
    S->num_staples++;
    S->num_domains += len;
    S->num_unassigned += len;
    return cs;
}

// takes the first entry equal to v out of the n entries at a
DEV void wave_list_remove(LArr<int16_t> a, int n, int v) {
#ifdef __HIP_DEVICE_COMPILE__
    int at = -1;
    for (int base = 0; base < n; base += 64) {
        int i = base + (int)(threadIdx.x & 63u);
        int x = i < n ? (int)a.lane(i) : -1;
        if (at < 0) {
            uint64_t m = __builtin_amdgcn_ballot_w64(i < n && x == v);
            at = m ? base + __builtin_ctzll(m) : -1;
        }
        if (at >= 0 && i > at && i < n) {
            *(LDO_LDS int16_t*)(a.p + 2 * (i - 1)) = (int16_t)x;
        }
    }
#else
    int k = 0;
    while (k < n && a[k] != v) {
        k++;
    }
    for (; k + 1 < n; k++) {
        a[k] = a[k + 1];
    }
#endif
}

// OrigamiSystem::delete_chain (:445-472)
DEVNI void WEng::delete_chain(int cs) {
    int ident = ch[cs].ident;
    int tc = tcount[ident];
    wave_list_remove(order, S->n_chains, cs);
    wave_list_remove(tlist + ident * P->L.tcap, tc, cs);
    tcount[ident] = (int16_t)(tc - 1);
    S->n_chains--;
    int len = ch[cs].len;
    S->num_domains -= len;
    S->num_staples--;
    S->num_unassigned -= len;
    ch[cs].ident = -1;
    freel[S->n_free++] = (int16_t)cs;
    S->energy -= init_e;
}

// MCMovetype::select_random_domain (movetypes.cpp:98-113): the scaffold comes
// first in the working order, then 64 staples at a time; their lengths (at
// most 8) are summed bit by bit
DEVIN int WEng::select_random_domain() {
    int idx = uniform_int(0, S->num_domains - 1);
    if (idx < ns) {
        return idx;
    }
    idx -= ns;
    int n = S->n_chains;
#ifdef __HIP_DEVICE_COMPILE__
    for (int base = 1; base < n; base += 64) {
        int w = base + plane();
        int cs = 0, len = 0;
        if (w < n) {
            cs = order.lane(w);
            len = *(LDO_LDS const int16_t*)(ch.p + cs * 8 + 6);
        }
        int before = 0, total = 0;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            uint64_t m = ballot((len >> b) & 1);
            before += below(m) << b;
            total += __builtin_popcountll(m) << b;
        }
        uint64_t hit = ballot(idx >= before && idx < before + len);
        if (hit) {
            int l = __builtin_ctzll(hit);
            return slot(lane_int(cs, l), idx - lane_int(before, l));
        }
        idx -= total;
    }
#else
    for (int w = 1; w < n; w++) {
        int cs = order[w], len = ch[cs].len;
        if (idx < len) {
            return slot(cs, idx);
        }
        idx -= len;
    }
#endif
    return LDO_NONE;
}

// MCMovetype::test_acceptance (movetypes.cpp:142-158)
DEVIN bool WEng::test_acceptance(double p_ratio) {
    double p_accept = fmin(1.0, p_ratio) * S->modifier;
    if (all_lanes(p_accept == 1)) {
        return true;
    }
    return all_lanes(p_accept > uniform_real());
}

// test_config_open (rg_movetypes.cpp:345-361)
DEVIN bool WEng::rg_test_open(double p) {
    p = fmin(1.0, p);
    if (all_lanes(p == 1)) {
        return true;
    }
    return all_lanes(p > uniform_real());
}

// ------------------------------------------------------------- CTCB growth
// Eng::ctcb_grow_chain_scaffold with the level being grown in registers: the
// stack in LDS is touched when a staple is entered or left.
DEVNI void WEng::ctcb_grow_chain_scaffold(int first, int count, int dir, bool first_gp) {
    int sp = 0;
    GrowFrame f;
    f.first = (int16_t)first;
    f.count = (int16_t)count;
    f.i = 1;
    f.prev = (int16_t)first;
    f.gold = 0;
    f.gnew = 0;
    f.dir = (int8_t)dir;
    f.kind = 0;
    f.phase = 0;
    f.pad = 0;
    bool have = count > 1;
    int enter = -1; // growthpoint to descend at
    if (first_gp && gp[first] >= 0) {
        enter = first;
    }
    while (S->status == ST_OK && !S->rejected) {
        if (enter >= 0) {
            if (have) {
                if (sp + 1 >= LDO_GROW_DEPTH) {
                    fail(ST_CAPACITY);
                    break;
                }
                gstack[sp++] = f;
            }
            have = true;
            f.gold = (int16_t)enter;
            f.kind = 1;
            f.phase = 0;
            enter = -1;
        }
        if (!have) {
            if (sp == 0) {
                break;
            }
            LGrowFrame g = gstack[--sp];
            f.first = g.first;
            f.count = g.count;
            f.i = g.i;
            f.prev = g.prev;
            f.gold = g.gold;
            f.gnew = g.gnew;
            f.dir = g.dir;
            f.kind = g.kind;
            f.phase = g.phase;
            have = true;
        }
        if (f.kind == 0) {
            if (f.i >= f.count) {
                have = false;
                continue;
            }
            int d = walk(f.prev, f.dir);
            int sd = seg[d], gd = gp[d], ed = inact[d];
            if (sd < 0) {
                seg[d] = 0; // get_dir's map insertion (top_constraint_points.cpp:179-185)
            }
            cb_select_and_set(d, f.prev);
            if (S->rejected) {
                break;
            }
            cp_remove_active(d);
            if (ed >= 0) {
                cp_add_active(ed, pos(d), seg[ed]);
            }
            f.prev = (int16_t)d;
            f.i++;
            enter = gd >= 0 ? d : -1;
            continue;
        }
        // staple growth from growthpoint f.gold: the growthpoint itself, then
        // the two ways from it
        if (f.phase == 2) {
            have = false;
            continue;
        }
        if (f.phase == 0) {
            int gnew = gp[f.gold];
            if (cslot_of(gnew) == 0) {
                have = false;
                continue;
            }
            if (S->regrow_old) {
                cb_set_old_growth_point(gnew, f.gold);
            }
            else {
                double de = set_growth_point(gnew, f.gold);
                S->bias *= exp(-de);
            }
            if (S->rejected) {
                break;
            }
            cp_update_endpoints(gnew);
            f.gnew = (int16_t)gnew;
        }
        int di = d_of(f.gnew);
        int n = f.phase == 0 ? ch[cslot_of(f.gnew)].len - di : di + 1;
        int way = f.phase == 0 ? 1 : -1;
        f.phase++;
        if (n > 1) {
            if (sp + 1 >= LDO_GROW_DEPTH) {
                fail(ST_CAPACITY);
                break;
            }
            gstack[sp++] = f;
            f.first = f.gnew;
            f.count = (int16_t)n;
            f.i = 1;
            f.prev = f.gnew;
            f.dir = (int8_t)way;
            f.kind = 0;
            f.phase = 0;
        }
    }
}

// ------------------------------------------------------ CTRG configurations
// the sites around the level's chain neighbour, before its attempts
DEVIN void WEng::rg_look(const RgCur& c) {
#ifdef __HIP_DEVICE_COMPILE__
    if (!c.stemd && six_d != c.d) {
        look_six(c.d, pos(c.ref));
        walk_six(c.d, seg[c.d], stem[c.d]);
    }
#endif
}

// select_trial_config (rg_movetypes.cpp:298-313): the k-th configuration left
// is the set bit with k below it
DEVIN void WEng::rg_select(RgCur& c, I3& p, int& o) {
    if (c.stemd) {
        FbRec r = rec(c.ref);
        p = i3(r.x, r.y, r.z);
        o = r.ore() ^ 1;
        return;
    }
    int k = uniform_int(0, __builtin_popcountll(c.avail) - 1);
#ifdef __HIP_DEVICE_COMPILE__
    int i = __builtin_ctzll(ballot(((c.avail >> plane()) & 1) && below(c.avail) == k));
#else
    int i = 0;
    for (uint64_t m = c.avail;; m &= m - 1) {
        if (k-- == 0) {
            i = __builtin_ctzll(m);
            break;
        }
    }
#endif
    c.avail &= ~(1ull << i);
    p = add3(pos(c.ref), unit3(i / 6));
    o = i % 6;
}

// calc_p_config_open (rg_movetypes.cpp:315-343)
DEVNI double WEng::rg_p_open(const RgCur& c, I3 p, int o) {
#ifdef __HIP_DEVICE_COMPILE__
    if (!c.stemd && six_d == c.d) {
        uint64_t at = ballot((six_p.x == p.x) & (six_p.y == p.y) & (six_p.z == p.z)) &
                      0x0000010101010101ull;
        if (at) {
            if (at & six_empty) {
                put_rec(c.d, p, pack(o, OCC_UNASSIGNED, LDO_NONE));
                S->site_empty++;
                return at & six_walk ? 1.0 : 0.0;
            }
            if (at & six_full) {
                return 0;
            }
            int l = __builtin_ctzll(at);
            Site t;
            t.occ = OCC_UNBOUND;
            t.s = lane_int(six_s, l);
            t.at = lane_int(six_at, l);
            t.home = lane_int(six_h, l);
            t.w = (uint32_t)lane_int((int)six_w, l);
            double de;
            int st;
            if (!try_bind(c.d, p, o, t, ident_of(c.d) == -ident_of(t.s), de, st) ||
                !(at & six_walk) ||
                !(cslot_of(t.s) == cslot_of(c.d) || (at & six_ends) != 0)) {
                return 0;
            }
            return fmin(1.0, exp(-de));
        }
    }
#endif
    double de = check_domain_constraints(c.d, p, o);
    if (S->violated) {
        S->violated = 0;
        return 0;
    }
    if (!cp_walks_remain(c.d, p)) {
        return 0;
    }
    Site t = find(p);
    if (t.occ == OCC_UNBOUND) {
        bool same_chain = cslot_of(t.s) == cslot_of(c.d);
        bool endpoint = cp_endpoint_reached(c.d, p);
        if (!(same_chain || endpoint || c.stemd)) {
            return 0;
        }
    }
    return fmin(1.0, exp(-de));
}

// -------------------------------------------------------- trial placement
#ifdef __HIP_DEVICE_COMPILE__
// Looks up the six sites around pp for the unassigned domain d.  Eight lanes
// read eight entries of a site's probe run at once; what the lane with the
// site's entry finds goes to the first of the eight.
__device__ __forceinline__ void WEng::look_six(int d, I3 pp) {
    int lane = plane();
    int v = lane >> 3, j = lane & 7;
    six_d = d;
    six_p = add3(pp, unit3(v));
    six_h = site_home(six_p.x, six_p.y, six_p.z, hbits);
    uint32_t en = hash.lane((six_h + j) & hmask);
    bool site = v < 6;
    // the group's free entries, and this lane's entry if it comes before them
    uint32_t gfree = (uint32_t)(ballot(en == LDO_HASH_EMPTY) >> (lane & 56)) & 255u;
    bool cand = site & ((int)(en >> 16) == six_h) & ((gfree & ((1u << j) - 1)) == 0);
    int s = cand ? (int)(en & 0xFFFFu) : 0;
    Quad r = *(LDO_LDS const Quad*)(dom.p + s * 16);
    bool hit = cand & ((int)r.x == six_p.x) & ((int)r.y == six_p.y) & ((int)r.z == six_p.z);
    uint32_t ghit = (uint32_t)(ballot(hit) >> (lane & 56)) & 255u;
    int src = ((lane & 56) | __builtin_ctz(ghit | 256u)) << 2;
    six_s = __builtin_amdgcn_ds_bpermute(src, s);
    six_w = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)r.w);
    six_at = (six_h + __builtin_ctz((ghit ? ghit : gfree) | 256u)) & hmask;
    bool found = ghit != 0;
    // a probe run longer than eight entries is followed entry by entry
    uint64_t more = ballot(site & (j == 0) & (ghit == 0) & (gfree == 0));
    for (; more; more &= more - 1) {
        int l = __builtin_ctzll(more);
        Site t = find(add3(pp, unit3(l >> 3)));
        bool me = lane == l;
        found = me ? t.s >= 0 : found;
        six_s = me ? (t.s >= 0 ? t.s : 0) : six_s;
        six_w = me ? t.w : six_w;
        six_at = me ? t.at : six_at;
    }
    bool first = site & (j == 0);
    six_empty = ballot(first & !found);
    six_unb = ballot(first & found & ((six_w & 0xFF00u) == (uint32_t)OCC_UNBOUND << 8));
    six_full = ballot(first & found) & ~six_unb;
}

// Of the six sites, those d's remaining walks allow (cp_walks_remain) and
// those that are an endpoint of d (cp_endpoint_reached): 64 endpoints are read
// at once, and each that concerns d's chain and segment is held against all
// six sites.
__device__ __forceinline__ void WEng::walk_six(int d, int sg, int std_) {
    int n = S->n_active;
    six_walk = ~0ull;
    six_ends = 0;
    if (n == 0) {
        return;
    }
    int sg2 = -2, sw = sg;
    if (std_ >= 0) {
        // a scaffold stem of a jump is held by its own pair of segments, any
        // other stem by none
        bool held = S->n_jsegs != 0 && cslot_of(d) == 0 && stemseg[d] >= 0;
        sw = held ? (int)stemseg[d] : -2;
        sg2 = held ? sw + 1 : -2;
    }
    int cs = cslot_of(d), dd = d_of(d);
    uint32_t key = (uint32_t)cs | (uint32_t)dd << 16;
    bool bad = false, end = false;
    for (int base = 0; base < n; base += 64) {
        int i = base + plane();
        uint32_t k = 0xFFFFu;
        int es = -1, ex = 0, ey = 0, ez = 0;
        if (base == 0) {
            LDO_LDS const Word* q = (LDO_LDS const Word*)(ep + i * (int)sizeof(Endpoint));
            k = (uint32_t)q[0];
            es = q[1];
            ex = q[2];
            ey = q[3];
            ez = q[4];
        }
        else if (i < n) {
            Endpoint e = active_at(i);
            k = (uint32_t)(uint16_t)e.cslot | (uint32_t)(uint16_t)e.d << 16;
            es = e.seg;
            ex = e.x;
            ey = e.y;
            ez = e.z;
        }
        bool mine = (i < n) & ((k & 0xFFFFu) == (uint32_t)cs);
        uint64_t m = ballot(mine & ((es == sg) | (es == sw) | (es == sg2)));
        for (; m; m &= m - 1) {
            int l = __builtin_ctzll(m);
            uint32_t ke = (uint32_t)lane_int((int)k, l);
            int se = lane_int(es, l), ed = (int)(ke >> 16);
            int ax = lane_int(ex, l) - six_p.x, ay = lane_int(ey, l) - six_p.y,
                az = lane_int(ez, l) - six_p.z;
            int l1 = (ax < 0 ? -ax : ax) + (ay < 0 ? -ay : ay) + (az < 0 ? -az : az);
            end = end | ((se == sg) & (ke == key) & (l1 == 0));
            if (se == sw || se == sg2) {
                int steps = ed > dd ? ed - dd : dd - ed;
                if (cyc && cs == 0) {
                    int dir = cp_seg_dir(cs, se);
                    if (dir > 0 && ed < dd) {
                        steps = ns + ed - dd;
                    }
                    else if (dir < 0 && ed > dd) {
                        steps = dd + ns - ed;
                    }
                    else if (dir == 0) {
                        steps = 0;
                    }
                }
                bad = bad | (l1 > steps) | (((steps - l1) & 1) != 0);
            }
        }
    }
    six_walk = ~ballot(bad);
    six_ends = ballot(end);
}
#endif

// CBMCMovetype::calc_biases + calc_bias + select_and_set_config
// (cb_movetypes.cpp:58-166, 363-387, 486-539).  The lane of each site carries
// it: table reads, exp and division run on all sites at once, and only a
// complementary occupant's FourBody checks are made site by site.  Lanes are
// in site order, so sums and the selection go in the reference's order (a site
// that is no candidate adds zero).  d is unassigned: every grower unassigns
// its domains first.
DEVNI void WEng::cb_select_and_set(int d, int prev_d) {
    bool ctcb = S->kind == LDO_MOVE_KIND_CTCB;
    // everything known of d and its neighbour, in one round of reads
    Quad q0 = *(LDO_LDS const Quad*)(dom.p + prev_d * 16);
    int q1 = *(LDO_LDS const int8_t*)(dom.p + d * 16 + 13);
    int q2 = dident.lane(d);
    int q3 = seg.lane(d), q4 = stem.lane(d);
    Quad q5 = *(LDO_LDS const Quad*)(old.p + d * 16);
    I3 pp = i3(uni((int32_t)q0.x), uni((int32_t)q0.y), uni((int32_t)q0.z));
    int id = uni(q2);
    if (uni(q1) != OCC_UNASSIGNED) {
        fail(ST_CONSTRAINT);
        S->rejected = 1;
        return;
    }
#ifdef __HIP_DEVICE_COMPILE__
    int lane = plane();
    look_six(d, pp);
    uint64_t mempty = six_empty, munb = six_unb;
    S->site_empty += __builtin_popcountll(mempty);
    uint64_t mc = mempty; // candidates
    double de = 0;
    int st = 0;
    double wt = 6.0;
    if (munb) {
        int ids = *(LDO_LDS const int16_t*)(dident.p + 2 * six_s);
        bool unb = (munb >> lane) & 1;
        uint64_t mcomp = munb & ballot(id + ident_lo == -(ids + ident_lo));
        uint64_t mmis = munb & ~mcomp;
        S->site_bind += __builtin_popcountll(mmis);
        if (mmis && mispot == 0) {
            // a misbound pair takes the opposing orientation and any energy
            mc |= mmis;
            if ((mmis >> lane) & 1) {
                de = t_hyb[(size_t)id * n_ident + ids];
            }
        }
        for (uint64_t m = mcomp; m; m &= m - 1) {
            int l = __builtin_ctzll(m);
            Site t;
            t.occ = OCC_UNBOUND;
            t.s = lane_int(six_s, l);
            t.at = 0;
            t.home = 0;
            t.w = (uint32_t)lane_int((int)six_w, l);
            double e1;
            int st1;
            if (try_bind(d, add3(pp, unit3(l >> 3)), (int)((t.w & 0xFFu) ^ 1u), t, true, e1, st1)) {
                mc |= 1ull << l;
                de = lane == l ? e1 : de;
                st = lane == l ? st1 : st;
            }
        }
        wt = (unb ? 1.0 : 6.0) * exp(-de);
    }
    uint64_t weigh = mc;
    if (ctcb) {
        walk_six(d, uni(q3), uni(q4));
        weigh &= six_walk;
        // an occupied site takes d only as an endpoint or of its own chain
        if (munb & weigh) {
            weigh &= ~munb | six_ends | ballot(cslot_of(six_s) == cslot_of(d));
        }
    }
    wt = (weigh >> lane) & 1 ? wt : 0.0;
    double sum = 0;
#pragma unroll
    for (int v = 0; v < 6; v++) {
        sum += lane_double(wt, 8 * v);
    }
    if (all_lanes(sum == 0)) {
        // a trial leaves its position on the unassigned domain
        if (mempty | munb) {
            int l = 63 - __builtin_clzll(mempty | munb);
            int o = (munb >> l) & 1 ? (lane_int((int)six_w, l) & 0xFF) ^ 1 : 0;
            put_rec(d, add3(pp, unit3(l >> 3)), pack(o, OCC_UNASSIGNED, LDO_NONE));
        }
        S->rejected = 1;
        return;
    }
    S->bias *= sum;
    I3 p;
    int o = -1;
    int l = -1; // the lane that holds the site
    if (!S->regrow_old) {
        double x = uniform_real();
        double part_l = wt / sum;
        double cum = 0, mine = 0;
#pragma unroll
        for (int v = 0; v < 6; v++) {
            cum += lane_double(part_l, 8 * v);
            mine = lane == 8 * v ? cum : mine;
        }
        uint64_t sel = ballot(x < mine) & mc;
        p = i3(0, 0, 0);
        if (sel) {
            l = __builtin_ctzll(sel);
            p = add3(pp, unit3(l >> 3));
            if ((munb >> l) & 1) {
                o = (lane_int((int)six_w, l) & 0xFF) ^ 1;
            }
        }
        if (o < 0) {
            o = uniform_int(0, 5);
        }
    }
    else {
        p = i3(uni((int32_t)q5.x), uni((int32_t)q5.y), uni((int32_t)q5.z));
        o = uni((int32_t)q5.w);
        uint64_t sel = ballot((six_p.x == p.x) & (six_p.y == p.y) & (six_p.z == p.z)) &
                       (mempty | munb | six_full);
        l = sel ? __builtin_ctzll(sel) : -1;
    }
    if (l >= 0) {
        // the lookup, and the trial's energy where it was of this very
        // configuration
        Site t;
        t.w = (uint32_t)lane_int((int)six_w, l);
        t.s = (mempty >> l) & 1 ? -1 : lane_int(six_s, l);
        t.occ = t.s < 0 ? OCC_UNASSIGNED : (int)((t.w >> 8) & 0xFFu);
        t.home = lane_int(six_h, l);
        t.at = lane_int(six_at, l);
        bool scored = ((munb & mc) >> l & 1) && o == (int)((t.w & 0xFFu) ^ 1u);
        set_checked_at(d, p, o, t, scored, lane_double(de, l), lane_int(st, l));
    }
    else {
        set_checked_domain_config(d, p, o);
    }
    push_assigned(d);
#else
    (void)q3;
    (void)q4;
    bool cand[6], unb[6];
    double wt[6], e1[6];
    int core[6], st1[6];
    Site site[6];
    double sum = 0;
    for (int v = 0; v < 6; v++) {
        I3 pn = add3(pp, unit3(v));
        Site t = site[v] = find(pn);
        cand[v] = false;
        unb[v] = t.occ == OCC_UNBOUND;
        core[v] = -1;
        wt[v] = 0;
        if (t.occ == OCC_UNASSIGNED) {
            cand[v] = true;
            put_rec(d, pn, pack(0, OCC_UNASSIGNED, LDO_NONE));
            S->site_empty++;
            wt[v] = 6.0;
        }
        else if (unb[v]) {
            core[v] = (int)((t.w & 0xFFu) ^ 1u);
            bool comp = id + ident_lo == -ident_of(t.s);
            if (try_bind(d, pn, core[v], t, comp, e1[v], st1[v])) {
                cand[v] = true;
                wt[v] = exp(-e1[v]);
            }
        }
        if (ctcb && cand[v]) {
            if (unb[v] && cslot_of(t.s) != cslot_of(d) && !cp_endpoint_reached(d, pn)) {
                wt[v] = 0;
            }
            if (!cp_walks_remain(d, pn)) {
                wt[v] = 0;
            }
        }
        sum += wt[v];
    }
    if (sum == 0) {
        S->rejected = 1;
        return;
    }
    S->bias *= sum;
    I3 p = i3(0, 0, 0);
    int o = -1, sel = -1;
    if (!S->regrow_old) {
        double x = uniform_real(), cum = 0;
        for (int v = 0; v < 6 && sel < 0; v++) {
            if (cand[v]) {
                cum += wt[v] / sum;
                sel = x < cum ? v : -1;
            }
        }
        if (sel >= 0) {
            p = add3(pp, unit3(sel));
            o = core[sel];
        }
        if (o < 0) {
            o = uniform_int(0, 5);
        }
    }
    else {
        p = i3((int32_t)q5.x, (int32_t)q5.y, (int32_t)q5.z);
        o = (int32_t)q5.w;
        for (int v = 0; v < 6; v++) {
            sel = eq3(p, add3(pp, unit3(v))) ? v : sel;
        }
    }
    if (sel >= 0) {
        bool scored = cand[sel] && unb[sel] && o == core[sel];
        set_checked_at(d, p, o, site[sel], scored, scored ? e1[sel] : 0.0, scored ? st1[sel] : 0);
    }
    else {
        set_checked_domain_config(d, p, o);
    }
    push_assigned(d);
#endif
}

// ------------------------------------------------------ active endpoints
// Constraintpoints::add_active_endpoint (:264-278)
DEVIN void WEng::cp_add_active(int s, I3 p, int sg) {
    six_d = -1;
    if (S->n_active >= ecap) {
        fail(ST_CAPACITY);
        return;
    }
    Endpoint e;
    e.cslot = (int16_t)cslot_of(s);
    e.d = (int16_t)d_of(s);
    e.seg = sg;
    e.x = p.x;
    e.y = p.y;
    e.z = p.z;
    active_put(S->n_active++, e);
}

// Constraintpoints::remove_active_endpoint (:299-320); see Eng's
DEVIN void WEng::cp_remove_active(int s, bool rec) {
    six_d = -1;
    int n = S->n_active;
    int k = 0, r = 0;
    int top = rec ? S->er_top : 0;
    int sg = n > 0 ? (int)seg[s] : 0;
    int cs = cslot_of(s), dd = d_of(s);
    for (int base = 0; base < n; base += width) {
        int i = base + plane();
        bool keep = false, drop = false;
        Endpoint e;
#ifdef __HIP_DEVICE_COMPILE__
        if (base == 0) {
            // two words tell which go; mostly none does
            LDO_LDS const Word* q = (LDO_LDS const Word*)(ep + i * (int)sizeof(Endpoint));
            drop = (i < n) & (q[0] == (cs | dd << 16)) & (q[1] == sg);
            if (ballot(drop) == 0) {
                k = n < 64 ? n : 64;
                continue;
            }
        }
#endif
        if (i < n) {
            e = active_at(i);
            keep = !(e.cslot == cs && e.seg == sg && e.d == dd);
            drop = !keep;
        }
#ifdef __HIP_DEVICE_COMPILE__
        uint64_t m = ballot(keep), md = ballot(drop);
        int kb = below(m), rb = below(md);
        int nm = __builtin_popcountll(m), nd = __builtin_popcountll(md);
#else
        int kb = 0, rb = 0, nm = keep ? 1 : 0, nd = drop ? 1 : 0;
#endif
        if (keep && (k != base || nd != 0)) {
            active_put(k + kb, e);
        }
        if (rec && drop) {
            int j = top + r + rb;
            if (j < ecap) {
                LDO_LDS Endpoint* q = (LDO_LDS Endpoint*)(erstk.p + j * (int)sizeof(Endpoint));
                q->cslot = e.cslot;
                q->d = e.d;
                q->seg = e.seg;
                q->x = e.x;
                q->y = e.y;
                q->z = e.z;
            }
        }
        k += nm;
        r += nd;
    }
    S->n_active = k;
    if (rec) {
        if (top + r > ecap || S->er_depth >= nslots) {
            fail(ST_CAPACITY);
            return;
        }
        ercnt[S->er_depth++] = (int16_t)r;
        S->er_top = top + r;
    }
}

// Constraintpoints::remove_activated_endpoint (:322-338): the first active
// endpoint of the inactive-endpoint domain paired with s
DEVIN void WEng::cp_remove_activated(int s) {
    six_d = -1;
    int e = inact[s];
    if (e < 0) {
        return;
    }
    int sg = seg[e];
    int cs = cslot_of(e), dd = d_of(e);
    int n = S->n_active;
    int at = -1;
    for (int base = 0; base < n; base += width) {
        int i = base + plane();
        Endpoint a;
        bool hit = false;
        if (i < n) {
            a = active_at(i);
            hit = a.cslot == cs && a.seg == sg && a.d == dd;
        }
        if (at < 0) {
#ifdef __HIP_DEVICE_COMPILE__
            uint64_t m = ballot(hit);
            at = m ? base + __builtin_ctzll(m) : -1;
#else
            at = hit ? i : -1;
#endif
        }
        if (at >= 0 && i > at && i < n) {
            active_put(i - 1, a);
        }
    }
    if (at >= 0) {
        S->n_active = n - 1;
    }
}

// Constraintpoints::endpoint_reached (:359-372)
DEVIN bool WEng::cp_endpoint_reached(int s, I3 p) {
    int sg = seg[s];
    int cs = cslot_of(s), dd = d_of(s);
    int n = S->n_active;
    bool hit = false;
    for (int i = plane(); i < n; i += width) {
        Endpoint e = active_at(i);
        hit = hit || (e.cslot == cs && e.seg == sg && e.d == dd && e.x == p.x && e.y == p.y &&
                      e.z == p.z);
    }
    return all_lanes(hit);
}

// Constraintpoints::walks_remain (:397-442, 571-601) for one segment; see
// Eng::cp_walks_remain
DEVIN bool WEng::cp_walks_seg(int s, I3 p, int sg) {
    int cs = cslot_of(s), dd = d_of(s);
    int dir = cyc && cs == 0 ? cp_seg_dir(cs, sg) : 0;
    int n = S->n_active;
    bool bad = false;
    for (int i = plane(); i < n; i += width) {
        Endpoint e = active_at(i);
        int ed = e.d;
        int steps = ed > dd ? ed - dd : dd - ed;
        if (cyc && cs == 0) {
            if (dir > 0 && ed < dd) {
                steps = ns + ed - dd;
            }
            else if (dir < 0 && ed > dd) {
                steps = dd + ns - ed;
            }
            else if (dir == 0) {
                steps = 0;
            }
        }
        int ax = e.x - p.x, ay = e.y - p.y, az = e.z - p.z;
        int l1 = (ax < 0 ? -ax : ax) + (ay < 0 ? -ay : ay) + (az < 0 ? -az : az);
        bad = bad || (e.cslot == cs && e.seg == sg && (l1 > steps || ((steps - l1) & 1)));
    }
    return !all_lanes(bad);
}

// the end of calculate_constraintpoints (top_constraint_points.cpp:220,
// 247): m_initial_active_endpoints = m_active_endpoints
DEVNI void WEng::cp_save_initial() {
    for (int i = plane(), n = S->n_active; i < n; i += width) {
        active0_put(i, active_at(i));
    }
    S->n_active0 = S->n_active;
}

// Constraintpoints::reset_active_endpoints (:295-297)
DEVNI void WEng::cp_restore_initial() {
    six_d = -1;
    for (int i = plane(), n = S->n_active0; i < n; i += width) {
        active_put(i, active0_at(i));
    }
    S->n_active = S->n_active0;
}

// Eng::ctcb_staples, 64 chains at a time
DEVNI int WEng::ctcb_staples() {
    LArr<int16_t> sl {sframes.p};
    int nst = 0;
    for (int base = 1; base < nchain; base += width) {
        int c = base + plane();
        bool take = c < nchain && regrow.lane(c) != 0 &&
                    *(LDO_LDS const int16_t*)(ch.p + c * 8 + 4) >= 0;
#ifdef __HIP_DEVICE_COMPILE__
        uint64_t m = ballot(take);
#else
        uint64_t m = take ? 1 : 0;
#endif
        for (; m; m &= m - 1) {
            int c2 = base + __builtin_ctzll(m);
            int uid = ch[c2].uid;
            int k = nst++;
            while (k > 0 && ch[sl[k - 1]].uid > uid) {
                sl[k] = sl[k - 1];
                k--;
            }
            sl[k] = (int16_t)c2;
        }
    }
    return nst;
}

// ------------------------------------------------------------------- bias
// Eng::window_op and calc_move_bias with the window's fields in registers;
// the grid value of the last order parameter is kept for the next one
DEVNI int WEng::window_op(int staple_offset) {
    return w_op == LDO_OP_NUMSTAPLES ? S->num_staples + staple_offset : S->num_fully;
}

DEVNI double WEng::calc_move_bias(int staple_offset) {
    if (!w_on) {
        return 0;
    }
    int p = window_op(staple_offset);
    double r;
    if (p < w_min) {
        r = w_slope * (w_min - p - 1) + w_minb;
    }
    else if (p > w_max) {
        r = w_slope * (p - w_max - 1) + w_minb;
    }
    else {
        r = w_well;
    }
    double g = w_off;
    if (p >= 0 && p < P->grid_len) {
        if (p != w_last) {
            w_grid = P->win_grid[(size_t)S->temp_slot * P->grid_len + p];
            w_last = p;
        }
        g = w_grid;
    }
    double diff = r - w_st0;
    diff += g - w_st1;
    w_st0 = r;
    w_st1 = g;
    return diff * w_mult;
}

// one more of a 64-bit count in device memory
DEV void wave_count(int64_t* p, int64_t n) {
#ifdef __HIP_DEVICE_COMPILE__
    // one lane, and nothing waits for it
    if ((threadIdx.x & 63u) == 0) {
        __hip_atomic_fetch_add(p, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#else
    *p += n;
#endif
}

DEVNI void WEng::count_window_op() {
    int p = window_op(0);
    int b = (p >= 0 && p < P->grid_len) ? p : P->grid_len;
    wave_count(&P->hist[(size_t)S->temp_slot * (P->grid_len + 1) + b], 1);
}

// ------------------------------------------------------------------- steps
// Where the tracking counters of move kind `kind` begin (Layout::off_track)
// and how far its accepts lie behind its attempts.
DEV void track_range(const Layout& L, int kind, int& at, int& width) {
    int T = L.ntypes, n1 = L.ns + 1, s1 = L.smax + 1;
    at = kind == 2 ? 4 * T
                   : (kind == 3 ? 6 * T
                                : (kind == 4 ? 6 * T + 2 * n1 + 2 * s1
                                             : (kind == 5 ? 6 * T + 4 * n1 + 2 * s1
                                                          : 6 * T + 4 * n1 + 2 * s1 + 2)));
    at = kind == 1 ? 0 : at;
    width = kind <= 2 ? T : (kind == 5 ? 1 : (kind == 6 ? s1 : n1));
}

// Eng::track_move on the counters in device memory
DEVIN void WEng::track_move(int m, bool acc) {
    S->last_move = m;
    S->last_acc = acc ? 1 : 0;
    int kind = kind_of(m), at, w;
#ifdef __HIP_DEVICE_COMPILE__
    at = lane_int(mv_track, m);
    w = lane_int(mv_width, m);
#else
    track_range(P->L, kind, at, w);
#endif
    if (kind == 0 || (kind == 2 && S->trk_nost)) {
        return;
    }
    int64_t* t = (int64_t*)(gblk + P->L.off_track);
    int key = kind == 1 ? (S->trk_ins ? 0 : 2 * w) + S->trk_type
                        : (kind == 2 ? S->trk_type
                                     : (kind == 5 ? 0 : (kind == 6 ? S->trk_nst : S->trk_len)));
    wave_count(t + at + key, 1);
    if (acc) {
        wave_count(t + at + key + w, 1);
    }
    if (kind == 3) {
        // a CTCB move counts its staples too
        int64_t* u = t + at + 2 * w + S->trk_nst;
        wave_count(u, 1);
        if (acc) {
            wave_count(u + P->L.smax + 1, 1);
        }
    }
}

#ifdef __HIP_DEVICE_COMPILE__
// the lanes' attempts and accepts to the block's counters
__device__ __forceinline__ void WEng::count_moves() {
    if (plane() < LDO_MAX_MOVES) {
        LDO_LDS int64_t* a = (LDO_LDS int64_t*)S->attempts.p + plane();
        LDO_LDS int64_t* c = (LDO_LDS int64_t*)S->accepts.p + plane();
        *a += mv_att;
        *c += mv_acc;
    }
    mv_att = 0;
    mv_acc = 0;
}
#endif

// GCMCSimulation::simulate (simulation.cpp:568-653) and select_movetype
// (:655-665)
DEVNI void WEng::simulate(int64_t steps) {
    int nm = P->n_moves;
    // steps to the next centring and constraint check
    int64_t to_center = P->centering_freq > 0 ? P->centering_freq - S->step % P->centering_freq : 0;
    int64_t to_check = P->check_freq > 0 ? P->check_freq - S->step % P->check_freq : 0;
#ifdef __HIP_DEVICE_COMPILE__
    int mine = plane() & (LDO_MAX_MOVES - 1);
    double cum = plane() < nm ? P->move_cum[mine] : 0.0;
    mv_kind = P->move_kind[mine];
    mv_maxreg = P->move_maxreg[mine];
    track_range(P->L, mv_kind, mv_track, mv_width);
    mv_att = 0;
    mv_acc = 0;
#endif
    for (int64_t n = 0; n < steps; n++) {
        if (S->status != ST_OK) {
            break;
        }
        S->step += 1;
        rng_begin();
        double prob = uniform_real();
#ifdef __HIP_DEVICE_COMPILE__
        uint64_t lt = ballot(prob < cum);
        int m = lt ? __builtin_ctzll(lt) : nm - 1;
#else
        int m = 0;
        while (m < nm - 1 && !(prob < P->move_cum[m])) {
            m++;
        }
#endif
        bool acc = attempt(m);
#ifdef __HIP_DEVICE_COMPILE__
        bool own = plane() == m;
        mv_att += own ? 1 : 0;
        mv_acc += own & acc ? 1 : 0;
        if ((n & 0x3FFFFFFF) == 0x3FFFFFFF) {
            count_moves();
        }
#else
        S->attempts[m]++;
        S->accepts[m] += acc ? 1 : 0;
#endif
        track_move(m, acc);
        if (!acc) {
            reset_origami();
            calc_move_bias(0);
        }
        if (to_center != 0 && --to_center == 0) {
            center();
            to_center = P->centering_freq;
        }
        if (to_check != 0 && --to_check == 0) {
            check_all_constraints();
            to_check = P->check_freq;
        }
        if (P->hist != nullptr && S->status == ST_OK) {
            count_window_op();
        }
    }
#ifdef __HIP_DEVICE_COMPILE__
    count_moves();
#endif
}

#undef S
#undef LDO_WAVE
#undef LDO_ENG
#undef DEVNI
#define DEVNI inline __host__ __device__ __noinline__

#endif
