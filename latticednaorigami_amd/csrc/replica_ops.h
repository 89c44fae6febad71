// replica_ops.h - the per-replica work of the sampler's kernels.
//
// Each function is the body a kernel runs for one replica (or, for the
// exchange, for the whole ladder).  They compile for the device, where the
// kernels in sampler.hip call them one replica per lane or per wavefront,
// and for the host, where a test build drives the same code replica by
// replica against the CPU oracle.
#ifndef LDO_REPLICA_OPS_H
#define LDO_REPLICA_OPS_H

#include "engine.h"
#include "engine_wave.h"
#include "layout.h"

// whether the moveset holds a recoil-growth or jump move
LDO_HD bool wave_all_kinds(const Params& P) {
    bool a = false;
    for (int m = 0; m < P.n_moves; m++) {
        a = a || P.move_kind[m] > LDO_MOVE_KIND_CTCB;
    }
    return a;
}

// Build (mode 0: OrigamiSystem constructor) or replace (mode 1: set_config)
// replica r's configuration.  c_idx/c_ident hold n_chains unique indices and
// identities, c_pos/c_ore three ints per domain in chain order.
DEV void init_replica(const Params& P, int r, const int32_t* c_idx, const int32_t* c_ident,
                      const int32_t* c_pos, const int32_t* c_ore, int n_chains, int mode,
                      const int32_t* rep_slot) {
    Eng e;
    char* blk = P.blocks + (size_t)r * P.L.bytes;
    RepScalars* S = (RepScalars*)blk;
    if (mode == 0) {
        S->temp_slot = rep_slot ? rep_slot[r] : r;
        S->init_slot = S->temp_slot;
        S->visited = 0;
        S->status = ST_OK;
        e.attach(&P, blk, r);
        for (int i = 0; i < P.L.hcap; i++) {
            e.hash[i] = LDO_HASH_EMPTY;
        }
        for (int c = 0; c < P.L.nchain; c++) {
            e.ch[c].ident = -1;
            e.ch[c].len = 0;
        }
        for (int t = 0; t < P.L.ntypes; t++) {
            e.tcount[t] = 0;
        }
        S->n_free = P.L.smax;
        for (int i = 0; i < P.L.smax; i++) {
            e.freel[i] = (int16_t)(P.L.smax - i);
        }
        // initialize_scaffold (origami_system.cpp:680-693)
        e.add_chain_with(0, c_idx[0]);
        S->num_staples--;
    }
    else {
        e.attach(&P, blk, r);
        // set_config (origami_system.cpp:327-341)
        for (int w = 0; w < S->n_chains; w++) {
            int cs = e.order[w];
            for (int d = 0; d < e.ch[cs].len; d++) {
                e.unassign_domain(e.slot(cs, d));
            }
        }
        for (int w = S->n_chains - 1; w != 0; w--) {
            e.delete_chain(e.order[w]);
        }
    }
    // initialize_staples (origami_system.cpp:659-678)
    int maxidx = c_idx[0];
    for (int c = 1; c < n_chains; c++) {
        e.add_chain_with(c_ident[c], c_idx[c]);
        maxidx = c_idx[c] > maxidx ? c_idx[c] : maxidx;
    }
    S->energy += (double)(S->n_chains - 1) * e.init_e;
    S->current_c_i = maxidx;
    // set_all_domains(config) (origami_system.cpp:588-616)
    int k = 0;
    for (int w = 0; w < S->n_chains; w++) {
        int cs = e.order[w];
        for (int d = 0; d < e.ch[cs].len; d++, k++) {
            int s = e.slot(cs, d);
            e.dom[s].x = c_pos[3 * k];
            e.dom[s].y = c_pos[3 * k + 1];
            e.dom[s].z = c_pos[3 * k + 2];
            I3 o = i3(c_ore[3 * k], c_ore[3 * k + 1], c_ore[3 * k + 2]);
            e.dom[s].ore = (int8_t)unit_index(o);
        }
    }
    e.set_all_domains();
}

// `steps` steps of GCMCSimulation::simulate (simulation.cpp:568-653); with a
// ladder (rep_slot) the replica first takes its slot's control variables
// (update_control_qs: a temperature switch recomputes the energy; windows
// swap only within a ladder of one temperature and change only the bias) and
// ends with its
// dependent quantities.
// One sweep of replica r on a caller-provided engine object and replica block
// (the block in device memory, or a copy of it held closer to the lane).
// par = 1: the 64 lanes of the calling wavefront all make this call (see
// Eng::par).
DEV void sweep_replica_on(Eng& e, const Params& P, int r, char* blk, int64_t steps,
                          const int32_t* rep_slot, int par = 0) {
    e.attach(&P, blk, r, par);
    if (e.S->status != ST_OK) {
        return;
    }
    if (rep_slot != nullptr) {
        // a window swap keeps the temperature; a temperature change
        // recomputes the energy (update_temp)
        int slot = rep_slot[r];
        bool moved = P.slot_key != nullptr && P.slot_key[slot] != P.slot_key[e.S->temp_slot];
        e.begin_interval(slot, P.exchange_mode != LDO_EXCHANGE_WINDOWS || moved);
    }
    e.simulate(steps);
    if (rep_slot != nullptr) {
        e.update_enthalpy_and_entropy();
    }
}

// The same with the wavefront engine, on a copy of the block's staged part in
// `lds` (wave_lds_bytes).  ALL: the moveset holds a recoil-growth or jump move.
template <bool ALL>
DEV void sweep_wave(const Params& P, int r, char* blk, lds_t lds, int64_t steps,
                    const int32_t* rep_slot) {
    WEng e;
    e.kinds = ALL;
    e.attach(&P, blk, lds, r);
    if (e.sc.status != ST_OK) {
        return;
    }
    if (rep_slot != nullptr) {
        int slot = uni(rep_slot[r]);
        bool moved = P.slot_key != nullptr &&
                     uni(P.slot_key[slot]) != uni(P.slot_key[e.sc.temp_slot]);
        e.begin_interval(slot, P.exchange_mode != LDO_EXCHANGE_WINDOWS || moved);
    }
    e.simulate(steps);
    if (rep_slot != nullptr) {
        e.update_enthalpy_and_entropy();
    }
    e.store_scalars();
}

DEV void sweep_replica(const Params& P, int r, int64_t steps, const int32_t* rep_slot,
                       int par = 0) {
    Eng e;
    sweep_replica_on(e, P, r, P.blocks + (size_t)r * P.L.bytes, steps, rep_slot, par);
}

// ldo_site_eval on a replica block (the caller's copy): the domain is taken
// off its site if placed (unassign_domain, origami_system.cpp:375-385) and
// checked at the query's site (check_domain_constraints, :343-355).  Returns
// false when the chain or the domain does not exist.
DEV bool site_eval_on(const Params& P, char* blk, const ldo_site_query& q, ldo_site_result& res) {
    Eng e;
    e.attach(&P, blk, q.replica);
    e.select_tables();
    res.unassign_delta = 0;
    res.delta = 0;
    res.violated = 0;
    res.pad = 0;
    int cs = -1;
    for (int w = 0; w < e.S->n_chains; w++) {
        if (e.ch[e.order[w]].uid == q.chain_index) {
            cs = e.order[w];
        }
    }
    if (cs < 0 || q.domain < 0 || q.domain >= e.ch[cs].len) {
        return false;
    }
    int s = e.slot(cs, q.domain);
    if (e.dom[s].state != OCC_UNASSIGNED) {
        res.unassign_delta = e.unassign_domain(s);
    }
    e.S->violated = 0;
    res.delta = e.check_domain_constraints(s, i3(q.pos[0], q.pos[1], q.pos[2]),
                                           unit_index(i3(q.ore[0], q.ore[1], q.ore[2])));
    res.violated = e.S->violated ? 1 : 0;
    return true;
}

// OrigamiSystem::update_enthalpy_and_entropy (origami_system.cpp:204-246)
DEV void dependent_replica(const Params& P, int r) {
    Eng e;
    e.attach(&P, P.blocks + (size_t)r * P.L.bytes, r);
    e.update_enthalpy_and_entropy();
}

#ifdef __HIP_DEVICE_COMPILE__
// The same by the 64 lanes of a wavefront on the block in device memory, with
// `rank` ([nchain] in LDS) for the chains' places in the working order.  A
// chain of dependent reads per domain bounds the serial form, so here every
// domain's partner and table entries are read side by side.  A pair counts at
// the domain that comes first in the working order, and the entries that
// count are added in that order.  A partner that does not point back (a state
// the caller forced) takes the serial form.  64-domain raster, 32 replicas:
// about 40 us less for each of the observables' 32 calls.
__device__ __forceinline__ void dependent_wave(const Params& P, int r, int16_t* rank) {
    const Layout& L = P.L;
    char* blk = P.blocks + (size_t)r * L.bytes;
    RepScalars* S = (RepScalars*)blk;
    const DomRec* dom = (const DomRec*)(blk + L.off_dom);
    const int16_t* dident = (const int16_t*)(blk + L.off_dident);
    const ChainRec* ch = (const ChainRec*)(blk + L.off_chain);
    const int16_t* order = (const int16_t*)(blk + L.off_order);
    int lane = threadIdx.x & 63, ns = L.ns, n = S->n_chains;
    size_t n2 = (size_t)P.n_ident * P.n_ident;
    const double* th = P.hyb_h + (size_t)S->temp_slot * n2;
    const double* ts = P.hyb_s + (size_t)S->temp_slot * n2;
    for (int c = lane; c < L.nchain; c += 64) {
        rank[c] = -1;
    }
    __syncthreads();
    for (int w = lane; w < n; w += 64) {
        rank[order[w]] = (int16_t)w;
    }
    __syncthreads();
    bool odd = false; // some partner does not point back
    double h = 0, e = 0;
    // one domain per lane: whether its pair counts here, and its entries
    auto add = [&](int s, int w, bool have) {
        bool counts = false;
        double x = 0, y = 0;
        if (have) {
            DomRec d = dom[s];
            if (d.state == OCC_BOUND || d.state == OCC_MISBOUND) {
                int b = d.bound;
                bool in = b >= 0 && b < L.nslots;
                DomRec o = dom[in ? b : s];
                int cb = !in || b < ns ? 0 : 1 + ((b - ns) >> L.lshift);
                int wb = rank[cb];
                if (!in || wb < 0 || o.bound != s ||
                    (o.state != OCC_BOUND && o.state != OCC_MISBOUND)) {
                    odd = true;
                } else {
                    counts = wb == w ? s < b : w < wb;
                    if (counts) {
                        size_t k = (size_t)dident[s] * P.n_ident + dident[b];
                        x = th[k];
                        y = ts[k];
                    }
                }
            }
        }
        for (uint64_t m = __builtin_amdgcn_ballot_w64(counts); m; m &= m - 1) {
            int l = __builtin_ctzll(m);
            h += lane_double(x, l);
            e += lane_double(y, l);
        }
    };
    for (int s0 = 0; s0 < ns; s0 += 64) {
        add(s0 + lane, 0, s0 + lane < ns);
    }
    // a lane for every slot of a staple's stride, several staples at a time
    int stride = 1 << L.lshift, per = stride < 64 ? 64 >> L.lshift : 1;
    for (int w0 = 1; w0 < n; w0 += per) {
        int w = stride < 64 ? w0 + (lane >> L.lshift) : w0;
        int cs = w < n ? order[w] : 0;
        int len = w < n ? ch[cs].len : 0;
        for (int d0 = 0; d0 < stride; d0 += 64) {
            int d = d0 + (lane & (stride - 1));
            add(ns + ((cs - 1) << L.lshift) + d, w, d < len);
        }
    }
    if (__builtin_amdgcn_ballot_w64(odd)) {
        if (lane == 0) {
            dependent_replica(P, r);
        }
        return;
    }
    h += (double)(n - 1) * P.init_h[S->init_slot];
    e += (double)(n - 1) * P.init_s[S->init_slot];
    if (lane == 0) {
        S->hyb_h = h;
        S->hyb_s = e;
        S->stack_e = S->energy - (h - e);
    }
}
#endif

DEV int32_t replica_status(const Params& P, int r) {
    return ((const RepScalars*)(P.blocks + (size_t)r * P.L.bytes))->status;
}

// Exchange state on the device
struct XState {
    int32_t* q_to_rep;
    int32_t* rep_slot;
    const double* ladder_t;
    const double* ladder_u;
    const double* ladder_s;
    const double* reduced_u; // [n_replicas * (ntypes-1)]
    double* rep_u;           // [n_replicas] each replica's chemical-potential multiplier
    // attempts, accepts, then per slot pair attempts[2R] and accepts[2R]
    // (element d * R + q: the pair of slot q with its neighbour in direction d)
    int64_t* counts;
};

// The exchange stream: Philox4x32-10 keyed by (seed, 0xFFFFFFFF), counter
// (draw, 0, exchange round of the context); or the recorded draws of replica
// 0's tape.
DEV double exchange_uniform(const Params& P, int64_t rng_ctr, uint32_t& idx) {
    if (P.rng_mode == 1) {
        RepScalars* S0 = (RepScalars*)P.blocks;
        int64_t pos = S0->tape_pos;
        if (pos >= P.tape_len[0]) {
            S0->status = ST_TAPE;
            return 0.0;
        }
        S0->tape_pos = pos + 1;
        return bits_to_double(P.tapes[P.tape_off[0] + pos]);
    }
    uint32_t c0 = idx++, c1 = 0u, c2 = (uint32_t)(uint64_t)rng_ctr,
             c3 = (uint32_t)((uint64_t)rng_ctr >> 32);
    uint32_t k0 = (uint32_t)P.seed, k1 = 0xFFFFFFFFu;
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
    uint64_t x = (uint64_t)c0 | ((uint64_t)c1 << 32);
    return (double)(x >> 11) * 0x1.0p-53;
}

// One pair's attempt: its slots and replicas, the counter of its direction,
// whether it may swap at all and the acceptance probability (1: without a
// draw).  The pairs of a set share no slot, so what is read for one does not
// depend on another's decision.
struct PairTry {
    int a, b, r1, r2;
    size_t at; // counter offset
    bool in;
    double p;
};

DEV void exchange_swap(const Params& P, const XState& X, const PairTry& t) {
    X.counts[2 + 2 * (size_t)P.n_replicas + t.at]++;
    X.q_to_rep[t.a] = t.r2;
    X.q_to_rep[t.b] = t.r1;
    X.rep_slot[t.r2] = t.a;
    X.rep_slot[t.r1] = t.b;
}

// test_acceptance (ptmc_simulation.cpp:300-313) and the swap
DEV void exchange_decide(const Params& P, const XState& X, const PairTry& t, int64_t rng_ctr,
                         uint32_t& idx) {
    X.counts[0]++;
    X.counts[2 + t.at]++;
    if (t.in && ((t.p == 1) ? true : (t.p > exchange_uniform(P, rng_ctr, idx)))) {
        X.counts[1]++;
        exchange_swap(P, X, t);
    }
}

#ifdef __HIP_DEVICE_COMPILE__
// exchange_decide for the pairs of a wavefront's lanes (`active` ones, in lane
// order) with Philox draws: a lane's draw is numbered by the drawing lanes
// before it.
__device__ __forceinline__ void exchange_decide_wave(const Params& P, const XState& X,
                                                     const PairTry& t, bool active,
                                                     int64_t rng_ctr, uint32_t& idx) {
    int lane = threadIdx.x & 63;
    bool draw = active && t.in && !(t.p == 1);
    uint64_t m = __builtin_amdgcn_ballot_w64(draw);
    bool accept = active && t.in;
    if (draw) {
        uint32_t k = idx + (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1));
        accept = t.p > exchange_uniform(P, rng_ctr, k);
    }
    idx += (uint32_t)__builtin_popcountll(m);
    uint64_t tried = __builtin_amdgcn_ballot_w64(active);
    uint64_t taken = __builtin_amdgcn_ballot_w64(accept);
    if (lane == 0) {
        X.counts[0] += __builtin_popcountll(tried);
        X.counts[1] += __builtin_popcountll(taken);
    }
    if (active) {
        X.counts[2 + t.at]++;
    }
    if (accept) {
        exchange_swap(P, X, t);
    }
}
#endif

// calc_acceptance_p (ptmc_simulation.cpp:255-298) for the replicas in slots a
// and b.  The per-staple
// chemical potential of a replica is reduced_u * T * (its own multiplier),
// as update_staple_us leaves m_staple_us (origami_system.cpp:624-628).
// d: direction of the pair (per-pair counters).
DEV PairTry exchange_pair(const Params& P, const XState& X, int a, int b, int d) {
    int nst = P.L.ntypes - 1;
    int r1 = X.q_to_rep[a], r2 = X.q_to_rep[b];
    RepScalars* S1 = (RepScalars*)(P.blocks + (size_t)r1 * P.L.bytes);
    RepScalars* S2 = (RepScalars*)(P.blocks + (size_t)r2 * P.L.bytes);
    const int16_t* tc1 = (const int16_t*)((char*)S1 + P.L.off_tcount);
    const int16_t* tc2 = (const int16_t*)((char*)S2 + P.L.off_tcount);
    double t1 = X.ladder_t[a], t2 = X.ladder_t[b];
    double sm1 = X.ladder_s[a], sm2 = X.ladder_s[b];
    double dbu_dn = 0;
    for (int k = 0; k < nst; k++) {
        double u1 = X.reduced_u[(size_t)r1 * nst + k] * t1 * X.rep_u[r1];
        double u2 = X.reduced_u[(size_t)r2 * nst + k] * t2 * X.rep_u[r2];
        dbu_dn += (u2 / t2 - u1 / t1) * ((double)tc2[k + 1] - (double)tc1[k + 1]);
    }
    double DB = 1 / t2 - 1 / t1;
    double DH = S2->hyb_h * t2 - S1->hyb_h * t1;
    double Dst = S2->stack_e * t2 - S1->stack_e * t1;
    double DBM = sm2 / t2 - sm1 / t1;
    double DBias = 0.0 * t2 - 0.0 * t1;
    double p = fmin(1.0, exp(DB * (DH + DBias) + DBM * Dst - dbu_dn));
    return PairTry {a, b, r1, r2, (size_t)d * P.n_replicas + a, true, p};
}

// One exchange round of the PT drivers: OneDPTGCMCSimulation::
// attempt_exchange (ptmc_simulation.cpp:360-412; swap_i picks the even or
// odd neighbour pairs) or TwoDPTGCMCSimulation::attempt_exchange (495-560;
// swap_i % 4 picks even or odd rows of temperature neighbours, or even or
// odd columns of stacking neighbours, in the grid of pt_dim2 columns), then
// master_send (212-226): with UT, HUT and 2D every replica takes its new
// slot's chemical-potential multiplier.  rng_ctr is the round's
// exchange-stream counter.
DEV void exchange_round(const Params& P, const XState& X, int64_t swap_i, int64_t rng_ctr) {
    int R = P.n_replicas;
    uint32_t idx = 0;
    if (P.exchange_mode == LDO_EXCHANGE_2D) {
        int v2 = P.pt_dim2, v1 = R / v2;
        int set = (int)(swap_i % 4);
        bool temps = set % 2 == 0; // sets 0 and 2 pair temperatures
        int i0 = set == 2 ? 1 : 0, j0 = set == 3 ? 1 : 0;
        int di = temps ? 2 : 1, dj = temps ? 1 : 2;
        int i1 = temps ? v1 - 1 : v1, j1 = temps ? v2 : v2 - 1;
        int step = temps ? v2 : 1;
        for (int i = i0; i < i1; i += di) {
            for (int j = j0; j < j1; j += dj) {
                int a = i * v2 + j;
                exchange_decide(P, X, exchange_pair(P, X, a, a + step, temps ? 0 : 1), rng_ctr,
                                idx);
            }
        }
    }
    else {
        for (int i = (int)(swap_i % 2); i < R - 1; i += 2) {
            exchange_decide(P, X, exchange_pair(P, X, i, i + 1, 0), rng_ctr, idx);
        }
    }
    int m = P.exchange_mode;
    if (m == LDO_EXCHANGE_TEMPERATURE || m == LDO_EXCHANGE_HUT || m == LDO_EXCHANGE_2D) {
        for (int q = 0; q < R; q++) {
            X.rep_u[X.q_to_rep[q]] = X.ladder_u[q];
        }
    }
}

// A replica's value of a window's order parameter (GridBiasFunction::get_point)
DEV int replica_window_op(const Params& P, int r, const ldo_window& w) {
    const RepScalars* S = (const RepScalars*)(P.blocks + (size_t)r * P.L.bytes);
    return w.op == LDO_OP_NUMSTAPLES ? S->num_staples : S->num_fully;
}

// grid bias of window q at point p as the exchange reads it (a GridFloats
// lookup: points without a value read 0)
DEV double exchange_grid(const Params& P, int q, int p) {
    return (p >= 0 && p < P.grid_len) ? P.win_grid[(size_t)q * P.grid_len + p] : 0.0;
}

// PTMWUSGCMCSimulation::attempt_exchange (us_simulation.cpp:770-864):
// adjacent windows swap configurations when each window's order parameter
// lies inside the other window.  Windows are ladder slots here, so a swap
// exchanges the two replicas' slots; each window keeps its stored biases.
DEV PairTry exchange_window_pair(const Params& P, const XState& X, int i) {
    const ldo_window& w1 = P.windows[i];
    const ldo_window& w2 = P.windows[i + 1];
    int r1 = X.q_to_rep[i], r2 = X.q_to_rep[i + 1];
    int p1 = replica_window_op(P, r1, w1);
    int p2 = replica_window_op(P, r2, w2);
    bool in = !(p2 < w1.min_op || p2 > w1.max_op || p1 < w2.min_op || p1 > w2.max_op);
    double p = 1;
    if (in && p1 != p2) {
        double d1 = exchange_grid(P, i, p1) - exchange_grid(P, i + 1, p1);
        double d2 = exchange_grid(P, i + 1, p2) - exchange_grid(P, i, p2);
        p = fmin(1.0, exp(d1 + d2));
    }
    return PairTry {i, i + 1, r1, r2, (size_t)i, in, p};
}

// Swap of the replicas in window w of two ladders at neighbouring
// temperatures (slots a < b, LDO_FLAG_WINDOW_TEMPERATURE_SWAPS): the PTMC log
// ratio of the two slots plus the grid biases of both windows at both
// replicas' order parameters; the windows' restraints are equal and cancel.
DEV PairTry exchange_window_temperatures(const Params& P, const XState& X, int a, int b) {
    int nst = P.L.ntypes - 1;
    int r1 = X.q_to_rep[a], r2 = X.q_to_rep[b];
    const RepScalars* S1 = (const RepScalars*)(P.blocks + (size_t)r1 * P.L.bytes);
    const RepScalars* S2 = (const RepScalars*)(P.blocks + (size_t)r2 * P.L.bytes);
    const int16_t* tc1 = (const int16_t*)((const char*)S1 + P.L.off_tcount);
    const int16_t* tc2 = (const int16_t*)((const char*)S2 + P.L.off_tcount);
    double t1 = X.ladder_t[a], t2 = X.ladder_t[b];
    double sm1 = X.ladder_s[a], sm2 = X.ladder_s[b];
    double dbu_dn = 0;
    for (int k = 0; k < nst; k++) {
        double u1 = X.reduced_u[(size_t)r1 * nst + k] * t1 * X.rep_u[r1];
        double u2 = X.reduced_u[(size_t)r2 * nst + k] * t2 * X.rep_u[r2];
        dbu_dn += (u2 / t2 - u1 / t1) * ((double)tc2[k + 1] - (double)tc1[k + 1]);
    }
    double DB = 1 / t2 - 1 / t1;
    double DH = S2->hyb_h * t2 - S1->hyb_h * t1;
    double Dst = S2->stack_e * t2 - S1->stack_e * t1;
    double DBM = sm2 / t2 - sm1 / t1;
    int p1 = replica_window_op(P, r1, P.windows[a]);
    int p2 = replica_window_op(P, r2, P.windows[b]);
    double dg = (exchange_grid(P, a, p1) - exchange_grid(P, b, p1)) +
                (exchange_grid(P, b, p2) - exchange_grid(P, a, p2));
    double p = fmin(1.0, exp(DB * DH + DBM * Dst - dbu_dn + P.windows[a].bias_mult * dg));
    return PairTry {a, b, r1, r2, (size_t)P.n_replicas + a, true, p};
}

// One exchange round over every window ladder.
DEV void exchange_windows_round(const Params& P, const XState& X, int64_t swap_i,
                                int64_t rng_ctr) {
    int R = P.n_replicas;
    uint32_t idx = 0;
    // each run of consecutive slots at one temperature is a window ladder of
    // its own (one PTMWUS run of the reference), paired from its first slot
    int W = R;
    for (int g0 = 0, g1; g0 < R; g0 = g1) {
        for (g1 = g0 + 1; g1 < R && X.ladder_t[g1] == X.ladder_t[g0]; g1++) {
        }
        if (g0 == 0) {
            W = g1;
        }
        for (int i = g0 + (int)(swap_i % 2); i < g1 - 1; i += 2) {
            exchange_decide(P, X, exchange_window_pair(P, X, i), rng_ctr, idx);
        }
    }
    if (P.flags & LDO_FLAG_WINDOW_TEMPERATURE_SWAPS) {
        for (int g = (int)(swap_i % 2); (g + 2) * W <= R; g += 2) {
            for (int w = 0; w < W; w++) {
                exchange_decide(P, X,
                                exchange_window_temperatures(P, X, g * W + w, (g + 1) * W + w),
                                rng_ctr, idx);
            }
        }
    }
}

#ifdef __HIP_DEVICE_COMPILE__
// Both rounds by a wavefront, for Philox draws: a pair per lane, the pairs of
// a set 64 at a time in the order above.  A pair reads some hundred values in
// dependent rounds (a staple type at a time), which is all an exchange takes:
// one lane needed 1.4 ms for the 192 pairs of 256 windows.
__device__ __forceinline__ void exchange_round_wave(const Params& P, const XState& X,
                                                    int64_t swap_i, int64_t rng_ctr) {
    int R = P.n_replicas, lane = threadIdx.x & 63;
    uint32_t idx = 0;
    bool grid = P.exchange_mode == LDO_EXCHANGE_2D;
    int v2 = grid ? P.pt_dim2 : 1, set = (int)(swap_i % 4);
    bool temps = !grid || set % 2 == 0;
    // pairs (i, j) of the grid from (i0, j0) in steps (di, dj), nj to a row
    int i0 = grid ? set == 2 : (int)(swap_i % 2), j0 = grid && set == 3 ? 1 : 0;
    int di = temps ? 2 : 1, dj = !grid || temps ? 1 : 2;
    int i1 = grid && !temps ? R / v2 : R / v2 - 1, j1 = temps ? v2 : v2 - 1;
    int ni = i1 > i0 ? (i1 - i0 + di - 1) / di : 0, nj = j1 > j0 ? (j1 - j0 + dj - 1) / dj : 0;
    int step = temps ? v2 : 1;
    for (int k0 = 0; k0 < ni * nj; k0 += 64) {
        int k = k0 + lane;
        bool active = k < ni * nj;
        PairTry t = {};
        if (active) {
            int a = (i0 + di * (k / nj)) * v2 + j0 + dj * (k % nj);
            t = exchange_pair(P, X, a, a + step, temps ? 0 : 1);
        }
        exchange_decide_wave(P, X, t, active, rng_ctr, idx);
    }
    __syncthreads();
    int m = P.exchange_mode;
    if (m == LDO_EXCHANGE_TEMPERATURE || m == LDO_EXCHANGE_HUT || m == LDO_EXCHANGE_2D) {
        for (int q = lane; q < R; q += 64) {
            X.rep_u[X.q_to_rep[q]] = X.ladder_u[q];
        }
    }
}

__device__ __forceinline__ void exchange_windows_round_wave(const Params& P, const XState& X,
                                                            int64_t swap_i, int64_t rng_ctr) {
    int R = P.n_replicas, lane = threadIdx.x & 63;
    uint32_t idx = 0;
    int W = R, g0 = 0; // the first ladder's windows; start of the current one
    for (int k0 = 0; k0 < R; k0 += 64) {
        int i = k0 + lane;
        bool first = i < R && i > 0 && X.ladder_t[i] != X.ladder_t[i - 1];
        uint64_t m = __builtin_amdgcn_ballot_w64(first);
        uint64_t below = m & (~0ull >> (63 - lane));
        int g = below ? k0 + 63 - __builtin_clzll(below) : g0;
        bool active = i < R - 1 && X.ladder_t[i + 1] == X.ladder_t[i] &&
                      (i - g) % 2 == (int)(swap_i % 2);
        PairTry t = {};
        if (active) {
            t = exchange_window_pair(P, X, i);
        }
        exchange_decide_wave(P, X, t, active, rng_ctr, idx);
        if (m) {
            W = W == R ? k0 + __builtin_ctzll(m) : W;
            g0 = k0 + 63 - __builtin_clzll(m);
        }
    }
    __syncthreads();
    if (P.flags & LDO_FLAG_WINDOW_TEMPERATURE_SWAPS) {
        // ladder pairs (g, g + 1), W windows each
        int s = (int)(swap_i % 2), n = R / W - s;
        n = n > 0 ? n / 2 * W : 0;
        for (int k0 = 0; k0 < n; k0 += 64) {
            int k = k0 + lane;
            PairTry t = {};
            if (k < n) {
                int a = (s + 2 * (k / W)) * W + k % W;
                t = exchange_window_temperatures(P, X, a, a + W);
            }
            exchange_decide_wave(P, X, t, k < n, rng_ctr, idx);
        }
    }
}
#endif

// the stored move-level bias of the window in ladder slot q (0 without
// windows).  The replica in slot q is rep_slot's inverse, not the block's
// temp_slot, which follows a swap only when the next interval begins.
DEV double slot_bias(const Params& P, int q) {
    if (P.windows == nullptr) {
        return 0;
    }
    return (P.win_stored[2 * q] + P.win_stored[2 * q + 1]) * P.windows[q].bias_mult;
}

// ------------------------------------------------------ learned proposal
// The lane parts of a learned-move attempt (Eng::learned_begin/finish): lane
// `lane` of `nl` handles sites lane, lane + nl, ... of the input box and
// hidden units lane, lane + nl, ...; every value is computed by one lane in a
// fixed order, so any lane count gives the same bits.

// the one-hot channels of the 7x7x7 box around the anchor (site index
// (dz+3)*49 + (dy+3)*7 + (dx+3)) and the six neighbour sites that can take d
// (at most one other domain there)
DEV void learned_context_lane(const Eng& e, LearnedMove& m, int lane, int nl) {
    for (int s = lane; s < 343; s += nl) {
        I3 p = i3(m.ax + s % 7 - 3, m.ay + (s / 7) % 7 - 3, m.az + s / 49 - 3);
        m.ch[s] = (uint8_t)e.site_channel(p, m.d);
    }
    for (int n = lane; n < 6; n += nl) {
        I3 p = add3(i3(m.ax, m.ay, m.az), unit3(n));
        m.legal[n] = e.site_count(p, m.d) <= 1 ? 1 : 0;
    }
}

// h[0] = relu(b1 + sum over sites of W1[site*13 + channel] + emb[id] W1e)
DEV void net_layer1_lane(const Params& P, LearnedMove& m, int lane, int nl) {
    const float* W = P.net;
    const float* e = W + P.net_off[1] + (int64_t)m.id * 16;
    for (int j = lane; j < 256; j += nl) {
        float s = W[P.net_off[3] + j];
        const float* w1 = W + P.net_off[0] + j;
        // 49 rows on their way at a time, added in site order
#pragma unroll 1
        for (int z = 0; z < 343; z += 49) {
            float w[49];
#pragma unroll
            for (int q = 0; q < 49; q++) {
                w[q] = w1[((z + q) * 13 + m.ch[z + q]) * 256];
            }
#pragma unroll
            for (int q = 0; q < 49; q++) {
                s += w[q];
            }
        }
        for (int k = 0; k < 16; k++) {
            s = fmaf(e[k], W[P.net_off[2] + k * 256 + j], s);
        }
        m.h[0][j] = fmaxf(s, 0.f);
    }
}

// out[j] = b[j] + sum_i in[i] W[i][j] (fused multiply-adds in i order),
// ReLU when `relu`
DEV void net_dense_lane(const float* W, const float* b, const float* in, float* out, int n_in,
                        int n_out, bool relu, int lane, int nl) {
    for (int j = lane; j < n_out; j += nl) {
        float s = b[j];
        // 32 rows on their way at a time (n_in is a multiple of 32)
#pragma unroll 1
        for (int i0 = 0; i0 < n_in; i0 += 32) {
            float w[32];
#pragma unroll
            for (int q = 0; q < 32; q++) {
                w[q] = W[(i0 + q) * n_out + j];
            }
#pragma unroll
            for (int q = 0; q < 32; q++) {
                s = fmaf(in[i0 + q], w[q], s);
            }
        }
        out[j] = relu ? fmaxf(s, 0.f) : s;
    }
}

// network phase `ph` (0: context, 1: layer 1, 2-3: hidden, 4: logits); the
// kernel separates phases with barriers, the host build runs them in order
DEV void learned_phase_lane(const Eng& e, const Params& P, LearnedMove& m, int ph, int lane,
                            int nl) {
    const float* W = P.net;
    switch (ph) {
    case 0:
        learned_context_lane(e, m, lane, nl);
        break;
    case 1:
        net_layer1_lane(P, m, lane, nl);
        break;
    case 2:
        net_dense_lane(W + P.net_off[4], W + P.net_off[5], m.h[0], m.h[1], 256, 256, true, lane, nl);
        break;
    case 3:
        net_dense_lane(W + P.net_off[6], W + P.net_off[7], m.h[1], m.h[0], 256, 256, true, lane, nl);
        break;
    case 4:
        net_dense_lane(W + P.net_off[8], W + P.net_off[9], m.h[0], m.logits, 256, 36, false, lane,
                       nl);
        break;
    }
}

#define LDO_LEARNED_PHASES 5

#endif
