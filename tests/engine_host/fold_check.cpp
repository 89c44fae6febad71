// fold_check.cpp - the FourBody checks on folded positions anywhere in the
// coordinate range, for the undefined-behaviour sanitizer: small networks of
// bound pairs score alike where they lie, whatever the offset.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <random>

#include "../../latticednaorigami_amd/csrc/replica_ops.h"

namespace {

constexpr int NS = 6, STRIDE = 2, STAPLES = 3, SLOTS = NS + STAPLES * STRIDE;
alignas(16) DomRec dom[SLOTS];
int16_t ident[SLOTS];

I3 step_from(I3 p, std::mt19937& g) { return add3(p, unit3((int)(g() % 6))); }

} // namespace

int main() {
    const I3 far[] = {i3(0, 0, 2044), i3(0, 0, -2052), i3(0, 0, 1000000), i3(0, 0, -1000000),
                      i3(1000000, -1000000, 1000000), i3(-1000000, 1000000, -1000000),
                      i3(1023, -1025, 4095)};
    std::mt19937 g(7);
    int wrong = 0, scored = 0;
    for (int n = 0; n < 4000; n++) {
        // a scaffold walk, staples bound to it at random, opposed orientations
        I3 p = i3(0, 0, 0);
        for (int s = 0; s < NS; s++, p = step_from(p, g)) {
            dom[s] = DomRec {p.x, p.y, p.z, (int8_t)(g() % 6), OCC_UNBOUND, LDO_NONE};
        }
        for (int s = NS; s < SLOTS; s++) {
            dom[s] = DomRec {0, 0, 0, 0, OCC_UNASSIGNED, LDO_NONE};
            int b = (int)(g() % NS);
            if (dom[b].state == OCC_UNBOUND) {
                dom[s] = dom[b];
                dom[s].ore = (int8_t)(dom[b].ore ^ 1);
                dom[s].state = dom[b].state = OCC_BOUND;
                dom[s].bound = (int16_t)b;
                dom[b].bound = (int16_t)s;
            }
        }
        int di = NS + (int)(g() % (SLOTS - NS));
        if (dom[di].state != OCC_BOUND) {
            continue;
        }
        int dj = dom[di].bound;
        bool half = n % 2 == 0;
        // flags: lmask | cyc << 8 | dtype << 9 | stack_one << 10
        FbArgs a {(lds_t)(char*)dom, (lds_t)(char*)ident, nullptr, -1.0,
                  (STRIDE - 1) | (half ? 0 : 1) << 9 | 1 << 10, NS, 1};
        auto terms = half ? wave_fb_terms<true, true> : wave_fb_terms<false, true>;
        FbOut at_origin = terms(a, di, dj);
        scored += at_origin.st != 0;
        for (I3 f : far) {
            DomRec keep[SLOTS];
            for (int s = 0; s < SLOTS; s++) {
                keep[s] = dom[s];
                dom[s].x += f.x;
                dom[s].y += f.y;
                dom[s].z += f.z;
            }
            FbOut o = terms(a, di, dj);
            wrong += o.viol != at_origin.viol || o.e != at_origin.e || o.st != at_origin.st;
            for (int s = 0; s < SLOTS; s++) {
                dom[s] = keep[s];
            }
        }
    }
    std::printf("%d wrong, %d scored\n", wrong, scored);
    return wrong != 0 || scored < 100;
}
