// The order of single causal tiles (sdpa_order.h) on the host: reads "heads nq last" a line, checks it, prints one line for each.
#define __host__
#define __device__
#include "sdpa_order.h"

#include <cstdio>
#include <vector>

int main() {
    long long heads, nq, resident;
    while (scanf("%lld %lld %lld", &heads, &nq, &resident) == 3) {
        const unsigned last = axhip::causal_last(heads, nq, resident), first = (unsigned)heads - last;
        std::vector<unsigned char> seen((size_t)(heads * nq));
        std::vector<int> xcd((size_t)heads, -1);
        const char *bad = first % 32 ? "groups" : last < 1 || last > heads ? "last" : nullptr;
        unsigned before = (unsigned)nq;
        for (unsigned block = 0; block < heads * nq && !bad; block++) {
            const axhip::CausalTile t = axhip::causal_tile(block, (unsigned)heads, (unsigned)nq, last);
            if (t.head >= heads || t.tile >= nq || seen[t.head * nq + t.tile]++) bad = "not every tile once";
            else if (block < first * nq) {
                if (t.head >= first) bad = "a late head early";
                if (xcd[t.head] >= 0 && xcd[t.head] != (int)(block % 8)) bad = "a head on two XCDs";
                xcd[t.head] = block % 8;
                // workgroups 8 apart are neighbours on an XCD: four of one length, for its four shader engines
                if (axhip::causal_tile(block / 32 * 32 + block % 8, (unsigned)heads, (unsigned)nq, last).tile != t.tile) bad = "lengths differ over shader engines";
            } else {
                if (t.tile > before) bad = "longer after shorter";
                before = t.tile;
            }
        }
        printf("%s %u %u\n", bad ? bad : "ok", first, last);
    }
}
