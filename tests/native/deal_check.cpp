// Host build of opfoundry_amd/csrc/dsa_deal.h (how the index scorer deals its
// chunks to workgroups) for tests/test_deal_cpu.py: the two HIP qualifiers are
// defined empty, so g++ compiles exactly the functions the kernel runs.
#define __host__
#define __device__
#include "../../opfoundry_amd/csrc/dsa_deal.h"

extern "C" {

uint32_t deal_start_units(void) { return dsa_deal::START; }

// Walks all workgroups over groups of chunks[0 .. n) chunks as the kernel does,
// G of them in runs or `parts` per group.  seen[c]: how often chunk c (all groups'
// chunks in a row) was taken; taken[x], begun[x]: chunks that workgroup x took, and
// groups that it took some of.
void deal_walk(const uint32_t* chunks, int n, uint32_t G, uint32_t parts, uint32_t* seen, uint32_t* taken,
               uint32_t* begun) {
    uint64_t all = 0, some = 0;
    for (int g = 0; g < n; ++g) {
        all += chunks[g];
        some += chunks[g] ? 1 : 0;
    }
    const dsa_deal::Deal d = dsa_deal::deal_of(all, some, G, dsa_deal::START);
    for (uint32_t x = 0; x < (parts ? parts * (uint32_t)n : G); ++x) {
        int g = 0, g_last = -1;
        uint32_t c_first = 0, c_last = 0;
        if (parts) {
            g = g_last = (int)(x / parts);
            dsa_deal::part_of(chunks[g], parts, x - (uint32_t)g * parts, &c_first, &c_last);
        } else {
            uint64_t first, last, end = 0;
            dsa_deal::run_of(d, x, &first, &last);
            for (int i = 0; first < last && i < n; ++i) {
                const uint64_t begin = end;
                end += dsa_deal::units(d, chunks[i]);
                if (begin <= first && first < end) {
                    g = i;
                    c_first = dsa_deal::chunks_before(d, first - begin);
                }
                if (begin < last && last <= end) {
                    g_last = i;
                    c_last = dsa_deal::chunks_before(d, last - begin);
                }
            }
        }
        uint64_t before = 0;
        for (int i = 0; i < g; ++i) before += chunks[i];
        for (; g <= g_last; before += chunks[g], ++g, c_first = 0) {
            const uint32_t end = g == g_last ? c_last : chunks[g];
            for (uint32_t c = c_first; c < end; ++c) ++seen[before + c];
            taken[x] += end > c_first ? end - c_first : 0;
            begun[x] += end > c_first ? 1 : 0;
        }
    }
}

}
