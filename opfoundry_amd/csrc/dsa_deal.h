// dsa_deal.h - how the index scorer deals the chunks of all its groups to
// workgroups, shared by the kernel (device) and its CPU unit test (host).
//
// A group (a sequence's tokens that share a workgroup) holds some chunks of
// positions.  The groups lie one after another on a line, each as long as it
// costs: `start` units for what a workgroup pays to begin a group (Q, weights,
// the first entries and rows), then a unit per chunk.  The line is cut into equal
// runs, one per workgroup, and a run takes the chunks whose unit lies in it: it
// costs its length, and one start more when it begins inside a group.  Equal
// numbers of chunks alone would give one workgroup 64 groups of one chunk and
// another a run inside one long group: causal scores of one prompt, 4096 tokens x
// 4096 positions of 64 heads, 356 us, with starts counted 184; 500 sequences of 60
// to 4000 positions 56 and 38 us.  (Up to one chunk to a run, starts are not
// counted: every run is one start and one chunk already.  Nor where equal groups are
// cut into equal runs without them, as many to a group: 4 groups of 512 chunks in 512
// runs, 4 chunks each, 30.5 us; 32.6 with 5 in some.)
//
// hipcc compiles these for host and device; a host-only test defines
// __host__ and __device__ as empty before including this file.
#ifndef DSA_DEAL_H_
#define DSA_DEAL_H_

#include <stdint.h>

namespace dsa_deal {

// A start in chunks: 2 where each k row is read once (a chunk then waits on HBM:
// 128 sequences x 2 tokens x 16 K positions of 32 heads 106 us, 110 with 3), else 3
// (4096 tokens x 4096 positions of 128 heads 351 us, 369 with 2).
constexpr uint32_t START_ONCE = 2, START = 3;

struct Deal {
    uint32_t start;      // units in front of a group's chunks
    uint64_t each, more; // a run's units; the first `more` runs have one more
};

// chunks: of all groups; some: groups that have any; G: workgroups.  (The division
// is done in 32 bits where that fits: in 64 it takes a microsecond.)
__host__ __device__ inline Deal deal_of(uint64_t chunks, uint64_t some, uint32_t G, uint32_t start) {
    Deal d;
    d.start = chunks > G ? start : 0u;
    if (d.start && some <= G && G % (uint32_t)some == 0 && (chunks >> 32 ? chunks % G : (uint32_t)chunks % G) == 0) d.start = 0;
    const uint64_t all = chunks + d.start * some;
    d.each = all >> 32 ? all / G : (uint64_t)((uint32_t)all / G);
    d.more = all - d.each * G;
    return d;
}

// Units [*first, *last) of workgroup x.
__host__ __device__ inline void run_of(const Deal& d, uint32_t x, uint64_t* first, uint64_t* last) {
    *first = d.each * x + (x < d.more ? x : d.more);
    *last = *first + d.each + (x < d.more ? 1 : 0);
}

// A group's units, and its chunks that lie before unit `at` of the group.
__host__ __device__ inline uint64_t units(const Deal& d, uint32_t chunks) { return chunks ? (uint64_t)chunks + d.start : 0; }
__host__ __device__ inline uint32_t chunks_before(const Deal& d, uint64_t at) {
    return at > d.start ? (uint32_t)(at - d.start) : 0u;
}

// Whole workgroups per group instead: chunks [*c0, *c1) of workgroup `part` of `parts`.
__host__ __device__ inline void part_of(uint32_t chunks, uint32_t parts, uint32_t part, uint32_t* c0, uint32_t* c1) {
    const uint32_t each = chunks / parts, more = chunks - each * parts;
    *c0 = each * part + (part < more ? part : more);
    *c1 = *c0 + each + (part < more ? 1 : 0);
}

}  // namespace dsa_deal

#endif  // DSA_DEAL_H_
