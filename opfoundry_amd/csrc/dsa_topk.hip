// DSA top-k index selection for gfx950: the step in front of the sparse-MLA
// kernels that turns one row of index scores per query token into the
// `indices` row those kernels gather (positions ascending, -1 padded).
//
// The reference leaves this step to its caller: "top-k semantics should
// already be reflected in kv_indices" (opus_attn/dsa_v4/README.md:185;
// opus_attn/dsa_v32/README.md:99).  The contract here is therefore this
// library's own and is spelled out in include/dsa_topk.h.
//
// Design.  One workgroup of 1024 threads (16 waves) per query token; a
// token's row is 4 B per position, so the path is HBM-bound byte work and
// uses no MFMA.  Each fp32 score maps to an order-preserving uint32 key
// (NaN highest, -0 == +0).  A radix select finds the k-th key: one pass
// histograms the top 12 key bits of every valid position into LDS, the bin
// holding the k-th key is found with a workgroup scan, and the bin's keys go
// to an LDS list over which the remaining bits are resolved.  The output is in
// position order without any ordered pass over the row: every four positions
// leave a byte of flags in LDS (taken, tied), and one scan over the flags gives
// each thread its slots (emit_flags).
// - Rows of at most 65,536 positions (dsa_topk_reg_kernel) are read once: their
//   keys stay in registers.
// - Rows whose flags fit LDS (TS_MAX_N positions, dsa_topk_stream_kernel) are
//   read twice: once for the histogram, once for the flags and the list.
// - Longer rows (dsa_topk_kernel): an ordered second read compacts positions and
//   candidates (k <= 4096 and <= 4096 keys in the bin), else 10-bit passes over
//   the row refine the threshold and a last pass compacts in position order.
// Loads are 16-byte vector loads of four positions per lane, coalesced
// across the wave; the passes after the first hit the L2 / MALL.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dsa_topk.h"
#include "dsa_lds.h"

namespace {

constexpr int TK_THREADS = 1024;
constexpr int TK_WAVES = TK_THREADS / 64;
constexpr int TK_FIRST_BITS = 12;          // first histogram: 4096 bins
constexpr int TK_NEXT_BITS = 10;           // refinement passes: 1024 bins
constexpr int TK_UNROLL = 8;               // float4 loads in flight per lane in a histogram pass
constexpr int TK_GROUP = 4;                // compaction: segments of 4096 positions loaded together
constexpr int TK_FAST_K = 4096;            // two-read path: top-k sizes whose positions LDS holds
constexpr int TK_CAND = 4096;              // two-read path: threshold-bin candidates LDS holds

// Order-preserving key: a > b as scores <=> key(a) > key(b) as uint32.  Every
// NaN maps to the largest key, and -0 to the key of +0.
__device__ __forceinline__ uint32_t order_key(float x) {
    const uint32_t b = __float_as_uint(x);
    const uint32_t mag = b & 0x7fffffffu;
    if (mag > 0x7f800000u) return 0xffffffffu;
    if (mag == 0) return 0x80000000u;
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// The key's top L bits (L in {0, 12, 22, 32}).
__device__ __forceinline__ uint32_t key_top(uint32_t key, int L) {
    return L == 0 ? 0u : (L == 32 ? key : key >> (32 - L));
}

// Keys in the bins above this thread's: the workgroup total minus the inclusive scan.
__device__ __forceinline__ uint32_t tot_minus(uint32_t incl, uint32_t tot) { return tot - incl; }

// Number of entries of the ascending list a[0, n) below x.
__device__ __forceinline__ uint32_t count_below(const uint32_t* a, uint32_t n, uint32_t x) {
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (a[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Inclusive scan of one uint32 per thread over the workgroup; *total gets the
// workgroup's sum.  All threads must call it (it holds barriers).
__device__ __forceinline__ uint32_t wg_scan(uint32_t v, uint32_t* part, uint32_t* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t u = __shfl_up(v, d, 64);
        if (lane >= d) v += u;
    }
    if (lane == 63) part[w] = v;
    __syncthreads();
    if (w == 0) {
        uint32_t p = lane < TK_WAVES ? part[lane] : 0u;
#pragma unroll
        for (int d = 1; d < TK_WAVES; d <<= 1) {
            const uint32_t u = __shfl_up(p, d, 64);
            if (lane >= d) p += u;
        }
        if (lane < TK_WAVES) part[lane] = p;
    }
    __syncthreads();
    const uint32_t before = w ? part[w - 1] : 0u;
    *total = part[TK_WAVES - 1];
    __syncthreads();
    return v + before;
}

// Two-read path, after the 12-bit histogram has found the bin P holding the k-th
// key: `above` keys lie in higher bins and the r-th of the bin's cnt keys is the
// k-th overall.  One ordered pass over the row stores the above-bin positions and
// the bin's (key, position) pairs in LDS, both ascending; the remaining 20 key bits
// are resolved over the candidates alone, the r chosen candidates are compacted in
// position order, and the two ascending lists are merged into the output.
__device__ __forceinline__ void select_in_lds(const float4* __restrict__ row, int n, int n4, int k, uint32_t P,
                                              uint32_t above, uint32_t r, uint32_t cnt, uint32_t* hist,
                                              uint32_t* above_pos, uint2* cand, uint32_t* part,
                                              uint32_t* found, int32_t* __restrict__ out) {
    const int tid = threadIdx.x;
    uint32_t run_gt = 0, run_eq = 0;
    for (int base = 0; base < n4; base += TK_THREADS) {
        const int i = base + tid;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < n4) v = row[i];
        const float e[4] = {v.x, v.y, v.z, v.w};
        uint32_t keys[4], flags = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            keys[c] = order_key(e[c]);
            if (i >= n4 || 4 * i + c >= n) continue;
            const uint32_t top = keys[c] >> (32 - TK_FIRST_BITS);
            if (top > P) flags |= 1u << c;
            else if (top == P) flags |= 16u << c;
        }
        const uint32_t mine = (uint32_t)__builtin_popcount(flags & 15u) |
                              ((uint32_t)__builtin_popcount(flags >> 4) << 16);
        uint32_t tot;
        const uint32_t ex = wg_scan(mine, part, &tot) - mine;
        uint32_t gb = run_gt + (ex & 0xffffu), eb = run_eq + (ex >> 16);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if ((flags >> c) & 1u) {
                if (gb < (uint32_t)TK_FAST_K) above_pos[gb] = (uint32_t)(4 * i + c);
                ++gb;
            } else if ((flags >> (4 + c)) & 1u) {
                if (eb < (uint32_t)TK_CAND) cand[eb] = make_uint2(keys[c], (uint32_t)(4 * i + c));
                ++eb;
            }
        }
        run_gt += tot & 0xffffu;
        run_eq += tot >> 16;
    }
    __syncthreads();
    // the rest of the key (20 bits) over the candidates: two 10-bit digits
    uint32_t Pc = P;
    int L = TK_FIRST_BITS;
    bool take_all = false;
    uint32_t rr = r;
    for (int pass = 0; pass < 2; ++pass) {
        const int shift = 32 - L - TK_NEXT_BITS;
        hist[tid] = 0;  // 1024 bins, one per thread
        __syncthreads();
        for (uint32_t j = tid; j < cnt; j += TK_THREADS) {
            const uint32_t key = cand[j].x;
            if ((key >> (32 - L)) == Pc) atomicAdd(&hist[(key >> shift) & 1023u], 1u);
        }
        __syncthreads();
        const uint32_t c = hist[tid];
        uint32_t tot;
        const uint32_t acc = tot_minus(wg_scan(c, part, &tot), tot);
        if (acc < rr && acc + c >= rr) {
            found[0] = (uint32_t)tid;
            found[1] = acc;
            found[2] = c;
        }
        __syncthreads();
        const uint32_t digit = found[0], abv = found[1], cn = found[2];
        __syncthreads();
        rr -= abv;
        Pc = (Pc << TK_NEXT_BITS) | digit;
        L += TK_NEXT_BITS;
        if (rr == cn) {
            take_all = true;
            break;
        }
    }
    // the r chosen candidates, ascending, into hist[0, r)
    const uint32_t r_eff = take_all ? 0xffffffffu : rr;
    uint32_t cg = 0, ce = 0;
    for (uint32_t base = 0; base < cnt; base += TK_THREADS) {
        const uint32_t j = base + tid;
        uint32_t gt = 0, eq = 0;
        uint2 kp = make_uint2(0u, 0u);
        if (j < cnt) {
            kp = cand[j];
            const uint32_t top = key_top(kp.x, L);
            gt = top > Pc;
            eq = top == Pc;
        }
        const uint32_t mine = gt | (eq << 16);
        uint32_t tot;
        const uint32_t ex = wg_scan(mine, part, &tot) - mine;
        const uint32_t gb = cg + (ex & 0xffffu), eb = ce + (ex >> 16);
        if (gt) {
            const uint32_t slot = gb + (eb < r_eff ? eb : r_eff);
            if (slot < r) hist[slot] = kp.y;
        } else if (eq && eb < r_eff && gb + eb < r) {
            hist[gb + eb] = kp.y;
        }
        cg += tot & 0xffffu;
        ce += tot >> 16;
    }
    __syncthreads();
    // merge: an entry's slot is its rank in its own list plus the entries of the
    // other list below it (positions are distinct)
    for (uint32_t j = tid; j < above; j += TK_THREADS) {
        const uint32_t x = above_pos[j];
        const uint32_t slot = j + count_below(hist, r, x);
        if (slot < (uint32_t)k) out[slot] = (int32_t)x;
    }
    for (uint32_t j = tid; j < r; j += TK_THREADS) {
        const uint32_t y = hist[j];
        const uint32_t slot = j + count_below(above_pos, above, y);
        if (slot < (uint32_t)k) out[slot] = (int32_t)y;
    }
}

__global__ __launch_bounds__(TK_THREADS) void dsa_topk_kernel(
    const float* __restrict__ scores, int64_t score_stride, const int32_t* __restrict__ lengths,
    int32_t n_max, int32_t k, int32_t* __restrict__ indices, int64_t idx_stride) {
    __shared__ uint32_t hist[1 << TK_FIRST_BITS];  // histograms; then the chosen candidates
    __shared__ uint32_t above_pos[TK_FAST_K];        // two-read path: positions above the bin
    __shared__ uint2 cand[TK_CAND];                  // two-read path: (key, position) in the bin
    __shared__ uint32_t part[TK_WAVES];
    __shared__ uint32_t found[3];  // digit, keys above its bin, keys in its bin

    const int tid = threadIdx.x;
    const int64_t t = blockIdx.x;
    int n = lengths ? lengths[t] : n_max;
    n = n < 0 ? 0 : (n > n_max ? n_max : n);
    const float4* row = reinterpret_cast<const float4*>(scores + t * score_stride);
    int32_t* out = indices + t * idx_stride;
    const int n4 = (n + 3) >> 2;

    // Selection state: keys whose top L bits exceed P are taken; of those equal
    // to P, all are taken (take_all) or the first r in position order.
    uint32_t P = 0, r = (uint32_t)k;
    int L = 0;
    bool take_all = true;
    if (n > k) {
        take_all = false;
        for (int pass = 0; pass < 3; ++pass) {
            const int bits = pass == 0 ? TK_FIRST_BITS : TK_NEXT_BITS;
            const int nbins = 1 << bits;
            const int shift = 32 - L - bits;
            for (int b = tid; b < nbins; b += TK_THREADS) hist[b] = 0;
            __syncthreads();
            for (int i0 = tid; i0 < n4; i0 += TK_THREADS * TK_UNROLL) {
                float4 v[TK_UNROLL];
#pragma unroll
                for (int j = 0; j < TK_UNROLL; ++j) {
                    const int i = i0 + j * TK_THREADS;
                    if (i < n4) v[j] = row[i];
                }
#pragma unroll
                for (int j = 0; j < TK_UNROLL; ++j) {
                    const int i = i0 + j * TK_THREADS;
                    if (i >= n4) continue;
                    const float e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        if (4 * i + c >= n) continue;
                        const uint32_t key = order_key(e[c]);
                        if (key_top(key, L) == P) atomicAdd(&hist[(key >> shift) & (nbins - 1)], 1u);
                    }
                }
            }
            __syncthreads();
            // Thread tid owns bins [tid * per, tid * per + per); higher bins belong to
            // higher threads, so the keys above a thread's bins are total - inclusive.
            const int per = nbins / TK_THREADS;
            uint32_t s = 0;
            for (int j = 0; j < per; ++j) s += hist[tid * per + j];
            uint32_t tot;
            const uint32_t incl = wg_scan(s, part, &tot);
            uint32_t acc = tot - incl;
            for (int j = per - 1; j >= 0; --j) {
                const uint32_t c = hist[tid * per + j];
                if (acc < r && acc + c >= r) {  // exactly one bin in the workgroup holds the r-th key
                    found[0] = (uint32_t)(tid * per + j);
                    found[1] = acc;
                    found[2] = c;
                }
                acc += c;
            }
            __syncthreads();
            const uint32_t digit = found[0], above = found[1], cnt = found[2];
            __syncthreads();
            r -= above;
            P = (P << bits) | digit;
            L += bits;
            if (r == cnt) {
                take_all = true;
                break;
            }
            if (pass == 0 && k <= TK_FAST_K && cnt <= TK_CAND) {
                select_in_lds(row, n, n4, k, P, above, r, cnt, hist, above_pos, cand, part, found, out);
                return;  // uniform: every thread takes this branch
            }
        }
    }

    // Compaction in position order.  Per 4096 positions, one scan of packed
    // counts (above-threshold in the low half, equal in the high half; each is
    // at most 4096) gives every lane the counts of earlier positions.  An
    // equal-key position is taken iff fewer than r equal keys precede it; a
    // position's slot is the number of taken positions before it.
    const uint32_t r_eff = take_all ? 0xffffffffu : r;
    uint32_t run_gt = 0, run_eq = 0;
    // Segments of 4096 positions are loaded TK_GROUP at a time, and the next group's
    // loads are issued before this group's scans, so the scans' barriers overlap the
    // memory latency instead of waiting on one load each.
    float4 cur[TK_GROUP], nxt[TK_GROUP];
#pragma unroll
    for (int j = 0; j < TK_GROUP; ++j) {
        const int i = j * TK_THREADS + tid;
        if (i < n4) cur[j] = row[i];
    }
    for (int gbase = 0; gbase < n4; gbase += TK_GROUP * TK_THREADS) {
        const int gnext = gbase + TK_GROUP * TK_THREADS;
#pragma unroll
        for (int j = 0; j < TK_GROUP; ++j) {
            const int i = gnext + j * TK_THREADS + tid;
            if (i < n4) nxt[j] = row[i];
        }
#pragma unroll
        for (int j = 0; j < TK_GROUP; ++j) {
            const int sbase = gbase + j * TK_THREADS;
            if (sbase >= n4) break;  // uniform: the same for every thread
            const int i = sbase + tid;
            uint32_t flags = 0;      // bit c: above; bit 4 + c: equal
            if (i < n4) {
                const float e[4] = {cur[j].x, cur[j].y, cur[j].z, cur[j].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if (4 * i + c >= n) continue;
                    const uint32_t top = key_top(order_key(e[c]), L);
                    if (top > P) flags |= 1u << c;
                    else if (top == P) flags |= 16u << c;
                }
            }
            const uint32_t mine = (uint32_t)__builtin_popcount(flags & 15u) |
                                  ((uint32_t)__builtin_popcount(flags >> 4) << 16);
            uint32_t tot;
            const uint32_t ex = wg_scan(mine, part, &tot) - mine;
            uint32_t gb = run_gt + (ex & 0xffffu), eb = run_eq + (ex >> 16);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                // slots stay below k when the row is not modified during the call; the
                // bound check keeps a caller's race on `scores` from writing past the row
                if ((flags >> c) & 1u) {
                    const uint32_t slot = gb + (eb < r_eff ? eb : r_eff);
                    if (slot < (uint32_t)k) out[slot] = 4 * i + c;
                    ++gb;
                } else if ((flags >> (4 + c)) & 1u) {
                    if (eb < r_eff && gb + eb < (uint32_t)k) out[gb + eb] = 4 * i + c;
                    ++eb;
                }
            }
            run_gt += tot & 0xffffu;
            run_eq += tot >> 16;
        }
#pragma unroll
        for (int j = 0; j < TK_GROUP; ++j) cur[j] = nxt[j];
    }
    const uint32_t taken = run_gt + (run_eq < r_eff ? run_eq : r_eff);
    for (uint32_t j = taken + (uint32_t)tid; j < (uint32_t)k; j += TK_THREADS) out[j] = -1;
}

// ---------------------------------------------------------------------------
// Flag-based selection, shared by the register-resident and the streaming
// kernel.  The threshold is a key range [t_lo, t_hi]: keys above it are taken,
// keys inside it are tied (the first r of them in position order are taken, or
// all).  Byte i of the flags covers positions 4 i .. 4 i + 3: bits 0..3 taken,
// bits 4..7 tied.
// ---------------------------------------------------------------------------
constexpr int TR_J = 16;                                   // most 16-byte pieces per lane
constexpr int TR_MAX_N = TK_THREADS * TR_J * 4;           // 65536 positions
constexpr int TR_CAND = 8192;                              // threshold-bin keys the LDS list holds; staged outputs
constexpr int TR_WAVE_LIST = 1536;                         // lists up to this long are refined by one wave

// order_key in five instructions: x + 0 turns -0 into +0 and keeps every other
// value (subnormals too), a sign-dependent mask orders the bits, and a NaN of
// either sign takes the largest key.
__device__ __forceinline__ uint32_t order_key_sel(float x) {
    const float z = x + 0.0f;
    const uint32_t b = __float_as_uint(z);
    const uint32_t k = b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
    return z != z ? 0xffffffffu : k;
}

// workgroup barrier over LDS only: outstanding global loads stay in flight
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Exclusive sum over the workgroup of one value per thread, *total the sum.  One
// barrier: `part` (TK_WAVES words) must not be in use, and a caller that scans
// again alternates between two of them.
__device__ __forceinline__ uint32_t wg_excl_scan(uint32_t v, uint32_t* part, uint32_t* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t incl = wave_incl_scan(v);
    if (lane == 63) part[w] = incl;
    __syncthreads();
    // (lanes past the waves add 0; every wave scans the 16 sums itself)
    const uint32_t sums = wave_incl_scan(lane < TK_WAVES ? part[lane] : 0u);
    *total = (uint32_t)__builtin_amdgcn_readlane((int)sums, TK_WAVES - 1);
    const uint32_t before = w ? (uint32_t)__builtin_amdgcn_readlane((int)sums, w - 1) : 0u;
    return before + incl - v;
}

// LDS shared by both kernels.
struct TopkLds {
    uint32_t hist[1 << TK_FIRST_BITS];
    uint32_t cand[TR_CAND];        // keys of the threshold bin (streaming: (key, position) pairs); then the output
    uint32_t part[2][TK_WAVES];
    uint32_t found[4];             // digit, keys above its bin, keys in its bin; [3]: list fill
    uint32_t sel[4];               // the threshold found by wave 0: P, L, r, take_all
};

// The bin of hist[0, nbins) holding the r-th key from the top: every thread gets
// its number, the keys in the bins above it and its own count.
template <int NBINS>
__device__ __forceinline__ void find_bin(TopkLds& s, uint32_t r, uint32_t& digit, uint32_t& above, uint32_t& cnt) {
    constexpr int per = NBINS / TK_THREADS;
    const int tid = threadIdx.x;
    uint32_t h[per], sum = 0;
#pragma unroll
    for (int j = 0; j < per; ++j) {
        h[j] = s.hist[tid * per + j];
        sum += h[j];
    }
    uint32_t tot;
    const uint32_t before = wg_excl_scan(sum, s.part[0], &tot);
    uint32_t acc = tot - before - sum;      // keys in the bins of higher threads
#pragma unroll
    for (int j = per - 1; j >= 0; --j) {
        if (acc < r && acc + h[j] >= r) {   // exactly one bin holds the r-th key
            s.found[0] = (uint32_t)(tid * per + j);
            s.found[1] = acc;
            s.found[2] = h[j];
        }
        acc += h[j];
    }
    __syncthreads();
    digit = s.found[0];
    above = s.found[1];
    cnt = s.found[2];
}

// Up to two 10-bit digits over the list of the threshold bin's keys (list[STEP j]): P, L,
// r and take_all refined in place.  The list is complete (after a barrier).  A
// short list is resolved by wave 0 alone (no workgroup barrier per step; lane l
// owns bins 16 l .. 16 l + 15), a long one by the workgroup.
template <int STEP>
__device__ __forceinline__ void resolve_list(TopkLds& s, const uint32_t* list, uint32_t cnt, uint32_t& P, int& L,
                                             uint32_t& r, bool& take_all) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (cnt > (uint32_t)TR_WAVE_LIST) {
        for (; L < 32 && !take_all;) {
            const int shift = 32 - L - TK_NEXT_BITS;
            s.hist[tid] = 0;  // 1024 bins, one per thread
            __syncthreads();
            for (uint32_t j = tid; j < cnt; j += TK_THREADS) {
                const uint32_t kk = list[STEP * j];
                if ((kk >> (32 - L)) == P) atomicAdd(&s.hist[(kk >> shift) & 1023u], 1u);
            }
            __syncthreads();
            uint32_t digit, abv, cn;
            find_bin<1 << TK_NEXT_BITS>(s, r, digit, abv, cn);
            r -= abv;
            P = (P << TK_NEXT_BITS) | digit;
            L += TK_NEXT_BITS;
            take_all = r == cn;
            __syncthreads();   // found is read before the next pass writes it
        }
        return;
    }
    if (w == 0) {
        for (; L < 32 && !take_all;) {
            const int shift = 32 - L - TK_NEXT_BITS;
#pragma unroll
            for (int q = 0; q < 16; ++q) s.hist[64 * q + lane] = 0;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            for (uint32_t j = lane; j < cnt; j += 64) {
                const uint32_t kk = list[STEP * j];
                if ((kk >> (32 - L)) == P) atomicAdd(&s.hist[(kk >> shift) & 1023u], 1u);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            uint32_t hb[16], sum = 0;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                hb[q] = s.hist[16 * lane + q];
                sum += hb[q];
            }
            const uint32_t inc = wave_incl_scan(sum);
            const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
            uint32_t acc = all - inc;   // keys in the bins of higher lanes
            int hit = -1;
            uint32_t h_abv = 0, h_cnt = 0;
#pragma unroll
            for (int q = 15; q >= 0; --q) {
                if (acc < r && acc + hb[q] >= r) {  // one bin of the wave holds the r-th key
                    hit = 16 * lane + q;
                    h_abv = acc;
                    h_cnt = hb[q];
                }
                acc += hb[q];
            }
            const int src = __builtin_ctzll(__ballot(hit >= 0));
            const uint32_t digit = (uint32_t)__builtin_amdgcn_readlane(hit, src);
            r -= (uint32_t)__builtin_amdgcn_readlane((int)h_abv, src);
            const uint32_t cn = (uint32_t)__builtin_amdgcn_readlane((int)h_cnt, src);
            P = (P << TK_NEXT_BITS) | digit;
            L += TK_NEXT_BITS;
            take_all = r == cn;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // bins read before the next clear
        }
        if (lane == 0) {
            s.sel[0] = P;
            s.sel[1] = (uint32_t)L;
            s.sel[2] = r;
            s.sel[3] = take_all ? 1u : 0u;
        }
    }
    __syncthreads();
    P = s.sel[0];
    L = (int)s.sel[1];
    r = s.sel[2];
    take_all = s.sel[3] != 0u;
}

// The key range of prefix P (its top L bits).
__device__ __forceinline__ void key_range(uint32_t P, int L, uint32_t& t_lo, uint32_t& t_hi) {
    t_lo = L == 32 ? P : P << (32 - L);
    t_hi = L == 32 ? P : t_lo | ((1u << (32 - L)) - 1u);
}

// Flags (complete, after a barrier) -> the output row.  Thread t owns dwords
// [D t, D t + D) of the flags, so thread order is position order.  With ties,
// each thread first turns its tied flags of rank below r into taken ones.
__device__ __forceinline__ void emit_flags(TopkLds& s, uint32_t* flags, int D, bool take_all, uint32_t r, int k,
                                           int32_t* __restrict__ out) {
    const int tid = threadIdx.x;
    uint32_t* const mine = flags + tid * D;
    uint32_t tot;
    if (!take_all) {
        uint32_t ties = 0;
        for (int d = 0; d < D; ++d) ties += (uint32_t)__builtin_popcount(mine[d] & 0xf0f0f0f0u);
        const uint32_t before = wg_excl_scan(ties, s.part[0], &tot);
        uint32_t quota = before < r ? r - before : 0u;
        for (int d = 0; d < D; ++d) {
            const uint32_t f = mine[d];
            uint32_t m = f & 0xf0f0f0f0u, take = 0;
            while (m && quota) {
                take |= m & (0u - m);
                m &= m - 1;
                --quota;
            }
            mine[d] = f | (take >> 4);
        }
    }
    uint32_t count = 0;
    for (int d = 0; d < D; ++d) count += (uint32_t)__builtin_popcount(mine[d] & 0x0f0f0f0fu);
    uint32_t slot = wg_excl_scan(count, s.part[1], &tot);
    // staged in LDS and left in coalesced rows when the output fits there (the
    // list is done with).  Slots stay below k when the row is not modified
    // during the call; the bound check keeps a caller's race on `scores` from
    // writing past the row.
    const bool staged = k <= TR_CAND;   // uniform
    for (int d = 0; d < D; ++d) {
        uint32_t m = mine[d] & 0x0f0f0f0fu;
        while (m) {
            const int bit = __builtin_ctz(m);
            m &= m - 1;
            const int pos = 16 * (tid * D + d) + 4 * (bit >> 3) + (bit & 7);
            if (slot < (uint32_t)k) {
                if (staged) s.cand[slot] = (uint32_t)pos;
                else out[slot] = pos;
            }
            ++slot;
        }
    }
    if (staged) {
        for (uint32_t j = tot + (uint32_t)tid; j < (uint32_t)k; j += TK_THREADS) s.cand[j] = 0xffffffffu;
        __syncthreads();
        for (int j = tid; j < k; j += TK_THREADS) out[j] = (int32_t)s.cand[j];
    } else {
        for (uint32_t j = tot + (uint32_t)tid; j < (uint32_t)k; j += TK_THREADS) out[j] = -1;
    }
}

// ---------------------------------------------------------------------------
// Register-resident kernel: rows of at most 4096 J positions.  The row is read
// from HBM once: lane tid keeps the keys of its J 16-byte pieces (positions
// 4 (j * 1024 + tid) + c) in registers.  J is the smallest that holds n_max; a
// row shorter than n_max skips the pieces past its end (a row of 1,152 of 65,536
// positions took 69 us when they were counted into one bin).
// What bounds it: 256 rows of 65,536 (67 MB) are loaded in about 17 us, with the
// keys and the histogram under the loads; the threshold, the flags and the
// output then run with the memory idle: 24.1 to 24.8 us in all (three score sets in
// turn; 26 with five, 320 MB, more than the MALL holds).  Ranking every key
// against ballots, prefix tables and a slot per key took 35.2 us; flags cost two
// to three instructions per key, and only taken positions pay for a slot.
// ---------------------------------------------------------------------------
template <int J>
__global__ __launch_bounds__(TK_THREADS) void dsa_topk_reg_kernel(
    const float* __restrict__ scores, int64_t score_stride, const int32_t* __restrict__ lengths,
    int32_t n_max, int32_t k, int32_t* __restrict__ indices, int64_t idx_stride) {
    __shared__ TopkLds s;
    constexpr int D = (J + 3) / 4;                          // dwords of flags per thread
    __shared__ __attribute__((aligned(16))) uint32_t flags[TK_THREADS * D];

    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t t = blockIdx.x;
    int n = lengths ? lengths[t] : n_max;
    n = n < 0 ? 0 : (n > n_max ? n_max : n);
    const float4* row = reinterpret_cast<const float4*>(scores + t * score_stride);
    int32_t* out = indices + t * idx_stride;
    if (n <= k) {  // uniform: every position, in order
        for (int j = tid; j < k; j += TK_THREADS) out[j] = j < n ? j : -1;
        return;
    }
    const int n4 = (n + 3) >> 2;
    const int nj = (n4 + TK_THREADS - 1) / TK_THREADS;      // pieces that hold positions
    const int full = n / (4 * TK_THREADS);                  // pieces without a position past the row

    // Pieces past the row re-read its last piece (in bounds); their keys are 0,
    // below every valid key (the smallest, -inf, is 0x007fffff).  The loads run
    // PF pieces ahead of the keys and the histogram, so that the waves of a SIMD
    // compute while later pieces are in flight.
    constexpr int PF = J < 7 ? J : 7;
    float4 v[J];
#pragma unroll
    for (int j = 0; j < PF; ++j) v[j] = row[min(j * TK_THREADS + tid, n4 - 1)];
    for (int b = tid; b < (1 << TK_FIRST_BITS); b += TK_THREADS) s.hist[b] = 0;
    if (J < 4) flags[tid] = 0;                              // bytes past the pieces
    if (tid == 0) s.found[3] = 0;
    lds_barrier();
    uint32_t key[J][4];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        if (j + PF < J) v[j + PF] = row[min((j + PF) * TK_THREADS + tid, n4 - 1)];
        const float e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) key[j][c] = order_key_sel(e[c]);
        if (j < full) {
#pragma unroll
            for (int c = 0; c < 4; ++c) atomicAdd(&s.hist[key[j][c] >> (32 - TK_FIRST_BITS)], 1u);
        } else {
            const int left = n - 4 * (j * TK_THREADS + tid);    // positions of this lane's piece in the row
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                key[j][c] = c < left ? key[j][c] : 0u;
                if (c < left) atomicAdd(&s.hist[key[j][c] >> (32 - TK_FIRST_BITS)], 1u);
            }
        }
    }
    __syncthreads();

    uint32_t t_lo, t_hi, r = (uint32_t)k, P, above, cnt;
    bool take_all = false;
    int L = TK_FIRST_BITS;
    find_bin<1 << TK_FIRST_BITS>(s, r, P, above, cnt);
    r -= above;
    take_all = r == cnt;
    if (!take_all && cnt <= (uint32_t)TR_CAND) {
        // the bin's keys into the LDS list (any order): per-lane counts, a wave
        // scan, one list reservation per wave
        uint32_t mine = 0;
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c) mine += (key[j][c] >> (32 - TK_FIRST_BITS)) == P ? 1u : 0u;
        const uint32_t incl = wave_incl_scan(mine);
        uint32_t base = 0;
        if (lane == 63) base = atomicAdd(&s.found[3], incl);
        uint32_t pos = (uint32_t)__builtin_amdgcn_readlane((int)base, 63) + incl - mine;
        if (mine) {
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if ((key[j][c] >> (32 - TK_FIRST_BITS)) == P) s.cand[pos++] = key[j][c];
        }
        __syncthreads();   // the list is complete
        resolve_list<1>(s, s.cand, cnt, P, L, r, take_all);
    } else if (!take_all) {
        // more tied keys than the list holds: the two digits over the registers;
        // a key outside the prefix counts in a bin of its lane's own (no two lanes
        // of a wave share it), so the code stays free of branches
        for (; L < 32 && !take_all;) {
            const int shift = 32 - L - TK_NEXT_BITS;
            __syncthreads();
            s.hist[tid] = 0;
            if (tid < 64) s.hist[1024 + tid] = 0;
            __syncthreads();
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint32_t kk = key[j][c];
                    const bool in = (kk >> (32 - L)) == P;
                    atomicAdd(&s.hist[in ? (kk >> shift) & 1023u : 1024u + lane], 1u);
                }
            __syncthreads();
            uint32_t digit, abv, cn;
            find_bin<1 << TK_NEXT_BITS>(s, r, digit, abv, cn);
            r -= abv;
            P = (P << TK_NEXT_BITS) | digit;
            L += TK_NEXT_BITS;
            take_all = r == cn;
        }
    }
    key_range(P, L, t_lo, t_hi);

    // flags: one compare per key when every tied key is taken, two otherwise
    unsigned char* const fb = reinterpret_cast<unsigned char*>(flags);
    const uint32_t taken_from = take_all ? t_lo : t_hi + 1u;    // (t_hi = 0xffffffff: nothing lies above)
    const bool none_above = !take_all && t_hi == 0xffffffffu;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        uint32_t f = 0;
        if (j < nj) {
#pragma unroll
            for (int c = 0; c < 4; ++c) f |= (key[j][c] >= taken_from ? 1u : 0u) << c;
            if (none_above) f = 0;
            if (!take_all) {
#pragma unroll
                for (int c = 0; c < 4; ++c) f |= (key[j][c] >= t_lo && key[j][c] <= t_hi ? 16u : 0u) << c;
            }
        }
        fb[j * TK_THREADS + tid] = (unsigned char)f;
    }
    __syncthreads();
    emit_flags(s, flags, D, take_all, r, k, out);
}

// ---------------------------------------------------------------------------
// Streaming kernel: rows of more than 65,536 and at most TS_MAX_N positions,
// whose flags fit LDS.  Two reads of the row: the 12-bit histogram; then the
// flags of the keys above the bin, and the bin's (key, position) pairs into the
// LDS list, whose threshold then sets the rest of the flags.  A bin with more
// keys than the list holds is refined by 10-bit passes over the row first.
// Against the ordered two-read kernel (one workgroup scan per 4096 positions):
// 263 rows of 102,073 positions 84 us instead of 130, 3 rows of 128,850 50.5
// instead of 76.6.
// ---------------------------------------------------------------------------
constexpr int TS_CAND = TR_CAND / 2;                        // (key, position) pairs the list holds
constexpr int TS_MAX_N = 393216;                            // 96 KB of flags
constexpr int TS_UNROLL = 8;                                // pieces in flight per lane

__global__ __launch_bounds__(TK_THREADS) void dsa_topk_stream_kernel(
    const float* __restrict__ scores, int64_t score_stride, const int32_t* __restrict__ lengths,
    int32_t n_max, int32_t k, int32_t* __restrict__ indices, int64_t idx_stride) {
    __shared__ TopkLds s;
    extern __shared__ __attribute__((aligned(16))) uint32_t ts_flags[];    // n_max / 4 bytes, whole dwords per thread

    const int tid = threadIdx.x;
    const int64_t t = blockIdx.x;
    int n = lengths ? lengths[t] : n_max;
    n = n < 0 ? 0 : (n > n_max ? n_max : n);
    const float4* row = reinterpret_cast<const float4*>(scores + t * score_stride);
    int32_t* out = indices + t * idx_stride;
    if (n <= k) {  // uniform: every position, in order
        for (int j = tid; j < k; j += TK_THREADS) out[j] = j < n ? j : -1;
        return;
    }
    const int n4 = (n + 3) >> 2;
    const int D = (n4 + 4 * TK_THREADS - 1) / (4 * TK_THREADS);     // dwords of flags per thread
    // one pass over the row: fn(piece, its four keys; 0 past the row, below every valid key)
    auto sweep = [&](auto&& fn) {
        for (int i0 = tid; i0 < n4; i0 += TK_THREADS * TS_UNROLL) {
            float4 v[TS_UNROLL];
#pragma unroll
            for (int j = 0; j < TS_UNROLL; ++j) v[j] = row[min(i0 + j * TK_THREADS, n4 - 1)];
#pragma unroll
            for (int j = 0; j < TS_UNROLL; ++j) {
                const int i = i0 + j * TK_THREADS;
                if (i >= n4) continue;
                const float e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
                uint32_t key[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) key[c] = 4 * i + c < n ? order_key_sel(e[c]) : 0u;
                fn(i, key);
            }
        }
    };
    uint32_t P = 0, r = (uint32_t)k, cnt = 0, above;
    int L = 0;
    bool take_all = false;
    // 12 bits, then 10 more at a time while the bin's keys do not fit the list
    for (int pass = 0; pass < 3 && !take_all; ++pass) {
        const int bits = pass == 0 ? TK_FIRST_BITS : TK_NEXT_BITS;
        const int shift = 32 - L - bits;
        for (int b = tid; b < (1 << bits); b += TK_THREADS) s.hist[b] = 0;
        if (tid == 0) s.found[3] = 0;
        __syncthreads();
        sweep([&](int, const uint32_t (&key)[4]) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (key[c] && key_top(key[c], L) == P) atomicAdd(&s.hist[(key[c] >> shift) & ((1u << bits) - 1u)], 1u);
        });
        __syncthreads();
        uint32_t digit;
        if (pass == 0) find_bin<1 << TK_FIRST_BITS>(s, r, digit, above, cnt);
        else find_bin<1 << TK_NEXT_BITS>(s, r, digit, above, cnt);
        r -= above;
        P = (P << bits) | digit;
        L += bits;
        take_all = r == cnt;
        __syncthreads();   // found is read before the next pass writes it
        if (cnt <= (uint32_t)TS_CAND) break;
    }
    const bool list = !take_all && L < 32;      // (cnt fits: a longer bin is refined to 32 bits)
    uint32_t t_lo, t_hi;
    key_range(P, L, t_lo, t_hi);
    unsigned char* const fb = reinterpret_cast<unsigned char*>(ts_flags);
    for (int i = n4 + tid; i < 4 * TK_THREADS * D; i += TK_THREADS) fb[i] = 0;    // past the row
    sweep([&](int i, const uint32_t (&key)[4]) {
        uint32_t f = 0, in = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            f |= (key[c] > t_hi ? 1u : 0u) << c;
            in |= (key[c] >= t_lo && key[c] <= t_hi ? 1u : 0u) << c;
        }
        if (take_all) f |= in;
        else if (!list) f |= in << 4;
        else if (in) {
            uint32_t at = atomicAdd(&s.found[3], (uint32_t)__builtin_popcount(in));
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if ((in >> c) & 1u) {
                    // (the list holds the bin when the row is not modified during the call)
                    if (at < (uint32_t)TS_CAND) {
                        s.cand[2 * at] = key[c];
                        s.cand[2 * at + 1] = (uint32_t)(4 * i + c);
                    }
                    ++at;
                }
        }
        fb[i] = (unsigned char)f;
    });
    __syncthreads();
    if (list) {
        const uint32_t held = min(min(s.found[3], cnt), (uint32_t)TS_CAND);
        resolve_list<2>(s, s.cand, held, P, L, r, take_all);
        key_range(P, L, t_lo, t_hi);
        for (uint32_t j = tid; j < held; j += TK_THREADS) {
            const uint32_t kk = s.cand[2 * j], pos = s.cand[2 * j + 1];
            const bool tied = kk >= t_lo && kk <= t_hi;
            const uint32_t bit = kk > t_hi || (tied && take_all) ? 1u : (tied ? 16u : 0u);
            if (bit) atomicOr(&ts_flags[pos >> 4], bit << (8 * ((pos >> 2) & 3) + (pos & 3)));
        }
        __syncthreads();
    }
    emit_flags(s, ts_flags, D, take_all, r, k, out);
}

template <int J>
void launch_reg(const float* scores, int64_t score_stride, const int32_t* lengths, int32_t n_tokens, int32_t n_max,
                int32_t topk, int32_t* indices, int64_t idx_stride, hipStream_t st) {
    hipLaunchKernelGGL(dsa_topk_reg_kernel<J>, dim3((unsigned)n_tokens), dim3(TK_THREADS), 0, st, scores, score_stride,
                       lengths, n_max, topk, indices, idx_stride);
}

}  // namespace

extern "C" {

int dsa_topk_indices(const float* scores, int64_t score_stride, const int32_t* lengths, int32_t n_tokens,
                     int32_t n_max, int32_t topk, int32_t* indices, int64_t idx_stride, void* stream) {
    if (n_tokens < 0 || n_max < 0 || topk < 0 || n_max > DSA_TOPK_MAX_N) return DSA_ERR_BAD_SHAPE;
    if (n_tokens == 0 || topk == 0) return DSA_OK;
    if (!indices || (n_max > 0 && !scores)) return DSA_ERR_NULL_POINTER;
    if (idx_stride < topk || score_stride < n_max) return DSA_ERR_BAD_SHAPE;
    if ((score_stride % 4) || ((uintptr_t)scores & 15) || ((uintptr_t)indices & 3)) return DSA_ERR_BAD_STRIDE;
    hipStream_t st = (hipStream_t)stream;
    if (n_max <= TR_MAX_N) {
        // the fewest pieces per lane that hold the row
        auto launch = n_max <= 4096 ? launch_reg<1>
                      : n_max <= 8192 ? launch_reg<2>
                      : n_max <= 16384 ? launch_reg<4>
                      : n_max <= 32768 ? launch_reg<8> : launch_reg<16>;
        launch(scores, score_stride, lengths, n_tokens, n_max, topk, indices, idx_stride, st);
    } else if (n_max <= TS_MAX_N) {
        const size_t flags = (size_t)((n_max + 16 * TK_THREADS - 1) / (16 * TK_THREADS)) * (4 * TK_THREADS);
        hipLaunchKernelGGL(dsa_topk_stream_kernel, dim3((unsigned)n_tokens), dim3(TK_THREADS), flags, st, scores,
                           score_stride, lengths, n_max, topk, indices, idx_stride);
    } else {
        hipLaunchKernelGGL(dsa_topk_kernel, dim3((unsigned)n_tokens), dim3(TK_THREADS), 0, st, scores, score_stride,
                           lengths, n_max, topk, indices, idx_stride);
    }
    return hipGetLastError() == hipSuccess ? DSA_OK : DSA_ERR_HIP;
}

}  // extern "C"
