// dsa_indexer.hip - the DSA index scorer for gfx950 (MI355X).
//
//   score[b][t][j] = sum_h weights[b][t][h] * max(0, q[b][t][h] . k[j])
//
// (the DeepSeek-V3.2 lightning indexer's score; the reference has no indexer,
// so the contract is the library's own and is spelled out in
// include/dsa_indexer.h).  It feeds dsa_topk_indices, which selects the
// top-k positions per query token.
//
// A GEMM per sequence, Q [tokens x H_I, 128] against K [positions, 128], with
// a ReLU and a weighted sum over the index heads fused into its epilogue:
// - a group is up to 128 (token, index head) rows of one sequence, so that the
//   MTP tokens of a sequence (H_I = 64: two tokens) read each k row once.  The
//   chunks of 128 positions of all groups are dealt out to at most 512 workgroups
//   (two per CU), each taking one run of them that counts what a group's start
//   (Q, lengths, first rows) costs (dsa_deal.h): whatever the lengths are, the
//   CUs finish together, and a short call still spreads over the chip.  Short
//   lists get whole workgroups per group instead (launch_ix).  With
//   a workgroup per 2048 positions the starts and the last, partly filled round
//   took a quarter of the time (2 tokens x 32 sequences of 35 K to 100 K
//   positions, 570 MB: 158 us, wave-private rings below alone 154 us; 512- and
//   1024-position workgroups 197 and 166 us);
// - Q stays in VGPRs as the A operand of v_mfma_f32_32x32x16_bf16 (NB blocks of
//   32 rows x 128 dims: 32 VGPRs per block); a call with fewer (token, head)
//   rows than 128 per sequence takes fewer blocks, so that no MFMA and no
//   epilogue is spent on rows of tokens that do not exist;
// - every wave works alone: of each 128 positions it takes 32, brings their k
//   rows by LDS-DMA (8 KB) into its own two-slot ring and reads them as the B
//   operand (NB x 8 MFMAs), then forms per position the weighted ReLU sum over
//   its token's rows (16 accumulator registers and one cross-half exchange per
//   row block).  A slot is refilled as soon as its last fragment is in
//   registers, before the epilogue; no barrier ties the waves together;
// - HBM bounds it when each k row is read once: 114 us for those 570 MB (5.0
//   TB/s, a plain copy moves 5.1), 131 us without the non-temporal mark on rows
//   that a single group reads.  Many tokens on one sequence (512 tokens x 16 K
//   positions) are bound by the MFMAs and the epilogue's two VALU instructions
//   per (head, position) instead.
// Bytes per position: one 256-byte k row per sequence (all its tokens), 4-byte
// scores per token; flops: 2 * 128 per (token, head, position).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <algorithm>

#include "../../include/dsa_indexer.h"
#include "dsa_deal.h"
#include "dsa_lds.h"

namespace {

constexpr int IX_D = DSA_INDEXER_D;        // 128 values per index vector
constexpr int IX_NTHR = 256;
constexpr int IX_NW = IX_NTHR / 64;
constexpr int IX_CHUNK = 128;              // positions per chunk (32 per wave)
constexpr int IX_WGS = 512;                // workgroups of a full grid: two per CU
constexpr int IX_TINY = 4, IX_SHORT = 16;  // chunks of the longest list that a call may hold
constexpr int IX_MOST_WGS = 1 << 20;       // workgroups of a grid of one per group (a grid has a limit, the even deal none)
constexpr int IX_LOOK = 4;                 // steps whose entries and rows a wave holds in LDS
constexpr int IX_KS = IX_D / 16;           // k-steps of 16
constexpr int IX_ROW = IX_D * 2;           // bytes of a k row (in LDS too: swizzled, unpadded)
constexpr int IX_SLOT = 32 * IX_ROW;       // a wave's rows of a chunk (8 KB); two slots per wave
constexpr int IX_LPW = 32 / 4;             // LDS-DMA loads (4 rows of 256 B each) per wave per chunk

typedef __bf16 ix_bf16x8 __attribute__((ext_vector_type(8)));

struct IxParams {
    const __bf16* q;
    int64_t q_sb, q_st, q_sh;
    const float* w;
    const unsigned char* k;
    int64_t k_rows, k_row_bytes;
    const int32_t* bt;
    int64_t bt_stride;
    int32_t bs, bs_shift;        // bs_shift: log2(bs) when a power of two, else -1
    int64_t groups;              // sequences x token groups
    int64_t k_bstride;
    const int32_t* seq_lens;
    float* scores;
    int64_t s_stride;
    int32_t s_q, n_cols, causal, tgroups;
    int32_t parts;               // > 0: workgroups per group; 0: an even deal of all chunks
};

// Positions j of token t of sequence b: j < min(len(b, t), n_cols).
__device__ __forceinline__ int64_t ix_len(const IxParams& p, int64_t L, int t) {
    const int64_t len = p.causal ? L - (p.s_q - 1 - t) : L;
    return min(max(len, (int64_t)0), (int64_t)p.n_cols);
}

// Inclusive sums over the workgroup, of one value per thread (*sum) and of the
// values that are not 0 (*some), and their totals.
__device__ __forceinline__ void ix_scan(uint32_t v, LDS_AS uint32_t* part, uint32_t* sum, uint32_t* some,
                                        uint32_t* all, uint32_t* all_some) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t any = __builtin_amdgcn_ballot_w64(v != 0);
    uint32_t cn = (uint32_t)__builtin_popcountll(any & (~0ull >> (63 - lane)));
    v = wave_incl_scan(v);
    if (lane == 63) {
        part[2 * wave] = v;
        part[2 * wave + 1] = cn;
    }
    __syncthreads();
    uint32_t a = 0, an = 0;
#pragma unroll
    for (int w = 0; w < IX_NW; ++w) {
        v += w < wave ? part[2 * w] : 0u;
        cn += w < wave ? part[2 * w + 1] : 0u;
        a += part[2 * w];
        an += part[2 * w + 1];
    }
    __syncthreads();
    *sum = v;
    *some = cn;
    *all = a;
    *all_some = an;
}

// max(x, 0), 0 for NaN, as the median of x, 0 and inf (an infinity that the
// compiler cannot see: it would turn the median into fmaxf, which takes a second
// instruction to quiet a signalling NaN first: a third of the epilogue).
__device__ __forceinline__ float relu(float x, float inf) { return __builtin_amdgcn_fmed3f(x, 0.0f, inf); }

// 4-byte LDS-DMA load: lane l's word lands at lds_wave_base + 4 l (tracked like
// lds_dma16 by explicit vmcnt waits).
__device__ __forceinline__ void ix_dma4(const void* gsrc, lds_ptr lds_wave_base) {
    const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds_wave_base);
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dword %1, off"
        :
        : "s"(m0v), "v"(gsrc)
        : "memory", "m0");
}

// lds_dma16 for rows that no other workgroup reads: marked non-temporal.
__device__ __forceinline__ void ix_dma16_once(const void* gsrc, lds_ptr lds_wave_base) {
    const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds_wave_base);
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, off nt"
        :
        : "s"(m0v), "v"(gsrc)
        : "memory", "m0");
}

template <int N>
__device__ __forceinline__ void ix_wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// HI index heads per token; NB 32-row blocks of Q, each of one token: 32 NB / HI
// tokens per group.  ONCE: one group per sequence, each k row is read once.
template <int HI, int NB, bool ONCE>
__global__ void __launch_bounds__(IX_NTHR) __attribute__((amdgpu_waves_per_eu(2, 2)))
dsa_indexer_kernel(const IxParams p) {
    constexpr int QROWS = 32 * NB;
    constexpr int TPW = QROWS / HI;
    __shared__ __attribute__((aligned(1024))) unsigned char s_k[IX_NW * 2 * IX_SLOT];
    __shared__ __attribute__((aligned(256))) int32_t s_ent[IX_NW * IX_LOOK * 64];   // block-table entries in flight
    __shared__ __attribute__((aligned(16))) uint64_t s_off[IX_NW * IX_LOOK * 32];   // byte offsets of the k rows
    __shared__ int32_t s_bad[IX_NW * IX_LOOK * 32];                                 // 1: the row is outside the cache
    __shared__ __attribute__((aligned(16))) float s_w[QROWS];
    __shared__ uint32_t s_part_arr[2 * IX_NW];
    __shared__ uint32_t s_at[4];              // the workgroup's first group and chunk, its last group and the chunk it ends before

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hi = lane >> 5, r32 = lane & 31;
    const bool any_rows = p.k_rows > 0;
    LDS_AS uint32_t* const s_part = (LDS_AS uint32_t*)s_part_arr;

    // ---- this workgroup's chunks: a run of all groups' chunks, in (sequence,
    // token group, position) order, or its part of one group (dsa_deal.h).  Group
    // g's list is its last token's (the lists grow with t).  A group holds at most
    // 2^24 chunks and a block of IX_NTHR groups fewer than 2^32; the totals are 64
    // bits ----
    auto seq_of = [&](int g) -> int { return ONCE ? g : (int)((unsigned)g / (unsigned)p.tgroups); };
    auto group_chunks = [&](int64_t g64) -> uint32_t {
        if (g64 >= p.groups) return 0u;
        const int g = (int)g64, b = seq_of(g), t0 = (g - b * p.tgroups) * TPW;
        return (uint32_t)((ix_len(p, p.seq_lens[b], min(t0 + TPW, p.s_q) - 1) + IX_CHUNK - 1) / IX_CHUNK);
    };
    const uint32_t G = gridDim.x, x = blockIdx.x;
    int g, g_last;
    uint32_t c_first, c_last;                      // first chunk of group g; end of group g_last's
    if (p.parts) {
        // whole workgroups per group
        g = g_last = (int)(x / (uint32_t)p.parts);
        dsa_deal::part_of(group_chunks(g), (uint32_t)p.parts, x - (uint32_t)g * (uint32_t)p.parts, &c_first, &c_last);
        if (c_first >= c_last) return;
    } else {
        uint64_t all = 0, some = 0;
        uint32_t n0 = 0, sum0 = 0, some0 = 0;      // of groups 0 .. IX_NTHR - 1
        for (int64_t g0 = 0; g0 < p.groups; g0 += IX_NTHR) {
            const uint32_t n = group_chunks(g0 + tid);
            uint32_t sum, cnt, tot, tot_n;
            ix_scan(n, s_part, &sum, &cnt, &tot, &tot_n);
            if (g0 == 0) { n0 = n; sum0 = sum; some0 = cnt; }
            all += tot;
            some += tot_n;
        }
        const dsa_deal::Deal deal = dsa_deal::deal_of(all, some, G, ONCE ? dsa_deal::START_ONCE : dsa_deal::START);
        uint64_t first, last;
        dsa_deal::run_of(deal, x, &first, &last);
        if (first >= last) return;
        // the groups holding units `first` and `last - 1`: exactly one thread finds each
        const bool once = p.groups <= IX_NTHR;
        uint64_t base = 0;
        for (int64_t g0 = 0; g0 < p.groups && base < last; g0 += IX_NTHR) {
            uint32_t n = n0, sum = sum0, cnt = some0, tot = 0, tot_n = 0;
            if (!once) {
                n = group_chunks(g0 + tid);
                ix_scan(n, s_part, &sum, &cnt, &tot, &tot_n);
            }
            const uint64_t end = base + sum + (uint64_t)deal.start * cnt, begin = end - dsa_deal::units(deal, n);
            if (begin <= first && first < end) {
                s_at[0] = (uint32_t)(g0 + tid);
                s_at[1] = dsa_deal::chunks_before(deal, first - begin);
            }
            if (begin < last && last <= end) {
                s_at[2] = (uint32_t)(g0 + tid);
                s_at[3] = dsa_deal::chunks_before(deal, last - begin);
            }
            base += tot + (uint64_t)deal.start * tot_n;
        }
        __syncthreads();
        g = __builtin_amdgcn_readfirstlane((int)s_at[0]);
        c_first = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_at[1]);
        g_last = __builtin_amdgcn_readfirstlane((int)s_at[2]);
        c_last = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_at[3]);
    }

    const lds_ptr ring = (lds_ptr)s_k + wave * 2 * IX_SLOT;
    LDS_AS int32_t* const ents = (LDS_AS int32_t*)s_ent + wave * IX_LOOK * 64;
    LDS_AS uint64_t* const offs = (LDS_AS uint64_t*)s_off + wave * IX_LOOK * 32;
    LDS_AS int32_t* const bads = (LDS_AS int32_t*)s_bad + wave * IX_LOOK * 32;

    float inf = INFINITY;
    asm volatile("" : "+s"(inf));
    for (; g <= g_last; ++g, c_first = 0) {
        const int b = seq_of(g);
        const int t0 = (g - b * p.tgroups) * TPW;
        const int ntok = min(TPW, p.s_q - t0);
        const int64_t L = p.seq_lens[b];
        const int32_t lmax = (int32_t)ix_len(p, L, t0 + ntok - 1);
        const uint32_t c_end = g == g_last ? c_last : (uint32_t)((lmax + (IX_CHUNK - 1ll)) / IX_CHUNK);
        if (c_first >= c_end) continue;        // (an empty list, or the run ends in its start units)
        const int c0 = (int)c_first, m = (int)(c_end - c_first);

        // ---- Q (A operand): lane (r32, hi) holds rows 32qb + r32, dims 16ks + 8hi .. +7 ----
        u32x4 qf[NB][IX_KS];
#pragma unroll
        for (int qb = 0; qb < NB; ++qb) {
            const int qrow = 32 * qb + r32;
            const int tl = min(qrow / HI, ntok - 1);   // rows of a missing token: a copy, never stored
            const __bf16* qp =
                p.q + (int64_t)b * p.q_sb + (int64_t)(t0 + tl) * p.q_st + (int64_t)(qrow % HI) * p.q_sh + 8 * hi;
#pragma unroll
            for (int ks = 0; ks < IX_KS; ++ks) qf[qb][ks] = *reinterpret_cast<const u32x4*>(qp + 16 * ks);
        }
        __syncthreads();                       // every wave is done with the last group's weights
        if (tid < QROWS) {
            const int tl = min(tid / HI, ntok - 1);
            s_w[tid] = p.w[((int64_t)b * p.s_q + t0 + tl) * HI + tid % HI];
        }
        int32_t len_t[TPW];
#pragma unroll
        for (int tk = 0; tk < TPW; ++tk) len_t[tk] = tk < ntok ? (int32_t)ix_len(p, L, t0 + tk) : 0;

        // This wave's step k: positions 128 (c0 + k) + 32 wave .. +31, below lmax
        // for k < n.  Three stages, each a fixed number of vector-memory
        // accesses, so that explicit vmcnt waits can count them:
        //   look(k)   (paged) the positions' block-table entries, one LDS-DMA load
        //   fetch(k)  their k rows -> ring slot k & 1, IX_LPW LDS-DMA loads: load i
        //             brings rows 4i .. 4i+3 (16 lanes x 16 bytes per row); a row's
        //             16-byte piece d is stored at slot position d ^ (row & 15), so
        //             the B-operand reads below (32 rows, one piece each) spread
        //             over the banks.  A row outside the cache is read from row 0
        //             and scored -inf; a position past the list copies the last.
        //   score(k)  the MFMAs, the weighted ReLU sums, and the stores
        // Step k issues fetch(k + 2) when its fragments are in registers, and
        // look(k + 4) behind it.
        const int64_t j00 = (int64_t)c0 * IX_CHUNK + 32 * wave;
        const int n = j00 < lmax ? min(m, (int)((lmax - j00 + IX_CHUNK - 1) / IX_CHUNK)) : 0;
        const int32_t* const bt = p.bt ? p.bt + (int64_t)b * p.bt_stride : nullptr;
        // (per-lane offsets from opaque copies of the lane id: hoisted out of the
        // loop they would spill beside Q and the accumulators)
        const int32_t j0 = (int32_t)j00;
        auto pos = [&](int k, int ln) -> int32_t {
            return (int32_t)min((uint32_t)j0 + (uint32_t)(k * IX_CHUNK + (ln & 31)), (uint32_t)lmax - 1u);
        };
        auto look = [&](int k) {
            const int32_t j = pos(k, opaque(lane));
            ix_dma4(bt + (p.bs_shift >= 0 ? j >> p.bs_shift : j / p.bs), (lds_ptr)(ents + (k & (IX_LOOK - 1)) * 64));
        };
        auto fetch = [&](int k) {
            const int ln = opaque(lane);
            const int32_t j = pos(k, ln);
            int64_t phys = (int64_t)b * p.k_bstride + j;
            if (bt)
                phys = (int64_t)ents[(k & (IX_LOOK - 1)) * 64 + ln] * p.bs +
                       (p.bs_shift >= 0 ? j & (p.bs - 1) : j % p.bs);
            // one lane per position forms the row's address (both halves the same);
            // the lanes that load a row read it back
            const int at = (k & (IX_LOOK - 1)) * 32;
            const bool in = phys >= 0 && phys < p.k_rows;
            offs[at + (ln & 31)] = in ? (uint64_t)phys * (uint64_t)p.k_row_bytes : 0;
            bads[at + (ln & 31)] = in ? 0 : 1;
            if (!any_rows) return;
            uint64_t off[IX_LPW];
#pragma unroll
            for (int i = 0; i < IX_LPW; ++i) off[i] = offs[at + 4 * i + (ln >> 4)];
#pragma unroll
            for (int i = 0; i < IX_LPW; ++i) {
                const int piece = (ln & 15) ^ ((4 * i + (ln >> 4)) & 15);
                const lds_ptr to = ring + (k & 1) * IX_SLOT + 4 * i * IX_ROW;
                if constexpr (ONCE) ix_dma16_once(p.k + off[i] + 16 * piece, to);
                else lds_dma16(p.k + off[i] + 16 * piece, to);
            }
        };
        float held[TPW];      // step k's scores, stored in step k + 1
        auto store = [&](int k) {
            const int ln = opaque(lane);
            const uint32_t j = (uint32_t)j0 + (uint32_t)(k * IX_CHUNK + (ln & 31));
            const bool bad = bads[(k & (IX_LOOK - 1)) * 32 + (ln & 31)] != 0;
#pragma unroll
            for (int tk = 0; tk < TPW; ++tk)
                // token tk's score leaves through the lanes of half (tk & 1)
                if ((tk & 1) == (ln >> 5) && j < (uint32_t)len_t[tk])
                    p.scores[((int64_t)b * p.s_q + t0 + tk) * p.s_stride + j] = bad ? -INFINITY : held[tk];
        };
        if (bt && n > 0) look(0);
        if (bt && n > 1) look(1);
        wait_vm<0>();                          // Q, weights (a wait that the compiler counts too)
        ix_wait_vm<0>();                       // and the first entries
        __syncthreads();
        if (n > 0) fetch(0);
        if (bt && n > 2) look(2);
        if (n > 1) fetch(1);
        if (bt && n > 3) look(3);
        for (int k = 0; k < n; ++k) {
            // fetch(k) landed.  Newer accesses: look(k + 2), the stores of k - 2
            // (counted as none), fetch(k + 1), look(k + 3).
            if (bt && k + 3 < n) ix_wait_vm<IX_LPW + 2>();
            else if (k + 1 < n) ix_wait_vm<IX_LPW>();
            else ix_wait_vm<0>();
            f32x16 acc[NB];
#pragma unroll
            for (int qb = 0; qb < NB; ++qb) acc[qb] = f32x16{};
            // B operand: lane (r32, hi) holds k row r32 of the slot, dims 16ks + 8hi .. +7
            const int ln = opaque(lane);
            const lds_cptr kr = ring + (k & 1) * IX_SLOT + (ln & 31) * IX_ROW;
            if (any_rows) {
#pragma unroll
                for (int ks = 0; ks < IX_KS; ++ks) {
                    const u32x4 kf = lds_ld<u32x4>(kr + 16 * ((2 * ks + (ln >> 5)) ^ (ln & 15)));
#pragma unroll
                    for (int qb = 0; qb < NB; ++qb)
                        acc[qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ix_bf16x8, qf[qb][ks]),
                                                                          __builtin_bit_cast(ix_bf16x8, kf), acc[qb],
                                                                          0, 0, 0);
                }
            }
            if (k > 0) store(k - 1);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // every read of the slot has returned
            if (k + 2 < n) {
                // look(k + 2) landed.  Newer: fetch(k + 1), look(k + 3), the stores of k - 2 and k - 1.
                if (bt && k + 3 < n) ix_wait_vm<IX_LPW + 1>();
                else if (bt) ix_wait_vm<IX_LPW>();
                fetch(k + 2);
                if (bt && k + 4 < n) look(k + 4);
            }
            // ---- lane (r32, hi) has position r32 of the step, and in register r of
            // row block qb the row 32qb + 8(r/4) + 4hi + r%4.  Token tk: row blocks
            // tk * HI / 32 .. (tk + 1) * HI / 32 - 1 ----
#pragma unroll
            for (int tk = 0; tk < TPW; ++tk) {
                f32x4 part = {0.0f, 0.0f, 0.0f, 0.0f};     // four chains: a single one is latency-bound
#pragma unroll
                for (int qb = tk * HI / 32; qb < (tk + 1) * HI / 32; ++qb) {
#pragma unroll
                    for (int r4 = 0; r4 < 4; ++r4) {
                        const f32x4 wv = lds_ld<f32x4>((lds_cptr)s_w + 4 * (32 * qb + 8 * r4 + 4 * (ln >> 5)));
#pragma unroll
                        for (int e = 0; e < 4; ++e) part[e] += wv[e] * relu(acc[qb][4 * r4 + e], inf);
                    }
                }
                const float sum = (part[0] + part[1]) + (part[2] + part[3]);
                held[tk] = sum + __shfl_xor(sum, 32, 64);
            }
        }
        if (n > 0) store(n - 1);
    }
}

template <int HI, int NB>
int launch_ix(IxParams& p, int B, hipStream_t st) {
    constexpr int TPW = 32 * NB / HI;
    p.tgroups = (p.s_q + TPW - 1) / TPW;
    p.groups = (int64_t)B * p.tgroups;
    // two workgroups per CU, but no more than the chunks the lists can hold
    const int64_t most = (p.n_cols + (int64_t)IX_CHUNK - 1) / IX_CHUNK;
    const bool once = p.tgroups == 1;          // (always for NB < 4: chosen by s_q)
    int64_t wgs = p.groups >= IX_WGS || most >= IX_WGS ? IX_WGS : std::min<int64_t>(p.groups * most, IX_WGS);
    // Whole workgroups per group, which start once and need no scan of the lengths
    // (about a microsecond):
    // - lists of up to IX_TINY chunks, in as many workgroups per group as one per CU
    //   gives: a second one there splits too few chunks to be worth its start (200
    //   sequences x 3 tokens x 300 positions of 64 heads 17.2 us, 20.9 dealt out; 128
    //   x 2 10.2 and 13.8);
    // - one sequence, or lists of up to IX_SHORT chunks, where they fill at least 7/8
    //   of the even deal's places: 1024 positions, 256 sequences x 2 tokens of 64
    //   heads 21.8 us, 26.3 dealt out.  One sequence's groups are as even as its
    //   lists are; several sequences' lists may differ by up to IX_SHORT chunks;
    // - lists of up to IX_SHORT chunks in two or more rounds of workgroups, one per
    //   group: the hardware hands them out as others end (causal, 2048 tokens x 2048
    //   positions of 128 heads 102 us, 119 dealt out; with 600 groups the second
    //   round is mostly empty, 51 and 46).
    const int64_t parts = wgs / p.groups;
    if (most <= IX_TINY && p.groups <= IX_MOST_WGS) {
        p.parts = (int32_t)std::max<int64_t>(1, std::min<int64_t>(IX_WGS / 2 / p.groups, most));
        wgs = p.parts * p.groups;
    } else if ((B == 1 || most <= IX_SHORT) && parts * p.groups >= wgs - wgs / 8) {
        p.parts = (int32_t)parts;
        wgs = parts * p.groups;
    } else if (most <= IX_SHORT && p.groups >= 2 * IX_WGS && p.groups <= IX_MOST_WGS) {
        p.parts = 1;
        wgs = p.groups;
    }
    if (once) hipLaunchKernelGGL((dsa_indexer_kernel<HI, NB, true>), dim3((unsigned)wgs), dim3(IX_NTHR), 0, st, p);
    else if constexpr (NB == 4)
        hipLaunchKernelGGL((dsa_indexer_kernel<HI, NB, false>), dim3((unsigned)wgs), dim3(IX_NTHR), 0, st, p);
    return hipGetLastError() == hipSuccess ? DSA_OK : DSA_ERR_HIP;
}

}  // namespace

extern "C" int dsa_indexer_scores(const dsa_indexer_args* a, void* stream) {
    if (!a) return DSA_ERR_NULL_POINTER;
    if (a->B < 0 || a->s_q <= 0 || a->n_cols < 0 || a->k_total_rows < 0 || a->k_total_rows > INT32_MAX)
        return DSA_ERR_BAD_SHAPE;
    if (a->H_I != 32 && a->H_I != 64 && a->H_I != 128) return DSA_ERR_UNSUPPORTED;
    if (a->block_table && a->block_size <= 0) return DSA_ERR_BAD_SHAPE;
    const int64_t k_stride = a->k_stride_row ? a->k_stride_row : DSA_INDEXER_D;
    if (k_stride < DSA_INDEXER_D || (k_stride % 8)) return DSA_ERR_BAD_STRIDE;
    if (a->score_stride < a->n_cols) return DSA_ERR_BAD_STRIDE;
    const int tpw = 128 / a->H_I;
    const int tgroups = (a->s_q + tpw - 1) / tpw;
    if ((int64_t)a->B * tgroups > INT32_MAX) return DSA_ERR_BAD_SHAPE;
    if (a->B == 0 || a->n_cols == 0) return DSA_OK;
    if (!a->q || !a->weights || !a->seq_lens || !a->scores || (a->k_total_rows > 0 && !a->k_cache))
        return DSA_ERR_NULL_POINTER;
    if ((a->q_stride_b % 8) || (a->q_stride_t % 8) || (a->q_stride_h % 8) || ((uintptr_t)a->q & 15) ||
        ((uintptr_t)a->k_cache & 15) || ((uintptr_t)a->scores & 3))
        return DSA_ERR_BAD_STRIDE;
    IxParams p{};
    p.q = (const __bf16*)a->q;
    p.q_sb = a->q_stride_b; p.q_st = a->q_stride_t; p.q_sh = a->q_stride_h;
    p.w = a->weights;
    p.k = (const unsigned char*)a->k_cache;
    p.k_rows = a->k_total_rows;
    p.k_row_bytes = 2 * k_stride;
    p.bt = a->block_table;
    p.bt_stride = a->block_table_stride;
    p.bs = a->block_table ? a->block_size : 1;
    p.bs_shift = (p.bs & (p.bs - 1)) == 0 ? __builtin_ctz((unsigned)p.bs) : -1;
    p.k_bstride = a->k_batch_stride;
    p.seq_lens = a->seq_lens;
    p.scores = a->scores;
    p.s_stride = a->score_stride;
    p.s_q = a->s_q; p.n_cols = a->n_cols; p.causal = a->causal ? 1 : 0;
    hipStream_t st = (hipStream_t)stream;
    // as many 32-row blocks as the sequence's (token, head) rows fill, up to four
    if (a->H_I == 32)
        return a->s_q == 1 ? launch_ix<32, 1>(p, a->B, st)
                           : (a->s_q == 2 ? launch_ix<32, 2>(p, a->B, st) : launch_ix<32, 4>(p, a->B, st));
    if (a->H_I == 64)
        return a->s_q == 1 ? launch_ix<64, 2>(p, a->B, st) : launch_ix<64, 4>(p, a->B, st);
    return launch_ix<128, 4>(p, a->B, st);
}
