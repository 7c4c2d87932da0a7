// Single-token decode over the KV cache: split-K over the context + combine.
//
// Replaces, for T == 1, what the reference runs below its flash threshold
// (src/nn/functional.cpp:397-421: matmul, div, softmax, matmul over a materialised score tensor)
// together with the two repeat_kv copies before it (src/nn/gqa_attention.cpp:140-141).
//
// One workgroup (4 wavefronts) handles one (batch row, kv head, context split).  The n_rep query
// heads that share the kv head ride in the N dimension of 16x16x32 MFMA tiles (padded to 16), so
// K and V are read from HBM exactly once per kv head:
//   S^T[key][head]  = K[key][:] . Q^T[:][head]        A = K rows as they lie in HBM (16-byte loads)
//   O^T[d][head]   += V^T[d][key] . P^T[key][head]    A = V^T, which the token-blocked V plane
//                                                     stores so that 8/16 tokens of one d are one load
// A wavefront consumes 64 keys per iteration.  MFMA row i of S^T tile jj (0..3) is key
// 16*(i/4) + 4*jj + i%4 of the group, which makes the four S values a lane gets from each tile
// line up with the contraction slots of the PV MFMAs (slot (t, g, e) = key 16*g + 8*t + e) without
// any cross-lane movement.  Online softmax in fp32, exp2 with the scale folded in.
#include <stdlib.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "kv_layout.hpp"
#include "kv_rows.hpp"
#include "vsp_common.hpp"

namespace vsp {
int check_kv_cache(const vsp_kv_cache* c);

namespace {

constexpr int kWaves = 4;
constexpr int kGroup = 64;  // keys per wave iteration
constexpr int kMinChunk = kWaves * kGroup;

struct DecodeArgs {
    const void* q;
    int64_t sq_b, sq_h, sq_t;  // q strides (elements) of dims 0, 1, 2
    int32_t T;                 // query tokens per sequence: token t sits at position L - T + t and sees the keys up to itself
    const void* k;
    const void* v;
    const void* k_scale;
    const void* v_scale;
    const int32_t* seq_lens;  // device, or nullptr
    int32_t len;              // used when seq_lens == nullptr
    int32_t B, Hq, Hkv, n_rep;
    int64_t S;  // physical token capacity of the planes
    int32_t S_max;  // logical capacity
    int32_t L_cap;  // min(S_max, the host's upper bound of the lengths): every length is clamped to it, because the
                    // grid, max_splits and the workspace are sized from that bound
    int32_t chunk;           // keys per split of a ragged batch
    int32_t uniform_splits;  // > 0: splits per row when the rows are about equally long (split_chunk)
    int32_t max_splits;
    float scale_log2;  // scale * log2(e)
    float* ws_o;       // [B][Hq][T][max_splits][D]
    float* ws_ml;      // [B][Hq][T][max_splits][2]  (m in log2 domain, l)
    // paged cache: sequence b's 64-key group starting at token t lives in page page_table[b * pages_per_seq +
    // t / page_tokens] (page_tokens is a multiple of 64, so a group never straddles two pages); S is then the
    // page size.  nullptr for a contiguous cache.
    const int32_t* page_table;
    int32_t page_tokens, pages_per_seq;
    // More than 16 query heads per kv head (one token per sequence): the heads are cut into n_cgroups groups of 16
    // columns, one workgroup per (item, kv head, group); col0 is the group's first head (set by each workgroup).
    int32_t n_cgroups, col0;
    // One launch per step: the last workgroup of a (batch row, kv head, column group) to leave its partials merges them into
    // `out`.  counters: one per such triple, zero between launches; nullptr: the partials are merged by a launch of
    // its own (launch_split_combine).
    uint32_t* counters;
    // The host knows the one length of all rows: the grid is (kv head, split, batch row) and no workgroup has to find its place (one
    // token of 2048 bf16 keys: 0.8 us from the start of a workgroup to its first load, integer divisions mostly).  n_splits: of
    // every row.  0 with lengths on the device or with column groups.
    int32_t direct, n_splits;
    int32_t range_wgs, range_slack;  // RANGE kernels: workgroups of the launch; how many groups longer than a range a part may be (RangeWalk)
    void* out;
    int64_t so_b, so_h, so_t;
    // STEP kernels: the step's token is not in the cache yet.  Its K and V rows enter the attention from registers and the cache at
    // position `len`, one past the keys that are read; with a table, q and k are rotated at that position first.
    const void* new_k;
    const void* new_v;
    int64_t sk_b, sk_h, sv_b, sv_h;  // strides (elements)
    const float* table;              // [positions][D/2][2] = {cos, sin}, or nullptr
    Round round;  // ROUND kernels
};

// Where the 64-key groups of (sequence b, kv head) lie: the [S][D] slab of the group at token `kbase` and its first token inside that slab.
// Of a paged cache, lane i holds the places of group i of the 64 from `first` on: one load of the table per 64 groups, where a load per group
// sits in the queue of the keys' loads and holds up the next group's until the current one's values are there.  A step with a load per group
// and this way: 8 x 8 rows of 500 to 8000 bf16 keys, D 128, four tokens, pages of 256, 46.5 and 45.1 us; 16 x 8, pages of 64, 74.9 and 72.6; one row of 1000 to
// 3000 14.5 and 12.9; Q8_0, 32 x 4 of 512 to 16384, 94 and 85 (32 x 8 of 1k to 32k, bf16: 450 and 452).
template <bool PAGED>
struct GroupPlaces {
    int64_t head;                 // contiguous cache: the slab
    int first, slab, local;       // paged: per lane
    __device__ void init(const DecodeArgs& a, int b, int kvh, int kbase, int lane) {
        if constexpr (PAGED) fetch(a, b, kvh, kbase, lane);
        else head = (int64_t)b * a.Hkv + kvh;
    }
    __device__ void fetch(const DecodeArgs& a, int b, int kvh, int kbase, int lane) {
        first = kbase;
        const int at = kbase + lane * kGroup;
        const int pg = (uint32_t)at / (uint32_t)a.page_tokens;
        slab = a.page_table[(int64_t)b * a.pages_per_seq + min(pg, a.pages_per_seq - 1)] * a.Hkv + kvh;
        local = at - pg * a.page_tokens;
    }
    __device__ int64_t at(const DecodeArgs& a, int b, int kvh, int kbase, int lane, int& token) {
        if constexpr (PAGED) {
            int i = __builtin_amdgcn_readfirstlane((kbase - first) / kGroup);
            if (i >= 64) {
                fetch(a, b, kvh, kbase, lane);
                i = 0;
            }
            token = __builtin_amdgcn_readlane(local, i);
            return __builtin_amdgcn_readlane(slab, i);
        } else {
            token = kbase;
            return head;
        }
    }
};

// The same of one token: its slab and its place in it.
template <bool PAGED>
__device__ inline int64_t token_slab(const DecodeArgs& a, int b, int kvh, int pos, int& local) {
    int64_t s = pos, slab_b = b;
    kv_locate(PAGED ? a.page_table : nullptr, a.page_tokens, a.pages_per_seq, slab_b, s);
    local = (int)s;
    return slab_b * a.Hkv + kvh;
}

__device__ inline float wave_max_over_groups(float x) {
    x = fmaxf(x, __shfl_xor(x, 16));
    x = fmaxf(x, __shfl_xor(x, 32));
    return x;
}
__device__ inline float wave_sum_over_groups(float x) {
    x += __shfl_xor(x, 16);
    x += __shfl_xor(x, 32);
    return x;
}

// Over the lanes with the same position in their row of 16, and over those of a row with the same position in their quad.
// (The swaps as asm: given one value twice, the builtins have come out as the sum of one result with itself.)
__device__ inline float rows_sum(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    float y;  // two wait states between a vector-ALU write and a permlane swap that reads it
    asm volatile("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(x), "=&v"(y));
    x += y;
    asm volatile("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "=&v"(y));
    x += y;
#endif
    return x;
}
template <int CTRL>  // DPP: 0x120 + n rotates the row by n
__device__ inline float row_rotated(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
#else
    return x;
#endif
}
__device__ inline float quads_sum(float x) {
    x += row_rotated<0x124>(x);
    return x + row_rotated<0x128>(x);
}
__device__ inline float quads_max(float x) {
    x = fmaxf(x, row_rotated<0x124>(x));
    return fmaxf(x, row_rotated<0x128>(x));
}

// The 16 MFMA columns of a work item are the (token, query head of the kv head) pairs of the call, token-major:
// column c = t * n_rep + r.  With one token per sequence (the plain decode step) a column is a query head.
struct Column {
    int t, r;
    bool live;
};
// Columns this workgroup owns: all (token, head) pairs, or its group of up to 16 heads.
__device__ inline int column_count(const DecodeArgs& a) { return a.n_cgroups > 1 ? min(16, a.n_rep - a.col0) : a.n_rep * a.T; }
__device__ inline Column column_of(const DecodeArgs& a, int c) {
    const int n = column_count(a), cc = min(c, n - 1);
    if (a.n_cgroups > 1 || a.T == 1) return Column{0, a.col0 + cc, c < n};  // col0 is 0 without groups
    return Column{cc / a.n_rep, cc % a.n_rep, c < n};
}
// Which (work item, kv head) a workgroup serves.  kv head fastest: every item that exists comes before the first
// surplus workgroup of the grid (which is sized for the longest possible batch), so the surplus ones start, find
// nothing and exit under the tail of the real work.  With column groups, the groups of one (item, kv head) get block
// ids 8 apart: the same XCD (ids are dealt round-robin to the 8 XCDs), so the K/V stream they share is fetched into
// one L2, once, and read from there by the others.
__device__ inline void block_coords(DecodeArgs& a, int& kvh, int& item) {
    if (a.direct) {
        kvh = blockIdx.x;
        item = 0;
        return;
    }
    int ik = blockIdx.x;
    if (a.n_cgroups > 1) {  // id = ((ik / 8) * n_cgroups + group) * 8 + ik % 8
        const int rest = blockIdx.x >> 3;
        a.col0 = 16 * (rest % a.n_cgroups);
        ik = (rest / a.n_cgroups) * 8 + (blockIdx.x & 7);
    }
    kvh = ik % a.Hkv;
    item = ik / a.Hkv;
}
// ---- STEP kernels: append and attention of one token per sequence in one launch -----------------------------------------
// A launch of its own for the append is most of a small step beside the attention's own latency (2.4 us and the gap to the next
// launch, of 9.2 us with 256 fp32 keys).  The token's key is scored from registers instead: the last wavefront of a row's last split
// starts its online softmax from it (m = its score, l = 1, O = its V, all as the cache's format rounds them) and writes the rows into
// the planes.  No workgroup reads them there: every one masks keys from `len` on.  Each workgroup rotates the query heads it serves
// itself, one piece of a row per thread through LDS while the first keys are on their way (every wavefront for itself: 1 us more, the
// time to fetch the instructions of four pieces).  A token step, two launches and one: 32 / 8 heads, D 128, 2047 bf16 keys 11.5 and
// 9.4 us (8.9 with plan_fine), 256 fp32 keys of 8 / 2 heads 9.2 and 7.1, 16 rows of 2047 bf16 keys 26.9 and 23.8.
__device__ inline bool step_owner(int split, int n_splits, int wave) {
    return split == n_splits - 1 && wave == kWaves - 1;
}
template <typename T>
__device__ inline const T* step_row(const void* base, int64_t sb, int64_t sh, int b, int h) {
    return (const T*)base + (int64_t)b * sb + (int64_t)h * sh;
}
// the {cos, sin} pairs of elements d0.. at the step's position
template <int D>
__device__ inline const float4* step_pairs(const DecodeArgs& a, int d0) {
    return (const float4*)((const float2*)a.table + (int64_t)a.len * (D / 2) + d0 / 2);
}
// The rows of a step are staged through LDS in pieces of W elements, one thread per piece: rows 0 .. n - 1 the workgroup's queries,
// n the token's key, n + 1 its value, PC pieces a row.
template <int PC>
struct StepPiece {
    int row, p;
    bool is_q, is_k, is_v;
    __device__ StepPiece(int i, int n) : row(i / PC), p(i % PC), is_q(row < n), is_k(row == n), is_v(row == n + 1) {}
};
template <typename T, int PC>
__device__ inline const T* step_source(const DecodeArgs& a, const StepPiece<PC>& s, int b, int kvh) {
    if (s.is_q) return step_row<T>(a.q, a.sq_b, a.sq_h, b, kvh * a.n_rep + a.col0 + s.row);
    return s.is_k ? step_row<T>(a.new_k, a.sk_b, a.sk_h, b, kvh) : step_row<T>(a.new_v, a.sv_b, a.sv_h, b, kvh);
}
// this wavefront's LDS writes have landed, then the barrier (a fence would also wait for the keys' loads)
__device__ inline void step_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Keys [0, limit) are visible to column col: token t of T sits at position L - T + t and attends up to itself.
__device__ inline int column_limit(const DecodeArgs& a, const Column& col, int L, int chunk_end) {
    return min(chunk_end, L - (a.T - 1 - col.t));
}
__device__ inline uint4 mask_tail_u16x8(uint4 v, int nvalid) {
    // keep the first nvalid 16-bit elements, zero the rest
    uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int rem = nvalid - 2 * i;
        w[i] = rem >= 2 ? w[i] : (rem == 1 ? (w[i] & 0xFFFFu) : 0u);
    }
    return uint4{w[0], w[1], w[2], w[3]};
}


// Keys per split, from the lengths on the device: the same answer in every workgroup of the decode and combine kernels.
// Rows of about one length (their sum at least 9/10 of what the longest would make) are cut into uniform_splits parts each,
// which makes one even round of workgroups; a ragged batch into splits of `chunk` keys, several rounds that the hardware deals
// out as workgroups finish.
// Every workgroup pays for this before its first load of K, so the reductions go over DPP lanes (row shifts and broadcasts: lane 63
// ends up with all of them), not over LDS: 32 x 8 rows of 1k to 32k keys, bf16, 443.7 us with shuffles, 442.3 with DPP; 8 x 8 rows of 500
// to 6525, 31.3 and 30.9.
// ROUND: a ragged batch's splits are as long as it takes to make one round of workgroups (plan_round says where, with times).  `chunk` comes from the host's bound
// of the lengths, which may be many times theirs (a decode_attention without max_len: the capacity), so it says nothing about how short a split may be: a row has
// max_splits at most, and shorter splits than `chunk` make a workgroup per CU at most.  Us a step, never shorter than `chunk` and as here: fp32, 7 x 4 rows of 1040 to 6525, two
// tokens, under a bound of 26100 45.2 and 24.0; bf16, D 64, pages, 7 x 8 of 1415 to 3000, two tokens, bound 12000 15.4 and 10.7; Q8_0, pages, 6 x 4 of 689 to 9000, bound
// 18000 17.7 and 15.9; 223 drawn batches with bounds of 2 to 8 times the longest row 1.14 faster, 237 with tight ones 1.007.  In kernels of their own (decode_*_round_kernel): a workgroup pays for the search before its first load of K,
// and the other steps' code stays as it is.
template <int CTRL>
__device__ inline int from_lane(int x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true); }  // 0 where there is no such lane
template <class Step>
__device__ inline void over_lanes(Step&& step) {  // lane 63 ends up with all
    step(std::integral_constant<int, 0x111>{});  // from 1, 2, 4, 8 lanes below in the row of 16,
    step(std::integral_constant<int, 0x112>{});
    step(std::integral_constant<int, 0x114>{});
    step(std::integral_constant<int, 0x118>{});
    step(std::integral_constant<int, 0x142>{});  // from lane 15 of the row below,
    step(std::integral_constant<int, 0x143>{});  // from lane 31
}
__device__ inline int lanes_total(int x) {
    over_lanes([&](auto ctrl) { x += from_lane<decltype(ctrl)::value>(x); });
    return __builtin_amdgcn_readlane(x, 63);
}
// ceil(groups / c), groups > 0: exact while groups stay below 2^21 (half a group is more than the product's rounding); plan_round
// takes rows of 2^20 at most (sixteen rounds of 512 splits of 8192 keys).
__device__ inline int parts_of(int groups, int c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return (int)(((float)(groups - 1) + 0.5f) * __builtin_amdgcn_rcpf((float)c)) + 1;
#else
    return 0;
#endif
}
__device__ inline int groups_of(int L) { return max((L + kGroup - 1) / kGroup, 1); }
// A row far shorter than a split of c groups: its one workgroup comes after all others (locate_work) and is not counted as one of the round, since it adds to one
// of the others' CUs at most what counting B / 2 such rows would add to every split (a split of c groups grows by c B / 2 / items).  One row of 50000 Q8_0 keys and fifteen
// of up to 200, 8 kv heads: counted 16 splits of the long row and 37.8 us, not counted 25 and 30.6; 16 x 8, half of them short, of 22 to 2305 17.7 and 15.9.  In the batch's order
// short rows before long ones leave two long splits on a CU: 12 x 8, half of them short, of 13 to 29441 88 us, not counted 143, not counted and last 87.6.
__device__ inline bool is_short(int groups, int c, int B, int items) { return 2 * items * groups <= B * c; }
// A length of a split, in groups and at least `least`, with which rows of `groups` groups (lane b: row b's; 0: no row) make at most `items` splits, short rows aside:
// the least of five between what no split could be shorter than and what always does.  Close enough (a fifth of B / items of it), and exact about the count: a round that a handful
// of workgroups overflow takes as long as two (8 x 8 rows of 500 to 8000: 264 workgroups 46 us, 248 37).  Two sums of 16 bits per reduction.
__device__ inline int round_groups(int groups, int total, int B, int least, int items, int round_items) {
    const int lo = max(least, (int)((uint32_t)(total + items - 1) / (uint32_t)items));
    const int hi = (int)((uint32_t)(total - B + items - B - 1) / (uint32_t)(items - B));  // the sum of ceil(g / c) is at most (total - B) / c + B
    if (hi <= lo) return lo;
    int best = hi;
#pragma unroll
    for (int k = 2; k >= 0; k -= 2) {
        const int c0 = lo + (hi - lo) * k / 5, c1 = lo + (hi - lo) * (k + 1) / 5;
        auto parts = [&](int c) { return is_short(groups, c, B, round_items) ? 0 : min(parts_of(groups, c), 1023); };
        const int n = lanes_total(parts(c0) | parts(c1) << 16);
        if ((n >> 16) <= items) best = c1;
        if ((n & 0xffff) <= items) best = c0;
    }
    return best;
}
template <bool ROUND>
__device__ inline int split_chunk(const int32_t* seq_lens, int B, int L_cap, int chunk, int uniform_splits, Round round, int lane) {
    if constexpr (ROUND) {
        const int groups = lane < B ? groups_of(min(max(seq_lens[lane], 0), L_cap)) : 0;
        int total = groups, longest = groups;
        over_lanes([&](auto ctrl) {
            total += from_lane<decltype(ctrl)::value>(total);
            longest = max(longest, from_lane<decltype(ctrl)::value>(longest));
        });
        total = __builtin_amdgcn_readlane(total, 63);
        longest = __builtin_amdgcn_readlane(longest, 63);
        if (uniform_splits > 0 && total * 10 >= longest * B * 9)
            return max((int)((uint32_t)(longest + uniform_splits - 1) / (uint32_t)uniform_splits) * kGroup, kMinChunk);
        int least = max(parts_of(longest, round.max_splits), kMinChunk / kGroup);
        // two workgroups a CU: shorter splits than `chunk` for one of them only (9 x 12 rows of 658 to 2111 under a bound of 4222: 13.7 us in 300 workgroups, 13.2 in 250;
        // 13 x 16 of 1 to 18054 33.5 and 31.9; 8 x 2 of 18 to 44808, four tokens, 20.9 and 18.9)
        if (round.per_cu < round.items)
            least = max(least, round.per_cu > B ? min(chunk / kGroup, round_groups(groups, total, B, least, round.per_cu, round.items)) : chunk / kGroup);
        const int one = round_groups(groups, total, B, least, round.items, round.items);
        if (!round.or_two) return one * kGroup;
        const int two = round_groups(groups, total, B, least, 2 * round.items, round.items);
        return (5 * one <= 11 * two ? one : two) * kGroup;
    }
    if (uniform_splits == 0) return chunk;
    float total = 0.f;  // the same rounding in every wavefront that asks
    int longest = 0;
    for (int b0 = 0; b0 < B; b0 += 64) {
        int mx = b0 + lane < B ? min(max(seq_lens[b0 + lane], 0), L_cap) : 0;
        float sum = (float)mx;
        over_lanes([&](auto ctrl) {
            constexpr int c = decltype(ctrl)::value;
            sum += __builtin_bit_cast(float, from_lane<c>(__builtin_bit_cast(int, sum)));
            mx = max(mx, from_lane<c>(mx));
        });
        total += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sum), 63));
        longest = max(longest, __builtin_amdgcn_readlane(mx, 63));
    }
    if (total * 10.f < (float)longest * (float)B * 9.f) return chunk;
    const int even = ((longest + uniform_splits - 1) / uniform_splits + kGroup - 1) / kGroup * kGroup;
    return max(even, kMinChunk);
}

// Work items are (batch row, split) pairs packed without gaps: item i belongs to the sequence b with
// offs(b) <= i < offs(b) + nsplits(b), nsplits(b) = ceil(L_b / chunk).  Lengths live on the device, so
// every workgroup locates its item itself: 64 sequences at a time, one per lane, wave-wide prefix sum.
// The grid is sized for the worst case; surplus workgroups sit at the END of the grid and exit at once
// (with the (split, b) grid of a naive mapping the empty workgroups of short sequences would be
// interleaved with real work and cost launch slots all the way through).
// With counters an empty row has one item all the same (it writes the zeros).
// ROUND: the rows that are short (is_short) come after the others.  Both prefix sums in one, 16 bits each (at most 64 rows and 640 splits).
template <bool ROUND = false>
__device__ inline bool locate_work(const DecodeArgs& a, int item, int lane, int& b, int& split, int& L, int& n_splits, int& chunk) {
    if (a.direct) {
        chunk = a.chunk;
        L = a.len;
        n_splits = a.n_splits;
        split = blockIdx.y;
        b = blockIdx.z;
        return true;
    }
    chunk = __builtin_amdgcn_readfirstlane(split_chunk<ROUND>(a.seq_lens, a.B, a.L_cap, a.chunk, a.uniform_splits, a.round, lane));
    const int at_least = a.counters ? 1 : 0;
    if (!a.seq_lens) {
        L = min(a.len, a.L_cap);
        n_splits = max((L + chunk - 1) / chunk, at_least);
        if (n_splits == 0 || item >= n_splits * a.B) return false;
        b = item / n_splits;
        split = item - b * n_splits;
        return true;
    }
    auto prefix_sum = [&](int x) {
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int t = __shfl_up(x, off);
            if (lane >= off) x += t;
        }
        return x;
    };
    if constexpr (ROUND) {
        const int Lb = lane < a.B ? min(max(a.seq_lens[lane], 0), a.L_cap) : 0;
        const int ns = lane < a.B ? max((Lb + chunk - 1) / chunk, at_least) : 0;
        const int ends = prefix_sum(is_short(groups_of(Lb), chunk / kGroup, a.B, a.round.items) ? ns << 16 : ns);
        const int total = __builtin_amdgcn_readlane(ends, 63), others = total & 0xffff;
        const bool among_short = item >= others;
        if (among_short) item -= others;
        if (among_short && item >= total >> 16) return false;
        const int end = among_short ? ends >> 16 : ends & 0xffff;
        b = __ffsll((long long)__ballot(end > item)) - 1;
        n_splits = __builtin_amdgcn_readlane(ns, b);
        split = item - (__builtin_amdgcn_readlane(end, b) - n_splits);
        L = __builtin_amdgcn_readlane(Lb, b);
        return true;
    }
    int base = 0;
    for (int b0 = 0; b0 < a.B; b0 += 64) {
        const int bb = b0 + lane;
        const int Lb = bb < a.B ? min(max(a.seq_lens[bb], 0), a.L_cap) : 0;
        const int ns = bb < a.B ? max((Lb + chunk - 1) / chunk, at_least) : 0;
        const int incl = prefix_sum(ns);
        const int total = __builtin_amdgcn_readlane(incl, 63);
        if (item < base + total) {
            const unsigned long long m = __ballot(base + incl > item);
            const int src = __ffsll((long long)m) - 1;
            b = b0 + src;  // all scalars: the branches on them are uniform to the compiler too
            n_splits = __builtin_amdgcn_readlane(ns, src);
            split = item - (base + __builtin_amdgcn_readlane(incl, src) - n_splits);
            L = __builtin_amdgcn_readlane(Lb, src);
            return true;
        }
        base += total;
    }
    return false;
}

// ---- RANGE kernels: a large batch with its lengths on the device --------------------------------------------------------
// The 64-key groups of all (batch row, kv head) pairs, one pair after the other, are cut into range_wgs ranges of equal length, one
// per workgroup, so that every workgroup has the same work whatever the lengths are; splits of one length make several rounds, the
// last of them ragged.  A workgroup serves the pairs its range touches one by one; a pair that it holds whole goes straight to the
// output, of the others it leaves a partial: the first piece of a range in slot 2 w, a last one that starts inside the range in slot
// 2 w + 1.  Rows of about one length are cut into uniform_splits parts each instead (split_chunk's test): one piece a workgroup, no
// seams inside a range.  So are others, into parts of one length, where one round of them is at most range_slack groups longer than a range (two seams
// less for at most 16 KB of keys: few pairs, or little work under a loose bound).  Ranges, parts: 8 x 8 rows of 500 to 6525 bf16 keys 35.2 and
// 34.6 us, 6 x 8 of 1500 to 24000, two tokens, 69.0 and 67.6, 8 x 12 of 100 to 3000, D 64, 21.0 and 19.0; where parts are longer by more, 12 x 8 of 300 to 7452
// 49.8 and 50.7, 32 x 8 of 100 to 2000 44.5 and 51.8.  Lane b of every wavefront holds row b's length (up to 64 rows); a prefix sum over the lanes says where each
// row begins.
constexpr int kRangeRows = 64, kRangeLeast = 4;  // rows at most; groups per workgroup at least (one per wavefront)
struct RangeWalk {
    int len, groups, end;         // per lane: its row's length, its groups of one kv head, where its pairs end
    int wgs, each, longer;        // ranges: the first `longer` are each + 1 groups, the others each;
    int part, parts, items;       // or part > 0: parts of `part` groups.  Per lane: its row's parts of one kv head, where its workgroups end
    int id;                       // the workgroup's range
    int r, r_first, r_end;        // the workgroup's range, what is left of it
    int b, kvh, off, row_groups, row_begin;  // the pair at r, and the group of it

    __device__ void scan(const DecodeArgs& a, int lane) {
        len = lane < a.B ? min(max(a.seq_lens[lane], 0), a.L_cap) : 0;
        groups = lane < a.B ? max((len + kGroup - 1) / kGroup, 1) : 0;  // an empty row has a group all the same (its zeros are written)
        auto from = [&](auto ctrl, auto rows, int y) { return __builtin_amdgcn_update_dpp(0, y, decltype(ctrl)::value, decltype(rows)::value, 0xf, decltype(rows)::value == 0xf); };
        auto over_lanes = [&](auto&& step) {
            using All = std::integral_constant<int, 0xf>;
            step(std::integral_constant<int, 0x111>{}, All{});  // from 1, 2, 4, 8 lanes below in the row of 16,
            step(std::integral_constant<int, 0x112>{}, All{});
            step(std::integral_constant<int, 0x114>{}, All{});
            step(std::integral_constant<int, 0x118>{}, All{});
            step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});  // from lane 15 of the row below into the odd rows,
            step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});  // from lane 31 into the upper half
        };
        int x = groups, longest = groups;
        over_lanes([&](auto ctrl, auto rows) {
            x += from(ctrl, rows, x);
            longest = max(longest, from(ctrl, rows, longest));
        });
        end = x * a.Hkv;
        const int rows_total = __builtin_amdgcn_readlane(x, 63), total = rows_total * a.Hkv, pairs = a.B * a.Hkv;
        longest = __builtin_amdgcn_readlane(longest, 63);
        wgs = min(a.range_wgs, max(total / kRangeLeast, 1));
        each = (uint32_t)total / (uint32_t)wgs;
        longer = total - each * wgs;
        part = 0;
        if (a.uniform_splits > 0 && (float)rows_total * 10.f >= (float)longest * (float)a.B * 9.f)
            part = max((uint32_t)(longest + a.uniform_splits - 1) / (uint32_t)a.uniform_splits, (uint32_t)kRangeLeast);
        else if (pairs < a.range_wgs) {  // every pair's last part is a short one: with the whole ones there are at most range_wgs
            const int p = max((uint32_t)(total + a.range_wgs - pairs - 1) / (uint32_t)(a.range_wgs - pairs), (uint32_t)kRangeLeast);
            if (p <= each + (longer > 0) + a.range_slack) part = p;
        }
        if (part > 0) {
            parts = (uint32_t)(groups + part - 1) / (uint32_t)part;
            int y = parts;
            over_lanes([&](auto ctrl, auto rows) { y += from(ctrl, rows, y); });
            items = y * a.Hkv;
            wgs = __builtin_amdgcn_readlane(items, 63);
        }
    }
    __device__ int begin_of(int w) const { return w * each + min(w, longer); }
    __device__ int range_at(int x) const {  // whose range group x is in
        const int head = longer * (each + 1);
        return x < head ? (uint32_t)x / (uint32_t)(each + 1) : longer + (uint32_t)(x - head) / (uint32_t)each;
    }
    __device__ bool start(const DecodeArgs& a, int lane, int w) {
        scan(a, lane);
        id = w;
        if (w >= wgs) return false;
        if (part > 0) {  // workgroup (row, part, kv head)
            b = __ffsll((long long)__ballot(items > w)) - 1;
            row(a);
            const int of_row = w - first_item(a), i = (uint32_t)of_row / (uint32_t)a.Hkv;
            kvh = of_row - i * a.Hkv;
            off = i * part;
            r_end = pair_begin() + min(off + part, row_groups);
        } else {
            const int first = begin_of(w);
            b = __ffsll((long long)__ballot(end > first)) - 1;
            row(a);
            kvh = (uint32_t)(first - row_begin) / (uint32_t)row_groups;
            off = first - pair_begin();
            r_end = begin_of(w + 1);
        }
        r = r_first = pair_begin() + off;
        return true;
    }
    __device__ int row_parts() const { return __builtin_amdgcn_readlane(parts, b); }
    __device__ int first_item(const DecodeArgs& a) const { return __builtin_amdgcn_readlane(items, b) - row_parts() * a.Hkv; }
    __device__ void row(const DecodeArgs& a) {
        row_groups = __builtin_amdgcn_readlane(groups, b);
        row_begin = __builtin_amdgcn_readlane(end, b) - row_groups * a.Hkv;
    }
    __device__ int pair_begin() const { return row_begin + kvh * row_groups; }
    __device__ int length() const { return __builtin_amdgcn_readlane(len, b); }
    __device__ int piece() const { return min(row_groups - off, r_end - r); }
    __device__ bool whole() const { return off == 0 && piece() == row_groups; }
    __device__ bool next(const DecodeArgs& a) {
        r += piece();
        if (r >= r_end) return false;
        off = 0;
        if (++kvh == a.Hkv) {
            kvh = 0;
            ++b;
            row(a);
        }
        return true;
    }
};
struct NoWalk {};
__device__ inline bool next_piece(const DecodeArgs&, NoWalk&) { return false; }
__device__ inline bool next_piece(const DecodeArgs& a, RangeWalk& walk) { return walk.next(a); }
// The partials of the walk's pair, in the order of its groups: rows slot * columns + column of the workspace.
struct RangeParts {
    int w_first, n, first_slot, apart;  // partial i is of range w_first + i * apart
    __device__ RangeParts(const DecodeArgs& a, const RangeWalk& k) {
        const int begin = k.pair_begin();
        if (k.part > 0) {
            w_first = k.first_item(a) + k.kvh;
            apart = a.Hkv;
            n = k.row_parts();
            first_slot = 2 * w_first;
        } else {
            w_first = k.range_at(begin);
            apart = 1;
            n = k.range_at(begin + k.row_groups - 1) - w_first + 1;
            first_slot = 2 * w_first + (k.begin_of(w_first) == begin ? 0 : 1);
        }
    }
    __device__ int slot(int i) const { return i == 0 ? first_slot : 2 * (w_first + i * apart); }
};

// Partials that another workgroup of the same launch reads: its die may have another L2, so they are written through and read
// past the caches (device-scope accesses, sc1).  No fence: one would write back and invalidate whole L2 slices; these accesses
// need only be complete (vmcnt) before the counter moves.  `r` spans the rows of one (batch row, kv head).
constexpr int kDeviceScope = 16;
__device__ inline void store_device(__amdgpu_buffer_rsrc_t r, int byte, f32x4_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), r, byte, 0, kDeviceScope);
#endif
}
__device__ inline void store_device(__amdgpu_buffer_rsrc_t r, int byte, float2 v) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, v), r, byte, 0, kDeviceScope);
#endif
}
__device__ inline void store_out(float* p, f32x4_t y) { *(f32x4_t*)p = y; }
__device__ inline void store_out(uint16_t* p, f32x4_t y) { *(u32x2_t*)p = u32x2_t{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])}; }

// Four outputs of one row (from d on) from its n_splits partials: what split_combine_kernel computes, operation for operation
// (one block for up to 32 splits, blocks of 32 beyond); up to 16 partial rows in flight.
// row_of(i): the row of partial i.
template <int BLK, int D, class RowOf>
__device__ inline f32x4_t merge_splits(__amdgpu_buffer_rsrc_t ro, __amdgpu_buffer_rsrc_t rml, RowOf&& row_of, int n_splits, int d) {
    constexpr int VB = BLK < 16 ? BLK : 16;
    float M = -INFINITY, l = 0.f;
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#if defined(__HIP_DEVICE_COMPILE__)
    for (int s0 = 0; s0 < n_splits; s0 += BLK) {
        float2 ml[BLK];
        f32x4_t v[VB];
        auto split_row = [&](int i) { return row_of(min(s0 + i, n_splits - 1)); };
        auto load_v = [&](int i0) {
#pragma unroll
            for (int i = 0; i < VB; ++i)
                v[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(ro, (split_row(i0 + i) * D + d) * 4, 0, kDeviceScope));
        };
#pragma unroll
        for (int i = 0; i < BLK; ++i) ml[i] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rml, split_row(i) * 8, 0, kDeviceScope));
        load_v(0);
        float Mb = M;
#pragma unroll
        for (int i = 0; i < BLK; ++i) Mb = fmaxf(Mb, ml[i].x);
        const float Mr = Mb == -INFINITY ? 0.f : Mb;
        const float keep = exp2f(M - Mr);
        o *= keep;
        l *= keep;
        M = Mb;
#pragma unroll
        for (int i0 = 0; i0 < BLK; i0 += VB) {
            if (i0 > 0) load_v(i0);
#pragma unroll
            for (int i = 0; i < VB; ++i)
                if (s0 + i0 + i < n_splits) {
                    const float w = exp2f(ml[i0 + i].x - Mr);
                    l += w * ml[i0 + i].y;
                    o += w * v[i];
                }
        }
    }
#endif
    f32x4_t y = {0.f, 0.f, 0.f, 0.f};
    if (l > 0.f) {
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = o[j] / l;
    }
    return y;
}

// The (m, l, O^T) of a workgroup's four wavefronts, left in LDS per column, merged into one split-K partial per column.
// First, one lane per column: the merged maximum, the four weights 2^(m_w - m), the merged sum and the partial's row
// (once per column, not once per element: the weights are four exp2 and the row takes integer divisions).  Then one
// element per thread: o = sum_w weight_w * O_w in wavefront order.  ZERO_FOR_EMPTY: a wavefront that saw no key of a
// short split, or a column with no key in it, carries m = -inf, l = 0 and zero sums, and gets the weight 0 explicitly;
// otherwise -inf is replaced by 0 as the reference point (a column without a key in this split: zero sums, m = -inf).
template <int D, class RowOf>
__device__ inline f32x4_t merge_all_splits(__amdgpu_buffer_rsrc_t ro, __amdgpu_buffer_rsrc_t rml, RowOf&& row_of, int n_splits, int d) {
    return n_splits <= 8    ? merge_splits<8, D>(ro, rml, row_of, n_splits, d)
           : n_splits <= 16 ? merge_splits<16, D>(ro, rml, row_of, n_splits, d)
                            : merge_splits<32, D>(ro, rml, row_of, n_splits, d);
}
// walk: the piece of a range that this is (RANGE kernels; split and n_splits are then not used), or NoWalk.
template <int D, bool ZERO_FOR_EMPTY, typename OutT, class Walk>
__device__ inline void merge_waves_and_store(const DecodeArgs& a, const float (&sm_o)[kWaves][16][D + 4], const float (&sm_m)[kWaves][16],
                                             const float (&sm_l)[kWaves][16], int b, int kvh, int split, int n_splits, int tid,
                                             const Walk& walk) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    __shared__ float sm_f[kWaves][16];
    __shared__ float sm_ll[16];
    __shared__ int sm_row[16];
    __shared__ int64_t sm_out[16];
    __shared__ uint32_t sm_before;
    constexpr bool RANGE = std::is_same_v<Walk, RangeWalk>;
    const int ncol = column_count(a);
    // the partials of (b, kvh) are consecutive rows; within them a column's splits are.  Of a range: slots of ncol rows.
    const int64_t base_row = RANGE ? 0 : ((int64_t)__builtin_amdgcn_readfirstlane(b) * a.Hq + (int64_t)__builtin_amdgcn_readfirstlane(kvh) * a.n_rep) * a.T * a.max_splits;
    const int n_rows = RANGE ? 2 * a.range_wgs * ncol : a.n_rep * a.T * a.max_splits;
    float* const po = a.ws_o + base_row * D;
    float* const pml = a.ws_ml + base_row * 2;
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(po, 0, n_rows * D * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rml = __builtin_amdgcn_make_buffer_rsrc(pml, 0, n_rows * 8, 0x00020000);
    int slot = 0;
    if constexpr (RANGE) {
        n_splits = walk.whole() ? 1 : 2;  // or more
        split = 0;
        slot = 2 * walk.id + (walk.r == walk.r_first ? 0 : 1);
    }
    if (tid < ncol) {
        const int hc = tid;
        float mm = sm_m[0][hc];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) mm = fmaxf(mm, sm_m[w][hc]);
        const float mm_ref = mm == -INFINITY ? 0.f : mm;
        float ll = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float f = ZERO_FOR_EMPTY ? (sm_m[w][hc] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sm_m[w][hc] - mm))
                                           : __builtin_amdgcn_exp2f(sm_m[w][hc] - mm_ref);
            sm_f[w][hc] = f;
            ll += f * sm_l[w][hc];
        }
        const Column col = column_of(a, hc);
        const int row = RANGE ? slot * ncol + hc : (col.r * a.T + col.t) * a.max_splits;
        sm_row[hc] = row;
        if (a.counters || RANGE) {
            sm_ll[hc] = ll;
            sm_out[hc] = (int64_t)b * a.so_b + (int64_t)(kvh * a.n_rep + col.r) * a.so_h + (int64_t)col.t * a.so_t;
            if (n_splits > 1 && !RANGE) store_device(rml, (row + split) * 8, float2{mm, ll});
        }
        if (RANGE ? n_splits > 1 : !a.counters) {
            *(float2*)(pml + (int64_t)(row + split) * 2) = float2{mm, ll};
        }
    }
    __syncthreads();
    auto merged = [&](int hc, int d) {
        f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWaves; ++w) o += sm_f[w][hc] * *(const f32x4_t*)&sm_o[w][hc][d];
        return o;
    };
    const int n_quads = ncol * (D / 4);
    if ((a.counters || RANGE) && n_splits == 1) {  // nothing to merge with: straight to the output
        for (int i = tid; i < n_quads; i += 256) {
            const int hc = i / (D / 4), d = 4 * (i % (D / 4));
            f32x4_t y = merged(hc, d);
            const float ll = sm_ll[hc];
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = ll > 0.f ? y[j] / ll : 0.f;
            store_out((OutT*)a.out + sm_out[hc] + d, y);
        }
        return;
    }
    for (int i = tid; i < n_quads; i += 256) {
        const int hc = i / (D / 4), d = 4 * (i % (D / 4));
        const f32x4_t o = merged(hc, d);
        if (!RANGE && a.counters) store_device(ro, ((sm_row[hc] + split) * D + d) * 4, o);
        else *(f32x4_t*)(po + (int64_t)(sm_row[hc] + split) * D + d) = o;
    }
    if (RANGE || !a.counters) return;
    // every thread's partials have reached the point all dies read from before the workgroup is counted
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint32_t* counter = a.counters + ((int64_t)b * a.Hkv + kvh) * a.n_cgroups + a.col0 / 16;
    if (tid == 0) sm_before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (sm_before != (uint32_t)n_splits - 1) return;
    if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int i = tid; i < n_quads; i += 256) {
        const int hc = i / (D / 4), d = 4 * (i % (D / 4));
        store_out((OutT*)a.out + sm_out[hc] + d, merge_all_splits<D>(ro, rml, [&](int k) { return sm_row[hc] + k; }, n_splits, d));
    }
#endif
}

// ---------------------------------------------------------------------------------------------
// bf16 cache
// ---------------------------------------------------------------------------------------------
template <int D, bool PAGED, bool STEP, bool RANGE, bool ROUND>
__device__ __forceinline__ void decode_bf16_body(DecodeArgs a) {
    constexpr int KS = D / 32;   // MFMA k-steps over the head dim
    constexpr int DB = D / 16;   // 16-row tiles of O^T
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ __attribute__((aligned(16))) float sm_o[kWaves][16][D + 4];
    __shared__ float sm_m[kWaves][16], sm_l[kWaves][16];
    std::conditional_t<RANGE, RangeWalk, NoWalk> walk;
    if constexpr (RANGE) {
        if (!walk.start(a, lane, blockIdx.x)) return;
    }
    do {  // one pass, or one per piece of the workgroup's range
    int kvh, b, split = 0, L, n_splits = 1, chunk_start, chunk_end;
    if constexpr (RANGE) {
        b = walk.b, kvh = walk.kvh, L = walk.length();
        chunk_start = walk.off * kGroup;
        chunk_end = min(L, chunk_start + walk.piece() * kGroup);
    } else {
        int item, chunk;
        block_coords(a, kvh, item);
        if (!locate_work<ROUND>(a, item, lane, b, split, L, n_splits, chunk)) return;
        chunk_start = split * chunk;
        chunk_end = min(L, chunk_start + chunk);
    }

    const int c = lane & 15, g = lane >> 4;
    GroupPlaces<PAGED> places;
    places.init(a, b, kvh, chunk_start, lane);

    // Q^T operands: column c = (token, query head of this kv head), zero beyond the last one
    const Column col = column_of(a, c);
    const int lim = column_limit(a, col, L, chunk_end);
    bf16x8_t qf[KS];
    const bool owner = STEP && step_owner(split, n_splits, wave);
    constexpr int PC = D / 8, PITCH = D + 8;
    [[maybe_unused]] uint4 piece;
    [[maybe_unused]] float4 pairs[2];
    [[maybe_unused]] const int n_pieces = (column_count(a) + 2) * PC;
    [[maybe_unused]] auto load_piece = [&](int i) {
        const StepPiece<PC> sp(i, column_count(a));
        piece = *(const uint4*)(step_source<uint16_t>(a, sp, b, kvh) + 8 * sp.p);
        if (a.table && !sp.is_v) pairs[0] = step_pairs<D>(a, 8 * sp.p)[0], pairs[1] = step_pairs<D>(a, 8 * sp.p)[1];
    };
    if constexpr (STEP) {
        if (tid < n_pieces) load_piece(tid);
    } else {
        const uint16_t* qrow = (const uint16_t*)a.q + (int64_t)b * a.sq_b + (int64_t)(kvh * a.n_rep + col.r) * a.sq_h + (int64_t)col.t * a.sq_t;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            uint4 w = *(const uint4*)(qrow + 32 * ks + 8 * g);
            if (!col.live) w = uint4{0, 0, 0, 0};
            qf[ks] = __builtin_bit_cast(bf16x8_t, w);
        }
    }
    const int krow = 16 * (c >> 2) + (c & 3);  // this lane's A-operand row: key offset before + 4*jj

    f32x4_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    // K rows (A operands of S^T) and V^T blocks (A operands of O^T) of one 64-key group.  The loop is
    // rotated: the loads of group i+1 are issued as soon as group i's registers have been consumed
    // (K after the S^T MFMAs, V after the O^T MFMAs), so every wavefront keeps HBM requests in flight
    // while it computes.
    uint4 kf[4][KS];
    uint4 vf[DB][2];
    auto load_k = [&](int kbase) {
        int local;
        const uint16_t* Kp = (const uint16_t*)a.k + places.at(a, b, kvh, kbase, lane, local) * a.S * D;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const uint16_t* kr = Kp + (int64_t)(local + krow + 4 * jj) * D + 8 * g;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) kf[jj][ks] = *(const uint4*)(kr + 32 * ks);
        }
    };
    auto load_v = [&](int kbase) {
        int local;
        const uint16_t* Vp = (const uint16_t*)a.v + places.at(a, b, kvh, kbase, lane, local) * a.S * D;
        const uint16_t* vb = Vp + ((int64_t)(local / kVBlkBf16 + 2 * g) * D + c) * kVBlkBf16;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int t = 0; t < 2; ++t) vf[db][t] = *(const uint4*)(vb + ((int64_t)t * D + 16 * db) * kVBlkBf16);
    };
    // Operands that one path leaves unset have had an MFMA's result put over the V pieces that the next ones read (fp32 prefill, seen in the
    // assembly): the loop stands inside the condition of its first loads, and where a step's rows are staged between them a wavefront without
    // keys sets its operands too.
    int kbase = chunk_start + wave * kGroup;
    const bool any = kbase < chunk_end;
    if constexpr (STEP) {
        if (any) {
            load_k(kbase);
            load_v(kbase);
        } else {
#pragma unroll
            for (int i = 0; i < 4 * KS; ++i) kf[i / KS][i % KS] = uint4{0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < 2 * DB; ++i) vf[i / 2][i % 2] = uint4{0, 0, 0, 0};
        }
        __shared__ __attribute__((aligned(16))) uint16_t sm_step[18 * PITCH];
        for (int i = tid; i < n_pieces; i += 256) {
            if (i >= 256) load_piece(i);
            const StepPiece<PC> sp(i, column_count(a));
            if (a.table && !sp.is_v) {
                float x[8];
                load8<uint16_t>((const uint16_t*)&piece, x);
                rope_pairs<8>(x, pairs);
                piece = pack8_bf16(x);
            }
            *(uint4*)(sm_step + sp.row * PITCH + 8 * sp.p) = piece;
        }
        step_barrier();
        const uint16_t* sk = sm_step + column_count(a) * PITCH;
        const uint16_t* sv = sk + PITCH;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            uint4 w = *(const uint4*)(sm_step + (col.r - a.col0) * PITCH + 32 * ks + 8 * g);
            if (!col.live) w = uint4{0, 0, 0, 0};
            qf[ks] = __builtin_bit_cast(bf16x8_t, w);
        }
        if (owner) {
            float x = 0.f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                float qx[8], kx[8];
                load8<uint16_t>((const uint16_t*)&qf[ks], qx);
                load8<uint16_t>(sk + 32 * ks + 8 * g, kx);
#pragma unroll
                for (int e = 0; e < 8; ++e) x = __builtin_fmaf(qx[e], kx[e], x);
            }
            m = wave_sum_over_groups(x) * a.scale_log2;
            l = g == 0 ? 1.f : 0.f;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const uint2 w = *(const uint2*)(sv + 16 * db + 4 * g);
                acc[db] = f32x4_t{__builtin_bit_cast(float, w.x << 16), __builtin_bit_cast(float, w.x & 0xffff0000u),
                                  __builtin_bit_cast(float, w.y << 16), __builtin_bit_cast(float, w.y & 0xffff0000u)};
            }
            if (a.col0 == 0) {  // the rows enter the planes
                int local;
                const int64_t slab = token_slab<PAGED>(a, b, kvh, a.len, local) * a.S * D;
                if (lane < PC) *(uint4*)((uint16_t*)a.k + slab + (int64_t)local * D + 8 * lane) = *(const uint4*)(sk + 8 * lane);
                uint16_t* vp = (uint16_t*)a.v + slab + (int64_t)(local / kVBlkBf16) * D * kVBlkBf16 + local % kVBlkBf16;
#pragma unroll
                for (int d = 0; d < D; d += 64) vp[(d + lane) * kVBlkBf16] = sv[d + lane];
            }
        }
    }
    if (any) {
    if constexpr (!STEP) {
        load_k(kbase);
        load_v(kbase);
    }
    for (;;) {
        const int knext = kbase + kWaves * kGroup;
        // ---- S^T
        f32x4_t s[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            s[jj] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                s[jj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[jj][ks]), qf[ks], s[jj], 0, 0, 0);
        }
        if (knext < chunk_end) load_k(knext);
        const bool tail = kbase + kGroup > chunk_end;               // keys past the end of the split: stale rows of the planes
        const bool tail_s = kbase + kGroup > chunk_end - (a.T - 1);  // keys past some column's limit
        float mloc = -INFINITY;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float t = s[jj][v] * a.scale_log2;
                if (tail_s && kbase + 16 * g + 4 * jj + v >= lim) t = -INFINITY;
                s[jj][v] = t;
                mloc = fmaxf(mloc, t);
            }
        mloc = wave_max_over_groups(mloc);
        const float m_new = fmaxf(m, mloc);
        // -inf while a column has seen no key yet (several tokens per sequence: the last keys of a context lie past the
        // earlier tokens' limits); its sums then stay zero
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - m_ref);
        float lsum = 0.f;
        uint32_t pw[2][4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            float p0 = __builtin_amdgcn_exp2f(s[jj][0] - m_ref), p1 = __builtin_amdgcn_exp2f(s[jj][1] - m_ref);
            float p2 = __builtin_amdgcn_exp2f(s[jj][2] - m_ref), p3 = __builtin_amdgcn_exp2f(s[jj][3] - m_ref);
            lsum += (p0 + p1) + (p2 + p3);
            pw[jj >> 1][2 * (jj & 1)] = pack_bf16x2(p0, p1);
            pw[jj >> 1][2 * (jj & 1) + 1] = pack_bf16x2(p2, p3);
        }
        l = l * alpha + lsum;
        m = m_new;
        if (tail) {
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int t = 0; t < 2; ++t) vf[db][t] = mask_tail_u16x8(vf[db][t], chunk_end - (kbase + 16 * g + 8 * t));
        }
        // ---- O^T
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            acc[db] *= alpha;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                bf16x8_t pf = __builtin_bit_cast(bf16x8_t, uint4{pw[t][0], pw[t][1], pw[t][2], pw[t][3]});
                acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vf[db][t]), pf, acc[db], 0, 0, 0);
            }
        }
        if (knext >= chunk_end) break;
        load_v(knext);
        kbase = knext;
    }
    }
    l = wave_sum_over_groups(l);

    // ---- combine the four wavefronts through LDS, write one partial per (b, head, split)
    if (col.live) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int v = 0; v < 4; ++v) sm_o[wave][c][16 * db + 4 * g + v] = acc[db][v];
        if (g == 0) {
            sm_m[wave][c] = m;
            sm_l[wave][c] = l;
        }
    }
    __syncthreads();
    merge_waves_and_store<D, false, uint16_t>(a, sm_o, sm_m, sm_l, b, kvh, split, n_splits, tid, walk);
    if constexpr (RANGE) __syncthreads();  // everyone is done with the exchange
    } while (next_piece(a, walk));
}
template <int D, bool PAGED, bool STEP, bool RANGE>
__global__ void __launch_bounds__(256, 2) decode_bf16_kernel(DecodeArgs a) { decode_bf16_body<D, PAGED, STEP, RANGE, false>(a); }
template <int D, bool PAGED>
__global__ void __launch_bounds__(256, 2) decode_bf16_round_kernel(DecodeArgs a) { decode_bf16_body<D, PAGED, false, false, true>(a); }

// ---------------------------------------------------------------------------------------------
// Q8_0 cache: int8 payload widened to fp16 in registers and scaled, fp16 MFMA.
// ---------------------------------------------------------------------------------------------
// 4 int8 (one dword, two's complement) -> 4 fp16 holding the same integers.  x ^ 0x80 is the
// biased value u = q + 128; 0x6400 | u is the fp16 1024 + u; subtracting 1152 is exact.
__device__ inline void i8x4_to_f16x4(uint32_t w, f16x2_t& lo, f16x2_t& hi) {
    const uint32_t x = w ^ 0x80808080u;
    const uint32_t a = __builtin_amdgcn_perm(0x64646464u, x, 0x04010400u);
    const uint32_t bq = __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u);
    const f16x2_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    lo = __builtin_bit_cast(f16x2_t, a) - bias;
    hi = __builtin_bit_cast(f16x2_t, bq) - bias;
}
__device__ inline uint32_t f16x2_bits(f16x2_t v) { return __builtin_bit_cast(uint32_t, v); }

template <int D, bool PAGED, bool STEP, bool ROUND>
__device__ __forceinline__ void decode_q8_body(DecodeArgs a) {
    constexpr int KS = D / 32;
    constexpr int DB = D / 16;
    constexpr int NH = D / 64;  // 16-byte K loads per row per lane
    constexpr int NQ = D / kQBlock;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ __attribute__((aligned(16))) float sm_o[kWaves][16][D + 4];
    __shared__ float sm_m[kWaves][16], sm_l[kWaves][16];
    int kvh, b, split, L, n_splits, item, chunk;
    block_coords(a, kvh, item);
    if (!locate_work<ROUND>(a, item, lane, b, split, L, n_splits, chunk)) return;
    const int chunk_start = split * chunk;
    const int chunk_end = min(L, chunk_start + chunk);

    const int c = lane & 15, g = lane >> 4;
    GroupPlaces<PAGED> places;
    places.init(a, b, kvh, chunk_start, lane);

    // Q^T operands in fp16.  Contraction slot (ks, g, e) is head-dim index
    // 64*(ks/2) + 16*g + 8*(ks%2) + e, so that one 16-byte K load (16 int8) feeds two k-steps.
    const Column col = column_of(a, c);
    const int lim = column_limit(a, col, L, chunk_end);
    f16x8_t qf[KS];
    const bool owner = STEP && step_owner(split, n_splits, wave);
    constexpr int PC = D / 8, PITCH = D + 8;
    auto q_operand = [&](int ks, uint4 w) {
        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float lo = bf16_bits_to_f32((uint16_t)(ww[i] & 0xFFFFu)), hi = bf16_bits_to_f32((uint16_t)(ww[i] >> 16));
            lo = fminf(fmaxf(lo, -65504.f), 65504.f);
            hi = fminf(fmaxf(hi, -65504.f), 65504.f);
            if (!col.live) lo = hi = 0.f;
            qf[ks][2 * i] = (_Float16)lo;
            qf[ks][2 * i + 1] = (_Float16)hi;
        }
    };
    [[maybe_unused]] uint4 piece;
    [[maybe_unused]] float4 pairs[2];
    [[maybe_unused]] const int n_pieces = (column_count(a) + 2) * PC;
    [[maybe_unused]] auto load_piece = [&](int i) {
        const StepPiece<PC> sp(i, column_count(a));
        piece = *(const uint4*)(step_source<uint16_t>(a, sp, b, kvh) + 8 * sp.p);
        if (a.table && !sp.is_v) pairs[0] = step_pairs<D>(a, 8 * sp.p)[0], pairs[1] = step_pairs<D>(a, 8 * sp.p)[1];
    };
    if constexpr (STEP) {
        if (tid < n_pieces) load_piece(tid);
    } else {
        const uint16_t* qrow = (const uint16_t*)a.q + (int64_t)b * a.sq_b + (int64_t)(kvh * a.n_rep + col.r) * a.sq_h + (int64_t)col.t * a.sq_t;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) q_operand(ks, *(const uint4*)(qrow + 64 * (ks >> 1) + 16 * g + 8 * (ks & 1)));
    }
    const int krow = 16 * (c >> 2) + (c & 3);

    f32x4_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    // loads of one 64-key group; rotated like the bf16 kernel (K re-issued after S^T, V after O^T)
    uint4 kq[4][NH];
    uint16_t ksc[4][NH];
    uint4 vq[DB];
    uint4 vsc[NQ][2];
    auto load_k = [&](int kbase) {
        int local;
        const int64_t head = places.at(a, b, kvh, kbase, lane, local);
        const int8_t* Kp = (const int8_t*)a.k + head * a.S * D;
        const uint16_t* KSp = (const uint16_t*)a.k_scale + head * a.S * NQ;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const int64_t key = local + krow + 4 * jj;
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                kq[jj][h] = *(const uint4*)(Kp + key * D + 64 * h + 16 * g);
                ksc[jj][h] = KSp[key * NQ + 2 * h + (g >> 1)];
            }
        }
    };
    auto load_v = [&](int kbase) {
        int local;
        const int64_t head = places.at(a, b, kvh, kbase, lane, local);
        const int8_t* Vp = (const int8_t*)a.v + head * a.S * D;
        const uint16_t* VSp = (const uint16_t*)a.v_scale + head * a.S * NQ;
        const int64_t blk = local / kVBlkQ8 + g;
#pragma unroll
        for (int db = 0; db < DB; ++db) vq[db] = *(const uint4*)(Vp + (blk * D + 16 * db + c) * kVBlkQ8);
#pragma unroll
        for (int qb = 0; qb < NQ; ++qb) {
            const uint4* sp = (const uint4*)(VSp + (blk * NQ + qb) * kVBlkQ8);
            vsc[qb][0] = sp[0];
            vsc[qb][1] = sp[1];
        }
    };
    // (as in decode_bf16_kernel)
    int kbase = chunk_start + wave * kGroup;
    const bool any = kbase < chunk_end;
    if constexpr (STEP) {
        if (any) {
            load_k(kbase);
            load_v(kbase);
        } else {
#pragma unroll
            for (int i = 0; i < 4 * NH; ++i) kq[i / NH][i % NH] = uint4{0, 0, 0, 0}, ksc[i / NH][i % NH] = 0;
#pragma unroll
            for (int i = 0; i < DB; ++i) vq[i] = uint4{0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < 2 * NQ; ++i) vsc[i / 2][i % 2] = uint4{0, 0, 0, 0};
        }
        __shared__ __attribute__((aligned(16))) uint16_t sm_step[16 * PITCH];
        __shared__ __attribute__((aligned(16))) uint32_t sm_q8[2][D / 4];  // the token's quantised K and V
        __shared__ uint16_t sm_sc[2][NQ];
        for (int i = tid; i < n_pieces; i += 256) {
            if (i >= 256) load_piece(i);
            const StepPiece<PC> sp(i, column_count(a));
            float x[8];
            load8<uint16_t>((const uint16_t*)&piece, x);
            if (a.table && !sp.is_v) rope_pairs<8>(x, pairs);
            if (sp.is_q) {
                *(uint4*)(sm_step + sp.row * PITCH + 8 * sp.p) = a.table ? pack8_bf16(x) : piece;
            } else {  // four lanes share a block of 32, as in append_q8_kernel
                float amax = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(x[j]));
                amax = fmaxf(amax, __shfl_xor(amax, 1));
                amax = fmaxf(amax, __shfl_xor(amax, 2));
                const q8_scale sc = q8_block_scale(amax);
                *(uint2*)&sm_q8[sp.is_v][2 * sp.p] = uint2{q8_pack4(x, sc.inverse), q8_pack4(x + 4, sc.inverse)};
                if (sp.p % 4 == 0) sm_sc[sp.is_v][sp.p / 4] = sc.bits;
            }
        }
        step_barrier();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) q_operand(ks, *(const uint4*)(sm_step + (col.r - a.col0) * PITCH + 64 * (ks >> 1) + 16 * g + 8 * (ks & 1)));
        if (owner) {
            float x = 0.f;
#pragma unroll
            for (int i = 0; i < D / 16; ++i) {  // four elements of K: d = 64 (i / 4) + 16 g + 4 (i % 4) ..
                const _Float16 sc = __builtin_bit_cast(_Float16, sm_sc[0][2 * (i >> 2) + (g >> 1)]);
                f16x2_t lo, hi;
                i8x4_to_f16x4(sm_q8[0][16 * (i >> 2) + 4 * g + (i & 3)], lo, hi);
                lo *= f16x2_t{sc, sc}, hi *= f16x2_t{sc, sc};
                const f16x8_t& qo = qf[i >> 1];
                const int e = 4 * (i & 1);
                x = __builtin_fmaf((float)qo[e], (float)lo[0], x);
                x = __builtin_fmaf((float)qo[e + 1], (float)lo[1], x);
                x = __builtin_fmaf((float)qo[e + 2], (float)hi[0], x);
                x = __builtin_fmaf((float)qo[e + 3], (float)hi[1], x);
            }
            m = wave_sum_over_groups(x) * a.scale_log2;
            l = g == 0 ? 1.f : 0.f;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const _Float16 sc = __builtin_bit_cast(_Float16, sm_sc[1][db >> 1]);
                f16x2_t lo, hi;
                i8x4_to_f16x4(sm_q8[1][4 * db + g], lo, hi);
                lo *= f16x2_t{sc, sc}, hi *= f16x2_t{sc, sc};
                acc[db] = f32x4_t{(float)lo[0], (float)lo[1], (float)hi[0], (float)hi[1]};
            }
            if (a.col0 == 0) {  // the rows enter the planes
                int local;
                const int64_t head = token_slab<PAGED>(a, b, kvh, a.len, local);
                if (lane < D / 4) {
                    *(uint32_t*)((int8_t*)a.k + (head * a.S + local) * D + 4 * lane) = sm_q8[0][lane];
                    int8_t* vp = (int8_t*)a.v + head * a.S * D + ((int64_t)(local / kVBlkQ8) * D + 4 * lane) * kVBlkQ8 + local % kVBlkQ8;
                    const uint32_t w = sm_q8[1][lane];
#pragma unroll
                    for (int j = 0; j < 4; ++j) vp[j * kVBlkQ8] = (int8_t)(w >> (8 * j));
                }
                if (lane < NQ) {
                    ((uint16_t*)a.k_scale)[(head * a.S + local) * NQ + lane] = sm_sc[0][lane];
                    ((uint16_t*)a.v_scale)[head * a.S * NQ + ((int64_t)(local / kVBlkQ8) * NQ + lane) * kVBlkQ8 + local % kVBlkQ8] = sm_sc[1][lane];
                }
            }
        }
    }
    if (any) {
    if constexpr (!STEP) {
        load_k(kbase);
        load_v(kbase);
    }
    for (;;) {
        const bool tail = kbase + kGroup > chunk_end;
        const bool tail_s = kbase + kGroup > chunk_end - (a.T - 1);
        const int knext = kbase + kWaves * kGroup;
        // ---- S^T
        f32x4_t s[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            s[jj] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const _Float16 sc = __builtin_bit_cast(_Float16, ksc[jj][h]);
                const f16x2_t sc2 = {sc, sc};
                const uint32_t w[4] = {kq[jj][h].x, kq[jj][h].y, kq[jj][h].z, kq[jj][h].w};
                uint32_t o[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    f16x2_t lo, hi;
                    i8x4_to_f16x4(w[i], lo, hi);
                    o[2 * i] = f16x2_bits(lo * sc2);
                    o[2 * i + 1] = f16x2_bits(hi * sc2);
                }
                f16x8_t k0 = __builtin_bit_cast(f16x8_t, uint4{o[0], o[1], o[2], o[3]});
                f16x8_t k1 = __builtin_bit_cast(f16x8_t, uint4{o[4], o[5], o[6], o[7]});
                s[jj] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0, qf[2 * h], s[jj], 0, 0, 0);
                s[jj] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k1, qf[2 * h + 1], s[jj], 0, 0, 0);
            }
        }
        if (knext < chunk_end) load_k(knext);
        float mloc = -INFINITY;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float t = s[jj][v] * a.scale_log2;
                if (tail_s && kbase + 16 * g + 4 * jj + v >= lim) t = -INFINITY;
                s[jj][v] = t;
                mloc = fmaxf(mloc, t);
            }
        mloc = wave_max_over_groups(mloc);
        const float m_new = fmaxf(m, mloc);
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;   // see decode_bf16_kernel
        const float alpha = __builtin_amdgcn_exp2f(m - m_ref);
        float lsum = 0.f;
        f16x8_t pf[2];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float p = __builtin_amdgcn_exp2f(s[jj][v] - m_ref);
                lsum += p;
                pf[jj >> 1][4 * (jj & 1) + v] = (_Float16)p;
            }
        l = l * alpha + lsum;
        m = m_new;
        // ---- O^T: dequantise V^T operands (16 tokens of one d per lane; per-token scales)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            acc[db] *= alpha;
            const int qb = (16 * db) / kQBlock;
            const uint32_t w[4] = {vq[db].x, vq[db].y, vq[db].z, vq[db].w};
            const uint32_t scw[8] = {vsc[qb][0].x, vsc[qb][0].y, vsc[qb][0].z, vsc[qb][0].w,
                                     vsc[qb][1].x, vsc[qb][1].y, vsc[qb][1].z, vsc[qb][1].w};
            uint32_t o[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                f16x2_t lo, hi;
                i8x4_to_f16x4(w[i], lo, hi);
                o[2 * i] = f16x2_bits(lo * __builtin_bit_cast(f16x2_t, scw[2 * i]));
                o[2 * i + 1] = f16x2_bits(hi * __builtin_bit_cast(f16x2_t, scw[2 * i + 1]));
            }
            uint4 v0 = uint4{o[0], o[1], o[2], o[3]}, v1 = uint4{o[4], o[5], o[6], o[7]};
            if (tail) {
                v0 = mask_tail_u16x8(v0, chunk_end - (kbase + 16 * g));
                v1 = mask_tail_u16x8(v1, chunk_end - (kbase + 16 * g + 8));
            }
            acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, v0), pf[0], acc[db], 0, 0, 0);
            acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, v1), pf[1], acc[db], 0, 0, 0);
        }
        if (knext >= chunk_end) break;
        load_v(knext);
        kbase = knext;
    }
    }
    l = wave_sum_over_groups(l);

    if (col.live) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int v = 0; v < 4; ++v) sm_o[wave][c][16 * db + 4 * g + v] = acc[db][v];
        if (g == 0) {
            sm_m[wave][c] = m;
            sm_l[wave][c] = l;
        }
    }
    __syncthreads();
    merge_waves_and_store<D, false, uint16_t>(a, sm_o, sm_m, sm_l, b, kvh, split, n_splits, tid, NoWalk{});
}
template <int D, bool PAGED, bool STEP>
__global__ void __launch_bounds__(256, 2) decode_q8_kernel(DecodeArgs a) { decode_q8_body<D, PAGED, STEP, false>(a); }
template <int D, bool PAGED>
__global__ void __launch_bounds__(256, 2) decode_q8_round_kernel(DecodeArgs a) { decode_q8_body<D, PAGED, false, true>(a); }

// ---------------------------------------------------------------------------------------------
// fp32 cache in the reference's own layout, any head size: plain fp32 arithmetic, one workgroup per
// (batch row, group of query heads, split).  Serves what decode_f32_mfma_kernel does not take (D other than 64 / 128,
// more than 16 query heads per kv head).
// ---------------------------------------------------------------------------------------------
// NH query heads of one kv head per workgroup (NH divides n_rep), so that K and V are read n_rep / NH times instead of
// n_rep times; a thread owns a key in the score phase and a (d, key residue) pair in the output phase.
template <int MAXD, int NH>
__global__ void __launch_bounds__(256) decode_f32_kernel(DecodeArgs a, int D) {
    const int tid = threadIdx.x;
    const int hq0 = blockIdx.y * NH;
    int b, split, L, n_splits, chunk;
    if (!locate_work(a, blockIdx.x, tid & 63, b, split, L, n_splits, chunk)) return;
    const int chunk_start = split * chunk;
    const int chunk_end = min(L, chunk_start + chunk);
    const int n = chunk_end - chunk_start;
    const int kvh = hq0 / a.n_rep;

    extern __shared__ float smem[];
    float* sq = smem;                    // [NH][MAXD]
    float* sp = smem + NH * MAXD;        // [NH][chunk]
    float* red = sp + NH * a.chunk;      // [256]
    for (int i = tid; i < NH * D; i += 256) {
        const int r = i / D, d = i - r * D;
        sq[r * MAXD + d] = ((const float*)a.q + (int64_t)b * a.sq_b + (int64_t)(hq0 + r) * a.sq_h)[d];
    }
    __syncthreads();
    const float* Kp = (const float*)a.k + (((int64_t)b * a.Hkv + kvh) * a.S + chunk_start) * D;
    const float* Vp = (const float*)a.v + (((int64_t)b * a.Hkv + kvh) * a.S + chunk_start) * D;
    float mloc[NH];
#pragma unroll
    for (int r = 0; r < NH; ++r) mloc[r] = -INFINITY;
    for (int j = tid; j < n; j += 256) {
        const float4* kr = (const float4*)(Kp + (int64_t)j * D);
        float s[NH];
#pragma unroll
        for (int r = 0; r < NH; ++r) s[r] = 0.f;
        for (int d4 = 0; d4 < D / 4; ++d4) {
            const float4 kk = kr[d4];
#pragma unroll
            for (int r = 0; r < NH; ++r) {
                const float* qr = sq + r * MAXD + 4 * d4;
                s[r] = fmaf(qr[0], kk.x, s[r]);
                s[r] = fmaf(qr[1], kk.y, s[r]);
                s[r] = fmaf(qr[2], kk.z, s[r]);
                s[r] = fmaf(qr[3], kk.w, s[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < NH; ++r) {
            const float t = s[r] * a.scale_log2;
            sp[r * a.chunk + j] = t;
            mloc[r] = fmaxf(mloc[r], t);
        }
    }
    float m[NH], l[NH];
#pragma unroll
    for (int r = 0; r < NH; ++r) {
        red[tid] = mloc[r];
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if (tid < st) red[tid] = fmaxf(red[tid], red[tid + st]);
            __syncthreads();
        }
        m[r] = red[0];
        __syncthreads();
        float lloc = 0.f;
        for (int j = tid; j < n; j += 256) {
            const float p = exp2f(sp[r * a.chunk + j] - m[r]);
            sp[r * a.chunk + j] = p;
            lloc += p;
        }
        red[tid] = lloc;
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if (tid < st) red[tid] += red[tid + st];
            __syncthreads();
        }
        l[r] = red[0];
        __syncthreads();
    }
    // PV: thread (d, part) sums keys part, part+P, ...; P = 256 / D' where D' = D rounded up to a power of two
    int Dp = 1;
    while (Dp < D) Dp <<= 1;
    const int P = 256 / Dp > 0 ? 256 / Dp : 1;
    const int d = tid % Dp, part = tid / Dp;
    float o[NH];
#pragma unroll
    for (int r = 0; r < NH; ++r) o[r] = 0.f;
    if (d < D && part < P)
        for (int j = part; j < n; j += P) {
            const float vv = Vp[(int64_t)j * D + d];
#pragma unroll
            for (int r = 0; r < NH; ++r) o[r] = fmaf(sp[r * a.chunk + j], vv, o[r]);
        }
#pragma unroll
    for (int r = 0; r < NH; ++r) {
        __syncthreads();
        red[tid] = o[r];
        __syncthreads();
        if (tid < D && tid < Dp) {
            float t = 0.f;
            for (int p = 0; p < P; ++p) t += red[p * Dp + tid];
            const int64_t row = ((int64_t)b * a.Hq + hq0 + r) * a.max_splits + split;
            a.ws_o[row * D + tid] = t;
            if (tid == 0) {
                a.ws_ml[row * 2] = m[r];
                a.ws_ml[row * 2 + 1] = l[r];
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// fp32 cache, D = 64 or 128, n_rep <= 16: the bf16 kernel's structure on fp32 matrix instructions
// (v_mfma_f32_16x16x4_f32), so that the reference's own cache layout is also read once per kv head and at the
// rate HBM delivers it.  One workgroup (4 wavefronts) per (batch row, kv head, context split); a wavefront
// consumes 32 keys per iteration as two 16-key tiles.
//   S^T[key][head] = K[key][:] . Q^T[:][head]: lane (row i, k-slot kk) of the A operand loads the 16 bytes
//     K[key i][16 cc + 4 kk .. + 3] and feeds its four floats to four MFMAs; MFMA (cc, e) contracts over
//     d = 16 cc + 4 kk + e, and the Q^T operand is laid out to match (scale * log2(e) folded in).
//   O^T[d][head] += V^T[d][key] . P^T[key][head]: the S^T result of a lane holds keys 4 g + v of the tile, so
//     k-step v of the PV product takes the keys {4 kk + v}: P needs no cross-lane movement and stays fp32.
//     Lane (row i, kk) loads the 16 bytes V[key 4 kk + v][64 vc + 4 i .. + 3] and feeds them to four MFMAs;
//     tile (vc, e) therefore holds the rows d = 64 vc + 4 i + e.
// Rows past the end of the split may hold anything and the planes are not padded: K is read from the split's last row instead and masked in S, V
// through a descriptor that ends with that row, beyond which it is zeros (an infinity in the row must not meet weights of 0).
//
// FEW, up to 4 columns (n_rep x tokens): v_mfma_f32_4x4x1_f32, whose 16 blocks of 4 x 4 use every column of theirs.  Of 16 columns 4 would
// leave three quarters of the matrix pipe's time to zeros: 2048 cycles a group at D 64 where these take 512, and fp32 MFMAs and vector
// instructions do not overlap.  Lane (c, g) belongs to the block (kq = c / 4, g):
//   S: row c % 4 is key 4 kq + c % 4 = c and the block sums over the d of its g, so the loads of K and Q are the same, with column c % 4; the
//     four g are added by two lane swaps, after which the lane holds the scores of the keys 4 kq + v.
//   O^T += V^T P^T: step v is key 4 kq + v, row i the four floats of the piece 4 g + i: a lane loads V[key 4 kq + v][64 vc + 16 g + 4 (c % 4) ..],
//     P again needs no movement, acc[vc][e][v] is the same d as above, and the four kq are added once at the end.
// Measured, us, 16 columns -> these: 8 / 2 heads, D 64, 256 keys 7.1 -> 6.5 (a token step); 4 x 32 / 8 heads, D 128, 256 keys 10.9 -> 9.4; 32 heads,
// 3000 keys 21.9 -> 20.1; 32 / 8 heads, 20000 keys 33.1 -> 31.2; 16 rows of 1000 to 16000 keys 226 -> 223.
// The error against 64 bits falls to a half to a third (D 64, 256 keys 3.0e-7 -> 1.5e-7): shorter chains, four of them added at the end.
// ---------------------------------------------------------------------------------------------
template <int D, bool STEP, bool RANGE, bool FEW, bool ROUND>
__device__ __forceinline__ void decode_f32_mfma_body(DecodeArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    constexpr int C4 = D / 16;  // 16-byte pieces of a K row per lane
    constexpr int VC = D / 64;  // 16-byte pieces of a V row per lane
    constexpr int KT = 2;       // 16-key tiles per wavefront iteration
    constexpr int GROUP = 16 * KT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ __attribute__((aligned(16))) float sm_o[kWaves][16][D + 4];
    __shared__ float sm_m[kWaves][16], sm_l[kWaves][16];
    std::conditional_t<RANGE, RangeWalk, NoWalk> walk;
    if constexpr (RANGE) {
        if (!walk.start(a, lane, blockIdx.x)) return;
    }
    do {  // one pass, or one per piece of the workgroup's range
    int kvh, b, split = 0, L, n_splits = 1, chunk_start, chunk_end;
    if constexpr (RANGE) {
        b = walk.b, kvh = walk.kvh, L = walk.length();
        chunk_start = walk.off * kGroup;
        chunk_end = min(L, chunk_start + walk.piece() * kGroup);
    } else {
        int item, chunk;
        block_coords(a, kvh, item);
        if (!locate_work<ROUND>(a, item, lane, b, split, L, n_splits, chunk)) return;
        chunk_start = split * chunk;
        chunk_end = min(L, chunk_start + chunk);
    }
    const int c = lane & 15, g = lane >> 4;

    // FEW: lane (c, g) is row or column c % 4 of the block (c / 4, g)
    const int cq = FEW ? c & 3 : c, kq = FEW ? c >> 2 : 0;
    const int key_of = FEW ? 4 * kq : 4 * g;  // + v: the keys of a tile whose scores the lane holds
    const Column col = column_of(a, cq);
    const int lim = column_limit(a, col, L, chunk_end);
    float qf[C4][4];
    const bool owner = STEP && step_owner(split, n_splits, wave);
    constexpr int PC = D / 4, PITCH = D + 4;
    [[maybe_unused]] float4 piece, pairs;
    [[maybe_unused]] const int n_pieces = (column_count(a) + 2) * PC;
    [[maybe_unused]] auto load_piece = [&](int i) {
        const StepPiece<PC> sp(i, column_count(a));
        piece = *(const float4*)(step_source<float>(a, sp, b, kvh) + 4 * sp.p);
        if (a.table && !sp.is_v) pairs = *step_pairs<D>(a, 4 * sp.p);
    };
    const float q_factor = col.live ? a.scale_log2 : 0.f;
    if constexpr (STEP) {
        if (tid < n_pieces) load_piece(tid);
    } else {
        const float* qrow = (const float*)a.q + (int64_t)b * a.sq_b + (int64_t)(kvh * a.n_rep + col.r) * a.sq_h + (int64_t)col.t * a.sq_t;
#pragma unroll
        for (int cc = 0; cc < C4; ++cc) {
            const float4 w = *(const float4*)(qrow + 16 * cc + 4 * g);
            qf[cc][0] = w.x * q_factor, qf[cc][1] = w.y * q_factor, qf[cc][2] = w.z * q_factor, qf[cc][3] = w.w * q_factor;
        }
    }
    const float* Kp = (const float*)a.k + ((int64_t)b * a.Hkv + kvh) * a.S * D;
    const float* Vp = (const float*)a.v + ((int64_t)b * a.Hkv + kvh) * a.S * D;

    f32x4_t acc[VC][4];
#pragma unroll
    for (int i = 0; i < VC; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    float4 kf[KT][C4];
    f32x4_t vf[KT][4][VC];
    const int last = chunk_end - 1;
    auto load_k = [&](int kbase) {
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            const float* kr = Kp + (int64_t)min(kbase + 16 * t + c, last) * D + 4 * g;
#pragma unroll
            for (int cc = 0; cc < C4; ++cc) kf[t][cc] = *(const float4*)(kr + 16 * cc);
        }
    };
    auto load_v = [&](int kbase) {
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(Vp + (int64_t)kbase * D), 0, min(GROUP, chunk_end - kbase) * D * 4, 0x00020000);
        int at = 4 * D * key_of + 16 * (FEW ? 4 * g + cq : c);
        if constexpr (RANGE && D == 128) {  // made anew for each group: this instance has no register left to keep it in
            int x = lane;
            asm volatile("" : "+v"(x));
            at = FEW ? 16 * D * ((x & 15) >> 2) + 64 * (x >> 4) + 16 * (x & 3) : 16 * D * (x >> 4) + 16 * (x & 15);
        }
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int vc = 0; vc < VC; ++vc)
                    vf[t][v][vc] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, at + 4 * D * (16 * t + v) + 256 * vc, 0, 0));
    };
    // (as in decode_bf16_kernel)
    int kbase = chunk_start + wave * GROUP;
    const bool any = kbase < chunk_end;
    if constexpr (STEP) {
        if (any) {
            load_k(kbase);
            load_v(kbase);
        } else {
#pragma unroll
            for (int t = 0; t < KT; ++t) {
#pragma unroll
                for (int i = 0; i < C4; ++i) kf[t][i] = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 4 * VC; ++i) vf[t][i / VC][i % VC] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        __shared__ __attribute__((aligned(16))) float sm_step[18 * PITCH];
        for (int i = tid; i < n_pieces; i += 256) {
            if (i >= 256) load_piece(i);
            const StepPiece<PC> sp(i, column_count(a));
            float x[4] = {piece.x, piece.y, piece.z, piece.w};
            if (a.table && !sp.is_v) rope_pairs<4>(x, &pairs);
            *(float4*)(sm_step + sp.row * PITCH + 4 * sp.p) = float4{x[0], x[1], x[2], x[3]};
        }
        step_barrier();
        const float* sk = sm_step + column_count(a) * PITCH;
        const float* sv = sk + PITCH;
#pragma unroll
        for (int cc = 0; cc < C4; ++cc) {
            const float4 w = *(const float4*)(sm_step + col.r * PITCH + 16 * cc + 4 * g);
            qf[cc][0] = w.x * q_factor, qf[cc][1] = w.y * q_factor, qf[cc][2] = w.z * q_factor, qf[cc][3] = w.w * q_factor;
        }
        if (owner) {
            float x = 0.f;
#pragma unroll
            for (int cc = 0; cc < C4; ++cc) {
                const float4 k = *(const float4*)(sk + 16 * cc + 4 * g);
                x = __builtin_fmaf(qf[cc][0], k.x, x), x = __builtin_fmaf(qf[cc][1], k.y, x);
                x = __builtin_fmaf(qf[cc][2], k.z, x), x = __builtin_fmaf(qf[cc][3], k.w, x);
            }
            m = wave_sum_over_groups(x);
            l = (FEW ? kq : g) == 0 ? 1.f : 0.f;
            const float mine = kq == 0 ? 1.f : 0.f;  // FEW: the four kq are added at the end
#pragma unroll
            for (int vc = 0; vc < VC; ++vc)
#pragma unroll
                for (int v = 0; v < 4; ++v) {  // acc[vc][e][v] is the row d = 64 vc + 16 g + 4 v + e
                    const float4 y = *(const float4*)(sv + 64 * vc + 16 * g + 4 * v);
                    acc[vc][0][v] = mine * y.x, acc[vc][1][v] = mine * y.y, acc[vc][2][v] = mine * y.z, acc[vc][3][v] = mine * y.w;
                }
            const int64_t row = (((int64_t)b * a.Hkv + kvh) * a.S + a.len) * D;  // the rows enter the planes
            if (lane < PC) {
                *(float4*)((float*)a.k + row + 4 * lane) = *(const float4*)(sk + 4 * lane);
                *(float4*)((float*)a.v + row + 4 * lane) = *(const float4*)(sv + 4 * lane);
            }
        }
    }
    if (any) {
    if constexpr (!STEP) {
        load_k(kbase);
        load_v(kbase);
    }
    for (;;) {
        const int knext = kbase + kWaves * GROUP;
        f32x4_t s[KT];
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            f32x4_t part[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int cc = 0; cc < C4; ++cc) {
                const float kk[4] = {kf[t][cc].x, kf[t][cc].y, kf[t][cc].z, kf[t][cc].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (FEW) part[e & 1] = __builtin_amdgcn_mfma_f32_4x4x1f32(kk[e], qf[cc][e], part[e & 1], 0, 0, 0);
                    else part[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[e], qf[cc][e], part[0], 0, 0, 0);
                }
            }
            s[t] = part[0];
            if constexpr (FEW) {
#pragma unroll
                for (int v = 0; v < 4; ++v) s[t][v] = rows_sum(part[0][v] + part[1][v]);
            }
        }
        if (knext < chunk_end) load_k(knext);
        const bool tail_s = kbase + GROUP > chunk_end - (a.T - 1);
        float mloc = -INFINITY;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float x = s[t][v];
                if (tail_s && kbase + 16 * t + key_of + v >= lim) x = -INFINITY;
                s[t][v] = x;
                mloc = fmaxf(mloc, x);
            }
        mloc = FEW ? quads_max(mloc) : wave_max_over_groups(mloc);
        const float m_new = fmaxf(m, mloc);
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;   // see decode_bf16_kernel
        const float alpha = __builtin_amdgcn_exp2f(m - m_ref);
        float lsum = 0.f;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                s[t][v] = __builtin_amdgcn_exp2f(s[t][v] - m_ref);
                lsum += s[t][v];
            }
        l = l * alpha + lsum;
        m = m_new;
#pragma unroll
        for (int vc = 0; vc < VC; ++vc)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[vc][e] *= alpha;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int vc = 0; vc < VC; ++vc) {
                    const f32x4_t vv = vf[t][v][vc];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if constexpr (FEW) acc[vc][e] = __builtin_amdgcn_mfma_f32_4x4x1f32(vv[e], s[t][v], acc[vc][e], 0, 0, 0);
                        else acc[vc][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[e], s[t][v], acc[vc][e], 0, 0, 0);
                    }
                }
        if (knext >= chunk_end) break;
        load_v(knext);
        kbase = knext;
    }
    }
    l = FEW ? quads_sum(l) : wave_sum_over_groups(l);
    if constexpr (FEW) {
#pragma unroll
        for (int vc = 0; vc < VC; ++vc)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[vc][e][v] = quads_sum(acc[vc][e][v]);
    }

    // ---- combine the four wavefronts through LDS, write one partial per (b, head, split)
    if (col.live && kq == 0) {
#pragma unroll
        for (int vc = 0; vc < VC; ++vc)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int v = 0; v < 4; ++v) sm_o[wave][c][64 * vc + 4 * (4 * g + v) + e] = acc[vc][e][v];
        if (g == 0) {
            sm_m[wave][c] = m;
            sm_l[wave][c] = l;
        }
    }
    __syncthreads();
    merge_waves_and_store<D, true, float>(a, sm_o, sm_m, sm_l, b, kvh, split, n_splits, tid, walk);
    if constexpr (RANGE) __syncthreads();  // everyone is done with the exchange
    } while (next_piece(a, walk));
#endif
}
template <int D, bool STEP, bool RANGE, bool FEW>
__global__ void __launch_bounds__(256, 2) decode_f32_mfma_kernel(DecodeArgs a) { decode_f32_mfma_body<D, STEP, RANGE, FEW, false>(a); }
template <int D, bool FEW>
__global__ void __launch_bounds__(256, 2) decode_f32_mfma_round_kernel(DecodeArgs a) { decode_f32_mfma_body<D, false, false, FEW, true>(a); }

// The partials of the pairs that more than one workgroup holds, kCombineQuads outputs of four elements per workgroup, one per thread, all partials of a pair
// in flight at once.  (A workgroup of four wavefronts per pair, 8 partials at a time: 5 x 8 rows of 200 to 12000 bf16 keys, four tokens, 40.8 us for 37.4; 6 x 8 of
// 1500 to 24000, two tokens, 70.5 and 68.9; 3 x 16 of 640 to 20501, D 64, 38.8 and 37.8.)
constexpr int kCombineQuads = 64;
template <typename OutT, int D>
__global__ void __launch_bounds__(kCombineQuads) range_combine_kernel(DecodeArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    RangeWalk k;
    k.scan(a, threadIdx.x & 63);
    k.b = blockIdx.y;
    k.kvh = blockIdx.x;
    k.row(a);
    const int ncol = column_count(a), rows = 2 * a.range_wgs * ncol, kvh = k.kvh;
    const RangeParts parts(a, k);
    if (parts.n == 1) return;
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(a.ws_o, 0, rows * D * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rml = __builtin_amdgcn_make_buffer_rsrc(a.ws_ml, 0, rows * 8, 0x00020000);
    const int i = blockIdx.z * kCombineQuads + threadIdx.x;
    if (i >= ncol * (D / 4)) return;
    const int hc = i / (D / 4), d = 4 * (i % (D / 4));
    const Column col = column_of(a, hc);
    OutT* p = (OutT*)a.out + (int64_t)k.b * a.so_b + (int64_t)(kvh * a.n_rep + col.r) * a.so_h + (int64_t)col.t * a.so_t + d;
    store_out(p, merge_all_splits<D>(ro, rml, [=](int n) { return parts.slot(n) * ncol + hc; }, parts.n, d));
#endif
}

// ---------------------------------------------------------------------------------------------
// combine: out[b][h][:] = sum_s w_s O_s / sum_s w_s l_s, w_s = 2^(m_s - max m); fixed order.
// ---------------------------------------------------------------------------------------------
struct CombineArgs {
    const float* ws_o;
    const float* ws_ml;
    const int32_t* seq_lens;
    int32_t len, chunk, max_splits, Hq, D, L_cap, T;
    void* out;
    int64_t so_b, so_h, so_t, rows;
    CombineExtra x;
};
template <typename OutT, int BLK, bool ROUND>
__device__ __forceinline__ void decode_combine_body(const CombineArgs& a) {
    const float *__restrict__ ws_o = a.ws_o, *__restrict__ ws_ml = a.ws_ml;
    const int32_t* __restrict__ seq_lens = a.seq_lens;
    OutT* __restrict__ out = (OutT*)a.out;
    const int max_splits = a.max_splits, Hq = a.Hq, D = a.D, T = a.T;
    const CombineExtra& x = a.x;
    const int hq = blockIdx.x / T, t = blockIdx.x % T, b = blockIdx.y, d = threadIdx.x;
    // the producers' clamp: [0, L_cap] in the decode step (locate_work); a chunk of a prompt is part of its context, so
    // there a row is at least as long as its chunk (prefill_bf16_pipe_kernel)
    const int len_floor = x.chunk_lens ? min(max(x.chunk_lens[b], 0), x.len_floor) : x.len_floor;
    const int L = min(max(seq_lens ? seq_lens[b] : a.len, len_floor), a.L_cap);
    const int chunk = split_chunk<ROUND>(seq_lens, x.B, a.L_cap, a.chunk, x.uniform_splits, x.round, threadIdx.x & 63);
    const int ns = min((L + chunk - 1) / chunk, max_splits);
    const int64_t row0 = (((int64_t)b * Hq + hq) * T + t) * max_splits;
    // One pass over blocks of BLK splits (8, 16 or 32, the smallest that covers the launch's split count): everything a block needs (maxima, sums, partial rows) is requested before any of
    // it is used, so the workgroup pays one memory latency per block instead of one per dependent step; across blocks
    // the reference point moves as in the online softmax.  Within a block and across blocks the sums run over the
    // splits in ascending order: the result does not depend on anything but the inputs.
    float M = -INFINITY, o = 0.f, l = 0.f;
    const float* po = ws_o + row0 * D + (d < D ? d : 0);
    for (int s0 = 0; s0 < ns; s0 += BLK) {
        float x[BLK], ms[BLK], ls[BLK];
#pragma unroll
        for (int i = 0; i < BLK; ++i) {
            const int64_t si = min(s0 + i, ns - 1);
            x[i] = po[si * D];
            ms[i] = ws_ml[(row0 + si) * 2];
            ls[i] = ws_ml[(row0 + si) * 2 + 1];
        }
        float Mb = M;
#pragma unroll
        for (int i = 0; i < BLK; ++i) Mb = fmaxf(Mb, ms[i]);   // indices past the end repeat the last split: harmless in a maximum
        const float keep = exp2f(M - Mb);                      // 0 for the first block (M = -inf, Mb finite)
        o *= keep;
        l *= keep;
        M = Mb;
#pragma unroll
        for (int i = 0; i < BLK; ++i)
            if (s0 + i < ns) {
                const float w = exp2f(ms[i] - M);
                l += w * ls[i];
                o += w * x[i];
            }
    }
    if (d < D) {
        const float r = (ns > 0 && l > 0.f) ? o / l : 0.f;   // l = 0: a token placed before the start of its context
        OutT* p = out + (int64_t)b * a.so_b + (int64_t)hq * a.so_h + (int64_t)t * a.so_t + d;
        if constexpr (sizeof(OutT) == 4) *p = r;
        else *p = f32_to_bf16_bits(r);
    }
    // LSE = m + log l (src/ops/flash_attention.cpp:359), here from the merged (M, l) in the log2 domain; a row that met
    // no key has l = 0 and reads -inf, as the unsplit kernels write it
    if (x.lse && d == 0) x.lse[(int64_t)b * x.sl[0] + (int64_t)hq * x.sl[1] + (int64_t)t * x.sl[2]] = (M + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
}
template <typename OutT, int BLK>
__global__ void __launch_bounds__(256) decode_combine_kernel(CombineArgs a) { decode_combine_body<OutT, BLK, false>(a); }
template <typename OutT, int BLK>
__global__ void __launch_bounds__(256) decode_combine_round_kernel(CombineArgs a) { decode_combine_body<OutT, BLK, true>(a); }

// The same merge for head_dim 64 / 128 and aligned output rows: D / 4 lanes per row, four columns each (16-byte loads of
// the partials, 8- or 16-byte stores), several rows per workgroup.  One row per workgroup with a column per thread is
// bound by the workgroups' start-up once there are thousands of rows: 16384 rows of four partials (a 512-token chunk over
// a split context) took 18 us for 38 MB.  Same operations in the same order per element as above.
template <typename OutT, int D, int BLK, bool ROUND>
__device__ __forceinline__ void split_combine_body(const CombineArgs& a) {
    const float *__restrict__ ws_o = a.ws_o, *__restrict__ ws_ml = a.ws_ml;
    const int32_t* __restrict__ seq_lens = a.seq_lens;
    OutT* __restrict__ out = (OutT*)a.out;
    const int max_splits = a.max_splits, Hq = a.Hq, T = a.T;
    const CombineExtra& x = a.x;
    constexpr int LPR = D / 4;
    const int64_t r = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / LPR;
    const int d = 4 * (threadIdx.x % LPR);
    const int chunk = split_chunk<ROUND>(seq_lens, x.B, a.L_cap, a.chunk, x.uniform_splits, x.round, threadIdx.x & 63);
    if (r >= a.rows) return;
    const int t = (int)(r % T), hq = (int)(r / T % Hq), b = (int)(r / T / Hq);
    const int len_floor = x.chunk_lens ? min(max(x.chunk_lens[b], 0), x.len_floor) : x.len_floor;
    const int L = min(max(seq_lens ? seq_lens[b] : a.len, len_floor), a.L_cap);
    const int ns = min((L + chunk - 1) / chunk, max_splits);
    const int64_t row0 = r * max_splits;
    float M = -INFINITY, l = 0.f;
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
    const float* po = ws_o + row0 * D + d;
    for (int s0 = 0; s0 < ns; s0 += BLK) {
        f32x4_t v[BLK];
        float ms[BLK], ls[BLK];
#pragma unroll
        for (int i = 0; i < BLK; ++i) {
            const int64_t si = min(s0 + i, ns - 1);
            v[i] = *(const f32x4_t*)(po + si * D);
            const float2 ml = *(const float2*)(ws_ml + (row0 + si) * 2);
            ms[i] = ml.x;
            ls[i] = ml.y;
        }
        float Mb = M;
#pragma unroll
        for (int i = 0; i < BLK; ++i) Mb = fmaxf(Mb, ms[i]);
        const float Mr = Mb == -INFINITY ? 0.f : Mb;  // no key so far: zero sums, weights 2^-inf
        const float keep = exp2f(M - Mr);
        o *= keep;
        l *= keep;
        M = Mb;
#pragma unroll
        for (int i = 0; i < BLK; ++i)
            if (s0 + i < ns) {
                const float w = exp2f(ms[i] - Mr);
                l += w * ls[i];
                o += w * v[i];
            }
    }
    f32x4_t y = {0.f, 0.f, 0.f, 0.f};
    if (ns > 0 && l > 0.f) {  // l = 0: a token placed before the start of its context
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = o[j] / l;
    }
    OutT* p = out + (int64_t)b * a.so_b + (int64_t)hq * a.so_h + (int64_t)t * a.so_t + d;
    if constexpr (sizeof(OutT) == 4) *(f32x4_t*)p = y;
    else *(u32x2_t*)p = u32x2_t{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    if (x.lse && d == 0) x.lse[(int64_t)b * x.sl[0] + (int64_t)hq * x.sl[1] + (int64_t)t * x.sl[2]] = (M + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
}
template <typename OutT, int D, int BLK>
__global__ void __launch_bounds__(256) split_combine_kernel(CombineArgs a) { split_combine_body<OutT, D, BLK, false>(a); }
template <typename OutT, int D, int BLK>
__global__ void __launch_bounds__(256) split_combine_round_kernel(CombineArgs a) { split_combine_body<OutT, D, BLK, true>(a); }

// ---------------------------------------------------------------------------------------------
// Output projection behind the combine: y[m][n] = sum_k x[m][k] W[n][k] + bias[n]
// (Linear::forward, src/nn/linear.cpp:41-49, as GroupedQueryAttention applies it to the merged heads,
// src/nn/gqa_attention.cpp:151-152).  x is the decode output [B][Hq*D] left in the workspace, so M = B is small and
// the job is one pass over W at HBM rate.  Workgroup (nb, ks) owns 128 output columns (16 per wavefront) and the
// ks-th of KS equal ranges of K.  Per 512-wide piece of its range every lane first issues its sixteen 16-byte loads
// of W rows (the A operands of 16x16x32 MFMAs, straight from HBM into registers), then the workgroup stages the
// matching piece of x in LDS once for its eight wavefronts (x^T is the B operand; up to MT tiles of 16 batch rows share
// the pass over W).  The fp32 partial tiles go to P[ks][m][n] (through LDS, so that P is written in whole rows);
// proj_reduce_kernel adds the KS partials in index order, the bias, and rounds.  The reduction is a second launch on
// purpose: folding it into the last workgroup to arrive needs device-scope fences, which on this multi-die part write
// back and invalidate the L2 slices and cost several times the whole projection.
// ---------------------------------------------------------------------------------------------
constexpr int kProjWaves = 8;     // wavefronts per workgroup, 16 output columns each
constexpr int kProjCols = 16 * kProjWaves;
constexpr int kProjThreads = 64 * kProjWaves;
constexpr int kProjPiece = 512;   // k values staged in LDS at a time
constexpr int kProjPitch = kProjPiece + 8;  // LDS row pitch (elements): 16 rows of one 16-byte read fall in 64 distinct banks
constexpr int kProjMaxSplit = 8;

template <int MT>
__global__ void __launch_bounds__(kProjThreads) proj_bf16_partial_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                                int64_t w_pitch, float* __restrict__ part, int32_t m0, int32_t M,
                                                                int32_t N, int32_t K, int32_t Kc) {
    __shared__ __attribute__((aligned(16))) uint16_t sx[16 * MT * kProjPitch];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * kProjCols + 16 * wave;
    const int ks = blockIdx.y;
    const int64_t wrow = min(n0 + r, N - 1);  // rows past N are computed from the last row and never stored
    const uint16_t* pw = w + wrow * w_pitch + g * 8;
    const int rows = min(M - m0, 16 * MT);
    f32x4_t acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    constexpr int kItems = 16 * MT * (kProjPiece / 8) / kProjThreads;  // 16-byte items of x a thread stages per piece
    for (int k0 = ks * Kc; k0 < (ks + 1) * Kc; k0 += kProjPiece) {
        const int piece = min(kProjPiece, (ks + 1) * Kc - k0);  // a multiple of 32
        const int n_slices = piece / 32;
        // x first, W behind it: loads return in order, so x can go to LDS while the W slices are still in flight and
        // the MFMAs start as the slices arrive
        u32x4_t xs[kItems];
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            const int e = threadIdx.x + i * kProjThreads, row = e / (kProjPiece / 8), c = e % (kProjPiece / 8);
            if (row < rows && 8 * c < piece) xs[i] = *(const u32x4_t*)(x + (int64_t)(m0 + row) * K + k0 + 8 * c);
        }
        bf16x8_t a[16];
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (u < n_slices) a[u] = *(const bf16x8_t*)(pw + k0 + 32 * u);
        __builtin_amdgcn_s_barrier();  // the previous piece's readers are done with sx (their LDS reads fed MFMAs already issued)
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            const int e = threadIdx.x + i * kProjThreads, row = e / (kProjPiece / 8), c = e % (kProjPiece / 8);
            if (row < rows && 8 * c < piece) *(u32x4_t*)(sx + row * kProjPitch + 8 * c) = xs[i];
        }
        // LDS writes landed, then the barrier: a fence here would also wait for the W loads
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            if (u < n_slices) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    // rows past `rows` hold whatever LDS held: they only reach output columns that are never stored
                    const bf16x8_t bx = *(const bf16x8_t*)(sx + (16 * t + r) * kProjPitch + 32 * u + 8 * g);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], bx, acc[t], 0, 0, 0);
                }
            }
        }
    }
    // The partial tile goes through LDS so that P is written in whole rows.  A lane holds batch row r of tile t, output
    // columns 16 wave + 4 g + i of the workgroup's 128.
    constexpr int kTilePitch = kProjCols + 4;  // floats; 16 rows of one 16-byte write fall in 64 distinct banks
    float* tile = (float*)sx;
    __builtin_amdgcn_s_barrier();  // every wavefront's reads of sx have returned (they fed its MFMAs)
#pragma unroll
    for (int t = 0; t < MT; ++t) *(f32x4_t*)(tile + (16 * t + r) * kTilePitch + 16 * wave + 4 * g) = acc[t];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const int nb0 = blockIdx.x * kProjCols;
    const bool vec = (N & 3) == 0;  // then a group of four columns is inside the row and 16-byte aligned in P
    for (int e = threadIdx.x; e < rows * (kProjCols / 4); e += kProjThreads) {
        const int m = e / (kProjCols / 4), c = (e % (kProjCols / 4)) * 4, n = nb0 + c;
        const f32x4_t v = *(const f32x4_t*)(tile + m * kTilePitch + c);
        float* dst = part + ((int64_t)ks * M + m0 + m) * N + n;
        if (vec && n < N) *(f32x4_t*)dst = v;
        else
            for (int i = 0; i < 4; ++i)
                if (n + i < N) dst[i] = v[i];
    }
}

// Up to 16 batch rows: one launch.  A workgroup owns 16 output columns; its eight wavefronts take the 32-wide slices of K
// round-robin (slice c goes to wavefront c % 8), x^T comes straight from L2 (16 rows at most: no staging pays), and the
// eight partial tiles meet in LDS, where they are added in wavefront order.  No partial buffer, no second launch.
__global__ void __launch_bounds__(512) proj_bf16_small_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                              int64_t w_pitch, const uint16_t* __restrict__ bias,
                                                              uint16_t* __restrict__ y, int64_t y_pitch, int32_t M, int32_t N,
                                                              int32_t K) {
    __shared__ float part[8][16][17];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const uint16_t* pw = w + (int64_t)min(n0 + r, N - 1) * w_pitch + g * 8;  // rows past N: computed, never stored
    const uint16_t* px = x + (int64_t)min(r, M - 1) * K + g * 8;             // likewise for batch rows past M
    const int n_slices = K / 32;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = wave; c0 < n_slices; c0 += 8 * 16) {  // sixteen slices of W (and of x) in flight per lane
        bf16x8_t a[16], b[16];
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (c0 + 8 * u < n_slices) a[u] = *(const bf16x8_t*)(pw + (int64_t)(c0 + 8 * u) * 32);
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (c0 + 8 * u < n_slices) b[u] = *(const bf16x8_t*)(px + (int64_t)(c0 + 8 * u) * 32);
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (c0 + 8 * u < n_slices) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], b[u], acc, 0, 0, 0);
    }
    // the tile a lane holds: batch row r, output columns 4 g + i
#pragma unroll
    for (int i = 0; i < 4; ++i) part[wave][r][4 * g + i] = acc[i];
    __syncthreads();
    if (threadIdx.x < 256) {
        const int m = threadIdx.x >> 4, n = threadIdx.x & 15;
        if (m < M && n0 + n < N) {
            float sum = part[0][m][n];
#pragma unroll
            for (int wv = 1; wv < 8; ++wv) sum += part[wv][m][n];
            if (bias) sum += bf16_bits_to_f32(bias[n0 + n]);
            y[(int64_t)m * y_pitch + n0 + n] = f32_to_bf16_bits(sum);
        }
    }
}

// y[m][n] = round(sum_ks P[ks][m][n] + bias[n]), the partials added in index order.  VEC consecutive outputs per thread
// (4 when N is a multiple of 4, so that a group never straddles two rows).
template <int VEC>
__global__ void __launch_bounds__(256) proj_reduce_kernel(const float* __restrict__ part, const uint16_t* __restrict__ bias,
                                                          uint16_t* __restrict__ y, int64_t y_pitch, int32_t M, int32_t N, int32_t KS) {
    typedef float vec_t __attribute__((ext_vector_type(VEC)));
    const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * VEC;
    const int64_t plane = (int64_t)M * N;
    if (e >= plane) return;
    const int m = (int)(e / N), n = (int)(e - (int64_t)m * N);
    vec_t v[kProjMaxSplit];
#pragma unroll
    for (int s = 0; s < kProjMaxSplit; ++s) v[s] = *(const vec_t*)(part + min(s, KS - 1) * plane + e);  // all loads in flight at once
    vec_t sum = v[0];
#pragma unroll
    for (int s = 1; s < kProjMaxSplit; ++s) sum += s < KS ? v[s] : vec_t(0.f);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
        float f = sum[j];
        if (bias) f += bf16_bits_to_f32(bias[n + j]);
        y[(int64_t)m * y_pitch + n + j] = f32_to_bf16_bits(f);
    }
}

// fp32 operands (the reference's own dtype): one wavefront per output column, lanes stride over k, eight batch rows
// per pass over the row of W.
__global__ void __launch_bounds__(256) proj_f32_kernel(const float* __restrict__ x, const float* __restrict__ w, int64_t w_pitch,
                                                       const float* __restrict__ bias, float* __restrict__ y, int64_t y_pitch,
                                                       int32_t M, int32_t N, int32_t K) {
    const int lane = threadIdx.x & 63;
    const int n = blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (n >= N) return;
    const float* pw = w + (int64_t)n * w_pitch;
    for (int m0 = 0; m0 < M; m0 += 8) {
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int k = lane; k < K; k += 64) {
            const float wk = pw[k];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = fmaf(x[(int64_t)min(m0 + j, M - 1) * K + k], wk, acc[j]);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float v = acc[j];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
            if (lane == 0 && m0 + j < M) y[(int64_t)(m0 + j) * y_pitch + n] = bias ? v + bias[n] : v;
        }
    }
}

// How the contexts are cut, and how long the splits of a ragged batch are that no other rule takes: of the ragged batches quoted here those of one to sixteen rounds of up to
// 64 rows are cut into a round instead (plan_round), large ones into ranges (plan_ranges); `chunk` then says which of them, and what a split need not be shorter than.  Every work item pays a fixed cost (locating itself, loading Q, merging four wavefronts, writing a
// partial) and every split is one more row to merge, so splits are as long as they can be while the launch still spreads evenly
// over the chip.  P = B * Hkv rows, counted with the host's upper bound of the lengths; rows `bytes` long per key.
//   whole rows, written to the output directly, where nearly every CU gets one and they are short: 32 rows of 100 to 700 keys of 8 kv
//     heads, bf16: 16.5 us in splits of 256, 13.8 whole; 12 x 16 rows of 1579 keys, Q8_0: 27.1 and 21.8.
//     Not where the rows leave the second to fourth round less than 9/10 full and one is more than 256 KB: 11 x 32 rows of 3426 keys, fp32:
//     259 us whole, 213 in halves; 26 x 16 of up to 1646, bf16: 47.3 whole, 44.0 in splits of 512; 10 x 32 of 306 keys: 16.9 either way.
//   uniform: one round of a workgroup per CU where that many parts fill 85/100 of the chip (four wavefronts keep enough of HBM in
//     flight: 16 x 16k keys of 8 kv heads, bf16, 189 us in splits of 1024, 174 in halves; 14 x 8 rows of 3540 keys, Q8_0: 30.5 in
//     halves, 34.9 in eighths; 4 x 16 rows of 14765, Q8_0: 49.6 in quarters, 52.5 in eighths), up to 24576 keys a part where a key is
//     less than 256 bytes (16 x 8 rows, Q8_0, in halves and in quarters: of 28k 168.4 and 173.4 us, 36k 212 and 218, 44k 264.5 and
//     265.4, 52k 308.5 and 308.3, 64k 387.8 and 379.5; D 64, bf16, 64k 362.6 and 353).  Else as few as make 9/10 of whole rounds
//     of `slots` workgroups, two per CU for keys of less than 256 bytes (Q8_0, D 64).
//   ragged: up to 1024 keys of D 128 (512 in fp32, in proportion for D 64): 8 rows of 1k to 32k keys, Q8_0: 82 us in splits of
//     8192, 60.5 in splits of 1024; 16 rows of 500 to 8000 in fp32: 131 in 1024, 123 in 512.  Shorter, down to 256, where fewer than one
//     item per CU would come of it by the bound and half the length still makes one round, by the 3/2 below (4 rows of up to 4000 keys,
//     bf16: 15.9 us in 1024, 12.7 in 512; 5 x 4 of 200 to 9680: 21.5 and 18.7; but 3 x 4 of 200 to 16106, 272 items of 512 keys: 23.0 and
//     25.5; 4 x 8 of 500 to 6525: 21.6 and 25.0, Q8_0 19.4 and 21.6, but over pages 22.8 in 1024 and 21.1 in 512), or fewer than four a row (32 x 16
//     rows of 100 to 3000, D 64: 46.9 in 2048, 41.4 in 512), and where one to four rounds would end raggedly (16 rows of 500 to 8000, bf16:
//     58.2 in 1024, 53.8 in 512; but 8 rows of up to 30k: 93.6 and 98.5, so only up to 16 splits a row).  Q8_0, whose items cost more beside their stream: up to 8192 keys while eight items per CU remain (5 x 32 rows
//     of up to 49729: 221 us in 1024, 201 in 4096).
//     Several tokens per sequence: a split's partials weigh that many times as much, so 2048 keys where more than eight rounds come of
//     it (32 x 8 rows of 1k to 32k, bf16, four tokens: 467 us, 475 in 1024, 471 in 4096; 24 x 8 of 5k to 30k, fp32: 692 and 731 in 512) or
//     half as many rounds as in 1024 (10 x 8 of 500 to 6525: 39.5 and 42.9, 42.6 in 512, fp32 68.1 and 83.5; 12 x 8 of 300 to 7452, two
//     tokens: 43.7 and 49.1 in 512; 8 x 8 of 2k to 20k: 85.5 and 92.5; but 14 x 8 of 500 to 7621, two rounds and three: 70.6 and 61.4).
//     A little over a round of 1024 is cut to 512 instead, all the more over pages, whose table is one more latency per group of keys
//     (7 x 8 of 500 to 6525: 36.0 paged, 41.1 in 1024, 42.0 in 2048; not paged 36.8, 41.5, 36.7).  A ragged batch has about two thirds
//     of the items its longest row would make of it: up to 3/2 per CU are a round.
// The partials of a ragged plan for one token are kept to what vsp_attn_decode_noalloc has room for (it takes one token; its results
// are vsp_attn_decode's, bit for bit).
struct DecodePlan {
    int chunk, uniform_splits, max_splits;
};
DecodePlan plan_decode(int format, int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t T, int64_t max_len, bool device_lens,
                       bool paged, size_t partials_limit) {
    if (max_len <= 0) return DecodePlan{kMinChunk, 0, 1};
    const int64_t cus = device_cu_count(), P = B * Hkv, most = ceil_div(max_len, kMinChunk);
    const int64_t bytes = D * (format == VSP_KV_F32 ? 4 : format == VSP_KV_BF16 ? 2 : 1), slots = bytes >= 256 ? cus : 2 * cus;
    const bool fair = P <= cus || P >= 4 * cus || P * 10 >= round_up(P, cus) * 9 || max_len * bytes <= 256 * 1024;
    if (P * 4 >= cus * 3 && max_len <= 4096 && fair) return DecodePlan{(int)round_up(max_len, kGroup), 0, 1};
    const int64_t one = std::min(cus / P, most);  // parts per row that make one round of a workgroup per CU
    int64_t even = one > 0 && P * one * 100 >= cus * 85 && (bytes >= 256 || max_len <= one * 24576) ? one : 0;
    for (int64_t n = 1; n <= most && !even; ++n)
        if (P * n * 10 >= slots * 9 && P * n * 10 >= round_up(P * n, cus) * 9) even = n;
    const int64_t even_chunk = even ? std::max<int64_t>(round_up(ceil_div(max_len, even), kGroup), kMinChunk) : 0;
    if (even && !device_lens) return DecodePlan{(int)even_chunk, 0, (int)ceil_div(max_len, even_chunk)};
    int64_t chunk = (format == VSP_KV_F32 ? 512 : 1024) * 128 / D;
    auto items_of = [&](int64_t keys) { return P * ceil_div(max_len, keys); };
    const bool whole_round = !(paged && format == VSP_KV_Q8_0);
    while (chunk > kMinChunk && ((items_of(chunk) < cus && !(whole_round && 2 * items_of(chunk / 2) >= 3 * cus)) || ceil_div(max_len, chunk) < 4)) chunk >>= 1;
    const int64_t items = items_of(chunk);
    if (bytes >= 256 && chunk > 512 && items > 2 * cus && items < 8 * cus && ceil_div(max_len, chunk) <= 16) chunk = 512;
    while (format == VSP_KV_Q8_0 && chunk < 8192 && P * ceil_div(max_len, 2 * chunk) >= 8 * cus) chunk <<= 1;
    if (T > 1 && bytes >= 256) {
        auto rounds = [&](int64_t keys) {
            const int64_t n = items_of(keys);
            return n <= cus * 3 / 2 ? 1 : n <= cus * 5 / 2 ? 2 : n <= cus * 9 / 2 ? 3 : 4;
        };
        const int64_t n = items_of(1024);
        if (chunk == 1024 && rounds(1024) > 1 && n * 4 <= cus * 7 && ceil_div(max_len, 1024) <= 16) chunk = 512;
        else if (items_of(2048) > 8 * cus || (2 * rounds(2048) <= rounds(1024) && !(paged && n <= 2 * cus))) chunk = 2048;
    }
    while (T == 1 && chunk < 8192 && (size_t)(B * Hq * ceil_div(max_len, chunk) * (D + 2) * 4) > partials_limit) chunk <<= 1;
    const int64_t splits = ceil_div(max_len, chunk);
    if (even_chunk == chunk) even = 0;
    return DecodePlan{(int)chunk, (int)even, (int)std::max(splits, even)};
}

// Workgroups of the RANGE kernels for a batch whose lengths are on the device, two per CU (what their registers leave room for), or 0: where (and a round does not come before
// them, as it does in many of the batches quoted here, round_before_ranges)
// the longest batch the host allows for is 22 groups of 64 keys a workgroup (28 of bf16 keys at D 128).  Below that the splits' shorter chains
// win (8 x 8 rows of 500 to 6525 bf16 keys, D 128, 10 groups: 32.4 us in splits, 37.6 in ranges; 12 x 8 of 300 to 7452, two tokens, 20 groups: 48.5 and
// 52.3).  Splits and ranges, us a step, keys that no cache holds: bf16, 32 x 8 rows of 1k to 32k 448 and 441; 6 x 8 of 1500 to 24000, two tokens, 75.0 and
// 71.5; D 64, 3 x 16 of 640 to 20501 47.1 and 41.1, 21 x 2 of 4871 to 19487 46.5 and 41.2; fp32, 16 x 8 of 500 to 8000 129 and 125, 20 x 2 of 8000 to 30000,
// D 64, 97 and 90, 6 x 8 of 1000 to 20000, two tokens, 156 and 108.  One workgroup per CU: 32 x 32 of 100 to 3000 219 us for 186; four: 32 x 8 of 1k
// to 32k 448 for 437.  The bound says how large the batch may be, not how large it is: splits and ranges (or the parts that RangeWalk makes of them)
// under bounds of 2, 4 and 8 times the longest row, times those at 1: 8 x 8 of 500 to 6525 (30.9 us) 34.6 34.6, 33.1 34.6, 35.7 34.8; 12 x 8 of 300 to 7452, two
// tokens (46.9), 52.3 50.0, 52.3 50.0, 49.0 48.8; 12 x 8 of 1000 to 4000, n_rep 8, (42.3) 40.6 40.6, 41.9 37.2, 45.8 37.3; 32 x 8 of 100 to 2000 (41.6) 41.7 41.7, 47.2
// 44.3, 48.1 45.0; 5 x 8 of 200 to 12000, four tokens, (36.0) 35.9 35.8, 35.9 36.7, 38.7 36.4; fp32, 7 x 4 of 500 to 6525, two tokens, (31.5) 32.0 32.0, 60.2 60.2, 60.7
// 33.8; D 64, 64 x 2 of 100 to 4000 (27.2) 25.8 27.4, -, 27.9 27.7; 48 x 2 of 100 to 6000 over pages (31.3) 29.6 30.1, -, 30.5 30.3.  33 batches under these
// bounds, splits / ranges: 1.08 (0.91 to 1.8).  Rows of one length keep their even parts (bf16 16 x 8 of 16384: 192 either way; as ranges 187 for 184).
// Not (has_ranges) for Q8_0 (ragged batches gain 2 to 10 %, but even ones, 8 x 8 of 64000, lose 3 to 6: the kernel's stream itself is slower inside
// the loop over pieces) nor for pages at D 128 (16 x 8 of 500 to 8000 72.6 and 75.5; 32 x 8 of 8000 188 and 195).
constexpr bool has_ranges(int format, int64_t D, bool paged) { return format != VSP_KV_Q8_0 && !(paged && D == 128); }
constexpr int range_line(int format, int64_t D) { return D == 128 && format == VSP_KV_BF16 ? 28 : 22; }
int plan_ranges(int format, int64_t B, int64_t Hkv, int64_t D, int64_t max_len, bool paged, int uniform_splits) {
    const int64_t wgs = 2 * (int64_t)device_cu_count(), groups = B * Hkv * ceil_div(max_len, kGroup);
    if (!has_ranges(format, D, paged) || B > kRangeRows || groups > INT32_MAX / 2) return 0;
    if (groups < wgs * range_line(format, D)) return 0;
    const int64_t n = std::max(wgs, B * Hkv * uniform_splits);
    // two slots a workgroup in the workspace that is documented for splits of 256 keys
    return 2 * n <= B * Hkv * ceil_div(max_len, 256) ? (int)n : 0;
}

// How many splits of a kv head's rows a ragged batch makes at most (items 0: the plan's splits as they are): where the bound of the lengths makes between one and sixteen rounds of
// those, one round of a workgroup per CU (two for keys of 64 bytes).  Every row's last split is a short one, so that one round of many rows' splits may be much longer than half of one
// of twice as many: with more than 2/5 as many rows as splits, whichever the lengths make better, two rounds from 2.2 times the length on (or_two).  Us a step, the plan's splits and one round,
// counted where counted_round allows it: bf16, 8 x 8 rows of 500 to 8000, four tokens, over
// pages 43.9 and 38.2, 9 x 8 of 1612 to 6451 45.2 and 38.4, D 64, 27 x 2 of 1780 to 7122 29.9 and 24.5; Q8_0, 6 x 4 of 13592 to 54370 63.2 and 50, 4 x 8
// of 6946 to 27785 53.2 and 40.4, 6 x 8 of 12662 to 50648 97 and 88, 12 x 8 of 1143 to 36580 112 and 104.
// More rows, the plan's splits, one round, two: bf16, four tokens, 22 x 8 of 864 to 3458 71 56 71; Q8_0, 14 x 8 of 136 to 4378 35.6 29.6 34.5, 11 x 16 of 202 to 6482, pages, 53 66 45,
// 23 x 8 of 302 to 9681 78 96 73; fp32, 16 heads, 11 rows of 612 to 2449 64 66 60.  113 drawn batches of these: 0.965 of the time (always two rounds 0.971), at most 1.04.
// One workgroup per CU of 64-byte keys: 28 x 2 of 12754 to 51018 68 and 75.
// Two rounds of the plan's splits and fewer: only from 140 KB of K a CU on, 200 where two lengths are searched for (or_two: 19 x 8 rows of 34 to 621 fp32 keys, 190 KB, 12.5 and 13.3; six drawn
// batches of 140 to 200 KB 0.97 of the speed of the plan's splits, 75 of 140 to 240 KB with one length 1.05); below, the search costs what it saves (10 x 16 rows of 131 to 527 Q8_0 keys 13.1 and 14.2, 20 x 8 of 139 to 557 15.5 and
// 16.6, bf16, 20 x 8 of 662, four tokens, 23.8 and 25.0; above, 23 x 4 of 906 to 3627, Q8_0, pages, 34.9 and 29.0, fp32, 15 x 4 of 118 to 3784 41.3 and 33.9).
Round plan_round(int format, int64_t B, int64_t Hkv, int64_t D, int64_t max_len, const DecodePlan& p) {
    const int64_t bytes = D * (format == VSP_KV_F32 ? 4 : format == VSP_KV_BF16 ? 2 : 1);
    const int64_t items = (bytes > 64 ? 1 : 2) * (int64_t)device_cu_count() / Hkv, n = B * ceil_div(max_len, p.chunk);
    const bool or_two = 5 * B > 2 * items;
    const bool worth = n * Hkv > 2 * (int64_t)device_cu_count() || B * Hkv * max_len * bytes >= (or_two ? 200 : 140) * 1024 * (int64_t)device_cu_count();
    return B <= 64 && 5 * B <= 4 * items && n > items && n <= 16 * items && worth ? Round{(int)items, or_two, (int)(device_cu_count() / Hkv)} : Round{};
}
// A round's partials are merged by the last workgroup to leave them where a row has few, whatever the lengths are: one long row among short ones makes all of
// a round's splits (most), and one workgroup then merges them one after the other.  One row of 30000 keys among short ones, merged by a launch of its own and by the
// last workgroup: fp32, 12 x 2 heads, four columns, 128 splits 16.8 us and 15.8; bf16, 8 kv heads, eight columns, 32 splits 23.1 and 22.0, Q8_0, 24 21.0 and 21.7, 49 28.2 and 29.4;
// sixteen columns, bf16, 15 splits 27.2 and 27.9, 18 14.5 and 18.8, Q8_0, 30 20.7 and 24.8, 49 24.2 and 31.7.  So 256 splits times columns, 512 with up to four columns.  Nor where
// few rows make as many splits each as a rule (two rows: 2 x 8 of 4184 to 9000, bf16, eight columns, 15.7 and 17.0; 2 x 8 of 2564 to 5619 12.5 and 13.9; 3 x 8 of 12410 to 49643, Q8_0, 51.7
// and 49.8), nor where rows of about one length would make more workgroups than are resident (11 x 16 of 4461, D 64, bf16, quarters: 45.8 and 50.3).
bool counted_round(const Round& r, int64_t B, int64_t Hkv, int64_t columns, int64_t uniform_splits, int64_t max_splits) {
    const int64_t longest = std::min(max_splits, std::max(uniform_splits, r.most())), usual = std::min(max_splits, r.most() / B);
    return B * Hkv * uniform_splits <= 2 * (int64_t)device_cu_count() && longest * columns <= (columns <= 4 ? 512 : 256) && usual * columns <= 96;
}
// Before ranges up to 64 groups of keys a workgroup of theirs, with splits as short as their one round takes whatever the lengths are (max_splits): those of the plan's length leave
// the chip to one long row (fp32, 8 x 4 rows, one of 24000 keys, the others short, four tokens, ranges 31.1 us a step, a round of twelve splits a row 45.6, of any number 27.3).  Us a step, ranges and a
// round: bf16, D 64, 10 x 8 rows of 348 to 11155, two tokens, 31.0 and 28.5, 7 x 8 of 5911 to 23645, pages, 52 and 49, 12 x 8 of 448 to 14366, D 128, 80 and 75.5; fp32, 6 x 12 of 414 to 13268, D 64, 56 and 53.  Two rounds only where the last workgroup merges: in a launch of its own (which searches for the split's length, too) 14 x 8 of 280
// to 8964, bf16, D 64, two tokens, 68 and 71, 15 x 8 of 424 to 1480, four, 11.8 and 13.5, 21 x 8 of 565 to 8739 32.5 and 35.3; one round: 6 x 4 of 4664 to 12000 under a bound of 48000, bf16, four tokens,
// 23.0 and 24.4, but 2 x 8 of 412 to 8662, fp32, 27.1 and 21.2, 8 x 2, one of 50000, bf16, D 64, 26.9 and 18.9.  50 drawn batches of these 1.07 faster than in ranges.  Above 64 groups ranges are as fast
// or up to 4 % faster (bf16, D 64, 22 x 8 of 817 to 26168, four tokens, 134 and 138).
bool round_before_ranges(const Round& r, int64_t B, int64_t Hkv, int64_t columns, int64_t max_len, int64_t uniform_splits, int64_t max_splits) {
    const int64_t resident = 2 * (int64_t)device_cu_count();
    return B * Hkv * ceil_div(max_len, kGroup) < 64 * resident && B * Hkv * uniform_splits <= resident && (!r.or_two || counted_round(r, B, Hkv, columns, uniform_splits, max_splits));
}

// One short length known on the host: up to 16 splits of 128 keys (one pass of two wavefronts over bf16 or Q8_0 keys, of four over fp32)
// while they make at most one workgroup per CU.  A workgroup's time is then what its CU takes to load 128 keys, and the merge of twice as
// many partials costs less than that saves.  A token step in splits of 256 and of 128 keys: 32 / 8 heads, 2047 bf16 keys 9.4 and 8.9 us, Q8_0
// 10.9 and 10.3; 16 / 4 heads, 1200 bf16 keys 8.6 and 7.7; fp32, 32 / 8 heads of 2048 keys 13.3 and 11.2, four rows of 1000 13.9
// and 11.5.  Not for 256 keys (7.4 and 7.6) nor beyond one round (four rows of 2047 bf16 keys: 10.1 and 12.8).
constexpr int kFineChunk = 128, kFineSplits = 16;
// (vsp_attn_decode keeps to splits that its documented workspace has room for.)
bool plan_fine(int64_t B, int64_t Hkv, int64_t max_len) {
    const int64_t splits = ceil_div(max_len, kFineChunk);
    return max_len > 256 && splits <= kFineSplits && B * Hkv * splits <= device_cu_count();
}

// decode_f32_kernel's tokens per split: the scores of a split are in LDS.
int pick_chunk(int format, int64_t B, int64_t Hkv, int64_t max_len, int64_t tokens) {
    const int64_t want = device_cu_count() / 2;
    const int cap = format == VSP_KV_Q8_0 ? 8192 : (tokens > 1 ? 2048 : 1024);
    for (int chunk = cap; chunk > 256; chunk >>= 1) {
        if (B * Hkv * ceil_div(max_len, chunk) >= want) return chunk;
    }
    return 256;
}

}  // namespace

// out[b][h][t][:] from the split-K partials ws_o [B][Hq][T][max_splits][D], ws_ml [..][2] = (m in the log2 domain, l): the
// combine of the decode step, also used by the context-split prefill over a cache.  A row's split count is
// ceil(its length / split_chunk's choice), its length seq_lens[b] (or len) clamped to [0, L_cap].
int launch_split_combine(const float* ws_o, const float* ws_ml, const int32_t* seq_lens, int32_t len, int32_t chunk, int32_t max_splits,
                         int64_t B, int64_t Hq, int64_t T, int64_t D, int32_t L_cap, vsp_tensor* out, hipStream_t st,
                         const CombineExtra& extra) {
    const int esz = out->dtype == VSP_F32 ? 4 : 2;
    const bool rows_aligned = ((uintptr_t)out->data % (4 * esz)) == 0 && out->stride[0] % 4 == 0 && out->stride[1] % 4 == 0 && (T == 1 || out->stride[2] % 4 == 0);
    const int64_t rows = B * Hq * T;
    const CombineArgs a{ws_o, ws_ml, seq_lens, len, chunk, max_splits, (int)Hq, (int)D, L_cap, (int)T, out->data, out->stride[0], out->stride[1], out->stride[2], rows, extra};
    if ((D == 64 || D == 128) && rows_aligned && is_aligned16(ws_o) && ((uintptr_t)ws_ml & 7) == 0) {
        const int threads = rows <= 4096 ? 64 : 256;  // few rows: more, smaller workgroups
        const int64_t wgs = ceil_div(rows, threads / (D / 4));
        if (wgs > INT32_MAX) return VSP_ERR_ARG;
        auto go = [&](auto out_tag, auto d, auto blk) {
            using OutT = decltype(out_tag);
            auto* kernel = extra.round.items > 0 ? split_combine_round_kernel<OutT, decltype(d)::value, decltype(blk)::value> : split_combine_kernel<OutT, decltype(d)::value, decltype(blk)::value>;
            hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(threads), 0, st, a);
        };
        auto pick_blk = [&](auto out_tag, auto d) {  // the smallest block of splits that covers the launch
            if (max_splits <= 4) go(out_tag, d, std::integral_constant<int, 4>{});
            else if (max_splits <= 8) go(out_tag, d, std::integral_constant<int, 8>{});
            else if (max_splits <= 16) go(out_tag, d, std::integral_constant<int, 16>{});
            else go(out_tag, d, std::integral_constant<int, 32>{});
        };
        auto pick_d = [&](auto out_tag) {
            if (D == 128) pick_blk(out_tag, std::integral_constant<int, 128>{});
            else pick_blk(out_tag, std::integral_constant<int, 64>{});
        };
        if (out->dtype == VSP_F32) pick_d(float{});
        else pick_d(uint16_t{});
        return check_launch();
    }
    dim3 cgrid((unsigned)(Hq * T), (unsigned)B);
    const int cthreads = D <= 64 ? 64 : (D <= 128 ? 128 : 256);
    auto combine = [&](auto out_tag, auto blk) {
        using OutT = decltype(out_tag);
        auto* kernel = extra.round.items > 0 ? decode_combine_round_kernel<OutT, decltype(blk)::value> : decode_combine_kernel<OutT, decltype(blk)::value>;
        hipLaunchKernelGGL(kernel, cgrid, dim3(cthreads), 0, st, a);
    };
    auto combine_blk = [&](auto out_tag) {
        if (max_splits <= 8) combine(out_tag, std::integral_constant<int, 8>{});
        else if (max_splits <= 16) combine(out_tag, std::integral_constant<int, 16>{});
        else combine(out_tag, std::integral_constant<int, 32>{});
    };
    if (out->dtype == VSP_F32) combine_blk(float{});
    else combine_blk(uint16_t{});
    return check_launch();
}

}  // namespace vsp

using namespace vsp;

namespace {

// Split-K partials for callers that cannot allocate (vsp_attn_decode_noalloc): one fixed array per GPU, part of
// the library's code object, held until the process ends.  In host code the array's name is only a handle for
// hipGetSymbolAddress; kernels and launches use the per-device address looked up through it.
constexpr size_t kScratchBytes = 32u << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices];  // per device, filled on the first call on that device
std::mutex g_scratch_mutex;

// Address of the current device's copy of `scratch` (each GPU holds its own at its own address).
int scratch_for_current_device(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        set_hip_error(e);
        return VSP_ERR_LAUNCH;
    }
    if (dev < 0 || dev >= kMaxDevices) return VSP_ERR_ARG;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_hip_error(e);
            return VSP_ERR_LAUNCH;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return VSP_OK;
}

// Partials of a call in whole splits.
size_t partials_bytes(int64_t rows, int64_t splits, int64_t D) { return (size_t)(rows * splits * (D + 2) * 4); }

// What a call runs: how its contexts are cut, by which kernels, in how many workgroups, and who merges the partials.
struct DecodeRoute {
    DecodePlan plan;
    int least_splits;    // of pick_chunk, which vsp_attn_decode_noalloc has to have room for
    Round round;         // round.items > 0: the *_round_kernels
    int32_t range_wgs;   // > 0: the RANGE kernels
    int32_t n_cgroups;
    int64_t wgs;         // the grid of the other kernels
    bool counted;        // one launch, with counters for all (sequence, kv head, group of 16 query heads)
};
struct DecodeShape {
    int format;
    bool paged, device_lens, step;
    int64_t B, Hq, Hkv, D, T;
    int32_t max_len;
};
// room: bytes of the caller's workspace (the library's scratch: kScratchBytes); quads: the output's rows take stores of four elements
DecodeRoute route_decode(const DecodeShape& s, size_t room, bool quads) {
    const int64_t cus = device_cu_count(), n_rep = s.Hq / s.Hkv, columns = n_rep * s.T, rows = s.B * s.Hq * s.T;
    const bool wide = s.D == 64 || s.D == 128;
    const bool by_columns = s.format != VSP_KV_F32 || (wide && n_rep <= 16);  // else decode_f32_kernel
    DecodeRoute r{};
    const int old_chunk = s.max_len > 0 ? pick_chunk(s.format, s.B, s.Hkv, s.max_len, s.T) : 256;
    r.least_splits = s.max_len > 0 ? (int)ceil_div(s.max_len, old_chunk) : 1;
    const DecodePlan old_plan{old_chunk, 0, r.least_splits};
    r.plan = by_columns ? plan_decode(s.format, s.B, s.Hq, s.Hkv, s.D, s.T, s.max_len, s.device_lens, s.paged, kScratchBytes) : old_plan;
    if (s.step && n_rep <= 16 && plan_fine(s.B, s.Hkv, s.max_len)) r.plan = DecodePlan{kFineChunk, 0, (int)ceil_div(s.max_len, kFineChunk)};
    // what the library's scratch has room for in longer splits is not refused for a finer plan (hundreds of query heads per kv head)
    if (s.T == 1 && partials_bytes(rows, r.plan.max_splits, s.D) > kScratchBytes && partials_bytes(rows, r.least_splits, s.D) <= kScratchBytes) r.plan = old_plan;
    const DecodePlan& plan = r.plan;
    r.n_cgroups = (s.format != VSP_KV_F32 && n_rep > 16) ? (int)((n_rep + 15) / 16) : 1;
    if (s.device_lens && by_columns && wide && r.n_cgroups == 1 && plan.max_splits > 1) {
        const size_t fits = std::min(room, kScratchBytes);
        r.round = plan_round(s.format, s.B, s.Hkv, s.D, s.max_len, plan);
        if (quads) r.range_wgs = plan_ranges(s.format, s.B, s.Hkv, s.D, s.max_len, s.paged, plan.uniform_splits);
        if (partials_bytes(2 * (int64_t)r.range_wgs * columns, 1, s.D) > fits) r.range_wgs = 0;
        if (r.round.items && r.range_wgs) {
            const int64_t splits = std::max<int64_t>(plan.max_splits, std::min(ceil_div(s.max_len, kMinChunk), r.round.most()));
            if (partials_bytes(rows, splits, s.D) <= fits && round_before_ranges(r.round, s.B, s.Hkv, columns, s.max_len, plan.uniform_splits, splits)) {
                r.range_wgs = 0;
                r.plan.max_splits = (int)splits;
            } else {
                r.round = Round{};
            }
        }
        r.round.max_splits = plan.max_splits;
    }
    // (item, kv head) pairs in the grid: one workgroup per pair and column group (pairs padded to a multiple of 8 when there are groups, see block_coords).
    // A round's splits and its short rows (one at least is not), or equal parts (split_chunk).
    const int64_t items = (int64_t)plan.max_splits * s.B;
    const int64_t pairs = (r.round.items ? std::min(items, std::max(r.round.most() + s.B - 1, s.B * plan.uniform_splits)) : items) * s.Hkv;
    r.wgs = r.n_cgroups > 1 ? round_up(pairs, 8) * r.n_cgroups : pairs;
    // Who merges.  Ranges: a launch of their own (in the same one: 1 to 3 % faster on some ragged batches, 3 to 9 slower on even ones).  Else one launch where no
    // row is split, and where all workgroups are resident at once and few partials meet in the last one: each then waits once for its partials to be visible (about
    // 3 us), under the others' work, and a launch is saved (one sequence, 2048 keys: 9.8 -> 8.7 us; a batch of ten rounds: 446 -> 477).
    const bool rows_fit = columns * plan.max_splits * s.D * 4 <= INT32_MAX;  // byte offsets of 32 bits within a (batch row, kv head)
    if (s.max_len > 0 && by_columns && quads && rows_fit && !r.range_wgs) {
        const int splits = plan.max_splits;
        r.counted = splits == 1 || (splits <= 8 && r.wgs <= 2 * cus)
                    // a token of 3 x 8 heads, 10005 Q8_0 keys, ten splits 22.3 -> 21.2, of 11 x 2 heads, 10837 fp32 keys, eleven 28.8 -> 27.7; 2 x 8, 3400 Q8_0, twelve 12.1 -> 13.2
                    || (splits <= 11 && columns <= 8 && r.wgs <= cus)
                    // a token of 4096 bf16 keys, 128 workgroups: 10.9 -> 10.0; 4000 fp32 keys of 16 heads, 256 workgroups: 10.9 -> 12.0
                    || (splits <= 16 && (2 * r.wgs <= cus || plan.chunk == kFineChunk))
                    || (r.round.items && counted_round(r.round, s.B, s.Hkv, columns, plan.uniform_splits, splits));
    }
    return r;
}

// The rows of a one-launch token step (vsp_attn_token_step): the context is [0, start_pos), the token's position start_pos.
struct StepRows {
    const vsp_tensor* k;
    const vsp_tensor* v;
    const float* table;
    int32_t start_pos;
};

// All decode entry points: validation, split sizing and the launches.  `own_scratch` selects the
// library's fixed per-device array instead of a caller workspace.
int decode_impl(const vsp_tensor* q, const vsp_kv_cache* cache, const int32_t* seq_lens, int32_t max_len, vsp_tensor* out,
                float scale, void* workspace, size_t workspace_bytes, bool own_scratch, void* stream, bool multi = false,
                uint32_t* counters = nullptr, size_t n_counters = 0, const StepRows* step = nullptr) {
    if (!q || !out) return VSP_ERR_NULL;
    int rc = check_kv_cache(cache);
    if (rc != VSP_OK) return rc;
    if (q->ndim != 4 || out->ndim != 4) return VSP_ERR_NDIM;
    const int64_t B = q->shape[0], Hq = q->shape[1], T = q->shape[2], D = q->shape[3];
    if ((multi ? T < 1 : T != 1) || B != cache->B || D != cache->D) return VSP_ERR_SHAPE;
    for (int i = 0; i < 4; ++i)
        if (out->shape[i] != q->shape[i]) return VSP_ERR_SHAPE;
    if (cache->Hkv <= 0 || Hq <= 0 || Hq % cache->Hkv != 0) return VSP_ERR_GQA_HEADS;
    const int n_rep = (int)(Hq / cache->Hkv);
    const int want_dtype = cache->format == VSP_KV_F32 ? VSP_F32 : VSP_BF16;
    if (q->dtype != out->dtype) return VSP_ERR_DTYPE;
    if (q->dtype != want_dtype) return VSP_ERR_UNSUPPORTED;
    // bf16 / Q8_0: the query heads of a kv head ride in the 16 columns of the matrix instructions; more than 16 are
    // served in groups of 16 (one token per sequence; ops::repeat_kv takes any n_rep, src/ops/attention_ops.cpp:92-155)
    if (cache->format == VSP_KV_F32 && D > 256) return VSP_ERR_UNSUPPORTED;
    // several tokens per sequence: they and the query heads of a kv head share the 16 columns of the matrix instructions
    if (T > 1 && (n_rep * T > 16 || (D != 64 && D != 128))) return VSP_ERR_UNSUPPORTED;
    if (B == 0) return VSP_OK;
    if (!q->data || !out->data) return VSP_ERR_NULL;
    if (q->stride[3] != 1 || out->stride[3] != 1) return VSP_ERR_STRIDE;
    const int esz = q->dtype == VSP_F32 ? 4 : 2;
    if (!is_aligned16(q->data) || (q->stride[0] * esz) % 16 || (q->stride[1] * esz) % 16 || (T > 1 && (q->stride[2] * esz) % 16))
        return VSP_ERR_ALIGN;
    if (max_len < 0 || max_len > cache->S_max) return VSP_ERR_ARG;
    // a host-side length above the bound the launch is sized from is a caller error; device-side lengths
    // cannot be read here and are clamped to the bound inside the kernels instead
    if (!seq_lens && max_len > 0 && cache->len > max_len) return VSP_ERR_ARG;
    const int32_t len = step ? step->start_pos : cache->len;  // keys in the cache (host-side length)
    if (max_len == 0) max_len = seq_lens ? cache->S_max : len;
    if (step) max_len = std::max(max_len, 1);  // the token itself
    hipStream_t st = (hipStream_t)stream;

    const bool columns = D == 64 || D == 128;
    const bool f32_columns = cache->format == VSP_KV_F32 && columns && n_rep <= 16;
    const bool out_quads = ((uintptr_t)out->data % (4 * esz)) == 0 && out->stride[0] % 4 == 0 && out->stride[1] % 4 == 0 && (T == 1 || out->stride[2] % 4 == 0);
    const DecodeRoute route = route_decode(DecodeShape{cache->format, cache->page_table != nullptr, seq_lens != nullptr, step != nullptr, B, Hq, cache->Hkv, D, T, max_len},
                                           own_scratch ? kScratchBytes : workspace_bytes, out_quads);
    const DecodePlan plan = route.plan;
    const int chunk = plan.chunk, max_splits = plan.max_splits;
    const size_t need = partials_bytes(B * Hq * T, max_splits, D);
    if (own_scratch) {
        // an empty context writes no partials
        if (max_len > 0 && std::max(need, partials_bytes(B * Hq * T, route.least_splits, D)) > kScratchBytes) return VSP_ERR_WORKSPACE;
        rc = scratch_for_current_device(&workspace);
        if (rc != VSP_OK) return rc;
    } else if (max_len > 0) {
        if (!workspace || workspace_bytes < need) return VSP_ERR_WORKSPACE;
        if (!is_aligned16(workspace)) return VSP_ERR_ALIGN;
    }
    DecodeArgs a;
    a.q = q->data;
    a.sq_b = q->stride[0];
    a.sq_h = q->stride[1];
    a.sq_t = q->stride[2];
    a.T = (int)T;
    a.k = cache->k;
    a.v = cache->v;
    a.k_scale = cache->k_scale;
    a.v_scale = cache->v_scale;
    a.seq_lens = seq_lens;
    a.len = len;
    a.B = (int)B;
    a.Hq = (int)Hq;
    a.Hkv = cache->Hkv;
    a.n_rep = n_rep;
    a.S = cache->page_table ? cache->page_tokens : kv_s_pad(cache->format, cache->S_max);
    a.S_max = cache->S_max;
    a.L_cap = max_len < cache->S_max ? max_len : cache->S_max;
    a.page_table = cache->page_table;
    a.page_tokens = cache->page_tokens;
    a.pages_per_seq = cache->pages_per_seq;
    a.chunk = chunk;
    a.uniform_splits = plan.uniform_splits;
    a.max_splits = max_splits;
    a.scale_log2 = scale * kLog2e;
    a.ws_o = (float*)workspace;
    a.ws_ml = a.ws_o ? a.ws_o + (size_t)B * Hq * T * max_splits * D : nullptr;
    a.n_cgroups = route.n_cgroups;
    a.col0 = 0;
    a.round = route.round;
    a.range_wgs = route.range_wgs;
    a.range_slack = 0;
    const int64_t wgs = route.wgs;
    if (wgs > INT32_MAX) return VSP_ERR_ARG;
    a.n_splits = (int)std::max<int64_t>(ceil_div(std::min(len, a.L_cap), chunk), 1);
    a.direct = !seq_lens && columns && a.n_cgroups == 1 && B <= 65535 && a.n_splits <= 65535 && std::min(len, a.L_cap) == len && (len > 0 || step);
    a.counters = route.counted && (size_t)(B * cache->Hkv * a.n_cgroups) <= n_counters ? counters : nullptr;
    a.out = out->data;
    a.so_b = out->stride[0];
    a.so_h = out->stride[1];
    a.so_t = out->stride[2];
    if (a.range_wgs) {
        a.range_slack = 256 / (int)(D * esz);  // 16 KB of keys (RangeWalk)
        a.ws_ml = a.ws_o + (size_t)2 * a.range_wgs * n_rep * T * D;
    }
    if (step) {
        if (!a.counters && len == 0) return VSP_ERR_UNSUPPORTED;  // no split of an empty context to own the token
        a.new_k = step->k->data;
        a.new_v = step->v->data;
        a.sk_b = step->k->stride[0], a.sk_h = step->k->stride[1];
        a.sv_b = step->v->stride[0], a.sv_h = step->v->stride[1];
        a.table = step->table;
    }
    if (max_len > 0) {
        const dim3 block(256), grid = a.range_wgs ? dim3((unsigned)a.range_wgs) : a.direct ? dim3((unsigned)a.Hkv, (unsigned)a.n_splits, (unsigned)B) : dim3((unsigned)wgs);
        enum Kind { kSplits, kStep, kRanges, kRound };
        // a combination without a kernel is an error, never a call that leaves the output as it was
        auto launch_columns = [&](auto d, auto paged, auto kind) -> int {
            constexpr int DD = decltype(d)::value;
            constexpr bool P = decltype(paged)::value, S = decltype(kind)::value == kStep, R = decltype(kind)::value == kRanges, O = decltype(kind)::value == kRound;
            if (cache->format == VSP_KV_BF16) {
                if constexpr (O) {
                    hipLaunchKernelGGL((decode_bf16_round_kernel<DD, P>), grid, block, 0, st, a);
                    return VSP_OK;
                } else if constexpr (!R || has_ranges(VSP_KV_BF16, DD, P)) {
                    hipLaunchKernelGGL((decode_bf16_kernel<DD, P, S, R>), grid, block, 0, st, a);
                    return VSP_OK;
                }
            } else if (cache->format == VSP_KV_Q8_0) {
                if constexpr (O) {
                    hipLaunchKernelGGL((decode_q8_round_kernel<DD, P>), grid, block, 0, st, a);
                    return VSP_OK;
                } else if constexpr (!R) {
                    hipLaunchKernelGGL((decode_q8_kernel<DD, P, S>), grid, block, 0, st, a);
                    return VSP_OK;
                }
                static_assert(!has_ranges(VSP_KV_Q8_0, DD, P));
            } else if constexpr (!P) {
                auto go = [&](auto few) {
                    if constexpr (O) hipLaunchKernelGGL((decode_f32_mfma_round_kernel<DD, decltype(few)::value>), grid, block, 0, st, a);
                    else hipLaunchKernelGGL((decode_f32_mfma_kernel<DD, S, R, decltype(few)::value>), grid, block, 0, st, a);
                };
                if (n_rep * T <= 4) go(std::true_type{});
                else go(std::false_type{});
                return VSP_OK;
            }
            return VSP_ERR_UNSUPPORTED;
        };
        if (cache->format != VSP_KV_F32 || f32_columns) {
            auto launch_paged = [&](auto paged) {
                auto launch_d = [&](auto kind) {
                    return D == 128 ? launch_columns(std::integral_constant<int, 128>{}, paged, kind) : launch_columns(std::integral_constant<int, 64>{}, paged, kind);
                };
                return step          ? launch_d(std::integral_constant<int, kStep>{})
                       : a.range_wgs ? launch_d(std::integral_constant<int, kRanges>{})
                       : a.round.items ? launch_d(std::integral_constant<int, kRound>{})
                                     : launch_d(std::integral_constant<int, kSplits>{});
            };
            if ((rc = cache->page_table ? launch_paged(std::true_type{}) : launch_paged(std::false_type{})) != VSP_OK) return rc;
        } else {
            // as many query heads of a kv head per workgroup as divide n_rep (up to four: 16 KB of scores each at chunk 1024)
            const int nh = n_rep % 4 == 0 ? 4 : (n_rep % 2 == 0 ? 2 : 1);
            dim3 grid((unsigned)(max_splits * B), (unsigned)(Hq / nh));
            const size_t smem = ((size_t)nh * 256 + (size_t)nh * chunk + 256) * sizeof(float);
            if (nh == 4) hipLaunchKernelGGL((decode_f32_kernel<256, 4>), grid, dim3(256), smem, st, a, (int)D);
            else if (nh == 2) hipLaunchKernelGGL((decode_f32_kernel<256, 2>), grid, dim3(256), smem, st, a, (int)D);
            else hipLaunchKernelGGL((decode_f32_kernel<256, 1>), grid, dim3(256), smem, st, a, (int)D);
        }
        rc = check_launch();
        if (rc != VSP_OK || a.counters) return rc;
        if (a.range_wgs) {
            const dim3 pairs_grid((unsigned)a.Hkv, (unsigned)B, (unsigned)ceil_div(n_rep * T * (D / 4), kCombineQuads));
            if (cache->format == VSP_KV_F32) {
                if (D == 128) hipLaunchKernelGGL((range_combine_kernel<float, 128>), pairs_grid, dim3(kCombineQuads), 0, st, a);
                else hipLaunchKernelGGL((range_combine_kernel<float, 64>), pairs_grid, dim3(kCombineQuads), 0, st, a);
            } else {
                if (D == 128) hipLaunchKernelGGL((range_combine_kernel<uint16_t, 128>), pairs_grid, dim3(kCombineQuads), 0, st, a);
                else hipLaunchKernelGGL((range_combine_kernel<uint16_t, 64>), pairs_grid, dim3(kCombineQuads), 0, st, a);
            }
            return check_launch();
        }
    }
    // with max_len == 0 every row is empty: the combine kernel reads nothing and writes zeros
    CombineExtra extra;
    extra.B = (int)B;
    extra.uniform_splits = plan.uniform_splits;
    extra.round = a.round;
    return launch_split_combine(a.ws_o, a.ws_ml, seq_lens, max_len > 0 ? len : 0, chunk, max_splits, B, Hq, T, D, a.L_cap,
                                out, st, extra);
}

// vsp_attn_decode_proj's workspace: the merged heads x [B][Hq*D] (4 bytes an element whatever the dtype), the
// projection's split-K partials [kProjMaxSplit][B][N] fp32, then the attention step's own partials; each part
// rounded up to 256 bytes.
size_t proj_x_bytes(int64_t B, int64_t Hq, int64_t D) { return (size_t)((B * Hq * D * 4 + 255) / 256 * 256); }
size_t proj_part_bytes(int64_t B, int64_t N) { return (size_t)((kProjMaxSplit * B * N * 4 + 255) / 256 * 256); }

// Equal ranges of K per workgroup row: as many as kProjMaxSplit while each stays a whole number of 32-wide slices.
int proj_split(int64_t K) {
    int ks = kProjMaxSplit;
    while (ks > 1 && K % (32 * ks) != 0) ks >>= 1;
    return ks;
}

}  // namespace

extern "C" {

size_t vsp_attn_decode_workspace_bytes(int32_t B, int32_t Hq, int32_t D, int32_t max_len) {
    if (B <= 0 || Hq <= 0 || D <= 0 || max_len <= 0) return 0;
    const int64_t splits = ceil_div(max_len, 256);
    return (size_t)((int64_t)B * Hq * splits * (D + 2) * 4);
}

int vsp_attn_decode_plan(const vsp_kv_cache* cache, int with_seq_lens, int32_t max_len, int32_t Hq, int32_t T, vsp_decode_plan* plan) {
    if (!cache || !plan) return VSP_ERR_NULL;
    const bool compact = cache->format == VSP_KV_BF16 || cache->format == VSP_KV_Q8_0;
    if ((!compact && cache->format != VSP_KV_F32) || (compact ? cache->D != 64 && cache->D != 128 : cache->D <= 0 || cache->D % 4 != 0)) return VSP_ERR_UNSUPPORTED;
    if (cache->B <= 0 || cache->Hkv <= 0 || Hq <= 0 || Hq % cache->Hkv != 0 || T <= 0) return VSP_ERR_SHAPE;
    if (max_len < 0 || max_len > cache->S_max || (!with_seq_lens && max_len > 0 && cache->len > max_len)) return VSP_ERR_ARG;
    if (cache->format == VSP_KV_F32 && cache->D > 256) return VSP_ERR_UNSUPPORTED;
    if (T > 1 && ((int64_t)Hq / cache->Hkv * T > 16 || (cache->D != 64 && cache->D != 128))) return VSP_ERR_UNSUPPORTED;
    if (max_len == 0) max_len = with_seq_lens ? cache->S_max : cache->len;
    const DecodeRoute r = route_decode(DecodeShape{cache->format, cache->page_table != nullptr, with_seq_lens != 0, false, cache->B, Hq, cache->Hkv, cache->D, T, max_len},
                                       vsp_attn_decode_workspace_bytes(cache->B * T, Hq, cache->D, max_len), true);
    *plan = vsp_decode_plan{r.plan.chunk, r.plan.uniform_splits, r.plan.max_splits, r.range_wgs, r.round.items, r.round.or_two, r.counted, r.range_wgs ? r.range_wgs : r.wgs};
    return VSP_OK;
}

int vsp_attn_decode(const vsp_tensor* q, const vsp_kv_cache* cache, const int32_t* seq_lens, int32_t max_len,
                    vsp_tensor* out, float scale, void* workspace, size_t workspace_bytes, void* stream) {
    return decode_impl(q, cache, seq_lens, max_len, out, scale, workspace, workspace_bytes, false, stream);
}

int vsp_attn_decode_multi(const vsp_tensor* q, const vsp_kv_cache* cache, const int32_t* seq_lens, int32_t max_len,
                          vsp_tensor* out, float scale, void* workspace, size_t workspace_bytes, void* stream) {
    return decode_impl(q, cache, seq_lens, max_len, out, scale, workspace, workspace_bytes, false, stream, true);
}

int vsp_attn_decode_counted(const vsp_tensor* q, const vsp_kv_cache* cache, const int32_t* seq_lens, int32_t max_len,
                            vsp_tensor* out, float scale, void* workspace, size_t workspace_bytes, uint32_t* counters,
                            size_t n_counters, void* stream) {
    if (n_counters && !counters) return VSP_ERR_NULL;
    return decode_impl(q, cache, seq_lens, max_len, out, scale, workspace, workspace_bytes, false, stream, true, counters, n_counters);
}

size_t vsp_attn_token_step_workspace_bytes(int32_t B, int32_t Hq, int32_t D, int32_t start_pos) {
    if (B <= 0 || Hq <= 0 || D <= 0 || start_pos < 0) return 0;
    const int64_t splits = std::max(ceil_div(std::max(start_pos, 1), 256), std::min<int64_t>(ceil_div(start_pos, kFineChunk), kFineSplits));
    return (size_t)((int64_t)B * Hq * splits * (D + 2) * 4);
}

int vsp_attn_token_step(vsp_kv_cache* cache, const vsp_tensor* q, const vsp_tensor* new_k, const vsp_tensor* new_v, const float* rope_table,
                        int64_t table_len, int64_t start_pos, vsp_tensor* out, float scale, void* workspace, size_t workspace_bytes,
                        uint32_t* counters, size_t n_counters, void* stream) {
    if (!q || !new_k || !new_v || !out) return VSP_ERR_NULL;
    int rc = check_kv_cache(cache);
    if (rc != VSP_OK) return rc;
    if (n_counters && !counters) return VSP_ERR_NULL;
    const int want = cache->format == VSP_KV_F32 ? VSP_F32 : VSP_BF16;
    if (q->ndim != 4 || q->shape[2] != 1 || (cache->D != 64 && cache->D != 128) || cache->Hkv <= 0 || (want == VSP_F32 && q->shape[1] > 16 * (int64_t)cache->Hkv)) return VSP_ERR_UNSUPPORTED;
    // the token is the last one of every row and inside the cache (and the table)
    if (start_pos < 0 || start_pos >= cache->S_max || start_pos + 1 < cache->len || (rope_table && start_pos >= table_len)) return VSP_ERR_UNSUPPORTED;
    if (rope_table && !is_aligned16(rope_table)) return VSP_ERR_UNSUPPORTED;
    const int esz = want == VSP_F32 ? 4 : 2;
    for (const vsp_tensor* t : {new_k, new_v}) {
        if (t->ndim != 4 || t->dtype != want || t->shape[0] != cache->B || t->shape[1] != cache->Hkv || t->shape[2] != 1 ||
            t->shape[3] != cache->D || t->stride[3] != 1 || !t->data || !is_aligned16(t->data) || (t->stride[0] * esz) % 16 || (t->stride[1] * esz) % 16)
            return VSP_ERR_UNSUPPORTED;
    }
    const StepRows step{new_k, new_v, rope_table, (int32_t)start_pos};
    vsp_kv_cache context = *cache;  // what the attention reads: the keys before the token
    context.len = (int32_t)start_pos;
    rc = decode_impl(q, &context, nullptr, 0, out, scale, workspace, workspace_bytes, false, stream, true, counters, n_counters, &step);
    if (rc == VSP_OK) cache->len = (int32_t)start_pos + 1;
    return rc;
}

int vsp_attn_decode_noalloc(const vsp_tensor* q, const vsp_kv_cache* cache, const int32_t* seq_lens, int32_t max_len,
                            vsp_tensor* out, float scale, void* stream) {
    return decode_impl(q, cache, seq_lens, max_len, out, scale, nullptr, 0, true, stream);
}

size_t vsp_attn_decode_proj_workspace_bytes(int32_t B, int32_t Hq, int32_t D, int32_t max_len, int32_t N) {
    if (B <= 0 || Hq <= 0 || D <= 0 || N < 0) return 0;
    return proj_x_bytes(B, Hq, D) + proj_part_bytes(B, N) + vsp_attn_decode_workspace_bytes(B, Hq, D, max_len);
}

int vsp_attn_decode_proj(const vsp_tensor* q, const vsp_kv_cache* cache, const int32_t* seq_lens, int32_t max_len,
                         const vsp_tensor* wo, const vsp_tensor* bias, vsp_tensor* y, float scale, void* workspace,
                         size_t workspace_bytes, void* stream) {
    if (!q || !wo || !y) return VSP_ERR_NULL;
    if (q->ndim != 4) return VSP_ERR_NDIM;
    if (wo->ndim != 2 || y->ndim != 3 || (bias && bias->ndim != 1)) return VSP_ERR_NDIM;
    const int64_t B = q->shape[0], Hq = q->shape[1], D = q->shape[3];
    const int64_t K = Hq * D, N = wo->shape[0];
    if (wo->shape[1] != K || y->shape[0] != B || y->shape[1] != 1 || y->shape[2] != N) return VSP_ERR_SHAPE;
    if (bias && bias->shape[0] != N) return VSP_ERR_SHAPE;
    if (wo->dtype != q->dtype || y->dtype != q->dtype || (bias && bias->dtype != q->dtype)) return VSP_ERR_DTYPE;
    if (wo->stride[1] != 1 || y->stride[2] != 1 || (bias && bias->stride[0] != 1)) return VSP_ERR_STRIDE;
    const int esz = q->dtype == VSP_F32 ? 4 : 2;
    if (N > 0 && B > 0) {
        if (!wo->data || !y->data || (bias && !bias->data)) return VSP_ERR_NULL;
        if (!is_aligned16(wo->data) || (wo->stride[0] * esz) % 16) return VSP_ERR_ALIGN;
    }
    if (B <= 0 || Hq <= 0 || D <= 0) {
        // shapes the attention step rejects are reported by it (it launches nothing for them); an empty batch has
        // nothing to project
        vsp_tensor none = *q;
        return decode_impl(q, cache, seq_lens, max_len, &none, scale, workspace, workspace_bytes, false, stream);
    }
    if (B > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return VSP_ERR_ARG;  // the projection kernels index with 32 bits
    // the attention step writes the merged heads x [B][Hq][D] (= [B][K]) to the head of the workspace
    const size_t pb_bytes = proj_part_bytes(B, N);
    const size_t xb = proj_x_bytes(B, Hq, D) + pb_bytes;
    if (!workspace || workspace_bytes < xb) return VSP_ERR_WORKSPACE;
    if (!is_aligned16(workspace)) return VSP_ERR_ALIGN;
    vsp_tensor x = *q;
    x.data = workspace;
    x.stride[0] = K;
    x.stride[1] = D;
    x.stride[2] = D;
    x.stride[3] = 1;
    int rc = decode_impl(q, cache, seq_lens, max_len, &x, scale, (char*)workspace + xb, workspace_bytes - xb, false, stream);
    if (rc != VSP_OK || N == 0) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (q->dtype == VSP_F32) {
        hipLaunchKernelGGL(proj_f32_kernel, dim3((unsigned)ceil_div(N, kWaves)), dim3(256), 0, st, (const float*)x.data,
                           (const float*)wo->data, wo->stride[0], bias ? (const float*)bias->data : nullptr,
                           (float*)y->data, y->stride[0], (int)B, (int)N, (int)K);
    } else {
        // K = Hq * D with D 64 or 128 (the bf16 attention kernels' head sizes): a whole number of 32-wide slices
        if (B <= 16) {
            hipLaunchKernelGGL(proj_bf16_small_kernel, dim3((unsigned)ceil_div(N, 16)), dim3(512), 0, st, (const uint16_t*)x.data,
                               (const uint16_t*)wo->data, wo->stride[0], bias ? (const uint16_t*)bias->data : nullptr,
                               (uint16_t*)y->data, y->stride[0], (int)B, (int)N, (int)K);
            return check_launch();
        }
        const int KS = proj_split(K);
        float* part = (float*)((char*)workspace + proj_x_bytes(B, Hq, D));
        const dim3 grid((unsigned)ceil_div(N, kProjCols), (unsigned)KS);
        const uint16_t* px = (const uint16_t*)x.data;
        const uint16_t* pw = (const uint16_t*)wo->data;
        for (int64_t m0 = 0; m0 < B; m0 += 64) {  // 64 batch rows share a pass over W
            const int64_t rows = B - m0;
            if (rows <= 16)
                hipLaunchKernelGGL(proj_bf16_partial_kernel<1>, grid, dim3(kProjThreads), 0, st, px, pw, wo->stride[0], part, (int)m0, (int)B,
                                   (int)N, (int)K, (int)(K / KS));
            else if (rows <= 32)
                hipLaunchKernelGGL(proj_bf16_partial_kernel<2>, grid, dim3(kProjThreads), 0, st, px, pw, wo->stride[0], part, (int)m0, (int)B,
                                   (int)N, (int)K, (int)(K / KS));
            else
                hipLaunchKernelGGL(proj_bf16_partial_kernel<4>, grid, dim3(kProjThreads), 0, st, px, pw, wo->stride[0], part, (int)m0, (int)B,
                                   (int)N, (int)K, (int)(K / KS));
        }
        rc = check_launch();
        if (rc != VSP_OK) return rc;
        const uint16_t* pbias = bias ? (const uint16_t*)bias->data : nullptr;
        if (N % 4 == 0)
            hipLaunchKernelGGL(proj_reduce_kernel<4>, dim3((unsigned)ceil_div(B * N, 1024)), dim3(256), 0, st, part, pbias,
                               (uint16_t*)y->data, y->stride[0], (int)B, (int)N, KS);
        else
            hipLaunchKernelGGL(proj_reduce_kernel<1>, dim3((unsigned)ceil_div(B * N, 256)), dim3(256), 0, st, part, pbias,
                               (uint16_t*)y->data, y->stride[0], (int)B, (int)N, KS);
    }
    return check_launch();
}

}  // extern "C"
