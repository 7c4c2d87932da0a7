// Causal GQA flash-attention prefill for gfx950.
//
// Replaces flash_attention_hip_dispatch (include/vesper/ops/flash_attention.h:74-78,
// src/ops/hip/flash_attention.hip:305-331) with repeat_kv (src/ops/attention_ops.cpp:30-57) folded
// into the head indexing.  Same mathematics as the reference's CPU forward
// (src/ops/flash_attention.cpp:218-364): online softmax over key tiles, O = acc / l,
// LSE = m + log l; the arithmetic is bf16 MFMA with fp32 accumulation (or fp32 MFMA for fp32 inputs).
//
// Two bf16 kernels share the tiles and the fragment layouts described here; prefill_bf16_pipe_kernel (D = 128,
// further down) reorders the work of a wavefront into a three-stage software pipeline, for long contexts on grids that
// fill the chip, prefill_bf16_kernel serves everything else (plan_prefill).
//
// A workgroup of 4 wavefronts owns 128 consecutive rows of one (batch, kv head) - its query heads' queries, token by token -,
// each wavefront 32 of them.  Key tiles of 32 go from global memory straight into LDS (buffer
// loads with the LDS modifier, a ring of slots, later tiles in flight while the current one is
// consumed, one barrier per tile).  LDS rows are unpadded; 16-byte chunks are XOR-swizzled so that
// both the ds_read_b128 of K and the transposing reads of V are bank-conflict free.  The vector ALU,
// not the matrix pipe, is what these kernels run out of first (vector-ALU work of one wavefront hardly
// overlaps with MFMAs of another wavefront on the same SIMD), so the loops are written to keep VALU
// instructions per MFMA minimal: addresses live in scalar registers, the mask and the rescale are rare
// branches.  Both GEMMs are computed transposed so that the softmax statistics of a query live in one
// lane (and its partner 32 lanes away):
//   S^T[key][q] = K[key][:] . Q^T[:][q]     32x32x16 MFMA, A = K rows from LDS, B = Q^T held in registers
//   O^T[d][q]  += V^T[d][key] . P^T[key][q]  A = V^T read from the row-major V tile with the
//                                            transposing LDS read, B = P^T straight from the S^T registers
// The exponent uses a per-row reference maximum that is only raised (and the accumulators rescaled)
// when the row has outgrown it by a wide margin; the result is mathematically the same
// softmax, without a rescale per tile.  Key tiles entirely above the causal diagonal are skipped;
// the mask is evaluated only on tiles that straddle it.
#include <math.h>

#include <algorithm>
#include <utility>

#include "kv_layout.hpp"
#include "kv_rows.hpp"
#include "vsp_common.hpp"

namespace vsp {
namespace {

struct PrefillArgs {
    const void* q;
    const void* k;
    const void* v;
    void* out;
    float* lse;  // nullable
    int64_t sq[3], sk[3], sv[3], so[3];  // strides of dims 0..2 (elements)
    int64_t sl[3];                       // lse strides dims 0..2
    int32_t B, Hq, Hkv, n_rep, T, L;
    int32_t causal;    // 0: no mask.  At the launch it becomes the grid row from which the lightest tiles come first, where masked (launch_row)
    int32_t n_qtiles;
    // bf16 kernels: query heads whose rows a workgroup mixes (n_rep or 1), and the divisors of a workgroup's number: workgroups of a share of
    // the context, of a row of tiles, (batch, kv head) pairs, kv heads; query heads per row's token
    int32_t pack;
    FastDiv by_share, by_bh, by_bkv, by_kv, by_pack;
    int32_t negate_q;  // scale < 0: flip the sign of Q (exact) and use |scale|
    int32_t s_pad;     // cache-plane mode: padded token capacity of the planes
    const int32_t* seq_lens;  // cache-plane mode: per-batch context lengths (device) or nullptr
    const int32_t* chunk_lens;  // cache-plane mode: per-batch number of valid query rows (device) or nullptr
    const int32_t* page_table;  // cache-plane mode, paged cache: [B][pages_per_seq] page indices (device) or nullptr
    int32_t page_tokens, pages_per_seq;
    float scale_log2;  // |scale| * log2(e) for bf16; scale * log2(e) for fp32
    // split-bf16 kernel (fp32 tensors as hi + lo bf16 terms): k / v above are the hi planes, these the lo planes; q is
    // the caller's fp32 tensor
    const void* k_lo;
    const void* v_lo;
    // cache-plane mode, context split over workgroups (n_splits > 1): split s of a query tile covers key tiles
    // [s * split_tiles, (s + 1) * split_tiles) and writes an unnormalised partial instead of the output, row
    // ((b * Hq + hq) * T + t) * n_splits + s of ws_o [..][D] and ws_ml [..][2] = (m in the log2 domain, l)
    int32_t n_splits, split_tiles;
    float* ws_o;
    float* ws_ml;
    int32_t D_true;  // fp32 kernel: the tensors' head_dim when the kernel's tile is wider (columns past it read as zeros)
    const float* rope_table;  // [positions][D/2][2] = {cos, sin}: row t of Q is rotated at position t first; or nullptr
    int32_t elementwise;  // fp32 kernel: rows are read element by element (any head_dim, any 4-byte aligned pitch)
};

constexpr int kBM = 128;       // queries per workgroup
[[maybe_unused]] constexpr float kRescaleThreshold = 8.0f;

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

__device__ inline uint32_t cvt_pk_bf16(float a, float b) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    f32x2_t v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// Reductions over the two half-waves (lane l and lane l ^ 32 hold the two halves of a query's keys).
// v_permlane32_swap exchanges the upper half of its first operand with the lower half of its second; with a
// copy of x in a second register both halves end up holding (lo[l], hi[l]) pairs: no LDS round trip.
__device__ inline float half_swap_max(float x) {
    float y;
    // two wait states between a vector-ALU write and a permlane swap that reads it
    asm volatile("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "=&v"(y));
    return fmaxf(x, y);
}
__device__ inline float half_swap_sum(float x) { return x + __shfl_xor(x, 32); }

// Transposing LDS read issued through inline asm: the compiler cannot prove that a builtin
// transposing read does not alias an outstanding direct-to-LDS load and would wait for every such
// load before it.  The asm form carries no such wait; tr_wait() below is the matching
// "all my LDS reads have returned" fence, tied to the values by data dependence.
template <int OFFSET_BYTES>
__device__ inline uint2 lds_read_tr16_b64_asm(uint32_t lds_byte_addr) {
    uint2 v;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(lds_byte_addr), "n"(OFFSET_BYTES));
    return v;
}
// `tie` is a value computed just before the point where the wait should sit: without it the compiler is free to
// hoist the wait above independent vector-ALU work, which would expose the LDS latency the early read hides.
__device__ inline void tr_wait(uint32_t& tie, uint2& a0, uint2& a1, uint2& a2, uint2& a3, uint2& a4, uint2& a5, uint2& a6, uint2& a7) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(tie), "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5), "+v"(a6), "+v"(a7));
}
__device__ inline void tr_wait(uint32_t& tie, uint2& a0, uint2& a1, uint2& a2, uint2& a3) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(tie), "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3));
}
// Plain 16-byte LDS read through inline asm, for the same reason; lds_wait<N>() waits until at most N of
// this wave's LDS operations are outstanding (they return in order) and ties the wait to a value.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
template <int OFFSET_BYTES>
__device__ inline u32x4_t lds_read_b128_asm(uint32_t lds_byte_addr) {
    u32x4_t v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(lds_byte_addr), "n"(OFFSET_BYTES));
    return v;
}
__device__ inline void lds_write_b128_asm(uint32_t lds_byte_addr, u32x4_t v) {
    asm volatile("ds_write_b128 %0, %1" ::"v"(lds_byte_addr), "v"(v) : "memory");
}
template <int N>
__device__ inline void lds_wait(u32x4_t& a0) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(a0) : "n"(N));
}
__device__ inline void lds_wait0(uint32_t& tie, u32x4_t& a0, u32x4_t& a1, u32x4_t& a2, u32x4_t& a3) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(tie), "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3));
}
__device__ inline void lds_wait0(uint32_t& tie, u32x4_t& a0, u32x4_t& a1) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(tie), "+v"(a0), "+v"(a1));
}
template <int... I, class F>
__device__ inline void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ inline void static_for(F&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}
__device__ inline uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

[[maybe_unused]] constexpr int kUnit = 32;  // keys per tile (one LDS ring slot)

// A lane's pieces of its row of Q (d = 16 ks + 8 h ..) and, for a prompt whose Q has not been rotated yet, of the table; then, once the
// first tiles are on their way, the operands.  Rotating Q here instead of in the append's launch takes two passes over Q out of a prompt
// (most of that launch: 8.4 -> 4.0 us at 777 tokens of 32 / 8 heads, D 128).  A prompt, us in all, rotated there -> here: 777 tokens 25.3 -> 21.2,
// 1500 42.4 -> 38.0, 4 x 2000 180 -> 165, 8000 519 -> 500; D 64, 2 x 16 heads, 777 18.9 -> 15.7.  With every lane rotating its operands' pieces
// in the key-group shapes too (G times the work, 32 rows touched per load) 777 tokens took 23.5 and 1500 took 46.
__device__ inline uint4 rotate8(uint4 w, const float4* cs) {
    float x[8];
    load8<uint16_t>((const uint16_t*)&w, x);
    rope_pairs<8>(x, cs);
    return uint4{cvt_pk_bf16(x[0], x[1]), cvt_pk_bf16(x[2], x[3]), cvt_pk_bf16(x[4], x[5]), cvt_pk_bf16(x[6], x[7])};
}
template <int D, bool ROPE>
__device__ inline void load_q_rows(const PrefillArgs& a, const uint16_t* Qrow, int pos, int h, uint4 (&raw)[D / 16], float4 (&pairs)[D / 16][2]) {
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) raw[ks] = *(const uint4*)(Qrow + 16 * ks + 8 * h);
    if constexpr (ROPE) {
        const float4* t = (const float4*)((const float2*)a.rope_table + (int64_t)pos * (D / 2) + 4 * h);
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) pairs[ks][0] = t[4 * ks], pairs[ks][1] = t[4 * ks + 1];
    }
}
template <int D, bool ROPE>
__device__ inline void finish_q_rows(const PrefillArgs& a, const uint4 (&raw)[D / 16], const float4 (&pairs)[D / 16][2], bf16x8_t (&qf)[D / 16]) {
    const uint32_t flip = a.negate_q ? 0x80008000u : 0u;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
        const uint4 w = ROPE ? rotate8(raw[ks], pairs[ks]) : raw[ks];
        qf[ks] = __builtin_bit_cast(bf16x8_t, uint4{w.x ^ flip, w.y ^ flip, w.z ^ flip, w.w ^ flip});
    }
}

// The query tile of the grid's row `from_last` (a row: all heads): the heaviest tiles first, and, where the kernel TURNS, from row a.causal on the lightest
// first (launch_fold; without a mask they weigh the same).  The row rides in a word that every kernel reads anyway: in one of its own it cost short calls 0.2 us.
template <bool TURNS>
__device__ inline int launch_row(const PrefillArgs& a, int from_last) {
    return !TURNS || from_last < a.causal ? a.n_qtiles - 1 - from_last : from_last - a.causal;
}

// A workgroup's rows are those of one kv head: its n_rep query heads' queries, token by token (row = token * n_rep + head), so that a block of 128 rows
// spans 128 / n_rep tokens.  Every head of the group reads the same keys, whatever its rows' order; tokens that lie closer together end closer to
// one another under the causal mask (a wavefront of 32 queries of one head idles through the tiles that only the later wavefronts' queries see, 1.5 of a
// workgroup's tiles on average, and through half of the last query block), and a chunk of a few tokens fills a workgroup with its group's heads.
struct GroupRow {
    int token, head;
    int64_t offset;   // from the group's first head's first row of Q, elements
};
__device__ inline GroupRow group_row(const PrefillArgs& a, int i) {
    const uint32_t r = (uint32_t)min(i, a.T * a.pack - 1), t = a.by_pack.div(r), head = a.by_pack.mod(r, t);
    return {(int)t, (int)head, (int64_t)head * a.sq[1] + (int64_t)t * a.sq[2]};
}

// A wavefront's 32 finished rows to the output, whole rows at a time.  As the accumulators lie, a lane has 8 bytes of its own row for each store instruction and
// the wavefront touches 32 rows with every one: 16 such instructions per wavefront took 1.7 us of a workgroup at D 128.  Through a patch of 32 x D bf16 of LDS (16-byte chunks
// permuted by the row: no bank conflicts either way) a store instruction covers 512 / D rows.  The patch belongs to the wavefront and no fetch is on its way to it.
template <int D>
__device__ inline void store_rows(const PrefillArgs& a, uint16_t* patch, const f32x16_t (&acc)[D / 32], float inv_l, int b, int h0, int q0, int lane) {
    constexpr int CPR = D / 8, RPI = 64 / CPR;   // chunks per row, rows per instruction
    const int ql = lane & 31, h = lane >> 5;
#pragma unroll
    for (int c = 0; c < CPR; ++c) {
        const f32x16_t& x = acc[c >> 2];
        const int v = 4 * (c & 3);
        *(uint2*)((char*)patch + ql * 2 * D + ((c ^ (ql % CPR)) << 4) + 8 * h) =
            uint2{cvt_pk_bf16(x[v] * inv_l, x[v + 1] * inv_l), cvt_pk_bf16(x[v + 2] * inv_l, x[v + 3] * inv_l)};  // round-to-nearest-even
    }
    const int rows = a.T * a.pack, c = lane % CPR;
    uint16_t* out = (uint16_t*)a.out + (int64_t)b * a.so[0] + (int64_t)h0 * a.so[1] + 8 * c;
#pragma unroll
    for (int i = 0; i < 32 / RPI; ++i) {
        const int r = RPI * i + lane / CPR;
        const uint4 w = *(const uint4*)((const char*)patch + r * 2 * D + ((c ^ (r % CPR)) << 4));
        const uint32_t row = (uint32_t)(q0 + r), t = a.by_pack.div(row), head = a.by_pack.mod(row, t);
        if (q0 + r < rows) *(uint4*)(out + (int64_t)head * a.so[1] + (int64_t)t * a.so[2]) = w;
    }
}

// VBLK: K and V are the planes of a bf16 KV cache (K row-major, V token-blocked by 8) instead of dense
// tensors, and the context length may come per batch row from a device array.  With 8 tokens of one d
// contiguous, a V^T operand is a plain 16-byte LDS read (no transposing read, no swizzle); to make the
// softmax registers line up with those 8 consecutive tokens, lane i of the K operand holds key
// (i with bits 2 and 3 swapped) of the tile.
// R x G wavefronts: R row groups of 32 queries (the workgroup's 32 R consecutive queries) times G key groups: key group g
// takes the key tiles g, g + G, ... and the G partial results (m, l, O^T) of a row group are merged through LDS at the end.
// R = 4, G = 1 is the shape for full grids; the others are for grids that leave the chip idle (a short prompt), where the
// time is the chain of the longest workgroup: fewer queries per workgroup make more workgroups, and G key groups cut the
// chain by G.  With R = 1 a tile belongs to one wavefront: no barrier in the loop, one K and one V slot, the next K
// tile requested when this one's scores are done, the next V tile when this one is consumed.  plan_prefill picks.
// MODE, bits: kSplit: the context may be cut into shares (a.n_splits > 1); kRope: Q is rotated here.
constexpr int kSplit = 1, kRope = 2;
template <int D, bool VBLK, int R, int G, int MODE>
__global__ void __launch_bounds__(64 * R * G, R * G == 4 && G == 1 ? 3 : 2) prefill_bf16_kernel(PrefillArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    constexpr bool SPLIT = (MODE & kSplit) != 0, ROPE = (MODE & kRope) != 0;
    constexpr int KS = D / 16;
    constexpr int DB = D / 32;
    constexpr int CPR = D / 8;
    constexpr int RP = 256 / (2 * D);
    constexpr int NR = 1024 / (2 * D);
    constexpr int NGRP = kUnit / NR;
    constexpr int NLD = (NGRP + R - 1) / R;   // load instructions per wavefront and tile operand
    constexpr bool PRIVATE = R == 1;          // a tile has one reader
    constexpr int NS = PRIVATE ? 1 : 2;       // ring slots
    constexpr int BM = 32 * R;                // queries per workgroup
    constexpr int SLOT = kUnit * D;
    constexpr int NKB = kUnit / 32;   // 32-key S^T blocks per tile
    constexpr int NJ = kUnit / 16;    // PV k-steps per tile

    // Ring slots per key group: K0 | K1 | V0 | V1 (one slot: K | V), SLOT elements each.  Every read of them is issued from
    // inline asm with the slot as an immediate offset, so the per-lane read addresses are loop constants.
    __shared__ __attribute__((aligned(1024))) uint16_t smem_all[G * 2 * NS * SLOT];
    constexpr int SLOTB = 2 * SLOT;  // bytes per slot

    // Block order: heaviest row blocks first (causal work grows with the block index).  Within one
    // of them, workgroups are dealt round-robin to the 8 XCDs by the hardware (id % 8); when the
    // number of (batch, kv head) groups is a multiple of 8, all workgroups of a group are given ids
    // of the same residue, so its K/V stays in one XCD's L2 instead of being fetched into all eight: the groups follow one
    // another, and where a workgroup has one head's rows, first each group's first head, then the second ones.
    int bid = blockIdx.x;
    int tile0 = 0;  // first key tile of this workgroup's share of the context (a context split over workgroups)
    int split = 0;
    if (SPLIT && a.n_splits > 1) {
        split = (int)a.by_share.div((uint32_t)bid);
        bid = (int)a.by_share.mod((uint32_t)bid, (uint32_t)split);
        tile0 = split * a.split_tiles;
    }
    const uint32_t from_last = a.by_bh.div((uint32_t)bid), pos = a.by_bh.mod((uint32_t)bid, from_last), rep = a.by_bkv.div(pos), g_kv = a.by_bkv.mod(pos, rep), ub = a.by_kv.div(g_kv);
    const int qt = launch_row<D == 128>(a, (int)from_last), b = (int)ub, kvh = (int)a.by_kv.mod(g_kv, ub), h0 = kvh * a.n_rep + (int)rep;   // h0: the workgroup's first query head
    int L = a.L;
    // cache mode: per-row context length (clamped to the bound a.L) and per-row chunk length n <= T:
    // query t < n sits at absolute position L - n + t; rows t >= n carry no query and their output is unspecified
    const int n_chunk = a.chunk_lens ? min(max(a.chunk_lens[b], 0), a.T) : a.T;
    if (a.seq_lens) L = min(max(a.seq_lens[b], n_chunk), a.L);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = G == 1 ? wave_id : wave_id % R;  // row group
    const int grp_k = G == 1 ? 0 : wave_id / R;       // key group
    uint16_t* smem = smem_all + grp_k * (2 * NS * SLOT);
    const uint32_t lds0 = lds_addr(smem);
    const int ql = lane & 31, h = lane >> 5;
    const int q0 = qt * BM + wave * 32;
    const int off = L - n_chunk;
    // this lane's row: query (token) tq of head hq
    const GroupRow row = group_row(a, q0 + ql);
    const int tq = row.token, hq = h0 + row.head;
    const int t_first = (int)a.by_pack.div((uint32_t)q0);   // of the wavefront's rows

    const uint16_t* Qp = (const uint16_t*)a.q + (int64_t)b * a.sq[0] + (int64_t)h0 * a.sq[1];
    const uint16_t* Kp = (const uint16_t*)a.k + (int64_t)b * a.sk[0] + (int64_t)kvh * a.sk[1];
    const uint16_t* Vp = (const uint16_t*)a.v + (int64_t)b * a.sv[0] + (int64_t)kvh * a.sv[1];

    // With key groups the G wavefronts of a row group hold the same rows of Q: a prompt's are rotated once, a 16-byte piece of a row per
    // thread and pass (whole rows of Q and of the table, where an operand's lanes would read 32 rows a piece at a time), and cross
    // through ring slots that no tile is on its way to yet: row group w through group w's second K slot, or, with one slot
    // each, through group 0's V slot, whose first tile is then requested afterwards.
    constexpr int NP = BM * CPR / 256;
    static_assert(G == 1 || (PRIVATE ? R == 1 : R <= G), "a slot per row group");
    uint16_t* const stage = PRIVATE ? smem_all + NS * SLOT : smem_all + SLOT;
    constexpr int STAGE_PITCH = 2 * NS * SLOT;
    constexpr bool STAGED = G > 1 && ROPE;
    uint4 qraw[KS];
    float4 pairs[KS][2];
    if constexpr (STAGED) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = tid + 256 * i, ch = p % CPR;
            const GroupRow r = group_row(a, qt * BM + p / CPR);
            qraw[i] = *(const uint4*)(Qp + r.offset + 8 * ch);
            const float4* t = (const float4*)((const float2*)a.rope_table + (int64_t)r.token * (D / 2) + 4 * ch);
            pairs[i][0] = t[0], pairs[i][1] = t[1];
        }
    } else {
        load_q_rows<D, ROPE>(a, Qp + row.offset, tq, h, qraw, pairs);
    }
    bf16x8_t qf[KS];  // ROPE: finished behind the request of the first tiles
    if constexpr (!ROPE) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            uint4 w = qraw[ks];
            if (a.negate_q) {
                w.x ^= 0x80008000u;
                w.y ^= 0x80008000u;
                w.z ^= 0x80008000u;
                w.w ^= 0x80008000u;
            }
            qf[ks] = __builtin_bit_cast(bf16x8_t, w);
        }
    }

    const int rows = a.T * a.pack;
    const int wg_qmax = (int)a.by_pack.div((uint32_t)min(qt * BM + BM - 1, rows - 1));
    const int kv_end_wg = a.causal ? min(L, wg_qmax + off + 1) : L;
    int n_tiles = (kv_end_wg + kUnit - 1) / kUnit;  // tiles [tile0, n_tiles)
    if (SPLIT && a.n_splits > 1) n_tiles = min(n_tiles, tile0 + a.split_tiles);
    const int wave_qmax = (int)a.by_pack.div((uint32_t)min(q0 + 31, rows - 1));
    int kv_end_wave = (q0 < rows) ? (a.causal ? min(L, wave_qmax + off + 1) : L) : 0;
    if (SPLIT && a.n_splits > 1) kv_end_wave = min(kv_end_wave, n_tiles * kUnit);  // a share may end in the middle of a step's G tiles

    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
    float m_ref = -INFINITY;
    float l = 0.f;

    // Global -> LDS through buffer loads with the LDS modifier: one wave-wide load fills 1024 contiguous
    // bytes of LDS (lane i -> bytes [16 i, 16 i + 16)), i.e. NR rows; the swizzle is applied by choosing
    // which 16-byte chunk of the global row each lane fetches.  The buffer descriptor is rebuilt per tile on
    // the scalar unit (base = first row of the tile, size = bytes up to the end of the context), so the
    // per-lane offsets are loop constants and rows past the end of the context read as zeros.
    const int ld_row = lane / CPR, ld_pos = lane % CPR;
    uint32_t voffK[NLD], voffV[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int r = NR * (wave + R * i) + ld_row;
        voffK[i] = (VBLK ? (uint32_t)r * (uint32_t)a.sk[2] * 2u : tile_row_offset(r, a.sk[2] * 2, a.L)) + 16u * (uint32_t)(ld_pos ^ ((r / RP) % CPR));
        if constexpr (VBLK) voffV[i] = (uint32_t)(wave + R * i) * 1024u + 16u * (uint32_t)lane;  // the tile is contiguous
        else voffV[i] = tile_row_offset(r, a.sv[2] * 2, a.L) + 16u * (uint32_t)(ld_pos ^ (((r / RP) % (CPR / 4)) << 2));
    }
    const int64_t rowK = a.sk[2] * 2, rowV = a.sv[2] * 2;  // bytes per key row
    auto load_tile = [&](int t, int slot, bool do_k, bool do_v) {
        const int key0 = t * kUnit;
        int rows = L - key0;  // > 0
        const char* kb = (const char*)Kp;
        const char* vb = (const char*)Vp;
        int local = key0, cap = a.s_pad;  // first token of the tile inside its [cap][D] slab
        if constexpr (VBLK) {
            if (a.page_table) {  // paged cache: a tile (32 tokens) never straddles a page (a multiple of 64 tokens)
                const int pg = key0 / a.page_tokens;
                local = key0 - pg * a.page_tokens;
                cap = a.page_tokens;
                const int64_t slab = (int64_t)a.page_table[(int64_t)b * a.pages_per_seq + pg] * a.Hkv + kvh;
                kb = (const char*)a.k + slab * cap * D * 2;
                vb = (const char*)a.v + slab * cap * D * 2;
                rows = min(rows, cap - local);
            }
        }
        __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(kb + (int64_t)local * rowK), 0, (int)((int64_t)rows * rowK), 0x00020000);
        // VBLK: 32 tokens = 4 token blocks = kUnit * D contiguous elements; bound = the rest of this head's slab
        const int64_t v_base = VBLK ? (int64_t)local * D * 2 : (int64_t)key0 * rowV;
        const int64_t v_bytes = VBLK ? ((int64_t)cap - local) * D * 2 : (int64_t)rows * rowV;
        __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(vb + v_base), 0, (int)v_bytes, 0x00020000);
        uint16_t* dstK = smem + slot * SLOT;
        uint16_t* dstV = smem + (NS + slot) * SLOT;
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int grp = wave + R * i;
            if (NGRP % R != 0 && grp >= NGRP) break;
            if (do_k) __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)(dstK + grp * 512), 16, voffK[i], 0, 0, 0);
            if (do_v) __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)(dstV + grp * 512), 16, voffV[i], 0, 0, 0);
        }
    };

    // Loop-constant LDS read addresses (slot 0; the slot is an immediate offset on the instruction).
    const int krow = VBLK ? ((ql & ~12) | ((ql & 4) << 1) | ((ql & 8) >> 1)) : ql;  // tile row this lane's S^T row holds
    const int kswz = (krow / RP) % CPR;
    uint32_t kaddr[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kaddr[ks] = lds0 + 2u * (uint32_t)(krow * D + 8 * ((2 * ks + h) ^ kswz));
    const int i16 = lane & 15;
    const int vswz = ((i16 >> 2) / RP) % (CPR / 4);
    const int v_lane_off = (4 * h + (i16 >> 2)) * D + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    uint32_t va[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
        va[db] = VBLK ? lds0 + 16u * (uint32_t)(h * D + ql) : lds0 + 2u * (uint32_t)v_lane_off + 64u * (uint32_t)(db ^ vswz);

    constexpr int PF = 4;  // K fragments in flight

    // one wavefront per tile: the V slot is free, the next tile's V may come (behind its K in the queue)
    auto next_v = [&](int tile) {
        if constexpr (PRIVATE) {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
            if (tile + G < n_tiles) load_tile(tile + G, 0, false, true);
        }
    };

    auto tile_step = [&](int t, auto slot_c) {
        constexpr int slot = decltype(slot_c)::value;
        constexpr int KOFF = slot * SLOTB;
        constexpr int VOFF = (NS + slot) * SLOTB;
        const int tile = G == 1 ? t : t * G + tile0 + grp_k;  // this key group's tile of the step
        if constexpr (PRIVATE) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NLD) : "memory");  // the K tile; the V tile may still be in flight
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (tile + G < n_tiles) load_tile(tile + G, slot ^ 1, true, true);
        }
        const int k0 = tile * kUnit;
        if (k0 >= kv_end_wave) return;

        static_assert(NKB == 1, "one 32-key block per tile");
        f32x16_t s[NKB];
#pragma unroll
        for (int j = 0; j < 16; ++j) s[0][j] = 0.f;
        u32x4_t kf[KS];
        static_for<PF>([&](auto i) { kf[i.value] = lds_read_b128_asm<KOFF>(kaddr[i.value]); });
        static_for<KS>([&](auto i) {
            constexpr int ks = i.value;
            constexpr int issued = (ks + PF < KS) ? ks + PF : KS;
            lds_wait<issued - ks - 1>(kf[ks]);
            s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kf[ks]), qf[ks], s[0], 0, 0, 0);
            if constexpr (ks + PF < KS) kf[ks + PF] = lds_read_b128_asm<KOFF>(kaddr[ks + PF]);
        });
        if constexpr (PRIVATE) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the V tile; every read of the K tile has returned
            if (tile + G < n_tiles) load_tile(tile + G, 0, true, false);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the first V fragments are requested now, so that their LDS latency passes under the softmax
        u32x4_t vcur[DB];
        uint2 tcur[DB][2];
        if constexpr (VBLK) {
            static_for<DB>([&](auto dbc) { vcur[dbc.value] = lds_read_b128_asm<VOFF + 512 * dbc.value>(va[dbc.value]); });
        } else {
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                tcur[db][0] = lds_read_tr16_b64_asm<VOFF>(va[db]);
                tcur[db][1] = lds_read_tr16_b64_asm<VOFF + 8 * D * 2>(va[db]);
            }
        }
        const bool need_mask = (a.causal && k0 + kUnit - 1 > t_first + off) || (k0 + kUnit > L);
        if (need_mask) {
            const int q_abs = tq + off;
            const int lim = a.causal ? min(q_abs, L - 1) : L - 1;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int key = VBLK ? k0 + 16 * (v >> 3) + 8 * h + (v & 7) : k0 + 8 * (v >> 2) + 4 * h + (v & 3);
                if (key > lim) s[0][v] = -INFINITY;
            }
        }
        // P is taken against the row's reference maximum as it stands, and the row sum says whether that reference
        // has fallen behind: below 2^10 no P of the tile exceeds 2^10, far from overflow in the fp32 accumulators.
        // Otherwise (rare on real data; always for the first tile, which has no reference yet) the true maximum of
        // these scores becomes the reference, what has been accumulated is rescaled and this tile's P is redone.  The
        // mathematics is the reference's online softmax (src/ops/flash_attention.cpp:309-343) with a reference point
        // that moves only when it has to, which takes the per-tile row maximum (16 max + a cross-half exchange) out of
        // the steady state.  The row sum is taken from the rounded bf16 P (packed dot product against (1, 1)): exactly
        // what the PV MFMAs accumulate.
        uint32_t pw[NJ][4];
        float lsum = 0.f;
        auto softmax = [&](float neg_m) {
            lsum = 0.f;
#pragma unroll
            for (int v = 0; v < 16; v += 2) {
                const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[0][v], a.scale_log2, neg_m));
                const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[0][v + 1], a.scale_log2, neg_m));
                const uint32_t pk = cvt_pk_bf16(p0, p1);
                pw[v >> 3][(v & 7) >> 1] = pk;
                lsum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pk), __builtin_bit_cast(bf16x2_t, 0x3f803f80u), lsum, false);
            }
        };
        const bool first = t == (G == 1 ? tile0 : 0);
        if (!first) softmax(m_ref == -INFINITY ? 0.f : -m_ref);
        if (first || __any(!(lsum < 1024.f))) {
            float mx = s[0][0];
#pragma unroll
            for (int v = 0; v < 16; ++v) mx = fmaxf(mx, s[0][v]);
            mx = half_swap_max(mx) * a.scale_log2;
            const float m_new = fmaxf(m_ref, mx);
            const float alpha = (m_new == -INFINITY || m_ref == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(m_ref - m_new);
            l *= alpha;
#pragma unroll
            for (int i = 0; i < DB; ++i)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[i][j] *= alpha;
            m_ref = m_new;
            softmax(m_ref == -INFINITY ? 0.f : -m_ref);
        }
        l += lsum;
        // PV
        if constexpr (VBLK) {
            u32x4_t vnext[DB];
            const bool tail = k0 + kUnit > L;  // the planes hold stale tokens past L: P is 0 there, V must not be NaN
            static_for<NJ>([&](auto jc) {
                constexpr int j = jc.value;
                if constexpr (DB == 4) lds_wait0(pw[j][3], vcur[0], vcur[1], vcur[2], vcur[3]);
                else lds_wait0(pw[j][3], vcur[0], vcur[1]);
                if constexpr (j + 1 < NJ)
                    static_for<DB>([&](auto dbc) {
                        vnext[dbc.value] = lds_read_b128_asm<VOFF + (2 * (j + 1) * D + 32 * dbc.value) * 16>(va[dbc.value]);
                    });
                if (tail) {
                    const int nvalid = L - (k0 + 16 * j + 8 * h);  // slots e >= nvalid are past the context
#pragma unroll
                    for (int db = 0; db < DB; ++db)
#pragma unroll
                        for (int w = 0; w < 4; ++w) {
                            uint32_t x = vcur[db][w];
                            if (2 * w + 1 >= nvalid) x &= 0x0000ffffu;
                            if (2 * w >= nvalid) x = 0;
                            vcur[db][w] = x;
                        }
                }
                const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, uint4{pw[j][0], pw[j][1], pw[j][2], pw[j][3]});
#pragma unroll
                for (int db = 0; db < DB; ++db)
                    acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vcur[db]), pf, acc[db], 0, 0, 0);
                if constexpr (j + 1 < NJ) {
#pragma unroll
                    for (int db = 0; db < DB; ++db) vcur[db] = vnext[db];
                }
            });
            next_v(tile);
            return;
        }
        uint2 tnext[DB][2];
        static_for<NJ>([&](auto jc) {
            constexpr int j = jc.value;
            if constexpr (DB == 4) tr_wait(pw[j][3], tcur[0][0], tcur[0][1], tcur[1][0], tcur[1][1], tcur[2][0], tcur[2][1], tcur[3][0], tcur[3][1]);
            else tr_wait(pw[j][3], tcur[0][0], tcur[0][1], tcur[1][0], tcur[1][1]);
            if constexpr (j + 1 < NJ) {
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    tnext[db][0] = lds_read_tr16_b64_asm<VOFF + (16 * (j + 1)) * D * 2>(va[db]);
                    tnext[db][1] = lds_read_tr16_b64_asm<VOFF + (16 * (j + 1) + 8) * D * 2>(va[db]);
                }
            }
            const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, uint4{pw[j][0], pw[j][1], pw[j][2], pw[j][3]});
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, uint4{tcur[db][0].x, tcur[db][0].y, tcur[db][1].x, tcur[db][1].y});
                acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, acc[db], 0, 0, 0);
            }
            if constexpr (j + 1 < NJ) {
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    tcur[db][0] = tnext[db][0];
                    tcur[db][1] = tnext[db][1];
                }
            }
        });
        next_v(tile);
    };

    if (tile0 + grp_k < n_tiles) load_tile(tile0 + grp_k, 0, true, !PRIVATE);
    if constexpr (STAGED) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = tid + 256 * i, r = (p / CPR) % 32, ch = p % CPR;
            const uint32_t at = lds_addr(stage + (p / CPR) / 32 * STAGE_PITCH + r * D + 8 * (ch ^ ((r / RP) % CPR)));
            lds_write_b128_asm(at, __builtin_bit_cast(u32x4_t, rotate8(qraw[i], pairs[i])));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        const uint32_t at = lds_addr(stage + wave * STAGE_PITCH);
        const uint32_t flip = a.negate_q ? 0x80008000u : 0u;
        u32x4_t w[KS];
        static_for<KS>([&](auto i) { w[i.value] = lds_read_b128_asm<0>(at + 2u * (uint32_t)(ql * D + 8 * ((2 * i.value + h) ^ ((ql / RP) % CPR)))); });
        static_for<KS>([&](auto i) {
            lds_wait<KS - 1 - i.value>(w[i.value]);
            qf[i.value] = __builtin_bit_cast(bf16x8_t, w[i.value] ^ flip);
        });
        if constexpr (PRIVATE) __builtin_amdgcn_s_barrier();  // every wavefront has its rows: the slot is free
    }
    if constexpr (PRIVATE) {
        __builtin_amdgcn_sched_barrier(0);
        if (tile0 + grp_k < n_tiles) load_tile(tile0 + grp_k, 0, false, true);
    }
    if constexpr (ROPE && !STAGED) finish_q_rows<D, ROPE>(a, qraw, pairs, qf);
    if constexpr (PRIVATE) {
        for (int t = 0; t * G + tile0 + grp_k < n_tiles; ++t) tile_step(t, std::integral_constant<int, 0>{});
    } else {
        // steps of G tiles, the same for every wavefront (they meet at the barriers)
        const int s0 = G == 1 ? tile0 : 0, s1 = G == 1 ? n_tiles : (n_tiles - tile0 + G - 1) / G;
        for (int t = s0; t < s1; t += 2) {
            tile_step(t, std::integral_constant<int, 0>{});
            if (t + 1 < s1) tile_step(t + 1, std::integral_constant<int, 1>{});
        }
    }

    l = half_swap_sum(l);
    const bool there = q0 + ql < rows;
    if constexpr (G > 1) {
        // Merge of the key groups: every wavefront leaves its (m, l) and its O^T registers in LDS as they lie (16-byte
        // quads of four consecutive d, one lane after the other), then takes 1 / G of the quads of its row group,
        // weights the G partials by 2^(m_g - M) and stores its columns.  A wavefront without a visible key has m = -inf,
        // l = 0 and the weight 0.
        constexpr int NQ = DB * 4;    // quads per wavefront
        constexpr int QPW = NQ / G;   // quads each wavefront finishes
        static_assert(NQ % G == 0 && R * G * NQ * 1024 <= G * 2 * NS * SLOT * 2, "the exchange fits the ring");
        __shared__ float sm_m[G][BM], sm_l[G][BM];
        float4* xch = (float4*)smem_all;  // [row group][key group][quad][lane]
        __syncthreads();  // every wavefront is done with the ring
        if (h == 0) {
            sm_m[grp_k][wave * 32 + ql] = l > 0.f ? m_ref : -INFINITY;
            sm_l[grp_k][wave * 32 + ql] = l;
        }
#pragma unroll
        for (int i = 0; i < NQ; ++i)
            xch[((wave * G + grp_k) * NQ + i) * 64 + lane] = float4{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
        __syncthreads();
        float M = -INFINITY;
#pragma unroll
        for (int g = 0; g < G; ++g) M = fmaxf(M, sm_m[g][wave * 32 + ql]);
        const float M_ref = M == -INFINITY ? 0.f : M;
        float f[G], lt = 0.f;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            f[g] = __builtin_amdgcn_exp2f(sm_m[g][wave * 32 + ql] - M_ref);
            lt += f[g] * sm_l[g][wave * 32 + ql];
        }
        if (!there) return;
        if (SPLIT && a.n_splits > 1) {  // the unnormalised partial of this share of the context; the combine kernel finishes the row
            const int64_t part = (((int64_t)b * a.Hq + hq) * a.T + tq) * a.n_splits + split;
#pragma unroll
            for (int i = 0; i < QPW; ++i) {
                const int quad = grp_k * QPW + i;
                float4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const float4 x = xch[((wave * G + g) * NQ + quad) * 64 + lane];
                    o.x += f[g] * x.x, o.y += f[g] * x.y, o.z += f[g] * x.z, o.w += f[g] * x.w;
                }
                *(float4*)(a.ws_o + part * D + 8 * quad + 4 * h) = o;
            }
            if (h == 0 && grp_k == 0) {
                a.ws_ml[part * 2] = M;
                a.ws_ml[part * 2 + 1] = lt;
            }
            return;
        }
        const float inv_l = lt > 0.f ? 1.0f / lt : 0.f;
        uint16_t* op = (uint16_t*)a.out + (int64_t)b * a.so[0] + (int64_t)hq * a.so[1] + (int64_t)tq * a.so[2];
#pragma unroll
        for (int i = 0; i < QPW; ++i) {
            const int quad = grp_k * QPW + i;
            float4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const float4 x = xch[((wave * G + g) * NQ + quad) * 64 + lane];
                o.x += f[g] * x.x, o.y += f[g] * x.y, o.z += f[g] * x.z, o.w += f[g] * x.w;
            }
            uint2 w;
            w.x = cvt_pk_bf16(o.x * inv_l, o.y * inv_l);  // round-to-nearest-even
            w.y = cvt_pk_bf16(o.z * inv_l, o.w * inv_l);
            *(uint2*)(op + 8 * quad + 4 * h) = w;
        }
        if (a.lse && h == 0 && grp_k == 0)
            a.lse[(int64_t)b * a.sl[0] + (int64_t)hq * a.sl[1] + (int64_t)tq * a.sl[2]] = (M + __builtin_amdgcn_logf(lt)) * 0.6931471805599453f;
        return;
    }
    if (SPLIT && a.n_splits > 1) {
        if (there) {
            const int64_t part = (((int64_t)b * a.Hq + hq) * a.T + tq) * a.n_splits + split;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int vq = 0; vq < 4; ++vq)
                    *(float4*)(a.ws_o + part * D + 32 * db + 8 * vq + 4 * h) = float4{acc[db][4 * vq], acc[db][4 * vq + 1], acc[db][4 * vq + 2], acc[db][4 * vq + 3]};
            if (h == 0) {  // a row that met no key in this share says so
                a.ws_ml[part * 2] = l > 0.f ? m_ref : -INFINITY;
                a.ws_ml[part * 2 + 1] = l;
            }
        }
        return;
    }
    if (a.pack == 1 && n_tiles - tile0 <= 4) {  // a call of a few tiles is its latencies: LDS and a barrier are 0.4 us of 4, and some of the wavefronts have no rows
        if (there) {
            const float inv_l = l > 0.f ? 1.0f / l : 0.f;
            uint16_t* op = (uint16_t*)a.out + (int64_t)b * a.so[0] + (int64_t)hq * a.so[1] + (int64_t)tq * a.so[2];
#pragma unroll
            for (int i = 0; i < 4 * DB; ++i)
                *(uint2*)(op + 8 * i + 4 * h) = uint2{cvt_pk_bf16(acc[i >> 2][4 * (i & 3)] * inv_l, acc[i >> 2][4 * (i & 3) + 1] * inv_l),
                                                      cvt_pk_bf16(acc[i >> 2][4 * (i & 3) + 2] * inv_l, acc[i >> 2][4 * (i & 3) + 3] * inv_l)};
            if (a.lse && h == 0) a.lse[(int64_t)b * a.sl[0] + (int64_t)hq * a.sl[1] + (int64_t)tq * a.sl[2]] = (m_ref + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
        }
        return;
    }
    __syncthreads();  // every wavefront has left the ring
    store_rows<D>(a, smem_all + wave_id * SLOT, acc, l > 0.f ? 1.0f / l : 0.f, b, h0, q0, lane);  // an empty context (cache mode, length 0) gives zeros
    if (there && a.lse && h == 0)
        a.lse[(int64_t)b * a.sl[0] + (int64_t)hq * a.sl[1] + (int64_t)tq * a.sl[2]] = (m_ref + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
#endif
}

// ---------------------------------------------------------------------------------------------
// fp32 tensors on the bf16 matrix cores.  Every operand x is split into two bf16 terms, x = hi + lo with hi = bf16(x)
// and lo = bf16(x - hi) (16 significant bits between them), and every product is taken as
//     a b  ~  hi_a hi_b + hi_a lo_b + lo_a hi_b          (fp32 accumulation; the dropped lo_a lo_b is 2^-16 of a b)
// for Q K^T and, with P split the same way after the exponential, for P V.  Three bf16 MFMAs per product at 16 times the
// fp32 MFMA rate, against the reference's fp32 arithmetic (src/ops/flash_attention.cpp:218-364) within its 1e-4 bar
// (observed: below 2e-5 of the output's magnitude).  A pre-pass writes the hi / lo planes of K and V, dense, into a
// caller workspace (Q is split by the wavefront that owns the rows); the attention kernel is prefill_bf16_kernel's
// structure over twice the tiles: R row groups times G key groups (split_row_groups), whose partial results are merged through LDS at the end.
// ---------------------------------------------------------------------------------------------
struct SplitPlan {  // K and V
    const float* src[2];
    uint16_t* hi[2];
    uint16_t* lo[2];
    int64_t s0[2], s1[2], s2[2];  // source strides of dims 0..2 (elements)
    FastDiv by_n, by_h;
    int64_t groups;               // 8-element groups per tensor
    int32_t D;                    // 64 or 128
};

__global__ void __launch_bounds__(256) split_f32_kernel(SplitPlan p) {
    const int t = blockIdx.y;
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (g >= p.groups) return;
    const int shift = p.D == 128 ? 4 : 3, d8 = (int)g & ((1 << shift) - 1);
    const uint32_t row = (uint32_t)(g >> shift), bh = p.by_n.div(row), n = p.by_n.mod(row, bh), b = p.by_h.div(bh), h = p.by_h.mod(bh, b);
    const float* src = p.src[t] + (int64_t)b * p.s0[t] + (int64_t)h * p.s1[t] + (int64_t)n * p.s2[t] + 8 * d8;
    const float4 x0 = *(const float4*)src, x1 = *(const float4*)(src + 4);
    const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    uint32_t hw[4], lw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        hw[i] = cvt_pk_bf16(x[2 * i], x[2 * i + 1]);
        const float r0 = x[2 * i] - __uint_as_float(hw[i] << 16), r1 = x[2 * i + 1] - __uint_as_float(hw[i] & 0xffff0000u);
        lw[i] = cvt_pk_bf16(r0, r1);
    }
    *(uint4*)(p.hi[t] + g * 8) = uint4{hw[0], hw[1], hw[2], hw[3]};
    *(uint4*)(p.lo[t] + g * 8) = uint4{lw[0], lw[1], lw[2], lw[3]};
}

template <int D, int R, int G>
__global__ void __launch_bounds__(256, D * G > 128 ? 1 : 2) prefill_split_kernel(PrefillArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    static_assert(R * G == 4);
    constexpr int KS = D / 16;
    constexpr int DB = D / 32;
    constexpr int CPR = D / 8;
    constexpr int RP = 256 / (2 * D);
    constexpr int NR = 1024 / (2 * D);
    constexpr int NGRP = kUnit / NR;
    constexpr int NLD = NGRP / R;
    constexpr int SLOT = kUnit * D;
    constexpr int NJ = kUnit / 16;
    constexpr int SLOTB = 2 * SLOT;  // bytes per tile
    // a key group's two ring slots hold four tiles each: K hi | K lo | V hi | V lo
    __shared__ __attribute__((aligned(1024))) uint16_t smem[G * 8 * SLOT];

    const int bid = blockIdx.x;
    const int nbh = a.B * a.Hq;
    const int qt = launch_row<D == 128>(a, bid / nbh);
    const int bh = xcd_grouped_head(bid % nbh, a.B * a.Hkv, a.n_rep);  // a kv group's query heads share one XCD's L2
    const int b = bh / a.Hq, hq = bh % a.Hq, kvh = hq / a.n_rep;
    const int L = a.L;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ql = lane & 31, h = lane >> 5;
    const int row = wave % R, group = wave / R;
    const int q0 = qt * (32 * R) + row * 32;
    const uint32_t lds0 = lds_addr(smem) + (uint32_t)(group * 8 * SLOTB);
    const int off = L - a.T;
    const int qrow = min(q0 + ql, a.T - 1);

    const int64_t ko = (int64_t)b * a.sk[0] + (int64_t)kvh * a.sk[1];
    const int64_t vo = (int64_t)b * a.sv[0] + (int64_t)kvh * a.sv[1];
    // Q comes as the caller's fp32 tensor (any strides) and is split here: each row is read by exactly one wavefront
    const float* qp = (const float*)a.q + (int64_t)b * a.sq[0] + (int64_t)hq * a.sq[1] + (int64_t)qrow * a.sq[2];
    bf16x8_t qh[KS], qlo[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const float4 x0 = *(const float4*)(qp + 16 * ks + 8 * h), x1 = *(const float4*)(qp + 16 * ks + 8 * h + 4);
        float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        uint32_t hw[4], lw[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float f0 = a.negate_q ? -x[2 * i] : x[2 * i], f1 = a.negate_q ? -x[2 * i + 1] : x[2 * i + 1];  // exact
            hw[i] = cvt_pk_bf16(f0, f1);
            lw[i] = cvt_pk_bf16(f0 - __uint_as_float(hw[i] << 16), f1 - __uint_as_float(hw[i] & 0xffff0000u));
        }
        qh[ks] = __builtin_bit_cast(bf16x8_t, uint4{hw[0], hw[1], hw[2], hw[3]});
        qlo[ks] = __builtin_bit_cast(bf16x8_t, uint4{lw[0], lw[1], lw[2], lw[3]});
    }

    const int wg_qmax = min(qt * (32 * R) + 32 * R - 1, a.T - 1);
    const int kv_end_wg = a.causal ? min(L, wg_qmax + off + 1) : L;
    const int n_stages = (kv_end_wg + kUnit * G - 1) / (kUnit * G);   // of G key tiles
    const int wave_qmax = min(q0 + 31, a.T - 1);
    const int kv_end_wave = (q0 < a.T) ? (a.causal ? min(L, wave_qmax + off + 1) : L) : 0;

    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
    float m_ref = -INFINITY;
    float l = 0.f;

    // global -> LDS as in prefill_bf16_kernel; the planes are dense, so K and V rows have the same pitch
    const int ld_row = lane / CPR, ld_pos = lane % CPR;
    uint32_t voffK[NLD], voffV[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int r = NR * (row + R * i) + ld_row;
        voffK[i] = (uint32_t)r * (uint32_t)(2 * D) + 16u * (uint32_t)(ld_pos ^ ((r / RP) % CPR));
        voffV[i] = (uint32_t)r * (uint32_t)(2 * D) + 16u * (uint32_t)(ld_pos ^ (((r / RP) % (CPR / 4)) << 2));
    }
    auto load_stage = [&](int st, int slot) {
        const int key0 = (st * G + group) * kUnit;
        const int bytes = max(L - key0, 0) * 2 * D;  // rows past the context read as zeros
        const char* bases[4] = {(const char*)((const uint16_t*)a.k + ko), (const char*)((const uint16_t*)a.k_lo + ko),
                                (const char*)((const uint16_t*)a.v + vo), (const char*)((const uint16_t*)a.v_lo + vo)};
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(bases[x] + (int64_t)key0 * 2 * D), 0, bytes, 0x00020000);
            uint16_t* dst = smem + (8 * group + 4 * slot + x) * SLOT;
#pragma unroll
            for (int i = 0; i < NLD; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(dst + (row + R * i) * 512), 16, x < 2 ? voffK[i] : voffV[i], 0, 0, 0);
        }
    };

    const int kswz = (ql / RP) % CPR;
    uint32_t kaddr[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kaddr[ks] = lds0 + 2u * (uint32_t)(ql * D + 8 * ((2 * ks + h) ^ kswz));
    const int i16 = lane & 15;
    const int vswz = ((i16 >> 2) / RP) % (CPR / 4);
    const int v_lane_off = (4 * h + (i16 >> 2)) * D + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    uint32_t va[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) va[db] = lds0 + 2u * (uint32_t)v_lane_off + 64u * (uint32_t)(db ^ vswz);

    auto stage_step = [&](int st, auto slot_c) {
        constexpr int slot = decltype(slot_c)::value;
        constexpr int KH = (4 * slot) * SLOTB, KL = (4 * slot + 1) * SLOTB, VH = (4 * slot + 2) * SLOTB, VL = (4 * slot + 3) * SLOTB;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (st + 1 < n_stages) load_stage(st + 1, slot ^ 1);
        const int k0 = (st * G + group) * kUnit;
        if (k0 >= kv_end_wave) return;

        // S^T = K_hi Q_hi^T + K_hi Q_lo^T + K_lo Q_hi^T; the operands of k-step ks + 1 are requested before those of ks are used
        f32x16_t s;
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = 0.f;
        u32x4_t kh[KS], kl[KS];
        kh[0] = lds_read_b128_asm<KH>(kaddr[0]);
        kl[0] = lds_read_b128_asm<KL>(kaddr[0]);
        static_for<KS>([&](auto i) {
            constexpr int ks = i.value;
            if constexpr (ks + 1 < KS) {
                kh[ks + 1] = lds_read_b128_asm<KH>(kaddr[ks + 1]);
                kl[ks + 1] = lds_read_b128_asm<KL>(kaddr[ks + 1]);
                lds_wait<3>(kh[ks]);
                lds_wait<2>(kl[ks]);
            } else {
                lds_wait<1>(kh[ks]);
                lds_wait<0>(kl[ks]);
            }
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kh[ks]), qh[ks], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kh[ks]), qlo[ks], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kl[ks]), qh[ks], s, 0, 0, 0);
        });
        const bool need_mask = (a.causal && k0 + kUnit - 1 > q0 + off) || (k0 + kUnit > L);
        if (need_mask) {
            const int q_abs = q0 + ql + off;
            const int lim = a.causal ? min(q_abs, L - 1) : L - 1;
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (k0 + 8 * (v >> 2) + 4 * h + (v & 3) > lim) s[v] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
        mx = half_swap_max(mx) * a.scale_log2;
        if (__any(mx > m_ref + kRescaleThreshold)) {  // P stays below 2^8 between raises: nothing to lose in fp32
            const float m_new = fmaxf(m_ref, mx);
            const float alpha = (m_new == -INFINITY || m_ref == -INFINITY) ? (m_ref == -INFINITY ? 0.f : 1.f) : __builtin_amdgcn_exp2f(m_ref - m_new);
            l *= alpha;
#pragma unroll
            for (int i = 0; i < DB; ++i)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[i][j] *= alpha;
            m_ref = m_new;
        }
        const float neg_m = (m_ref == -INFINITY) ? 0.f : -m_ref;
        // P = exp2(s scale - m) in fp32, summed in fp32, then split like the inputs
        uint32_t ph[NJ][4], pl[NJ][4];
        float lsum = 0.f;
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], a.scale_log2, neg_m));
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v + 1], a.scale_log2, neg_m));
            lsum += p0 + p1;
            const uint32_t hw = cvt_pk_bf16(p0, p1);
            ph[v >> 3][(v & 7) >> 1] = hw;
            pl[v >> 3][(v & 7) >> 1] = cvt_pk_bf16(p0 - __uint_as_float(hw << 16), p1 - __uint_as_float(hw & 0xffff0000u));
        }
        l += lsum;
        // O^T += V_hi^T P_hi + V_hi^T P_lo + V_lo^T P_hi, one (key half, d block) at a time, the next operands in flight
        uint2 vh[2], vl[2], nh[2], nl[2];
        vh[0] = lds_read_tr16_b64_asm<VH>(va[0]);
        vh[1] = lds_read_tr16_b64_asm<VH + 8 * D * 2>(va[0]);
        vl[0] = lds_read_tr16_b64_asm<VL>(va[0]);
        vl[1] = lds_read_tr16_b64_asm<VL + 8 * D * 2>(va[0]);
        static_for<NJ * DB>([&](auto ic) {
            constexpr int idx = ic.value, j = idx / DB, db = idx % DB;
            if constexpr (idx + 1 < NJ * DB) {
                constexpr int j2 = (idx + 1) / DB, db2 = (idx + 1) % DB;
                nh[0] = lds_read_tr16_b64_asm<VH + (16 * j2) * D * 2>(va[db2]);
                nh[1] = lds_read_tr16_b64_asm<VH + (16 * j2 + 8) * D * 2>(va[db2]);
                nl[0] = lds_read_tr16_b64_asm<VL + (16 * j2) * D * 2>(va[db2]);
                nl[1] = lds_read_tr16_b64_asm<VL + (16 * j2 + 8) * D * 2>(va[db2]);
                asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(vh[0]), "+v"(vh[1]), "+v"(vl[0]), "+v"(vl[1]));
            } else {
                asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(vh[0]), "+v"(vh[1]), "+v"(vl[0]), "+v"(vl[1]));
            }
            const bf16x8_t pfh = __builtin_bit_cast(bf16x8_t, uint4{ph[j][0], ph[j][1], ph[j][2], ph[j][3]});
            const bf16x8_t pfl = __builtin_bit_cast(bf16x8_t, uint4{pl[j][0], pl[j][1], pl[j][2], pl[j][3]});
            const bf16x8_t vfh = __builtin_bit_cast(bf16x8_t, uint4{vh[0].x, vh[0].y, vh[1].x, vh[1].y});
            const bf16x8_t vfl = __builtin_bit_cast(bf16x8_t, uint4{vl[0].x, vl[0].y, vl[1].x, vl[1].y});
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vfh, pfh, acc[db], 0, 0, 0);
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vfh, pfl, acc[db], 0, 0, 0);
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vfl, pfh, acc[db], 0, 0, 0);
            if constexpr (idx + 1 < NJ * DB) {
                vh[0] = nh[0];
                vh[1] = nh[1];
                vl[0] = nl[0];
                vl[1] = nl[1];
            }
        });
    };

    if (n_stages > 0) load_stage(0, 0);
    for (int st = 0; st < n_stages; st += 2) {
        stage_step(st, std::integral_constant<int, 0>{});
        if (st + 1 < n_stages) stage_step(st + 1, std::integral_constant<int, 1>{});
    }

    l = half_swap_sum(l);
    const int qi = q0 + ql;
    float* op = (float*)a.out + (int64_t)b * a.so[0] + (int64_t)hq * a.so[1] + (int64_t)qi * a.so[2];
    float* lp = a.lse ? a.lse + (int64_t)b * a.sl[0] + (int64_t)hq * a.sl[1] + (int64_t)qi * a.sl[2] : nullptr;
    constexpr int NQ = 4 * DB, MINE = NQ / G;
    if constexpr (G == 1) {
        if (qi < a.T) {
            const float inv_l = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
            for (int i = 0; i < NQ; ++i)
                *(float4*)(op + 8 * i + 4 * h) = float4{acc[i >> 2][4 * (i & 3)] * inv_l, acc[i >> 2][4 * (i & 3) + 1] * inv_l, acc[i >> 2][4 * (i & 3) + 2] * inv_l, acc[i >> 2][4 * (i & 3) + 3] * inv_l};
            if (lp && h == 0) *lp = (m_ref + log2f(l)) * 0.6931471805599453f;
        }
    } else {   // the key groups' partial results meet in the ring; each wavefront merges and stores a G-th of its rows' columns
        __shared__ float sM[4][32], sL[4][32];
        auto image = [&](int w) { return (f32x4_t*)smem + w * (NQ * 64) + lane; };
        __syncthreads();   // every wavefront has left the last stage
#pragma unroll
        for (int i = 0; i < NQ; ++i) image(wave)[64 * i] = f32x4_t{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
        if (h == 0) sM[wave][ql] = m_ref, sL[wave][ql] = l;
        __syncthreads();
        float m = sM[row][ql], w[G];
#pragma unroll
        for (int g = 1; g < G; ++g) m = fmaxf(m, sM[row + g * R][ql]);
        l = 0.f;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const float mg = sM[row + g * R][ql];
            w[g] = mg == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mg - m);   // a group without a visible key weighs nothing
            l += w[g] * sL[row + g * R][ql];
        }
        if (qi < a.T) {
            const float inv_l = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
            for (int g = 0; g < G; ++g) w[g] *= inv_l;
#pragma unroll
            for (int i = 0; i < MINE; ++i) {
                f32x4_t sum = w[0] * image(row)[64 * (MINE * group + i)];
#pragma unroll
                for (int g = 1; g < G; ++g) sum += w[g] * image(row + g * R)[64 * (MINE * group + i)];
                *(f32x4_t*)(op + 8 * (MINE * group + i) + 4 * h) = sum;
            }
            if (lp && h == 0 && group == 0) *lp = (m + log2f(l)) * 0.6931471805599453f;
        }
    }
#endif
}

// ---------------------------------------------------------------------------------------------
// Software-pipelined bf16 kernel, D = 128, dense K/V.  Same tiles, fragment layouts and arithmetic as
// prefill_bf16_kernel; what changes is the order of work inside a wavefront.  Step tau of a wavefront issues, as
// three independent instruction streams,
//     S(tau+2) = K(tau+2) Q^T          8 MFMAs into the "next" score registers
//     P(tau+1) = exp2(S(tau+1) - m)    the vector-ALU work, on scores finished one step earlier
//     O       += V(tau)^T P(tau)       8 MFMAs with the P computed one step earlier
// so no MFMA of a step waits for vector-ALU work of the same step and vice versa: the matrix pipe and the vector ALU
// of one SIMD run side by side from a single wavefront's instruction stream.  The 16 MFMAs of a step are "slots";
// each slot is followed by its share of the softmax instructions and by the LDS reads of the operand needed kLead
// slots later (the reads run ahead across step boundaries).  Four ring slots per operand in LDS: the tiles a step
// needs were requested three steps earlier and published by the barrier one step earlier, so neither the barrier nor
// the global loads sit on a wavefront's critical path.
// Vector-ALU instructions of one wavefront hardly overlap with MFMAs of ANOTHER wavefront on the same SIMD (a wavefront
// of nothing but vector-ALU work gets about one instruction in per MFMA of its neighbour), while those that follow an
// MFMA in the same instruction stream are nearly free; hence this structure, and the diet of the softmax stage:
//   - -m / c (m: the row's reference maximum, c = |scale| * log2(e)) enters as the C operand of the first QK^T MFMA,
//     so P is one multiply and one exp2 per score (Q is not pre-multiplied by c: rounding Q * c to bf16 again costs
//     2^-9 of every score, which shows in the output once logits reach the tens);
//   - the row sum uses plain adds (v_dot2c_f32_bf16 occupies the matrix pipe);
//   - no row maximum per tile: m is raised only when the row sum shows that it has fallen behind (rare), and is
//     kept integer-valued (log2 domain) so that the rescale factor is a power of two and the P tile that has been
//     computed but not yet multiplied into O rescales exactly.
// ---------------------------------------------------------------------------------------------
constexpr int kLead = 6;  // LDS operand reads run this many MFMA slots ahead

// MFMA slot order of a step: Q = a QK^T MFMA (k-step index), P = a PV MFMA (index p: key half p / 4, d block p % 4).
// The QK chain finishes at slot 10, so that the row maximum of the new scores is taken under the last PV MFMAs.
constexpr int kSlotIsQ[16] = {1, 1, 0, 1, 1, 0, 1, 1, 0, 1, 1, 0, 0, 0, 0, 0};
[[maybe_unused]] constexpr int kSlotIdx[16] = {0, 1, 0, 2, 3, 1, 4, 5, 2, 6, 7, 3, 4, 5, 6, 7};
// LDS read instructions per operand: one ds_read_b128 for K rows and for V^T taken from a token-blocked plane, two
// transposing reads for V^T taken from row-major V
template <bool VBLK>
constexpr int slot_reads(int s) { return (kSlotIsQ[s & 15] || VBLK) ? 1 : 2; }
// LDS reads issued after the operand of slot s and before the wait at slot s: those of slots s+1 .. s+kLead-1
template <bool VBLK>
constexpr int reads_behind(int s) {
    int n = 0;
    for (int k = 1; k < kLead; ++k) n += slot_reads<VBLK>(s + k);
    return n;
}

struct Frag {  // one MFMA A operand on its way from LDS
    u32x4_t k;     // K rows (ds_read_b128)
    uint2 t0, t1;  // V^T halves (two transposing reads)
};

template <int N>
__device__ inline void frag_wait_k(u32x4_t& k) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(k) : "n"(N));
}
template <int N>
__device__ inline void frag_wait_v(uint2& t0, uint2& t1) {
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(t0), "+v"(t1) : "n"(N));
}

// VBLK: K and V are the planes of a bf16 KV cache (K row-major, V token-blocked by 8), possibly paged, with the context
// length per batch row from a device array; see prefill_bf16_kernel for the operand layouts this implies.
template <bool VBLK, bool ROPE>
__global__ void __launch_bounds__(256, 2) prefill_bf16_pipe_kernel(PrefillArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    constexpr int D = 128;
    constexpr int KS = D / 16;
    constexpr int DB = D / 32;
    constexpr int CPR = D / 8;
    constexpr int RP = 256 / (2 * D);
    constexpr int NR = 1024 / (2 * D);
    constexpr int NGRP = kUnit / NR;
    constexpr int NLD = NGRP / 4;
    constexpr int SLOT = kUnit * D;
    constexpr int SLOTB = 2 * SLOT;
    constexpr int NRING = 4;
    static_assert(KS == 8 && DB == 4 && NLD == 2, "written for D = 128");

    // K ring (4 slots) | V ring (4 slots)
    __shared__ __attribute__((aligned(1024))) uint16_t smem[2 * NRING * SLOT];
    const uint32_t lds0 = lds_addr(smem);

    int bid = blockIdx.x;
    int tile0 = 0;  // first key tile of this workgroup's share of the context (a split context: cache-plane mode only)
    int split = 0;
    if constexpr (VBLK) {
        if (a.n_splits > 1) {
            split = (int)a.by_share.div((uint32_t)bid);
            bid = (int)a.by_share.mod((uint32_t)bid, (uint32_t)split);
            tile0 = split * a.split_tiles;
        }
    }
    const uint32_t from_last = a.by_bh.div((uint32_t)bid), pos = a.by_bh.mod((uint32_t)bid, from_last), rep = a.by_bkv.div(pos), g_kv = a.by_bkv.mod(pos, rep), ub = a.by_kv.div(g_kv);
    const int qt = launch_row<D == 128>(a, (int)from_last), b = (int)ub, kvh = (int)a.by_kv.mod(g_kv, ub), h0 = kvh * a.n_rep + (int)rep;   // h0: the workgroup's first query head
    int L = a.L;
    // cache mode: per-row context length (clamped to the bound a.L) and per-row chunk length n <= T: query t < n sits
    // at absolute position L - n + t; rows t >= n carry no query and their output is unspecified
    int n_chunk = a.T;
    if constexpr (VBLK) {
        if (a.chunk_lens) n_chunk = min(max(a.chunk_lens[b], 0), a.T);
        if (a.seq_lens) L = min(max(a.seq_lens[b], n_chunk), a.L);
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ql = lane & 31, h = lane >> 5;
    const int q0 = qt * kBM + wave * 32;
    const int off = L - n_chunk;
    // this lane's row: query (token) tq of head hq
    const GroupRow row = group_row(a, q0 + ql);
    const int tq = row.token, hq = h0 + row.head;
    const int t_first = (int)a.by_pack.div((uint32_t)q0);   // of the wavefront's rows

    const uint16_t* Qp = (const uint16_t*)a.q + (int64_t)b * a.sq[0] + (int64_t)h0 * a.sq[1];
    const uint16_t* Kp = (const uint16_t*)a.k + (int64_t)b * a.sk[0] + (int64_t)kvh * a.sk[1];
    const uint16_t* Vp = (const uint16_t*)a.v + (int64_t)b * a.sv[0] + (int64_t)kvh * a.sv[1];

    uint4 qraw[KS];
    float4 pairs[KS][2];
    load_q_rows<D, ROPE>(a, Qp + row.offset, tq, h, qraw, pairs);
    bf16x8_t qf[KS];
    // Q goes into the MFMAs as stored (a negative scale flips its sign bits: exact); |scale| * log2(e) multiplies the
    // fp32 scores in front of the exp2, so the scores carry no rounding beyond the fp32 accumulation
    const float cexp = a.scale_log2;
    const float inv_cexp = 1.0f / cexp;
    auto prescale_q = [&]() { finish_q_rows<D, ROPE>(a, qraw, pairs, qf); };

    const int rows = a.T * a.pack;
    const int wg_qmax = (int)a.by_pack.div((uint32_t)min(qt * kBM + kBM - 1, rows - 1));
    const int kv_end_wg = a.causal ? min(L, wg_qmax + off + 1) : L;
    int n_tiles = (kv_end_wg + kUnit - 1) / kUnit;  // tiles the workgroup loads
    const int wave_qmax = (int)a.by_pack.div((uint32_t)min(q0 + 31, rows - 1));
    const int kv_end_wave = (q0 < rows) ? (a.causal ? min(L, wave_qmax + off + 1) : L) : 0;
    int nt_w = (kv_end_wave + kUnit - 1) / kUnit;  // tiles this wavefront uses
    // first tile of this wavefront that needs the mask (straddles the diagonal or the end of the context)
    int first_masked = min(nt_w, L / kUnit);
    if (a.causal) first_masked = min(first_masked, t_first + off - 31 < 0 ? 0 : (t_first + off - 31) / kUnit + 1);
    if constexpr (VBLK) {
        if (a.n_splits > 1) {  // this workgroup's share: tiles [tile0, tile0 + split_tiles), counted from tile0 below
            n_tiles = max(0, min(n_tiles, tile0 + a.split_tiles) - tile0);
            nt_w = min(max(0, nt_w - tile0), n_tiles);
            first_masked = min(max(0, first_masked - tile0), nt_w);
        }
    }
    const int n_fast = max(0, first_masked - 2);  // steps [0, n_fast): all three stages active, no mask
    const int n_mid = max(0, nt_w - 2);           // steps [0, n_mid): all three stages active

    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
    float m_ref = -INFINITY;
    float l = 0.f;

    // global -> LDS, as in prefill_bf16_kernel
    const int ld_row = lane / CPR, ld_pos = lane % CPR;
    uint32_t voffK[NLD], voffV[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int r = NR * (wave + 4 * i) + ld_row;
        // (contexts of more than two tiles only: 31 rows of a head are less than 2^31 bytes)
        voffK[i] = (uint32_t)r * (uint32_t)a.sk[2] * 2u + 16u * (uint32_t)(ld_pos ^ ((r / RP) % CPR));
        if constexpr (VBLK) voffV[i] = (uint32_t)(wave + 4 * i) * 1024u + 16u * (uint32_t)lane;  // the tile is contiguous
        else voffV[i] = (uint32_t)r * (uint32_t)a.sv[2] * 2u + 16u * (uint32_t)(ld_pos ^ (((r / RP) % (CPR / 4)) << 2));
    }
    const int64_t rowK = a.sk[2] * 2, rowV = a.sv[2] * 2;
    // where the 32-token tile starting at key0 lives: the head's slab and the first token inside it (a tile never
    // straddles a page: pages are multiples of 64 tokens)
    auto locate_tile = [&](int key0, const char*& kb, const char*& vb, int& local, int& cap, int& rows) {
        kb = (const char*)Kp;
        vb = (const char*)Vp;
        local = key0;
        cap = a.s_pad;
        rows = L - key0;
        if constexpr (VBLK) {
            if (a.page_table) {
                const int pg = key0 / a.page_tokens;
                local = key0 - pg * a.page_tokens;
                cap = a.page_tokens;
                const int64_t slab = (int64_t)a.page_table[(int64_t)b * a.pages_per_seq + pg] * a.Hkv + kvh;
                kb = (const char*)a.k + slab * cap * D * 2;
                vb = (const char*)a.v + slab * cap * D * 2;
                rows = min(rows, cap - local);
            }
        }
    };
    auto load_k_tile = [&](int t, int slot) {
        const char *kb, *vb;
        int local, cap, rows;
        locate_tile((tile0 + t) * kUnit, kb, vb, local, cap, rows);
        __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(kb + (int64_t)local * rowK), 0, (int)((int64_t)rows * rowK), 0x00020000);
        uint16_t* dst = smem + slot * SLOT;
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)(dst + (wave + 4 * i) * 512), 16, voffK[i], 0, 0, 0);
    };
    auto load_v_tile = [&](int t, int slot) {
        const char *kb, *vb;
        int local, cap, rows;
        locate_tile((tile0 + t) * kUnit, kb, vb, local, cap, rows);
        // VBLK: 32 tokens = 4 token blocks = kUnit * D contiguous elements; bound = the rest of this head's slab
        const int64_t v_base = VBLK ? (int64_t)local * D * 2 : (int64_t)local * rowV;
        const int64_t v_bytes = VBLK ? ((int64_t)cap - local) * D * 2 : (int64_t)rows * rowV;
        __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(vb + v_base), 0, (int)v_bytes, 0x00020000);
        uint16_t* dst = smem + (NRING + slot) * SLOT;
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)(dst + (wave + 4 * i) * 512), 16, voffV[i], 0, 0, 0);
    };

    // loop-constant LDS read addresses (ring slot 0 of each operand; the slot is an immediate offset)
    const int krow = VBLK ? ((ql & ~12) | ((ql & 4) << 1) | ((ql & 8) >> 1)) : ql;  // tile row this lane's S^T row holds
    const int kswz = (krow / RP) % CPR;
    uint32_t kaddr[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kaddr[ks] = lds0 + 2u * (uint32_t)(krow * D + 8 * ((2 * ks + h) ^ kswz));
    const int i16 = lane & 15;
    const int vswz = ((i16 >> 2) / RP) % (CPR / 4);
    const int v_lane_off = (4 * h + (i16 >> 2)) * D + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    uint32_t va[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
        va[db] = VBLK ? lds0 + 16u * (uint32_t)(h * D + ql) : lds0 + 2u * (uint32_t)v_lane_off + 64u * (uint32_t)(db ^ vswz);

    Frag fr[16];         // operand of MFMA slot s of the current step (slots < kLead: already requested)
    // With c = |scale| * log2(e), scores are kept as u = q.k - m / c: -m / c (m = the row's reference maximum in the
    // log2 domain) enters as the C operand of the first QK^T MFMA from a tile of 16 registers that all hold it, and
    // P = exp2(c * u).
    f32x16_t sb[2];      // step tau finishes S'(tau+2) in sb[tau & 1] and consumes S'(tau+1) from sb[(tau+1) & 1]
    uint32_t pb[2][8];   // packed bf16 P: step tau consumes P(tau) from pb[tau & 1] and writes P(tau+1) to pb[(tau+1) & 1]
    f32x16_t negm;       // every element = -m_ref / c of this lane's query
#pragma unroll
    for (int j = 0; j < 16; ++j) negm[j] = 0.f;
    m_ref = 0.f;  // "no reference yet": the first tile sets it

    // Request the operand of MFMA slot S of the step whose ring slot is RS.
    auto request = [&](auto s_c, auto rs_c) {
        constexpr int S = decltype(s_c)::value;
        constexpr int RS = decltype(rs_c)::value;
        if constexpr (kSlotIsQ[S]) {
            constexpr int ks = kSlotIdx[S];
            fr[S].k = lds_read_b128_asm<RS * SLOTB>(kaddr[ks]);
        } else {
            constexpr int p = kSlotIdx[S], j = p / 4, db = p % 4;
            if constexpr (VBLK) {  // token block 2j + h of the tile, rows d = 32 db + ql: one 16-byte read
                fr[S].k = lds_read_b128_asm<(NRING + RS) * SLOTB + (2 * j * D + 32 * db) * 16>(va[db]);
            } else {
                constexpr int VOFF = (NRING + RS) * SLOTB + 16 * j * D * 2;
                fr[S].t0 = lds_read_tr16_b64_asm<VOFF>(va[db]);
                fr[S].t1 = lds_read_tr16_b64_asm<VOFF + 8 * D * 2>(va[db]);
            }
        }
    };

    // One step.  PH = tau & 3 (ring slot of the step's tiles: K(tau+2), V(tau)).  MODE 0: all three stages are active
    // and the new scores need no mask, so the body is one straight line of code; 1: the same with the mask applied
    // under one wavefront-uniform branch; 2: every stage guarded (the first and last steps of a wavefront).
    auto step = [&](int tau, auto ph_c, auto fast_c) {
        constexpr int PH = decltype(ph_c)::value;
        constexpr int MODE = decltype(fast_c)::value;
        constexpr bool FAST = MODE < 2;     // all three stages active: no per-slot guards
        constexpr bool MASK = MODE > 0;     // the new scores may need the mask
        constexpr bool FIRST = MODE == 4;   // step -1: the softmax stage sees tile 0 and sets the reference
        f32x16_t& s_cur = sb[(PH + 1) & 1];
        f32x16_t& s_nxt = sb[PH & 1];
        uint32_t(&p_cur)[8] = pb[PH & 1];
        uint32_t(&p_nxt)[8] = pb[(PH + 1) & 1];

        if constexpr (MODE == 3) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");  // first step: K(1) has landed
        else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");  // the tiles of step tau+1 have landed; those of tau+2 may be in flight
        __builtin_amdgcn_s_barrier();  // waits are explicit: no fence, which would drain every load in flight
        // always four loads per wavefront and step, so that the vmcnt arithmetic holds: past the end the tile index is
        // clamped (the rows fall outside the buffer bound and arrive as zeros, or re-read the last tile; never consumed)
        if constexpr (MODE != 3) {
            load_k_tile(min(tau + 5, n_tiles - 1), (PH + 3) & 3);
            load_v_tile(min(tau + 3, n_tiles - 1), (PH + 3) & 3);
        }

        const bool qk_on = FAST || (tau + 2 < nt_w);
        const bool sm_on = FAST || (tau + 1 >= 0 && tau + 1 < nt_w);
        const bool pv_on = FAST || (tau >= 0 && tau < nt_w);

        float es[16];
        float lsum = 0.f, lsum2 = 0.f;
        // instruction i of the 32 that turn s_cur into p_nxt: per pair of scores 2 exp2, 1 pack, and the row sum.
        // Steady-state steps sum the fp32 values with plain adds (a dot2 occupies the matrix pipe); against the sum of
        // the bf16-rounded P that the PV MFMAs consume this is zero-mean rounding noise of relative size
        // 2^-9 / sqrt(keys), and such steps only exist in contexts of more than a hundred keys.  The first and last
        // steps of a wavefront sum the rounded values themselves (packed dot product against (1, 1)), so that short
        // contexts are normalised by exactly what was accumulated (a single key reproduces V bit for bit).
        auto softmax_op = [&](auto i_c) {
            constexpr int i = decltype(i_c)::value, p = i / 4, k = i % 4;
            if constexpr (k == 0) {  // both multiplies first: neither exp2 waits on the instruction right before it
                es[2 * p] = s_cur[2 * p] * cexp;
                es[2 * p + 1] = s_cur[2 * p + 1] * cexp;
                es[2 * p] = __builtin_amdgcn_exp2f(es[2 * p]);
            } else if constexpr (k == 1) es[2 * p + 1] = __builtin_amdgcn_exp2f(es[2 * p + 1]);
            else if constexpr (k == 2) p_nxt[p] = cvt_pk_bf16(es[2 * p], es[2 * p + 1]);
            else if constexpr (FAST && !MASK) { lsum += es[2 * p]; lsum2 += es[2 * p + 1]; }
            else lsum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, p_nxt[p]), __builtin_bit_cast(bf16x2_t, 0x3f803f80u), lsum, false);
        };

        static_for<16>([&](auto s_c) {
            constexpr int S = decltype(s_c)::value;
            // ---- the MFMA of this slot
            if constexpr (kSlotIsQ[S]) {
                constexpr int ks = kSlotIdx[S];
                frag_wait_k<reads_behind<VBLK>(S)>(fr[S].k);
                if (qk_on) {
                    if constexpr (ks == 0) s_nxt = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fr[S].k), qf[ks], negm, 0, 0, 0);
                    else s_nxt = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fr[S].k), qf[ks], s_nxt, 0, 0, 0);
                }
            } else {
                constexpr int p = kSlotIdx[S], j = p / 4, db = p % 4;
                if constexpr (VBLK) frag_wait_k<reads_behind<VBLK>(S)>(fr[S].k);
                else frag_wait_v<reads_behind<VBLK>(S)>(fr[S].t0, fr[S].t1);
                if (pv_on) {
                    if constexpr (VBLK && MODE >= 2) {
                        // the planes hold stale tokens past L: P is 0 there, V must not be NaN
                        const int nvalid = L - ((tile0 + tau) * kUnit + 16 * j + 8 * h);  // slots e >= nvalid are past the context
                        if (nvalid < 8) {
#pragma unroll
                            for (int w = 0; w < 4; ++w) {
                                uint32_t x = fr[S].k[w];
                                if (2 * w + 1 >= nvalid) x &= 0x0000ffffu;
                                if (2 * w >= nvalid) x = 0;
                                fr[S].k[w] = x;
                            }
                        }
                    }
                    const bf16x8_t vf = VBLK ? __builtin_bit_cast(bf16x8_t, fr[S].k)
                                             : __builtin_bit_cast(bf16x8_t, uint4{fr[S].t0.x, fr[S].t0.y, fr[S].t1.x, fr[S].t1.y});
                    const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, uint4{p_cur[4 * j], p_cur[4 * j + 1], p_cur[4 * j + 2], p_cur[4 * j + 3]});
                    acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, acc[db], 0, 0, 0);
                }
            }
            // ---- the operand of the slot kLead ahead (next step's tiles once the index wraps)
            if constexpr (S + kLead < 16) request(std::integral_constant<int, S + kLead>{}, std::integral_constant<int, PH>{});
            else request(std::integral_constant<int, S + kLead - 16>{}, std::integral_constant<int, (PH + 1) & 3>{});
            // ---- this slot's share of the vector-ALU work
            if constexpr (!FIRST) {
                if (sm_on) static_for<2>([&](auto k_c) { softmax_op(std::integral_constant<int, 2 * S + decltype(k_c)::value>{}); });
            }
            if constexpr (MASK && S == 12) {
                if (qk_on) {
                    const int k0 = (tile0 + tau + 2) * kUnit;
                    if ((a.causal && k0 + kUnit - 1 > t_first + off) || (k0 + kUnit > L)) {
                        const int q_abs = tq + off;
                        const int lim = a.causal ? min(q_abs, L - 1) : L - 1;
#pragma unroll
                        for (int v = 0; v < 16; ++v)
                            if ((VBLK ? k0 + 16 * (v >> 3) + 8 * h + (v & 7) : k0 + 8 * (v >> 2) + 4 * h + (v & 3)) > lim) s_nxt[v] = -INFINITY;
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if (sm_on) {
            // A reference that has fallen behind shows in the row sum: below 2^10 no P of the tile exceeds 2^10, far
            // from overflow; otherwise (rare; and always for the first tile, which has no reference yet) take the true
            // maximum of these scores, raise the reference to an integer at or above it (alpha is then a power of
            // two, so everything computed against the old reference rescales exactly) and redo this tile's P.
            constexpr bool first = FIRST;
            if (first || __any(!(lsum + lsum2 < 1024.f))) {
                float mx = s_cur[0];
#pragma unroll
                for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s_cur[v]);
                mx = half_swap_max(mx);
                // raise (first tile: set) the reference by delta, an integer in the log2 domain; the scores move by du
                float delta = (mx == -INFINITY) ? 0.f : ceilf(mx * cexp);
                if (!first) delta = fmaxf(delta, 0.f);
                const float du = delta == 0.f ? 0.f : delta * inv_cexp;  // (a scale in the denormal range has 1 / c = inf)
                if constexpr (!first) {  // nothing has been accumulated before the first tile
                    const float alpha = __builtin_amdgcn_exp2f(-delta);
                    l *= alpha;
#pragma unroll
                    for (int i = 0; i < DB; ++i)
#pragma unroll
                        for (int j = 0; j < 16; ++j) acc[i][j] *= alpha;
                }
                lsum = lsum2 = 0.f;
#pragma unroll
                for (int v = 0; v < 16; ++v) s_cur[v] -= du;
                static_for<32>([&](auto i_c) { softmax_op(i_c); });
                if (qk_on) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) s_nxt[v] -= du;  // finished this step against the old reference
                }
                m_ref += delta;
#pragma unroll
                for (int j = 0; j < 16; ++j) negm[j] = m_ref == 0.f ? 0.f : -m_ref * inv_cexp;
            }
            l += lsum + lsum2;
        }
    };

    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using Fast = std::integral_constant<int, 0>;
    using Mid = std::integral_constant<int, 1>;
    using Slow = std::integral_constant<int, 2>;
    using First = std::integral_constant<int, 3>;   // step -2: Slow, and the tiles three steps ahead were requested by the prologue
    using Second = std::integral_constant<int, 4>;  // step -1: Slow, and its softmax stage sets the reference from tile 0

    if (n_tiles > 0) {  // an empty context (cache mode, length 0) has nothing to attend to: zeros below
    // prologue: the tiles of steps -2 and -1 (K(0), K(1)) are requested here, published by the barrier below
    load_k_tile(0, 2);
    load_k_tile(min(1, n_tiles - 1), 3);
    // tiles of steps 0 and 1 (K(2), V(0), K(3), V(1)); from step -1 on every step requests the tiles three steps ahead
    load_k_tile(min(2, n_tiles - 1), 0);
    load_v_tile(0, 0);
    load_k_tile(min(3, n_tiles - 1), 1);
    load_v_tile(min(1, n_tiles - 1), 1);
    prescale_q();
    asm volatile("s_waitcnt vmcnt(10)" ::: "memory");  // K(0) has landed
    __builtin_amdgcn_s_barrier();  // waits are explicit: no fence, which would drain every load in flight
    static_for<kLead>([&](auto s_c) { request(s_c, I2{}); });

    step(-2, I2{}, First{});
    step(-1, I3{}, Second{});
    int tau = 0;
    for (; tau + 4 <= n_fast; tau += 4) {
        step(tau, I0{}, Fast{});
        step(tau + 1, I1{}, Fast{});
        step(tau + 2, I2{}, Fast{});
        step(tau + 3, I3{}, Fast{});
    }
    for (; tau + 4 <= n_mid; tau += 4) {
        step(tau, I0{}, Mid{});
        step(tau + 1, I1{}, Mid{});
        step(tau + 2, I2{}, Mid{});
        step(tau + 3, I3{}, Mid{});
    }
    for (; tau < n_tiles; tau += 4) {
        step(tau, I0{}, Slow{});
        if (tau + 1 < n_tiles) step(tau + 1, I1{}, Slow{});
        if (tau + 2 < n_tiles) step(tau + 2, I2{}, Slow{});
        if (tau + 3 < n_tiles) step(tau + 3, I3{}, Slow{});
    }
    // operands requested for a step that does not exist are still in flight: let them land before the registers die
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
        prescale_q();
    }

    l = half_swap_sum(l);
    const bool there = q0 + ql < rows;
    if constexpr (VBLK) {
        if (a.n_splits > 1) {  // the unnormalised partial of this share of the context; the combine kernel finishes the row
            if (there) {
                const int64_t part = (((int64_t)b * a.Hq + hq) * a.T + tq) * a.n_splits + split;
                float* po = a.ws_o + part * D;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int vq = 0; vq < 4; ++vq)
                        *(float4*)(po + 32 * db + 8 * vq + 4 * h) = float4{acc[db][4 * vq], acc[db][4 * vq + 1], acc[db][4 * vq + 2], acc[db][4 * vq + 3]};
                if (h == 0) {  // a row that met no key in this share (masked, or the share lies past its diagonal) says so
                    a.ws_ml[part * 2] = l > 0.f ? m_ref : -INFINITY;
                    a.ws_ml[part * 2 + 1] = l;
                }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            return;
        }
    }
    // the clamped tile requests of the last steps write LDS: they have landed before the ring is used for the output
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // every wavefront has left the ring
    store_rows<D>(a, smem + wave * SLOT, acc, l > 0.f ? 1.0f / l : 0.f, b, h0, q0, lane);
    if (there && a.lse && h == 0)
        a.lse[(int64_t)b * a.sl[0] + (int64_t)hq * a.sl[1] + (int64_t)tq * a.sl[2]] = (m_ref + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
#endif
}

// A row's reference in prefill_f32_kernel's LAG instances may lag 2^kLag behind its maximum, which saves most rescalings of the accumulators and makes
// the sums up to 2^kLag larger.  A sum that this makes overflow (|V| above 2^120 / the keys that weigh) is not finite to the end; the workgroup sees it
// in what it stores and does its tiles again with the reference at the running maximum, where no weight is above 1.  From kLagTiles key tiles on: us at the
// running maximum, with the lag: D 128, 32 heads, 777 tokens 69.1 and 66.7, 1500 220 and 209; 2 x 32, 2048 572 and 554; D 64, 32 heads, 2557 240 and
// 232; but 8 x 12 heads, 128 tokens 9.8 and 10.5, D 128, 8 x 64, 43 tokens 20.2 and 20.4.
constexpr float kLag = 8.f;
constexpr int kLagTiles = 16;

// ---------------------------------------------------------------------------------------------
// fp32 kernel (fp32 inputs, fp32 MFMA 32x32x2, fp32 softmax): the precision the reference computes
// in.  R row groups of 32 queries times G key groups, one wavefront each, as in prefill_bf16_kernel: key group g takes the
// 32-key tiles g, g + G, ..., and the G partial results of a row group meet in LDS at the end.
// GEN: the tensors' head_dim a.D_true is any value up to the tile width D (the reference's forward takes any
// head_dim, src/ops/flash_attention.cpp:235-238): columns past it are zero in the operands (they add nothing to a
// score) and are not stored; rows are read element by element, so they need no 16-byte alignment.
// Bound by the fp32 matrix pipe (64 cycles per 32x32x2 MFMA, D of them per tile), which the vector ALU's work adds to: fp32 MFMAs and
// vector instructions of the two wavefronts of a SIMD were busy 0.55 + 0.29 of the cycles one beside the other, hardly together
// (D 64, 32 heads, 2557 tokens), so every vector instruction counts.  The next tile travels in registers under the MFMAs of the current
// one, by descriptors whose base is scalar; contraction slot (4 c + e, h) of Q K^T is d = 8 c + 4 h + e, so that one 16-byte LDS
// read (and one 16-byte load of Q) feeds four MFMAs; masks are a branch of the tiles that need them, a weight is one fma and one
// exp2 (weights below 2^-126 of a row's reference are 0), and accumulators are rescaled only when a row's reference moves (kLag).  A key
// group of one wavefront needs no barrier.
// MFMA busy 0.55 -> 0.73 there and 302 -> 230 us; 2 x 32 heads, D 128, 2048 tokens 747 -> 554; 4 x 16 heads, D 64, 1775 tokens 252 -> 222.
// Tiles kept twice in LDS (one barrier per tile) gave 3 % to 128-query workgroups of D 128 and took 3 to 7 % where the LDS then holds
// fewer workgroups: not kept.
// ---------------------------------------------------------------------------------------------
template <int D, bool GEN, int R, int G, bool LAG>
__global__ void __launch_bounds__(64 * R * G, D <= 64 || (D == 128 && R == 4) ? 2 : 1) prefill_f32_kernel(PrefillArgs a) {
    constexpr int BN = 32;
    constexpr int BM = 32 * R;
    constexpr int PITCH = D + 8;  // 4 rows apart = 32 banks apart: the two half-waves of a V read do not meet
    constexpr int DB = D / 32;
    constexpr int NC = D / 8;     // 16-byte pieces of a row per half-wave
    constexpr int TILE = BN * PITCH;
    constexpr int NLD = BN * D / 4 / (64 * R);  // 16-byte pieces of a tile per thread of its key group
    extern __shared__ __attribute__((aligned(16))) float smem_f32[];  // per key group: K tile | V tile
    __shared__ float sm_m[G][BM], sm_l[G][BM];
    [[maybe_unused]] __shared__ int sm_again;
    const int Dt = GEN ? a.D_true : D;

    const int bid = blockIdx.x;
    const int qt = launch_row<true>(a, bid / (a.B * a.Hq));
    const int bh = xcd_grouped_head(bid % (a.B * a.Hq), a.B * a.Hkv, a.n_rep);
    const int b = bh / a.Hq, hq = bh % a.Hq, kvh = hq / a.n_rep;
    const int n_chunk = a.chunk_lens ? min(max(a.chunk_lens[b], 0), a.T) : a.T;  // cache mode, as in the bf16 kernel
    const int L = a.seq_lens ? min(max(a.seq_lens[b], n_chunk), a.L) : a.L;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave_id % R, grp_k = wave_id / R;
    const int gt = tid - grp_k * (64 * R);  // thread of the key group
    float* sK = smem_f32 + grp_k * (2 * TILE);
    float* sV = sK + TILE;
    const int ql = lane & 31, h = lane >> 5;
    const int q0 = qt * BM + wave * 32;
    const int off = L - n_chunk;
    const int qrow = min(q0 + ql, a.T - 1);

    const float* Qp = (const float*)a.q + (int64_t)b * a.sq[0] + (int64_t)hq * a.sq[1] + (int64_t)qrow * a.sq[2];
    const float* Kp = (const float*)a.k + (int64_t)b * a.sk[0] + (int64_t)kvh * a.sk[1];
    const float* Vp = (const float*)a.v + (int64_t)b * a.sv[0] + (int64_t)kvh * a.sv[1];

    // Q^T operands: column ql, contraction slot (4 c + e, h) is d = 8 c + 4 h + e
    float qf[NC][4];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int d = 8 * c + 4 * h;
        if constexpr (GEN) {
#pragma unroll
            for (int e = 0; e < 4; ++e) qf[c][e] = d + e < Dt ? Qp[d + e] : 0.f;
        } else {
            const float4 w = *(const float4*)(Qp + d);
            qf[c][0] = w.x, qf[c][1] = w.y, qf[c][2] = w.z, qf[c][3] = w.w;
        }
    }

    const int wg_qmax = min(qt * BM + BM - 1, a.T - 1);
    const int kv_end_wg = a.causal ? min(L, wg_qmax + off + 1) : L;
    const int n_tiles = (kv_end_wg + BN - 1) / BN;
    const int wave_qmax = min(q0 + 31, a.T - 1);
    const int kv_end_wave = (q0 < a.T) ? (a.causal ? min(L, wave_qmax + off + 1) : L) : 0;

    f32x16_t acc[DB];
    float m_ref, neg, l;  // neg = -m_ref sc, as rounded: what every weight is taken relative to
    float lag = LAG ? kLag : 0.f;

    f32x4_t kreg[NLD], vreg[NLD];
    auto fetch = [&](int kt) {
        if constexpr (!GEN) {  // rows past L fall outside the descriptor and arrive as zeros
            constexpr int RS = 64 * R / (D / 4);
            const int rows = min(BN, L - kt * BN), row = gt / (D / 4), col = 16 * (gt % (D / 4));
            const int rowK = (int)a.sk[2] * 4, rowV = (int)a.sv[2] * 4;
            const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(Kp + (int64_t)kt * BN * a.sk[2]), 0, (rows - 1) * rowK + 4 * D, 0x00020000);
            const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(Vp + (int64_t)kt * BN * a.sv[2]), 0, (rows - 1) * rowV + 4 * D, 0x00020000);
            auto piece = [&](int i) {
                kreg[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, (row + i * RS) * rowK + col, 0, 0));
                vreg[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, (row + i * RS) * rowV + col, 0, 0));
            };
#pragma unroll
            for (int i = 0; i < NLD; ++i) piece(i);
            return;
        }
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int id = gt + i * (64 * R), row = id / (D / 4), col = 4 * (id % (D / 4)), key = kt * BN + row;
            float4 kk = {0.f, 0.f, 0.f, 0.f}, vv = kk;
            if (key < L) {
                const float *pk = Kp + (int64_t)key * a.sk[2] + col, *pv = Vp + (int64_t)key * a.sv[2] + col;
                if (col < Dt) kk.x = pk[0], vv.x = pv[0];
                if (col + 1 < Dt) kk.y = pk[1], vv.y = pv[1];
                if (col + 2 < Dt) kk.z = pk[2], vv.z = pv[2];
                if (col + 3 < Dt) kk.w = pk[3], vv.w = pv[3];
            }
            kreg[i] = f32x4_t{kk.x, kk.y, kk.z, kk.w};
            vreg[i] = f32x4_t{vv.x, vv.y, vv.z, vv.w};
        }
    };
    // a negative scale goes into Q's sign: the running maximum is then that of the raw scores (a scale of zero is refused)
    const float sc = fabsf(a.scale_log2);
    auto tile_step = [&](int kt) {
        const int k0 = kt * BN;
        if (k0 >= kv_end_wave) return;
        f32x16_t s;
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = 0.f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const float4 w = *(const float4*)(sK + ql * PITCH + 8 * c + 4 * h);
            const float kk[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kk[e], qf[c][e], s, 0, 0, 0);
        }
        if (k0 + BN - 1 > (a.causal ? min(q0 + off, L - 1) : L - 1)) {  // some query here does not see all of the tile
            const int lim = a.causal ? min(q0 + ql + off, L - 1) : L - 1;
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (k0 + 8 * (v >> 2) + 4 * h + (v & 3) > lim) s[v] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
        mx = half_swap_max(mx);
        if (__builtin_amdgcn_ballot_w64(LAG ? (mx - m_ref) * sc > lag : mx > m_ref) != 0) {
            const float m_new = fmaxf(m_ref, mx), neg_new = m_new == -INFINITY ? 0.f : -m_new * sc;
            const float alpha = m_ref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(neg_new - neg);
            m_ref = m_new;
            neg = neg_new;
            l *= alpha;
#pragma unroll
            for (int i = 0; i < DB; ++i)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[i][j] *= alpha;
        }
        float p[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            p[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], sc, neg));
            l += p[v];
        }
        // O^T += V^T . P^T : contraction slot h of step v is key 8*(v/4) + 4*h + v%4, the key p[v] belongs to
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int krow = 8 * (v >> 2) + 4 * h + (v & 3);
#pragma unroll
            for (int db = 0; db < DB; ++db)
                acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(sV[krow * PITCH + 32 * db + ql], p[v], acc[db], 0, 0, 0);
        }
    };

    auto meet = [] {  // a key group of one wavefront has its tiles to itself, and a wavefront's LDS accesses are done in order
        if constexpr (R == 1) asm volatile("" ::: "memory");
        else __syncthreads();
    };
    constexpr bool AHEAD = D <= 128;  // the widest tile has no registers left to fetch ahead into
    if (AHEAD && grp_k < n_tiles) fetch(grp_k);
    if (LAG && tid == 0) sm_again = 0;
    if (a.scale_log2 < 0.f) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) qf[c][e] = -qf[c][e];
    }
    for (;;) {  // once; twice where a sum overflowed (kLag)
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
    m_ref = -INFINITY, neg = 0.f, l = 0.f;
    for (int t0 = 0; t0 < n_tiles; t0 += G) {  // the same number of steps for every wavefront: they meet at the barriers
        const int kt = t0 + grp_k;
        meet();  // the previous tiles' readers are done
        if (kt < n_tiles) {
            if (!AHEAD) fetch(kt);
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                const int id = gt + i * (64 * R), at = id / (D / 4) * PITCH + 4 * (id % (D / 4));
                *(f32x4_t*)(sK + at) = kreg[i];
                *(f32x4_t*)(sV + at) = vreg[i];
            }
        }
        meet();
        if (AHEAD && kt + G < n_tiles) fetch(kt + G);
        if (kt < n_tiles) tile_step(kt);
    }

    l = half_swap_sum(l);
    int qi = q0 + ql;
    if constexpr (LAG) asm volatile("" : "+v"(qi));  // addresses of the output are made here and take no registers before
    float* op = (float*)a.out + (int64_t)b * a.so[0] + (int64_t)hq * a.so[1] + (int64_t)min(qi, a.T - 1) * a.so[2];
    auto store = [&](int quad, float4 o) {  // columns d = 8 quad + 4 h .. + 3
        const int d = 8 * quad + 4 * h;
        if constexpr (GEN) {
            if (d < Dt) op[d] = o.x;
            if (d + 1 < Dt) op[d + 1] = o.y;
            if (d + 2 < Dt) op[d + 2] = o.z;
            if (d + 3 < Dt) op[d + 3] = o.w;
        } else {
            *(float4*)(op + d) = o;
        }
    };
    constexpr int NQ = DB * 4, QPW = NQ / G;
    const float m_run = m_ref == -INFINITY ? -INFINITY : -neg;
    float f[G], M = m_run, lt = l;
    f[0] = 1.f;
    float4* xch = (float4*)smem_f32;  // [row group][key group][quad][lane]
    if constexpr (G > 1) {            // as in prefill_bf16_kernel
        static_assert(NQ % G == 0 && R * G * NQ * 256 <= G * 2 * TILE, "the exchange fits the tiles");
        __syncthreads();
        if (h == 0) {
            sm_m[grp_k][wave * 32 + ql] = m_run;  // -inf without a visible key
            sm_l[grp_k][wave * 32 + ql] = l;
        }
#pragma unroll
        for (int i = 0; i < NQ; ++i)
            xch[((wave * G + grp_k) * NQ + i) * 64 + lane] = float4{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
        __syncthreads();
        M = -INFINITY;
#pragma unroll
        for (int g = 0; g < G; ++g) M = fmaxf(M, sm_m[g][wave * 32 + ql]);
        lt = 0.f;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            f[g] = exp2f(sm_m[g][wave * 32 + ql] - (M == -INFINITY ? 0.f : M));
            lt += f[g] * sm_l[g][wave * 32 + ql];
        }
    }
    if (!LAG && qi >= a.T) return;
    float largest = 0.f;
    if (qi < a.T) {
        const float inv_l = lt > 0.f ? 1.0f / lt : 0.f;  // an empty context (cache mode, length 0) gives zeros
#pragma unroll
        for (int i = 0; i < QPW; ++i) {
            float4 o;
            if constexpr (G == 1) {
                o = float4{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
            } else {
                o = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const float4 x = xch[((wave * G + g) * NQ + grp_k * QPW + i) * 64 + lane];
                    o.x += f[g] * x.x, o.y += f[g] * x.y, o.z += f[g] * x.z, o.w += f[g] * x.w;
                }
            }
            if constexpr (LAG)  // (a NaN stays one)
                for (float x : {o.x, o.y, o.z, o.w}) largest = __builtin_elementwise_maximum(largest, fabsf(x));
            store(grp_k * QPW + i, float4{o.x * inv_l, o.y * inv_l, o.z * inv_l, o.w * inv_l});
        }
        if (a.lse && h == 0 && grp_k == 0)
            a.lse[(int64_t)b * a.sl[0] + (int64_t)hq * a.sl[1] + (int64_t)qi * a.sl[2]] = (M + log2f(lt)) * 0.6931471805599453f;
    }
    if (!LAG || lag == 0.f) return;
    if (!(largest < INFINITY)) sm_again = 1;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(sm_again) == 0) return;
    lag = 0.f;
    if (AHEAD && grp_k < n_tiles) fetch(grp_k);
    }
}

// ---------------------------------------------------------------------------------------------
// fp32, small grids: 16 queries per workgroup and four wavefronts, each of which takes groups of 32 keys (w, w + 4, ...) on its own, in the
// operand layouts of the decode step's fp32 kernel (v_mfma_f32_16x16x4_f32; the 16 columns are queries of one head).
// Few workgroups are bound by what one wavefront does in a row: 32 queries x 32 keys are 4096 matrix-pipe cycles at D 64, with a round
// trip through LDS and two barriers before them, while most SIMDs have nothing to do.  Here twice the workgroups exist, a group of
// keys is 2048 cycles, and K and V go from memory to the operands directly (a group has one reader), the next group's K under P V and
// its V under the following Q K^T.  What is left is the latency of the loads: a long context reaches half of the matrix pipe.
// Eight wavefronts pay more in the merge than they gain except past 4000 keys (50 for 51 us).
// Measured, us, before -> this: D 64, 8 / 2 heads, 256 tokens 10.3 -> 6.5; 16 heads, 175 tokens, not causal 10.0 -> 6.4; 32 / 8 heads, 26
// tokens after 5617 149 -> 63; D 128, 16 heads, 60 tokens 10.7 -> 6.6; 2 x 32 / 8 heads, 34 tokens after 4199 215 -> 87.
// ---------------------------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(256, 2) prefill_f32_narrow_kernel(PrefillArgs a) {
    constexpr int NW = 4;
    constexpr int C4 = D / 16;  // 16-byte pieces of a K row per lane
    constexpr int VC = D / 64;  // 16-byte pieces of a V row per lane
    constexpr int KT = 2;       // 16-key tiles of a group
    constexpr int GROUP = 16 * KT;
    __shared__ __attribute__((aligned(16))) float sm_o[NW][16][D + 4];
    __shared__ float sm_m[NW][16], sm_l[NW][16], sm_f[NW][16], sm_inv[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int bh = xcd_grouped_head(blockIdx.x, a.B * a.Hkv, a.n_rep), qt = launch_row<true>(a, (int)blockIdx.y);
    const int b = bh / a.Hq, hq = bh - b * a.Hq, kvh = hq / a.n_rep;
    const int n_chunk = a.chunk_lens ? min(max(a.chunk_lens[b], 0), a.T) : a.T;  // cache mode, as in the bf16 kernel
    const int L = a.seq_lens ? min(max(a.seq_lens[b], n_chunk), a.L) : a.L;
    const int q0 = qt * 16, off = L - n_chunk;
    const int kv_end = a.causal ? min(L, min(q0 + 15, a.T - 1) + off + 1) : L;  // keys that some query here sees
    const int lim = a.causal ? min(L, q0 + c + off + 1) : L;                   // column c sees keys [0, lim)

    const float* qrow = (const float*)a.q + (int64_t)b * a.sq[0] + (int64_t)hq * a.sq[1] + (int64_t)min(q0 + c, a.T - 1) * a.sq[2] + 4 * g;
    const float* Kp = (const float*)a.k + (int64_t)b * a.sk[0] + (int64_t)kvh * a.sk[1] + 4 * g;
    const float* Vp = (const float*)a.v + (int64_t)b * a.sv[0] + (int64_t)kvh * a.sv[1];
    float4 qf[C4], kf[KT][C4];
    f32x4_t vf[KT][4][VC];
#pragma unroll
    for (int cc = 0; cc < C4; ++cc) qf[cc] = *(const float4*)(qrow + 16 * cc);
    const int last = kv_end - 1;
    auto load_k = [&](int kbase) {  // keys past the last one are read from it and masked
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            const float* kr = Kp + (int64_t)min(kbase + 16 * t + c, last) * a.sk[2];
#pragma unroll
            for (int cc = 0; cc < C4; ++cc) kf[t][cc] = *(const float4*)(kr + 16 * cc);
        }
    };
    const int rowV = (int)a.sv[2] * 4;
    auto load_v = [&](int kbase) {  // and the V of keys past the last one are zeros: an infinity in its row must not meet their weights of 0
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(Vp + (int64_t)kbase * a.sv[2]), 0, (min(GROUP, kv_end - kbase) - 1) * rowV + 4 * D, 0x00020000);
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int vc = 0; vc < VC; ++vc)
                    vf[t][v][vc] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, (16 * t + 4 * g + v) * rowV + 16 * c + 256 * vc, 0, 0));
    };
    const float sc = fabsf(a.scale_log2);
    f32x4_t acc[4 * VC];  // acc[4 vc + e][v]: row d = 64 vc + 16 g + 4 v + e of O^T, column c
    float m_ref = -INFINITY, neg = 0.f, l = 0.f;  // as in prefill_f32_kernel
#pragma unroll
    for (int i = 0; i < 4 * VC; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (a.scale_log2 < 0.f) {
#pragma unroll
        for (int cc = 0; cc < C4; ++cc) qf[cc] = float4{-qf[cc].x, -qf[cc].y, -qf[cc].z, -qf[cc].w};
    }
    // the loop stands inside the condition of its first loads: with operands that a path around them leaves unset, the register allocator
    // has let an MFMA's result overwrite the V pieces that the next ones read (found in the assembly of an earlier form)
    if (int kbase = wave * GROUP; kbase < kv_end) {
        load_k(kbase);
        load_v(kbase);
        for (;;) {
            const int next = kbase + NW * GROUP;
            f32x4_t s[KT];
#pragma unroll
            for (int t = 0; t < KT; ++t) {
                s[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int cc = 0; cc < C4; ++cc) {
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][cc].x, qf[cc].x, s[t], 0, 0, 0);
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][cc].y, qf[cc].y, s[t], 0, 0, 0);
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][cc].z, qf[cc].z, s[t], 0, 0, 0);
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][cc].w, qf[cc].w, s[t], 0, 0, 0);
                }
            }
            if (next < kv_end) load_k(next);
            if (kbase + GROUP > (a.causal ? min(L, q0 + off + 1) : L)) {  // some column does not see all of the group
#pragma unroll
                for (int t = 0; t < KT; ++t)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (kbase + 16 * t + 4 * g + v >= lim) s[t][v] = -INFINITY;
            }
            float mx = s[0][0];
#pragma unroll
            for (int t = 0; t < KT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) mx = fmaxf(mx, s[t][v]);
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            if (__builtin_amdgcn_ballot_w64(mx > m_ref) != 0) {  // the running maximum: kLag saves this kernel's short calls nothing
                const float m_new = fmaxf(m_ref, mx), neg_new = m_new == -INFINITY ? 0.f : -m_new * sc;
                const float alpha = m_ref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(neg_new - neg);
                m_ref = m_new;
                neg = neg_new;
                l *= alpha;
#pragma unroll
                for (int i = 0; i < 4 * VC; ++i) acc[i] *= alpha;
            }
#pragma unroll
            for (int t = 0; t < KT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    s[t][v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][v], sc, neg));
                    l += s[t][v];
                }
#pragma unroll
            for (int t = 0; t < KT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int vc = 0; vc < VC; ++vc) {
                        acc[4 * vc] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t][v][vc][0], s[t][v], acc[4 * vc], 0, 0, 0);
                        acc[4 * vc + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t][v][vc][1], s[t][v], acc[4 * vc + 1], 0, 0, 0);
                        acc[4 * vc + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t][v][vc][2], s[t][v], acc[4 * vc + 2], 0, 0, 0);
                        acc[4 * vc + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t][v][vc][3], s[t][v], acc[4 * vc + 3], 0, 0, 0);
                    }
            if (next >= kv_end) break;
            load_v(next);
            kbase = next;
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);

    // the wavefronts' (m, l, O^T) meet in LDS; a wavefront without a visible key has m = -inf, l = 0 and the weight 0
    float* mine = sm_o[wave][c];
#pragma unroll
    for (int vc = 0; vc < VC; ++vc)
#pragma unroll
        for (int v = 0; v < 4; ++v) *(float4*)(mine + 64 * vc + 16 * g + 4 * v) = float4{acc[4 * vc][v], acc[4 * vc + 1][v], acc[4 * vc + 2][v], acc[4 * vc + 3][v]};
    if (g == 0) {
        sm_m[wave][c] = m_ref == -INFINITY ? -INFINITY : -neg;
        sm_l[wave][c] = l;
    }
    __syncthreads();
    if (tid < 16) {
        float M = -INFINITY, lt = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) M = fmaxf(M, sm_m[w][tid]);
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = exp2f(sm_m[w][tid] - (M == -INFINITY ? 0.f : M));
            sm_f[w][tid] = f;
            lt += f * sm_l[w][tid];
        }
        sm_inv[tid] = lt > 0.f ? 1.0f / lt : 0.f;  // an empty context (cache mode, length 0) gives zeros
        if (a.lse && q0 + tid < a.T)
            a.lse[(int64_t)b * a.sl[0] + (int64_t)hq * a.sl[1] + (int64_t)(q0 + tid) * a.sl[2]] = (M + log2f(lt)) * 0.6931471805599453f;
    }
    __syncthreads();
    for (int i = tid; i < 16 * (D / 4); i += 64 * NW) {
        const int row = i / (D / 4), d = 4 * (i % (D / 4));
        if (q0 + row >= a.T) continue;
        f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) o += sm_f[w][row] * *(const f32x4_t*)(sm_o[w][row] + d);
        *(f32x4_t*)((float*)a.out + (int64_t)b * a.so[0] + (int64_t)hq * a.so[1] + (int64_t)(q0 + row) * a.so[2] + d) = o * sm_inv[row];
    }
}

int check_tensor4(const vsp_tensor* t, int esz) {
    if (t->stride[3] != 1) return VSP_ERR_STRIDE;
    if (!t->data) return VSP_ERR_NULL;
    if (!is_aligned16(t->data)) return VSP_ERR_ALIGN;
    for (int i = 0; i < 3; ++i)
        if ((t->stride[i] * esz) % 16 != 0) return VSP_ERR_ALIGN;
    return VSP_OK;
}

// fp32 tensors whose head_dim is not one of the native tiles: element-wise access, so 4-byte alignment is all it takes
int check_tensor4_any_d(const vsp_tensor* t) {
    if (t->stride[3] != 1) return VSP_ERR_STRIDE;
    if (!t->data) return VSP_ERR_NULL;
    if ((reinterpret_cast<uintptr_t>(t->data) & 3u) != 0) return VSP_ERR_ALIGN;
    return VSP_OK;
}
bool native_head_dim(int dtype, int64_t D) { return D == 64 || D == 128 || (D == 32 && dtype == VSP_F32); }
// the fp32 kernels' tile width for a head_dim they do not hold natively (0: none)
int64_t padded_head_dim(int dtype, int64_t D) {
    if (dtype != VSP_F32 || D < 1 || D > 256) return 0;
    return D <= 32 ? 32 : D <= 64 ? 64 : D <= 128 ? 128 : 256;
}

// Where the order of a grid's rows turns from falling to rising weight (launch_row).  Heaviest first lets the short workgroups of a causal grid
// fill the ends, but where all of them are on the chip at once nothing waits, and what counts is which two share a CU: the one that comes after the first round
// of a workgroup per CU joins the one of its place in that round, so the second round's lightest goes to the heaviest.  us, all falling -> turned: bf16, D 128, prompts
// of 32/8 heads, 777 tokens 20.5 -> 19.8, 2048 52.1 -> 51.3, 16/4, 4000 84.5 -> 82.9; forward, 32/8, 2048 42.8 -> 41.3, 64/8, 900 22.6 -> 21.9; fp32 tensors on the
// bf16 cores, forward and backward, 2048 487.4 -> 481.2; exact fp32, D 64, 8/2, 700 14.5 -> 13.0, 2000 55.9 -> 46.2, 12, 1229 37.5 -> 32.2; D 128, 16, 500 24.9 -> 21.0,
// 32/8, 256 15.6 -> 14.1.  Grids of two to three workgroups per CU, which wait: bf16, 32/8, 2 x 1500 44.4 -> 46.4, 16/4, 4 x 1300 33.1 -> 38.0; exact fp32, D 64, 3 x 8/2, 400
// 13.2 -> 14.7.  bf16 with one row group, whose chains are a fourth as long: 32/8, 400 12.3 -> 12.5; bf16 at D 64, whose CUs hold more: no difference.
// A row of tiles that straddles the first round spoils the pairs, so the turn may fall before it or behind it, or nowhere: whichever leaves the heaviest CU lightest.
int64_t heaviest_pair(int64_t n_qtiles, int64_t per_row, int64_t fold) {   // in tiles of the heaviest workgroup's n_qtiles
    const int64_t cus = device_cu_count();
    auto weight = [&](int64_t row) { return row < fold ? n_qtiles - row : row - fold + 1; };
    int64_t worst = n_qtiles;
    for (int64_t row = cus / per_row; row < n_qtiles; ++row)
        worst = std::max(worst, weight(row) + weight((std::max(row * per_row, cus) - cus) / per_row));
    return worst;
}
int launch_fold(int64_t n_qtiles, int64_t per_row) {
    const int64_t cus = device_cu_count(), before = std::max<int64_t>(1, cus / per_row), behind = ceil_div(cus, per_row);
    if (n_qtiles * per_row <= cus || n_qtiles * per_row > 2 * cus) return (int)n_qtiles;
    int64_t best = n_qtiles;
    for (const int64_t fold : {behind, before})
        if (fold < n_qtiles && heaviest_pair(n_qtiles, per_row, fold) < heaviest_pair(n_qtiles, per_row, best)) best = fold;
    return (int)best;
}

template <int DP, bool GEN, int R, int G, bool LAG>
int launch_prefill_f32_instance(PrefillArgs a, hipStream_t st) {
    constexpr size_t lds = (size_t)G * 2 * 32 * (DP + 8) * sizeof(float);
    if constexpr (lds > 65536) {  // beyond the default limit of a launch: raised once per process
        static const hipError_t e = hipFuncSetAttribute((const void*)prefill_f32_kernel<DP, GEN, R, G, LAG>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            set_hip_error(e);
            return VSP_ERR_LAUNCH;
        }
    }
    a.n_qtiles = (int)ceil_div(a.T, 32 * R);
    const int64_t blocks = (int64_t)a.n_qtiles * a.B * a.Hq;
    if (blocks > INT32_MAX) return VSP_ERR_ARG;
    if (a.causal) a.causal = (DP <= 64 || (DP == 128 && R == 4)) ? launch_fold(a.n_qtiles, (int64_t)a.B * a.Hq) : a.n_qtiles;
    hipLaunchKernelGGL((prefill_f32_kernel<DP, GEN, R, G, LAG>), dim3((unsigned)blocks), dim3(64 * R * G), lds, st, a);
    return check_launch();
}

template <int DP, bool GEN, int R, int G>
int launch_prefill_f32_shape(const PrefillArgs& a, hipStream_t st) {
    if constexpr (!GEN) {  // (the element-wise fetch leaves no registers for a second round)
        if (a.L > 32 * (kLagTiles - 1)) return launch_prefill_f32_instance<DP, GEN, R, G, true>(a, st);
    }
    return launch_prefill_f32_instance<DP, GEN, R, G, false>(a, st);
}

// Where 16-query workgroups pay (prefill_f32_narrow_kernel): their rows of K and V are read once per 16 queries, so the CUs must not
// have to take turns.  One workgroup per CU always gains.  Beyond that (us, the other shapes' best -> narrow, w workgroups per CU):
// a causal grid without context (L == T), whose short workgroups fill the gaps of the long ones, to the w that two or three of them side by
//   side hold: D 64, 8 x 16 heads, 64 tokens, w 2.0 6.9 -> 6.6, 6 x 32, w 3.0 7.0 -> 7.4; 32 heads, 300 tokens, w 2.4 13.7 -> 12.2; 2 x 32, 200,
//   w 3.25 12.0 -> 11.3, 256, w 4.0 12.9 -> 14.1; D 128, 4 x 32, 64, w 2.0 11.4 -> 10.2, 6 x 32, 42, w 2.25 10.9 -> 12.8; 2 x 32, 160, w 2.5
//   20.1 -> 15.3, 256, w 4.0 26.2 -> 26.3;
// others while the four wavefronts have a single turn, L below 128, and two workgroups a CU: D 128, 4 x 32 heads, 42 tokens, w 1.5
//   10.7 -> 9.7; D 64 6.8 -> 6.2; but 200 tokens, not causal, w 1.6 16.9 -> 18.0, and 48 tokens after 952, w 1.5 45.7 -> 58.9.
bool f32_narrow_pays(const PrefillArgs& a, int64_t D) {
    const int64_t cus = device_cu_count(), blocks = ceil_div(a.T, 16) * a.B * a.Hq;
    if (blocks <= cus) return true;
    if (a.causal && a.T == a.L) return 2 * blocks <= ((D == 64 ? 5 : 4) + (a.T > 128 ? 1 : 0)) * cus;
    return a.L < 128 && blocks <= 2 * cus;
}

template <int D>
int launch_prefill_f32_narrow(PrefillArgs a, hipStream_t st) {
    a.n_qtiles = (int)ceil_div(a.T, 16);
    if (a.causal) a.causal = launch_fold(a.n_qtiles, (int64_t)a.B * a.Hq);
    hipLaunchKernelGGL((prefill_f32_narrow_kernel<D>), dim3((unsigned)(a.B * a.Hq), (unsigned)a.n_qtiles), dim3(256), 0, st, a);
    return check_launch();
}

// Every tile costs its wavefront 2 D MFMAs of 64 cycles, so what counts is how evenly the tiles spread over the SIMDs, and beside
// that what a workgroup costs to start and to merge (`fixed`, in tiles; paid again in every round, in full where only one or two
// workgroups fit a CU's LDS, D 128; not where a causal grid's short workgroups hide it).  The three shapes' times are estimated from the
// workgroups per CU, how many of them a CU holds, their tiles (a causal grid: the mean of its rows, the heaviest first; while all are on
// the chip, what lands on the CU of the heaviest: of two workgroups at most the heaviest pair, but not less than a fitted 1 + 0.6 (2 - x) of the longest chain, x to a CU) and the
// time per tile: D 128 runs two 128-query workgroups beside one another (0.92) and one of
// the others; D 64 takes 1.17 where a SIMD has a single wavefront.  The cheapest is taken: within 3 % of the best of the three in all
// but one of 115 shapes measured, us, R 1 / 2 / 4: D 64: 8 / 2 heads, 1115 tokens of context 26 / 47 / 81; 16 heads, 1775 tokens, batch 4
// 236 / 222 / 254; 4 heads, 4000 tokens, not causal 142 / 157 / 279; D 128: 32 heads, 777 tokens 78 / 65 / 108; 2 x 32 heads, 2048 tokens
// 744 / 674 / 554 (the turned order moved 32 / 8, 2000 tokens from R 2 to R 4, 336 -> 285, and 2 x 900 164 -> 151); 32 heads, 512 tokens after 3488 296 / 310 / 524.
template <int DP, bool GEN>
int launch_prefill_f32(const PrefillArgs& a, hipStream_t st) {
    if constexpr (!GEN && DP >= 64) {
        if (f32_narrow_pays(a, DP)) return launch_prefill_f32_narrow<DP>(a, st);
    }
    if constexpr (DP <= 128) {
        const int64_t cus = device_cu_count(), tiles = ceil_div(a.L, 32);
        const bool triangle = a.causal && a.T == a.L;
        auto cost = [&](int R, int G, int resident, double rate, double alone, double fixed) {
            const double x = (double)(ceil_div(a.T, 32 * R) * a.B * a.Hq) / (double)cus;  // workgroups per CU
            const double whole = (double)((int64_t)x + ((double)(int64_t)x < x ? 1 : 0)), full = (double)ceil_div(tiles, G);
            double rounds = triangle || x > resident ? x : whole, work;
            if (triangle) {  // the mean of the rows; not less than what lands on the CU of the heaviest rows at the start
                double first = 0;
                if (x > 1 && x <= 2 && resident >= 2) {  // two to a CU, paired by launch_fold
                    const int64_t n_q = ceil_div(a.T, 32 * R), per_row = (int64_t)a.B * a.Hq;
                    const double pair = (double)heaviest_pair(n_q, per_row, launch_fold(n_q, per_row)) / (double)n_q, slow = 1 + 0.6 * (2 - x);
                    first = full * (pair > slow ? pair : slow);
                } else {
                    for (int k = 0; k < resident && k < whole; ++k) first += full * (1 - k / x);
                }
                work = rounds * (full + 1) / 2 + full / 4;
                if (work < first) work = first;
            } else {
                if (x > resident) rounds = (x + whole) / 2;
                work = rounds * full;
            }
            const double start = DP == 128 ? (rounds > 1 ? rounds : 1) : rounds > 1 ? (triangle ? 0.75 + 0.25 * rounds : 0.3 + 0.7 * rounds) : 1;
            return (work + fixed * start) * (x <= 1 ? alone : rate);
        };
        double c1, c2, c4;
        if (DP == 128) c1 = cost(1, 4, 1, 1, 1, 1.1), c2 = cost(2, 2, 1, triangle ? 1.02 : 1.04, triangle ? 1.02 : 1.04, 0.9), c4 = cost(4, 1, 2, 0.92, 0.92, 0.5);
        else c1 = cost(1, 4, 2, 1, 1.17, 1.5), c2 = cost(2, 2, 3, 1, 1.17, 1.3), c4 = cost(4, 1, 4, 1, 1.08, 0.9);
        if (GEN) c1 *= 1.25, c2 *= 1.05;  // element by element, the loads are work of their own: each tile has 4 / R rows per thread to fetch
        if (c1 < c2 && c1 < c4) return launch_prefill_f32_shape<DP, GEN, 1, 4>(a, st);
        if (c2 < c4) return launch_prefill_f32_shape<DP, GEN, 2, 2>(a, st);
    }
    return launch_prefill_f32_shape<DP, GEN, 4, 1>(a, st);
}

// Which bf16 kernel a call runs, and into how many shares its context is cut.
// pipe: the software-pipelined kernel (D = 128; 128 rows per workgroup, the fastest steady state).  Otherwise the general
// kernel with R row groups and G key groups.  n_splits > 1: shares of split_tiles key tiles, merged by the combine kernel.
// pack: a workgroup's rows are all heads' of a kv head.
struct PrefillPlan {
    int R, G;
    bool pipe;
    int n_splits, split_tiles;
    bool pack;
};
// A full grid is bound by its throughput, which is best with four row groups and, once contexts pay for filling and draining a pipeline, with the pipelined
// kernel; a grid that leaves the chip idle is bound by the chain of key tiles of its longest workgroup, which key groups cut and shares of the context, at the
// price of more K / V traffic per row and of the launch that merges the shares; few rows over a long context are bound by reading it.  The shape with the least
// estimate runs.  An estimate is no time (it is 0.55 to 0.7 of one from 15 us on, and 3 to 6 us less than one below): its constants were fitted to the
// order of the shapes alone.  Start + the root of the sum of the squares of
//   chain: tiles of the longest workgroup / G, at `chain` a tile,
//   work: workgroups per CU (in whole rounds of what a CU holds where their chains are about equal) x (their mean tiles / G + fill, and half a tile with key
//   groups), at `work` a tile, and
//   K and V once from memory,
// and with shares the merge's launch and the partial rows' traffic.  Fitted to 250 drawn shapes (prompts, chunks and plain calls of more than 128 tokens), each run as
// every shape and, over a cache, in 1 to 32 shares.  On 774 others the choice was 1.3 % (D 128) and 1.4 % (D 64) from the best of them on average, more than 5 % for a tenth,
// and at worst 31 % (3 x 32 heads, 58 tokens of 4794: 61.1 in two shares of 32-row workgroups, 46.5 whole) and 50 % (D 64, 12 heads, 26 tokens of 4500: 19.9 in 16 shares, 13.2 in 8).
// Constants fitted to all of these were no better on 373 more (mean 1.00, 0.86 to 1.12 of this choice's time), nor was a term for rounds in which some CUs have a workgroup more
// than others (1.004, 0.89 to 1.15): what is left is not in the sum's form.
// us, R 1 / R 2 / R 4 / pipelined: D 128, 32 / 8 heads: 777 tokens (prompt) 20.8 / 20.4 / 25.3 / 24.3, 2 x 3109 261 / 216 / 190 / 185; 16 heads, 5 x 901 48.9 / 37.9 / 29.4 / 32.3;
// 45 tokens after 1266, 64 / 8 17.1 / 20.2 / 22.6 / 23.0 (in 1, 4, 8, 4 shares); 512 after 32256, 32 / 8 418 / 337 / 309 / 265; D 64: 16 heads, 2 x 1500, not causal 34.2 / 28.3 / 32.1;
// 8 / 2, 3 x 3986 78.7 / 65.9 / 69.1; 113 after 9542, 2 x 8 / 2 22.1 / 23.5 / 25.4 (in 8, 8, 16 shares).
// Short contexts are a launch and one chain of memory latencies: 128 rows of one head a workgroup, whose wavefronts past the last row have nothing to do, spread a
// call over the most CUs (not packed; a kv head's workgroups still on one XCD: in the heads' own order 4 x 64 / 8 heads, 64 tokens took 6.2 instead of 5.3, 4 x 128 10.1 instead of
// 8.8, a prompt of 4 x 45 10.8 instead of 9.8): 4 x 32 tokens, D 128, 32 / 8 heads 4.0, with the group's rows packed 5.9 (R 4), 5.4 (R 1); three and four tiles only
// where 32-row workgroups do not fit the CUs at once: 2 x 74, 64 / 8 6.0, packed 7.0 (R 1), 6.5 (R 2).  rope (a prompt whose Q is rotated in the kernel): 32 rows a workgroup from two
// tiles on, where they are rotated once through LDS: 62 tokens, 32 heads 9.0, not 10.0.
// Partials take at most kPartialBytes: their room is a block that the Python view keeps for the stream, and without the bound a large batch's would be gigabytes.  Shapes that it
// changes, us, as many shares as the estimate likes -> in the bound: D 64, 32 / 8 heads, 1186 tokens after 31236 387 -> 379, 3 x 16, 1536 after 20925 505 -> 505; D 128, 3 x 64 / 8,
// 714 after 6633 (Q8_0) 554 -> 522.
constexpr float kPartialBytes = 140e6f;
constexpr int64_t kMostShares = 32;
// Row numbers are 32-bit integers that are added to: more rows than this stay with their own head (which has fewer: T is checked at the entry points).
constexpr int64_t kMaxRows = INT32_MAX / 2;
// max_shares: of the context, as many as there is room for (1: it stays whole).
PrefillPlan plan_prefill(int64_t B, int64_t Hkv, int64_t n_rep, int64_t T, int64_t L, int64_t D, bool causal, bool pipe_ok, bool pipe_splits, int64_t max_shares, bool rope) {
    const int64_t tiles = ceil_div(L, kUnit), rows = T * n_rep, groups = B * Hkv;
    const int64_t ncu = device_cu_count();
    if (tiles <= 2) return rope && tiles == 2 && ceil_div(T, 32) * groups * n_rep <= 2 * ncu ? PrefillPlan{1, 4, false, 1, 0, false} : PrefillPlan{4, 1, false, 1, 0, false};
    if (tiles <= 4 && T == L && !rope && ceil_div(rows, 32) * groups > ncu && groups * n_rep <= ncu) return {4, 1, false, 1, 0, false};
    struct Cost {
        int R, resident;   // workgroups a CU holds
        bool pipe;
        float chain, work, start, fill;
    };
    static const Cost k128[] = {{1, 2, false, 0.79f, 0.707f, -1.9f, 1.9f}, {2, 2, false, 0.629f, 0.422f, 0.13f, 2.07f}, {4, 3, false, 0.485f, 0.295f, 0.34f, 1.55f}, {4, 2, true, 0.351f, 0.286f, 2.5f, 2.98f}};
    static const Cost k64[] = {{1, 4, false, 0.52f, 0.233f, 0.2f, 1.48f}, {2, 4, false, 0.352f, 0.18f, 0.74f, 1.73f}, {4, 4, false, 0.328f, 0.133f, 0.31f, -0.32f}};
    const Cost* costs = D == 128 ? k128 : k64;
    const float merge = D == 128 ? 2.2f : 2.3f, partials = D == 128 ? 3.7e6f : 5.3e6f;   // us; bytes per us
    const float kv = (float)groups * (float)L * (float)(4 * D) / (D == 128 ? 6.5e6f : 3.4e6f);
    const float mean_tiles = (float)tiles - (causal ? 0.5f * (float)T / kUnit : 0.f);
    const float share_bytes = (float)(rows * groups) * (float)((D + 2) * (int64_t)sizeof(float));   // partials of one share
    const int64_t most = std::max<int64_t>(1, std::min({kMostShares, max_shares, (int64_t)(kPartialBytes / std::max(share_bytes, 1.f))}));
    PrefillPlan best{4, 1, false, 1, 0, rows <= kMaxRows};
    float least = INFINITY;
    for (int i = 0; i < (D == 128 ? 4 : 3); ++i) {
        const Cost& c = costs[i];
        if (c.pipe && !pipe_ok) continue;
        const float wgs = (float)(ceil_div(rows, 32 * c.R) * groups) / (float)ncu;   // per CU
        const int G = 4 / c.R;
        for (int64_t want = 1; want <= most; want = want < most ? std::min(2 * want, most) : most + 1) {
            if (want > 1 && ((c.pipe && !pipe_splits) || 4 * want > tiles)) break;
            const int64_t share = ceil_div(tiles, want), n = ceil_div(tiles, share);
            const float chain = (float)ceil_div(share, G) * c.chain;
            float all = wgs * (float)n;
            if (all > (float)c.resident && mean_tiles >= 0.75f * (float)tiles) all = ceilf(all / (float)c.resident) * (float)c.resident;   // equal chains: whole rounds
            const float work = all * (mean_tiles / (float)(n * G) + (G > 1 ? 0.5f : 0.f) + c.fill) * c.work;
            const float us = c.start + sqrtf(chain * chain + work * work + kv * kv) + (n > 1 ? merge + 2.f * (float)n * share_bytes / partials : 0.f);
            if (us < least) {
                least = us;
                best.R = c.R, best.G = G, best.pipe = c.pipe;
                best.n_splits = (int)n, best.split_tiles = n > 1 ? (int)share : 0;
            }
        }
    }
    return best;
}
size_t plan_partial_bytes(const PrefillPlan& p, int64_t B, int64_t Hq, int64_t T, int64_t D) {
    return p.n_splits > 1 ? (size_t)B * (size_t)Hq * (size_t)T * (size_t)p.n_splits * (size_t)(D + 2) * sizeof(float) : 0;
}

// bf16, over cache planes or dense K/V
int launch_prefill_bf16(PrefillArgs& a, int64_t D, bool cache_planes, const PrefillPlan& p, hipStream_t st) {
    a.pack = p.pack ? a.n_rep : 1;
    const int64_t rows = (int64_t)a.T * a.pack, groups = a.Hq / a.pack;
    a.n_splits = p.n_splits;
    a.split_tiles = p.split_tiles;
    a.by_bh = FastDiv::of(a.B * groups), a.by_bkv = FastDiv::of((int64_t)a.B * a.Hkv), a.by_kv = FastDiv::of(a.Hkv), a.by_pack = FastDiv::of(a.pack);
    auto launch = [&](auto r, auto planes, auto rope) -> int {
        constexpr int R = decltype(r)::value;
        constexpr bool VBLK = decltype(planes)::value, ROPE = decltype(rope)::value;
        a.n_qtiles = (int)ceil_div(rows, 32 * R);
        const int64_t blocks = (int64_t)a.n_qtiles * a.B * groups * p.n_splits;
        if (blocks > INT32_MAX || rows > kMaxRows) return VSP_ERR_ARG;
        a.by_share = FastDiv::of(blocks / p.n_splits);
        if (a.causal) a.causal = D == 128 && p.n_splits == 1 && R > 1 ? launch_fold(a.n_qtiles, a.B * groups) : a.n_qtiles;
        const dim3 grid((unsigned)blocks);
        if (p.pipe) {
            if constexpr (R == 4) {
                if (D != 128) return VSP_ERR_UNSUPPORTED;
                hipLaunchKernelGGL((prefill_bf16_pipe_kernel<VBLK, ROPE>), grid, dim3(256), 0, st, a);
                return check_launch();
            }
            return VSP_ERR_UNSUPPORTED;
        }
        auto general = [&](auto d) {
            constexpr int DD = decltype(d)::value, kR = ROPE ? kRope : 0;
            if (R == 4 && p.n_splits <= 1) hipLaunchKernelGGL((prefill_bf16_kernel<DD, VBLK, 4, 1, kR>), grid, dim3(256), 0, st, a);
            else hipLaunchKernelGGL((prefill_bf16_kernel<DD, VBLK, R, 4 / R, kSplit | kR>), grid, dim3(256), 0, st, a);
        };
        if (D == 128) general(std::integral_constant<int, 128>{});
        else general(std::integral_constant<int, 64>{});
        return check_launch();
    };
    return with_row_groups<4, 2, 1>(p.R, [&](auto r) {
        if (cache_planes) return a.rope_table ? launch(r, std::true_type{}, std::true_type{}) : launch(r, std::true_type{}, std::false_type{});
        return a.rope_table ? launch(r, std::false_type{}, std::true_type{}) : launch(r, std::false_type{}, std::false_type{});
    });
}

int launch_prefill(PrefillArgs a, int dtype, int64_t D, bool cache_planes, void* stream) {
    const int64_t blocks = (int64_t)a.n_qtiles * a.B * a.Hq;
    if (blocks > INT32_MAX) return VSP_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == VSP_BF16) {
        // the software-pipelined kernel over dense K/V takes one context length for the batch; per-row lengths (a Q8_0
        // cache read out into the workspace) stay with the general kernel
        const bool pipe_ok = D == 128 && (cache_planes || (!a.seq_lens && !a.chunk_lens));
        PrefillArgs x = a;
        return launch_prefill_bf16(x, D, cache_planes, plan_prefill(a.B, a.Hkv, a.n_rep, a.T, a.L, D, a.causal != 0, pipe_ok, false, 1, false), st);
    } else {
        if (a.L == 1) a.sv[2] = D;  // any pitch will do
        // the native tiles address 32 rows of K or V with 31-bit offsets and count on rows of V past the end lying past the last row
        auto rows_ok = [&](int64_t stride) { return stride >= D && stride <= (1 << 23); };
        if (!a.elementwise && (a.sk[2] == 0 || rows_ok(a.sk[2])) && rows_ok(a.sv[2])) {
            if (D == 128) return launch_prefill_f32<128, false>(a, st);
            if (D == 64) return launch_prefill_f32<64, false>(a, st);
            if (D == 32) return launch_prefill_f32<32, false>(a, st);
        }
        switch (padded_head_dim(dtype, D)) {  // a.D_true == D
            case 32: return launch_prefill_f32<32, true>(a, st);
            case 64: return launch_prefill_f32<64, true>(a, st);
            case 128: return launch_prefill_f32<128, true>(a, st);
            case 256: return launch_prefill_f32<256, true>(a, st);
            default: return VSP_ERR_UNSUPPORTED;
        }
    }
    return check_launch();
}

}  // namespace

int check_kv_cache(const vsp_kv_cache* c);  // kv_cache.hip
int kv_append_rotated(vsp_kv_cache* cache, const vsp_tensor* q, const vsp_tensor* new_k, const vsp_tensor* new_v, const float* rope_table,
                      int64_t table_len, int64_t start_pos, void* dense_k, void* dense_v, bool* dense_written, void* stream);

}  // namespace vsp

using namespace vsp;

namespace {
// The host-side bound of the context lengths a cached-prefill call is planned on: max_len when given, else the
// cache's own length, or its capacity when the lengths live on the device.
int64_t cached_len_bound(const vsp_kv_cache* cache, bool with_seq_lens, int32_t max_len) {
    if (max_len > 0) return std::min<int64_t>(max_len, cache->S_max);
    return with_seq_lens ? cache->S_max : cache->len;
}
}  // namespace

extern "C" size_t vsp_attn_prefill_cached_workspace_bytes(const vsp_kv_cache* cache, int with_seq_lens, int32_t max_len) {
    if (!cache || cache->format != VSP_KV_Q8_0 || max_len < 0) return 0;
    const int64_t rows = cached_len_bound(cache, with_seq_lens != 0, max_len);
    return (size_t)2 * (size_t)cache->B * (size_t)cache->Hkv * (size_t)rows * (size_t)cache->D * 2;  // K and V, bf16
}

namespace {
// What a Q8_0 cache's dequantised rows take at the head of the workspace (0 for the other formats); partials follow.
size_t plan_base_bytes(const vsp_kv_cache* cache, bool with_seq_lens, int32_t max_len) {
    return (vsp_attn_prefill_cached_workspace_bytes(cache, with_seq_lens, max_len) + 255) / 256 * 256;
}
PrefillPlan plan_cached(const vsp_kv_cache* cache, int64_t Hq, int64_t T, int64_t L, bool ragged, int64_t max_shares, bool rope = false) {
    const bool planes = cache->format == VSP_KV_BF16;
    return plan_prefill(cache->B, cache->Hkv, Hq / cache->Hkv, T, L, cache->D, true, cache->D == 128 && (planes || !ragged), planes, max_shares, rope);
}
}  // namespace

// For shares of at least 16 tiles (512 keys): as many as the plan takes of them, and not fewer than it takes to reach two workgroups of 128 queries of one head per CU.
extern "C" size_t vsp_attn_prefill_cached_split_workspace_bytes(const vsp_kv_cache* cache, int with_seq_lens, int32_t max_len,
                                                                int32_t Hq, int32_t T) {
    if (!cache || Hq <= 0 || T <= 0 || max_len < 0 || cache->format != VSP_KV_BF16 || cache->D != 128 || cache->B <= 0 || cache->Hkv <= 0 || Hq < cache->Hkv) return 0;
    const int64_t L = cached_len_bound(cache, with_seq_lens != 0, max_len), tiles = ceil_div(L, kUnit), most = std::min<int64_t>(tiles / 16, 64);
    if (most <= 1) return 0;
    PrefillPlan p = plan_cached(cache, Hq, T, L, with_seq_lens != 0, most);
    const int64_t workgroups = ceil_div(T, kBM) * cache->B * Hq, slots = 2 * (int64_t)device_cu_count();
    if (2 * workgroups <= slots) p.n_splits = std::max(p.n_splits, (int)ceil_div(tiles, ceil_div(tiles, std::min(ceil_div(slots, workgroups), most))));
    return plan_partial_bytes(p, cache->B, Hq, T, cache->D);
}

extern "C" size_t vsp_attn_prefill_cached_best_workspace_bytes(const vsp_kv_cache* cache, int with_seq_lens, int32_t max_len,
                                                               int32_t Hq, int32_t T) {
    if (!cache || Hq <= 0 || T <= 0 || max_len < 0 || cache->format == VSP_KV_F32 || cache->Hkv <= 0 || Hq < cache->Hkv) return 0;
    const int64_t L = cached_len_bound(cache, with_seq_lens != 0, max_len);
    const PrefillPlan p = plan_cached(cache, Hq, T, L, with_seq_lens != 0, kMostShares);
    const size_t part = plan_partial_bytes(p, cache->B, Hq, T, cache->D);
    return part ? plan_base_bytes(cache, with_seq_lens != 0, max_len) + part
                : vsp_attn_prefill_cached_workspace_bytes(cache, with_seq_lens, max_len);
}

extern "C" int vsp_attn_prefill_cached_plan(const vsp_kv_cache* cache, int with_seq_lens, int32_t max_len, int32_t Hq, int32_t T, int prompt,
                                            vsp_attn_plan* plan) {
    if (!cache || !plan) return VSP_ERR_NULL;
    if (cache->format == VSP_KV_F32 || (cache->D != 64 && cache->D != 128)) return VSP_ERR_UNSUPPORTED;
    if (cache->B <= 0 || cache->Hkv <= 0 || Hq <= 0 || Hq % cache->Hkv != 0 || T <= 0) return VSP_ERR_SHAPE;
    if (max_len < 0 || T > INT32_MAX / 2) return VSP_ERR_ARG;
    const int64_t L = prompt ? T : cached_len_bound(cache, with_seq_lens != 0, max_len);
    if (T > L) return VSP_ERR_SHAPE;
    const PrefillPlan p = plan_cached(cache, Hq, T, L, with_seq_lens != 0, kMostShares, prompt != 0);
    *plan = vsp_attn_plan{p.R, p.G, p.pipe, p.pack, p.n_splits};
    return VSP_OK;
}

extern "C" int vsp_kv_read(const vsp_kv_cache* cache, int64_t start, int64_t count, vsp_tensor* k_out, vsp_tensor* v_out,
                           void* stream);

// rope_table: Q is a prompt's own, not rotated yet (row t at position t).  dense_ready: the workspace holds the rows of a Q8_0 cache already
static int prefill_cached(const vsp_tensor* q, const vsp_kv_cache* cache, const int32_t* seq_lens, int32_t max_len, const int32_t* chunk_lens,
                          vsp_tensor* out, vsp_tensor* lse, float scale, int is_causal, void* workspace, size_t workspace_bytes, void* stream,
                          const float* rope_table, bool dense_ready) {
    if (!q || !out) return VSP_ERR_NULL;
    int rc = check_kv_cache(cache);
    if (rc != VSP_OK) return rc;
    if (q->ndim != 4 || out->ndim != 4) return VSP_ERR_NDIM;
    const int64_t B = q->shape[0], Hq = q->shape[1], T = q->shape[2], D = q->shape[3];
    const int64_t Hkv = cache->Hkv;
    if (B != cache->B || D != cache->D) return VSP_ERR_SHAPE;
    if (Hkv <= 0 ? Hq != 0 : (Hq % Hkv != 0)) return VSP_ERR_SHAPE;
    // the bound every plan below is made on; device-side lengths are clamped to it inside the kernels, a host-side
    // length above it is a caller error (as in vsp_attn_decode)
    if (max_len < 0 || max_len > cache->S_max) return VSP_ERR_ARG;
    if (!seq_lens && max_len > 0 && cache->len > max_len) return VSP_ERR_ARG;
    const int64_t L = cached_len_bound(cache, seq_lens != nullptr, max_len);
    if (T > L) return VSP_ERR_SHAPE;                          // the chunk is part of the context
    for (int i = 0; i < 4; ++i)
        if (out->shape[i] != q->shape[i]) return VSP_ERR_SHAPE;
    if (out->dtype != q->dtype) return VSP_ERR_DTYPE;
    if (q->dtype != (cache->format == VSP_KV_F32 ? VSP_F32 : VSP_BF16)) return VSP_ERR_DTYPE;
    if (lse) {
        if (lse->ndim != 3 || lse->shape[0] != B || lse->shape[1] != Hq || lse->shape[2] != T) return VSP_ERR_SHAPE;
        if (lse->dtype != VSP_F32) return VSP_ERR_DTYPE;
    }
    if (B * Hq * T * D == 0) return VSP_OK;
    // bf16: head_dim 64 or 128; fp32: any head_dim up to 256 (the native tiles 32 / 64 / 128, or the next one padded)
    const bool native = native_head_dim(q->dtype, D);
    if (!native && !padded_head_dim(q->dtype, D)) return VSP_ERR_UNSUPPORTED;
    if (!(fabsf(scale) > 0.0f) || !(fabsf(scale) < INFINITY)) return VSP_ERR_ARG;
    const int esz = q->dtype == VSP_F32 ? 4 : 2;
    bool elementwise = !native;
    if (native && ((rc = check_tensor4(q, esz)) != VSP_OK || (rc = check_tensor4(out, esz)) != VSP_OK)) {
        if (q->dtype != VSP_F32 || rc != VSP_ERR_ALIGN) return rc;
        elementwise = true;  // fp32 rows that are not 16-byte aligned: the element-wise kernel takes them
    }
    if (elementwise && ((rc = check_tensor4_any_d(q)) != VSP_OK || (rc = check_tensor4_any_d(out)) != VSP_OK)) return rc;
    if (lse && !lse->data) return VSP_ERR_NULL;
    if (T > INT32_MAX / 2) return VSP_ERR_ARG;

    PrefillArgs a{};
    a.D_true = (int)D;
    a.elementwise = elementwise ? 1 : 0;
    a.q = q->data;
    a.k = cache->k;
    a.v = cache->v;
    a.rope_table = rope_table;
    a.out = out->data;
    a.lse = lse ? (float*)lse->data : nullptr;
    int64_t s_phys = kv_s_pad(cache->format, cache->S_max);
    for (int i = 0; i < 3; ++i) {
        a.sq[i] = q->stride[i];
        a.so[i] = out->stride[i];
        a.sl[i] = lse ? lse->stride[i] : 0;
    }
    if (cache->format == VSP_KV_Q8_0) {
        // Compute-bound path: dequantising inside the MFMA loop would add vector-ALU work to a kernel that is
        // already short of it, while reading the context out once costs ~0.2 % of the attention time.  The rows
        // [0, L) are dequantised to dense bf16 in the workspace and the dense kernel runs over that.
        const size_t need = vsp_attn_prefill_cached_workspace_bytes(cache, seq_lens != nullptr, max_len);
        if (!workspace || workspace_bytes < need) return VSP_ERR_WORKSPACE;
        if (!is_aligned16(workspace)) return VSP_ERR_ALIGN;
        vsp_tensor kt{}, vt{};
        kt.dtype = vt.dtype = VSP_BF16;
        kt.ndim = vt.ndim = 4;
        const int64_t shp[4] = {B, Hkv, L, D};
        for (int i = 0; i < 4; ++i) kt.shape[i] = vt.shape[i] = shp[i];
        kt.stride[3] = vt.stride[3] = 1;
        kt.stride[2] = vt.stride[2] = D;
        kt.stride[1] = vt.stride[1] = L * D;
        kt.stride[0] = vt.stride[0] = Hkv * L * D;
        kt.data = workspace;
        vt.data = (char*)workspace + need / 2;
        if (!dense_ready && (rc = vsp_kv_read(cache, 0, L, &kt, &vt, stream)) != VSP_OK) return rc;
        a.k = kt.data;
        a.v = vt.data;
        s_phys = L;
    }
    a.sk[0] = a.sv[0] = Hkv * s_phys * D;
    a.sk[1] = a.sv[1] = s_phys * D;
    a.sk[2] = a.sv[2] = D;
    a.B = (int)B;
    a.Hq = (int)Hq;
    a.Hkv = (int)Hkv;
    a.n_rep = (int)(Hq / Hkv);
    a.T = (int)T;
    a.L = (int)L;
    a.s_pad = (int)s_phys;
    a.seq_lens = seq_lens;
    a.chunk_lens = chunk_lens;
    if (cache->page_table && cache->format == VSP_KV_BF16) {
        a.page_table = cache->page_table;
        a.page_tokens = cache->page_tokens;
        a.pages_per_seq = cache->pages_per_seq;
        a.s_pad = cache->page_tokens;
    }
    a.causal = is_causal ? 1 : 0;
    a.n_qtiles = (int)ceil_div(T, kBM);
    a.negate_q = (q->dtype == VSP_BF16 && scale < 0.0f) ? 1 : 0;
    a.scale_log2 = (q->dtype == VSP_BF16 ? fabsf(scale) : scale) * kLog2e;
    if (q->dtype == VSP_F32) return launch_prefill(a, q->dtype, D, false, stream);
    // a caller that brings room for partials behind what the format itself needs gets the context split over workgroups
    // when the grid would otherwise leave the chip idle; the combine kernel finishes the rows (and their lse)
    const bool planes = cache->format == VSP_KV_BF16;
    const size_t base = plan_base_bytes(cache, seq_lens != nullptr, max_len);
    const bool room = workspace && is_aligned16(workspace) && workspace_bytes > base;
    const size_t share = (size_t)B * (size_t)Hq * (size_t)T * (size_t)(D + 2) * sizeof(float);
    const int64_t max_shares = room ? (int64_t)std::min<size_t>((workspace_bytes - base) / share, kMostShares) : 1;
    const PrefillPlan p = plan_cached(cache, Hq, T, L, seq_lens || chunk_lens, max_shares, rope_table != nullptr);
    if (p.n_splits > 1) {
        a.ws_o = (float*)((char*)workspace + base);
        a.ws_ml = a.ws_o + (size_t)B * Hq * T * p.n_splits * D;
    }
    if ((rc = launch_prefill_bf16(a, D, planes, p, (hipStream_t)stream)) != VSP_OK || p.n_splits <= 1) return rc;
    CombineExtra x;
    x.chunk_lens = chunk_lens;
    x.len_floor = (int)T;
    x.lse = a.lse;
    for (int i = 0; i < 3; ++i) x.sl[i] = a.sl[i];
    return launch_split_combine(a.ws_o, a.ws_ml, seq_lens, cache->len, p.split_tiles * kUnit, p.n_splits, B, Hq, T, D, (int)L, out,
                                (hipStream_t)stream, x);
}

extern "C" int vsp_attn_prefill_cached(const vsp_tensor* q, const vsp_kv_cache* cache, const int32_t* seq_lens, int32_t max_len,
                                       const int32_t* chunk_lens, vsp_tensor* out, vsp_tensor* lse, float scale,
                                       int is_causal, void* workspace, size_t workspace_bytes, void* stream) {
    return prefill_cached(q, cache, seq_lens, max_len, chunk_lens, out, lse, scale, is_causal, workspace, workspace_bytes, stream, nullptr, false);
}

extern "C" int vsp_attn_prompt_step(vsp_kv_cache* cache, const vsp_tensor* q, const vsp_tensor* new_k, const vsp_tensor* new_v,
                                    const float* rope_table, int64_t table_len, vsp_tensor* out, float scale, void* workspace,
                                    size_t workspace_bytes, void* stream) {
    if (!q || !new_k || !new_v || !out || !rope_table) return VSP_ERR_NULL;
    int rc = check_kv_cache(cache);
    if (rc != VSP_OK) return rc;
    if (cache->format == VSP_KV_F32) return VSP_ERR_UNSUPPORTED;  // rotating in the fp32 kernel was no faster: 2 x 16 heads, 1000 tokens 71.5 -> 73.5 us
    const int64_t T = q->ndim == 4 ? q->shape[2] : 0;
    // what vsp_rope_kv_append and vsp_attn_prefill_cached take, of a prompt that fills the cache from its start
    if (T < 2 || T < cache->len || T > cache->S_max || q->dtype != VSP_BF16 || out->dtype != VSP_BF16 || out->ndim != 4 || (cache->D != 64 && cache->D != 128) ||
        q->shape[3] != cache->D || !is_aligned16(rope_table) || check_tensor4(q, 2) != VSP_OK || check_tensor4(out, 2) != VSP_OK || !(fabsf(scale) > 0.0f) || !(fabsf(scale) < INFINITY))
        return VSP_ERR_UNSUPPORTED;
    for (int i = 0; i < 4; ++i)
        if (q->shape[i] <= 0 || out->shape[i] != q->shape[i]) return VSP_ERR_UNSUPPORTED;
    if (cache->Hkv <= 0 || q->shape[0] != cache->B || q->shape[1] % cache->Hkv != 0) return VSP_ERR_UNSUPPORTED;
    void *dense_k = nullptr, *dense_v = nullptr;
    if (cache->format == VSP_KV_Q8_0) {
        // The append leaves the rows that prefill_cached would read out into the workspace, which was a launch that read the planes back.  us:
        // 32 / 8 heads, D 128, 777 tokens 31.6 -> 21.5, 2000 x 2 117 -> 99; 16 heads, D 64, 6 x 368 33.5 -> 22.3; 2 x 32 / 8, 60 tokens 13.6 -> 9.9
        const size_t need = vsp_attn_prefill_cached_workspace_bytes(cache, 0, (int32_t)T);
        if (workspace_bytes < need || !workspace || !is_aligned16(workspace)) return VSP_ERR_WORKSPACE;
        dense_k = workspace;
        dense_v = (char*)workspace + need / 2;
    }
    bool dense_ready = false;
    if ((rc = kv_append_rotated(cache, q, new_k, new_v, rope_table, table_len, 0, dense_k, dense_v, &dense_ready, stream)) != VSP_OK) return rc;
    return prefill_cached(q, cache, nullptr, (int32_t)T, nullptr, out, nullptr, scale, 1, workspace, workspace_bytes, stream, rope_table, dense_ready);
}

namespace {
// Bytes of the hi / lo bf16 planes of Q, K and V (dense [B,H,N,D] each, 256-byte aligned starts).
size_t split_plane_bytes(int64_t elems) { return (size_t)((elems * 2 + 255) / 256 * 256); }

int prefill_entry(const vsp_tensor* q, const vsp_tensor* k, const vsp_tensor* v, vsp_tensor* out, vsp_tensor* lse, float scale,
                  int is_causal, float dropout_p, int training, bool split, void* workspace, size_t workspace_bytes, void* stream);
}  // namespace

extern "C" int vsp_attn_prefill(const vsp_tensor* q, const vsp_tensor* k, const vsp_tensor* v, vsp_tensor* out,
                                vsp_tensor* lse, float scale, int is_causal, float dropout_p, int training,
                                void* stream) {
    return prefill_entry(q, k, v, out, lse, scale, is_causal, dropout_p, training, false, nullptr, 0, stream);
}

extern "C" size_t vsp_attn_prefill_split_workspace_bytes(int32_t B, int32_t Hq, int32_t Hkv, int32_t T, int32_t L, int32_t D) {
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || T <= 0 || L <= 0 || D <= 0) return 0;
    return 4 * split_plane_bytes((int64_t)B * Hkv * L * D);  // hi and lo planes of K and of V
}

extern "C" int vsp_attn_prefill_split(const vsp_tensor* q, const vsp_tensor* k, const vsp_tensor* v, vsp_tensor* out,
                                      vsp_tensor* lse, float scale, int is_causal, void* workspace, size_t workspace_bytes,
                                      void* stream) {
    return prefill_entry(q, k, v, out, lse, scale, is_causal, 0.0f, 0, true, workspace, workspace_bytes, stream);
}

namespace {
// The split forward's workgroup: R row groups of 32 queries times 4 / R key groups, for the reasons at plan_prefill: a grid that leaves the chip idle takes
// as long as its longest workgroup's chain of key tiles (0.9 to 1.6 us a tile), a full one is fastest with the fewest reads of a tile.  us, R = 4 / 2 / 1
// (w: workgroups of 128 queries):
// D 128 (R 2: one workgroup per CU, R 4: two): 32 heads, 445 tokens, not causal (w 128) 32.7 / 28.0; 16 heads, 1491 (w 192) 70.7 / 54.4; 64 / 8, 2 x 175 (w 256)
//   16.1 / 20.1; 16 heads, 3 x 1130 (w 432) 77.5 / 92.2;
// D 64: 8 / 2, 3 x 248 (w 48) 13.0 / 10.4 / 9.4; 12 heads, 3 x 71 (w 36) 8.7 / 8.6 / 10.7; 8 / 2, 1613 (w 104) 47.6 / 29.8 / 24.2; 2 x 1339 (w 176) 40.5 / 28.6 / 34.3;
//   32 / 8, 3 x 177 (w 192) 11.5 / 11.1 / 16.9; 12 heads, 2 x 1433 (w 288) 50.0 / 38.2 / 57; 8 / 2, 6 x 862 (w 336) 33.5 / 28.7 / 49.5; 16 heads, 7 x 482 (w 448) 31 / 33 / 55.
int split_row_groups(int64_t B, int64_t Hq, int64_t T, int64_t L, int64_t D, bool causal) {
    const int64_t cus = device_cu_count(), w = ceil_div(T, kBM) * B * Hq, tiles = ceil_div(L, kUnit);
    if (tiles < 3) return 4;
    if (D == 64 && ((tiles >= 6 && 4 * w <= cus) || (causal && tiles >= 24 && 2 * w <= cus))) return 1;
    if (2 * w <= cus) return 2;
    if (D == 64) return (tiles >= 6 && w <= cus) || (causal && tiles >= 24 && 2 * w <= 3 * cus) ? 2 : 4;
    return causal && tiles >= 32 && w <= cus ? 2 : 4;
}

template <int D>
int launch_prefill_split(PrefillArgs a, hipStream_t st) {
    auto launch = [&](auto r) {
        constexpr int R = decltype(r)::value;
        a.n_qtiles = (int)ceil_div(a.T, 32 * R);
        const dim3 grid((unsigned)((int64_t)a.n_qtiles * a.B * a.Hq));
        if (a.causal) a.causal = D == 128 && R == 4 ? launch_fold(a.n_qtiles, (int64_t)a.B * a.Hq) : a.n_qtiles;
        hipLaunchKernelGGL((prefill_split_kernel<D, R, 4 / R>), grid, dim3(256), 0, st, a);
        return check_launch();
    };
    const int r = split_row_groups(a.B, a.Hq, a.T, a.L, D, a.causal != 0);
    if constexpr (D == 64) return with_row_groups<4, 2, 1>(r, launch);
    else return with_row_groups<4, 2>(r, launch);
}

int prefill_entry(const vsp_tensor* q, const vsp_tensor* k, const vsp_tensor* v, vsp_tensor* out, vsp_tensor* lse, float scale,
                  int is_causal, float dropout_p, int training, bool split, void* workspace, size_t workspace_bytes, void* stream) {
    if (!q || !k || !v || !out) return VSP_ERR_NULL;
    // validation in the reference's order, src/ops/flash_attention.cpp:45-59
    if (q->ndim != 4 || k->ndim != 4 || v->ndim != 4) return VSP_ERR_NDIM;
    const int64_t B = q->shape[0], Hq = q->shape[1], T = q->shape[2], D = q->shape[3];
    const int64_t Hkv = k->shape[1], L = k->shape[2];
    for (int i = 0; i < 4; ++i)
        if (k->shape[i] != v->shape[i]) return VSP_ERR_SHAPE;
    if (k->shape[0] != B || k->shape[3] != D) return VSP_ERR_SHAPE;
    if (Hkv <= 0 ? Hq != 0 : (Hq % Hkv != 0)) return VSP_ERR_SHAPE;
    if (is_causal && T > L) return VSP_ERR_SHAPE;
    if (q->dtype != k->dtype || k->dtype != v->dtype) return VSP_ERR_DTYPE;
    if (dropout_p < 0.0f || dropout_p >= 1.0f) return VSP_ERR_DROPOUT;
    // inference only: dropout is active in the reference iff training && dropout_p > 0 (:241)
    if (training && dropout_p > 0.0f) return VSP_ERR_UNSUPPORTED;
    if (out->ndim != 4) return VSP_ERR_NDIM;
    for (int i = 0; i < 4; ++i)
        if (out->shape[i] != q->shape[i]) return VSP_ERR_SHAPE;
    if (out->dtype != q->dtype) return VSP_ERR_DTYPE;
    if (q->dtype != VSP_BF16 && q->dtype != VSP_F32) return VSP_ERR_UNSUPPORTED;
    if (lse) {
        if (lse->ndim != 3 || lse->shape[0] != B || lse->shape[1] != Hq || lse->shape[2] != T) return VSP_ERR_SHAPE;
        if (lse->dtype != VSP_F32) return VSP_ERR_DTYPE;
    }
    if (B * Hq * T * D == 0) return VSP_OK;
    // bf16: head_dim 64 or 128; fp32: any head_dim up to 256, as the reference's forward takes any (:235-238): the native
    // tiles 32 / 64 / 128, or the next one with the columns past head_dim padded with zeros inside the kernel
    const bool native = native_head_dim(q->dtype, D);
    if (!native && (split || !padded_head_dim(q->dtype, D))) return VSP_ERR_UNSUPPORTED;
    if (L == 0) return VSP_ERR_SHAPE;  // softmax over an empty context is undefined
    if (!(fabsf(scale) > 0.0f) || !(fabsf(scale) < INFINITY)) return VSP_ERR_ARG;
    const int esz = q->dtype == VSP_F32 ? 4 : 2;
    int rc;
    bool elementwise = !native;
    if (native && ((rc = check_tensor4(q, esz)) != VSP_OK || (rc = check_tensor4(k, esz)) != VSP_OK ||
                   (rc = check_tensor4(v, esz)) != VSP_OK || (rc = check_tensor4(out, esz)) != VSP_OK)) {
        if (q->dtype != VSP_F32 || split || rc != VSP_ERR_ALIGN) return rc;
        elementwise = true;  // fp32 rows that are not 16-byte aligned: the element-wise kernel takes them
    }
    if (elementwise && ((rc = check_tensor4_any_d(q)) != VSP_OK || (rc = check_tensor4_any_d(k)) != VSP_OK ||
                        (rc = check_tensor4_any_d(v)) != VSP_OK || (rc = check_tensor4_any_d(out)) != VSP_OK))
        return rc;
    if (lse && !lse->data) return VSP_ERR_NULL;
    if (T > INT32_MAX / 2 || L > INT32_MAX / 2) return VSP_ERR_ARG;
    // the tile loads address one head's rows through a 32-bit buffer descriptor
    if (k->stride[2] < 0 || v->stride[2] < 0) return VSP_ERR_STRIDE;
    if (q->dtype == VSP_BF16 && (L * k->stride[2] * 2 > INT32_MAX || L * v->stride[2] * 2 > INT32_MAX)) return VSP_ERR_STRIDE;

    PrefillArgs a{};
    a.D_true = (int)D;
    a.elementwise = elementwise ? 1 : 0;
    a.q = q->data;
    a.k = k->data;
    a.v = v->data;
    a.out = out->data;
    a.lse = lse ? (float*)lse->data : nullptr;
    for (int i = 0; i < 3; ++i) {
        a.sq[i] = q->stride[i];
        a.sk[i] = k->stride[i];
        a.sv[i] = v->stride[i];
        a.so[i] = out->stride[i];
        a.sl[i] = lse ? lse->stride[i] : 0;
    }
    a.B = (int)B;
    a.Hq = (int)Hq;
    a.Hkv = (int)Hkv;
    a.n_rep = (int)(Hq / Hkv);
    a.T = (int)T;
    a.L = (int)L;
    a.causal = is_causal ? 1 : 0;
    a.n_qtiles = (int)ceil_div(T, kBM);
    a.negate_q = (q->dtype == VSP_BF16 && scale < 0.0f) ? 1 : 0;
    a.scale_log2 = (q->dtype == VSP_BF16 ? fabsf(scale) : scale) * kLog2e;
    if (split) {
        // fp32 tensors through the bf16 matrix cores: split planes in the workspace, then the attention kernel over them
        if (q->dtype != VSP_F32 || (D != 64 && D != 128)) return VSP_ERR_UNSUPPORTED;
        const int64_t nk = B * Hkv * L * D;
        if (L * D * 2 > INT32_MAX || nk / 8 > INT32_MAX * 256LL) return VSP_ERR_ARG;
        const size_t need = 4 * split_plane_bytes(nk);
        if (!workspace || workspace_bytes < need) return VSP_ERR_WORKSPACE;
        if (!is_aligned16(workspace)) return VSP_ERR_ALIGN;
        uint16_t* planes[4];
        for (int i = 0; i < 4; ++i) planes[i] = (uint16_t*)((char*)workspace + i * split_plane_bytes(nk));
        SplitPlan sp{};
        const vsp_tensor* src[2] = {k, v};
        for (int t = 0; t < 2; ++t) {
            sp.src[t] = (const float*)src[t]->data;
            sp.hi[t] = planes[2 * t];
            sp.lo[t] = planes[2 * t + 1];
            sp.s0[t] = src[t]->stride[0];
            sp.s1[t] = src[t]->stride[1];
            sp.s2[t] = src[t]->stride[2];
        }
        sp.by_n = FastDiv::of(L), sp.by_h = FastDiv::of(Hkv);
        sp.groups = nk / 8;
        sp.D = (int)D;
        hipStream_t st = (hipStream_t)stream;
        hipLaunchKernelGGL(split_f32_kernel, dim3((unsigned)ceil_div(nk / 8, 256), 2), dim3(256), 0, st, sp);
        rc = check_launch();
        if (rc != VSP_OK) return rc;
        a.k = planes[0];
        a.k_lo = planes[1];
        a.v = planes[2];
        a.v_lo = planes[3];
        a.sk[0] = Hkv * L * D, a.sk[1] = L * D, a.sk[2] = D;
        a.sv[0] = a.sk[0], a.sv[1] = a.sk[1], a.sv[2] = D;
        a.negate_q = scale < 0.0f ? 1 : 0;
        a.scale_log2 = fabsf(scale) * kLog2e;
        return D == 128 ? launch_prefill_split<128>(a, st) : launch_prefill_split<64>(a, st);
    }
    return launch_prefill(a, q->dtype, D, false, stream);
}
}  // namespace

extern "C" int vsp_attn_prefill_plan(int32_t B, int32_t Hq, int32_t Hkv, int32_t T, int32_t L, int32_t D, int is_causal, int split, vsp_attn_plan* plan) {
    if (!plan) return VSP_ERR_NULL;
    if (D != 64 && D != 128) return VSP_ERR_UNSUPPORTED;
    if (B <= 0 || Hkv <= 0 || Hq <= 0 || Hq % Hkv != 0 || T <= 0 || L <= 0 || (is_causal && T > L)) return VSP_ERR_SHAPE;
    if (T > INT32_MAX / 2 || L > INT32_MAX / 2) return VSP_ERR_ARG;
    if (split) {
        const int r = split_row_groups(B, Hq, T, L, D, is_causal != 0);
        *plan = vsp_attn_plan{r, 4 / r, 0, 0, 1};
    } else {
        const PrefillPlan p = plan_prefill(B, Hkv, Hq / Hkv, T, L, D, is_causal != 0, D == 128, false, 1, false);
        *plan = vsp_attn_plan{p.R, p.G, p.pipe, p.pack, p.n_splits};
    }
    return VSP_OK;
}
