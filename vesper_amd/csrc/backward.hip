// Flash-attention backward for gfx950.
//
// Replaces flash_attention_backward_hip_dispatch (include/vesper/ops/flash_attention.h:80-92,
// src/ops/hip/flash_attention.hip:183-299) with the mathematics of the reference's CPU backward
// (src/ops/flash_attention.cpp:366-482): with P = exp(scale q.k - lse) recomputed from the forward's
// log-sum-exp,  Di = rowsum(dO * O),  dV = P^T dO,  dP = dO V^T,  dS = P * (dP - Di),
// dQ = scale dS K,  dK = scale dS^T Q.  Differences from the reference's HIP kernel: matrix cores
// instead of scalar FMAs, D in {64, 128} (and 32 for fp32 operands), grouped-query heads folded in
// (dK / dV of a kv head sum over its query heads, the gradient of ops::repeat_kv), and no atomics:
// dQ is produced by one pass that owns query rows, dK / dV by a second pass that owns key rows, so the
// result is bitwise reproducible (the reference accumulates dQ with atomicAdd).  Both passes compute dS; with the
// larger of the two workspaces (bf16 operands) the dK / dV pass runs first and leaves dS behind as bf16 tiles, and dQ is
// one product over those tiles (bwd_rowstats_bf16_kernel, bwd_dkdv_bf16_kernel<D, true>, bwd_dq_stream_kernel).
//
// fp32 operands: fp32 MFMA (32x32x2) throughout.  bf16 operands: bf16 MFMA (32x32x16) with fp32 accumulation
// and fp32 softmax algebra; P and dS are rounded to bf16 (round-to-nearest-even) between the products, as P is
// in the forward kernel, and the gradients are rounded to bf16 on store.  The fp32 kernels use plain padded LDS
// tiles filled by ordinary loads; the bf16 kernels use dense XOR-swizzled tiles filled by direct-to-LDS loads
// through a ring of slots (see the comments at bwd_dq_bf16 and bwd_dkdv_bf16).
#include <math.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "vsp_common.hpp"

namespace vsp {
namespace {

struct BwdArgs {
    const void *dout, *q, *k, *v, *out;
    const float* lse;
    void *dq, *dk, *dv;
    float* delta;                          // workspace: Di [B][Hq][N]
    float* lse2;                           // workspace: lse * log2(e) [B][Hq][N] (bf16 and split kernels)
    int64_t s_do[3], s_q[3], s_k[3], s_v[3], s_o[3], s_l[3], s_dq[3], s_dk[3], s_dv[3];
    int32_t B, Hq, Hkv, n_rep, N;
    int32_t causal;
    float scale;
    int64_t lo_q, lo_kv;                   // split operands: elements from a hi plane to its lo plane (q-shaped, kv-shaped)
    int32_t D_true;                        // fp32 kernels: the tensors' head_dim (<= the kernel's tile width; columns past it are zero)
    // bf16, one-pass dS: the dK / dV pass leaves every dS tile (32 keys x 32 queries, bf16, [key][query], 2 KB) in the
    // workspace at [b][hq][query tile][key tile], and dQ is one product over those tiles
    uint16_t* ds_tiles;
    int32_t n_qt32, n_kt32;                // query tiles per head, key tiles per head (an even number: key blocks come in pairs)
    // dK / dV pass in parts: a part of a key block is part_heads of the group's query heads times part_tiles query tiles
    // (counted from the last one down), one workgroup each, which leaves its accumulators in `parts` (fp32, register
    // images); bwd_dkdv_reduce_kernel adds them
    int32_t part_heads, part_tiles;        // part_heads 0: one workgroup per key block, gradients stored directly
    int32_t part_ranges, n_parts;          // ranges of part_tiles per head; head groups times ranges
    float* parts;                          // [part][workgroup's keys][key block of 32][dV, dK][quad][lane][4]
};
// bf16 passes: divisors of a workgroup's number: key blocks of a part, B * Hkv, Hkv, n_rep
struct BwdDivisors {
    FastDiv by_blocks, by_bkv, by_hkv, by_rep, by_n, by_hq;
};

// Di[b][h][i] = sum_d dO[i][d] * O[i][d]   (src/ops/flash_attention.cpp:416-423); one wavefront per row.
__global__ void __launch_bounds__(256) bwd_delta_kernel(BwdArgs a, int D) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int64_t rows = (int64_t)a.B * a.Hq * a.N;
    if (row >= rows) return;
    const int i = (int)(row % a.N);
    const int64_t bh = row / a.N;
    const int h = (int)(bh % a.Hq), b = (int)(bh / a.Hq);
    const float* po = (const float*)a.out + (int64_t)b * a.s_o[0] + (int64_t)h * a.s_o[1] + (int64_t)i * a.s_o[2];
    const float* pd = (const float*)a.dout + (int64_t)b * a.s_do[0] + (int64_t)h * a.s_do[1] + (int64_t)i * a.s_do[2];
    float s = 0.f;
    for (int d = lane; d < D; d += 64) s += pd[d] * po[d];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) a.delta[row] = s;
}

// bf16 operands: Di as above and lse * log2(e), the two per-row constants of both passes.  D / 8 lanes per row, 16 bytes of O and dO each.
template <int D>
__global__ void __launch_bounds__(256) bwd_rowstats_bf16_kernel(BwdArgs a, BwdDivisors dv) {
    constexpr int LPR = D / 8, RPB = 256 / LPR;
    const uint32_t row = blockIdx.x * RPB + threadIdx.x / LPR, rows = (uint32_t)a.B * a.Hq * a.N, rr = min(row, rows - 1);
    const int piece = threadIdx.x % LPR;
    const uint32_t bh = dv.by_n.div(rr), i = dv.by_n.mod(rr, bh), b = dv.by_hq.div(bh), h = dv.by_hq.mod(bh, b);
    const uint4 wo = *(const uint4*)((const uint16_t*)a.out + (int64_t)b * a.s_o[0] + (int64_t)h * a.s_o[1] + (int64_t)i * a.s_o[2] + 8 * piece);
    const uint4 wd = *(const uint4*)((const uint16_t*)a.dout + (int64_t)b * a.s_do[0] + (int64_t)h * a.s_do[1] + (int64_t)i * a.s_do[2] + 8 * piece);
    const uint32_t o4[4] = {wo.x, wo.y, wo.z, wo.w}, d4[4] = {wd.x, wd.y, wd.z, wd.w};
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        s += __uint_as_float(o4[j] << 16) * __uint_as_float(d4[j] << 16);
        s += __uint_as_float(o4[j] & 0xffff0000u) * __uint_as_float(d4[j] & 0xffff0000u);
    }
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (row < rows && piece == 0) {
        a.delta[row] = s;
        a.lse2[row] = 1.4426950408889634f * a.lse[(int64_t)b * a.s_l[0] + (int64_t)h * a.s_l[1] + (int64_t)i * a.s_l[2]];
    }
}

constexpr int kBQ = 128;  // rows (queries or keys) per workgroup, 32 per wavefront
constexpr int kBT = 32;   // rows of the streamed tile

// ---- dQ: a wavefront owns 32 query rows and walks the key tiles (the forward's structure) ----
//   S^T[key][q]  = K . Q^T      A = K tile (LDS), B = Q^T (registers)
//   dP^T[key][q] = V . dO^T     A = V tile (LDS), B = dO^T (registers)
//   dS^T = exp(scale S^T - lse[q]) * (dP^T - Di[q])        a lane owns one query column: lse, Di are per lane
//   dQ^T[d][q]  += K^T . dS^T   A = K^T (the same tile read column-wise), B = dS^T straight from registers
template <int D>
__global__ void __launch_bounds__(256) bwd_dq_kernel(BwdArgs a) {
    constexpr int PITCH = D + 1;
    constexpr int DB = D / 32;
    __shared__ float sK[kBT * PITCH];
    __shared__ float sV[kBT * PITCH];
    const int n_qtiles = (a.N + kBQ - 1) / kBQ;
    const int bid = blockIdx.x;
    const int qt = n_qtiles - 1 - bid / (a.B * a.Hq);
    const int bh = xcd_grouped_head(bid % (a.B * a.Hq), a.B * a.Hkv, a.n_rep);  // a kv group's query heads share one XCD's L2
    const int b = bh / a.Hq, hq = bh % a.Hq, kvh = hq / a.n_rep;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ql = lane & 31, h = lane >> 5;
    const int q0 = qt * kBQ + wave * 32;
    const int qi = q0 + ql;
    const int qrow = min(qi, a.N - 1);

    const float* Qp = (const float*)a.q + (int64_t)b * a.s_q[0] + (int64_t)hq * a.s_q[1] + (int64_t)qrow * a.s_q[2];
    const float* Op = (const float*)a.dout + (int64_t)b * a.s_do[0] + (int64_t)hq * a.s_do[1] + (int64_t)qrow * a.s_do[2];
    const float* Kp = (const float*)a.k + (int64_t)b * a.s_k[0] + (int64_t)kvh * a.s_k[1];
    const float* Vp = (const float*)a.v + (int64_t)b * a.s_v[0] + (int64_t)kvh * a.s_v[1];
    float qf[D / 2], dof[D / 2];
    const int Dt = a.D_true;  // the reference's backward takes any head_dim (src/ops/flash_attention.cpp:366-482)
#pragma unroll
    for (int ks = 0; ks < D / 2; ++ks) {
        qf[ks] = 2 * ks + h < Dt ? Qp[2 * ks + h] : 0.f;
        dof[ks] = 2 * ks + h < Dt ? Op[2 * ks + h] : 0.f;
    }
    const float lse_q = a.lse[(int64_t)b * a.s_l[0] + (int64_t)hq * a.s_l[1] + (int64_t)qrow * a.s_l[2]];
    const float di_q = a.delta[((int64_t)b * a.Hq + hq) * a.N + qrow];

    const int wg_qmax = min(qt * kBQ + kBQ - 1, a.N - 1);
    const int kv_end_wg = a.causal ? min(a.N, wg_qmax + 1) : a.N;
    const int n_tiles = (kv_end_wg + kBT - 1) / kBT;
    const int kv_end_wave = (q0 < a.N) ? (a.causal ? min(a.N, min(q0 + 31, a.N - 1) + 1) : a.N) : 0;

    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;

    for (int kt = 0; kt < n_tiles; ++kt) {
        __syncthreads();
        for (int id = tid; id < kBT * D; id += 256) {
            const int row = id / D, col = id % D, key = kt * kBT + row;
            const bool ok = key < a.N && col < Dt;
            sK[row * PITCH + col] = ok ? Kp[(int64_t)key * a.s_k[2] + col] : 0.f;
            sV[row * PITCH + col] = ok ? Vp[(int64_t)key * a.s_v[2] + col] : 0.f;
        }
        __syncthreads();
        const int k0 = kt * kBT;
        if (k0 >= kv_end_wave) continue;
        f32x16_t s, dp;
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = dp[j] = 0.f;
#pragma unroll
        for (int ks = 0; ks < D / 2; ++ks) {
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(sK[ql * PITCH + 2 * ks + h], qf[ks], s, 0, 0, 0);
            dp = __builtin_amdgcn_mfma_f32_32x32x2f32(sV[ql * PITCH + 2 * ks + h], dof[ks], dp, 0, 0, 0);
        }
        const int lim = a.causal ? min(qi, a.N - 1) : a.N - 1;
        float ds[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int key = k0 + 8 * (v >> 2) + 4 * h + (v & 3);
            const float p = key <= lim ? expf(s[v] * a.scale - lse_q) : 0.f;
            ds[v] = p * (dp[v] - di_q);
        }
        // dQ^T += K^T . dS^T : contraction slot h of step v is key 8*(v/4) + 4*h + v%4, the key ds[v] belongs to
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int krow = 8 * (v >> 2) + 4 * h + (v & 3);
#pragma unroll
            for (int db = 0; db < DB; ++db)
                acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(sK[krow * PITCH + 32 * db + ql], ds[v], acc[db], 0, 0, 0);
        }
    }
    if (qi < a.N) {
        float* op = (float*)a.dq + (int64_t)b * a.s_dq[0] + (int64_t)hq * a.s_dq[1] + (int64_t)qi * a.s_dq[2];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int d = 32 * db + 8 * (v >> 2) + 4 * h + (v & 3);
                if (d < Dt) op[d] = a.scale * acc[db][v];
            }
    }
}

// ---- dK, dV: a wavefront owns 32 key rows of one kv head and walks the query heads of the group and their
// query tiles (the forward's structure with the roles of queries and keys exchanged) ----
//   S[q][key]  = Q . K^T        A = Q tile (LDS), B = K^T (registers);  a lane owns one key column
//   dP[q][key] = dO . V^T       A = dO tile (LDS), B = V^T (registers)
//   P = exp(scale S - lse[q]),  dS = P * (dP - Di[q])      lse, Di per row: read from LDS
//   dV^T[d][key] += dO^T . P    A = dO^T (tile read column-wise), B = P from registers
//   dK^T[d][key] += Q^T . dS    A = Q^T, B = dS
template <int D>
__global__ void __launch_bounds__(256) bwd_dkdv_kernel(BwdArgs a) {
    constexpr int PITCH = D + 1;
    constexpr int DB = D / 32;
    __shared__ float sQ[kBT * PITCH];
    __shared__ float sO[kBT * PITCH];
    __shared__ float sL[kBT], sD[kBT];
    const int n_ktiles = (a.N + kBQ - 1) / kBQ;
    const int bid = blockIdx.x;
    const int kt = bid / (a.B * a.Hkv);  // causal: early key tiles see the most queries -> dispatched first
    const int bh = bid % (a.B * a.Hkv);
    const int b = bh / a.Hkv, kvh = bh % a.Hkv;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kl = lane & 31, h = lane >> 5;
    const int key0 = kt * kBQ + wave * 32;
    const int ki = key0 + kl;
    const int krow = min(ki, a.N - 1);
    (void)n_ktiles;

    const float* Kp = (const float*)a.k + (int64_t)b * a.s_k[0] + (int64_t)kvh * a.s_k[1] + (int64_t)krow * a.s_k[2];
    const float* Vp = (const float*)a.v + (int64_t)b * a.s_v[0] + (int64_t)kvh * a.s_v[1] + (int64_t)krow * a.s_v[2];
    float kf[D / 2], vf[D / 2];
    const int Dt = a.D_true;
#pragma unroll
    for (int ks = 0; ks < D / 2; ++ks) {
        kf[ks] = 2 * ks + h < Dt ? Kp[2 * ks + h] : 0.f;
        vf[ks] = 2 * ks + h < Dt ? Vp[2 * ks + h] : 0.f;
    }
    f32x16_t acck[DB], accv[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acck[i][j] = accv[i][j] = 0.f;

    // query tiles that can see any key of this workgroup / of this wavefront
    const int wg_kmin = kt * kBQ;
    const int qt_begin_wg = a.causal ? wg_kmin / kBT : 0;
    const int n_qt = (a.N + kBT - 1) / kBT;
    const int q_begin_wave = a.causal ? key0 : 0;

    for (int r = 0; r < a.n_rep; ++r) {
        const int hq = kvh * a.n_rep + r;
        const float* Qp = (const float*)a.q + (int64_t)b * a.s_q[0] + (int64_t)hq * a.s_q[1];
        const float* Op = (const float*)a.dout + (int64_t)b * a.s_do[0] + (int64_t)hq * a.s_do[1];
        const float* Lp = a.lse + (int64_t)b * a.s_l[0] + (int64_t)hq * a.s_l[1];
        const float* Dp = a.delta + ((int64_t)b * a.Hq + hq) * a.N;
        for (int qt = qt_begin_wg; qt < n_qt; ++qt) {
            __syncthreads();
            for (int id = tid; id < kBT * D; id += 256) {
                const int row = id / D, col = id % D, qi = qt * kBT + row;
                const bool ok = qi < a.N && col < Dt;
                sQ[row * PITCH + col] = ok ? Qp[(int64_t)qi * a.s_q[2] + col] : 0.f;
                sO[row * PITCH + col] = ok ? Op[(int64_t)qi * a.s_do[2] + col] : 0.f;
            }
            if (tid < kBT) {
                const int qi = qt * kBT + tid;
                sL[tid] = qi < a.N ? Lp[(int64_t)qi * a.s_l[2]] : 0.f;
                sD[tid] = qi < a.N ? Dp[qi] : 0.f;
            }
            __syncthreads();
            const int qb = qt * kBT;
            if (key0 >= a.N || qb + kBT - 1 < q_begin_wave) continue;  // no query of this tile sees these keys
            f32x16_t s, dp;
#pragma unroll
            for (int j = 0; j < 16; ++j) s[j] = dp[j] = 0.f;
#pragma unroll
            for (int ks = 0; ks < D / 2; ++ks) {
                s = __builtin_amdgcn_mfma_f32_32x32x2f32(sQ[kl * PITCH + 2 * ks + h], kf[ks], s, 0, 0, 0);
                dp = __builtin_amdgcn_mfma_f32_32x32x2f32(sO[kl * PITCH + 2 * ks + h], vf[ks], dp, 0, 0, 0);
            }
            float p[16], ds[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = 8 * (v >> 2) + 4 * h + (v & 3);
                const int qi = qb + row;
                const bool ok = qi < a.N && ki < a.N && (!a.causal || ki <= qi);
                p[v] = ok ? expf(s[v] * a.scale - sL[row]) : 0.f;
                ds[v] = p[v] * (dp[v] - sD[row]);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = 8 * (v >> 2) + 4 * h + (v & 3);
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    accv[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(sO[row * PITCH + 32 * db + kl], p[v], accv[db], 0, 0, 0);
                    acck[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(sQ[row * PITCH + 32 * db + kl], ds[v], acck[db], 0, 0, 0);
                }
            }
        }
    }
    if (ki < a.N) {
        float* pk = (float*)a.dk + (int64_t)b * a.s_dk[0] + (int64_t)kvh * a.s_dk[1] + (int64_t)ki * a.s_dk[2];
        float* pv = (float*)a.dv + (int64_t)b * a.s_dv[0] + (int64_t)kvh * a.s_dv[1] + (int64_t)ki * a.s_dv[2];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int d = 32 * db + 8 * (v >> 2) + 4 * h + (v & 3);
                if (d < Dt) {
                    pk[d] = a.scale * acck[db][v];
                    pv[d] = accv[db][v];
                }
            }
    }
}

// =============================================================================================
// bf16 operands: the same two passes on bf16 matrix cores (v_mfma_f32_32x32x16_bf16), fp32 accumulation and
// fp32 softmax algebra.  Tiles are bf16 in LDS with a padded pitch; the operand that a product contracts
// over rows (K^T, Q^T, dO^T) is fetched with the transposing LDS read, as V^T is in the forward kernel, and
// P / dS go from the accumulator registers into the next MFMA without leaving the lane.
// =============================================================================================
typedef short s16x4b_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// ---- a [32][D] bf16 tile in LDS ----
// Rows are dense (2 D bytes); the 16-byte chunks of a row are permuted by an XOR that depends on the row, chosen
// so that both access patterns the kernels use are free of bank conflicts: 16 lanes reading the same chunk of
// 16 consecutive rows (the row-major MFMA operand), and a 4-row x 64-byte block (the transposing read).
template <int D>
__device__ inline int tile_swz(int row) {
    return D == 128 ? (((row & 3) << 2) | ((row >> 2) & 3)) : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
}
template <int D>
__device__ inline int tile_off(int row, int chunk) { return row * (2 * D) + ((chunk ^ tile_swz<D>(row)) << 4); }
// MFMA operand, contraction over the row's elements: lane (row r = lane % 32, half h) takes elements 16 ks + 8 h ..
template <int D>
__device__ inline bf16x8_t load_row(const uint16_t* tile, int ks, int lane) {
    return __builtin_bit_cast(bf16x8_t, *(const uint4*)((const char*)tile + tile_off<D>(lane & 31, 2 * ks + (lane >> 5))));
}
__device__ inline uint2 lds_tr16(const char* p) {
    s16x4b_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4b_t*)p);
    return __builtin_bit_cast(uint2, v);
}
// MFMA operand, contraction over the tile's rows: lane (column 32 db + lane % 32, half h) takes, as slot e of
// k-step j, row 16 j + 8 (e / 4) + 4 h + e % 4 - the row that accumulator register 8 j + e of this lane half
// belongs to, so a product's result feeds the next product without leaving the lane.
template <int D>
__device__ inline bf16x8_t load_transposed(const uint16_t* tile, int j, int db, int lane) {
    const int h = lane >> 5, row = 16 * j + 4 * h + ((lane & 15) >> 2);
    const int chunk = 4 * db + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), o8 = (lane & 1) * 8;
    const uint2 lo = lds_tr16((const char*)tile + tile_off<D>(row, chunk) + o8);
    const uint2 hi = lds_tr16((const char*)tile + tile_off<D>(row + 8, chunk) + o8);
    return __builtin_bit_cast(bf16x8_t, uint4{lo.x, lo.y, hi.x, hi.y});
}
// Global -> LDS without passing through registers: a wavefront instruction moves 64 x 16 bytes to 1 KB of
// consecutive LDS, so the lane that lands on (row, physical chunk) fetches the row's chunk `physical ^ swizzle`.
// Rows at or past `valid_rows` fall outside the buffer descriptor's range and arrive as zeros.
template <int D, int W = 4>   // W wavefronts bring a tile
struct TileDma {
    static constexpr int CPR = D / 8, RPG = 64 / CPR, NLD = CPR / (2 * W);   // chunks per row, rows per instruction, instructions per wavefront
    uint32_t voff[NLD];
    __device__ inline void init(int64_t row_stride, int n_rows, int wave, int lane) {   // of a head's n_rows
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int r = (wave + W * i) * RPG + lane / CPR;
            voff[i] = tile_row_offset(r, row_stride * 2, n_rows) + 16u * (uint32_t)((lane % CPR) ^ tile_swz<D>(r));
        }
    }
    __device__ inline void load(uint16_t* dst, const uint16_t* row0, int valid_rows, int64_t row_stride, int wave) const {
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)row0, 0, (int)((int64_t)max(valid_rows, 0) * row_stride * 2), 0x00020000);
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)((char*)dst + (wave + W * i) * 1024), 16, voff[i], 0, 0, 0);
    }
};
// One float per lane (element stride `stride`) to 64 consecutive LDS words; lanes at or past `valid` bring zeros.  src and valid are the
// same in all lanes, and said to be: where the compiler does not see it, it loops over the lanes' descriptors, and it has put
// register spills behind such a loop before the lanes are back on (registers that are reloaded as garbage).
__device__ inline void row_dma(float* dst, const float* src, int valid, int64_t stride, int lane) {
    const uint64_t p = (uint64_t)(uintptr_t)src;
    const uint64_t base = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)p);
    valid = __builtin_amdgcn_readfirstlane(valid);
    __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)base, 0, (int)((int64_t)valid * stride * 4), 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 4, (uint32_t)lane * (uint32_t)stride * 4u, 0, 0, 0);
}
__device__ inline void dma_wait_all() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

constexpr float kLog2e = 1.4426950408889634f;

// two fp32 -> packed bf16x2 (lo = a, hi = b), round-to-nearest-even in one instruction
__device__ inline uint32_t cvt_pk_bf16(float a, float b) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    f32x2_t v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// four consecutive gradient elements: bf16 (rounded to nearest even) or fp32
template <bool F32>
__device__ inline void store_quad(void* base, int64_t elem, float f, f32x4_t x) {
    if constexpr (F32) *(f32x4_t*)((float*)base + elem) = f32x4_t{f * x[0], f * x[1], f * x[2], f * x[3]};
    else *(uint2*)((uint16_t*)base + elem) = uint2{cvt_pk_bf16(f * x[0], f * x[1]), cvt_pk_bf16(f * x[2], f * x[3])};
}
// ... from accumulator registers v .. v + 3
template <bool F32>
__device__ inline void store4(void* base, int64_t elem, float f, const f32x16_t& acc, int v) {
    store_quad<F32>(base, elem, f, f32x4_t{acc[v], acc[v + 1], acc[v + 2], acc[v + 3]});
}

// ---- dK, dV (bf16) ----
// A workgroup owns 64 key rows of one kv head: two blocks of 32, each worked by a pair of wavefronts that share
// the arithmetic of a (query tile, key block) step by product instead of by rows, which halves what each has to
// keep in registers (one of K / V, one of dK / dV):
//   wavefront P:  S = Q K^T  ->  P = exp2(..)  ->  hands P (bf16) to its partner through LDS  ->  dV^T += dO^T P
//   wavefront D:  dP = dO V^T                  ->  takes P  ->  dS = P (dP - Di)               ->  dK^T += Q^T dS
// Both see the same accumulator layout, so lane l of one reads exactly the words lane l of the other wrote.
// An iteration is 16 MFMA slots: the first products of tile t + 1 (8), then the second products of tile t (8); P(t + 1)
// crosses to the partner over the iteration's only barrier.  What bounds a wavefront is its instruction issue (one in 4 to 5
// cycles, 32 to an MFMA) and, per CU, the LDS port (1 KB of operands per MFMA), so the stream is laid out by hand, as in the
// forward's pipelined kernel: every slot is followed by the LDS read of the operand due kLead slots later (inline asm with the
// ring slot as an immediate offset: one address register per operand for all slots, and no wait the compiler would add for
// the direct-to-LDS loads in flight), by a pair of the vector work - the D wavefront's dS(t) under its dP(t + 1), the P
// wavefront's exp of S(t + 1) under its dV(t) - and by an instruction of the fetch; tile addresses are running scalars; the only
// branch in an iteration is the mask's (fetches past the end ask for nothing; the last four iterations are the tail's instances).
// Whole backward, compiler-scheduled stream -> this one, on one card: B 1, 32 / 8 heads, D 128, N 2048: 249.5 -> 217 us; 8 x 32 x 8
// heads, N 300, not causal: 97 -> 85.5 us; 2 x 12 x 12 heads, D 64, N 1024: 47.4 -> 41.5 us; B 1, D 64, N 8192: 1123 -> 1089 us.
// Filling the chip (D 128, N 8192) it takes 8.5 % fewer cycles, but at a clock of 1.9 instead of 2.03 GHz (the card's power
// limit): dK / dV 1184 -> 1156 us.
constexpr int kBK = 64;   // key rows per workgroup in the dK / dV pass

typedef __attribute__((address_space(3))) char lds_char_t;
typedef __attribute__((address_space(3))) f32x4_t lds_f32x4_t;

// A wavefront's 32 finished rows, whole rows at a time: as the accumulators lie, a lane has 8 bytes of its own row for each store instruction and the
// wavefront touches 32 rows with every one.  Through a patch of LDS of its own (16-byte chunks permuted by the row) an instruction covers 512 / D rows.  row(r): where row r goes
// (elements from base), or below 0.  Whole bf16 training steps with grids of a few rounds, us: 32 heads, D 128, 6 x 1172 435 -> 420, 2 x 161 27.0 -> 25.3.  Not for
// the fp32 rows of the split operands, whose pieces have 16 bytes and whose workgroups have a CU each: 1 to 4 % slower.
template <int D, class Row>
__device__ inline void store_rows(lds_char_t* patch, const f32x16_t (&acc)[D / 32], float f, int lane, void* base, Row&& row) {
    constexpr int CH = D / 8, RPI = 64 / CH;   // chunks per row, rows per instruction
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) u32x2_t lds_u2;
    typedef __attribute__((address_space(3))) u32x4_t lds_u4;
    const int ql = lane & 31, h = lane >> 5;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const f32x16_t& x = acc[i >> 2];
        const int v = 4 * (i & 3);
        *(lds_u2*)(patch + ql * D * 2 + ((i ^ (ql % CH)) << 4) + 8 * h) = u32x2_t{cvt_pk_bf16(f * x[v], f * x[v + 1]), cvt_pk_bf16(f * x[v + 2], f * x[v + 3])};
    }
    const int c = lane % CH;
#pragma unroll
    for (int i = 0; i < 32 / RPI; ++i) {
        const int r = RPI * i + lane / CH;
        const u32x4_t w = *(const lds_u4*)(patch + r * D * 2 + ((c ^ (r % CH)) << 4));
        const int64_t at = row(r);
        if (at >= 0) *(u32x4_t*)((char*)base + at * 2 + 16 * c) = w;
    }
}

template <int OFFSET>
__device__ inline u32x4_t ds_b128(uint32_t addr) {
    u32x4_t v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFFSET));
    return v;
}
template <int OFFSET>
__device__ inline uint2 ds_tr16(uint32_t addr) {
    uint2 v;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFFSET));
    return v;
}
__device__ inline uint32_t lds_byte_addr(const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }
template <int... I, class F>
__device__ inline void for_each_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ inline void for_each(F&& f) { for_each_impl(std::make_integer_sequence<int, N>{}, f); }

// Bit i: query row base + i is there and sees key ki.
__device__ inline uint32_t rows_that_see(const BwdArgs& a, int ki, int base) {
    const int lo = a.causal ? max(ki - base, 0) : 0, hi = min(a.N - base, 32);
    return ki < a.N && lo < hi ? (~0u << lo) & (~0u >> (32 - hi)) : 0u;
}
__device__ inline uint32_t bit_mask(uint32_t bits, int i) { return (uint32_t)((int32_t)(bits << (31 - i)) >> 31); }  // all ones where bit i is set

// LDS of the launches that hold both passes (see lds_start): what the dK / dV pass's variables take, asserted beside them, and what the launch takes in all
template <int D>
constexpr int kDkdvLds = D == 128 ? 4 * 16384 + 8 * 256 + 8192 : 4 * 8192 + 8 * 256 + 8192;           // bwd_dkdv_bf16
template <int D>
constexpr int kPassLds = D == 128 ? 80 * 1024 : kDkdvLds<64>;                                          // bwd_pass_kernel: two workgroups per CU, three
template <int D>
constexpr int kDkdvSplitLds = D == 128 ? 16 * 8192 + 8 * 256 + 16384 : 12 * 4096 + 6 * 256 + 24576;   // bwd_dkdv_split
template <int D>
constexpr int kSplitLds = D == 128 ? 160 * 1024 : 80 * 1024;                                           // bwd_split_pass_kernel: one workgroup per CU, two

// SPILL: the D wavefront also leaves dS of every (query tile, key block) in the workspace (a.ds_tiles), from where
// bwd_dq_stream_kernel takes dQ with one product instead of the three of bwd_dq_bf16.
template <int D, bool SPILL>
__device__ __forceinline__ void bwd_dkdv_bf16(const BwdArgs& a, const BwdDivisors& d, int block) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    constexpr int KS = D / 16, DB = D / 32;
    constexpr int NF = KS, NS = 2 * DB, NSLOT = NF + NS;   // MFMA slots: first products, second products
    constexpr int kLead = 4;
    constexpr int NR = 4;                                  // ring slots; a tile is requested three iterations ahead of its last use
    constexpr int TILEB = kBT * D * 2, SLOTB = 2 * TILEB;  // bytes of a tile; of a ring slot (Q tile | dO tile)
    __shared__ __attribute__((aligned(1024))) char ring[NR * SLOTB];
    __shared__ __attribute__((aligned(256))) float sL0[64], sL1[64], sL2[64], sL3[64];   // lse and Di of the tile's rows (32 used; a
    __shared__ __attribute__((aligned(256))) float sD0[64], sD1[64], sD2[64], sD3[64];   // wavefront instruction fills 64 words)
    __shared__ __attribute__((aligned(1024))) uint4 sP[2][2][2][64];                     // [parity of the tile][key block][words][lane]
    static_assert(sizeof(ring) + 4 * sizeof(sL0) + 4 * sizeof(sD0) + sizeof(sP) == kDkdvLds<D>);
    auto pick = [](auto s, auto* x0, auto* x1, auto* x2, auto* x3) { if constexpr (s.value == 0) return x0; else if constexpr (s.value == 1) return x1; else if constexpr (s.value == 2) return x2; else return x3; };
    auto tl = [&](auto s) { return pick(s, sL0, sL1, sL2, sL3); };
    auto td = [&](auto s) { return pick(s, sD0, sD1, sD2, sD3); };
    const int n_blocks = (a.N + kBK - 1) / kBK * a.B * a.Hkv;
    const int part = (int)d.by_blocks.div((uint32_t)block);   // 0 where there are none
    const int bid = (int)d.by_blocks.mod((uint32_t)block, (uint32_t)part);
    const int kt = (int)d.by_bkv.div((uint32_t)bid);          // causal work falls with the key tile: heaviest first
    const int bh = (int)d.by_bkv.mod((uint32_t)bid, (uint32_t)kt);
    const int b = (int)d.by_hkv.div((uint32_t)bh), kvh = (int)d.by_hkv.mod((uint32_t)bh, (uint32_t)b);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kb = wave >> 1;
    // which wavefront of a pair takes which role alternates between workgroups, so that the exp-heavy role of two
    // co-resident workgroups does not always fall on the same SIMDs
    const bool role_d = __builtin_amdgcn_readfirstlane((wave ^ __builtin_popcount(bid >> 3)) & 1);
    const int kl = lane & 31, h = lane >> 5;
    const int key0 = kt * kBK + kb * 32;
    const int ki = key0 + kl;
    const int krow = min(ki, a.N - 1);

    // the stationary operand: K rows for the P wavefront, V rows for the D wavefront
    const uint16_t* Xp = role_d ? (const uint16_t*)a.v + (int64_t)b * a.s_v[0] + (int64_t)kvh * a.s_v[1] + (int64_t)krow * a.s_v[2]
                                : (const uint16_t*)a.k + (int64_t)b * a.s_k[0] + (int64_t)kvh * a.s_k[1] + (int64_t)krow * a.s_k[2];
    bf16x8_t xf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) xf[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Xp + 16 * ks + 8 * h));
    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;

    const int qt_begin = a.causal ? (kt * kBK) / kBT : 0;
    const int n_qt = (a.N + kBT - 1) / kBT - qt_begin;   // query tiles per head
    int r0 = 0, r1 = a.n_rep, t0 = 0, t1 = n_qt;         // heads of the group, query tiles from the last one down
    if (!SPILL && a.part_heads) {                        // this workgroup's part of them
        r0 = part / a.part_ranges * a.part_heads;
        r1 = min(a.n_rep, r0 + a.part_heads);
        t0 = part % a.part_ranges * a.part_tiles;
        t1 = min(n_qt, t0 + a.part_tiles);
        if (t0 >= t1) return;                            // a lighter key block has fewer tiles
    }
    const int n_it = (r1 - r0) * (t1 - t0);              // the loop runs over (head of the group, query tile)
    // SPILL: where the D wavefront leaves its next dS tile; query tiles of a head are n_kt32 tiles apart, heads
    // n_qt32 * n_kt32
    char* ds_tile = nullptr;
    int64_t ds_step_t = 0, ds_step_r = 0;   // to the next query tile; from the last query tile of a head to the first of the next
    int se_t = 0;
    if constexpr (SPILL) {
        ds_step_t = -(int64_t)a.n_kt32 * 2048;
        ds_step_r = (int64_t)a.n_qt32 * a.n_kt32 * 2048 - (int64_t)(n_qt - 1) * ds_step_t;
        ds_tile = (char*)a.ds_tiles + ((((int64_t)b * a.Hq + kvh * a.n_rep) * a.n_qt32 + qt_begin + n_qt - 1) * a.n_kt32 + (key0 >> 5)) * 2048;
    }
    const float scale_log2 = a.scale * kLog2e;

    TileDma<D> dq_, do_;
    dq_.init(a.s_q[2], a.N, wave, lane);
    do_.init(a.s_do[2], a.N, wave, lane);
    // The tile being fetched, as running addresses (the stride arithmetic of a tile is a hundred scalar instructions): its first
    // rows, the bytes from there to the end of the head, and its row constants.
    const int64_t step_q = (int64_t)kBT * a.s_q[2] * 2, step_o = (int64_t)kBT * a.s_do[2] * 2;   // bytes per tile
    const int n_tl = t1 - t0;
    const char *pq, *po;
    const float* pr;   // lse (even wavefronts) or Di (odd ones: two write the same words)
    int nq, no, nr, ld_t = 0, n_left = n_it;
    {
        const int hq = kvh * a.n_rep + r0, qb = (qt_begin + (n_qt - 1 - t0)) * kBT;
        pq = (const char*)((const uint16_t*)a.q + (int64_t)b * a.s_q[0] + (int64_t)hq * a.s_q[1] + (int64_t)qb * a.s_q[2]);
        po = (const char*)((const uint16_t*)a.dout + (int64_t)b * a.s_do[0] + (int64_t)hq * a.s_do[1] + (int64_t)qb * a.s_do[2]);
        pr = ((wave & 1) ? a.delta : a.lse2) + ((int64_t)b * a.Hq + hq) * a.N + qb;
        nr = a.N - qb;
        nq = (int)((int64_t)nr * a.s_q[2] * 2);
        no = (int)((int64_t)nr * a.s_do[2] * 2);
    }
    const int64_t head_q = a.s_q[1] * 2 + (n_tl - 1) * step_q, head_o = a.s_do[1] * 2 + (n_tl - 1) * step_o;   // last tile of a head to the first of the next
    constexpr int NLD = TileDma<D>::NLD, NFETCH = 2 * NLD;
    constexpr int PER_TILE = NFETCH + 1;   // memory instructions per wavefront and tile
    // one instruction of the fetch: the NLD of Q, then of dO (and the row constants with the first)
    auto fetch = [&](auto buf, int i) {
        const bool is_q = i < NLD;
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(is_q ? pq : po), 0, is_q ? nq : no, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(ring + buf.value * SLOTB + (is_q ? 0 : TILEB) + (wave + 4 * (i % NLD)) * 1024), 16,
                                                 (is_q ? dq_ : do_).voff[i % NLD], 0, 0, 0);
        if (i == 0) row_dma((wave & 1) ? td(buf) : tl(buf), pr, max(min(nr, kBT), 0), 1, lane);
    };
    // past the last tile the fetch goes on with nothing in range (zeros, no memory touched): no branch in the steady state
    auto next_tile = [&]() {
        if (--n_left <= 0) {
            nq = no = nr = 0;
        } else if (++ld_t == n_tl) {
            ld_t = 0;
            pq += head_q, po += head_o;
            pr += a.N + (n_tl - 1) * kBT;
            nr -= (n_tl - 1) * kBT;
            nq -= (int)((n_tl - 1) * step_q), no -= (int)((n_tl - 1) * step_o);
        } else {
            pq -= step_q, po -= step_o;
            pr -= kBT;
            nr += kBT;
            nq += (int)step_q, no += (int)step_o;
        }
    };
    int fi_t = t0;   // query tile of the tile whose first products are due

    // Operand addresses within a tile (see load_row, load_transposed): the ring slot, the tile and the k-step of a transposed read
    // are immediate offsets.
    const uint32_t lds0 = lds_byte_addr(ring);
    uint32_t a_row[NF], a_lo[DB], a_hi[DB];
#pragma unroll
    for (int ks = 0; ks < NF; ++ks) a_row[ks] = lds0 + (uint32_t)tile_off<D>(lane & 31, 2 * ks + h);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        const int row = 4 * h + ((lane & 15) >> 2), chunk = 4 * db + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), o8 = (lane & 1) * 8;
        a_lo[db] = lds0 + (uint32_t)(tile_off<D>(row, chunk) + o8);
        a_hi[db] = lds0 + (uint32_t)(tile_off<D>(row + 8, chunk) + o8);
    }

    // The loop exists once per role.
    auto run = [&](auto role) {
    constexpr bool RD = decltype(role)::value;
    constexpr int ROWS = RD ? TILEB : 0, COLS = RD ? 0 : TILEB;   // the first products read dO rows (D) or Q rows (P)
    constexpr int STORES = RD && SPILL ? 2 : 0;
    f32x16_t s_cur, s_nxt;                 // D: dP of this tile and of the next; P: scores of the next
    uint32_t pw[2][4], pw_n[2][4];         // what the second products of this tile (the next tile) take
    // the next tile's rows: their lse, and which of them see this lane's key (bit i: row i + 4 h of the tile)
    float lq[16];
    bool edge = false;
    uint32_t seen = 0;
    auto load_lq = [&](const float* rows) {
#pragma unroll
        for (int g = 0; g < 4; ++g) *(float4*)&lq[4 * g] = *(const float4*)&rows[8 * g + 4 * h];
        const int qb = (qt_begin + (n_qt - 1 - fi_t)) * kBT;
        if (++fi_t == t1) fi_t = t0;
        edge = (a.causal && qb < key0 + 31) || qb + kBT > a.N || key0 + 32 > a.N;   // same for the wavefront
        if (edge) seen = rows_that_see(a, ki, qb + 4 * h);
    };
    // P of masked positions is 0, whatever came of their scores (NaN and overflow too).  Done on the finished words: a branch in the
    // tiles that the diagonal or the end of the sequence crosses, nothing in the others.
    auto mask = [&](uint32_t (&w)[2][4]) {
        if (edge)
#pragma unroll
            for (int v = 0; v < 16; v += 2)
                w[v >> 3][(v & 7) >> 1] &= (bit_mask(seen, 8 * (v >> 2) + (v & 3)) & 0x0000ffffu) | (bit_mask(seen, 8 * (v >> 2) + (v & 3) + 1) & 0xffff0000u);
    };
    auto exp_pair = [&](const f32x16_t& s, int v, uint32_t (&w)[2][4]) {
        w[v >> 3][(v & 7) >> 1] = cvt_pk_bf16(__builtin_amdgcn_exp2f(fmaf(s[v], scale_log2, -lq[v])), __builtin_amdgcn_exp2f(fmaf(s[v + 1], scale_log2, -lq[v + 1])));
    };
    auto post = [&](int parity, const uint32_t (&w)[2][4]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) sP[parity][kb][j][lane] = uint4{w[j][0], w[j][1], w[j][2], w[j][3]};
    };
    // The MFMA slots FROM .. TO - 1 of an iteration: first products of the tile in ring slot NX into s, second products of the tile
    // in ring slot CU.  work(slot) is what is placed behind each.
    auto slots = [&](auto from, auto to, auto nx, auto cu, f32x16_t& s, auto&& work) {
        constexpr int FROM = decltype(from)::value, TO = decltype(to)::value;
        constexpr int OFF_ROW = nx.value * SLOTB + ROWS, OFF_COL = cu.value * SLOTB + COLS;
        u32x4_t fr[NF];
        uint2 fl[NS], fh[NS];
        auto request = [&](auto sc) {
            constexpr int x = decltype(sc)::value;
            if constexpr (x < NF) fr[x] = ds_b128<OFF_ROW>(a_row[x]);
            else if constexpr (x < TO) {
                constexpr int g = x - NF, o = OFF_COL + (g / DB) * 16 * 2 * D;
                fl[g] = ds_tr16<o>(a_lo[g % DB]);
                fh[g] = ds_tr16<o>(a_hi[g % DB]);
            }
        };
        for_each<kLead>([&](auto i) { request(std::integral_constant<int, FROM + i.value>{}); });
        for_each<TO - FROM>([&](auto i) {
            constexpr int x = FROM + i.value;
            // reads issued behind this slot's operand
            constexpr int last = x + kLead - 1 < TO - 1 ? x + kLead - 1 : TO - 1;
            constexpr int rows_behind = x < NF ? ((last < NF ? last : NF - 1) - x) : 0;
            constexpr int cols_behind = last < NF ? 0 : last - (x >= NF ? x : NF - 1);
            constexpr int behind = rows_behind + 2 * cols_behind;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (x < NF) {
                asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(fr[x]) : "n"(behind));
                const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fr[x]), xf[x], x == 0 ? zero : s, 0, 0, 0);
            } else {
                constexpr int g = x - NF, j = g / DB, db = g % DB;
                asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(fl[g]), "+v"(fh[g]) : "n"(behind));
                acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, uint4{fl[g].x, fl[g].y, fh[g].x, fh[g].y}),
                                                                  __builtin_bit_cast(bf16x8_t, uint4{pw[j][0], pw[j][1], pw[j][2], pw[j][3]}), acc[db], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (x + kLead < TO) request(std::integral_constant<int, x + kLead>{});
            work(std::integral_constant<int, x>{});
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    using FIRST = std::integral_constant<int, NF>;
    using ALL = std::integral_constant<int, NSLOT>;
    auto fetch_all = [&](auto slot) {
        for (int i = 0; i < NFETCH; ++i) fetch(slot, i);
        next_tile();
    };
    fetch_all(S0{});
    fetch_all(S1{});
    fetch_all(S2{});
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PER_TILE) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    slots(S0{}, FIRST{}, S0{}, S0{}, s_cur, [](auto) {});
    if constexpr (!RD) {
        load_lq(tl(S0{}));
#pragma unroll
        for (int v = 0; v < 16; v += 2) exp_pair(s_cur, v, pw);
        mask(pw);
        post(0, pw);
    }
    if constexpr (STORES > 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_TILE) : "memory");   // tile 1: no store stands behind it yet
    int left = n_it - 1;   // iterations before the last one
    int at = 0;            // tail: the ring slot of the tile (the operand addresses have moved there)
    // One iteration, for the tile in ring slot `buf`; more: another tile follows.  tail: the slot is `at`, not an immediate, and
    // nothing is fetched but the last tile of all.
    auto step = [&](auto buf, auto more_c, auto tail_c) {
        constexpr bool more = decltype(more_c)::value, tail = decltype(tail_c)::value;
        using B1 = std::integral_constant<int, (buf.value + 1) % NR>;
        using BF = std::integral_constant<int, (buf.value + 3) % NR>;
        // tile it + 1 is in LDS (tile it + 2 may still be on its way, and dS stores behind either: no fence, it would wait for them
        // too), P(it) has been posted; every wavefront has left tile it - 1, whose slot is filled next
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(tail ? 0 : PER_TILE + STORES) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int parity = tail ? at & 1 : buf.value & 1;
        if constexpr (RD) {
            float di[16];
            uint32_t p[8];
#pragma unroll
            for (int j = 0; j < 2; ++j) *(uint4*)&p[4 * j] = sP[parity][kb][j][lane];
            const float* rows = td(buf);
            if constexpr (tail) rows = at == 0 ? sD0 : at == 1 ? sD1 : at == 2 ? sD2 : sD3;
#pragma unroll
            for (int g = 0; g < 4; ++g) *(float4*)&di[4 * g] = *(const float4*)&rows[8 * g + 4 * h];
            if constexpr (tail && more)
                if (left == 3) fetch_all(S3{});
            auto ds_pair = [&](int v) {
                const float p0 = __uint_as_float(p[v >> 1] << 16), p1 = __uint_as_float(p[v >> 1] & 0xffff0000u);
                pw[v >> 3][(v & 7) >> 1] = cvt_pk_bf16(p0 * (s_cur[v] - di[v]), p1 * (s_cur[v + 1] - di[v + 1]));
            };
            // the tile as this wavefront's registers hold it, [j][lane][4 words]: lane (key kl, half h) holds, in pw[j][2c],
            // pw[j][2c + 1], the queries 16 j + 8 c + 4 h .. + 3.  Two instructions of 1 KB each, written once and read once: kept
            // out of the way of the tiles the L2 is holding.
            auto spill = [&](int j) {
                __builtin_nontemporal_store(u32x4_t{pw[j][0], pw[j][1], pw[j][2], pw[j][3]}, (u32x4_t*)(ds_tile + lane * 16) + 64 * j);
                if (j == 1) {
                    const bool end = ++se_t == n_qt;
                    ds_tile += end ? ds_step_r : ds_step_t;
                    se_t = end ? 0 : se_t;
                }
            };
            if constexpr (more) {
                // pair i is due at slot NF (i < 4) or NF + DB: from the third slot on, where P has arrived
                slots(S0{}, ALL{}, B1{}, buf, s_nxt, [&](auto xc) {
                    constexpr int x = decltype(xc)::value;
                    if constexpr (x < NFETCH && !tail) fetch(BF{}, x);
                    constexpr int per = D == 128 ? 1 : 2, i0 = (x - (D == 128 ? 2 : 1)) * per;   // D = 64 has half the slots
                    if constexpr (i0 >= 0 && i0 < 8)
#pragma unroll
                        for (int i = i0; i < i0 + per; ++i) ds_pair(2 * i);
                    if constexpr (SPILL && x == NF + 2) spill(0);
                    if constexpr (SPILL && x == NF + 3) spill(1);
                });
                s_cur = s_nxt;
                if constexpr (!tail) next_tile();
            } else {
#pragma unroll
                for (int v = 0; v < 16; v += 2) ds_pair(v);
                if constexpr (SPILL) spill(0), spill(1);
                slots(FIRST{}, ALL{}, B1{}, buf, s_nxt, [](auto) {});
            }
        } else {
            if constexpr (more) {
                const float* rows = tl(B1{});
                if constexpr (tail) rows = at == 0 ? sL1 : at == 1 ? sL2 : sL3;
                load_lq(rows);
                if constexpr (tail)
                    if (left == 3) fetch_all(S3{});
                slots(S0{}, ALL{}, B1{}, buf, s_nxt, [&](auto xc) {
                    constexpr int x = decltype(xc)::value;
                    if constexpr (x < NFETCH && !tail) fetch(BF{}, x);
                    // the scores are complete two slots behind their last MFMA
                    constexpr int y = x - NF - 1, room = NS - 2;
                    if constexpr (y >= 1) {
#pragma unroll
                        for (int i = 8 * (y - 1) / room; i < 8 * y / room; ++i) exp_pair(s_nxt, 2 * i, pw_n);
                    }
                });
                mask(pw_n);
                post(parity ^ 1, pw_n);
                if constexpr (!tail) next_tile();
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int w = 0; w < 4; ++w) pw[j][w] = pw_n[j][w];
            } else {
                slots(FIRST{}, ALL{}, B1{}, buf, s_nxt, [](auto) {});
            }
        }
    };
    const std::true_type more{};
    const std::false_type last{};
    // Four iterations as one block, then up to three and the last one through a single instance of each: with an instance per ring
    // slot the compiler spilled registers at their ends (backward, 8 x 32 x 8 heads, D 128, N 300, not causal: 89.4 us, 77 now; one
    // sequence, 32 / 8 heads, N 2048: 175, 165; N 8192 with dS kept: 1675, 1652).
    const std::false_type ring_slot{};
    const std::true_type tail{};
    for (; left >= 4; left -= 4) step(S0{}, more, ring_slot), step(S1{}, more, ring_slot), step(S2{}, more, ring_slot), step(S3{}, more, ring_slot);
    for (; left > 0; --left) {
        step(S0{}, more, tail);
        ++at;
#pragma unroll
        for (int x = 0; x < NF; ++x) a_row[x] += SLOTB;
#pragma unroll
        for (int x = 0; x < DB; ++x) a_lo[x] += SLOTB, a_hi[x] += SLOTB;
    }
    step(S0{}, last, tail);
    dma_wait_all();        // the fetches past the last tile write LDS: they land before the workgroup gives it back
    };
    if (role_d) run(std::true_type{});
    else run(std::false_type{});
    if (!SPILL && a.part_heads) {
        float4* img = (float4*)a.parts + ((((int64_t)part * n_blocks + bid) * 2 + kb) * 2 + (role_d ? 1 : 0)) * (DB * 4 * 64) + lane;
#pragma unroll
        for (int i = 0; i < DB * 4; ++i)
            img[64 * i] = float4{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
        return;
    }
    __syncthreads();   // every wavefront has left the ring
    {
        const int64_t head = role_d ? (int64_t)b * a.s_dk[0] + (int64_t)kvh * a.s_dk[1] : (int64_t)b * a.s_dv[0] + (int64_t)kvh * a.s_dv[1];
        const int64_t pitch = role_d ? a.s_dk[2] : a.s_dv[2];
        store_rows<D>((lds_char_t*)ring + wave * (32 * D * 2), acc, role_d ? a.scale : 1.f, lane, role_d ? a.dk : a.dv,
                             [&](int r) { return key0 + r < a.N ? head + (int64_t)(key0 + r) * pitch : (int64_t)-1; });
    }
#endif
}

template <int D, bool SPILL>
__global__ void __launch_bounds__(256, 2) bwd_dkdv_bf16_kernel(BwdArgs a, BwdDivisors d) {   // by itself: where dS is kept
    bwd_dkdv_bf16<D, SPILL>(a, d, (int)blockIdx.x);
}

// ---- LDS of a launch that holds both passes ----
// A workgroup is of one of them.  The dK / dV pass's LDS are variables (the compiler has to see that its reads of one do not touch a fetch into
// another); the dQ pass, whose reads are all laid out by hand, uses the same bytes from the start on.
__device__ inline lds_char_t* lds_start() {
    uint32_t at = 0;
    asm("" : "+s"(at));   // a literal zero would be the null pointer, which is another address there
    return (lds_char_t*)(uintptr_t)at;
}
// ---- dQ (bf16) ----
// Rows are all query heads' of a kv head, token by token, as in the forward (prefill.hip: a block of rows spans fewer tokens, which end closer to one another under the
// causal mask; 16 / 4 heads, D 128, 5 x 591, whole step 71.7 -> 68.8 us with the stores above).
// S^T = K Q^T, dP^T = V dO^T, dQ^T += K^T dS^T, as bwd_dq_kernel, R row groups of 32 queries times G key groups: key group g takes the tiles g, g + G, ..., and the G sums of
// a row group meet in LDS at the end (dq_row_groups() says which shape runs when).  The stream is laid out by hand, as in bwd_dq_split: an
// iteration is groups of two MFMAs, first the first products of the key group's next tile (S and dP in turn), then the second products of this
// tile; behind each MFMA stand the LDS operands of the group kAhead ahead, dS of this tile under the next one's first products, the fetch.  Two wavefronts share a
// SIMD (three at head_dim 64), in a launch with the dK / dV pass's.  What bounds it is vector and LDS issue beside the MFMAs.
template <int D, int R, int G>
__device__ __forceinline__ void bwd_dq_bf16(const BwdArgs& a, const BwdDivisors& d, int bid) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    static_assert(R * G == 4);
    constexpr int KS = D / 16, DB = D / 32, ROWS = 32 * R;
    constexpr int NF = KS, NS = DB, NG = NF + NS;          // groups of two MFMAs: first products (S and dP), second products (two column blocks of dQ)
    constexpr int kAhead = D == 128 ? 3 : 2;               // groups from an operand's request to its use
    constexpr int LEAD = G == 1 ? 3 : 2;                   // iterations from a tile's request to its second products
    // D 128, G 1: rings of one length, so that four iterations have their slots as immediate offsets (1 to 2 % of a full grid's whole backward against
    // adding them; at D 64 the registers of three wavefronts per SIMD do not take it: 0.5 to 1.5 % slower)
    constexpr bool IMM = G == 1 && D == 128;
    constexpr int NK = LEAD + 1, NV = IMM ? NK : LEAD;
    constexpr int TILEB = kBT * D * 2, GROUPB = (NK + NV) * TILEB;
    static_assert(G * GROUPB <= kPassLds<D>);
    lds_char_t* const ring = lds_start();
    const int rows = a.N * a.n_rep;   // of a kv head
    const int n_qtiles = (rows + ROWS - 1) / ROWS;
    const uint32_t from_last = d.by_bkv.div((uint32_t)bid), bh = d.by_bkv.mod((uint32_t)bid, from_last), ub = d.by_hkv.div(bh);
    const int qt = n_qtiles - 1 - (int)from_last, b = (int)ub, kvh = (int)d.by_hkv.mod(bh, ub);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = wave % R, group = wave / R;
    const int ql = lane & 31, h = lane >> 5;
    const int q0 = qt * ROWS + row * 32;
    // this lane's row: query (token) qi of head hq
    const uint32_t ur = (uint32_t)min(q0 + ql, rows - 1), ut = d.by_rep.div(ur);
    const int qi = (int)ut, hq = kvh * a.n_rep + (int)d.by_rep.mod(ur, ut);
    const int t_first = (int)d.by_rep.div((uint32_t)q0);   // of the wavefront's rows

    const int wg_qmax = (int)d.by_rep.div((uint32_t)min(qt * ROWS + ROWS - 1, rows - 1));
    const int kv_end_wg = a.causal ? wg_qmax + 1 : a.N;
    const int n_it = (kv_end_wg + kBT * G - 1) / (kBT * G);   // stages of G key tiles
    // of which this wavefront's key group has work for its rows
    const int kv_end_wave = q0 < rows ? (a.causal ? (int)d.by_rep.div((uint32_t)min(q0 + 31, rows - 1)) + 1 : a.N) : 0;
    const int n_w = max(((kv_end_wave + kBT - 1) / kBT - group + G - 1) / G, 0);

    // The tile being fetched, as running scalars: its first rows, the bytes from there to the end of the head, its ring slots.  Past the last tile
    // nothing is in range.
    TileDma<D, R> dk_, dv_;
    dk_.init(a.s_k[2], a.N, row, lane);
    dv_.init(a.s_v[2], a.N, row, lane);
    constexpr int NLD = TileDma<D, R>::NLD, NFETCH = 2 * NLD, PERG = (NFETCH + NF - 1) / NF;   // instructions of a tile's fetch; behind each group
    const int64_t row_k = a.s_k[2] * 2, row_v = a.s_v[2] * 2;   // bytes
    const char* pk = (const char*)a.k + ((int64_t)b * a.s_k[0] + (int64_t)kvh * a.s_k[1]) * 2 + group * kBT * row_k;
    const char* pv = (const char*)a.v + ((int64_t)b * a.s_v[0] + (int64_t)kvh * a.s_v[1]) * 2 + group * kBT * row_v;
    // (a head spans less than 2^31 bytes, a step of a few rows far apart may be more)
    int nk = (int)(max(a.N - group * kBT, 0) * row_k), nv = (int)(max(a.N - group * kBT, 0) * row_v), fk = 0, fv = 0;
    const int step_k = (int)min(G * kBT * row_k, (int64_t)INT32_MAX), step_v = (int)min(G * kBT * row_v, (int64_t)INT32_MAX);
    lds_char_t* const mine = ring + group * GROUPB;
    auto fetch = [&](int i) {   // K, V: NLD instructions each
        const bool is_v = i >= NLD;
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(is_v ? pv : pk), 0, max(is_v ? nv : nk, 0), 0x00020000);
        lds_char_t* dst = mine + (is_v ? NK * TILEB + fv * TILEB : fk * TILEB) + (row + R * (i % NLD)) * 1024;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 16, (is_v ? dv_ : dk_).voff[i % NLD], 0, 0, 0);
    };
    auto next_tile = [&]() {
        pk += G * kBT * row_k, pv += G * kBT * row_v;
        nk -= nk > 0 ? step_k : 0, nv -= nv > 0 ? step_v : 0;
        fk = fk + 1 == NK ? 0 : fk + 1;
        fv = fv + 1 == NV ? 0 : fv + 1;
    };
    for (int t = 0; t < LEAD; ++t) {
#pragma unroll
        for (int i = 0; i < NFETCH; ++i) fetch(i);
        next_tile();
    }

    const uint16_t* Qp = (const uint16_t*)a.q + (int64_t)b * a.s_q[0] + (int64_t)hq * a.s_q[1] + (int64_t)qi * a.s_q[2];
    const uint16_t* Op = (const uint16_t*)a.dout + (int64_t)b * a.s_do[0] + (int64_t)hq * a.s_do[1] + (int64_t)qi * a.s_do[2];
    bf16x8_t qf[KS], dof[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        qf[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Qp + 16 * ks + 8 * h));
        dof[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Op + 16 * ks + 8 * h));
    }
    const float di_q = a.delta[((int64_t)b * a.Hq + hq) * a.N + qi];
    const float lse_q = a.lse2[((int64_t)b * a.Hq + hq) * a.N + qi];
    const float scale_log2 = a.scale * kLog2e;
    const int lim = a.causal ? qi : a.N - 1;   // the last key this lane's query sees

    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;

    // operand addresses within a tile (see load_row, load_transposed)
    const uint32_t lds0 = (uint32_t)(uintptr_t)mine;
    uint32_t a_row[NF], a_lo[DB], a_hi[DB];
#pragma unroll
    for (int ks = 0; ks < NF; ++ks) a_row[ks] = lds0 + (uint32_t)tile_off<D>(lane & 31, 2 * ks + h);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        const int r = 4 * h + ((lane & 15) >> 2), chunk = 4 * db + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), o8 = (lane & 1) * 8;
        a_lo[db] = lds0 + (uint32_t)(tile_off<D>(r, chunk) + o8);
        a_hi[db] = lds0 + (uint32_t)(tile_off<D>(r + 8, chunk) + o8);
    }

    uint32_t pw[2][4];   // dS of this tile, bf16 pairs
    float e0 = 0.f, e1 = 0.f;
    // dS of a pair of positions in two halves
    auto ds_half = [&](const f32x16_t& s, const f32x16_t& dp, int v, int half) {
        if (half == 0) {
            e0 = __builtin_amdgcn_exp2f(fmaf(s[v], scale_log2, -lse_q));
            e1 = __builtin_amdgcn_exp2f(fmaf(s[v + 1], scale_log2, -lse_q));
        } else {
            pw[v >> 3][(v & 7) >> 1] = cvt_pk_bf16(e0 * (dp[v] - di_q), e1 * (dp[v + 1] - di_q));
        }
    };
    // dS of masked positions is 0, whatever came of their scores: done on the finished words, in the tiles that the diagonal or the end crosses
    auto mask = [&](int k0) {
        if ((a.causal && k0 + kBT - 1 > t_first) || k0 + kBT > a.N) {   // same for the wavefront
            const int n = lim - (k0 + 4 * h) + 1;
            const uint32_t seen = n >= 32 ? ~0u : n <= 0 ? 0u : (1u << n) - 1u;
#pragma unroll
            for (int v = 0; v < 16; v += 2)
                pw[v >> 3][(v & 7) >> 1] &= (bit_mask(seen, 8 * (v >> 2) + (v & 3)) & 0x0000ffffu) | (bit_mask(seen, 8 * (v >> 2) + (v & 3) + 1) & 0xffff0000u);
        }
    };
    // The groups FROM .. TO - 1 of an iteration: first products of the tile in the slots at kn, vn (bytes from the ring's start) into s, dp; second
    // products of the tile whose K is at kc; slots as scalars, which are added to the addresses, or as immediate offsets.  work(group, u) is what is placed behind MFMA u of a group; between() stands before the second products.
    auto row_at = [](uint32_t at, auto slot) {
        if constexpr (std::is_same_v<decltype(slot), uint32_t>) return ds_b128<0>(at + slot);
        else return ds_b128<slot.value>(at);
    };
    auto col_at = [](uint32_t at, auto slot, auto o) {
        if constexpr (std::is_same_v<decltype(slot), uint32_t>) return ds_tr16<o.value>(at + slot);
        else return ds_tr16<slot.value + o.value>(at);
    };
    auto groups = [&](auto from, auto to, auto kn, auto vn, auto kc, f32x16_t& s, f32x16_t& dp, auto&& work, auto&& between) {
        constexpr int FROM = decltype(from)::value, TO = decltype(to)::value;
        u32x4_t kr[NF], vr[NF];
        uint2 tr[NS][2][2];   // [group][column block of the two][rows + 0, + 8]
        auto request = [&](auto xc, auto piece) {   // the reads of group x in two pieces
            constexpr int x = decltype(xc)::value, p = decltype(piece)::value;
            if constexpr (x < NF && x < TO) {
                if constexpr (p == 0) kr[x] = row_at(a_row[x], kn);
                else vr[x] = row_at(a_row[x], vn);
            } else if constexpr (x < TO) {
                constexpr int g = x - NF, j = g / (DB / 2), db = 2 * (g % (DB / 2)) + p, o = j * 16 * 2 * D;
                tr[g][p][0] = col_at(a_lo[db], kc, std::integral_constant<int, o>{});
                tr[g][p][1] = col_at(a_hi[db], kc, std::integral_constant<int, o>{});
            }
        };
        using P0 = std::integral_constant<int, 0>;
        using P1 = std::integral_constant<int, 1>;
        for_each<kAhead>([&](auto i) {
            using X = std::integral_constant<int, FROM + i.value>;
            request(X{}, P0{}), request(X{}, P1{});
        });
        for_each<TO - FROM>([&](auto ic) {
            constexpr int x = FROM + ic.value;
            using AHEAD = std::integral_constant<int, x + kAhead>;
            // reads of the groups behind this one that have been requested
            constexpr int last = x + kAhead - 1 < TO - 1 ? x + kAhead - 1 : TO - 1;
            constexpr int firsts = last < NF ? last - x : x < NF ? NF - 1 - x : 0;
            constexpr int behind = 2 * firsts + 4 * (last - x - firsts);
            if constexpr (x == NF) between();
            __builtin_amdgcn_sched_barrier(0);
            auto mf = [&](f32x16_t& c, u32x4_t op, bf16x8_t y, bool zero) {
                const f32x16_t z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, op), y, zero ? z : c, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            if constexpr (x < NF) {
                asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(kr[x]), "+v"(vr[x]) : "n"(behind));
                mf(s, kr[x], qf[x], x == 0);
                request(AHEAD{}, P0{}), work(x, 0), __builtin_amdgcn_sched_barrier(0);
                mf(dp, vr[x], dof[x], x == 0);
                request(AHEAD{}, P1{}), work(x, 1);
            } else {
                constexpr int g = x - NF, j = g / (DB / 2), db = 2 * (g % (DB / 2));
                asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(tr[g][0][0]), "+v"(tr[g][0][1]), "+v"(tr[g][1][0]), "+v"(tr[g][1][1]) : "n"(behind));
                const bf16x8_t ph = __builtin_bit_cast(bf16x8_t, u32x4_t{pw[j][0], pw[j][1], pw[j][2], pw[j][3]});
                auto cat = [](const uint2 (&t)[2]) { return u32x4_t{t[0].x, t[0].y, t[1].x, t[1].y}; };
                mf(acc[db], cat(tr[g][0]), ph, false);
                request(AHEAD{}, P0{}), work(x, 0), __builtin_amdgcn_sched_barrier(0);
                mf(acc[db + 1], cat(tr[g][1]), ph, false);
                request(AHEAD{}, P1{}), work(x, 1);
            }
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    using G0 = std::integral_constant<int, 0>;
    using GF = std::integral_constant<int, NF>;
    using GA = std::integral_constant<int, NG>;
    auto nothing = [](int, int) {};
    auto none = []() {};
    uint32_t kc = 0, kn = TILEB, vn = NK * TILEB + TILEB;   // slots of this tile's K, of the next tile's K and V
    // tile it + 1 is in LDS (younger requests may be on their way: no fence, it would wait for them too); every wavefront has left K of tile it - 1 and
    // V of tile it, whose slots are filled next
    auto arrive = [&]() {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((LEAD - 2) * NFETCH) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto advance = [&]() {
        next_tile();
        kc = kn;
        kn = kn + TILEB == NK * TILEB ? 0 : kn + TILEB;
        vn = vn + TILEB == (NK + NV) * TILEB ? NK * TILEB : vn + TILEB;
    };
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((LEAD - 1) * NFETCH) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int it = 0;
    if (n_w > 0) {
        f32x16_t s0, dp0, s1, dp1;
        groups(G0{}, GF{}, 0u, (uint32_t)(NK * TILEB), 0u, s0, dp0, nothing, none);
        int k0 = group * kBT;
        // one iteration: this tile's scores in s, dp, the next tile's into s2, dp2
        auto step = [&](f32x16_t& s, f32x16_t& dp, f32x16_t& s2, f32x16_t& dp2, auto next_k, auto next_v, auto cur_k) {
            arrive();
            groups(G0{}, GA{}, next_k, next_v, cur_k, s2, dp2, [&](int x, int u) {
                if (x < NF) {
#pragma unroll
                    for (int i = 0; i < PERG; ++i)
                        if (i % 2 == u && x * PERG + i < NFETCH) fetch(x * PERG + i);
                    if constexpr (NF == 8) ds_half(s, dp, 2 * x, u);
                    else ds_half(s, dp, 4 * x + 2 * u, 0), ds_half(s, dp, 4 * x + 2 * u, 1);   // a pair under each MFMA
                }
            }, [&]() { mask(k0); });
            k0 += G * kBT;
        };
        if constexpr (IMM) {
            auto in_slot = [&](auto c, f32x16_t& s, f32x16_t& dp, f32x16_t& s2, f32x16_t& dp2) {
                constexpr int n = (c.value + 1) % NK;
                step(s, dp, s2, dp2, std::integral_constant<int, n * TILEB>{}, std::integral_constant<int, (NK + n) * TILEB>{}, std::integral_constant<int, c.value * TILEB>{});
                next_tile();
            };
            for (; it + 4 < n_w; it += 4) {
                in_slot(std::integral_constant<int, 0>{}, s0, dp0, s1, dp1), in_slot(std::integral_constant<int, 1>{}, s1, dp1, s0, dp0);
                in_slot(std::integral_constant<int, 2>{}, s0, dp0, s1, dp1), in_slot(std::integral_constant<int, 3>{}, s1, dp1, s0, dp0);
            }
            for (; it + 1 < n_w; ++it) {
                step(s0, dp0, s1, dp1, kn, vn, kc);
                advance();
                s0 = s1, dp0 = dp1;
            }
        } else {
            for (; it + 2 < n_w; it += 2) {
                step(s0, dp0, s1, dp1, kn, vn, kc);
                advance();
                step(s1, dp1, s0, dp0, kn, vn, kc);
                advance();
            }
            if (it + 1 < n_w) {
                step(s0, dp0, s1, dp1, kn, vn, kc);
                advance();
                s0 = s1, dp0 = dp1;
                ++it;
            }
        }
        arrive();
#pragma unroll
        for (int i = 0; i < NFETCH; ++i) fetch(i);
#pragma unroll
        for (int v = 0; v < 16; v += 2) ds_half(s0, dp0, v, 0), ds_half(s0, dp0, v, 1);
        groups(GF{}, GA{}, kn, vn, kc, s1, dp1, nothing, [&]() { mask(k0); });
        advance();
        ++it;
    }
    for (; it < n_it; ++it) {   // the other wavefronts' tiles
        arrive();
#pragma unroll
        for (int i = 0; i < NFETCH; ++i) fetch(i);
        next_tile();
    }
    dma_wait_all();        // the fetches past the last tile write LDS: they land before the workgroup gives it back
    if constexpr (G == 1) {
        __syncthreads();   // every wavefront has left the ring
        store_rows<D>(ring + wave * (32 * D * 2), acc, a.scale, lane, a.dq, [&](int r) {
            const uint32_t i = (uint32_t)(q0 + r), t = d.by_rep.div(i);
            return q0 + r < rows ? (int64_t)b * a.s_dq[0] + (int64_t)(kvh * a.n_rep + (int)d.by_rep.mod(i, t)) * a.s_dq[1] + (int64_t)t * a.s_dq[2] : (int64_t)-1;
        });
    } else {   // the key groups' sums meet in the ring; each wavefront adds and stores a G-th of its rows' columns
        const uint32_t i0 = (uint32_t)min(q0 + ql, rows - 1), t0 = d.by_rep.div(i0);
        const int64_t out_row = (int64_t)b * a.s_dq[0] + (int64_t)(kvh * a.n_rep + (int)d.by_rep.mod(i0, t0)) * a.s_dq[1] + (int64_t)t0 * a.s_dq[2];
        __syncthreads();
        constexpr int NQ = 4 * DB, MINE = NQ / G;
        auto image = [&](int w) { return (lds_f32x4_t*)ring + w * (NQ * 64) + lane; };
#pragma unroll
        for (int i = 0; i < NQ; ++i) image(wave)[64 * i] = f32x4_t{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
        __syncthreads();
        if (q0 + ql < rows)
#pragma unroll
            for (int i = 0; i < MINE; ++i) {
                f32x4_t sum = image(row)[64 * (MINE * group + i)];
#pragma unroll
                for (int g = 1; g < G; ++g) sum += image(row + g * R)[64 * (MINE * group + i)];
                store_quad<false>(a.dq, out_row + 8 * (MINE * group + i) + 4 * h, a.scale, sum);
            }
    }
#endif
}

// Both passes in one launch, as bwd_split_pass_kernel.  Di comes from a launch of its own (which is what the dQ pass's prologue took and what the dK / dV pass
// would have to wait for).  Forward and backward, two launches with the compiler's schedule of the dQ pass -> this, us: 16 heads, D 128, 180 tokens 23.6 -> 18.3;
// 32 / 8, D 128, 1 x 8192 2284 -> 2202, 4 x 64 / 8 heads, 1054, not causal 781 -> 673, 8 / 2, D 64, 3 x 5849 582 -> 530; 16 heads, D 64, 8 x 5431 2363 -> 2391 (reading O and
// dO ahead of the passes); 60 drawn shapes 1.07 (0.97 to 1.29).  The passes of the same code in two launches, Di from the dQ pass: 9 % slower.
template <int D, int R, int G>
__global__ void __launch_bounds__(256, D == 64 ? 3 : 2) bwd_pass_kernel(BwdArgs a, BwdDivisors d, int n_dkdv) {
    if constexpr (kPassLds<D> > kDkdvLds<D>) {
        __shared__ __attribute__((aligned(256))) char rest[kPassLds<D> - kDkdvLds<D>];
        asm volatile("" ::"v"(lds_byte_addr(rest)));   // part of the workgroup's LDS, whatever the dQ pass's shape needs of it
    }
    if ((int)blockIdx.x < n_dkdv) bwd_dkdv_bf16<D, false>(a, d, (int)blockIdx.x);
    else bwd_dq_bf16<D, R, G>(a, d, (int)blockIdx.x - n_dkdv);
}

// ---- dK, dV of the split-operand path ----
// The pairs of wavefronts of bwd_dkdv_bf16 with the hi and lo tiles of Q and dO in every ring slot (one workgroup per CU,
// one wavefront per SIMD), three MFMAs per operand pair (hi hi + hi lo + lo hi), P crossing to the partner as fp32 and what feeds a
// second product (P or dS) split into two bf16 terms.  With nothing else on the SIMD, whatever a wavefront waits for is lost,
// so its stream is laid out by hand.  An iteration is 16 groups of three MFMAs (96 cycles): first the first products of
// tile t + 1 (S or dP), then the second products of tile t (dV or dK).  Behind each MFMA stand a few of the other
// instructions: the LDS operands of the group kLead groups ahead, the D wavefront's dS(t) = P (dP - Di) under its dP(t + 1), the P
// wavefront's exp of S(t + 1) under its dV(t), one instruction of the next tile's fetch per group.  No branch in an iteration but the
// mask's: fetches past the end ask for nothing, and the last iteration is its own instance.  As an instance of the bf16 kernel this
// pass took 421 us (one sequence, 32 / 8 heads, D 128, 2048 tokens) and 1.2 ms (four); the stream brought it to 311, the parts
// (plan_parts) to 200 and the fourth ring slot the batch of four to 740.
template <int D>
__device__ __forceinline__ void bwd_dkdv_split(const BwdArgs& a, int block) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    constexpr int KS = D / 16, DB = D / 32;
    constexpr int kLead = 3;
    // Ring slots: at head_dim 128 four (150 KB of LDS), a tile has two iterations to arrive (-4 % on a full grid, where it comes
    // from past the L2); at 64 three, which lets a CU hold two workgroups.
    constexpr int NR = D == 128 ? 4 : 3;
    __shared__ __attribute__((aligned(1024))) uint16_t sQ0[kBT * D], sQ1[kBT * D], sQ2[kBT * D], sQ3[NR == 4 ? kBT * D : 8];
    __shared__ __attribute__((aligned(1024))) uint16_t sO0[kBT * D], sO1[kBT * D], sO2[kBT * D], sO3[NR == 4 ? kBT * D : 8];
    __shared__ __attribute__((aligned(1024))) uint16_t sQl0[kBT * D], sQl1[kBT * D], sQl2[kBT * D], sQl3[NR == 4 ? kBT * D : 8];
    __shared__ __attribute__((aligned(1024))) uint16_t sOl0[kBT * D], sOl1[kBT * D], sOl2[kBT * D], sOl3[NR == 4 ? kBT * D : 8];
    __shared__ __attribute__((aligned(256))) float sL0[64], sL1[64], sL2[64], sL3[64];   // lse and Di of the tile's rows
    __shared__ __attribute__((aligned(256))) float sD0[64], sD1[64], sD2[64], sD3[64];
    __shared__ __attribute__((aligned(1024))) float4 sP[NR == 4 ? 2 : 3][2][4][64];   // [tile][key block][quad][lane]: posted in one iteration, read in the next
    static_assert(NR * (sizeof(sQ0) + sizeof(sO0) + sizeof(sQl0) + sizeof(sOl0) + sizeof(sL0) + sizeof(sD0)) + sizeof(sP) == kDkdvSplitLds<D>);   // (a fourth slot that is not used takes nothing)
    auto pick = [](auto s, auto* x0, auto* x1, auto* x2, auto* x3) { if constexpr (s.value == 0) return x0; else if constexpr (s.value == 1) return x1; else if constexpr (s.value == 2) return x2; else return x3; };
    auto tq = [&](auto s) { return pick(s, sQ0, sQ1, sQ2, sQ3); };
    auto to = [&](auto s) { return pick(s, sO0, sO1, sO2, sO3); };
    auto tql = [&](auto s) { return pick(s, sQl0, sQl1, sQl2, sQl3); };
    auto tol = [&](auto s) { return pick(s, sOl0, sOl1, sOl2, sOl3); };
    auto tl = [&](auto s) { return pick(s, sL0, sL1, sL2, sL3); };
    auto td = [&](auto s) { return pick(s, sD0, sD1, sD2, sD3); };
    const int n_blocks = (a.N + kBK - 1) / kBK * a.B * a.Hkv;
    const int part = a.part_heads ? block / n_blocks : 0;
    const int bid = a.part_heads ? block % n_blocks : block;
    const int kt = bid / (a.B * a.Hkv);          // causal work falls with the key tile: heaviest first
    const int bh = bid % (a.B * a.Hkv);
    const int b = bh / a.Hkv, kvh = bh % a.Hkv;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kb = wave >> 1;
    const bool role_d = wave & 1;
    const int kl = lane & 31, h = lane >> 5;
    const int key0 = kt * kBK + kb * 32;
    const int ki = key0 + kl;
    const int krow = min(ki, a.N - 1);

    // the stationary operand: K rows for the P wavefront, V rows for the D wavefront
    const uint16_t* Xp = role_d ? (const uint16_t*)a.v + (int64_t)b * a.s_v[0] + (int64_t)kvh * a.s_v[1] + (int64_t)krow * a.s_v[2]
                                : (const uint16_t*)a.k + (int64_t)b * a.s_k[0] + (int64_t)kvh * a.s_k[1] + (int64_t)krow * a.s_k[2];
    bf16x8_t xf[KS], xfl[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        xf[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Xp + 16 * ks + 8 * h));
        xfl[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Xp + a.lo_kv + 16 * ks + 8 * h));
    }
    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;

    const int qt_begin = a.causal ? (kt * kBK) / kBT : 0;
    const int n_qt = (a.N + kBT - 1) / kBT - qt_begin;   // query tiles per head
    int r0 = 0, r1 = a.n_rep, t0 = 0, t1 = n_qt;         // heads of the group, query tiles from the last one down
    if (a.part_heads) {                                  // this workgroup's part of them
        r0 = part / a.part_ranges * a.part_heads;
        r1 = min(a.n_rep, r0 + a.part_heads);
        t0 = part % a.part_ranges * a.part_tiles;
        t1 = min(n_qt, t0 + a.part_tiles);
        if (t0 >= t1) return;                            // a lighter key block has fewer tiles
    }
    const int n_it = (r1 - r0) * (t1 - t0);              // the loop runs over (head of the group, query tile)
    const float scale_log2 = a.scale * kLog2e;

    TileDma<D> dq_, do_;
    dq_.init(a.s_q[2], a.N, wave, lane);
    do_.init(a.s_do[2], a.N, wave, lane);
    // The tile being fetched, as running addresses (the stride arithmetic of a tile is a hundred scalar instructions): the
    // first row of its hi tiles, the bytes from there to the end of the head, and its row constants.
    const int64_t step_q = (int64_t)kBT * a.s_q[2] * 2, step_o = (int64_t)kBT * a.s_do[2] * 2;   // bytes per tile
    const int n_tl = t1 - t0;
    const char *pq, *po;
    const float* pr;   // lse (even wavefronts) or Di (odd ones: two write the same words)
    int nq, no, nr, ld_t = 0, n_left = n_it;
    {
        const int hq = kvh * a.n_rep + r0, qb = (qt_begin + (n_qt - 1 - t0)) * kBT;
        pq = (const char*)((const uint16_t*)a.q + (int64_t)b * a.s_q[0] + (int64_t)hq * a.s_q[1] + (int64_t)qb * a.s_q[2]);
        po = (const char*)((const uint16_t*)a.dout + (int64_t)b * a.s_do[0] + (int64_t)hq * a.s_do[1] + (int64_t)qb * a.s_do[2]);
        pr = ((wave & 1) ? a.delta : a.lse2) + ((int64_t)b * a.Hq + hq) * a.N + qb;
        nr = a.N - qb;
        nq = (int)((int64_t)nr * a.s_q[2] * 2);
        no = (int)((int64_t)nr * a.s_do[2] * 2);
    }
    const int64_t head_q = a.s_q[1] * 2 + (n_tl - 1) * step_q, head_o = a.s_do[1] * 2 + (n_tl - 1) * step_o;   // last tile of a head to the first of the next
    const int64_t lo_b = a.lo_q * 2;
    constexpr int NLD = TileDma<D>::NLD;
    // one instruction of the fetch: the NLD of Q hi, dO hi, Q lo, dO lo in turn (and the row constants with the first)
    auto fetch = [&](auto buf, int i) {
        const bool is_q = (i / NLD) % 2 == 0, lo = i / NLD >= 2;
        const char* base = (is_q ? pq : po) + (lo ? lo_b : 0);
        uint16_t* dst = is_q ? (lo ? tql(buf) : tq(buf)) : (lo ? tol(buf) : to(buf));
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, is_q ? nq : no, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)((char*)dst + (wave + 4 * (i % NLD)) * 1024), 16, (is_q ? dq_ : do_).voff[i % NLD], 0, 0, 0);
        if (i == 0) row_dma((wave & 1) ? td(buf) : tl(buf), pr, max(min(nr, kBT), 0), 1, lane);
    };
    // past the last tile the fetch goes on with nothing in range (zeros, no memory touched): no branch in the steady state
    auto next_tile = [&]() {
        if (--n_left <= 0) {
            nq = no = nr = 0;
        } else if (++ld_t == n_tl) {
            ld_t = 0;
            pq += head_q, po += head_o;
            pr += a.N + (n_tl - 1) * kBT;
            nr -= (n_tl - 1) * kBT;
            nq -= (int)((n_tl - 1) * step_q), no -= (int)((n_tl - 1) * step_o);
        } else {
            pq -= step_q, po -= step_o;
            pr -= kBT;
            nr += kBT;
            nq += (int)step_q, no += (int)step_o;
        }
    };
    int fi_t = t0;   // query tile of the tile whose first products are due
    // The loop exists once per role, so that each wavefront's code reads its tiles from named variables.
    auto run = [&](auto role) {
    constexpr bool RD = decltype(role)::value;
    constexpr int NF = KS, NS = 2 * DB;          // groups of the first and of the second products
    constexpr int PF = 8 / NF, PS = 8 / NS;      // pairs of elements of the vector-ALU work per group
    auto rows_hi = [&](auto buf) { if constexpr (RD) return to(buf); else return tq(buf); };
    auto rows_lo = [&](auto buf) { if constexpr (RD) return tol(buf); else return tql(buf); };
    auto cols_hi = [&](auto buf) { if constexpr (RD) return tq(buf); else return to(buf); };
    auto cols_lo = [&](auto buf) { if constexpr (RD) return tql(buf); else return tol(buf); };
    // two bf16 terms of a pair of values, in two halves: x0, x1 -> hi, and what is left -> lo
    float x0 = 0.f, x1 = 0.f;
    uint32_t xw = 0;
    auto term_hi = [&](int v, uint32_t (&hi)[2][4]) { hi[v >> 3][(v & 7) >> 1] = xw = cvt_pk_bf16(x0, x1); };
    auto term_lo = [&](int v, uint32_t (&lo)[2][4]) { lo[v >> 3][(v & 7) >> 1] = cvt_pk_bf16(x0 - __uint_as_float(xw << 16), x1 - __uint_as_float(xw & 0xffff0000u)); };
    // First products of a tile (S or dP) into s; `work(g, u)` is what is placed behind MFMA u of group g.
    auto first = [&](auto buf, f32x16_t& s, auto&& work) {
        const uint16_t *th = rows_hi(buf), *tlo = rows_lo(buf);
        bf16x8_t oh[NF], ol[NF];
#pragma unroll
        for (int g = 0; g < kLead; ++g) oh[g] = load_row<D>(th, g, lane), ol[g] = load_row<D>(tlo, g, lane);
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = 0.f;
#pragma unroll
        for (int g = 0; g < NF; ++g) {
            __builtin_amdgcn_sched_barrier(0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(oh[g], xf[g], s, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (g + kLead < NF) oh[g + kLead] = load_row<D>(th, g + kLead, lane), ol[g + kLead] = load_row<D>(tlo, g + kLead, lane);
            work(g, 0);
            __builtin_amdgcn_sched_barrier(0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(oh[g], xfl[g], s, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            work(g, 1);
            __builtin_amdgcn_sched_barrier(0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ol[g], xf[g], s, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            work(g, 2);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Second products of a tile: acc += (dO or Q)^T (P or dS)
    auto second = [&](auto buf, const uint32_t (&pw)[2][4], const uint32_t (&pl)[2][4], auto&& work) {
        const uint16_t *th = cols_hi(buf), *tlo = cols_lo(buf);
        bf16x8_t oh[NS], ol[NS];
#pragma unroll
        for (int g = 0; g < kLead; ++g) oh[g] = load_transposed<D>(th, g / DB, g % DB, lane), ol[g] = load_transposed<D>(tlo, g / DB, g % DB, lane);
        bf16x8_t ph[2], plo[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            ph[j] = __builtin_bit_cast(bf16x8_t, uint4{pw[j][0], pw[j][1], pw[j][2], pw[j][3]});
            plo[j] = __builtin_bit_cast(bf16x8_t, uint4{pl[j][0], pl[j][1], pl[j][2], pl[j][3]});
        }
#pragma unroll
        for (int g = 0; g < NS; ++g) {
            const int j = g / DB, db = g % DB, g2 = g + kLead;
            __builtin_amdgcn_sched_barrier(0);
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(oh[g], ph[j], acc[db], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (g2 < NS) oh[g2] = load_transposed<D>(th, g2 / DB, g2 % DB, lane), ol[g2] = load_transposed<D>(tlo, g2 / DB, g2 % DB, lane);
            work(g, 0);
            __builtin_amdgcn_sched_barrier(0);
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(oh[g], plo[j], acc[db], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            work(g, 1);
            __builtin_amdgcn_sched_barrier(0);
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ol[g], ph[j], acc[db], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            work(g, 2);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // P of a tile from its scores; lse and masked positions as in bwd_dkdv_bf16
    float lq[16], p_out[16];
    bool edge = false;
    uint32_t seen = 0;
    auto load_lq = [&](auto buf) {
#pragma unroll
        for (int g = 0; g < 4; ++g) *(float4*)&lq[4 * g] = *(const float4*)&tl(buf)[8 * g + 4 * h];
        const int qb = (qt_begin + (n_qt - 1 - fi_t)) * kBT;
        if (++fi_t == t1) fi_t = t0;
        edge = (a.causal && qb < key0 + 31) || qb + kBT > a.N || key0 + 32 > a.N;   // same for the wavefront
        if (edge) seen = rows_that_see(a, ki, qb + 4 * h);
    };
    auto mask = [&](uint32_t (&hi)[2][4], uint32_t (&lo)[2][4]) {
        if (edge)
#pragma unroll
            for (int v = 0; v < 16; v += 2) {
                const uint32_t k0 = bit_mask(seen, 8 * (v >> 2) + (v & 3)), k1 = bit_mask(seen, 8 * (v >> 2) + (v & 3) + 1);
                const uint32_t pair = (k0 & 0x0000ffffu) | (k1 & 0xffff0000u);
                p_out[v] = __uint_as_float(__float_as_uint(p_out[v]) & k0);
                p_out[v + 1] = __uint_as_float(__float_as_uint(p_out[v + 1]) & k1);
                hi[v >> 3][(v & 7) >> 1] &= pair;
                lo[v >> 3][(v & 7) >> 1] &= pair;
            }
    };
    auto exp_hi = [&](const f32x16_t& s, int v, uint32_t (&hi)[2][4]) {
        p_out[v] = x0 = __builtin_amdgcn_exp2f(fmaf(s[v], scale_log2, -lq[v]));
        p_out[v + 1] = x1 = __builtin_amdgcn_exp2f(fmaf(s[v + 1], scale_log2, -lq[v + 1]));
        term_hi(v, hi);
    };
    auto post = [&](auto buf) {
#pragma unroll
        for (int g = 0; g < 4; ++g) sP[NR == 4 ? buf.value & 1 : buf.value][kb][g][lane] = float4{p_out[4 * g], p_out[4 * g + 1], p_out[4 * g + 2], p_out[4 * g + 3]};
    };

    f32x16_t s_cur, s_nxt;                                  // D: dP of this tile and of the next; P: scores of the next
    uint32_t pw[2][4], pl[2][4], pw_n[2][4], pl_n[2][4];    // what the second products of this tile (the next tile) take
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    constexpr int PER_TILE = 4 * NLD + 1;   // memory instructions per wavefront and tile
    auto nothing = [](int, int) {};
    auto fetch_all = [&](auto slot) {
        for (int i = 0; i < 4 * NLD; ++i) fetch(slot, i);
        next_tile();
    };
    fetch_all(S0{});
    fetch_all(S1{});
    if constexpr (NR == 4) fetch_all(S2{});
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NR - 2) * PER_TILE) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    first(S0{}, s_cur, nothing);
    if constexpr (!RD) {
        load_lq(S0{});
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
            exp_hi(s_cur, v, pw);
            term_lo(v, pl);
        }
        mask(pw, pl);
        post(S0{});
    }
    // one iteration, for the tile in ring slot `buf`; more: another tile follows
    auto step = [&](auto buf, auto more_c) {
        constexpr bool more = decltype(more_c)::value;
        using B1 = std::integral_constant<int, (buf.value + 1) % NR>;
        using BF = std::integral_constant<int, (buf.value + NR - 1) % NR>;
        // tile it + 1 is in LDS (with four slots tile it + 2 may still be on its way: no fence, it would wait for that too), P(it)
        // has been posted; every wavefront has left tile it - 1, whose slot is filled next
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NR - 3) * PER_TILE) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // an instruction of the fetch behind every group of the first products: together they would hold the wavefront up for
        // some 40 ns each
        auto dma = [&](int g) {
#pragma unroll
            for (int u = 0; u < 4 * NLD / NF; ++u) fetch(BF{}, g * (4 * NLD / NF) + u);
        };
        if constexpr (RD) {
            float di[16], p[16];
#pragma unroll
            for (int g = 0; g < 4; ++g) *(float4*)&p[4 * g] = sP[NR == 4 ? buf.value & 1 : buf.value][kb][g][lane];
#pragma unroll
            for (int g = 0; g < 4; ++g) *(float4*)&di[4 * g] = *(const float4*)&td(buf)[8 * g + 4 * h];
            auto ds_hi = [&](int v) {
                x0 = p[v] * (s_cur[v] - di[v]), x1 = p[v + 1] * (s_cur[v + 1] - di[v + 1]);
                term_hi(v, pw);
            };
            if constexpr (more) {
                first(B1{}, s_nxt, [&](int g, int u) {
                    if (u == 0) dma(g);
#pragma unroll
                    for (int i = 0; i < PF; ++i) {
                        const int v = 2 * (PF * g + i);
                        if (u == 1) ds_hi(v), (PF > 1 ? term_lo(v, pl) : void());
                        if (u == 2 && PF == 1) term_lo(v, pl);
                    }
                });
            } else {
#pragma unroll
                for (int v = 0; v < 16; v += 2) ds_hi(v), term_lo(v, pl);
            }
            second(buf, pw, pl, nothing);
            s_cur = s_nxt;
            if constexpr (more) next_tile();
        } else {
            if constexpr (more) {
                load_lq(B1{});
                first(B1{}, s_nxt, [&](int g, int u) { if (u == 0) dma(g); });
                second(buf, pw, pl, [&](int g, int u) {
#pragma unroll
                    for (int i = 0; i < PS; ++i) {
                        const int v = 2 * (PS * g + i);
                        if (u == 1) exp_hi(s_nxt, v, pw_n), (PS > 1 ? term_lo(v, pl_n) : void());
                        if (u == 2 && PS == 1) term_lo(v, pl_n);
                    }
                });
                mask(pw_n, pl_n);
                post(B1{});
                next_tile();
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int w = 0; w < 4; ++w) pw[j][w] = pw_n[j][w], pl[j][w] = pl_n[j][w];
            } else {
                second(buf, pw, pl, nothing);
            }
        }
    };
    const std::true_type more{};
    const std::false_type last{};
    int left = n_it - 1;   // iterations before the last one
    if constexpr (NR == 4) {
        for (; left >= 4; left -= 4) step(S0{}, more), step(S1{}, more), step(S2{}, more), step(S3{}, more);
        if (left == 3) step(S0{}, more), step(S1{}, more), step(S2{}, more), step(S3{}, last);
    } else {
        for (; left >= 3; left -= 3) step(S0{}, more), step(S1{}, more), step(S2{}, more);
    }
    if (left == 0) step(S0{}, last);
    else if (left == 1) step(S0{}, more), step(S1{}, last);
    else if (left == 2) step(S0{}, more), step(S1{}, more), step(S2{}, last);
    dma_wait_all();        // the fetches past the last tile write LDS: they land before the workgroup gives it back
    };
    if (role_d) run(std::true_type{});
    else run(std::false_type{});
    if (a.part_heads) {
        float4* img = (float4*)a.parts + ((((int64_t)part * n_blocks + bid) * 2 + kb) * 2 + (role_d ? 1 : 0)) * (DB * 4 * 64) + lane;
#pragma unroll
        for (int i = 0; i < DB * 4; ++i)
            img[64 * i] = float4{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
        return;
    }
    if (ki < a.N) {
        const float f = role_d ? a.scale : 1.f;
        void* po = role_d ? a.dk : a.dv;
        const int64_t row = role_d ? (int64_t)b * a.s_dk[0] + (int64_t)kvh * a.s_dk[1] + (int64_t)ki * a.s_dk[2]
                                   : (int64_t)b * a.s_dv[0] + (int64_t)kvh * a.s_dv[1] + (int64_t)ki * a.s_dv[2];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int vq = 0; vq < 4; ++vq) store4<true>(po, row + 32 * db + 8 * vq + 4 * h, f, acc[db], 4 * vq);
    }
#endif
}

// ---- dQ of the split-operand path ----
// Operands are two bf16 terms each (planes written by bwd_split_kernel), every product is hi hi + hi lo + lo hi, and dS is split the same way after
// the fp32 algebra.  A wavefront owns 32 query rows (Q and dO, hi and lo, in registers); R row groups times G key groups as in bwd_dq_bf16.
// One wavefront per SIMD at head_dim 128, so the stream is laid out by hand: an iteration is groups of six MFMAs (192 cycles), first the
// first products of the key group's next tile (S and dP in turn), then the second products of this tile (two 32-column blocks of dQ in turn).  Behind
// each MFMA stand a few of the other instructions: the LDS operands of the group two ahead, dS of this tile under the first products of the
// next, the fetch.  K is needed for an iteration longer than V (rows for S, columns for dQ): a tile's K and V lie in rings of their own, LEAD + 1 and
// LEAD slots.  One instance of the iteration: the ring slots are scalars that are added to the operands' addresses.
// As an instance of a compiler-scheduled kernel with two slots -> this: 4 x 16 heads, D 128, N 2552 546 -> 449 us (1.07 PFLOP/s of executed products);
// 32 / 8 heads, 2048 181 -> 147; 16 / 4, 1357 93 -> 68, with two key groups 46; D 64, 2 x 12 heads, 5300 380 -> 337.  Operands requested across the
// iterations' border and scores of two tiles in registers of their own measured the same: the matrix pipe is busy 0.8 of the time as it is.
template <int D, int R, int G>
__device__ __forceinline__ void bwd_dq_split(const BwdArgs& a, int bid) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins
    static_assert(R * G == 4);
    constexpr int KS = D / 16, DB = D / 32, ROWS = 32 * R;
    constexpr int NF = KS, NS = DB, NG = NF + NS;          // groups of six MFMAs: first products, second products
    constexpr int LEAD = G == 1 ? 3 : 2;                   // iterations from a tile's request to its second products
    constexpr int NK = LEAD + 1, NV = LEAD;
    constexpr int TILEB = kBT * D * 2, PAIRB = 2 * TILEB;  // bytes of a tile; of its hi and lo terms
    constexpr int GROUPB = (NK + NV) * PAIRB;
    static_assert(G * GROUPB <= kSplitLds<D>);
    lds_char_t* const ring = lds_start();
    const int n_qtiles = (a.N + ROWS - 1) / ROWS;
    const int qt = n_qtiles - 1 - bid / (a.B * a.Hq);
    const int bh = xcd_grouped_head(bid % (a.B * a.Hq), a.B * a.Hkv, a.n_rep);
    const int b = bh / a.Hq, hq = bh % a.Hq, kvh = hq / a.n_rep;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = wave % R, group = wave / R;
    const int ql = lane & 31, h = lane >> 5;
    const int q0 = qt * ROWS + row * 32;
    const int qi = q0 + ql;
    const int qrow = min(qi, a.N - 1);

    const int wg_qmax = min(qt * ROWS + ROWS - 1, a.N - 1);
    const int kv_end_wg = a.causal ? wg_qmax + 1 : a.N;
    const int n_it = (kv_end_wg + kBT * G - 1) / (kBT * G);   // stages of G key tiles
    // of which this wavefront's key group has work for its rows
    const int kv_end_wave = q0 < a.N ? (a.causal ? min(q0 + 32, a.N) : a.N) : 0;
    const int n_w = max(((kv_end_wave + kBT - 1) / kBT - group + G - 1) / G, 0);

    // The tile being fetched, as running scalars: its first K row (V and the lo planes lie at fixed distances), the bytes from there to the end of the
    // head, its ring slots.  Past the last tile nothing is in range.
    TileDma<D, R> dma;
    dma.init(D, a.N, row, lane);
    constexpr int NLD = TileDma<D, R>::NLD, NFETCH = 4 * NLD, STEPB = G * kBT * D * 2;
    const int64_t head = ((int64_t)b * a.s_k[0] + (int64_t)kvh * a.s_k[1]) * 2, lo_b = a.lo_kv * 2;
    const char* pk = (const char*)a.k + head + group * kBT * D * 2;
    const int64_t v_b = (const char*)a.v - (const char*)a.k;
    int in_range = (a.N - group * kBT) * D * 2, fk = 0, fv = 0;
    lds_char_t* const mine = ring + group * GROUPB;
    auto fetch = [&](int i) {   // K hi, V hi, K lo, V lo, NLD instructions each
        const bool is_v = i / NLD % 2, lo = i / NLD >= 2;
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(pk + (is_v ? v_b : 0) + (lo ? lo_b : 0)), 0, max(in_range, 0), 0x00020000);
        lds_char_t* dst = mine + (is_v ? NK * PAIRB + fv * PAIRB : fk * PAIRB) + (lo ? TILEB : 0) + (row + R * (i % NLD)) * 1024;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 16, dma.voff[i % NLD], 0, 0, 0);
    };
    auto next_tile = [&]() {
        pk += STEPB;
        in_range -= in_range > 0 ? STEPB : 0;
        fk = fk + 1 == NK ? 0 : fk + 1;
        fv = fv + 1 == NV ? 0 : fv + 1;
    };
    for (int t = 0; t < LEAD; ++t) {
#pragma unroll
        for (int i = 0; i < NFETCH; ++i) fetch(i);
        next_tile();
    }

    const uint16_t* Qp = (const uint16_t*)a.q + (int64_t)b * a.s_q[0] + (int64_t)hq * a.s_q[1] + (int64_t)qrow * a.s_q[2];
    const uint16_t* Op = (const uint16_t*)a.dout + (int64_t)b * a.s_do[0] + (int64_t)hq * a.s_do[1] + (int64_t)qrow * a.s_do[2];
    bf16x8_t qh[KS], qlo[KS], doh[KS], dol[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        qh[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Qp + 16 * ks + 8 * h));
        doh[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Op + 16 * ks + 8 * h));
        qlo[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Qp + a.lo_q + 16 * ks + 8 * h));
        dol[ks] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(Op + a.lo_q + 16 * ks + 8 * h));
    }
    const float di_q = a.delta[((int64_t)b * a.Hq + hq) * a.N + qrow];
    const float lse_q = a.lse2[((int64_t)b * a.Hq + hq) * a.N + qrow];
    const float scale_log2 = a.scale * kLog2e;
    const int lim = a.causal ? min(qi, a.N - 1) : a.N - 1;   // the last key this lane's query sees

    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;

    // operand addresses within a tile (see load_row, load_transposed)
    const uint32_t lds0 = (uint32_t)(uintptr_t)mine;
    uint32_t a_row[NF], a_lo[DB], a_hi[DB];
#pragma unroll
    for (int ks = 0; ks < NF; ++ks) a_row[ks] = lds0 + (uint32_t)tile_off<D>(lane & 31, 2 * ks + h);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        const int r = 4 * h + ((lane & 15) >> 2), chunk = 4 * db + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), o8 = (lane & 1) * 8;
        a_lo[db] = lds0 + (uint32_t)(tile_off<D>(r, chunk) + o8);
        a_hi[db] = lds0 + (uint32_t)(tile_off<D>(r + 8, chunk) + o8);
    }

    f32x16_t s_cur, dp_cur, s_nxt, dp_nxt;
    uint32_t pw[2][4], pl[2][4];   // dS of this tile, hi and lo terms
    float e0 = 0.f, e1 = 0.f;
    uint32_t xw = 0;
    // dS of a pair of positions in five pieces
    auto ds_piece = [&](int v, int piece) {
        if (piece == 0) e0 = __builtin_amdgcn_exp2f(fmaf(s_cur[v], scale_log2, -lse_q));
        else if (piece == 1) e1 = __builtin_amdgcn_exp2f(fmaf(s_cur[v + 1], scale_log2, -lse_q));
        else if (piece == 2) e0 *= dp_cur[v] - di_q, e1 *= dp_cur[v + 1] - di_q;
        else if (piece == 3) pw[v >> 3][(v & 7) >> 1] = xw = cvt_pk_bf16(e0, e1);
        else pl[v >> 3][(v & 7) >> 1] = cvt_pk_bf16(e0 - __uint_as_float(xw << 16), e1 - __uint_as_float(xw & 0xffff0000u));
    };
    // dS of masked positions is 0, whatever came of their scores: done on the finished words, in the tiles that the diagonal or the end crosses
    auto mask = [&](int k0) {
        if ((a.causal && k0 + kBT - 1 > q0) || k0 + kBT > a.N) {   // same for the wavefront
            const int n = lim - (k0 + 4 * h) + 1;
            const uint32_t seen = n >= 32 ? ~0u : n <= 0 ? 0u : (1u << n) - 1u;
#pragma unroll
            for (int v = 0; v < 16; v += 2) {
                const uint32_t pair = (bit_mask(seen, 8 * (v >> 2) + (v & 3)) & 0x0000ffffu) | (bit_mask(seen, 8 * (v >> 2) + (v & 3) + 1) & 0xffff0000u);
                pw[v >> 3][(v & 7) >> 1] &= pair;
                pl[v >> 3][(v & 7) >> 1] &= pair;
            }
        }
    };
    // The groups FROM .. TO - 1 of an iteration: first products of the tile in the slots at kn, vn (bytes from the ring's start) into s, dp; second
    // products of the tile whose K is at kc.  work(group, u) is what is placed behind MFMA u of a group; between() stands before the second products.
    auto groups = [&](auto from, auto to, uint32_t kn, uint32_t vn, uint32_t kc, f32x16_t& s, f32x16_t& dp, auto&& work, auto&& between) {
        constexpr int FROM = decltype(from)::value, TO = decltype(to)::value;
        u32x4_t kh[NF], kl[NF], vh[NF], vl[NF];
        uint2 th[NS][2][2], tl[NS][2][2];   // [group][column block of the two][rows + 0, + 8]
        // the reads of group x in four pieces
        auto request = [&](auto xc, auto piece) {
            constexpr int x = decltype(xc)::value, p = decltype(piece)::value;
            if constexpr (x < NF && x < TO) {
                if constexpr (p == 0) kh[x] = ds_b128<0>(a_row[x] + kn);
                else if constexpr (p == 1) vh[x] = ds_b128<0>(a_row[x] + vn);
                else if constexpr (p == 2) kl[x] = ds_b128<TILEB>(a_row[x] + kn);
                else vl[x] = ds_b128<TILEB>(a_row[x] + vn);
            } else if constexpr (x < TO) {
                constexpr int g = x - NF, j = g / (DB / 2), c = p & 1, db = 2 * (g % (DB / 2)) + c, o = j * 16 * 2 * D + (p >= 2 ? TILEB : 0);
                auto& t = p >= 2 ? tl[g][c] : th[g][c];
                t[0] = ds_tr16<o>(a_lo[db] + kc);
                t[1] = ds_tr16<o>(a_hi[db] + kc);
            }
        };
        using P0 = std::integral_constant<int, 0>;
        using P1 = std::integral_constant<int, 1>;
        using P2 = std::integral_constant<int, 2>;
        using P3 = std::integral_constant<int, 3>;
        for_each<2>([&](auto i) {
            using X = std::integral_constant<int, FROM + i.value>;
            request(X{}, P0{}), request(X{}, P1{}), request(X{}, P2{}), request(X{}, P3{});
        });
        for_each<TO - FROM>([&](auto ic) {
            constexpr int x = FROM + ic.value;
            using AHEAD = std::integral_constant<int, x + 2>;
            constexpr int behind = x + 1 >= TO ? 0 : x + 1 < NF ? 4 : 8;   // reads of the next group
            if constexpr (x == NF) between();
            __builtin_amdgcn_sched_barrier(0);
            auto mf = [&](f32x16_t& c, u32x4_t op, bf16x8_t y, bool zero) {
                const f32x16_t z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, op), y, zero ? z : c, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            if constexpr (x < NF) {
                asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(kh[x]), "+v"(vh[x]), "+v"(kl[x]), "+v"(vl[x]) : "n"(behind));
                mf(s, kh[x], qh[x], x == 0);
                request(AHEAD{}, P0{}), work(x, 0), __builtin_amdgcn_sched_barrier(0);
                mf(dp, vh[x], doh[x], x == 0);
                request(AHEAD{}, P1{}), work(x, 1), __builtin_amdgcn_sched_barrier(0);
                mf(s, kh[x], qlo[x], false);
                request(AHEAD{}, P2{}), work(x, 2), __builtin_amdgcn_sched_barrier(0);
                mf(dp, vh[x], dol[x], false);
                request(AHEAD{}, P3{}), work(x, 3), __builtin_amdgcn_sched_barrier(0);
                mf(s, kl[x], qh[x], false);
                work(x, 4), __builtin_amdgcn_sched_barrier(0);
                mf(dp, vl[x], doh[x], false);
                work(x, 5);
            } else {
                constexpr int g = x - NF, j = g / (DB / 2), db = 2 * (g % (DB / 2));
                asm volatile("s_waitcnt lgkmcnt(%8)" : "+v"(th[g][0][0]), "+v"(th[g][0][1]), "+v"(th[g][1][0]), "+v"(th[g][1][1]), "+v"(tl[g][0][0]), "+v"(tl[g][0][1]),
                             "+v"(tl[g][1][0]), "+v"(tl[g][1][1]) : "n"(behind));
                const bf16x8_t ph = __builtin_bit_cast(bf16x8_t, u32x4_t{pw[j][0], pw[j][1], pw[j][2], pw[j][3]});
                const bf16x8_t plo = __builtin_bit_cast(bf16x8_t, u32x4_t{pl[j][0], pl[j][1], pl[j][2], pl[j][3]});
                auto cat = [](const uint2 (&t)[2]) { return u32x4_t{t[0].x, t[0].y, t[1].x, t[1].y}; };
                mf(acc[db], cat(th[g][0]), ph, false);
                request(AHEAD{}, P0{}), work(x, 0), __builtin_amdgcn_sched_barrier(0);
                mf(acc[db + 1], cat(th[g][1]), ph, false);
                request(AHEAD{}, P1{}), work(x, 1), __builtin_amdgcn_sched_barrier(0);
                mf(acc[db], cat(th[g][0]), plo, false);
                request(AHEAD{}, P2{}), work(x, 2), __builtin_amdgcn_sched_barrier(0);
                mf(acc[db + 1], cat(th[g][1]), plo, false);
                request(AHEAD{}, P3{}), work(x, 3), __builtin_amdgcn_sched_barrier(0);
                mf(acc[db], cat(tl[g][0]), ph, false);
                work(x, 4), __builtin_amdgcn_sched_barrier(0);
                mf(acc[db + 1], cat(tl[g][1]), ph, false);
                work(x, 5);
            }
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    using G0 = std::integral_constant<int, 0>;
    using GF = std::integral_constant<int, NF>;
    using GA = std::integral_constant<int, NG>;
    auto nothing = [](int, int) {};
    auto none = []() {};
    uint32_t kc = 0, kn = PAIRB, vn = NK * PAIRB + PAIRB;   // slots of this tile's K, of the next tile's K and V
    // tile it + 1 is in LDS (younger requests may be on their way: no fence, it would wait for them too); every wavefront has left K of tile it - 1 and
    // V of tile it, whose slots are filled next
    auto arrive = [&]() {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((LEAD - 2) * NFETCH) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto advance = [&]() {
        next_tile();
        kc = kn;
        kn = kn + PAIRB == NK * PAIRB ? 0 : kn + PAIRB;
        vn = vn + PAIRB == (NK + NV) * PAIRB ? NK * PAIRB : vn + PAIRB;
    };
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((LEAD - 1) * NFETCH) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int it = 0;
    if (n_w > 0) {
        groups(G0{}, GF{}, 0, NK * PAIRB, 0, s_cur, dp_cur, nothing, none);
        int k0 = group * kBT;
        for (; it < n_w - 1; ++it, k0 += G * kBT) {
            arrive();
            groups(G0{}, GA{}, kn, vn, kc, s_nxt, dp_nxt, [&](int x, int u) {
                if (x < NF) {
                    if (u < NFETCH / NF) fetch(x * (NFETCH / NF) + u);
                    if (D == 128) {
                        if (u >= 1) ds_piece(2 * x, u - 1);
                    } else {   // two pairs under a group
                        const int v = 4 * x + 2 * (u / 3);
                        if (u % 3 == 0) ds_piece(v, 0), ds_piece(v, 1);
                        else if (u % 3 == 1) ds_piece(v, 2), ds_piece(v, 3);
                        else ds_piece(v, 4);
                    }
                }
            }, [&]() { mask(k0); });
            s_cur = s_nxt, dp_cur = dp_nxt;
            advance();
        }
        arrive();
#pragma unroll
        for (int i = 0; i < NFETCH; ++i) fetch(i);
#pragma unroll
        for (int v = 0; v < 16; v += 2)
#pragma unroll
            for (int i = 0; i < 5; ++i) ds_piece(v, i);
        groups(GF{}, GA{}, kn, vn, kc, s_nxt, dp_nxt, nothing, [&]() { mask(k0); });
        advance();
        ++it;
    }
    for (; it < n_it; ++it) {   // the other wavefronts' tiles
        arrive();
#pragma unroll
        for (int i = 0; i < NFETCH; ++i) fetch(i);
        next_tile();
    }
    dma_wait_all();        // the fetches past the last tile write LDS: they land before the workgroup gives it back
    const int64_t out_row = (int64_t)b * a.s_dq[0] + (int64_t)hq * a.s_dq[1] + (int64_t)qi * a.s_dq[2];
    if constexpr (G == 1) {
        if (qi < a.N)
#pragma unroll
            for (int i = 0; i < 4 * DB; ++i) store4<true>(a.dq, out_row + 8 * i + 4 * h, a.scale, acc[i >> 2], 4 * (i & 3));
    } else {   // the key groups' sums meet in the ring; each wavefront adds and stores a G-th of its rows' columns
        __syncthreads();
        constexpr int NQ = 4 * DB, MINE = NQ / G;
        auto image = [&](int w) { return (lds_f32x4_t*)ring + w * (NQ * 64) + lane; };
#pragma unroll
        for (int i = 0; i < NQ; ++i) image(wave)[64 * i] = f32x4_t{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
        __syncthreads();
        if (qi < a.N)
#pragma unroll
            for (int i = 0; i < MINE; ++i) {
                f32x4_t sum = image(row)[64 * (MINE * group + i)];
#pragma unroll
                for (int g = 1; g < G; ++g) sum += image(row + g * R)[64 * (MINE * group + i)];
                store_quad<true>(a.dq, out_row + 8 * (MINE * group + i) + 4 * h, a.scale, sum);
            }
    }
#endif
}

// Both passes in one launch: they share nothing but their inputs, and either by itself ends in a tail of few workgroups or never fills the chip.  The
// first n_dkdv workgroups are the dK / dV pass's, whose chains are longer (all query heads of a kv head), the dQ pass's fill what these leave.
// Forward and backward of fp32 tensors, two launches -> one, us: 12 heads, D 64, 74 tokens 24.3 -> 18.7; 32, D 128, 265 60.9 -> 48.2; 32 / 8, D 128, 714
// 142 -> 120, 3 x 731, not causal 518 -> 402; 8 / 2, D 64, 4297, not causal 648 -> 545; 16, D 128, 3251, not causal 1163 -> 1046; 50 drawn shapes 1.12 (1.00 to 1.32).
template <int D, int R, int G>
__global__ void __launch_bounds__(256, D == 64 ? 2 : 1) bwd_split_pass_kernel(BwdArgs a, int n_dkdv) {
    __shared__ __attribute__((aligned(256))) char rest[kSplitLds<D> - kDkdvSplitLds<D>];
    asm volatile("" ::"v"(lds_byte_addr(rest)));   // part of the workgroup's LDS, whatever the dQ pass's shape needs of it
    if ((int)blockIdx.x < n_dkdv) bwd_dkdv_split<D>(a, (int)blockIdx.x);
    else bwd_dq_split<D, R, G>(a, (int)blockIdx.x - n_dkdv);
}

// dK, dV from the parts of the dK / dV pass: the register images of a key half's gradient, added in the order of the parts
// (bitwise reproducible), scaled and stored.  One wavefront per (key block, half, gradient, quad of columns), eight parts' loads in flight: bound by the
// latency of the parts' first touch, which wants many short wavefronts.  Forward and backward, us, with four quads each, four parts in flight and divisions ->
// now: fp32, D 128, 16/4 heads, 236 tokens 41.7 -> 39.4; 5 x 16/4, 286 75.4 -> 73.8; D 64, 32/8, 66 21.4 -> 20.9; bf16, D 64, 2 x 8/2, 240 19.7 -> 18.7;
// D 128, 3 x 64/8, 223, not causal 53.3 -> 51.5; 32/8, 2048 193.0 -> 191.3.
template <int D, bool F32>
__global__ void __launch_bounds__(256) bwd_dkdv_reduce_kernel(BwdArgs a, BwdDivisors dv) {
    constexpr int NQ = D / 8, WGS = NQ / 4;   // quads; workgroups per (key block, half, gradient)
    const int n_blocks = (a.N + kBK - 1) / kBK * a.B * a.Hkv;
    const uint32_t item = blockIdx.x / WGS, bid = item >> 2;
    const int kb = (item >> 1) & 1, grad = item & 1;   // grad 0: dV, 1: dK
    const uint32_t ut = dv.by_bkv.div(bid), bh = dv.by_bkv.mod(bid, ut), b = dv.by_hkv.div(bh), kvh = dv.by_hkv.mod(bh, b);
    const int kt = (int)ut, lane = threadIdx.x & 63, quad = blockIdx.x % WGS * 4 + (threadIdx.x >> 6);
    const int qt_begin = a.causal ? (kt * kBK) / kBT : 0;
    const int n_qt = (a.N + kBT - 1) / kBT - qt_begin;
    const int ranges = min(a.part_ranges, (n_qt + a.part_tiles - 1) / a.part_tiles);   // of them exist for this key block
    const int n_parts = a.n_parts / a.part_ranges * ranges;
    const int ki = kt * kBK + kb * 32 + (lane & 31), h = lane >> 5;
    const int64_t step = (int64_t)n_blocks * 4 * (NQ * 64), skip = (a.part_ranges - ranges) * step;
    const f32x4_t* img = (const f32x4_t*)a.parts + (((int64_t)bid * 2 + kb) * 2 + grad) * (NQ * 64) + quad * 64 + lane;
    int left = ranges;   // of the heads' group that img is in
    auto next = [&]() {
        const f32x4_t x = *img;
        img += step;
        if (--left == 0) left = ranges, img += skip;
        return x;
    };
    f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
    int p = 0;
    for (; p + 8 <= n_parts; p += 8) {
        f32x4_t x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = next();
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += x[u];
    }
    for (; p + 2 <= n_parts; p += 2) {
        const f32x4_t x0 = next(), x1 = next();
        sum += x0;
        sum += x1;
    }
    if (p < n_parts) sum += next();
    if (ki >= a.N) return;
    void* po = grad ? a.dk : a.dv;
    const int64_t row = grad ? (int64_t)b * a.s_dk[0] + (int64_t)kvh * a.s_dk[1] + (int64_t)ki * a.s_dk[2]
                             : (int64_t)b * a.s_dv[0] + (int64_t)kvh * a.s_dv[1] + (int64_t)ki * a.s_dv[2];
    store_quad<F32>(po, row + 8 * quad + 4 * h, grad ? a.scale : 1.f, sum);
}

// ---- dQ from the dS tiles the dK / dV pass left behind (bf16) ----
// A wavefront owns 32 query rows and walks the key tiles.  Its own dS tile (2 KB, consecutive key tiles consecutive in
// the workspace) comes straight into registers, several tiles ahead; the workgroup's shared K tile comes through a
// ring of four LDS slots.  The tile is the register image of the wavefront that wrote it (a lane = a key), and this
// product contracts over keys, so it passes through a 2 KB patch of LDS of the wavefront's own: written as it came,
// read back with the transposing read (a lane = a query).  Then dQ^T[d][q] += K^T . dS^T, A = the K tile read
// column-wise.  One product instead of the three of bwd_dq_bf16: the pass runs at the rate the tiles stream in.
// Masked positions hold zeros in the tiles, so no mask is applied here.
template <int D>
__global__ void __launch_bounds__(256, 2) bwd_dq_stream_kernel(BwdArgs a) {
    constexpr int DB = D / 32;
    constexpr int PER_STAGE = TileDma<D>::NLD + 2;   // memory instructions a wavefront issues per ring stage
    __shared__ __attribute__((aligned(1024))) uint16_t sK0[kBT * D], sK1[kBT * D], sK2[kBT * D], sK3[kBT * D];
    __shared__ __attribute__((aligned(1024))) char sT[4][2048];   // per wavefront
    auto tk = [&](auto s) -> uint16_t* { if constexpr (s.value == 0) return sK0; else if constexpr (s.value == 1) return sK1; else if constexpr (s.value == 2) return sK2; else return sK3; };
    const int n_qtiles = (a.N + kBQ - 1) / kBQ;
    const int bid = blockIdx.x;
    const int qt = n_qtiles - 1 - bid / (a.B * a.Hq);
    const int bh = xcd_grouped_head(bid % (a.B * a.Hq), a.B * a.Hkv, a.n_rep);
    const int b = bh / a.Hq, hq = bh % a.Hq, kvh = hq / a.n_rep;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ql = lane & 31, h = lane >> 5;
    const int q0 = qt * kBQ + wave * 32;
    const int qi = q0 + ql;

    const int wg_qmax = min(qt * kBQ + kBQ - 1, a.N - 1);
    const int n_tiles = ((a.causal ? wg_qmax + 1 : a.N) + kBT - 1) / kBT;          // key tiles the workgroup walks
    const int nt_w = q0 < a.N ? ((a.causal ? min(q0 + 31, a.N - 1) + 1 : a.N) + kBT - 1) / kBT : 0;   // of which this wavefront uses

    const uint16_t* Kp = (const uint16_t*)a.k + (int64_t)b * a.s_k[0] + (int64_t)kvh * a.s_k[1];
    const u32x4_t* Sp = (const u32x4_t*)((const char*)a.ds_tiles + ((((int64_t)b * a.Hq + hq) * a.n_qt32 + min(q0 >> 5, a.n_qt32 - 1)) * a.n_kt32) * 2048) + lane;
    TileDma<D> dk_;
    dk_.init(a.s_k[2], a.N, wave, lane);
    constexpr int NI = 8, AHEAD = 6;   // dS tiles: register ring, and how many tiles ahead they are requested
    u32x4_t img[NI][2];
    // Every step issues the same number of loads, so that the wait counts below hold: past the end the tile index is
    // clamped (the tile is fetched again and not used).
    auto load_k = [&](int t, auto slot) {
        const int kt = min(t, n_tiles - 1);
        dk_.load(tk(slot), Kp + (int64_t)kt * kBT * a.s_k[2], a.N - kt * kBT, a.s_k[2], wave);
    };
    auto load_s = [&](int t, auto islot) {
        const u32x4_t* tile = Sp + (int64_t)min(t, max(nt_w - 1, 0)) * 128;
        img[islot.value][0] = __builtin_nontemporal_load(tile);
        img[islot.value][1] = __builtin_nontemporal_load(tile + 64);
    };
    f32x16_t acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
    // The patch holds the image as [j][position of the writing lane][4 words], the lane (key kl, half hh) at position
    // 2 kl + hh, rotated by 128 bytes for j = 1: the 16 lanes of a transposing read then fetch 4 keys x 32 bytes =
    // 128 consecutive bytes, and the four such groups of an instruction fall in different banks.
    char* patch = sT[wave];
    const int wr_off = (2 * ql + h) * 16;
    const int i16 = lane & 15, g4 = (lane >> 4) & 1;
    // k-step j', keys 16 j' + 4 h + (i16 >> 2) (+ 8), queries 16 g4 + 4 (i16 & 3) .. + 3: words 2c, 2c + 1 of the lane
    // (key, hh) with hh = i16 & 1, c = (i16 >> 1) & 1, in half j = g4 of the image
    const int rd_off = 32 * (4 * h + (i16 >> 2)) + 16 * (i16 & 1) + 8 * ((i16 >> 1) & 1);
    auto step = [&](int t, auto idx) {
        using KS = std::integral_constant<int, idx.value % 4>;
        using KL = std::integral_constant<int, (idx.value + 3) % 4>;
        using IL = std::integral_constant<int, (idx.value + AHEAD) % NI>;
        // This wavefront's share of K tile t has landed.  Younger in its memory queue, and possibly still in flight: the
        // dS tile requested right behind it and the two steps' requests since.  No fence: it would drain them.
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 + 2 * PER_STAGE) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const u32x4_t i0 = img[idx.value % NI][0], i1 = img[idx.value % NI][1];
        load_k(t + 3, KL{});   // into the slot every wavefront left before this barrier
        load_s(t + AHEAD, IL{});
        if (t >= nt_w) return;
        using slot_t = KS;
        const slot_t slot{};
        const uint16_t* tK = tk(slot);
        *(u32x4_t*)(patch + wr_off) = i0;
        *(u32x4_t*)(patch + 1024 + ((wr_off + 128) & 1023)) = i1;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const char* half = patch + 1024 * g4;
            const uint2 lo = lds_tr16(half + ((rd_off + 512 * j + 128 * g4) & 1023));
            const uint2 hi = lds_tr16(half + ((rd_off + 512 * j + 256 + 128 * g4) & 1023));
            const bf16x8_t dsf = __builtin_bit_cast(bf16x8_t, uint4{lo.x, lo.y, hi.x, hi.y});
#pragma unroll
            for (int db = 0; db < DB; ++db) acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(load_transposed<D>(tK, j, db, lane), dsf, acc[db], 0, 0, 0);
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using I4 = std::integral_constant<int, 4>;
    using I5 = std::integral_constant<int, 5>;
    using I6 = std::integral_constant<int, 6>;
    using I7 = std::integral_constant<int, 7>;
    // the order of the first requests gives every K tile at least as many younger requests as the steady state does
    load_k(0, I0{});
    load_s(0, I0{});
    load_s(1, I1{});
    load_s(2, I2{});
    load_s(3, I3{});
    load_k(1, I1{});
    load_s(4, I4{});
    load_k(2, I2{});
    load_s(5, I5{});
    for (int t = 0; t < n_tiles; t += 8) {
        step(t, I0{});
        if (t + 1 < n_tiles) step(t + 1, I1{});
        if (t + 2 < n_tiles) step(t + 2, I2{});
        if (t + 3 < n_tiles) step(t + 3, I3{});
        if (t + 4 < n_tiles) step(t + 4, I4{});
        if (t + 5 < n_tiles) step(t + 5, I5{});
        if (t + 6 < n_tiles) step(t + 6, I6{});
        if (t + 7 < n_tiles) step(t + 7, I7{});
    }
    dma_wait_all();   // the clamped requests of the last steps write LDS: they land before the workgroup gives it back
    if (qi < a.N) {
        const int64_t row = (int64_t)b * a.s_dq[0] + (int64_t)hq * a.s_dq[1] + (int64_t)qi * a.s_dq[2];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int vq = 0; vq < 4; ++vq) store4<false>(a.dq, row + 32 * db + 8 * vq + 4 * h, a.scale, acc[db], 4 * vq);
    }
}

// Instantiated explicitly: the host pass of this compiler drops the implicit instantiation of the launch stubs.
template __global__ void bwd_dkdv_bf16_kernel<128, true>(BwdArgs, BwdDivisors);
template __global__ void bwd_dkdv_bf16_kernel<64, true>(BwdArgs, BwdDivisors);
template __global__ void bwd_dq_stream_kernel<128>(BwdArgs);
template __global__ void bwd_dq_stream_kernel<64>(BwdArgs);
template __global__ void bwd_rowstats_bf16_kernel<128>(BwdArgs, BwdDivisors);
template __global__ void bwd_rowstats_bf16_kernel<64>(BwdArgs, BwdDivisors);
template __global__ void bwd_pass_kernel<128, 4, 1>(BwdArgs, BwdDivisors, int);
template __global__ void bwd_pass_kernel<128, 2, 2>(BwdArgs, BwdDivisors, int);
template __global__ void bwd_pass_kernel<64, 4, 1>(BwdArgs, BwdDivisors, int);
template __global__ void bwd_pass_kernel<64, 2, 2>(BwdArgs, BwdDivisors, int);
template __global__ void bwd_split_pass_kernel<128, 4, 1>(BwdArgs, int);
template __global__ void bwd_split_pass_kernel<128, 2, 2>(BwdArgs, int);
template __global__ void bwd_split_pass_kernel<64, 4, 1>(BwdArgs, int);
template __global__ void bwd_split_pass_kernel<64, 2, 2>(BwdArgs, int);
template __global__ void bwd_dkdv_reduce_kernel<128, false>(BwdArgs, BwdDivisors);
template __global__ void bwd_dkdv_reduce_kernel<64, false>(BwdArgs, BwdDivisors);
template __global__ void bwd_dkdv_reduce_kernel<128, true>(BwdArgs, BwdDivisors);
template __global__ void bwd_dkdv_reduce_kernel<64, true>(BwdArgs, BwdDivisors);

// ---- pre-pass of the split-operand path: every fp32 operand as two bf16 planes, Di and lse * log2(e) ----
struct SplitArgs {
    const float *q, *dout, *out, *k, *v, *lse;
    int64_t s_q[3], s_do[3], s_o[3], s_k[3], s_v[3], s_l[3];
    uint16_t *qh, *doh, *kh, *vh;          // hi planes, dense [B][H][N][D]; the lo plane follows at lo_q / lo_kv elements
    int64_t lo_q, lo_kv;
    float *delta, *lse2;
    int32_t B, Hq, Hkv, N, D;
    FastDiv by_n, by_hq, by_hkv;
};
// Four neighbouring elements; rows begin at multiples of 8 bytes only, which a 16-byte global load takes.
typedef float f32x4_rows_t __attribute__((ext_vector_type(4), aligned(8)));
__device__ inline void split_quad(f32x4_rows_t x, uint16_t* hi, uint16_t* lo) {
    const uint32_t h0 = cvt_pk_bf16(x[0], x[1]), h1 = cvt_pk_bf16(x[2], x[3]);
    *(uint2*)hi = uint2{h0, h1};
    *(uint2*)lo = uint2{cvt_pk_bf16(x[0] - __uint_as_float(h0 << 16), x[1] - __uint_as_float(h0 & 0xffff0000u)),
                        cvt_pk_bf16(x[2] - __uint_as_float(h1 << 16), x[3] - __uint_as_float(h1 & 0xffff0000u))};
}
// D / 4 lanes per row, 16 bytes of each operand: rows [0, B Hq N) are query rows (Q, dO, and Di = rowsum(dO * O) in fp32,
// src/ops/flash_attention.cpp:416-423), the rest are key rows (K, V).  Bound by the bytes, 12 read and 8 written per element of a query row, 8 and 8 of a key row; with a
// wavefront per row (half of it idle at D 64), 8-byte pieces and 64-bit divisions it was bound by its instructions.  Forward and backward, us, before -> now:
// D 64, 4 x 32/8 heads, 300 tokens 66.7 -> 58.8; 3 x 12, 1034 122.9 -> 112.8; D 128, 2 x 64/8, 396 151.7 -> 146.4; 32/8, 2048 483.0 -> 474.3; 30 21.1 -> 20.5.
template <int D>
__global__ void __launch_bounds__(256) bwd_split_kernel(SplitArgs a) {
    constexpr int LPR = D / 4, RPB = 256 / LPR;
    const uint32_t rows_q = (uint32_t)a.B * a.Hq * a.N, rows_kv = (uint32_t)a.B * a.Hkv * a.N;
    const uint32_t row = blockIdx.x * RPB + threadIdx.x / LPR, d = 4 * (threadIdx.x % LPR);
    if (row < rows_q) {   // (all lanes of a row alike)
        const uint32_t bh = a.by_n.div(row), i = a.by_n.mod(row, bh), b = a.by_hq.div(bh), h = a.by_hq.mod(bh, b);
        const f32x4_rows_t xq = *(const f32x4_rows_t*)(a.q + (int64_t)b * a.s_q[0] + (int64_t)h * a.s_q[1] + (int64_t)i * a.s_q[2] + d);
        const f32x4_rows_t xd = *(const f32x4_rows_t*)(a.dout + (int64_t)b * a.s_do[0] + (int64_t)h * a.s_do[1] + (int64_t)i * a.s_do[2] + d);
        const f32x4_rows_t xo = *(const f32x4_rows_t*)(a.out + (int64_t)b * a.s_o[0] + (int64_t)h * a.s_o[1] + (int64_t)i * a.s_o[2] + d);
        const int64_t at = (int64_t)row * D + d;
        split_quad(xq, a.qh + at, a.qh + a.lo_q + at);
        split_quad(xd, a.doh + at, a.doh + a.lo_q + at);
        float di = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) di += xd[e] * xo[e];
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) di += __shfl_xor(di, o);
        if (d == 0) {
            a.delta[row] = di;
            a.lse2[row] = kLog2e * a.lse[(int64_t)b * a.s_l[0] + (int64_t)h * a.s_l[1] + (int64_t)i * a.s_l[2]];
        }
    } else if (row - rows_q < rows_kv) {
        const uint32_t r = row - rows_q, bh = a.by_n.div(r), i = a.by_n.mod(r, bh), b = a.by_hkv.div(bh), h = a.by_hkv.mod(bh, b);
        const f32x4_rows_t xk = *(const f32x4_rows_t*)(a.k + (int64_t)b * a.s_k[0] + (int64_t)h * a.s_k[1] + (int64_t)i * a.s_k[2] + d);
        const f32x4_rows_t xv = *(const f32x4_rows_t*)(a.v + (int64_t)b * a.s_v[0] + (int64_t)h * a.s_v[1] + (int64_t)i * a.s_v[2] + d);
        const int64_t at = (int64_t)r * D + d;
        split_quad(xk, a.kh + at, a.kh + a.lo_kv + at);
        split_quad(xv, a.vh + at, a.vh + a.lo_kv + at);
    }
}

int check4(const vsp_tensor* t, int64_t B, int64_t H, int64_t N, int64_t D, int dtype) {
    if (!t) return VSP_ERR_NULL;
    if (t->ndim != 4) return VSP_ERR_NDIM;
    if (t->shape[0] != B || t->shape[1] != H || t->shape[2] != N || t->shape[3] != D) return VSP_ERR_SHAPE;
    if (t->dtype != dtype) return VSP_ERR_DTYPE;
    if (t->stride[3] != 1) return VSP_ERR_STRIDE;
    if (B * H * N * D > 0 && !t->data) return VSP_ERR_NULL;
    return VSP_OK;
}

// How the dK / dV pass is cut into parts (heads 0: not at all).  A workgroup per key block (64 keys of a kv head) leaves the
// chip idle on two counts: few key blocks, and, under the causal mask, the first block's chain being twice the average one.
// The steps of a block are cut by query head, then by ranges of query tiles.  Cut that way, the workgroups
// of one (kv head, part) still walk the same Q / dO tiles at the same time, whatever their key block, and find them in their
// XCD's L2 (equal lengths of the (head, tile) sequence do not: 2 x the time at 2048 tokens).
// The number of parts is the one with the least estimate of the launch that holds both passes, in us:
//   the larger of  work = (7/4 of the dK / dV steps, for the dQ pass's three products beside its four, and 3 a part to start) a slot, at tau_work a step
//   and            chain = (the longest part's steps + 3), at tau_chain a step, which is shorter where a lone workgroup on a CU runs faster,
//   and, where there are parts, 4 for the launch that adds them and their traffic at 3 MB / us.
// Fitted to 105 drawn shapes with 1, 2, 3, 4, 6, 8, 12 and 16 parts, forward and backward, us, one part / as chosen / twice as many: bf16, D 128, 32 / 8 heads, 842, not
// causal 103.9 / 84.5 / 87.0; 64 / 8, 4 x 1482 705.7 / 705.7 / 755.6; 16 / 4, 754 72.7 / 40.9 / 40.9; D 64, 8 / 2, 2082 138.5 / 57.3 / -; split, D 128, 32 / 8, 2 x 836,
// not causal 352.4 / 352.4 / 364.5; 64 / 8, 558 223.9 / 127.1 / 136.3; D 64, 8 / 2, 2849 344.2 / 156.6 / 170.3.  On average 1 % from the best of the eight.
// bf16 chains of fewer than 24 steps stay whole (21.0 us for 17.2 at 8 / 2 heads, D 64, 3 x 160): their parts would need more room than kept dS tiles, and a short
// call's bits would depend on which of the two workspaces it was given.
struct PartPlan {
    int heads, tiles, ranges, parts;
};
PartPlan plan_parts(int64_t B, int64_t Hkv, int64_t n_rep, int64_t N, int64_t D, bool causal, bool split) {
    const int64_t blocks = ceil_div(N, kBK) * B * Hkv, n_qt = ceil_div(N, kBT), steps = n_rep * n_qt;
    // workgroups the chip holds; us a step of 32 queries x 64 keys
    const int64_t slots = device_cu_count() * (split ? (D == 64 ? 2 : 1) : D == 64 ? 3 : 2);
    const float tau_work = split ? 1.f : D == 64 ? 0.7f : 0.85f, tau_chain = split ? (D == 64 ? 0.9f : 1.3f) : D == 64 ? 0.63f : 0.65f;
    const float work = 1.75f * (float)blocks * (float)n_rep * (causal ? 0.5f * (float)(n_qt + 2) : (float)n_qt);
    PartPlan best{0, 0, 1, 1};
    if (!split && steps < 24) return best;
    float least = std::max(work / (float)slots * tau_work, (float)(steps + 3) * tau_chain);
    for (const int64_t want : {2, 3, 4, 6, 8, 12, 16, 24, 32}) {
        if (want > steps / 2) break;
        const int64_t heads = std::max<int64_t>(1, n_rep / want), groups = ceil_div(n_rep, heads);
        const int64_t tiles = ceil_div(n_qt, std::max<int64_t>(1, want / groups)), ranges = ceil_div(n_qt, tiles), parts = groups * ranges;
        if (parts <= 1) continue;
        const float us = std::max((work + 3.f * (float)(parts * blocks)) / (float)slots * tau_work, (float)(heads * tiles + 3) * tau_chain) + 4.f +
                         (float)(parts * blocks) * (float)(4 * kBK * D * (int64_t)sizeof(float)) / 3e6f;
        if (us < least) least = us, best = {(int)heads, (int)tiles, (int)ranges, (int)parts};
    }
    return best;
}
size_t parts_bytes(const PartPlan& p, int64_t B, int64_t Hkv, int64_t N, int64_t D) {
    return p.parts > 1 ? (size_t)p.parts * (size_t)(ceil_div(N, kBK) * B * Hkv) * 2 * kBK * (size_t)D * sizeof(float) : 0;
}

// The dQ workgroups of the launch: 128 queries, or 64 with two key groups, which halves the longest chain of key tiles where the workgroups are few and the
// chains long.  128 / 64 queries, forward and backward, us (w: workgroups of 128 queries): D 128, 16 / 4 heads, 754 (w 96) 46.3 / 41.0; 32 / 8, 842, not causal
// (w 224) 96.1 / 93.0; 2 x 507, 32 heads (w 256) 47.1 / 46.1; 16 heads, 2 x 161 (w 96) 27.4 / 29.1; 32 / 8, 2 x 1031 (w 576) 128 / 131; D 64, 8 / 2, 2082 (w 136) 70.8 / 59.4;
// 32 / 8, 3 x 611 (w 480) 59.1 / 56.8; 8 / 2, 2 x 5254 (w 672) 324 / 308; 12 heads, 472 (w 48) 19.3 / 19.5; 32 / 8, 2 x 3706 (w 1856) 554 / 568.
int dq_row_groups(int64_t B, int64_t Hkv, int64_t n_rep, int64_t N, int64_t D) {
    const int64_t cus = device_cu_count(), w = ceil_div(N * n_rep, kBQ) * B * Hkv, tiles = ceil_div(N, kBT);
    return D == 64 ? (tiles >= 20 && 2 * w <= 5 * cus ? 2 : 4) : tiles >= 16 && w <= cus ? 2 : 4;
}

// Query rows of all heads that the bf16 passes number in 32 bits, with a workgroup's rows to spare (2^31 rows of 64 columns are 256 GB a tensor)
constexpr int64_t kMaxRows = INT32_MAX - 127;

BwdDivisors divisors(const BwdArgs& a) {
    const int64_t heads = (int64_t)a.B * a.Hkv;
    return {FastDiv::of(ceil_div(a.N, kBK) * heads), FastDiv::of(heads), FastDiv::of(a.Hkv), FastDiv::of(a.n_rep), FastDiv::of(a.N), FastDiv::of(a.Hq)};
}

// Whether a gradient [B, Hkv, N, D] and an operand [B, heads, N, D], bf16, lie in overlapping memory (the bytes from the first element to the last: more than they are)
bool may_overlap(const BwdArgs& a, int64_t D, const void* grad, const int64_t (&sg)[3], const void* x, const int64_t (&sx)[3], int64_t heads) {
    auto span = [&](const void* p, const int64_t (&s)[3], int64_t h) {
        int64_t lo = 0, hi = D;
        for (const int64_t last : {(int64_t)(a.B - 1) * s[0], (h - 1) * s[1], (int64_t)(a.N - 1) * s[2]}) (last < 0 ? lo : hi) += last;
        return std::pair<intptr_t, intptr_t>{(intptr_t)p + 2 * lo, (intptr_t)p + 2 * hi};
    };
    const auto u = span(grad, sg, a.Hkv), v = span(x, sx, heads);
    return u.first < v.second && v.first < u.second;
}

// Gradients that replace operands in their memory: the dK / dV pass writes a key block's when it has read that block of K and V and every Q and dO of its heads (of
// one key block, Q and dO may be replaced too), the dQ pass reads all of them, so it comes first, in a launch of its own.  (Where there are parts, the launch that adds them is the
// one that writes.)
template <int D>
int launch_bf16_passes(const BwdArgs& a, const BwdDivisors& d, hipStream_t st) {
    auto replaces = [&](const void* grad, const int64_t (&sg)[3]) {
        return may_overlap(a, D, grad, sg, a.k, a.s_k, a.Hkv) || may_overlap(a, D, grad, sg, a.v, a.s_v, a.Hkv) || may_overlap(a, D, grad, sg, a.q, a.s_q, a.Hq) ||
               may_overlap(a, D, grad, sg, a.dout, a.s_do, a.Hq);
    };
    const bool in_place = !a.part_heads && (replaces(a.dk, a.s_dk) || replaces(a.dv, a.s_dv));
    const int64_t rows = (int64_t)a.B * a.Hq * a.N, blocks = ceil_div(a.N, kBK) * a.B * a.Hkv, n_dkdv = blocks * (a.part_heads ? a.n_parts : 1);
    hipLaunchKernelGGL((bwd_rowstats_bf16_kernel<D>), dim3((unsigned)ceil_div(rows, 4 * (512 / D))), dim3(256), 0, st, a, d);
    const int rc = with_row_groups<4, 2>(dq_row_groups(a.B, a.Hkv, a.n_rep, a.N, D), [&](auto r) {
        constexpr int R = decltype(r)::value;
        const int64_t n_dq = ceil_div((int64_t)a.N * a.n_rep, 32 * R) * a.B * a.Hkv;
        if (in_place) hipLaunchKernelGGL((bwd_pass_kernel<D, R, 4 / R>), dim3((unsigned)n_dq), dim3(256), 0, st, a, d, 0);
        hipLaunchKernelGGL((bwd_pass_kernel<D, R, 4 / R>), dim3((unsigned)(n_dkdv + (in_place ? 0 : n_dq))), dim3(256), 0, st, a, d, (int)n_dkdv);
        return VSP_OK;
    });
    if (rc == VSP_OK && a.part_heads) hipLaunchKernelGGL((bwd_dkdv_reduce_kernel<D, false>), dim3((unsigned)(D / 8 * blocks)), dim3(256), 0, st, a, d);
    return rc == VSP_OK ? check_launch() : rc;
}

int launch_backward_bf16(const BwdArgs& a, int64_t D, hipStream_t st) {
    const int64_t rows = (int64_t)a.B * a.Hq * a.N;
    if (rows > kMaxRows) return VSP_ERR_ARG;
    const BwdDivisors d = divisors(a);
    if (!a.ds_tiles) return D == 128 ? launch_bf16_passes<128>(a, d, st) : launch_bf16_passes<64>(a, d, st);
    // one-pass dS: row constants, dK / dV (leaving the dS tiles), dQ from the tiles
    const dim3 gq((unsigned)(ceil_div(a.N, kBQ) * a.B * a.Hq)), gk((unsigned)(ceil_div(a.N, kBK) * a.B * a.Hkv));
    if (D == 128) {
        hipLaunchKernelGGL((bwd_rowstats_bf16_kernel<128>), dim3((unsigned)ceil_div(rows, 16)), dim3(256), 0, st, a, d);
        hipLaunchKernelGGL((bwd_dkdv_bf16_kernel<128, true>), gk, dim3(256), 0, st, a, d);
        hipLaunchKernelGGL((bwd_dq_stream_kernel<128>), gq, dim3(256), 0, st, a);
    } else {
        hipLaunchKernelGGL((bwd_rowstats_bf16_kernel<64>), dim3((unsigned)ceil_div(rows, 32)), dim3(256), 0, st, a, d);
        hipLaunchKernelGGL((bwd_dkdv_bf16_kernel<64, true>), gk, dim3(256), 0, st, a, d);
        hipLaunchKernelGGL((bwd_dq_stream_kernel<64>), gq, dim3(256), 0, st, a);
    }
    return check_launch();
}

int launch_backward_f32(const BwdArgs& a, int64_t D, hipStream_t st) {
    const int64_t rows = (int64_t)a.B * a.Hq * a.N, tiles = ceil_div(a.N, kBQ);
    hipLaunchKernelGGL(bwd_delta_kernel, dim3((unsigned)ceil_div(rows, 4)), dim3(256), 0, st, a, (int)D);
    const int rc = check_launch();
    if (rc != VSP_OK) return rc;
    const dim3 gq((unsigned)(tiles * a.B * a.Hq)), gk((unsigned)(tiles * a.B * a.Hkv));
    if (D > 64) {  // the kernels take any head_dim up to their tile width (a.D_true)
        hipLaunchKernelGGL((bwd_dq_kernel<128>), gq, dim3(256), 0, st, a);
        hipLaunchKernelGGL((bwd_dkdv_kernel<128>), gk, dim3(256), 0, st, a);
    } else if (D > 32) {
        hipLaunchKernelGGL((bwd_dq_kernel<64>), gq, dim3(256), 0, st, a);
        hipLaunchKernelGGL((bwd_dkdv_kernel<64>), gk, dim3(256), 0, st, a);
    } else {
        hipLaunchKernelGGL((bwd_dq_kernel<32>), gq, dim3(256), 0, st, a);
        hipLaunchKernelGGL((bwd_dkdv_kernel<32>), gk, dim3(256), 0, st, a);
    }
    return check_launch();
}

// The split dQ pass: 128 queries per workgroup, or 64 with two key groups, for the reasons at dq_row_groups.  D 128 has one workgroup per CU (112 and
// 160 KB of LDS), so that two rounds of halves are no shorter than one of wholes except where causal chains differ much; D 64 has two.  Whole backward,
// us, 128 / 64 queries (w: workgroups of 128): D 128, 32 heads, 445, not causal (w 128) 68.9 / 61.3; 64 / 8, 490, not causal (w 256) 122 / 126; 16 heads, 1491
// (w 192) 153 / 133; 64 / 8, 2 x 175 (w 256) 55.9 / 61.0; 16 heads, 3 x 1130 (w 432) 237 / 248; D 64, 8 / 2, 1613 (w 104) 91.2 / 73.2; 2 x 1446 (w 192) 109 / 98;
// 12 heads, 2 x 1433 (w 288) 114 / 105; 32 / 8, 5 x 196 (w 320) 56.1 / 58.5; 16 heads, 7 x 482 (w 448) 91 / 95.  32 queries and four key groups, D 64: slower throughout.
// Those are of the dQ pass in a launch of its own; beside the dK / dV pass's workgroups the rule is, over 51 shapes, within 1 % of the better shape of each on average
// (always 128 queries 0.2 % slower, always 64 0.8 %), as plan_parts' is (no parts 6 % slower, half or twice as many within 0.7 %).
int dq_split_row_groups(int64_t B, int64_t Hq, int64_t N, int64_t D, bool causal) {
    const int64_t cus = device_cu_count(), w = ceil_div(N, kBQ) * B * Hq, tiles = ceil_div(N, kBT);
    if (tiles < 3) return 4;
    if (2 * w <= cus) return 2;
    if (D == 64) return tiles >= (causal ? 12 : 24) && 4 * w <= 5 * cus ? 2 : 4;
    return causal && tiles >= 32 && w <= cus ? 2 : 4;
}

template <int D>
int launch_split_passes(const BwdArgs& a, hipStream_t st) {
    const int64_t blocks = ceil_div(a.N, kBK) * a.B * a.Hkv, n_dkdv = blocks * (a.part_heads ? a.n_parts : 1);
    const int rc = with_row_groups<4, 2>(dq_split_row_groups(a.B, a.Hq, a.N, D, a.causal != 0), [&](auto r) {
        constexpr int R = decltype(r)::value;
        const dim3 grid((unsigned)(n_dkdv + ceil_div(a.N, 32 * R) * a.B * a.Hq));
        hipLaunchKernelGGL((bwd_split_pass_kernel<D, R, 4 / R>), grid, dim3(256), 0, st, a, (int)n_dkdv);
        return VSP_OK;
    });
    if (rc == VSP_OK && a.part_heads) hipLaunchKernelGGL((bwd_dkdv_reduce_kernel<D, true>), dim3((unsigned)(D / 8 * blocks)), dim3(256), 0, st, a, divisors(a));
    return rc == VSP_OK ? check_launch() : rc;
}

int launch_backward_split(const SplitArgs& sa, const BwdArgs& a, int64_t D, hipStream_t st) {
    const int64_t rows = (int64_t)a.B * (a.Hq + a.Hkv) * a.N;
    if (D == 128) {
        hipLaunchKernelGGL((bwd_split_kernel<128>), dim3((unsigned)ceil_div(rows, 8)), dim3(256), 0, st, sa);
        return launch_split_passes<128>(a, st);
    } else {
        hipLaunchKernelGGL((bwd_split_kernel<64>), dim3((unsigned)ceil_div(rows, 16)), dim3(256), 0, st, sa);
        return launch_split_passes<64>(a, st);
    }
}

size_t align16(size_t n) { return (n + 15) & ~(size_t)15; }
size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// The dK / dV pass in parts when the workspace has room behind its `base` bytes and the grid calls for it.
void take_parts(BwdArgs& a, int64_t D, bool split, void* workspace, size_t base, size_t workspace_bytes) {
    const PartPlan p = plan_parts(a.B, a.Hkv, a.n_rep, a.N, D, a.causal != 0, split);
    if (p.parts <= 1 || !is_aligned16(workspace) || workspace_bytes < align256(base) + parts_bytes(p, a.B, a.Hkv, a.N, D)) return;
    a.part_heads = p.heads, a.part_tiles = p.tiles, a.part_ranges = p.ranges, a.n_parts = p.parts;
    a.parts = (float*)((char*)workspace + align256(base));
}

}  // namespace
}  // namespace vsp

using namespace vsp;

extern "C" size_t vsp_attn_backward_workspace_bytes(int32_t B, int32_t Hq, int32_t N) {
    if (B <= 0 || Hq <= 0 || N <= 0) return 0;
    return 2 * (size_t)B * (size_t)Hq * (size_t)N * sizeof(float);   // Di and the rescaled log-sum-exp
}

extern "C" size_t vsp_attn_backward_fast_workspace_bytes(int32_t B, int32_t Hq, int32_t N) {
    if (B <= 0 || Hq <= 0 || N <= 0) return 0;
    const size_t base = (vsp_attn_backward_workspace_bytes(B, Hq, N) + 255) & ~(size_t)255;
    const size_t n_qt32 = ((size_t)N + 31) / 32, n_kt32 = 2 * (((size_t)N + 63) / 64);
    return base + (size_t)B * (size_t)Hq * n_qt32 * n_kt32 * 2048;   // one 32 x 32 bf16 dS tile per (query tile, key tile)
}

extern "C" size_t vsp_attn_backward_split_workspace_bytes(int32_t B, int32_t Hq, int32_t Hkv, int32_t N, int32_t D);

extern "C" size_t vsp_attn_backward_parts_workspace_bytes(int32_t B, int32_t Hq, int32_t Hkv, int32_t N, int32_t D, int is_causal, int split) {
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || N <= 0 || (D != 64 && D != 128)) return 0;
    const size_t base = split ? vsp_attn_backward_split_workspace_bytes(B, Hq, Hkv, N, D) : vsp_attn_backward_workspace_bytes(B, Hq, N);
    const PartPlan p = plan_parts(B, Hkv, Hq / Hkv, N, D, is_causal != 0, split != 0);
    return p.parts > 1 ? align256(base) + parts_bytes(p, B, Hkv, N, D) : base;
}

extern "C" int vsp_attn_backward_plan(int32_t B, int32_t Hq, int32_t Hkv, int32_t N, int32_t D, int is_causal, int split, vsp_attn_plan* plan) {
    if (!plan) return VSP_ERR_NULL;
    if (D != 64 && D != 128) return VSP_ERR_UNSUPPORTED;
    if (B <= 0 || Hkv <= 0 || Hq <= 0 || Hq % Hkv != 0 || N <= 0) return VSP_ERR_SHAPE;
    if (N > INT32_MAX / 2 || (!split && (int64_t)B * Hq * N > kMaxRows)) return VSP_ERR_ARG;
    const int r = split ? dq_split_row_groups(B, Hq, N, D, is_causal != 0) : dq_row_groups(B, Hkv, Hq / Hkv, N, D);
    *plan = vsp_attn_plan{r, 4 / r, 0, !split, plan_parts(B, Hkv, Hq / Hkv, N, D, is_causal != 0, split != 0).parts};
    return VSP_OK;
}

// keep_ds: a workspace large enough for the dS tiles selects the path that stores them
static int backward_entry(const vsp_tensor* dout, const vsp_tensor* q, const vsp_tensor* k, const vsp_tensor* v, const vsp_tensor* out,
                          const vsp_tensor* lse, vsp_tensor* dq, vsp_tensor* dk, vsp_tensor* dv, float scale, int is_causal,
                          void* workspace, size_t workspace_bytes, bool keep_ds, void* stream) {
    if (!q || !k || !v) return VSP_ERR_NULL;
    if (q->ndim != 4 || k->ndim != 4 || v->ndim != 4) return VSP_ERR_NDIM;
    const int64_t B = q->shape[0], Hq = q->shape[1], N = q->shape[2], D = q->shape[3];
    const int64_t Hkv = k->shape[1];
    if (Hkv <= 0 ? Hq != 0 : (Hq % Hkv != 0)) return VSP_ERR_SHAPE;
    const int dt = q->dtype;
    if (dt != VSP_F32 && dt != VSP_BF16) return VSP_ERR_UNSUPPORTED;
    int rc;
    if ((rc = check4(q, B, Hq, N, D, dt)) || (rc = check4(dout, B, Hq, N, D, dt)) || (rc = check4(out, B, Hq, N, D, dt)) ||
        (rc = check4(dq, B, Hq, N, D, dt)) || (rc = check4(k, B, Hkv, N, D, dt)) || (rc = check4(v, B, Hkv, N, D, dt)) ||
        (rc = check4(dk, B, Hkv, N, D, dt)) || (rc = check4(dv, B, Hkv, N, D, dt)))
        return rc;
    if (!lse) return VSP_ERR_NULL;
    if (lse->ndim != 3 || lse->shape[0] != B || lse->shape[1] != Hq || lse->shape[2] != N) return VSP_ERR_SHAPE;
    if (lse->dtype != VSP_F32) return VSP_ERR_DTYPE;
    if (B * Hq * N * D == 0) return VSP_OK;
    if (!lse->data) return VSP_ERR_NULL;
    // bf16: head_dim 64 or 128; fp32: any head_dim up to 128, as the reference's backward takes any
    if (dt == VSP_BF16 ? (D != 64 && D != 128) : D > 128) return VSP_ERR_UNSUPPORTED;
    if (!(fabsf(scale) < INFINITY)) return VSP_ERR_ARG;
    if (N > INT32_MAX / 2) return VSP_ERR_ARG;
    if (!workspace || workspace_bytes < vsp_attn_backward_workspace_bytes((int32_t)B, (int32_t)Hq, (int32_t)N)) return VSP_ERR_WORKSPACE;
    if (((uintptr_t)workspace & 3) != 0) return VSP_ERR_ALIGN;
    if (dt == VSP_BF16) {  // 16-byte row segments are moved whole
        for (const vsp_tensor* t : {dout, q, k, v, out, (const vsp_tensor*)dq, (const vsp_tensor*)dk, (const vsp_tensor*)dv}) {
            if (!is_aligned16(t->data)) return VSP_ERR_ALIGN;
            for (int i = 0; i < 3; ++i)
                if ((t->stride[i] * 2) % 16 != 0) return VSP_ERR_ALIGN;
            if (t->stride[2] < D) return VSP_ERR_STRIDE;   // whole rows are fetched under a byte-range check
            if ((uint64_t)N * (uint64_t)t->stride[2] * 2u > 0x7fffffffull) return VSP_ERR_STRIDE;
        }
    }

    BwdArgs a{};
    a.dout = dout->data;
    a.q = q->data;
    a.k = k->data;
    a.v = v->data;
    a.out = out->data;
    a.lse = (const float*)lse->data;
    a.dq = dq->data;
    a.dk = dk->data;
    a.dv = dv->data;
    a.delta = (float*)workspace;
    a.lse2 = a.delta + B * Hq * N;
    for (int i = 0; i < 3; ++i) {
        a.s_do[i] = dout->stride[i];
        a.s_q[i] = q->stride[i];
        a.s_k[i] = k->stride[i];
        a.s_v[i] = v->stride[i];
        a.s_o[i] = out->stride[i];
        a.s_l[i] = lse->stride[i];
        a.s_dq[i] = dq->stride[i];
        a.s_dk[i] = dk->stride[i];
        a.s_dv[i] = dv->stride[i];
    }
    a.B = (int)B;
    a.Hq = (int)Hq;
    a.Hkv = (int)Hkv;
    a.n_rep = (int)(Hq / Hkv);
    a.N = (int)N;
    a.causal = is_causal ? 1 : 0;
    a.scale = scale;
    a.D_true = (int)D;
    // bf16 with the larger workspace: dS is computed once (see include/vsp_attn.h)
    if (dt == VSP_BF16 && keep_ds && workspace_bytes >= vsp_attn_backward_fast_workspace_bytes((int32_t)B, (int32_t)Hq, (int32_t)N) && is_aligned16(workspace)) {
        a.ds_tiles = (uint16_t*)((char*)workspace + ((vsp_attn_backward_workspace_bytes((int32_t)B, (int32_t)Hq, (int32_t)N) + 255) & ~(size_t)255));
        a.n_qt32 = (int)ceil_div(N, 32);
        a.n_kt32 = (int)(2 * ceil_div(N, 64));
    } else if (dt == VSP_BF16) {
        take_parts(a, D, false, workspace, vsp_attn_backward_workspace_bytes((int32_t)B, (int32_t)Hq, (int32_t)N), workspace_bytes);
    }
    return dt == VSP_F32 ? launch_backward_f32(a, D, (hipStream_t)stream) : launch_backward_bf16(a, D, (hipStream_t)stream);
}

extern "C" int vsp_attn_prefill_backward(const vsp_tensor* dout, const vsp_tensor* q, const vsp_tensor* k,
                                         const vsp_tensor* v, const vsp_tensor* out, const vsp_tensor* lse,
                                         vsp_tensor* dq, vsp_tensor* dk, vsp_tensor* dv, float scale, int is_causal,
                                         void* workspace, size_t workspace_bytes, void* stream) {
    return backward_entry(dout, q, k, v, out, lse, dq, dk, dv, scale, is_causal, workspace, workspace_bytes, true, stream);
}

extern "C" int vsp_attn_prefill_backward_parts(const vsp_tensor* dout, const vsp_tensor* q, const vsp_tensor* k,
                                               const vsp_tensor* v, const vsp_tensor* out, const vsp_tensor* lse,
                                               vsp_tensor* dq, vsp_tensor* dk, vsp_tensor* dv, float scale, int is_causal,
                                               void* workspace, size_t workspace_bytes, void* stream) {
    return backward_entry(dout, q, k, v, out, lse, dq, dk, dv, scale, is_causal, workspace, workspace_bytes, false, stream);
}

// fp32 tensors, the arithmetic on the bf16 matrix cores with every operand as two bf16 terms (see include/vsp_attn.h).
extern "C" size_t vsp_attn_backward_split_workspace_bytes(int32_t B, int32_t Hq, int32_t Hkv, int32_t N, int32_t D) {
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0 || D <= 0) return 0;
    const size_t rows_q = (size_t)B * (size_t)Hq * (size_t)N, rows_kv = (size_t)B * (size_t)Hkv * (size_t)N;
    return align16(2 * rows_q * sizeof(float)) + 4 * (rows_q + rows_kv) * (size_t)D * sizeof(uint16_t);   // Q, dO, K, V: hi and lo
}

extern "C" int vsp_attn_prefill_backward_split(const vsp_tensor* dout, const vsp_tensor* q, const vsp_tensor* k,
                                               const vsp_tensor* v, const vsp_tensor* out, const vsp_tensor* lse,
                                               vsp_tensor* dq, vsp_tensor* dk, vsp_tensor* dv, float scale, int is_causal,
                                               void* workspace, size_t workspace_bytes, void* stream) {
    if (!q || !k || !v) return VSP_ERR_NULL;
    if (q->ndim != 4 || k->ndim != 4 || v->ndim != 4) return VSP_ERR_NDIM;
    const int64_t B = q->shape[0], Hq = q->shape[1], N = q->shape[2], D = q->shape[3];
    const int64_t Hkv = k->shape[1];
    if (Hkv <= 0 ? Hq != 0 : (Hq % Hkv != 0)) return VSP_ERR_SHAPE;
    if (q->dtype != VSP_F32) return VSP_ERR_UNSUPPORTED;
    int rc;
    if ((rc = check4(q, B, Hq, N, D, VSP_F32)) || (rc = check4(dout, B, Hq, N, D, VSP_F32)) || (rc = check4(out, B, Hq, N, D, VSP_F32)) ||
        (rc = check4(dq, B, Hq, N, D, VSP_F32)) || (rc = check4(k, B, Hkv, N, D, VSP_F32)) || (rc = check4(v, B, Hkv, N, D, VSP_F32)) ||
        (rc = check4(dk, B, Hkv, N, D, VSP_F32)) || (rc = check4(dv, B, Hkv, N, D, VSP_F32)))
        return rc;
    if (!lse) return VSP_ERR_NULL;
    if (lse->ndim != 3 || lse->shape[0] != B || lse->shape[1] != Hq || lse->shape[2] != N) return VSP_ERR_SHAPE;
    if (lse->dtype != VSP_F32) return VSP_ERR_DTYPE;
    if (B * Hq * N * D == 0) return VSP_OK;
    if (!lse->data) return VSP_ERR_NULL;
    if (D != 64 && D != 128) return VSP_ERR_UNSUPPORTED;
    if (!(fabsf(scale) < INFINITY)) return VSP_ERR_ARG;
    if (N > INT32_MAX / 2 || (uint64_t)N * (uint64_t)D * 2u > 0x7fffffffull) return VSP_ERR_ARG;
    if (!workspace || workspace_bytes < vsp_attn_backward_split_workspace_bytes((int32_t)B, (int32_t)Hq, (int32_t)Hkv, (int32_t)N, (int32_t)D))
        return VSP_ERR_WORKSPACE;
    if (!is_aligned16(workspace)) return VSP_ERR_ALIGN;
    for (const vsp_tensor* t : {dout, q, k, v, out}) {   // rows are read in 8-byte pieces
        if (((uintptr_t)t->data & 7) != 0) return VSP_ERR_ALIGN;
        for (int i = 0; i < 3; ++i)
            if (t->stride[i] % 2 != 0) return VSP_ERR_ALIGN;
    }
    for (const vsp_tensor* t : {(const vsp_tensor*)dq, (const vsp_tensor*)dk, (const vsp_tensor*)dv}) {   // and written in 16-byte ones
        if (!is_aligned16(t->data)) return VSP_ERR_ALIGN;
        for (int i = 0; i < 3; ++i)
            if (t->stride[i] % 4 != 0) return VSP_ERR_ALIGN;
    }

    const int64_t rows_q = B * Hq * N, rows_kv = B * Hkv * N;
    SplitArgs sa{};
    sa.q = (const float*)q->data, sa.dout = (const float*)dout->data, sa.out = (const float*)out->data;
    sa.k = (const float*)k->data, sa.v = (const float*)v->data, sa.lse = (const float*)lse->data;
    for (int i = 0; i < 3; ++i) {
        sa.s_q[i] = q->stride[i], sa.s_do[i] = dout->stride[i], sa.s_o[i] = out->stride[i];
        sa.s_k[i] = k->stride[i], sa.s_v[i] = v->stride[i], sa.s_l[i] = lse->stride[i];
    }
    sa.delta = (float*)workspace;
    sa.lse2 = sa.delta + rows_q;
    sa.qh = (uint16_t*)((char*)workspace + align16(2 * (size_t)rows_q * sizeof(float)));
    sa.doh = sa.qh + 2 * rows_q * D;
    sa.kh = sa.doh + 2 * rows_q * D;
    sa.vh = sa.kh + 2 * rows_kv * D;
    sa.lo_q = rows_q * D, sa.lo_kv = rows_kv * D;
    sa.B = (int)B, sa.Hq = (int)Hq, sa.Hkv = (int)Hkv, sa.N = (int)N, sa.D = (int)D;
    sa.by_n = FastDiv::of(N), sa.by_hq = FastDiv::of(Hq), sa.by_hkv = FastDiv::of(Hkv);

    BwdArgs a{};
    a.dout = sa.doh, a.q = sa.qh, a.k = sa.kh, a.v = sa.vh;
    a.dq = dq->data, a.dk = dk->data, a.dv = dv->data;
    a.delta = sa.delta, a.lse2 = sa.lse2;
    const int64_t sq[3] = {Hq * N * D, N * D, D}, skv[3] = {Hkv * N * D, N * D, D};
    for (int i = 0; i < 3; ++i) {
        a.s_do[i] = a.s_q[i] = sq[i];
        a.s_k[i] = a.s_v[i] = skv[i];
        a.s_dq[i] = dq->stride[i], a.s_dk[i] = dk->stride[i], a.s_dv[i] = dv->stride[i];
    }
    a.lo_q = sa.lo_q, a.lo_kv = sa.lo_kv;
    a.B = (int)B, a.Hq = (int)Hq, a.Hkv = (int)Hkv, a.n_rep = (int)(Hq / Hkv), a.N = (int)N;
    a.causal = is_causal ? 1 : 0;
    a.scale = scale;
    take_parts(a, D, true, workspace, vsp_attn_backward_split_workspace_bytes((int32_t)B, (int32_t)Hq, (int32_t)Hkv, (int32_t)N, (int32_t)D), workspace_bytes);
    return launch_backward_split(sa, a, D, (hipStream_t)stream);
}
