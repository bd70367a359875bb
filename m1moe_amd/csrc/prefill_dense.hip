// prefill_dense.hip — the dense part of the decoder for T prompt tokens at once.
//
// The reference forwards a prompt token by token (Sources/bench/main.swift:
// 139-141, Sources/chat/main.swift:143-149), so every weight is read once
// per token.  Here each layer's dense work for the T tokens is one pass over
// its weights:
//
//   embed_rows     the token rows of the bf16 embedding -> f32 [T][h]
//                  (InferenceEngine.swift:482-488)
//   rmsnorm_rows   x * rsqrt(mean(x^2) + eps) * w per row (Shaders.metal:96-134)
//   gemm_parts     Y[T][N] = X[T][K] W[N][K]^T (+ R): f32 activations, split
//                  exactly into three bf16 parts by the kernel that produces
//                  them, each part multiplied with the bf16 weights on
//                  v_mfma_f32_32x32x16_bf16 (exact products, f32
//                  accumulation: the arithmetic of matvecBF16,
//                  Shaders.metal:328-358, in another order)
//   rope_kv_rows   per token and head: the per-head q/k RMSNorm and RoPE at
//                  the token's position (InferenceEngine.swift:521-548), k and
//                  v rows into the caches (:215-220)
//   attn_split     causal attention of the T queries over positions 0 .. their
//                  own (Shaders.metal:209-326 for every token) on bf16 MFMA
//                  with the f32 operands split exactly, online softmax over
//                  key blocks (head_dim 64, 128; attn_causal, on the SIMD
//                  units, for head_dim 256)
//
// The MoE block runs through the grouped prefill (prefill.hip).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "internal.hpp"

namespace m1moe {
namespace {

// ---- embedding and row norms ----------------------------------------------------------

__global__ __launch_bounds__(256) void embed_rows_kernel(PfDenseArgs a) {
    const int t = blockIdx.x;
    int tok = a.tokens[t];
    if (tok < 0 || tok >= a.vocab) {
        if (threadIdx.x == 0) flag_error(a.err, 16u);
        tok = 0;
    }
    const uint16_t* row = a.embed + (size_t)tok * a.h;
    float* out = a.res + (size_t)t * a.h;
    for (int d = threadIdx.x; d < a.h; d += 256) out[d] = bf16_to_f32(row[d]);
}

// The three bf16 parts of a GEMM's f32 input, made by the kernel that produces
// it (row norms, attention): plane p of [3][T][n] holds part p of every value.
// hi = x with the low 16 bits cleared, mid = the same of x - hi, lo = x - hi -
// mid: 24 significant bits = 8 + 8 + 8, so the parts add up to x exactly.
// N = 4 or 2 consecutive values at `at`.
template <int N>
__device__ __forceinline__ void store_parts(uint16_t* at, int64_t plane, const float (&x)[N]) {
    uint32_t h[N], m[N], l[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        h[i] = __float_as_uint(x[i]) & 0xffff0000u;
        const float r = x[i] - __uint_as_float(h[i]);
        m[i] = __float_as_uint(r) & 0xffff0000u;
        l[i] = __float_as_uint(r - __uint_as_float(m[i]));
    }
    auto put = [&](uint16_t* p, const uint32_t (&v)[N]) {
        if constexpr (N == 4)
            *reinterpret_cast<uint2*>(p) = make_uint2(v[0] >> 16 | (v[1] & 0xffff0000u),
                                                      v[2] >> 16 | (v[3] & 0xffff0000u));
        else
            *reinterpret_cast<uint32_t*>(p) = v[0] >> 16 | (v[1] & 0xffff0000u);
    };
    put(at, h);
    put(at + plane, m);
    put(at + 2 * plane, l);
}

// One workgroup per row: out = x * rsqrt(sum(x^2) / n + eps) * w, as f32 (out)
// or as the three parts of a GEMM's input (parts, rows of n).  n % 4 == 0, n <=
// 1024 NV: a thread keeps its NV groups of four in registers, so x is read
// once (2048 rows of 4096: 18.0 -> 13.0 us).
template <int NV>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const float* x, const uint16_t* w, float* out,
                                                           uint16_t* parts, int64_t plane, int n, float eps) {
    __shared__ float s_red[4];
    const size_t row = (size_t)blockIdx.x * n;
    const int tid = threadIdx.x, n4 = n >> 2;
    float4 v[NV];
    uint2 b[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = min(tid + 256 * j, n4 - 1);
        v[j] = reinterpret_cast<const float4*>(x + row)[i];
        b[j] = reinterpret_cast<const uint2*>(w)[i];
    }
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (tid + 256 * j < n4)
            acc = fmaf(v[j].w, v[j].w, fmaf(v[j].z, v[j].z, fmaf(v[j].y, v[j].y, fmaf(v[j].x, v[j].x, acc))));
    acc = wave_sum(acc);
    if ((tid & 63) == 0) s_red[tid >> 6] = acc;
    __syncthreads();
    const float ss = ((s_red[0] + s_red[1]) + s_red[2]) + s_red[3];
    const float rms = rsqrtf(ss / (float)n + eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = tid + 256 * j;
        if (i >= n4) continue;
        const float y[4] = {v[j].x * rms * bf16_to_f32(b[j].x & 0xFFFFu), v[j].y * rms * bf16_to_f32(b[j].x >> 16),
                            v[j].z * rms * bf16_to_f32(b[j].y & 0xFFFFu), v[j].w * rms * bf16_to_f32(b[j].y >> 16)};
        if (parts)
            store_parts<4>(parts + row + 4 * i, plane, y);
        else
            *reinterpret_cast<float4*>(out + row + 4 * i) = float4{y[0], y[1], y[2], y[3]};
    }
}

// ---- q/k norm, RoPE, KV rows ----------------------------------------------------------

// Token blockIdx.x, heads kRopeHeads blockIdx.y .. (the q heads, then the kv
// heads): a q head rotated into qkv, a kv head's k normalised and rotated, k
// and v stored at cache row p0 + t.  G lanes per head, lane i with dims i, i +
// G, .. and their partners HD / 2 on: whole 64-lane rows of loads, no LDS.  The
// projections come as qkv, or as the GEMM's split partials (splits > 1), summed
// here in the order s = 0 .. S - 1; cos and sin from the decoder's table
// (rope_table_kernel).  Bound by the bytes at long prompts (32 + 8 heads of
// 128, T = 2048: 30.9 -> 19.4 us for 100 MB; before, one wave per head computed
// the powers, sines and cosines of its angles); 16 + 16 heads T = 333 8.8 -> 6.8,
// T = 128 with 4 splits 5.0 + 5.0 for their own sum -> 7.5.
constexpr int kRopeHeads = 8;
template <int HD>
__global__ __launch_bounds__(256) void rope_kv_rows_kernel(PfDenseArgs a) {
    constexpr int H2 = HD / 2, G = H2 < 64 ? H2 : 64, NP = H2 / G;   // lanes per head, pairs per lane
    constexpr int kSlots = 256 / G, PASS = (kRopeHeads + kSlots - 1) / kSlots;
    const int t = blockIdx.x, slot = threadIdx.x / G, i = threadIdx.x % G;
    const int p = *a.pos + t, heads = a.num_heads + a.num_kv_heads;
    const bool past = p >= a.max_seq;
    if (past && threadIdx.x == 0 && blockIdx.y == 0) flag_error(a.err, 32u);
    if (past && a.splits <= 1) return;
    // value at column c of the token's projections
    const size_t at = (size_t)t * a.ldqkv, step = (size_t)a.T * a.ldqkv;
    auto value = [&](int c) {
        if (a.splits <= 1) return a.qkv[at + c];
        float y[kGemmMaxSplits];   // every split's load in flight together
#pragma unroll
        for (int z = 0; z < kGemmMaxSplits; ++z)
            if (z < a.splits) y[z] = a.part[z * step + at + c];
        float v = y[0];
#pragma unroll
        for (int z = 1; z < kGemmMaxSplits; ++z)
            if (z < a.splits) v += y[z];
        return v;
    };
#pragma unroll
    for (int k = 0; k < PASS; ++k) {
        const int head = kRopeHeads * (int)blockIdx.y + k * kSlots + slot;
        if (head >= heads) continue;   // (uniform over the head's lanes)
        const bool is_q = head < a.num_heads;
        const int kvh = head - a.num_heads;
        const int c0 = is_q ? head * HD : a.qd + kvh * HD;
        if (past) {   // (flagged) no row of the table or the caches; the query as it was projected
            for (int d = i; is_q && d < HD; d += G) a.qkv[at + c0 + d] = value(c0 + d);
            continue;
        }
        const uint16_t* nw = is_q ? a.q_norm : a.k_norm;
        float x0[NP], x1[NP], v0[NP], v1[NP];
        float2 r[NP];
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int d = i + G * j;
            x0[j] = value(c0 + d);
            x1[j] = value(c0 + d + H2);
            if (!is_q) {
                v0[j] = value(c0 + a.kvd + d);
                v1[j] = value(c0 + a.kvd + d + H2);
            }
            r[j] = reinterpret_cast<const float2*>(a.rope)[(size_t)p * H2 + d];
            ss = fmaf(x0[j], x0[j], fmaf(x1[j], x1[j], ss));
        }
        if (nw) {
#pragma unroll
            for (int o = 1; o < G; o <<= 1) ss += __shfl_xor(ss, o);
            const float rms = 1.0f / sqrtf(ss / (float)HD + a.eps);
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                x0[j] *= rms * bf16_to_f32(nw[i + G * j]);
                x1[j] *= rms * bf16_to_f32(nw[i + G * j + H2]);
            }
        }
        float* dst = is_q ? a.qkv + at + c0 : a.kcache + (size_t)p * a.kvd + (size_t)kvh * HD;
        float* vdst = a.vcache + (size_t)p * a.kvd + (size_t)kvh * HD;
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int d = i + G * j;
            dst[d] = x0[j] * r[j].x - x1[j] * r[j].y;
            dst[d + H2] = x0[j] * r[j].y + x1[j] * r[j].x;
            if (!is_q) {
                vdst[d] = v0[j];
                vdst[d + H2] = v1[j];
            }
        }
    }
}

// ---- causal attention ------------------------------------------------------------------

// Workgroup (head, 16 queries): thread (q = tid/16, j = tid%16).  Key blocks
// of KB = 4096/HD positions are staged in LDS; thread j scores keys j, j+16,
// ... of its query, the 16 threads of a query reduce max and sum, then
// accumulate dims j, j+16, ... of the output.  Queries at positions p0+t see
// keys 0 .. p0+t.
template <int HD>
__global__ __launch_bounds__(256) void attn_causal_kernel(PfDenseArgs a) {
    constexpr int QB = 16, KB = 4096 / HD, KPT = KB / 16, DPT = HD / 16;
    __shared__ __attribute__((aligned(16))) float sQ[QB][HD];
    __shared__ float sK[KB][HD + 1];
    __shared__ __attribute__((aligned(16))) float sV[KB][HD];
    __shared__ float sP[QB][KB];
    const int h = blockIdx.x, tb = blockIdx.y * QB;
    const int tid = threadIdx.x, qi = tid >> 4, j = tid & 15;
    const int p0 = *a.pos;
    const int kvh = h / a.hpkv;
    const int t = tb + qi;
    const bool live = t < a.T;
    const int qpos = min(p0 + t, a.max_seq - 1);
    const int last = min(p0 + min(tb + QB, a.T) - 1, a.max_seq - 1);  // the block's last query position
    for (int e = tid; e < QB * HD; e += 256) {
        const int r = e / HD, d = e - r * HD;
        sQ[r][d] = tb + r < a.T ? a.qkv[(size_t)(tb + r) * a.ldqkv + (size_t)h * HD + d] : 0.f;
    }
    float m = -INFINITY, l = 0.f, acc[DPT];
#pragma unroll
    for (int e = 0; e < DPT; ++e) acc[e] = 0.f;
    for (int k0 = 0; k0 <= last; k0 += KB) {
        __syncthreads();  // (sQ published; the previous block's sK/sV/sP consumed)
        for (int e = tid; e < KB * HD / 4; e += 256) {
            const int r = e / (HD / 4), d = (e - r * (HD / 4)) * 4;
            const int kp = min(k0 + r, last);
            const size_t off = (size_t)kp * a.kvd + (size_t)kvh * HD + d;
            const float4 kv = *reinterpret_cast<const float4*>(a.kcache + off);
            const float4 vv = *reinterpret_cast<const float4*>(a.vcache + off);
            sK[r][d] = kv.x, sK[r][d + 1] = kv.y, sK[r][d + 2] = kv.z, sK[r][d + 3] = kv.w;
            *reinterpret_cast<float4*>(&sV[r][d]) = vv;
        }
        __syncthreads();
        float s[KPT];
        float bm = -INFINITY;
#pragma unroll
        for (int e = 0; e < KPT; ++e) {
            const int kk = j + 16 * e;
            float d = 0.f;
#pragma unroll 8
            for (int c = 0; c < HD; ++c) d = fmaf(sQ[qi][c], sK[kk][c], d);
            s[e] = (live && k0 + kk <= qpos) ? d * a.scale : -INFINITY;
            bm = fmaxf(bm, s[e]);
        }
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) bm = fmaxf(bm, __shfl_xor(bm, o));
        const float mn = fmaxf(m, bm);
        const float f = m == -INFINITY ? 0.f : expf(m - mn);
        float ls = 0.f;
#pragma unroll
        for (int e = 0; e < KPT; ++e) {
            const float pe = s[e] == -INFINITY ? 0.f : expf(s[e] - mn);
            sP[qi][j + 16 * e] = pe;
            ls += pe;
        }
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) ls += __shfl_xor(ls, o);
        l = fmaf(l, f, ls);
        m = mn;
#pragma unroll
        for (int e = 0; e < DPT; ++e) acc[e] *= f;
        __syncthreads();  // sP complete
        for (int kk = 0; kk < KB; ++kk) {
            const float pk = sP[qi][kk];
#pragma unroll
            for (int e = 0; e < DPT; ++e) acc[e] = fmaf(pk, sV[kk][j + 16 * e], acc[e]);
        }
    }
    if (live) {
        uint16_t* out = a.attn + (size_t)t * a.qd + (size_t)h * HD;
#pragma unroll
        for (int e = 0; e < DPT; ++e) {
            // (values of the thread's neighbour, so that pairs are stored)
            const float x = acc[e] / l, y = __shfl_xor(x, 1);
            if (j % 2 == 0) store_parts<2>(out + j + 16 * e, a.attn_plane, {x, y});
        }
    }
}

__global__ void advance_pos_kernel(int32_t* pos, int32_t by, int32_t max_seq) {
    *pos = min(*pos + by, max_seq);
}
// ---- GEMM on bf16 MFMA with the f32 input split three ways ---------------------------

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16v __attribute__((ext_vector_type(16)));

// C[M][N] = X[M][K] W[N][K]^T (+ R), X f32 as its three bf16 parts
// (store_parts), W bf16: each part multiplied with the weights on
// v_mfma_f32_32x32x16_bf16, whose products are exact, into one f32 accumulator:
// the arithmetic of the f32 GEMM (exact products, f32 sums) at a third of the
// bf16 rate.
// Tile BM tokens x BN weight rows, WM x WN waves of RM x RN blocks of 32 x 32.
// MFMA A = weight rows, B = tokens (lane l: row l % 32, k 8 (l / 32) .. + 7), so
// a lane's accumulators are four consecutive outputs of one token.  Every
// operand byte of a k-block (BK) is copied global -> LDS by the loads
// themselves (lds_copy16: no registers, no vector work in the loop) into a
// ring of NS stages, NS - 1 blocks ahead.  A stage is rows of 2 BK bytes, the X
// parts' then the weights'; 16-byte unit u of row r lies at position u ^ (r & 7)
// (BK 64) or u ^ ((r >> 2) & 3) (BK 32), so that eight lanes read by one
// ds_read_b128 hit distinct banks.  Before, f32 tiles were loaded to registers,
// split and stored to LDS by every workgroup between two barriers per k-block.
// Bound: MFMA and the operands' way through L2 (a 64 x 128 tile reads 40 KB per
// 24 MFMAs of each wave).  q, k and v of one layer, N x K 6144 x 2048: T = 37
// 12.1 -> 12.0 us, 128 19.5 -> 18.8, 333 59.9 -> 45.6, 1000 147 -> 80.5; 6144 x
// 4096: T = 100 32.6 -> 25.7, 500 139 -> 104, 2048 469 -> 333 (928 TFLOP/s of
// bf16 products; a plain bf16 product of 8192^3 reaches 1170 here); o_proj, 4096
// x 4096 at 2048 269 -> 198.
template <int RM, int RN, int WM, int WN, int BK, int NS>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_parts_kernel(GemmArgs g, int gm, int gn) {
    constexpr int BM = 32 * RM * WM, BN = 32 * RN * WN, NW = WM * WN;
    constexpr int RB = 2 * BK, U = BK / 8;                        // bytes and 16-byte units per row
    constexpr int kX = 3 * BM * RB, kStage = kX + BN * RB;
    constexpr int kPieces = kStage / 1024, kOps = kPieces / NW;   // 1 KB copies per stage, per wave
    static_assert(kPieces % NW == 0 && kOps * (NS - 2) < 64, "whole copies per wave");
    __shared__ __attribute__((aligned(1024))) uint8_t s_ring[NS * kStage];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // an XCD (workgroup id mod 8) takes consecutive tiles, eight token tiles
    // of each weight tile in a row: their operands meet in its L2
    const int total = gm * gn, bid = (int)blockIdx.x;
    const int o = total % 8 == 0 ? (bid & 7) * (total / 8) + (bid >> 3) : bid;
    const int mg = o / (8 * gn), mh = min(8, gm - 8 * mg), in = o - mg * 8 * gn;
    const int m0 = (8 * mg + in % mh) * BM, n0 = in / mh * BN;
    // the weights' segment (its borders are multiples of BN)
    const uint16_t* w = !g.W1 || n0 < g.n1 ? g.W + (size_t)n0 * g.K
                        : n0 < g.n2        ? g.W1 + (size_t)(n0 - g.n1) * g.K
                                           : g.W2 + (size_t)(n0 - g.n2) * g.K;
    const uint8_t* xb = reinterpret_cast<const uint8_t*>(g.X);
    const uint8_t* wb = reinterpret_cast<const uint8_t*>(w);
    auto swizzle = [](int row) { return U == 4 ? (row >> 2) & 3 : row & 7; };
    uint32_t voff[kOps];
#pragma unroll
    for (int i = 0; i < kOps; ++i) {
        const int row = (64 / U) * (wave * kOps + i) + lane / U;   // of the stage
        const int u = lane % U ^ swizzle(row);
        const bool isx = row < 3 * BM;
        const int r = isx ? row % BM : row - 3 * BM;
        const uint32_t at = isx ? (uint32_t)min(m0 + r, g.M - 1) : (uint32_t)min(r, g.N - 1 - n0);
        voff[i] = (isx ? (uint32_t)(row / BM) * (uint32_t)(g.xplane * 2) : 0u) + at * (uint32_t)(g.K * 2) + u * 16;
    }
    const int nkb = g.K / BK, S = (int)gridDim.y, z = (int)blockIdx.y;
    const int kbeg = z * nkb / S, kend = (z + 1) * nkb / S;
    const uint32_t ring = lds_addr(s_ring);
    // block kb's copies into its slot (past the last block that block is read
    // again, into a slot no step reads, so every wave always has the same
    // number of copies behind a block's)
    auto issue = [&](int kb, int slot) {
        const size_t ko = (size_t)min(kb, kend - 1) * RB;
#pragma unroll
        for (int i = 0; i < kOps; ++i) {
            const int p = wave * kOps + i;
            lds_copy16(voff[i], (p < kX / 1024 ? xb : wb) + ko, ring + slot * kStage + p * 1024);
        }
    };
    f32x16v acc[RN][RM];
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][i][e] = 0.f;
    const int r32 = lane & 31, h = lane >> 5, wm = (wave % WM) * 32 * RM, wn = (wave / WM) * 32 * RN;
    const int sw = swizzle(r32);
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) issue(kbeg + s, s);
    int slot = 0;
    for (int kb = kbeg; kb < kend; ++kb) {
        wait_vm<kOps * (NS - 2)>();   // block kb's copies are in (the next NS - 2 may not be)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        issue(kb + NS - 1, slot == 0 ? NS - 1 : slot - 1);
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t* st = s_ring + slot * kStage;
        // the operands of k-step ks + 1 are read while step ks is multiplied
        bf16x8 af[2][RN], bf[2][3][RM];
        auto read = [&](int ks, int at) {
            const int u = ((2 * ks + h) ^ sw) * 16;
#pragma unroll
            for (int j = 0; j < RN; ++j)
                af[at][j] = *reinterpret_cast<const bf16x8*>(st + kX + (wn + 32 * j + r32) * RB + u);
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int i = 0; i < RM; ++i)
                    bf[at][p][i] = *reinterpret_cast<const bf16x8*>(st + (p * BM + wm + 32 * i + r32) * RB + u);
        };
        read(0, 0);
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
            if (ks + 1 < BK / 16) read(ks + 1, (ks + 1) & 1);
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int i = 0; i < RM; ++i)
#pragma unroll
                    for (int j = 0; j < RN; ++j)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][j], bf[ks & 1][p][i],
                                                                            acc[j][i], 0, 0, 0);
        }
        slot = slot + 1 == NS ? 0 : slot + 1;
    }
    wait_vm<0>();   // no copy into LDS may still be in flight when the workgroup ends
#pragma unroll
    for (int i = 0; i < RM; ++i) {
        const int m = m0 + wm + 32 * i + r32;
        if (m >= g.M) continue;
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int n = n0 + wn + 32 * j + 8 * v + 4 * h;
                if (n >= g.N) continue;   // (N % 4 == 0)
                float4 y{acc[j][i][4 * v], acc[j][i][4 * v + 1], acc[j][i][4 * v + 2], acc[j][i][4 * v + 3]};
                if (S > 1) {
                    *reinterpret_cast<float4*>(g.part + ((size_t)z * g.M + m) * g.N + n) = y;
                } else {
                    if (g.R) {
                        const float4 r = *reinterpret_cast<const float4*>(g.R + (size_t)m * g.ldc + n);
                        y.x += r.x, y.y += r.y, y.z += r.z, y.w += r.w;
                    }
                    *reinterpret_cast<float4*>(g.C + (size_t)m * g.ldc + n) = y;
                }
            }
    }
}

// C = sum over s = 0 .. S-1 of the split-K partials (in that order, at most
// kGemmMaxSplits) + R, one output row per workgroup, then that row's RMSNorm with the arithmetic of rmsnorm_rows_kernel
// (each thread's squares summed in its own column order, four at a time).
__global__ __launch_bounds__(256) void splitk_sum_norm_kernel(GemmArgs g) {
    __shared__ float s_red[4];
    const size_t m = blockIdx.x, mn4 = (size_t)g.M * g.N / 4;
    const float4* p = reinterpret_cast<const float4*>(g.part) + m * (g.N / 4);
    float* c = g.C + m * g.ldc;
    float acc = 0.f;
    for (int i = threadIdx.x; i < g.N / 4; i += 256) {
        float4 v[kGemmMaxSplits];  // every split's load in flight together
#pragma unroll
        for (int z = 0; z < kGemmMaxSplits; ++z)
            if (z < g.splits) v[z] = p[(size_t)z * mn4 + i];
        float4 y = v[0];
#pragma unroll
        for (int z = 1; z < kGemmMaxSplits; ++z)
            if (z < g.splits) y.x += v[z].x, y.y += v[z].y, y.z += v[z].z, y.w += v[z].w;
        if (g.R) {
            const float4 r = *reinterpret_cast<const float4*>(g.R + m * g.ldc + 4 * i);
            y.x += r.x, y.y += r.y, y.z += r.z, y.w += r.w;
        }
        *reinterpret_cast<float4*>(c + 4 * i) = y;
        acc = fmaf(y.x, y.x, acc);
        acc = fmaf(y.y, y.y, acc);
        acc = fmaf(y.z, y.z, acc);
        acc = fmaf(y.w, y.w, acc);
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = acc;
    __syncthreads();
    const float ss = ((s_red[0] + s_red[1]) + s_red[2]) + s_red[3];
    const float rms = rsqrtf(ss / (float)g.N + g.norm_eps);
    float* o = g.norm_out + m * g.ldc;
    for (int i = threadIdx.x; i < g.N; i += 256) o[i] = c[i] * rms * bf16_to_f32(g.norm_w[i]);
}

}  // namespace

int launch_pf_embed(const PfDenseArgs& a, void* stream) {
    hipLaunchKernelGGL(embed_rows_kernel, dim3((unsigned)a.T), dim3(256), 0, static_cast<hipStream_t>(stream), a);
    return (int)hipGetLastError();
}

int launch_rmsnorm_rows(const float* x, const uint16_t* w, float* out, uint16_t* parts, int64_t plane, int rows,
                        int n, float eps, void* stream) {
    if (n % 4 || n <= 0 || n > 8192) return (int)hipErrorInvalidValue;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid((unsigned)rows);
    if (n <= 2048)
        hipLaunchKernelGGL(rmsnorm_rows_kernel<2>, grid, dim3(256), 0, st, x, w, out, parts, plane, n, eps);
    else if (n <= 4096)
        hipLaunchKernelGGL(rmsnorm_rows_kernel<4>, grid, dim3(256), 0, st, x, w, out, parts, plane, n, eps);
    else
        hipLaunchKernelGGL(rmsnorm_rows_kernel<8>, grid, dim3(256), 0, st, x, w, out, parts, plane, n, eps);
    return (int)hipGetLastError();
}

namespace {
template <int RM, int RN, int WM, int WN, int BK, int NS>
void launch_gemm_tile(const GemmArgs& g, hipStream_t st) {
    const int gm = (g.M + 32 * RM * WM - 1) / (32 * RM * WM), gn = (g.N + 32 * RN * WN - 1) / (32 * RN * WN);
    hipLaunchKernelGGL((gemm_parts_kernel<RM, RN, WM, WN, BK, NS>), dim3((unsigned)(gm * gn), (unsigned)g.splits),
                       dim3(64 * WM * WN), 0, st, g, gm, gn);
}
}  // namespace

int64_t gemm_part_floats(int cus) { return 3LL * cus * 64 * 64; }

namespace {
// Tiles of 64 x 128, two workgroups per CU: measured best or within a few
// percent at every size but one, a grid of 128 x 256 tiles that is more than
// three quarters of one round of the CUs (of 256, M x N x K: 256 of them, 2048 x
// 4096 x 4096, 200 us, 1024 of 64 x 128 215; 216, 1100 x 6144 x 4096, 175 against
// 207; four layers of 1280 x 5120 x 4096, 200, a prompt 1823 against 1935 us; but 192
// at 1000 x 6144 x 2048 84 against 82, 384 at 2048 x 6144 x 4096 342 against 307).
// The weight segments' borders must be tile borders.  Fewer tiles than CUs: the
// k-blocks are split over gridDim.y (at least 4 blocks of 64 per split: 6 of them
// 279 -> 291 us a prompt of 17 tokens, hidden 1536, four layers; at most two
// workgroups per CU and gemm_part_floats of partials in all) and the partials summed
// in a fixed order, so results do not depend on timing.  The workspace's 12 MB is
// what limits the splits from 384 workgroups of whole tiles on; with 16 MB, two per
// CU, four layers of hidden 4096 would take 657 us in place of 677 at 128 tokens, 854
// in place of 948 at 300, of hidden 2048 440 in place of 445 at 128.
struct GemmPlan {
    bool big, wide;
    int splits;
};
GemmPlan gemm_plan(const GemmArgs& g) {
    const long gm64 = (g.M + 63) / 64, gn128 = (g.N + 127) / 128, gn64 = (g.N + 63) / 64;
    const long big = (long)((g.M + 127) / 128) * ((g.N + 255) / 256);
    GemmPlan p{};
    // (instead of one column of tiles, two narrow ones: one layer of hidden 128 at 5 /
    // 1000 tokens 55.2 -> 54.0, 83.2 -> 81.8 us a prompt)
    p.wide = g.N > 128 && (!g.W1 || (g.n1 % 128 == 0 && g.n2 % 128 == 0));
    p.big = 4 * big > 3 * g.cus && big <= g.cus && (!g.W1 || (g.n1 % 256 == 0 && g.n2 % 256 == 0));
    const long tiles = p.wide ? gn128 * gm64 : gn64 * gm64, nkb = g.K / 64;
    long S = !p.big && g.part && tiles < g.cus ? std::min(2 * g.cus / tiles, nkb / 4) : 1;
    S = std::min({S, (long)kGemmMaxSplits, (long)(gemm_part_floats(g.cus) / ((int64_t)g.M * g.N))});
    p.splits = (int)std::max(S, 1l);
    return p;
}
}  // namespace

int gemm_splits(const GemmArgs& g) { return gemm_plan(g).splits; }

int launch_gemm(const GemmArgs& g0, void* stream) {
    GemmArgs g = g0;
    if (g.K % 64 || g.K <= 0 || g.M <= 0 || g.N <= 0 || g.N % 4 || g.ldc % 4 || (uintptr_t)g.C % 16 ||
        (uintptr_t)g.R % 16 || g.xplane < (int64_t)g.M * g.K || 6 * g.xplane >= (1ll << 32) ||
        2ll * 128 * g.K >= (1ll << 32) || g.cus <= 0)
        return (int)hipErrorInvalidValue;
    if (g.W1 && (!g.W2 || g.n1 < 0 || g.n1 > g.n2 || g.n2 > g.N || g.n1 % 64 || g.n2 % 64))
        return (int)hipErrorInvalidValue;
    if (g.norm_w && (!g.norm_out || g.ldc != g.N)) return (int)hipErrorInvalidValue;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const GemmPlan plan = gemm_plan(g);
    g.splits = plan.splits;
    if (plan.big)
        launch_gemm_tile<2, 2, 2, 4, 32, 3>(g, st);
    else if (plan.wide)
        launch_gemm_tile<1, 2, 2, 2, 64, 2>(g, st);
    else
        launch_gemm_tile<1, 1, 2, 2, 64, 2>(g, st);
    if (g.splits > 1 && g.norm_w)  // the sum makes the row norm too
        hipLaunchKernelGGL(splitk_sum_norm_kernel, dim3((unsigned)g.M), dim3(256), 0, st, g);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !g.norm_w || g.splits > 1) return (int)e;
    return launch_rmsnorm_rows(g.C, g.norm_w, g.norm_out, nullptr, 0, g.M, g.N, g.norm_eps, stream);
}

int launch_pf_rope_kv(const PfDenseArgs& a, void* stream) {
    if (!a.rope || (a.splits > 1 && (!a.part || a.splits > kGemmMaxSplits))) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)a.T, (unsigned)((a.num_heads + a.num_kv_heads + kRopeHeads - 1) / kRopeHeads));
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (a.head_dim) {
        case 64: hipLaunchKernelGGL(rope_kv_rows_kernel<64>, grid, dim3(256), 0, st, a); break;
        case 128: hipLaunchKernelGGL(rope_kv_rows_kernel<128>, grid, dim3(256), 0, st, a); break;
        case 256: hipLaunchKernelGGL(rope_kv_rows_kernel<256>, grid, dim3(256), 0, st, a); break;
        default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

// ---- causal attention on bf16 MFMA with f32 operands split three ways ----------------

// Three bf16 parts of eight f32 values, two per word: hi = bf16(x), mid =
// bf16(x - hi), lo = bf16(x - hi - mid), each rounded to nearest: 24
// significant bits, so the parts add up to x exactly.  The differences of a
// pair are one v_dot2 each, (hi0, hi1) . (-1, 0) + x0 and (hi0, hi1) . (0, -1)
// + x1 (exact: the result fits f32), 3.5 instructions per value against 5.5
// with the parts unpacked and subtracted.  The constants live in scalar
// registers: as literals the compiler makes them inline operands, which the
// instruction reads as f32, not as a bf16 pair.
struct Split8 {
    bf16x8 h, m, l;
};
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ Split8 split8_rne(const float (&v)[8]) {
    uint32_t c0, c1;
    asm("s_mov_b32 %0, 0xbf80" : "=s"(c0));
    asm("s_mov_b32 %0, 0xbf800000" : "=s"(c1));
    const bf16x2 n0 = __builtin_bit_cast(bf16x2, c0), n1 = __builtin_bit_cast(bf16x2, c1);
    uint32_t h[4], m[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x0 = v[2 * i], x1 = v[2 * i + 1];
        const bf16x2 hi = __builtin_convertvector(f32x2v{x0, x1}, bf16x2);
        const float r0 = __builtin_amdgcn_fdot2_f32_bf16(hi, n0, x0, false);
        const float r1 = __builtin_amdgcn_fdot2_f32_bf16(hi, n1, x1, false);
        const bf16x2 mid = __builtin_convertvector(f32x2v{r0, r1}, bf16x2);
        const float t0 = __builtin_amdgcn_fdot2_f32_bf16(mid, n0, r0, false);
        const float t1 = __builtin_amdgcn_fdot2_f32_bf16(mid, n1, r1, false);
        h[i] = __builtin_bit_cast(uint32_t, hi);
        m[i] = __builtin_bit_cast(uint32_t, mid);
        l[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{t0, t1}, bf16x2));
    }
    Split8 s;
    s.h = __builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3]));
    s.m = __builtin_bit_cast(bf16x8, make_uint4(m[0], m[1], m[2], m[3]));
    s.l = __builtin_bit_cast(bf16x8, make_uint4(l[0], l[1], l[2], l[3]));
    return s;
}

// acc += A B over 16 contraction slots with both f32 operands split: the six
// part products down to 2^-16 of the largest, small ones first.  The three left
// out add up to at most 2^-23 of a product and 2^-27.4 of it in the root mean square, of
// either sign (an f32 product's rounding: 2^-24 and 2^-25.2).  The prompts' error
// against 64 bits did not grow over the exact products of f32 MFMA (last logits of
// two layers, relative 2-norm, mean of six: 16 heads of 128 at 333 tokens 2.76e-7 ->
// 2.72e-7, 32 q / 8 kv heads at 1500 7.51e-7 -> 7.59e-7, with queries eight times as
// large 5.37e-5 -> 5.28e-5, 8 q / 2 kv heads of 64 at 333 2.45e-7 -> 2.44e-7).
__device__ __forceinline__ void mfma_split(const Split8& a, const Split8& b, f32x16v& acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.l, b.h, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.l, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.m, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.h, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.m, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.h, acc, 0, 0, 0);
}

__device__ __forceinline__ float halves_max(float v) {  // lanes l and l ^ 32
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_add(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// One wave's 32 queries of one head: its running softmax and the transposed
// output accumulators.  Lane l holds query l % 32 (both halves the same one):
// of the scores S^T = K Q^T of a 32-key block the 16 keys 8 (v / 4) + 4 h + v
// % 4 (h = l / 32), of O^T (NT tiles of 32 rows) the rows in the same order;
// dim NT r + t of the head is row r of tile t, so that a lane's V and output
// values of all tiles are NT consecutive floats.
// Contraction slots: lane half h, element e of k-step s is dim (or key) 16 s
// + 4 h + e for e < 4 and 16 s + 8 + 4 h + e - 4 above: the accumulator's row
// order, so P multiplies V straight from the lanes that computed it.
template <int HD>
struct AttnWave {
    static constexpr int NT = HD / 32, NS = HD / 16;
    typedef float vecT __attribute__((ext_vector_type(NT)));
    const float *qrow, *kbase, *vbase;   // the lane's query; the kv head's columns
    int kvd, r32, h, t, qpos, first, last, nblk;
    float scale, m, l;                   // m: the running maximum, in exponents of two
    f32x16v acc[NT];

    __device__ __forceinline__ void init(const PfDenseArgs& a, int head, int t0, int lane) {
        const int p0 = *a.pos, kvh = head / a.hpkv;
        r32 = lane & 31;
        h = lane >> 5;
        kvd = a.kvd;
        scale = a.scale;
        t = min(t0 + r32, a.T - 1);
        qpos = min(p0 + t, a.max_seq - 1);
        first = min(p0 + t0, a.max_seq - 1);                       // the tile's first and
        last = min(p0 + min(t0 + 31, a.T - 1), a.max_seq - 1);     // last query position
        nblk = last / 32 + 1;
        qrow = a.qkv + (size_t)t * a.ldqkv + (size_t)head * HD;
        kbase = a.kcache + (size_t)kvh * HD;
        vbase = a.vcache + (size_t)kvh * HD;
        clear();
    }
    __device__ __forceinline__ void clear() {
        m = -INFINITY;
        l = 0.f;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
    }
    // k-step s of the lane's query, scaled (Log2Scale) and split
    __device__ __forceinline__ Split8 query(int s) const {
        const Log2Scale c(scale);
        const float4 x0 = *reinterpret_cast<const float4*>(qrow + 16 * s + 4 * h);
        const float4 x1 = *reinterpret_cast<const float4*>(qrow + 16 * s + 8 + 4 * h);
        return split8_rne({c(x0.x), c(x0.y), c(x0.z), c(x0.w), c(x1.x), c(x1.y), c(x1.z), c(x1.w)});
    }
    // The running softmax (Shaders.metal:245-289 in pieces) over the lane's 16
    // keys and the other half's: s (scores as exponents of two) becomes the
    // numerators, acc is rescaled.
    __device__ __forceinline__ void softmax(int k0, f32x16v& s) {
        if (k0 + 31 > first) {   // (uniform) some query of the tile does not see the whole block
#pragma unroll
            for (int v = 0; v < 16; ++v)
                s[v] = k0 + 8 * (v >> 2) + 4 * h + (v & 3) <= qpos ? s[v] : -INFINITY;
        }
        float bm = -INFINITY;
#pragma unroll
        for (int v = 0; v < 16; ++v) bm = fmaxf(bm, s[v]);
        const float mn = fmaxf(m, halves_max(bm));
        const float mc = mn == -INFINITY ? 0.f : mn;   // (no key seen yet: every numerator 0)
        const float f = __builtin_amdgcn_exp2f(m - mc);
        float ls = 0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            s[v] = __builtin_amdgcn_exp2f(s[v] - mc);
            ls += s[v];
        }
        l = fmaf(l, f, ls);
        m = mn;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][v] *= f;
    }
    // Whether some score (odd: a sum of them times 0) or output of the wave is
    // not finite: an infinity or NaN among its q, k and v, or a value so
    // large that its bf16 part rounds to infinity (its parts then add up to NaN).
    __device__ __forceinline__ bool not_finite(float odd) const {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) odd = fmaf(acc[i][v], 0.f, odd);
        return __any(odd != 0.f);
    }
    // Blocks b0, b0 + step, ... again on f32 MFMA, for such a wave: lane half h
    // supplies dims 8 j + 4 h + e of Q and K, then the lane's own keys of P.
    __device__ __forceinline__ void f32_blocks(int b0, int step) {
        clear();
#pragma unroll 1
        for (int b = b0; b < nblk; b += step) {
            const int k0 = 32 * b;
            f32x16v s;
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll 1
            for (int j = 0; j < 2 * NS; ++j) {
                const float4 q = *reinterpret_cast<const float4*>(qrow + 8 * j + 4 * h);
                const float4 k = *reinterpret_cast<const float4*>(
                    kbase + (size_t)min(k0 + r32, last) * kvd + 8 * j + 4 * h);
                const Log2Scale c(scale);
                s = __builtin_amdgcn_mfma_f32_32x32x2f32(k.x, c(q.x), s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_32x32x2f32(k.y, c(q.y), s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_32x32x2f32(k.z, c(q.z), s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_32x32x2f32(k.w, c(q.w), s, 0, 0, 0);
            }
            softmax(k0, s);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const vecT x = *reinterpret_cast<const vecT*>(
                    vbase + (size_t)min(k0 + 8 * (v >> 2) + 4 * h + (v & 3), last) * kvd + NT * r32);
#pragma unroll
                for (int i = 0; i < NT; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i], s[v], acc[i], 0, 0, 0);
            }
        }
    }
};

// Causal attention, head_dim 64 or 128, on v_mfma_f32_32x32x16_bf16 with the
// f32 operands split (mfma_split): six bf16 MFMAs in place of one f32 MFMA at
// a sixteenth of the rate.  Workgroup = (head, 32 queries); wave w takes key
// blocks w, w + 4, ... with a running softmax of its own, the four merged
// through LDS at the end.  K and V come straight from the cache into the lanes
// that split and multiply them: no barrier in the loop, and heads x T / 32
// workgroups, so a short prompt still spreads over the chip.  Before, 64
// queries per workgroup on f32 MFMA with K and V staged in LDS: 16 heads of
// 128, T = 128 26.1 -> 10.5 us, T = 333 65.4 -> 17.4; 32 q / 8 kv heads, T =
// 2048 632 -> 285 us.  Bound at long prompts by the vector unit (the splits of
// K and V, ~800 instructions per 96 MFMAs) and the K loads' 32-byte pieces
// (data return busy 78% of the time).  128 queries per workgroup sharing
// each block's split through LDS took 255 us there (eight waves; their
// barriers keep the splits and the MFMAs of a SIMD's two waves in step), the
// same as this form at T = 1500 and 132 -> 178 us at 16 heads, T = 2000.
template <int HD>
__global__ __launch_bounds__(256, 2) void attn_split_kernel(PfDenseArgs a) {
    constexpr int NT = HD / 32, NS = HD / 16;
    typedef typename AttnWave<HD>::vecT vecT;
    // the split queries (an operand image per part and k-step), then the
    // waves' partial outputs
    constexpr int kQBytes = 3 * NS * 64 * 16, kOBytes = 4 * 16 * NT * 64 * 4;
    __shared__ __attribute__((aligned(16))) uint8_t s_buf[kQBytes > kOBytes ? kQBytes : kOBytes];
    __shared__ float s_m[4][32], s_l[4][32];
    bf16x8* sQ = reinterpret_cast<bf16x8*>(s_buf);  // [3][NS][64]
    float* sO = reinterpret_cast<float*>(s_buf);    // [4][16 NT][64]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    // longest tiles first; with heads in multiples of 8 an XCD (workgroup id
    // mod 8) takes consecutive heads, whose K and V share its L2
    const int H = a.num_heads, nq = (a.T + 31) / 32, id = (int)blockIdx.x;
    const int hx = H % 8 == 0 ? H / 8 : H, j = H % 8 == 0 ? id >> 3 : id;
    const int head = (H % 8 == 0 ? (id & 7) * hx : 0) + j % hx, t0 = (nq - 1 - j / hx) * 32;
    AttnWave<HD> w;
    w.init(a, head, t0, lane);
    float4 kf[2 * NS];
    vecT vf[16];
    // half `part` of a block's K dims or V keys; the loads are kept where they
    // are written (the registers of both whole blocks do not fit two waves per SIMD)
    auto load_k = [&](int k0, int part) {
        const float* row = w.kbase + (size_t)min(k0 + w.r32, w.last) * w.kvd + 4 * w.h;
#pragma unroll
        for (int i = part * NS; i < (part + 1) * NS; ++i) kf[i] = *reinterpret_cast<const float4*>(row + 8 * i);
        asm volatile("" ::: "memory");
    };
    auto load_v = [&](int k0, int part) {
#pragma unroll
        for (int v = 8 * part; v < 8 * part + 8; ++v)
            vf[v] = *reinterpret_cast<const vecT*>(
                w.vbase + (size_t)min(k0 + 8 * (v >> 2) + 4 * w.h + (v & 3), w.last) * w.kvd + NT * w.r32);
        asm volatile("" ::: "memory");
    };
    if (wave < w.nblk) {
        load_k(32 * wave, 0);
        load_k(32 * wave, 1);
    }
    for (int s = wave; s < NS; s += 4) {
        const Split8 q = w.query(s);
        sQ[(0 * NS + s) * 64 + lane] = q.h;
        sQ[(1 * NS + s) * 64 + lane] = q.m;
        sQ[(2 * NS + s) * 64 + lane] = q.l;
    }
    __syncthreads();
    float odd = 0.f;
    for (int b = wave; b < w.nblk; b += 4) {
        const int k0 = 32 * b;
        load_v(k0, 0);
        f32x16v s;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const Split8 q{sQ[(0 * NS + i) * 64 + lane], sQ[(1 * NS + i) * 64 + lane],
                           sQ[(2 * NS + i) * 64 + lane]};
            mfma_split(split8_rne({kf[2 * i].x, kf[2 * i].y, kf[2 * i].z, kf[2 * i].w, kf[2 * i + 1].x,
                                   kf[2 * i + 1].y, kf[2 * i + 1].z, kf[2 * i + 1].w}), q, s);
        }
        load_v(k0, 1);
        load_k(k0 + 128, 0);  // (rows past the last are read again, not used)
#pragma unroll
        for (int v = 0; v < 16; ++v) odd = fmaf(s[v], 0.f, odd);
        w.softmax(k0, s);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const Split8 p = split8_rne({s[8 * k], s[8 * k + 1], s[8 * k + 2], s[8 * k + 3], s[8 * k + 4],
                                         s[8 * k + 5], s[8 * k + 6], s[8 * k + 7]});
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = vf[8 * k + e][i];
                mfma_split(split8_rne(x), p, w.acc[i]);
            }
            if (k == 0) load_k(k0 + 128, 1);
        }
    }
    if (w.not_finite(odd)) w.f32_blocks(wave, 4);
    // the four waves' partials: out = sum_w acc_w e^(m_w - M) / sum_w l_w e^(m_w - M)
    const float l = halves_add(w.l);
    __syncthreads();  // (every wave is done with the queries)
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) sO[(wave * 16 * NT + v * NT + i) * 64 + lane] = w.acc[i][v];
    if (w.h == 0) {
        s_m[wave][w.r32] = w.m;
        s_l[wave][w.r32] = l;
    }
    __syncthreads();
    float f[4], M = -INFINITY, L = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) M = fmaxf(M, s_m[k][w.r32]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f[k] = s_m[k][w.r32] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_m[k][w.r32] - M);
        L = fmaf(s_l[k][w.r32], f[k], L);
    }
    if (t0 + w.r32 >= a.T) return;
    // wave w: accumulator rows 8 w + 4 h .. + 3 of every tile
    uint16_t* out = a.attn + (size_t)w.t * a.qd + (size_t)head * HD;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        float o[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            float x = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                x = fmaf(sO[(k * 16 * NT + (4 * wave + v) * NT + i) * 64 + lane], f[k], x);
            o[i] = x / L;
        }
        store_parts<NT>(out + NT * (8 * wave + 4 * w.h + v), a.attn_plane, o);
    }
}

int launch_pf_attention(const PfDenseArgs& a, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid_s((unsigned)a.num_heads * (unsigned)((a.T + 31) / 32));
    const dim3 grid((unsigned)a.num_heads, (unsigned)((a.T + 15) / 16));
    switch (a.head_dim) {
        case 64: hipLaunchKernelGGL(attn_split_kernel<64>, grid_s, dim3(256), 0, st, a); break;
        case 128: hipLaunchKernelGGL(attn_split_kernel<128>, grid_s, dim3(256), 0, st, a); break;
        case 256: hipLaunchKernelGGL(attn_causal_kernel<256>, grid, dim3(256), 0, st, a); break;
        default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

int launch_advance_pos(int32_t* pos, int32_t by, int32_t max_seq, void* stream) {
    hipLaunchKernelGGL(advance_pos_kernel, dim3(1), dim3(1), 0, static_cast<hipStream_t>(stream), pos, by, max_seq);
    return (int)hipGetLastError();
}

}  // namespace m1moe
