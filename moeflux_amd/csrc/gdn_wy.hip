// The delta rule over a prompt chunk in blocked form, on the matrix cores.
//
// The reference steps the recurrence token by token (crates/moeflux/src/riir/
// linear_attn.rs:373-411; eval_prompt is a token loop, riir/mod.rs:1196-1214):
//   S <- g_t S;  d_t = beta_t (v_t - S k_t);  S <- S + d_t k_t^T;  o_t = S q_t.
// For a block of C = 64 tokens that starts from state S0, with L_t = sum_{i<=t} log g_i,
//   A[i][j] = beta_i e^{L_i-L_j} (k_i . k_j)  (j < i),      T = (I + A)^-1,
//   W  = T diag(beta e^L) K,   U = T diag(beta) V,   M[i][j] = e^{L_i-L_j} (q_i . k_j)  (j <= i),
//   D  = U - W S0^T                      (the d_t of the block, one row per token)
//   O  = diag(e^L) Q S0^T + M D
//   S' = e^{L_C} S0 + D^T diag(e^{L_C-L}) K
// are the same d_t, o_t and final state (exact arithmetic; f32 rounding differs at 1e-6).
// A token whose decay is zero (the reference's exp underflows, or its softplus overflows) starts L
// afresh: factors across it are exactly 0, as they are token by token.
// Everything before D depends on the inputs only and is computed for all blocks of the
// chunk at once (gdn_wy_kernel, one workgroup per (block, value head)); the four
// products that involve the state run block after block with the state in registers
// (gdn_wy_recur_kernel, one workgroup per 32 rows of a head's state, rows being
// independent).  The products are v_mfma_f32_16x16x32_bf16 over operands split into three bf16 numbers (see wy_split4), the
// inversion's small ones v_mfma_f32_16x16x4_f32.
//
// Operand conventions of the f32 instruction (lane l, m = n = l % 16, g = l / 16):
// A[m][g], B[g][n] in; D[4g+i][n], i = 0..3, out.  A contraction over 16 values is done as
// 4 instructions i = 0..3 in which lane group g contributes value number 4g+i: then one
// float4 (values 4g..4g+3) feeds the four instructions, and a D tile can be used as the
// B operand of a contraction over its rows without moving data between lanes.
#include <type_traits>

#include "gdn_device.h"
#include "sdpa_wave.h"

namespace mfa {

typedef __attribute__((ext_vector_type(4))) float wy_f32x4;

static constexpr int kC = 64;  // tokens per block

__device__ inline wy_f32x4 mfma4(float4 a, float4 b, wy_f32x4 acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
    return acc;
}
__device__ inline float4 lds_f4(const float *p) {
    const gdn_f32x4 v = *reinterpret_cast<const gdn_f32x4 *>(p);
    return float4{v.x, v.y, v.z, v.w};
}
// Value head served by the workgroups with x index bx.  Workgroups go to the 8 XCDs in turn, so with a
// head count that is a multiple of 8 a head's workgroups share an XCD and its L2; heads that share a
// k head (and read the same q and k inputs) are given x indices 8 apart, the same XCD, so that the
// second reader of a line finds it in that L2 (block precompute 22.3 -> 21.6 us per 512 tokens).
__device__ inline int wy_head_of(int bx, int Hk, int Hv) {
    const int r = Hv / Hk;
    if (Hv % 8 != 0 || (Hv / 8) % r != 0) return bx;
    const int x = bx & 7, j = bx >> 3;
    return (x + 8 * (j / r)) * r + j % r;
}
__device__ inline float4 as_f4(wy_f32x4 v) { return float4{v[0], v[1], v[2], v[3]}; }
// a 16-byte load kept as a vector register value (members of a struct of operands)
__device__ inline wy_f32x4 load_v4(const float *p) { return *reinterpret_cast<const wy_f32x4 *>(p); }

// An f32 x as the sum of three bf16 numbers, h = bf16(x), m = bf16(x - h), l = x - h - m: exact, 24 bits are 8 + 8 + 8, and bf16 has
// f32's exponents, so that every value keeps its own scale, whatever lies beside it in a tile.  (Two f16 parts are half the terms
// and two bytes less, but share a scale along a contraction: a token 1e8 times the others took the bits of the tokens ahead of it, and
// small W, T or K' under a fixed scale lost theirs.)  Below 2^-102 l loses its last bits; within 2^-9 of the largest f32 h is infinite.
// Of a product all but m l, l m and l l is formed and summed in f32: what is left out is below 2^-24 of it.  Six
// instructions take 96 clocks for 32 contracted values, f32 instructions 256.
// Contractions over a block's tokens go in steps of 32, and of 16 where the next 16 lie past the diagonal: zeros
// there would carry a later token's infinity or NaN into earlier ones.
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;   // (LDS holding f32 and bf16 parts in turn is read and written as vectors, which alias anything)
struct WyFour { u32x2 p[3]; };    // h, m, l of four values
struct WyEight { u32x4 p[3]; };
__device__ inline void wy_split2(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l) {
    auto low = [](uint32_t x) { return __builtin_bit_cast(float, x << 16); };
    auto high = [](uint32_t x) { return __builtin_bit_cast(float, x & 0xffff0000u); };
    h = pack_bf16(a, b);
    a -= low(h), b -= high(h);
    m = pack_bf16(a, b);
    l = pack_bf16(a - low(m), b - high(m));
}
__device__ inline WyFour wy_split4(float a, float b, float c, float d) {
    uint32_t h0, h1, m0, m1, l0, l1;
    wy_split2(a, b, h0, m0, l0);
    wy_split2(c, d, h1, m1, l1);
    return {{u32x2{h0, h1}, u32x2{m0, m1}, u32x2{l0, l1}}};
}
__device__ inline WyFour wy_split4(const wy_f32x4 &x) { return wy_split4(x[0], x[1], x[2], x[3]); }
__device__ inline WyEight wy_join(const WyFour &x, const WyFour &y) {
    WyEight r;
#pragma unroll
    for (int i = 0; i < 3; i++) r.p[i] = u32x4{x.p[i][0], x.p[i][1], y.p[i][0], y.p[i][1]};
    return r;
}
// the four values whose parts these are
__device__ inline wy_f32x4 wy_whole(const WyFour &x) {
    wy_f32x4 r;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        auto low = [&](int k) { return __builtin_bit_cast(float, (uint32_t)x.p[k][i] << 16); };
        auto high = [&](int k) { return __builtin_bit_cast(float, (uint32_t)x.p[k][i] & 0xffff0000u); };
        r[2 * i] = low(0) + (low(1) + low(2));
        r[2 * i + 1] = high(0) + (high(1) + high(2));
    }
    return r;
}
__device__ inline wy_f32x4 wy_fma(wy_f32x4 a, float s, wy_f32x4 c) {
    return wy_f32x4{fmaf(a[0], s, c[0]), fmaf(a[1], s, c[1]), fmaf(a[2], s, c[2]), fmaf(a[3], s, c[3])};
}
static constexpr int kWyA[6] = {2, 0, 1, 1, 0, 0}, kWyB[6] = {0, 2, 1, 0, 1, 0};   // parts of the terms, smallest first
__device__ inline wy_f32x4 wy_mfma(u32x4 a, u32x4 b, wy_f32x4 acc) {   // 32 contracted values: the lane group's four of one 16, then of the next
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}
__device__ inline wy_f32x4 wy_mfma_first(u32x4 a, u32x4 b, wy_f32x4 acc) {   // the first 16 of them
    typedef short i16x4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, u32x2{a[0], a[1]}), __builtin_bit_cast(i16x4, u32x2{b[0], b[1]}), acc, 0, 0, 0);
}

// Per (block, value head) outputs, block-major then head, each cut into tiles that are stored the way the recurrence kernel's lanes
// read them, 1 KiB of 16 bytes per lane (a row-major matrix read as an A operand has neighbouring lanes 512 bytes apart, which the
// memory pipeline serves at a fraction of its rate).  A tile of W, q^ or K' is 16 rows by 32 contracted values and consists of three
// such pieces, the bf16 parts h, m and l; M and U stay f32, in tiles of 16 by 16:
//   Wt [token tile w][32 channels s], Qt likewise (in the slot of the first value head that shares q^), Kt [col tile c][32 tokens p]
//   (= diag(e^{L_C-L}) K transposed): lane (m, g) holds X[16 row-tile + m][32 col-tile + 4g + i] and [.. + 16 + 4g + i];
//   Mt [w][token tile tau]: lane (m, g) holds M[16w + m][16 tau + 4g + i];
//   Ut [w][col tile c]: lane (n, g) holds U[16w + 4g + i][16c + n]  (a D tile as computed);
//   eL [64] (e^{L_t}; eL[63] = e^{L_C} because padded tokens do not decay).
// Tokens past the end of the chunk are padded with beta = 0, log g = 0, k = q = v = 0.
//
// grid (Hv, blocks), one wave per 16 columns of K (DK/16 waves: two per SIMD at DK = 128, so that one
// has matrix work while the other waits for LDS or stores a tile).
// A workgroup's 31 k clocks (39 k on f32 instructions) are 9 k until its inputs are there, 3.6 k of norms and their splits, 5 k for the two
// triangles, 3 k for the diagonal blocks beside K', 3.5 k for the levels beside phase 3's operands, 1.4 k for T's parts and 4 to 6 k for W and U;
// 512 tokens of 32 heads 20.9 us on f32 instructions, 19.4.  It takes 245 registers and 120 KiB, a CU to a workgroup.
// Measured beside: q^ split by the wave that multiplies it, and the triangles' jobs by whole row tiles (20.2, the longest job 6.5 k clocks);
// q^ out as f32 and split by the recurrence (19.0, but 26.7 there).
// FUSED: the block's inputs come straight from the layer's inputs (WyInputs): what
// gdn_chunk_pre_kernel computes for the token-by-token form is done here per (block, value head) -
// conv + SiLU of the head's q, k and v channels, the per-token q/k norm, the decay's logarithm and
// beta - so the chunk needs no launch and no arrays for them.  A k-head's q and k are formed by
// each of the value heads that share it; q^ goes out once, each of them writing a part.
template <int DK, bool FUSED>
__global__ __launch_bounds__(DK * 4) void gdn_wy_kernel(
    int Hk, int Hv, int T, const float *__restrict__ qn, const float *__restrict__ kn,
    const float *__restrict__ vv, const float *__restrict__ lg, const float *__restrict__ bg,
    u32x4 *__restrict__ Wt, u32x4 *__restrict__ Qt, float *__restrict__ Ut, float *__restrict__ Mt,
    u32x4 *__restrict__ Kt, float *__restrict__ eLc, WyInputs in) {
    constexpr int DV = DK;
    constexpr int NK = DK / 16, NS = DK / 32;
    // row strides (4-byte units) chosen so that 16-byte row reads by 8 lanes hit all banks (LDK 4 to 52 past the parts: within 0.5 % of each other)
    constexpr int LDK = 3 * DK / 2 + 20, LDC = kC + 4;
    constexpr int NW = NK;        // waves; wave c owns columns 16c .. 16c+15 of U
    constexpr int NTHR = 64 * NW;
    // A row of k^ or q^ is f32 until it is normed and then its bf16 parts in its place (h of all channels, m, l; of each 32 channels in the
    // order of an operand's lanes), v stays in the registers of the wave that multiplies it.  T lies where q^ was, its parts behind it
    // and where k^ was.
    constexpr int TPARTS = 6 * 3 * 64 * 4;           // parts of T times a factor per token: [(token tile, 32-token step)][h|m|l][64] x 16 bytes
    constexpr int KROOM = kC * LDK > TPARTS ? kC * LDK : TPARTS;
    constexpr int QROOM = kC * LDK > kC * LDC + TPARTS ? kC * LDK : kC * LDC + TPARTS;
    __shared__ __align__(16) float sKroom[KROOM];    // k^, later T diag(beta e^L)
    __shared__ __align__(16) float sQroom[QROOM];    // q^, later T and T diag(beta)
    __shared__ __align__(16) float sA[10][16][20];   // tile (I, J <= I) at I (I + 1) / 2 + J
    float(*sK)[LDK] = reinterpret_cast<float(*)[LDK]>(&sKroom[0]);
    float(*sQ)[LDK] = reinterpret_cast<float(*)[LDK]>(&sQroom[0]);
    float(*sT)[LDC] = reinterpret_cast<float(*)[LDC]>(&sQroom[0]);
    u32x4(*sTu)[3][64] = reinterpret_cast<u32x4(*)[3][64]>(&sQroom[kC * LDC]);
    u32x4(*sTw)[3][64] = reinterpret_cast<u32x4(*)[3][64]>(&sKroom[0]);
    __shared__ __align__(16) float sL[kC], sB[kC], sCw[kC], sKd[kC];
    __shared__ __align__(16) int sR[kC];

    // heads along x: a head's blocks are produced on the XCD whose L2 the recurrence kernel
    // (heads along x as well) will read them through
    const int vh = wy_head_of(blockIdx.x, Hk, Hv), blk = blockIdx.y, heads = Hv / Hk, kh = vh / heads;
    const int t0 = blk * kC;
    const int nt = (T - t0 < kC) ? T - t0 : kC;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    const size_t slot = (size_t)blk * Hv + vh;

    // ---- phase 0: k^, q^ of the block, cumulative log decay, beta ---------------------
    // Everything the block reads is requested here, in the order of use (loads return in the
    // order of their requests): the gates, k^ and q^, and v, which waits in registers for phase 2.
    float lg_in = 0.f, bg_in = 0.f;
    float vreg[4][4];   // v of tokens 16 s + 4 g + i, channel 16 wave + m, phase 3's operand
    // Cumulative log decay (wave 0), restarted after every token whose decay is zero: where the
    // reference's exp() underflows (log g below log FLT_MIN; -inf when its softplus overflows,
    // linear_attn.rs:357-370) the token forgets everything before it, and no factor e^{L_i-L_j}
    // may be formed across it (-inf - -inf).  sR[t] is the last such token up to and
    // including t (-1: none); a pair (row, col) decays to exactly 0 when sR[row] > col.
    auto scan_gates = [&]() __attribute__((always_inline)) {
        const bool dead = lg_in < -87.3f;
        float l = dead ? 0.f : lg_in;
        bool seg = dead;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const float u = __shfl_up(l, d, 64);
            const int su = __shfl_up((int)seg, d, 64);
            if (lane >= d) {
                if (!seg) l += u;
                seg = seg || su;
            }
        }
        const unsigned long long kills = __ballot(dead) & ((2ull << lane) - 1ull);
        const int r = kills ? 63 - __builtin_clzll(kills) : -1;
        const float el = r >= 0 ? 0.f : expf(l);      // decay since the block's first token
        sL[lane] = l;
        sR[lane] = r;
        sB[lane] = bg_in;
        sCw[lane] = bg_in * el;
        eLc[slot * kC + lane] = el;
        sKd[lane] = __shfl(r, 63, 64) > lane ? 0.f : expf(__shfl(l, 63, 64) - l);  // e^{L_C - L_t}
    };
    // four channels c .. c + 3 of a row of k^ or q^ as their parts
    auto put4 = [&](float *row, int c, float4 y) __attribute__((always_inline)) {
        const WyFour x = wy_split4(y.x, y.y, y.z, y.w);
        uint32_t *r = reinterpret_cast<uint32_t *>(row) + 16 * (c >> 5) + 4 * ((c >> 2) & 3) + 2 * ((c >> 4) & 1);
#pragma unroll
        for (int part = 0; part < 3; part++) *reinterpret_cast<u32x2 *>(r + part * (DK / 2)) = x.p[part];
    };
    if constexpr (FUSED) {
        constexpr int NCONV = 2 * DK, TT = 16;               // q and k channels of the head; tokens per run
        constexpr int NU = NCONV * (kC / TT) / NTHR;          // (channel, run) units per thread
        static_assert(NCONV * (kC / TT) % NTHR == 0, "whole units per thread");
        const int C = 2 * Hk * DK + Hv * DV;
        float a_in = 0.f, b_in = 0.f, al_in = 0.f, dt_in = 0.f;
        if (wave == 0 && lane < nt) {
            a_in = in.alpha[(size_t)(t0 + lane) * Hv + vh];
            b_in = in.beta[(size_t)(t0 + lane) * Hv + vh];
            al_in = in.a_log[vh];
            dt_in = bf16_bits_to_f32(in.dt_bias[vh]);
        }
        // conv + SiLU (linear_attn.rs:132-154) of channel c over a run of 16 tokens per unit.
        // First every request of every unit: a run's TT + 3 inputs, oldest first, are rows of the
        // chunk, or ring slots for inputs from before it.  Every load is unconditional (the address
        // is selected; rows past the chunk's end re-read its last row and only feed outputs that
        // are zeroed below), so all of a thread's requests are in flight at once instead of one
        // memory round trip per input or per unit.
        // (Conv width 4 only; the launcher sends other widths through the separate first kernel.)
        float xs[NU][TT + 3];
        uint2 wbits[NU];
        const float *blk_rows = in.qkv + (size_t)t0 * C;   // the block's first row: offsets from here fit 32 bits
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const int unit = tid + u * NTHR, c = unit % NCONV, run = unit / NCONV;
            const int ch = c < DK ? kh * DK + c : Hk * DK + kh * DK + (c - DK);
            wbits[u] = *(const uint2 *)(in.conv_w + (unsigned)ch * 4u);
#pragma unroll
            for (int j = 0; j < TT + 3; j++) {
                const int rel = TT * run - 3 + j;          // row relative to the block's first
                const int idx = t0 + rel;
                const int last = T - 1 - t0;
                if (rel < 0) {                              // compile-time for all but the first run
                    const int off = (idx < 0 ? ((in.step_mod + idx + 4) & 3) : rel) * C + ch;
                    xs[u][j] = (idx < 0 ? in.ring : blk_rows)[off];
                } else {
                    xs[u][j] = blk_rows[(rel > last ? last : rel) * C + ch];
                }
            }
        }
        // v the same way, in runs of four tokens (seven inputs each)
        const int vch = 2 * Hk * DK + vh * DV + 16 * wave + m;
        const uint2 vw = *(const uint2 *)(in.conv_w + (unsigned)vch * 4u);
        float xv[4][7];
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < 7; j++) {
                const int rel = 16 * s + 4 * g + j - 3, idx = t0 + rel, last = T - 1 - t0;
                if (s == 0 && j < 3) {   // the block's first tokens look back before it
                    const int off = (idx < 0 ? ((in.step_mod + idx + 4) & 3) : rel > last ? last : rel) * C + vch;
                    xv[s][j] = (idx < 0 ? in.ring : blk_rows)[off];
                } else {
                    xv[s][j] = blk_rows[(rel > last ? last : rel) * C + vch];
                }
            }
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const int unit = tid + u * NTHR, c = unit % NCONV, run = unit / NCONV;
            const int tr = t0 + TT * run;
            int ntr = T - tr;
            ntr = ntr < 0 ? 0 : ntr > TT ? TT : ntr;
            const float wt[4] = {bf16_bits_to_f32((uint16_t)(wbits[u].x & 0xffffu)), bf16_bits_to_f32((uint16_t)(wbits[u].x >> 16)),
                                 bf16_bits_to_f32((uint16_t)(wbits[u].y & 0xffffu)), bf16_bits_to_f32((uint16_t)(wbits[u].y >> 16))};
            float(*dst)[LDK] = c < DK ? sQ : sK;
            const int cc = c < DK ? c : c - DK;
#pragma unroll
            for (int i = 0; i < TT; i++) {
                float acc = 0.f;
#pragma unroll
                for (int k = 0; k < 4; k++) acc = fmaf(xs[u][i + k], wt[k], acc);
                dst[TT * run + i][cc] = i < ntr ? silu_f(acc) : 0.f;
            }
        }
        {
            const float wt[4] = {bf16_bits_to_f32((uint16_t)(vw.x & 0xffffu)), bf16_bits_to_f32((uint16_t)(vw.x >> 16)),
                                 bf16_bits_to_f32((uint16_t)(vw.y & 0xffffu)), bf16_bits_to_f32((uint16_t)(vw.y >> 16))};
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float acc = 0.f;
#pragma unroll
                    for (int k = 0; k < 4; k++) acc = fmaf(xv[s][i + k], wt[k], acc);
                    vreg[s][i] = 16 * s + 4 * g + i < nt ? silu_f(acc) : 0.f;
                }
        }
        if (wave == 0 && lane < nt) {
            // shaders.metal:1321-1326; the decay enters as its logarithm
            const float a_cap = expf(al_in);
            const float sp = logf(1.0f + expf(a_in + dt_in));
            lg_in = -a_cap * sp;
            bg_in = 1.0f / (1.0f + expf(-b_in));
        }
        if (wave == 0) scan_gates();   // ahead of the barrier, which waves 4 .. 7 reach last
        __syncthreads();
        // per-token norm of q and k (infer.m:2655-2667: x * inv_rms, then q *= (1/sqrt(dk))^2,
        // k *= 1/sqrt(dk)): NTHR / (2 kC) lanes per (token, q|k) row, in place
        constexpr int LPP = NTHR / (2 * kC), EPL = DK / LPP;   // lanes per row, elements per lane
        static_assert(LPP == 2 || LPP == 4, "lanes per normed row");
        {
            const int p = tid / LPP, sub = tid % LPP, tt = p % kC;
            const bool is_q = p < kC;
            float *row = is_q ? sQ[tt] : sK[tt];
            float4 x[EPL / 4];
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < EPL / 4; i++) {
                x[i] = lds_f4(row + 4 * (LPP * i + sub));
                ss += x[i].x * x[i].x + x[i].y * x[i].y + x[i].z * x[i].z + x[i].w * x[i].w;
            }
            ss = dpp_add<0xB1>(ss);
            if (LPP == 4) ss = dpp_add<0x4E>(ss);
            const float inv_scale = 1.0f / sqrtf((float)DK);
            const float inv_rms = 1.0f / sqrtf(ss / (float)DK + 1e-6f);
            const float sc = is_q ? inv_scale * inv_scale : inv_scale;
            wave_lds_order();   // a row's lanes are one wave's: all have read it
#pragma unroll
            for (int i = 0; i < EPL / 4; i++) {
                float4 y = {x[i].x * inv_rms, x[i].y * inv_rms, x[i].z * inv_rms, x[i].w * inv_rms};
                y.x *= sc; y.y *= sc; y.z *= sc; y.w *= sc;
                put4(row, 4 * (LPP * i + sub), y);
            }
        }
    } else {
        if (wave == 0) {
            if (lane < nt) {
                lg_in = lg[(size_t)(t0 + lane) * Hv + vh];
                bg_in = bg[(size_t)(t0 + lane) * Hv + vh];
            }
            scan_gates();
        }
        constexpr int NL = kC * (DK / 4) / NTHR;
        float4 a[NL], b[NL];
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int i = tid + u * NTHR, tt = i / (DK / 4), x = (i % (DK / 4)) * 4;
            const size_t src = ((size_t)(t0 + (tt < nt ? tt : nt - 1)) * Hk + kh) * DK + x;
            a[u] = load_f4(kn + src);
            b[u] = load_f4(qn + src);
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int tt = 16 * s + 4 * g + i;
                vreg[s][i] = vv[((size_t)(t0 + (tt < nt ? tt : nt - 1)) * Hv + vh) * DV + 16 * wave + m];
                if (tt >= nt) vreg[s][i] = 0.f;
            }
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int i = tid + u * NTHR, tt = i / (DK / 4), x = (i % (DK / 4)) * 4;
            const float keep = tt < nt ? 1.f : 0.f;  // padded tokens are zero rows
            put4(sK[tt], x, float4{a[u].x * keep, a[u].y * keep, a[u].z * keep, a[u].w * keep});
            put4(sQ[tt], x, float4{b[u].x * keep, b[u].y * keep, b[u].z * keep, b[u].w * keep});
        }
    }
    __syncthreads();

    // Operands from the rows: eight channels of a row; four tokens (t .. t + 3, t = 16 tau + 4 g) of channel 16 c + m.
    auto row_of = [&](const float *row, int s) __attribute__((always_inline)) {
        WyEight r;
#pragma unroll
        for (int part = 0; part < 3; part++)
            r.p[part] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const uint32_t *>(row) + part * (DK / 2) + 16 * s + 4 * g);
        return r;
    };
    auto col_of = [&](int tau, int c) __attribute__((always_inline)) {
        typedef short i16x4 __attribute__((ext_vector_type(4)));
        const uint32_t *p = reinterpret_cast<const uint32_t *>(sK[16 * tau + 4 * g + (m >> 2)]) + 16 * (c >> 1) + 4 * (m & 3) + 2 * (c & 1);
        WyFour r;
#pragma unroll
        for (int part = 0; part < 3; part++)
            r.p[part] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (i16x4 __attribute__((address_space(3))) *)(__attribute__((address_space(3))) uint32_t *)(p + part * (DK / 2))));
        return r;
    };
    const wy_f32x4 zero = {0.f, 0.f, 0.f, 0.f};

    // ---- phase 1: the lower tiles of K K^T (-> A) and of Q K^T (-> M) -----------------
    // A job is two tiles of M, or three, of which M's (that take longer) is at most one.  Written
    // out per job, so that the reads of a tile's operands overlap the tile before it.
    auto gram = [&](auto kind_tag, auto I_tag, auto from_tag, auto to_tag) __attribute__((always_inline)) {
        constexpr int kind = decltype(kind_tag)::value, I = decltype(I_tag)::value, J0 = decltype(from_tag)::value, J1 = decltype(to_tag)::value;
        WyEight own[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) own[s] = row_of(kind ? sQ[16 * I + m] : sK[16 * I + m], s);
#pragma unroll
        for (int J = J0; J <= J1; J++) {
            WyEight other[NS];
#pragma unroll
            for (int s = 0; s < NS; s++) other[s] = row_of(sK[16 * J + m], s);
            wy_f32x4 term[6];
#pragma unroll
            for (int t = 0; t < 6; t++) term[t] = zero;
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int t = 0; t < 6; t++)
                    // K K^T: lane (n = m, g) gets rows 16I + 4g + i of column 16J + n.  Q K^T as the tile transposed (k^ as the A side):
                    // columns 16J + 4g + i of row 16I + n, which is this lane's part of tile (I, J) in A-operand order
                    term[t] = kind ? wy_mfma(other[s].p[kWyA[t]], own[s].p[kWyB[t]], term[t]) : wy_mfma(own[s].p[kWyA[t]], other[s].p[kWyB[t]], term[t]);
            const wy_f32x4 acc = ((term[0] + term[1]) + term[2]) + (term[3] + term[4]) + term[5];
            const int one = kind ? 16 * I + m : 16 * J + m, four = (kind ? 16 * J : 16 * I) + 4 * g;   // this lane's row (column), columns (rows)
            const float4 l4 = lds_f4(&sL[four]);
            const float lf[4] = {l4.x, l4.y, l4.z, l4.w}, l1 = sL[one];
            wy_f32x4 y;
            if constexpr (kind) {
                const int r1 = sR[one];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float d = r1 > four + i ? 0.f : __builtin_amdgcn_exp2f(fminf(l1 - lf[i], 0.f) * 1.4426950408889634f);  // v_exp_f32: 1 ulp
                    y[i] = (I > J || four + i <= one) ? d * acc[i] : 0.f;
                }
                *reinterpret_cast<wy_f32x4 *>(Mt + (((slot * 4 + I) * 4 + J) * 64 + lane) * 4) = y;
            } else {
                const float4 b4 = lds_f4(&sB[four]);
                const int4 r4 = *reinterpret_cast<const int4 *>(&sR[four]);
                const float bf[4] = {b4.x, b4.y, b4.z, b4.w};
                const int rf[4] = {r4.x, r4.y, r4.z, r4.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float d = rf[i] > one ? 0.f : __builtin_amdgcn_exp2f(fminf(lf[i] - l1, 0.f) * 1.4426950408889634f);
                    sA[I * (I + 1) / 2 + J][4 * g + i][m] = (I > J || one < four + i) ? bf[i] * d * acc[i] : 0.f;
                }
            }
        }
    };
#pragma unroll
    for (int r = 0; r < 8 / NW; r++) {
        const std::integral_constant<int, 0> c0{};
        const std::integral_constant<int, 1> c1{};
        const std::integral_constant<int, 2> c2{};
        const std::integral_constant<int, 3> c3{};
        switch (wave + NW * r) {   // uniform over the wave
            case 0: gram(c0, c0, c0, c0); gram(c0, c1, c0, c1); break;
            case 1: gram(c0, c2, c0, c2); break;
            case 2: gram(c0, c3, c0, c1); gram(c1, c0, c0, c0); break;
            case 3: gram(c0, c3, c2, c3); gram(c1, c2, c2, c2); break;
            case 4: gram(c1, c3, c0, c1); break;
            case 5: gram(c1, c3, c2, c3); break;
            case 6: gram(c1, c1, c0, c1); break;
            default: gram(c1, c2, c0, c1); break;
        }
    }
#pragma unroll
    for (int u = 0; u < 4 * NS / NW; u++) {  // q^ tiles, before T takes their place: once per k head, by its value heads in turn
        if (u % heads != vh % heads) continue;
        const int tile = wave + NW * u;
        const WyEight x = row_of(sQ[16 * (tile / NS) + m], tile % NS);
#pragma unroll
        for (int part = 0; part < 3; part++) Qt[(((slot - vh % heads) * 4 * NS + tile) * 3 + part) * 64 + lane] = x.p[part];
    }
    __syncthreads();

    // ---- phase 2: diag(e^{L_C - L}) K transposed goes out, and
    //      T = (I + A)^-1 by blocks of 16: the diagonal blocks by forward substitution (one
    //      per wave, a column per lane), the blocks below them level by level from
    //      T_IJ = -T_II sum_{J <= K < I} A_IK T_KJ on the matrix cores -----------------------
    if (NW == 4 || wave < 4) {
        // block `wave`; the four lane groups compute the same 16 columns, group 0 stores
        const int r0 = 16 * wave;
        float t[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            float acc = (i == m) ? 1.f : 0.f;
#pragma unroll
            for (int j4 = 0; j4 < i; j4 += 4) {
                const float4 a = lds_f4(&sA[wave * (wave + 1) / 2 + wave][i][j4]);  // the same address in every lane
                acc = fmaf(-a.x, t[j4], acc);
                if (j4 + 1 < i) acc = fmaf(-a.y, t[j4 + 1], acc);
                if (j4 + 2 < i) acc = fmaf(-a.z, t[j4 + 2], acc);
                if (j4 + 3 < i) acc = fmaf(-a.w, t[j4 + 3], acc);
            }
            t[i] = acc;
            if (g == 0) sT[r0 + i][r0 + m] = acc;
        }
    }
    // the waves without a diagonal block take the tiles of K' (all waves where each has one)
    if (NW == 4 || wave >= 4) {
#pragma unroll
        for (int u = 0; u < NK / 2; u++) {
            const int tile = (wave & 3) + 4 * u, c = tile >> 1, p = tile & 1;
            WyFour x[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float4 e = lds_f4(&sKd[32 * p + 16 * h + 4 * g]);
                const wy_f32x4 k = wy_whole(col_of(2 * p + h, c));
                x[h] = wy_split4(k[0] * e.x, k[1] * e.y, k[2] * e.z, k[3] * e.w);
            }
            const WyEight y = wy_join(x[0], x[1]);
#pragma unroll
            for (int part = 0; part < 3; part++) Kt[((slot * NK * 2 + tile) * 3 + part) * 64 + lane] = y.p[part];
        }
    }
    __syncthreads();
    // phase 3's operands, for all four token tiles: here, where most waves would wait for the levels.  V of the wave's 16 columns; K of
    // 32 columns, of which the wave forms W for two of the four token tiles: the first and the last, or those between
    static_assert(NW == 2 * NS, "two waves to 32 columns");
    const int wcol = wave % NS;
    WyEight vu[2], kw[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++) {
        vu[p] = wy_join(wy_split4(vreg[2 * p][0], vreg[2 * p][1], vreg[2 * p][2], vreg[2 * p][3]),
                        wy_split4(vreg[2 * p + 1][0], vreg[2 * p + 1][1], vreg[2 * p + 1][2], vreg[2 * p + 1][3]));
#pragma unroll
        for (int ct = 0; ct < 2; ct++) kw[ct][p] = wy_join(col_of(2 * p, 2 * wcol + ct), col_of(2 * p + 1, 2 * wcol + ct));
    }
#pragma unroll
    for (int lvl = 1; lvl < 4; lvl++) {
        if (wave < 4 - lvl) {  // block (I, J) = (wave + lvl, wave)
            const int I = wave + lvl, J = wave;
            wy_f32x4 x = zero;
            for (int K = J; K < I; K++) {
                float4 bt;
                bt.x = sT[16 * K + 4 * g + 0][16 * J + m];
                bt.y = sT[16 * K + 4 * g + 1][16 * J + m];
                bt.z = sT[16 * K + 4 * g + 2][16 * J + m];
                bt.w = sT[16 * K + 4 * g + 3][16 * J + m];
                x = mfma4(lds_f4(&sA[I * (I + 1) / 2 + K][m][4 * g]), bt, x);
            }
            // x is held as rows 4g+i of column m: already the B operand of T_II x
            wy_f32x4 r = zero;
            r = mfma4(lds_f4(&sT[16 * I + m][16 * I + 4 * g]), as_f4(x), r);
#pragma unroll
            for (int i = 0; i < 4; i++) sT[16 * I + 4 * g + i][16 * J + m] = -r[i];
        }
        __syncthreads();
    }
    // The parts of T diag(beta e^L) and T diag(beta), tile (tau, s <= tau) at tau (tau + 1) / 2 + s
#pragma unroll
    for (int u = 0; u < (10 + NW - 1) / NW; u++) {
        const int tile = wave + NW * u;
        if (tile < 10) {
            const int tau = tile >= 6 ? 3 : tile >= 3 ? 2 : tile >= 1 ? 1 : 0, s = tile - tau * (tau + 1) / 2;
            const int at = (tau < 2 ? tau : 2 * tau - 2) + (s >> 1);
            const float4 t = lds_f4(&sT[16 * tau + m][16 * s + 4 * g]);
            const float4 cw = lds_f4(&sCw[16 * s + 4 * g]), cb = lds_f4(&sB[16 * s + 4 * g]);
            const WyFour x = wy_split4(t.x * cw.x, t.y * cw.y, t.z * cw.z, t.w * cw.w);
            const WyFour y = wy_split4(t.x * cb.x, t.y * cb.y, t.z * cb.z, t.w * cb.w);
#pragma unroll
            for (int part = 0; part < 3; part++) {
                reinterpret_cast<u32x2 *>(&sTw[at][part][lane])[s & 1] = x.p[part];
                reinterpret_cast<u32x2 *>(&sTu[at][part][lane])[s & 1] = y.p[part];
            }
        }
    }
    __syncthreads();

    // ---- phase 3: W = T diag(beta e^L) K and U = T diag(beta) V -------------------------
    auto times_t = [&](auto first) __attribute__((always_inline)) {
        WyEight tu[2][2], tw[2][2];   // [token tile % 2][step]
        auto is_mine = [](int tau) { return (tau == 0 || tau == 3) == decltype(first)::value; };   // whether the wave forms W of these tokens
        auto read_t = [&](int tau) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p <= tau / 2; p++)
#pragma unroll
                for (int part = 0; part < 3; part++) {
                    const int at = tau < 2 ? tau : 2 * tau - 2 + p;
                    tu[tau % 2][p].p[part] = sTu[at][part][lane];
                    if (is_mine(tau)) tw[tau % 2][p].p[part] = sTw[at][part][lane];
                }
        };
        read_t(0);
#pragma unroll
        for (int tau = 0; tau < 4; tau++) {
            if (tau < 3) read_t(tau + 1);
            __builtin_amdgcn_sched_barrier(0);   // the next tile's reads ahead of this one's products
            const bool mine = is_mine(tau);
            wy_f32x4 au[2] = {zero, zero}, aw[2][2] = {{zero, zero}, {zero, zero}};
#pragma unroll
            for (int p = 0; p <= tau / 2; p++) {
                const bool half = 2 * p == tau;
                const WyEight &u8 = tu[tau % 2][p], &w8 = tw[tau % 2][p];
#pragma unroll
                for (int t = 0; t < 6; t++) {
                    const int x = (t & 1) * 3 + t / 2, a = kWyA[x], b = kWyB[x];   // the two sums in turn
                    wy_f32x4 &u = au[x >= 3];
                    u = half ? wy_mfma_first(u8.p[a], vu[p].p[b], u) : wy_mfma(u8.p[a], vu[p].p[b], u);
                    if (mine) {
                        // W transposed (K as the A side): lane (n = m, g) then holds columns 16c + 4g + i of
                        // token 16 tau + n, its part of the tile in A-operand order
#pragma unroll
                        for (int ct = 0; ct < 2; ct++) {
                            wy_f32x4 &w = aw[ct][x >= 3];
                            w = half ? wy_mfma_first(kw[ct][p].p[a], w8.p[b], w) : wy_mfma(kw[ct][p].p[a], w8.p[b], w);
                        }
                    }
                }
            }
            // U as computed (a D tile), W in A-operand order
            *reinterpret_cast<wy_f32x4 *>(Ut + ((slot * 4 + tau) * NK + wave) * 256 + lane * 4) = au[0] + au[1];
            if (mine) {
                const WyEight w = wy_join(wy_split4(aw[0][0] + aw[0][1]), wy_split4(aw[1][0] + aw[1][1]));
#pragma unroll
                for (int part = 0; part < 3; part++) Wt[(((slot * 4 + tau) * NS + wcol) * 3 + part) * 64 + lane] = w.p[part];
            }
        }
    };
    if (wave < NS) times_t(std::true_type{});
    else times_t(std::false_type{});
}

// grid (Hv, DV/32), 512 threads: 32 rows of one head's state, as two groups of 16.  Waves 0-3 are the chain that each block waits
// for: wave w forms D of tokens 16w .. 16w+15 from W, and owns columns 32w .. 32w+31 of the state, in f32, which it updates
// and hands to all waves as parts.  Waves 4-7 form O of the same tokens: q^ S0^T while the chain updates the state, M D while it
// forms the next block's D, so that LDS and matrix core are shared evenly.  (Lane (n, g) of a tile that the update leaves holds row n,
// columns 16c+4g+i: with c = 2w, 2w+1 its own eight values are the B operand of a 32-wide contraction over them, k-slot e < 4 being
// column 32w+4g+e, e >= 4 column 32w+16+4g+e-4; two tiles of D likewise tokens 32p+4g+i and 32p+16+4g+i of row n.)
// A block takes 6.0 k clocks, 5.0 k without its operand requests (timing only): a chain of two exchanges through LDS, 96 matrix and 250 vector
// instructions, and 160 KB of operands a CU.  512 tokens of 32 heads on half the CUs 23.8 us (f32 instructions, 16 rows a
// workgroup: 25.4 on all of them; q^ S0^T beside the next block's D, and requests after the last product: 25.2).
// A layer with this and the block precompute above against both on f32 instructions, with three sequences side by side / one call after
// the other: 512 tokens of 32 heads 40.0 / 54.5 -> 36.9 / 52.3 us, 1000 79.1 / 89.2 -> 73.4 / 89.6, 2000 156 / 159 -> 144 / 163,
// 512 of 64 heads 84.4 / 89.3 -> 73.7 / 78.7.  (f16 pairs: 31.2 / 47.1, 57.9 / 77.9, 114 / 138, 60.3 / 64.3.)
template <int DK>
__global__ __launch_bounds__(512, 2) void gdn_wy_recur_kernel(
    int Hk, int Hv, int T, const u32x4 *__restrict__ Wt, const u32x4 *__restrict__ Qt,
    const float *__restrict__ Ut, const float *__restrict__ Mt, const u32x4 *__restrict__ Kt,
    const float *__restrict__ eLc, float *__restrict__ ssm, float *__restrict__ o_raw) {
    constexpr int DV = DK;
    constexpr int NK = DK / 16;   // column tiles of the state
    constexpr int NS = DK / 32;   // 32-column steps of a contraction over them
    __shared__ u32x4 s_s[2][2][NS][3][64];   // state [block % 2][row group][step][h|m|l]
    __shared__ u32x4 s_d[2][2][2][3][64];    // D [block % 2][row group][32 tokens][h|m|l]

    const int vh = wy_head_of(blockIdx.x, Hk, Hv), row0 = blockIdx.y * 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, g = lane >> 4, w = wave & 3, lane16 = lane * 16;
    const int nblk = (T + kC - 1) / kC;
    // Requests go through a descriptor of the block's operand, so that they cost no vector addition.  Past the last block: that one again.
    auto slot_of = [&](int blk) { return (size_t)(blk < nblk ? blk : nblk - 1) * Hv + vh; };
    const int shared = vh % (Hv / Hk);   // q^ is its k head's, in the slot of the first of the value heads
    auto load = [&](__amdgpu_buffer_rsrc_t r, int tile) __attribute__((always_inline)) {
        return __builtin_amdgcn_raw_buffer_load_b128(r, lane16, tile * 1024, 0);
    };
    WyEight pw[NS];   // W, or q^, of tokens 16w .. 16w+15: a register takes the next block's request as soon as it has been used
    auto w_of = [&](const u32x4 *X, int back, int blk) { return buffer_of(X + ((slot_of(blk) - back) * 4 + w) * NS * 3 * 64); };
    auto fetch_w = [&](__amdgpu_buffer_rsrc_t r, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int part = 0; part < 3; part++) pw[s].p[part] = load(r, 3 * s + part);
    };
    auto fetch_all_w = [&](const u32x4 *X, int back) __attribute__((always_inline)) {
        const auto r = w_of(X, back, 0);
#pragma unroll
        for (int s = 0; s < NS; s++) fetch_w(r, s);
    };
    // X S0^T of this wave's 16 tokens, X = W or q^ (which lies `back` slots ahead of the head's own), both row groups
    auto times_state = [&](const u32x4 *X, int back, int blk, wy_f32x4 (&p)[2]) __attribute__((always_inline)) {
        // All LDS reads first, and four sums in turn, so that no instruction waits for the one
        // before it (left alone the compiler reads each operand just ahead of its product).
        WyEight st[NS][2];
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int rg = 0; rg < 2; rg++)
#pragma unroll
                for (int part = 0; part < 3; part++) st[s][rg].p[part] = s_s[blk & 1][rg][s][part][lane];
        __builtin_amdgcn_sched_barrier(0);
        const wy_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        wy_f32x4 acc[2][2] = {{zero, zero}, {zero, zero}};
        const auto r = w_of(X, back, blk + 1);
#pragma unroll
        for (int s = 0; s < NS; s += 2) {
#pragma unroll
            for (int t = 0; t < 6; t++)
#pragma unroll
                for (int x = 0; x < 2; x++)
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) acc[x][rg] = wy_mfma(pw[s + x].p[kWyA[t]], st[s + x][rg].p[kWyB[t]], acc[x][rg]);
            __builtin_amdgcn_sched_barrier(0);
            fetch_w(r, s);
            fetch_w(r, s + 1);
        }
#pragma unroll
        for (int rg = 0; rg < 2; rg++) p[rg] = acc[0][rg] + acc[1][rg];
    };

    if (wave < 4) {
        // ================= the chain: D, and the state =================
        __builtin_amdgcn_s_setprio(1);   // the other waves' work is wanted a block later
        const bool owner = w < NS;       // of columns 32w .. 32w+31 of the state
        float *srow = ssm + ((size_t)vh * DV + row0 + m) * DK + 32 * (owner ? w : 0) + 4 * g;
        wy_f32x4 st[2][2];               // [row group][column tile]
#pragma unroll
        for (int rg = 0; rg < 2; rg++)
#pragma unroll
            for (int ct = 0; ct < 2; ct++) st[rg][ct] = load_v4(srow + 16 * rg * DK + 16 * ct);
        auto publish_state = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int rg = 0; rg < 2; rg++) {
                const WyEight x = wy_join(wy_split4(st[rg][0]), wy_split4(st[rg][1]));
#pragma unroll
                for (int part = 0; part < 3; part++) s_s[buf][rg][w][part][lane] = x.p[part];
            }
        };
        WyEight kd[2][2];   // [column tile][32 tokens]
        wy_f32x4 pu[2];
        float elc;
        auto u_of = [&](int blk) { return buffer_of(Ut + ((slot_of(blk) * 4 + w) * NK + 2 * blockIdx.y) * 256); };
        auto k_of = [&](int blk) { return buffer_of(Kt + (slot_of(blk) * NK + 2 * (owner ? w : 0)) * 2 * 3 * 64); };
        auto fetch_elc = [&](int blk) __attribute__((always_inline)) {
            elc = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buffer_of(eLc + slot_of(blk) * kC + kC - 1), 0, 0, 0));
        };
        auto fetch_k = [&](__amdgpu_buffer_rsrc_t r, int p) __attribute__((always_inline)) {
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int part = 0; part < 3; part++) kd[ct][p].p[part] = load(r, (2 * ct + p) * 3 + part);
        };
        fetch_all_w(Wt, 0);
        {
            const auto ru = u_of(0), rk = k_of(0);
#pragma unroll
            for (int rg = 0; rg < 2; rg++) pu[rg] = __builtin_bit_cast(wy_f32x4, load(ru, rg));
            fetch_elc(0);
            fetch_k(rk, 0);
            fetch_k(rk, 1);
        }
        if (owner) publish_state(0);
        __syncthreads();
        for (int blk = 0; blk < nblk; blk++) {
            // ---- D = U - W S0^T: lane (n, g) holds tokens 16w+4g+i of state row n of the group ----
            wy_f32x4 p[2];
            times_state(Wt, 0, blk, p);
            const wy_f32x4 d[2] = {pu[0] - p[0], pu[1] - p[1]};
            const auto ru = u_of(blk + 1);
#pragma unroll
            for (int rg = 0; rg < 2; rg++) pu[rg] = __builtin_bit_cast(wy_f32x4, load(ru, rg));
#pragma unroll
            for (int rg = 0; rg < 2; rg++) {
                const WyFour x = wy_split4(d[rg]);
#pragma unroll
                for (int part = 0; part < 3; part++) reinterpret_cast<u32x2 *>(&s_d[blk & 1][rg][w >> 1][part][lane])[w & 1] = x.p[part];
            }
            __syncthreads();
            // ---- S' = e^{L_C} S0 + D^T diag(e^{L_C-L}) K, this wave's columns ------
            if (owner) {
const auto rk = k_of(blk + 1);
                WyEight dd[2][2];
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int rg = 0; rg < 2; rg++)
#pragma unroll
                        for (int part = 0; part < 3; part++) dd[p][rg].p[part] = s_d[blk & 1][rg][p][part][lane];
                __builtin_amdgcn_sched_barrier(0);
                const wy_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                wy_f32x4 acc[2][2] = {{zero, zero}, {zero, zero}};
#pragma unroll
                for (int p = 0; p < 2; p++) {
#pragma unroll
                    for (int t = 0; t < 6; t++)
#pragma unroll
                        for (int rg = 0; rg < 2; rg++)
#pragma unroll
                            for (int ct = 0; ct < 2; ct++) acc[rg][ct] = wy_mfma(kd[ct][p].p[kWyA[t]], dd[p][rg].p[kWyB[t]], acc[rg][ct]);
                    fetch_k(rk, p);
                }
#pragma unroll
                for (int rg = 0; rg < 2; rg++)
#pragma unroll
                    for (int ct = 0; ct < 2; ct++) st[rg][ct] = wy_fma(st[rg][ct], elc, acc[rg][ct]);
                fetch_elc(blk + 1);
                publish_state((blk + 1) & 1);
            }
            __syncthreads();
        }
        if (owner) {
#pragma unroll
            for (int rg = 0; rg < 2; rg++)
#pragma unroll
                for (int ct = 0; ct < 2; ct++) *reinterpret_cast<wy_f32x4 *>(srow + 16 * rg * DK + 16 * ct) = st[rg][ct];
        }
    } else {
        // ================= O = diag(e^L) q^ S0^T + M D, a block behind =================
        // M comes as f32 and is split here: these waves wait for the chain's D
        wy_f32x4 rm[4], el;
        auto fetch_m = [&](int blk) __attribute__((always_inline)) {
            const auto r = buffer_of(Mt + (slot_of(blk) * 4 + w) * 4 * 256);
#pragma unroll
            for (int tau = 0; tau < 4; tau++) rm[tau] = __builtin_bit_cast(wy_f32x4, load(r, tau <= w ? tau : w));   // (past the diagonal there is nothing)
        };
        auto fetch_el = [&](int blk) __attribute__((always_inline)) {
            el = __builtin_bit_cast(wy_f32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer_of(eLc + slot_of(blk) * kC + 16 * w), g * 16, 0, 0));
        };
        const int stride = Hv * DV;
        fetch_all_w(Qt, shared);
        fetch_el(0);
        fetch_m(0);
        __syncthreads();
        __syncthreads();
        for (int blk = 0; blk < nblk; blk++) {
            // beside the update of this block's state
            wy_f32x4 o[2];
            times_state(Qt, shared, blk, o);
            o[0] *= el;
            o[1] *= el;
            fetch_el(blk + 1);
            __syncthreads();
            // beside the next block's D
WyEight dd[2][2];
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int rg = 0; rg < 2; rg++)
#pragma unroll
                    for (int part = 0; part < 3; part++) dd[p][rg].p[part] = s_d[blk & 1][rg][p][part][lane];
            __builtin_amdgcn_sched_barrier(0);
            const wy_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            wy_f32x4 acc[2][2] = {{zero, zero}, {zero, zero}};
            auto add = [&](int p, auto half) __attribute__((always_inline)) {
                const WyEight mt = wy_join(wy_split4(rm[2 * p]), decltype(half)::value ? WyFour{} : wy_split4(rm[2 * p + 1]));
#pragma unroll
                for (int t = 0; t < 6; t++)
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) {
                        const int x = (t & 1) * 3 + t / 2;   // the two sums in turn
                        const u32x4 a = mt.p[kWyA[x]], b = dd[p][rg].p[kWyB[x]];
                        acc[t & 1][rg] = decltype(half)::value ? wy_mfma_first(a, b, acc[t & 1][rg]) : wy_mfma(a, b, acc[t & 1][rg]);
                    }
            };
#pragma unroll
            for (int p = 0; p < 2; p++) {
                if (2 * p < w) add(p, std::false_type{});
                else if (2 * p == w) add(p, std::true_type{});
            }
#pragma unroll
            for (int rg = 0; rg < 2; rg++) o[rg] += acc[0][rg] + acc[1][rg];
            fetch_m(blk + 1);
            const int left = T - (blk * kC + 16 * w) - 4 * g;   // tokens from this lane's first on
            float *dst = o_raw + ((size_t)(blk * kC + 16 * w) * Hv + vh) * DV + row0;
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i < left) {
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) dst[(4 * g + i) * stride + m + 16 * rg] = o[rg][i];
                }
            if (blk + 1 < nblk) __syncthreads();   // this block's D may be written over
        }
    }
}

size_t gdn_wy_scratch_elems(int Hv, int dk, int dv, int T) {
    const size_t nblk = ((size_t)T + kC - 1) / kC;
    return nblk * Hv * (9 * (size_t)kC * dk / 2 + (size_t)kC * dv + (size_t)kC * kC + kC);
}

// o_raw [T, Hv*dv].  The blocks' inputs come from the layer's inputs (`in`; qn .. bg are then unused
// and may be null) or, when in is null, from qn, kn [T, Hk, dk]; vv [T, Hv, dv]; lg, bg [T, Hv] (log
// decay, beta gate) as gdn_chunk_pre_kernel leaves them.
int launch_gdn_wy(hipStream_t s, int Hk, int Hv, int dk, int dv, int T, const float *qn, const float *kn,
                  const float *vv, const float *lg, const float *bg, float *scratch, float *ssm,
                  float *o_raw, const WyInputs *in) {
    if (dk != dv || (dk != 64 && dk != 128))
        return fail(MFA_ERR_SHAPE, "gdn blocked form: dk=%d dv=%d not supported", dk, dv);
    const size_t nblk = ((size_t)T + kC - 1) / kC;
    if (nblk > 65535) return fail(MFA_ERR_SHAPE, "gdn blocked form: too many tokens in one call");
    const size_t slots = nblk * Hv;
    // (the parts of W, q^ and K' take six bytes a value)
    u32x4 *Wt = reinterpret_cast<u32x4 *>(scratch);
    u32x4 *Qt = Wt + slots * kC * dk * 3 / 8;
    u32x4 *Kt = Qt + slots * kC * dk * 3 / 8;
    float *Ut = reinterpret_cast<float *>(Kt + slots * kC * dk * 3 / 8);
    float *Mt = Ut + slots * kC * dv;
    float *eLc = Mt + slots * kC * kC;
    const WyInputs none{};
#define MFA_WY(DKK, FU)                                                                                             \
    hipLaunchKernelGGL((gdn_wy_kernel<DKK, FU>), dim3(Hv, (unsigned)nblk), dim3(DKK * 4), 0, s, Hk, Hv, T, qn, kn, vv, \
                       lg, bg, Wt, Qt, Ut, Mt, Kt, eLc, in ? *in : none)
    if (dk == 128) {
        if (in) MFA_WY(128, true); else MFA_WY(128, false);
        hipLaunchKernelGGL((gdn_wy_recur_kernel<128>), dim3(Hv, dv / 32), dim3(512), 0, s, Hk, Hv, T, Wt, Qt, Ut,
                           Mt, Kt, eLc, ssm, o_raw);
    } else {
        if (in) MFA_WY(64, true); else MFA_WY(64, false);
        hipLaunchKernelGGL((gdn_wy_recur_kernel<64>), dim3(Hv, dv / 32), dim3(512), 0, s, Hk, Hv, T, Wt, Qt, Ut,
                           Mt, Kt, eLc, ssm, o_raw);
    }
#undef MFA_WY
    MFA_HIP(hipGetLastError());
    return MFA_OK;
}

}  // namespace mfa
