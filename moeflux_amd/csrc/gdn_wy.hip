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
// independent).  The products are v_mfma_f32_16x16x32_f16 over operands split into two f16 numbers (see wy_split4), the
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

// f32 x scaled by a power of two as the sum of two f16 numbers, hi = f16(x), lo = f16(x - hi): 22 bits, what is left out is below
// 2^-24 of x (2^-39 of the scale for x below 2^-16 of it, where lo is subnormal), the size of x's own rounding.
// Of a product hi hi + hi lo + lo hi is formed (lo lo too where it costs nothing) and summed in f32, as the f32 instruction does,
// in 16 clocks for 32 contracted values and term instead of 256.  W, q^, the decayed k^ and M are at most 1 by construction
// (unit keys, beta <= 1, decays <= 1, and every row of W is beta e^L k^ under a chain of contractions), so they carry a fixed
// scale; the state's and D's scales are those of the largest value of a tile's row, taken as the tile is formed.
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;   // (LDS holding f32 and f16 parts in turn is read and written as vectors, which alias anything)
static constexpr float kWyScale = 16384.f;   // 2^14: the largest f16 is 65504
// Four values times scale as 16 bytes: hi of all, lo of all.  v_fma_mix*_f16 multiplies, subtracts hi where there is one, and
// rounds, in one instruction per value and part (multiply, convert, convert back, subtract, convert are four).
// The compiler does not see into the assembly: a result that went to the upper half of its register may be read one wait state
// later at the earliest, which the order of the eight and the last no-op keep; and no result of a matrix instruction may come in
// directly (its wait states are the compiler's to place), which callers see to with an instruction in between.
__device__ inline u32x4 wy_split4(float a, float b, float c, float d, float scale) {
    uint32_t h0, h1, l0, l1;
    asm("v_fma_mixlo_f16 %0, %4, %8, 0\n\t"
        "v_fma_mixlo_f16 %1, %6, %8, 0\n\t"
        "v_fma_mixhi_f16 %0, %5, %8, 0\n\t"
        "v_fma_mixhi_f16 %1, %7, %8, 0\n\t"
        "v_fma_mixlo_f16 %2, %4, %8, -%0 op_sel:[0,0,0] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %3, %6, %8, -%1 op_sel:[0,0,0] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %2, %5, %8, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %3, %7, %8, -%1 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "s_nop 0"
        : "=&v"(h0), "=&v"(h1), "=&v"(l0), "=&v"(l1) : "v"(a), "v"(b), "v"(c), "v"(d), "v"(scale));
    return u32x4{h0, h1, l0, l1};
}
__device__ inline u32x4 wy_split4_unit(float a, float b, float c, float d) { return wy_split4(a, b, c, d, kWyScale); }   // of values of at most 1
__device__ inline wy_f32x4 wy_fma(wy_f32x4 a, float s, wy_f32x4 c) {
    return wy_f32x4{fmaf(a[0], s, c[0]), fmaf(a[1], s, c[1]), fmaf(a[2], s, c[2]), fmaf(a[3], s, c[3])};
}
// The scale of values of at most mx (2^14 <= mx scale < 2^15, less for mx below 2^-87) and what undoes it together with kWyScale.
__device__ inline void wy_scale(float mx, float &scale, float &undo) {
    const int e = max((int)(__builtin_bit_cast(uint32_t, mx) >> 23), 40);   // mx >= 0
    scale = __builtin_bit_cast(float, (uint32_t)(268 - e) << 23);
    undo = __builtin_bit_cast(float, (uint32_t)(e - 28) << 23);
}
__device__ inline wy_f32x4 wy_mfma(u32x4 a, u32x4 b, wy_f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
}

// Per (block, value head) outputs, block-major then head, each cut into 16x16 tiles that
// are stored the way the recurrence kernel's lanes read them, 16 bytes per lane (four f32 values of Ut, the two f16 parts of
// four values of the others) and 1 KiB per tile (a row-major matrix read as an A operand has neighbouring lanes 512
// bytes apart, which the memory pipeline serves at a fraction of its rate):
//   Wt [token tile w][col tile c], Qt likewise (in the slot of the first value head that shares q^), Mt [w][token tile tau], Kt [col tile c][tau]
//   (= diag(e^{L_C-L}) K transposed): lane (m, g) holds X[16 row-tile + m][16 col-tile + 4g + i];
//   Ut [w][col tile c]: lane (n, g) holds U[16w + 4g + i][16c + n]  (a D tile as computed);
//   eL [64] (e^{L_t}; eL[63] = e^{L_C} because padded tokens do not decay).
// Tokens past the end of the chunk are padded with beta = 0, log g = 0, k = q = v = 0.
//
// grid (Hv, blocks), one wave per 16 columns of K (DK/16 waves: two per SIMD at DK = 128, so that one
// has matrix work while the other waits for LDS or stores a tile).
// A workgroup's 28 k clocks (39 k on f32 instructions) are 9 k until its inputs are there, 3 k of norms, 3.5 k for the two
// triangles, 2.3 k for the diagonal blocks beside K', 4.7 k for the levels beside phase 3's operands, 4 k for W and U: 512 tokens of 32
// heads 21.5 -> 15.8 us.  At 128 registers, so that a CU holds two (it takes 144 and holds one), it spills: no faster at 2000
// tokens with three sequences side by side (120.5 us a pass either way), 2 us slower at 512.
// FUSED: the block's inputs come straight from the layer's inputs (WyInputs): what
// gdn_chunk_pre_kernel computes for the token-by-token form is done here per (block, value head) -
// conv + SiLU of the head's q, k and v channels, the per-token q/k norm, the decay's logarithm and
// beta - so the chunk needs no launch and no arrays for them.  A k-head's q and k are formed by
// each of the value heads that share it; q^ goes out once, each of them writing a part (a layer's 512 tokens with three sequences side by
// side: 2 value heads a k head 31.7 -> 31.3 us, 4 64.2 -> 59.9; 2000 tokens of 2 117.4 -> 114.4).
template <int DK, bool FUSED>
__global__ __launch_bounds__(DK * 4) void gdn_wy_kernel(
    int Hk, int Hv, int T, const float *__restrict__ qn, const float *__restrict__ kn,
    const float *__restrict__ vv, const float *__restrict__ lg, const float *__restrict__ bg,
    u32x4 *__restrict__ Wt, u32x4 *__restrict__ Qt, float *__restrict__ Ut, u32x4 *__restrict__ Mt,
    u32x4 *__restrict__ Kt, float *__restrict__ eLc, WyInputs in) {
    constexpr int DV = DK;
    constexpr int NK = DK / 16, NS = DK / 32;
    constexpr int LDK = DK + 4;  // row strides (4-byte units) chosen so that 16-byte row reads by 8 lanes hit all banks
    constexpr int LDC = kC + 4;
    constexpr int NW = NK;        // waves; wave c owns columns 16c .. 16c+15 of W and of U
    constexpr int NTHR = 64 * NW;
    // A row of k^ or q^ is f32 until it is normed and then the f16 parts in its place (hi of all channels, then lo of all), v stays
    // in the registers of the wave that multiplies it, T and its f16 parts lie where q^ and A were.
    __shared__ __align__(16) float sK[kC][LDK];
    constexpr int TPARTS = 6 * 2 * 64 * 4;           // f16 parts of T times a factor per token: [(token tile, 32-token step)][hi|lo][64] x 16 bytes
    constexpr int QROOM = kC * LDK > kC * LDC + TPARTS ? kC * LDK : kC * LDC + TPARTS;
    __shared__ __align__(16) float sQroom[QROOM];    // q^, later T and T diag(beta)
    __shared__ __align__(16) float sA[10][16][20];   // tile (I, J <= I) at I (I + 1) / 2 + J; later T diag(beta e^L)
    float(*sQ)[LDK] = reinterpret_cast<float(*)[LDK]>(&sQroom[0]);
    float(*sT)[LDC] = reinterpret_cast<float(*)[LDC]>(&sQroom[0]);
    u32x4(*sTu)[2][64] = reinterpret_cast<u32x4(*)[2][64]>(&sQroom[kC * LDC]);
    u32x4(*sTw)[2][64] = reinterpret_cast<u32x4(*)[2][64]>(&sA[0][0][0]);
    static_assert(TPARTS * sizeof(float) <= sizeof(sA), "T's parts fit where A was");
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
    // a row of k^ or q^ as its f16 parts: channels c .. c + 3, y scale (at most 1)
    auto put4 = [&](float *row, int c, float4 y, float scale) __attribute__((always_inline)) {
        const u32x4 x = wy_split4(y.x, y.y, y.z, y.w, scale * kWyScale);
        uint32_t *r = reinterpret_cast<uint32_t *>(row);
        *reinterpret_cast<u32x2 *>(r + c / 2) = u32x2{x[0], x[1]};
        *reinterpret_cast<u32x2 *>(r + DK / 2 + c / 2) = u32x2{x[2], x[3]};
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
            float *row = (is_q ? sQ[tt] : sK[tt]) + EPL * sub;
            float4 x[EPL / 4];
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < EPL / 4; i++) {
                x[i] = lds_f4(row + 4 * i);
                ss += x[i].x * x[i].x + x[i].y * x[i].y + x[i].z * x[i].z + x[i].w * x[i].w;
            }
            ss = dpp_add<0xB1>(ss);
            if (LPP == 4) ss = dpp_add<0x4E>(ss);
            const float inv_scale = 1.0f / sqrtf((float)DK);
            const float inv_rms = 1.0f / sqrtf(ss / (float)DK + 1e-6f);
            const float sc = inv_rms * (is_q ? inv_scale * inv_scale : inv_scale);
#pragma unroll
            for (int i = 0; i < EPL / 4; i++) put4(is_q ? sQ[tt] : sK[tt], EPL * sub + 4 * i, x[i], sc);   // (a row's lanes are one wave's: all have read it)
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
            put4(sK[tt], x, float4{a[u].x * keep, a[u].y * keep, a[u].z * keep, a[u].w * keep}, 1.f);
            put4(sQ[tt], x, float4{b[u].x * keep, b[u].y * keep, b[u].z * keep, b[u].w * keep}, 1.f);
        }
    }
    __syncthreads();

    // Operands from the rows: eight channels of a row; four tokens (t .. t + 3, t = 16 tau + 4 g) of channel 16 c + m.
    auto row_part = [&](const float *row, int s, int part) __attribute__((always_inline)) {
        return *reinterpret_cast<const u32x4 *>(reinterpret_cast<const uint32_t *>(row) + part * (DK / 2) + 16 * s + 4 * g);
    };
    auto col_part = [&](int tau, int c, int part) __attribute__((always_inline)) {
        typedef short i16x4 __attribute__((ext_vector_type(4)));
        const uint32_t *p = reinterpret_cast<const uint32_t *>(sK[16 * tau + 4 * g + (m >> 2)]) + part * (DK / 2) + 8 * c + 2 * (m & 3);
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (i16x4 __attribute__((address_space(3))) *)(__attribute__((address_space(3))) uint32_t *)p));
    };
    const wy_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    constexpr float kUnscale2 = 1.f / (kWyScale * kWyScale);

    // ---- phase 1: the lower tiles of K K^T (-> A) and of Q K^T (-> M) -----------------
    // A job is a row tile I of one of the two and its tiles J <= I; the jobs of a SIMD's two waves add up to five tiles.  Written
    // out per job, so that the reads of a tile's operands overlap the tile before it.
    auto gram = [&](auto kind_tag, auto I_tag) __attribute__((always_inline)) {
        constexpr int kind = decltype(kind_tag)::value, I = decltype(I_tag)::value;
        u32x4 ih[NS], il[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const float *row = kind ? sQ[16 * I + m] : sK[16 * I + m];
            ih[s] = row_part(row, s, 0);
            il[s] = row_part(row, s, 1);
        }
#pragma unroll
        for (int J = 0; J <= I; J++) {
            u32x4 jh[NS], jl[NS];
#pragma unroll
            for (int s = 0; s < NS; s++) jh[s] = row_part(sK[16 * J + m], s, 0), jl[s] = row_part(sK[16 * J + m], s, 1);
            wy_f32x4 lh = zero, hl = zero, hh = zero;
#pragma unroll
            for (int s = 0; s < NS; s++) {
                // K K^T: lane (n = m, g) gets rows 16I + 4g + i of column 16J + n.  Q K^T as the tile transposed (k^ as the A side):
                // columns 16J + 4g + i of row 16I + n, which is this lane's 16 bytes of tile (I, J) in A-operand order
                lh = kind ? wy_mfma(jl[s], ih[s], lh) : wy_mfma(il[s], jh[s], lh);
                hl = kind ? wy_mfma(jh[s], il[s], hl) : wy_mfma(ih[s], jl[s], hl);
                hh = kind ? wy_mfma(jh[s], ih[s], hh) : wy_mfma(ih[s], jh[s], hh);
            }
            const wy_f32x4 acc = ((lh + hl) + hh) * kUnscale2;
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
                Mt[((slot * 4 + I) * 4 + J) * 64 + lane] = wy_split4_unit(y[0], y[1], y[2], y[3]);
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
        using std::integral_constant;
        switch (wave + NW * r) {   // uniform over the wave
            case 0: gram(integral_constant<int, 0>{}, integral_constant<int, 0>{}); break;
            case 1: gram(integral_constant<int, 0>{}, integral_constant<int, 1>{}); break;
            case 2: gram(integral_constant<int, 0>{}, integral_constant<int, 2>{}); break;
            case 3: gram(integral_constant<int, 0>{}, integral_constant<int, 3>{}); break;
            case 4: gram(integral_constant<int, 1>{}, integral_constant<int, 3>{}); break;
            case 5: gram(integral_constant<int, 1>{}, integral_constant<int, 2>{}); break;
            case 6: gram(integral_constant<int, 1>{}, integral_constant<int, 1>{}); break;
            default: gram(integral_constant<int, 1>{}, integral_constant<int, 0>{}); break;
        }
    }
#pragma unroll
    for (int u = 0; u < 4 * NK / NW; u++) {  // q^ tiles, before T takes their place: once per k head, by its value heads in turn
        if (u % heads != vh % heads) continue;
        const int tile = wave + NW * u, w = tile / NK, c = tile % NK;
        const uint32_t *row = reinterpret_cast<const uint32_t *>(sQ[16 * w + m]) + 8 * c + 2 * g;
        const u32x2 hi = *reinterpret_cast<const u32x2 *>(row), lo = *reinterpret_cast<const u32x2 *>(row + DK / 2);
        Qt[((slot - vh % heads) * 4 * NK + tile) * 64 + lane] = u32x4{hi[0], hi[1], lo[0], lo[1]};
    }
    __syncthreads();

    // ---- phase 2: diag(e^{L_C - L}) K transposed goes out, and
    //      T = (I + A)^-1 by blocks of 16: the diagonal blocks by forward substitution (one
    //      per wave, a column per lane), the blocks below them level by level from
    //      T_IJ = -T_II sum_{J <= K < I} A_IK T_KJ on the matrix cores -----------------------
    // k^ of four tokens from its parts (exact), times kWyScale
    auto whole = [&](u32x2 hi, u32x2 lo) __attribute__((always_inline)) {
        const f16x2 h0 = __builtin_bit_cast(f16x2, (uint32_t)hi[0]), h1 = __builtin_bit_cast(f16x2, (uint32_t)hi[1]), l0 = __builtin_bit_cast(f16x2, (uint32_t)lo[0]), l1 = __builtin_bit_cast(f16x2, (uint32_t)lo[1]);
        return float4{(float)h0[0] + (float)l0[0], (float)h0[1] + (float)l0[1], (float)h1[0] + (float)l1[0], (float)h1[1] + (float)l1[1]};
    };
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
        for (int u = 0; u < NK; u++) {
            const int tile = (wave & 3) + 4 * u, c = tile >> 2, tau = tile & 3;
            const float4 e = lds_f4(&sKd[16 * tau + 4 * g]);
            const float4 k = whole(col_part(tau, c, 0), col_part(tau, c, 1));
            Kt[(slot * NK * 4 + tile) * 64 + lane] = wy_split4(k.x * e.x, k.y * e.y, k.z * e.z, k.w * e.w, 1.f);
        }
    }
    __syncthreads();
    // phase 3's K and V operands of the wave's columns, for all four token tiles: here, where most waves would wait for the levels
    u32x4 kwh[2], kwl[2], vuh[2], vul[2];
    float v_undo;
    {
        float mx = 0.f, sc;
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 4; i++) mx = fmaxf(mx, fabsf(vreg[s][i]));
        wy_scale(rows_max(mx), sc, v_undo);
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const u32x2 h0 = col_part(2 * p, wave, 0), h1 = col_part(2 * p + 1, wave, 0), l0 = col_part(2 * p, wave, 1), l1 = col_part(2 * p + 1, wave, 1);
            kwh[p] = u32x4{h0[0], h0[1], h1[0], h1[1]};
            kwl[p] = u32x4{l0[0], l0[1], l1[0], l1[1]};
            const u32x4 y0 = wy_split4(vreg[2 * p][0], vreg[2 * p][1], vreg[2 * p][2], vreg[2 * p][3], sc);
            const u32x4 y1 = wy_split4(vreg[2 * p + 1][0], vreg[2 * p + 1][1], vreg[2 * p + 1][2], vreg[2 * p + 1][3], sc);
            vuh[p] = u32x4{y0[0], y0[1], y1[0], y1[1]};
            vul[p] = u32x4{y0[2], y0[3], y1[2], y1[3]};
        }
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
    // The f16 parts of T diag(beta e^L) and T diag(beta) (T is at most 1: its column j is what an impulse at token j leaves of itself in
    // later ones); step p of token tile tau holds tokens 32p .. 32p+31, zeros above the diagonal
#pragma unroll
    for (int u = 0; u < 12 / NW + (12 % NW != 0); u++) {
        const int half = wave + NW * u;   // (tau, token tile): (0,0) (0,1) (1,0) (1,1) (2,0) .. (3,3)
        if (half < 12) {
            const int tau = half < 4 ? half >> 1 : 2 + ((half - 4) >> 2), s = half < 4 ? half & 1 : (half - 4) & 3;
            const float4 t = s <= tau ? lds_f4(&sT[16 * tau + m][16 * s + 4 * g]) : float4{0.f, 0.f, 0.f, 0.f};
            const float4 cw = lds_f4(&sCw[16 * s + 4 * g]), cb = lds_f4(&sB[16 * s + 4 * g]);
            const u32x4 x = wy_split4_unit(t.x * cw.x, t.y * cw.y, t.z * cw.z, t.w * cw.w);
            const u32x4 y = wy_split4_unit(t.x * cb.x, t.y * cb.y, t.z * cb.z, t.w * cb.w);
#pragma unroll
            for (int part = 0; part < 2; part++) {
                reinterpret_cast<u32x2 *>(&sTw[half >> 1][part][lane])[half & 1] = u32x2{x[2 * part], x[2 * part + 1]};
                reinterpret_cast<u32x2 *>(&sTu[half >> 1][part][lane])[half & 1] = u32x2{y[2 * part], y[2 * part + 1]};
            }
        }
    }
    __syncthreads();

    // ---- phase 3: W = T diag(beta e^L) K and U = T diag(beta) V -------------------------
    u32x4 tw[6][2], tu[6][2];
#pragma unroll
    for (int at = 0; at < 6; at++)
#pragma unroll
        for (int part = 0; part < 2; part++) tw[at][part] = sTw[at][part][lane], tu[at][part] = sTu[at][part][lane];
    __builtin_amdgcn_sched_barrier(0);   // all reads ahead of the first product
#pragma unroll
    for (int tau = 0; tau < 4; tau++) {
        wy_f32x4 aw = zero, au = zero;
#pragma unroll
        for (int p = 0; p <= tau / 2; p++) {
            const int at = tau < 2 ? tau : 2 + 2 * (tau - 2) + p;
            // W transposed (K as the A side): lane (n = m, g) then holds columns 16c + 4g + i of
            // token 16 tau + n, its 16 bytes of the tile in A-operand order
            aw = wy_mfma(kwl[p], tw[at][0], aw);
            au = wy_mfma(tu[at][1], vuh[p], au);
            aw = wy_mfma(kwh[p], tw[at][1], aw);
            au = wy_mfma(tu[at][0], vul[p], au);
            aw = wy_mfma(kwh[p], tw[at][0], aw);
            au = wy_mfma(tu[at][0], vuh[p], au);
        }
        const size_t tile = (slot * 4 + tau) * NK + wave;
        // U as computed (a D tile), W in A-operand order
        *reinterpret_cast<wy_f32x4 *>(Ut + tile * 256 + lane * 4) = au * v_undo;
        const wy_f32x4 w4 = aw * (1.f / kWyScale);   // (the instruction between the product and wy_split4)
        Wt[tile * 64 + lane] = wy_split4(w4[0], w4[1], w4[2], w4[3], 1.f);
    }
}

// grid (Hv, DV/32), 512 threads: 32 rows of one head's state, as two groups of 16.  Waves 0-3 are the chain that each block waits
// for: wave w forms D of tokens 16w .. 16w+15 from W, and owns columns 32w .. 32w+31 of the state, in f32, which it updates
// and hands to all waves as f16 parts with the scale of each row's largest value there.  Waves 4-7 form O of the same
// tokens from q^, a block later, beside the chain.  (Lane (n, g) of a tile that the update leaves holds row n, columns 16c+4g+i: with
// c = 2w, 2w+1 its own eight values are the B operand of a 32-wide contraction over them, k-slot e < 4 being column 32w+4g+e,
// e >= 4 column 32w+16+4g+e-4; a tile of D likewise tokens 16w+4g+i of row n.  The A side has hi and lo of the same four values in its
// k-slots 0-3 and 4-7, so against a D operand that repeats its values one instruction adds two of the products.)
// Bound by the chain: 4.4 k clocks a block (two exchanges through LDS, 56 matrix and 300 vector instructions in a row), on half the
// CUs at 32 heads.  512 tokens of 32 heads 25.4 us (f32 instructions, 16 rows a workgroup, all CUs) -> 21.2 us; six layers'
// chunks with this and the block precompute above 238 -> 180 us a pass with three sequences side by side, one sequence 54.8 -> 47.6 a layer;
// 2000 tokens 162 -> 118 and 163 -> 144, of 64 heads 337 -> 231 and 331 -> 241.  Tried and not kept: the operands touched two blocks
// ahead to have them in the L2 (24.5 us), O beside D of the same block (24.6).
template <int DK>
__global__ __launch_bounds__(512, 2) void gdn_wy_recur_kernel(
    int Hk, int Hv, int T, const u32x4 *__restrict__ Wt, const u32x4 *__restrict__ Qt,
    const float *__restrict__ Ut, const u32x4 *__restrict__ Mt, const u32x4 *__restrict__ Kt,
    const float *__restrict__ eLc, float *__restrict__ ssm, float *__restrict__ o_raw) {
    constexpr int DV = DK;
    constexpr int NK = DK / 16;   // column tiles of the state
    constexpr int NS = DK / 32;   // 32-column steps of a contraction over them
    __shared__ u32x4 s_s[2][2][NS][2][64];   // state [block % 2][row group][step][hi|lo]
    __shared__ u32x4 s_d[2][2][4][2][64];    // D [block % 2][row group][token tile][hi twice|lo twice]
    __shared__ float s_su[2][2][NS][16], s_du[2][2][4][16];   // what undoes their scales, per row

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
    u32x4 pw[NK];   // W, or q^, of tokens 16w .. 16w+15: a register takes the next block's request as soon as it has been used
    auto w_of = [&](const u32x4 *X, int back, int blk) { return buffer_of(X + ((slot_of(blk) - back) * 4 + w) * NK * 64); };
    auto fetch_all_w = [&](const u32x4 *X, int back) __attribute__((always_inline)) {
        const auto r = w_of(X, back, 0);
#pragma unroll
        for (int c = 0; c < NK; c++) pw[c] = load(r, c);
    };
    // X S0^T of this wave's 16 tokens, X = W or q^ (which lies `back` slots ahead of the head's own), both row groups
    auto times_state = [&](const u32x4 *X, int back, int blk, wy_f32x4 (&p)[2]) __attribute__((always_inline)) {
        // All LDS reads first, and the three terms of every (step, row group) in turn, so that no instruction waits for the one
        // before it (left alone the compiler reads each operand just ahead of its product: 5.2 k clocks a block instead of 4.4 k).
        u32x4 sh[NS][2], sl[NS][2];
        float un[NS][2];
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int rg = 0; rg < 2; rg++) sh[s][rg] = s_s[blk & 1][rg][s][0][lane], sl[s][rg] = s_s[blk & 1][rg][s][1][lane];
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int rg = 0; rg < 2; rg++) un[s][rg] = s_su[blk & 1][rg][s][m];
        __builtin_amdgcn_sched_barrier(0);
        wy_f32x4 acc[NS][2];
        u32x4 hi[NS], lo[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const u32x4 a = pw[2 * s], b = pw[2 * s + 1];
            hi[s] = u32x4{a[0], a[1], b[0], b[1]};
            lo[s] = u32x4{a[2], a[3], b[2], b[3]};
        }
        const wy_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int rg = 0; rg < 2; rg++) acc[s][rg] = wy_mfma(lo[s], sh[s][rg], zero);
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int rg = 0; rg < 2; rg++) acc[s][rg] = wy_mfma(hi[s], sl[s][rg], acc[s][rg]);
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int rg = 0; rg < 2; rg++) acc[s][rg] = wy_mfma(hi[s], sh[s][rg], acc[s][rg]);
        const auto r = w_of(X, back, blk + 1);
#pragma unroll
        for (int c = 0; c < NK; c++) pw[c] = load(r, c);
#pragma unroll
        for (int rg = 0; rg < 2; rg++) {
            p[rg] = acc[0][rg] * un[0][rg];
#pragma unroll
            for (int s = 1; s < NS; s++) p[rg] = wy_fma(acc[s][rg], un[s][rg], p[rg]);
        }
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
            float mx[2];
#pragma unroll
            for (int rg = 0; rg < 2; rg++) {
                mx[rg] = 0.f;
#pragma unroll
                for (int i = 0; i < 4; i++) mx[rg] = fmaxf(fmaxf(mx[rg], fabsf(st[rg][0][i])), fabsf(st[rg][1][i]));
            }
            rows_max2(mx[0], mx[1]);
#pragma unroll
            for (int rg = 0; rg < 2; rg++) {
                float sc, un;
                wy_scale(mx[rg], sc, un);
                const u32x4 a = wy_split4(st[rg][0][0], st[rg][0][1], st[rg][0][2], st[rg][0][3], sc);
                const u32x4 b = wy_split4(st[rg][1][0], st[rg][1][1], st[rg][1][2], st[rg][1][3], sc);
                s_s[buf][rg][w][0][lane] = u32x4{a[0], a[1], b[0], b[1]};
                s_s[buf][rg][w][1][lane] = u32x4{a[2], a[3], b[2], b[3]};
                if (g == 0) s_su[buf][rg][w][m] = un;
            }
        };
        u32x4 kd[2][4];
        wy_f32x4 pu[2];
        float elc;
        auto u_of = [&](int blk) { return buffer_of(Ut + ((slot_of(blk) * 4 + w) * NK + 2 * blockIdx.y) * 256); };
        auto k_of = [&](int blk) { return buffer_of(Kt + (slot_of(blk) * NK + 2 * (owner ? w : 0)) * 4 * 64); };
        auto fetch_elc = [&](int blk) __attribute__((always_inline)) {
            elc = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buffer_of(eLc + slot_of(blk) * kC + kC - 1), 0, 0, 0));
        };
        fetch_all_w(Wt, 0);
        {
            const auto ru = u_of(0), rk = k_of(0);
#pragma unroll
            for (int rg = 0; rg < 2; rg++) pu[rg] = __builtin_bit_cast(wy_f32x4, load(ru, rg));
            fetch_elc(0);
#pragma unroll
            for (int tau = 0; tau < 4; tau++)
#pragma unroll
                for (int ct = 0; ct < 2; ct++) kd[ct][tau] = load(rk, 4 * ct + tau);
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
            float mx[2];
#pragma unroll
            for (int rg = 0; rg < 2; rg++)
                mx[rg] = fmaxf(fmaxf(fabsf(d[rg][0]), fabsf(d[rg][1])), fmaxf(fabsf(d[rg][2]), fabsf(d[rg][3])));
            rows_max2(mx[0], mx[1]);
#pragma unroll
            for (int rg = 0; rg < 2; rg++) {
                float sc, un;
                wy_scale(mx[rg], sc, un);
                const u32x4 x = wy_split4(d[rg][0], d[rg][1], d[rg][2], d[rg][3], sc);
                s_d[blk & 1][rg][w][0][lane] = u32x4{x[0], x[1], x[0], x[1]};
                s_d[blk & 1][rg][w][1][lane] = u32x4{x[2], x[3], x[2], x[3]};
                if (g == 0) s_du[blk & 1][rg][w][m] = un;
            }
            __syncthreads();
            // ---- S' = e^{L_C} S0 + D^T diag(e^{L_C-L}) K, this wave's columns ------
            if (owner) {
#pragma unroll
                for (int rg = 0; rg < 2; rg++)
#pragma unroll
                    for (int ct = 0; ct < 2; ct++) st[rg][ct] *= elc;
                const auto rk = k_of(blk + 1);
                fetch_elc(blk + 1);
                u32x4 dh[4][2], dl[4][2];
                float un[4][2];
#pragma unroll
                for (int tau = 0; tau < 4; tau++)
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) dl[tau][rg] = s_d[blk & 1][rg][tau][1][lane], dh[tau][rg] = s_d[blk & 1][rg][tau][0][lane];
#pragma unroll
                for (int tau = 0; tau < 4; tau++)
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) un[tau][rg] = s_du[blk & 1][rg][tau][m];
                __builtin_amdgcn_sched_barrier(0);
                const wy_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int th = 0; th < 4; th += 2) {
                    wy_f32x4 acc[2][2][2];
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int rg = 0; rg < 2; rg++)
#pragma unroll
                            for (int ct = 0; ct < 2; ct++) acc[t][rg][ct] = wy_mfma(kd[ct][th + t], dl[th + t][rg], zero);
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int rg = 0; rg < 2; rg++)
#pragma unroll
                            for (int ct = 0; ct < 2; ct++) acc[t][rg][ct] = wy_mfma(kd[ct][th + t], dh[th + t][rg], acc[t][rg][ct]);
#pragma unroll
                    for (int t = 0; t < 2; t++) {
#pragma unroll
                        for (int rg = 0; rg < 2; rg++)
#pragma unroll
                            for (int ct = 0; ct < 2; ct++) st[rg][ct] = wy_fma(acc[t][rg][ct], un[th + t][rg], st[rg][ct]);
#pragma unroll
                        for (int ct = 0; ct < 2; ct++) kd[ct][th + t] = load(rk, 4 * ct + th + t);
                    }
                }
                publish_state((blk + 1) & 1);
            }
            __syncthreads();
        }
        __syncthreads();   // the other waves' last block
        if (owner) {
#pragma unroll
            for (int rg = 0; rg < 2; rg++)
#pragma unroll
                for (int ct = 0; ct < 2; ct++) *reinterpret_cast<wy_f32x4 *>(srow + 16 * rg * DK + 16 * ct) = st[rg][ct];
        }
    } else {
        // ================= O = diag(e^L) q^ S0^T + M D, a block behind =================
        u32x4 mt[4];
        wy_f32x4 el;
        auto fetch_m = [&](int blk) __attribute__((always_inline)) {
            const auto r = buffer_of(Mt + (slot_of(blk) * 4 + w) * 4 * 64);
#pragma unroll
            for (int tau = 0; tau < 4; tau++) mt[tau] = load(r, tau <= w ? tau : w);
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
        __syncthreads();   // block 0: its D and the state behind it are there
        for (int blk = 0; blk < nblk; blk++) {
            wy_f32x4 o[2];
            times_state(Qt, shared, blk, o);
            o[0] *= el;
            o[1] *= el;
            fetch_el(blk + 1);
            __syncthreads();   // the state of this block may be written over
            // (tiles past the diagonal repeat the last one; their products are left out of the sum)
            u32x4 dh[4][2], dl[4][2];
            float un[4][2];
#pragma unroll
            for (int tau = 0; tau < 4; tau++)
#pragma unroll
                for (int rg = 0; rg < 2; rg++) dl[tau][rg] = s_d[blk & 1][rg][tau][1][lane], dh[tau][rg] = s_d[blk & 1][rg][tau][0][lane];
#pragma unroll
            for (int tau = 0; tau < 4; tau++)
#pragma unroll
                for (int rg = 0; rg < 2; rg++) un[tau][rg] = s_du[blk & 1][rg][tau][m];
            __builtin_amdgcn_sched_barrier(0);
            const wy_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            wy_f32x4 acc[4][2];
#pragma unroll
            for (int tau = 0; tau < 4; tau++)
                if (tau <= w) {
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) acc[tau][rg] = wy_mfma(mt[tau], dl[tau][rg], zero);
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) acc[tau][rg] = wy_mfma(mt[tau], dh[tau][rg], acc[tau][rg]);
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) o[rg] = wy_fma(acc[tau][rg], un[tau][rg], o[rg]);
                }
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
    return nblk * Hv * (3 * (size_t)kC * dk + (size_t)kC * dv + (size_t)kC * kC + kC);
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
    // (an operand's two f16 parts take the four bytes of the f32 value they stand for)
    u32x4 *Wt = reinterpret_cast<u32x4 *>(scratch);
    u32x4 *Qt = Wt + slots * kC * dk / 4;
    u32x4 *Kt = Qt + slots * kC * dk / 4;
    float *Ut = reinterpret_cast<float *>(Kt + slots * kC * dk / 4);
    u32x4 *Mt = reinterpret_cast<u32x4 *>(Ut + slots * kC * dv);
    float *eLc = reinterpret_cast<float *>(Mt + slots * kC * kC / 4);
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
