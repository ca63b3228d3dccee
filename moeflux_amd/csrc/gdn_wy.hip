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
// independent).  The products before D are v_mfma_f32_16x16x4_f32; those that involve the state are
// v_mfma_f32_16x16x32_f16 over operands split into two f16 numbers (see wy_split4).
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
static constexpr float kWyScale = 16384.f;   // 2^14: the largest f16 is 65504
__device__ inline uint32_t wy_pack(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2)); }
__device__ inline void wy_split2(float a, float b, uint32_t &hi, uint32_t &lo) {
    const f16x2 h = __builtin_convertvector(f32x2{a, b}, f16x2);
    hi = __builtin_bit_cast(uint32_t, h);
    lo = wy_pack(a - (float)h[0], b - (float)h[1]);
}
// four values as 16 bytes: hi of all, lo of all
__device__ inline u32x4 wy_split4(float a, float b, float c, float d) {
    uint32_t h0, h1, l0, l1;
    wy_split2(a, b, h0, l0);
    wy_split2(c, d, h1, l1);
    return u32x4{h0, h1, l0, l1};
}
__device__ inline u32x4 wy_split4_unit(float a, float b, float c, float d) {   // of values of at most 1
    return wy_split4(a * kWyScale, b * kWyScale, c * kWyScale, d * kWyScale);
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
//   Wt [token tile w][col tile c], Qt likewise, Mt [w][token tile tau], Kt [col tile c][tau]
//   (= diag(e^{L_C-L}) K transposed): lane (m, g) holds X[16 row-tile + m][16 col-tile + 4g + i];
//   Ut [w][col tile c]: lane (n, g) holds U[16w + 4g + i][16c + n]  (a D tile as computed);
//   eL [64] (e^{L_t}; eL[63] = e^{L_C} because padded tokens do not decay).
// Tokens past the end of the chunk are padded with beta = 0, log g = 0, k = q = v = 0.
//
// grid (Hv, blocks), one wave per 16 columns of K (DK/16 waves: two per SIMD at DK = 128, so that one
// has matrix work while the other waits for LDS or stores a tile).
// FUSED: the block's inputs come straight from the layer's inputs (WyInputs): what
// gdn_chunk_pre_kernel computes for the token-by-token form is done here per (block, value head) -
// conv + SiLU of the head's q, k and v channels, the per-token q/k norm, the decay's logarithm and
// beta - so the chunk needs no launch and no arrays for them.  A k-head's q and k are formed by
// each of the value heads that share it.
template <int DK, bool FUSED>
__global__ __launch_bounds__(DK * 4) void gdn_wy_kernel(
    int Hk, int Hv, int T, const float *__restrict__ qn, const float *__restrict__ kn,
    const float *__restrict__ vv, const float *__restrict__ lg, const float *__restrict__ bg,
    u32x4 *__restrict__ Wt, u32x4 *__restrict__ Qt, float *__restrict__ Ut, u32x4 *__restrict__ Mt,
    u32x4 *__restrict__ Kt, float *__restrict__ eLc, WyInputs in) {
    constexpr int DV = DK;
    constexpr int NK = DK / 16;
    constexpr int LDK = DK + 4;  // row strides chosen so that 16-byte row reads by 8 lanes hit all banks
    constexpr int LDC = kC + 4;
    constexpr int NW = NK;        // waves
    constexpr int NTHR = 64 * NW;
    constexpr int NCT = 1;        // 16-wide column tiles of W (and of U) per wave
    static_assert(!FUSED || NCT == 1, "a wave's v is one column tile");
    __shared__ __align__(16) float sK[kC][LDK];
    // FUSED keeps to half a CU's LDS (81664 bytes of 163840; it was 137472), so that a CU holds two workgroups, of one launch or
    // of two sequences': v stays in the registers of the wave that multiplies it, A is its ten lower tiles, and T lies
    // where q^ was.  The kernel waits on memory, LDS and its substitution chain far more than on its products (512 tokens,
    // six layers 261 -> 237 us a pass with three sequences side by side; 2000 tokens of one layer 176 -> 154).
    __shared__ __align__(16) float sQ[kC][LDK];  // q^, later v (FUSED: later T)
    __shared__ __align__(16) float sA[10][16][20];   // tile (I, J <= I) at I (I + 1) / 2 + J
    __shared__ __align__(16) float sTown[FUSED ? 1 : kC][LDC];
    static_assert(LDC <= LDK, "T fits where q^ was");
    float(*sT)[LDC] = FUSED ? reinterpret_cast<float(*)[LDC]>(&sQ[0][0]) : sTown;
    __shared__ __align__(16) float sL[kC], sB[kC], sCw[kC], sKd[kC];
    __shared__ int sR[kC];

    // heads along x: a head's blocks are produced on the XCD whose L2 the recurrence kernel
    // (heads along x as well) will read them through
    const int vh = wy_head_of(blockIdx.x, Hk, Hv), blk = blockIdx.y, kh = vh / (Hv / Hk);
    const int t0 = blk * kC;
    const int nt = (T - t0 < kC) ? T - t0 : kC;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, g = lane >> 4;
    const size_t slot = (size_t)blk * Hv + vh;

    // ---- phase 0: k^, q^ of the block, cumulative log decay, beta ---------------------
    // Everything the block reads is requested here, in the order of use (loads return in the
    // order of their requests): the gates, k^ and q^, and v, which waits in registers for phase 2.
    float lg_in = 0.f, bg_in = 0.f;
    constexpr int NLV = kC * (DV / 4) / NTHR;
    float4 va[FUSED ? 1 : NLV];
    float vreg[4][4];   // FUSED: v of tokens 16 s + 4 g + i, channel 16 wave + m, phase 3's operand
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
            const float sc = is_q ? inv_scale * inv_scale : inv_scale;
#pragma unroll
            for (int i = 0; i < EPL / 4; i++) {
                float4 y = {x[i].x * inv_rms, x[i].y * inv_rms, x[i].z * inv_rms, x[i].w * inv_rms};
                y.x *= sc; y.y *= sc; y.z *= sc; y.w *= sc;
                *(float4 *)(row + 4 * i) = y;
            }
        }
    } else {
    if (wave == 0 && lane < nt) {
        lg_in = lg[(size_t)(t0 + lane) * Hv + vh];
        bg_in = bg[(size_t)(t0 + lane) * Hv + vh];
    }
    {
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
        for (int u = 0; u < NLV; u++) {
            const int i = tid + u * NTHR, tt = i / (DV / 4), x = (i % (DV / 4)) * 4;
            va[u] = load_f4(vv + ((size_t)(t0 + (tt < nt ? tt : nt - 1)) * Hv + vh) * DV + x);
        }
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int i = tid + u * NTHR, tt = i / (DK / 4), x = (i % (DK / 4)) * 4;
            const float keep = tt < nt ? 1.f : 0.f;  // padded tokens are zero rows
            *(float4 *)&sK[tt][x] = float4{a[u].x * keep, a[u].y * keep, a[u].z * keep, a[u].w * keep};
            *(float4 *)&sQ[tt][x] = float4{b[u].x * keep, b[u].y * keep, b[u].z * keep, b[u].w * keep};
        }
    }
    }
    if (wave == 0) {
        // Cumulative log decay, restarted after every token whose decay is zero: where the
        // reference's exp() underflows (log g below log FLT_MIN; -inf when its softplus overflows,
        // linear_attn.rs:357-370) the token forgets everything before it, and no factor e^{L_i-L_j}
        // may be formed across it (-inf - -inf).  sR[t] is the last such token up to and
        // including t (-1: none); a pair (row, col) decays to exactly 0 when sR[row] > col.
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
        const float b = bg_in;
        const float el = r >= 0 ? 0.f : expf(l);      // decay since the block's first token
        sL[lane] = l;
        sR[lane] = r;
        sB[lane] = b;
        sCw[lane] = b * el;
        eLc[slot * kC + lane] = el;
        sKd[lane] = __shfl(r, 63, 64) > lane ? 0.f : expf(__shfl(l, 63, 64) - l);  // e^{L_C - L_t}
    }
    __syncthreads();

    // ---- phase 1: the lower tiles of K K^T (-> A) and of Q K^T (-> M) -----------------
    // 10 tiles (I, J <= I) each; 20 jobs of DK/4 instructions dealt round the waves.
#pragma unroll
    for (int r = 0; r < (20 + NW - 1) / NW; r++) {
        const int job = wave + NW * r;
        if (job >= 20) break;   // uniform over the wave
        const int kind = job / 10, idx = job % 10;
        const int I = idx >= 6 ? 3 : idx >= 3 ? 2 : idx >= 1 ? 1 : 0;
        const int J = idx - I * (I + 1) / 2;
        wy_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        if (kind == 0) {
#pragma unroll
            for (int s = 0; s < DK / 16; s++)
                acc = mfma4(lds_f4(&sK[16 * I + m][16 * s + 4 * g]), lds_f4(&sK[16 * J + m][16 * s + 4 * g]), acc);
            // lane (n = m, g) holds rows 16I + 4g + i of column 16J + n
            const int col = 16 * J + m;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = 16 * I + 4 * g + i;
                const float dl = sL[row] - sL[col];
                const float d = sR[row] > col ? 0.f : __builtin_amdgcn_exp2f((dl < 0.f ? dl : 0.f) * 1.4426950408889634f);  // v_exp_f32: 1 ulp
                sA[idx][4 * g + i][m] = (col < row) ? sB[row] * d * acc[i] : 0.f;
            }
        } else {
            // the tile transposed (k^ as the A side): lane (n = m, g) then holds columns 16J + 4g + i of
            // row 16I + n, which is this lane's 16 bytes of tile (I, J) in A-operand order
#pragma unroll
            for (int s = 0; s < DK / 16; s++)
                acc = mfma4(lds_f4(&sK[16 * J + m][16 * s + 4 * g]), lds_f4(&sQ[16 * I + m][16 * s + 4 * g]), acc);
            const int row = 16 * I + m;
            wy_f32x4 mv;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int col = 16 * J + 4 * g + i;
                const float dl = sL[row] - sL[col];
                const float d = sR[row] > col ? 0.f : __builtin_amdgcn_exp2f((dl < 0.f ? dl : 0.f) * 1.4426950408889634f);
                mv[i] = (col <= row) ? d * acc[i] : 0.f;
            }
            Mt[((slot * 4 + I) * 4 + J) * 64 + lane] = wy_split4_unit(mv[0], mv[1], mv[2], mv[3]);
        }
    }
    for (int i = tid; i < 4 * NK * 64; i += NTHR) {  // q^ tiles, before v takes its place
        const int tile = i >> 6, l = i & 63, w = tile / NK, c = tile % NK;
        const float4 q = lds_f4(&sQ[16 * w + (l & 15)][16 * c + 4 * (l >> 4)]);
        Qt[(slot * 4 * NK + tile) * 64 + l] = wy_split4_unit(q.x, q.y, q.z, q.w);
    }
    __syncthreads();

    // ---- phase 2: diag(e^{L_C - L}) K transposed goes out, v comes in, and
    //      T = (I + A)^-1 by blocks of 16: the diagonal blocks by forward substitution (one
    //      per wave, a column per lane), the blocks below them level by level from
    //      T_IJ = -T_II sum_{J <= K < I} A_IK T_KJ on the matrix cores -----------------------
    {
#pragma unroll
        for (int u = 0; u < NK * 4 * 64 / NTHR; u++) {
            const int i = tid + u * NTHR, tile = i >> 6, l = i & 63, c = tile >> 2, tau = tile & 3;
            const int kk = 16 * c + (l & 15), j4 = 16 * tau + 4 * (l >> 4);
            const float4 e = lds_f4(&sKd[j4]);
            Kt[(slot * NK * 4 + tile) * 64 + l] = wy_split4_unit(e.x * sK[j4 + 0][kk], e.y * sK[j4 + 1][kk], e.z * sK[j4 + 2][kk], e.w * sK[j4 + 3][kk]);
        }
        if constexpr (!FUSED) {
#pragma unroll
            for (int u = 0; u < NLV; u++) {
                const int i = tid + u * NTHR, tt = i / (DV / 4), x = (i % (DV / 4)) * 4;
                const float keep = tt < nt ? 1.f : 0.f;
                *(float4 *)&sQ[tt][x] = float4{va[u].x * keep, va[u].y * keep, va[u].z * keep, va[u].w * keep};
            }
        }
    }
    if (wave < 4) {
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
    __syncthreads();
#pragma unroll
    for (int lvl = 1; lvl < 4; lvl++) {
        if (wave < 4 - lvl) {  // block (I, J) = (wave + lvl, wave)
            const int I = wave + lvl, J = wave;
            wy_f32x4 x = {0.f, 0.f, 0.f, 0.f};
            for (int K = J; K < I; K++) {
                float4 bt;
                bt.x = sT[16 * K + 4 * g + 0][16 * J + m];
                bt.y = sT[16 * K + 4 * g + 1][16 * J + m];
                bt.z = sT[16 * K + 4 * g + 2][16 * J + m];
                bt.w = sT[16 * K + 4 * g + 3][16 * J + m];
                x = mfma4(lds_f4(&sA[I * (I + 1) / 2 + K][m][4 * g]), bt, x);
            }
            // x is held as rows 4g+i of column m: already the B operand of T_II x
            wy_f32x4 r = {0.f, 0.f, 0.f, 0.f};
            r = mfma4(lds_f4(&sT[16 * I + m][16 * I + 4 * g]), as_f4(x), r);
#pragma unroll
            for (int i = 0; i < 4; i++) sT[16 * I + 4 * g + i][16 * J + m] = -r[i];
        }
        __syncthreads();
    }

    // ---- phase 3: W = T diag(beta e^L) K and U = T diag(beta) V -------------------------
    // Wave w owns column tiles NCT*w .. of both; the K and V operands of those columns are
    // read once and serve all four token tiles.
    float bK[4][NCT][4], bV[4][NCT][4];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int ct = 0; ct < NCT; ct++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                bK[s][ct][i] = sK[16 * s + 4 * g + i][16 * (NCT * wave + ct) + m];
                bV[s][ct][i] = FUSED ? vreg[s][i] : sQ[16 * s + 4 * g + i][16 * (NCT * wave + ct) + m];
            }
#pragma unroll
    for (int tau = 0; tau < 4; tau++) {
        wy_f32x4 aw4[NCT], au4[NCT];
#pragma unroll
        for (int ct = 0; ct < NCT; ct++) aw4[ct] = au4[ct] = wy_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s <= tau; s++) {
            const float4 t4 = lds_f4(&sT[16 * tau + m][16 * s + 4 * g]);
            const float4 cw = lds_f4(&sCw[16 * s + 4 * g]), cb = lds_f4(&sB[16 * s + 4 * g]);
            const float4 tw = {t4.x * cw.x, t4.y * cw.y, t4.z * cw.z, t4.w * cw.w};
            const float4 tu = {t4.x * cb.x, t4.y * cb.y, t4.z * cb.z, t4.w * cb.w};
#pragma unroll
            for (int ct = 0; ct < NCT; ct++) {
                // W transposed (K as the A side): lane (n = m, g) then holds columns 16c + 4g + i of
                // token 16 tau + n, its 16 bytes of the tile in A-operand order
                aw4[ct] = mfma4(float4{bK[s][ct][0], bK[s][ct][1], bK[s][ct][2], bK[s][ct][3]}, tw, aw4[ct]);
                au4[ct] = mfma4(tu, float4{bV[s][ct][0], bV[s][ct][1], bV[s][ct][2], bV[s][ct][3]}, au4[ct]);
            }
        }
#pragma unroll
        for (int ct = 0; ct < NCT; ct++) {
            const wy_f32x4 aw = aw4[ct], au = au4[ct];
            const size_t tile = (slot * 4 + tau) * NK + NCT * wave + ct;
            // U as computed (a D tile), W in A-operand order
            *reinterpret_cast<wy_f32x4 *>(Ut + tile * 256 + lane * 4) = au;
            Wt[tile * 64 + lane] = wy_split4_unit(aw[0], aw[1], aw[2], aw[3]);
        }
    }
}

// grid (Hv, DV/32), 512 threads: 32 rows of one head's state, as two groups of 16.  Waves w and w + 4 serve tokens 16w .. 16w+15
// of each block, the first with W (and then D), the second with q^ (and then O); in the update of the state wave 4 rg + s owns
// columns 32s .. 32s+31 of row group rg, in f32, and hands them to all waves as f16 parts with the scale of each row's largest
// value there.  (Lane (n, g) of a tile that the update leaves holds row n, columns 16c+4g+i: with c = 2s, 2s+1 its own eight
// values are the B operand of a 32-wide contraction over them, k-slot e < 4 being column 32s+4g+e, e >= 4 column 32s+16+4g+e-4;
// a tile of D likewise tokens 16w+4g+i of row n.  The A side has hi and lo of the same four values in its k-slots 0-3 and 4-7, so
// against a D operand that repeats its values one instruction adds two of the products.)
// Bound by the two exchanges a block and by the CU's 64 bytes a clock of operands.  512 tokens of 32 heads take 25 us on half the
// CUs (f32 instructions, 16 rows a workgroup: 25 us on all of them): six layers 241 -> 205 us a pass with three sequences side by
// side, 2000 tokens of one layer 162 -> 128, of 64 heads 337 -> 261.
template <int DK>
__global__ __launch_bounds__(512, 2) void gdn_wy_recur_kernel(
    int Hk, int Hv, int T, const u32x4 *__restrict__ Wt, const u32x4 *__restrict__ Qt,
    const float *__restrict__ Ut, const u32x4 *__restrict__ Mt, const u32x4 *__restrict__ Kt,
    const float *__restrict__ eLc, float *__restrict__ ssm, float *__restrict__ o_raw) {
    constexpr int DV = DK;
    constexpr int NK = DK / 16;   // column tiles of the state
    constexpr int NS = DK / 32;   // 32-column steps of a contraction over them
    __shared__ u32x4 s_s[2][NS][2][64];    // state [row group][step][hi|lo]
    __shared__ u32x4 s_d[2][2][4][2][64];  // D [block % 2][row group][token tile][hi twice|lo twice]
    __shared__ float s_su[2][NS][16], s_du[2][2][4][16];   // what undoes their scales, per row

    const int vh = wy_head_of(blockIdx.x, Hk, Hv), row0 = blockIdx.y * 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int w = wave & 3, rgu = wave >> 2;   // token tile; of the update: row group, and step w
    const bool owner = w < NS;
    const int nblk = (T + kC - 1) / kC;
    auto slot_of = [&](int blk) { return (size_t)(blk < nblk ? blk : nblk - 1) * Hv + vh; };   // past the end: the last block again

    float *srow = ssm + ((size_t)vh * DV + row0 + 16 * rgu + m) * DK + 32 * (owner ? w : 0) + 4 * g;
    wy_f32x4 st[2] = {load_v4(srow), load_v4(srow + 16)};
    auto publish_state = [&]() __attribute__((always_inline)) {
        float mx = 0.f, sc, un;
#pragma unroll
        for (int ct = 0; ct < 2; ct++)
#pragma unroll
            for (int i = 0; i < 4; i++) mx = fmaxf(mx, fabsf(st[ct][i]));
        wy_scale(rows_max(mx), sc, un);
        const u32x4 a = wy_split4(st[0][0] * sc, st[0][1] * sc, st[0][2] * sc, st[0][3] * sc);
        const u32x4 b = wy_split4(st[1][0] * sc, st[1][1] * sc, st[1][2] * sc, st[1][3] * sc);
        s_s[rgu][w][0][lane] = u32x4{a[0], a[1], b[0], b[1]};
        s_s[rgu][w][1][lane] = u32x4{a[2], a[3], b[2], b[3]};
        if (g == 0) s_su[rgu][w][m] = un;
    };

    // ROLE 0: W, D; ROLE 1: q^, O.  D and the state are the chain that the next block waits for; O of a block is formed a block
    // later, beside the chain (its waves give way to the others: s_setprio).  An operand's register takes the next block's
    // request as soon as it has been used.  Requests go through a descriptor of the block's operand, so that they cost a
    // scalar addition each and no vector one.
    const int lane16 = lane * 16;
    auto run = [&](auto role_tag) __attribute__((always_inline)) {
        constexpr int ROLE = decltype(role_tag)::value;
        u32x4 pw[NK], mt[4], kd[2][4];
        wy_f32x4 pu[2], el, o[2];
        float elc;
        auto load = [&](__amdgpu_buffer_rsrc_t r, int tile) __attribute__((always_inline)) {
            return __builtin_amdgcn_raw_buffer_load_b128(r, lane16, tile * 1024, 0);
        };
        auto w_of = [&](int blk) { return buffer_of((ROLE == 0 ? Wt : Qt) + (slot_of(blk) * 4 + w) * NK * 64); };
        auto fetch_u = [&](int blk) __attribute__((always_inline)) {
            const auto r = buffer_of(Ut + ((slot_of(blk) * 4 + w) * NK + 2 * blockIdx.y) * 256);
#pragma unroll
            for (int rg = 0; rg < 2; rg++) pu[rg] = __builtin_bit_cast(wy_f32x4, load(r, rg));
        };
        auto fetch_el = [&](int blk) __attribute__((always_inline)) {
            el = __builtin_bit_cast(wy_f32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer_of(eLc + slot_of(blk) * kC + 16 * w), g * 16, 0, 0));
        };
        auto fetch_m = [&](int blk) __attribute__((always_inline)) {
            const auto r = buffer_of(Mt + (slot_of(blk) * 4 + w) * 4 * 64);
#pragma unroll
            for (int tau = 0; tau < 4; tau++) mt[tau] = load(r, tau <= w ? tau : w);
        };
        auto fetch_k = [&](int blk) __attribute__((always_inline)) {
            const size_t slot = slot_of(blk);
            const auto r = buffer_of(Kt + (slot * NK + 2 * (owner ? w : 0)) * 4 * 64);
            elc = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buffer_of(eLc + slot * kC + kC - 1), 0, 0, 0));
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int tau = 0; tau < 4; tau++) kd[ct][tau] = load(r, 4 * ct + tau);
        };
        // O of block blk = (what diag(e^L) q^ S0^T left in o) + M D
        auto finish_o = [&](int blk) __attribute__((always_inline)) {
            const u32x4(*sd)[4][2][64] = s_d[blk & 1];
            const float(*du)[4][16] = s_du[blk & 1];
#pragma unroll
            for (int tau = 0; tau < 4; tau++)
                if (tau <= w) {
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) {
                        wy_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                        acc = wy_mfma(mt[tau], sd[rg][tau][1][lane], acc);
                        acc = wy_mfma(mt[tau], sd[rg][tau][0][lane], acc);
                        o[rg] += acc * du[rg][tau][m];
                    }
                }
            const int rows = T - (blk * kC + 16 * w) - 4 * g;   // tokens from this lane's first on
            float *dst = o_raw + ((size_t)(blk * kC + 16 * w) * Hv + vh) * DV + row0;
            const int stride = Hv * DV, off = 4 * g * stride + m;
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i < rows) {
#pragma unroll
                    for (int rg = 0; rg < 2; rg++) dst[off + i * stride + 16 * rg] = o[rg][i];
                }
        };
        {
            const auto r = w_of(0);
#pragma unroll
            for (int c = 0; c < NK; c++) pw[c] = load(r, c);
        }
        if (ROLE == 0) fetch_u(0);
        else fetch_el(0);
        fetch_k(0);
        if (owner) publish_state();
        __syncthreads();
        for (int blk = 0; blk < nblk; blk++) {
            // ---- W S0^T, or q^ S0^T, for this wave's 16 tokens ------------------------------
            if constexpr (ROLE == 0) __builtin_amdgcn_s_setprio(1);
            if constexpr (ROLE == 1) {
                if (blk > 0) {
                    finish_o(blk - 1);
                }
                fetch_m(blk);
            }
            wy_f32x4 p[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            const auto r = w_of(blk + 1);
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const u32x4 a = pw[2 * s], b = pw[2 * s + 1];
                const u32x4 hi = {a[0], a[1], b[0], b[1]}, lo = {a[2], a[3], b[2], b[3]};
#pragma unroll
                for (int rg = 0; rg < 2; rg++) {
                    const u32x4 sh = s_s[rg][s][0][lane], sl = s_s[rg][s][1][lane];
                    wy_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                    acc = wy_mfma(lo, sh, acc);
                    acc = wy_mfma(hi, sl, acc);
                    acc = wy_mfma(hi, sh, acc);
                    p[rg] += acc * s_su[rg][s][m];
                }
                pw[2 * s] = load(r, 2 * s);
                pw[2 * s + 1] = load(r, 2 * s + 1);
            }
            if constexpr (ROLE == 0) {
                // ---- D = U - W S0^T: lane (n, g) holds tokens 16w+4g+i of state row n of the group ----
                const wy_f32x4 d[2] = {pu[0] - p[0], pu[1] - p[1]};
                fetch_u(blk + 1);
#pragma unroll
                for (int rg = 0; rg < 2; rg++) {
                    float sc, un;
                    wy_scale(rows_max(fmaxf(fmaxf(fabsf(d[rg][0]), fabsf(d[rg][1])), fmaxf(fabsf(d[rg][2]), fabsf(d[rg][3])))), sc, un);
                    const u32x4 x = wy_split4(d[rg][0] * sc, d[rg][1] * sc, d[rg][2] * sc, d[rg][3] * sc);
                    s_d[blk & 1][rg][w][0][lane] = u32x4{x[0], x[1], x[0], x[1]};
                    s_d[blk & 1][rg][w][1][lane] = u32x4{x[2], x[3], x[2], x[3]};
                    if (g == 0) s_du[blk & 1][rg][w][m] = un;
                }
            } else {
#pragma unroll
                for (int rg = 0; rg < 2; rg++) o[rg] = el * p[rg];
                fetch_el(blk + 1);
            }
            __syncthreads();
            // ---- S' = e^{L_C} S0 + D^T diag(e^{L_C-L}) K, this wave's columns and rows ------
            if (owner) {
#pragma unroll
                for (int ct = 0; ct < 2; ct++) st[ct] *= elc;
#pragma unroll
                for (int tau = 0; tau < 4; tau++) {
                    const u32x4 dh = s_d[blk & 1][rgu][tau][0][lane], dl = s_d[blk & 1][rgu][tau][1][lane];
                    const float un = s_du[blk & 1][rgu][tau][m];
#pragma unroll
                    for (int ct = 0; ct < 2; ct++) {
                        wy_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                        acc = wy_mfma(kd[ct][tau], dl, acc);
                        acc = wy_mfma(kd[ct][tau], dh, acc);
                        st[ct] += acc * un;
                    }
                }
                publish_state();
                fetch_k(blk + 1);
            }
            __syncthreads();
        }
        if constexpr (ROLE == 1) finish_o(nblk - 1);
    };
    if (rgu == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});
    if (owner) {
#pragma unroll
        for (int ct = 0; ct < 2; ct++) *reinterpret_cast<wy_f32x4 *>(srow + 16 * ct) = st[ct];
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
