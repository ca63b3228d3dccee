// Attention over a compressed (latent) cache for gfx950: the folded form of multi-head
// latent attention, one query token.
//
// Per head h:  s[t] = (q'[h] . latent[t] + q_pe[h] . rope_k[t]) * scale,  w = softmax(s),
//              out[h] = sum_t w[t] latent[t].
// Every head reads the same keys ([latent | rope_k], R + P wide) and the same values
// (latent): the heads are the free dimension of both products, so they form one side of
// the MFMA tiles and a workgroup reads its positions once for all of its heads.
//
// Both products run on the bf16 matrix pipeline at f32-like accuracy: every f32 operand x
// is split into bf16 parts hi = bf16(x), lo = bf16(x - hi)  (x = hi + lo to 2^-18 x), and a
// product a b is evaluated as a_hi b_hi + a_hi b_lo + a_lo b_hi with f32 accumulation.
//
// Two kernels (mla_plan chooses); partials (unnormalised O, running max and sum per head) go to the workspace in the
// layout of the decode kernel's partials, and sdpa_merge_kernel combines them.
//
//   mla_rounds_kernel<NHT>   a workgroup (8 waves) serves 16 NHT heads and walks its share of the cache in rounds of 128
//     positions, each in two phases:
//       scores   a wave owns 16 positions of the round and forms their scores against every head of the workgroup: keys
//                come from memory in whole lines and change lanes through 4 KiB of the wave's own LDS (mla_operands); the queries,
//                split once per workgroup, are B operands in LDS;
//       values   a wave owns 64 channels: lane (n, g) reads channels 4 n .. 4 n + 3 of positions 4 g + e and 16 + 4 g + e
//                (256 contiguous bytes per row), so that the four channels are B operands of four tiles and no value is ever
//                transposed; the probabilities are A operands in LDS, in exactly the registers the scores left them in.
//     Nothing passes between waves but the rows' maxima and the probabilities: two barriers a round.  For caches of few rounds:
//     its workgroups start 3 us sooner than the other kernel's, and with 16 or 32 heads each they leave a half or a quarter of the
//     partials.  It converts each row twice per workgroup, so that with more than
//     two rounds of 32 heads the vector ALU (10 k of a round's 19 k clocks at 32 heads) costs more than that saves.
//
//   mla_stream_kernel<R, P>   grid (splits, ceil(H / 64)); 8 waves in two roles.  Wave hg
//     (0..3) computes the scores and the softmax of head group hg, wave 4 + hg accumulates
//     that group's values; the two share a SIMD and run one block apart, so that one of
//     them always has matrix work while the other converts, exponentiates or stores:
//       iteration it:   score waves   S(it + 1): 16 positions x 16 heads over R + P channels,
//                                     online softmax, weights to LDS as bf16 hi/lo operands
//                       value waves   V(it):  O[channel][head] += X[slot][channel] P[slot][head]
//       and both stage block it + 2 (one barrier per iteration).
//     A block of 16 positions lives in LDS once, split but not transposed:
//       krow[hi|lo][position][channel], three buffers (scored, accumulated, being written);
//     rows are 1184 bytes apart, the stride at which both kinds of read below run without
//     bank conflicts.  The scores read it as an A operand directly (a lane's 8 channels of
//     one position are contiguous).  The values need 8 positions of one channel per lane:
//     ds_read_b64_tr_b16 delivers exactly that from the row-major block (within 16 lanes,
//     lane j receives element j % 4 of the 8 bytes addressed by lanes j/4, j/4 + 4, j/4 + 8,
//     j/4 + 12; with lane L pointing at position L/4, channels 4 (L % 4) .. + 3, lane j
//     ends up with channel j at four positions).  The value product's 32 slots are the hi
//     parts of the 16 positions followed by their lo parts, so that with P = [p_hi | p_hi]
//     one instruction adds x_hi p_hi + x_lo p_hi and a second with [p_lo | p_lo] adds x_hi p_lo
//     (and x_lo p_lo, which comes for free).
//     The value waves fetch and split 6 of a block's 16 latent rows (four channels of every second one per
//     thread), the score waves the other 10 and the rotary keys (4 or 8 for the value waves are no faster).
#include <algorithm>
#include <type_traits>

#include "sdpa_wave.h"

namespace mfa {

__device__ inline f32x4 mla_load4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }

static constexpr int kMlaWaves = 8;

// hi and lo operand halves of eight values
__device__ inline void mla_split8(const f32x4 &a, const f32x4 &b, bf16x8 &hi, bf16x8 &lo) {
    uint4 h, l;
    split_pair(a[0], a[1], h.x, l.x);
    split_pair(a[2], a[3], h.y, l.y);
    split_pair(b[0], b[1], h.z, l.z);
    split_pair(b[2], b[3], h.w, l.w);
    hi = as_bf16x8(h);
    lo = as_bf16x8(l);
}

// 16 rows x 64 channels, read as four requests of four rows (256 contiguous bytes each: lane l has channels 4 (l % 16) .. + 3 of row
// 4 r + l / 16), as the operands of two 32-channel steps: step k takes channels 32 k + 8 g .. + 7 of row n into lane (n, g).  They
// change lanes through 4 KiB of LDS of the wave's own (LDS executes a wave's instructions in order: no barrier).  Requested in
// operand order instead, neighbouring lanes in different rows, a request takes 49 clocks of the CU's 16; exchanged by DPP selects
// (32 for the 16 values a lane holds) these cost 20 clocks each as soon as a SIMD has two waves.
static constexpr int kMlaRow = 68;   // floats from row to row: 16 neighbouring lanes then read 16 different groups of four banks
__device__ inline void mla_operands(const f32x4 (&x)[4], float *buf, int lane, bf16x8 (&hi)[2], bf16x8 (&lo)[2]) {
    const int n = lane & 15, g = lane >> 4;
#pragma unroll
    for (int r = 0; r < 4; r++) *reinterpret_cast<f32x4 *>(buf + (4 * r + g) * kMlaRow + 4 * n) = x[r];
    wave_lds_order();
    f32x4 y[2][2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const float *at = buf + n * kMlaRow + 32 * k + 8 * g;
        y[k][0] = mla_load4(at), y[k][1] = mla_load4(at + 4);
    }
    wave_lds_order();   // ahead of the next call's writes
#pragma unroll
    for (int k = 0; k < 2; k++) mla_split8(y[k][0], y[k][1], hi[k], lo[k]);
}

// Workgroup id -> (split, head group).  Workgroups go to the 8 XCDs in turn; those of one split read the same rows and sit on
// one XCD, one after the other, so that the rows come through its L2 once.
template <int NHT>
__global__ __launch_bounds__(kMlaWaves * 64, 2) void mla_rounds_kernel(
    const float *__restrict__ q_prime, const float *__restrict__ q_pe, const float *__restrict__ latent,
    const float *__restrict__ rope_k, int H, int L, int nsplit, int ngroups, int per_split, float qscale,
    float *__restrict__ part_o, float *__restrict__ part_ml) {
    constexpr int R = 512, P = 64;
    constexpr int NS = (R + P) / 64, NSL = R / 64;   // 64-channel steps of the scores; of which latent
    constexpr int HW = 16 * NHT;                     // heads of a workgroup
    constexpr int WPOS = 16, ROUND = kMlaWaves * WPOS;   // positions of a wave, of a round
    constexpr int D = 2;                             // steps of keys in flight
    __shared__ uint4 sq[2 * NS][NHT][2][64];         // queries [32 channels][head tile][hi|lo], operand order
    __shared__ uint4 sp[ROUND / 32][NHT][2][64];     // probabilities [32 positions][head tile][hi|lo], operand order
    __shared__ __attribute__((aligned(16))) float smax[HW][kMlaWaves];
    __shared__ float ssum[kMlaWaves][HW];
    __shared__ __attribute__((aligned(16))) float kbuf[kMlaWaves][16 * kMlaRow];   // see mla_operands

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    float *buf = kbuf[wave];
    const int id = blockIdx.x, xi = id >> 3;
    const int split = (xi / ngroups) * 8 + (id & 7), group = xi % ngroups;
    if (split >= nsplit) return;   // uniform over the workgroup, ahead of every barrier
    const int h0 = group * HW;
    const int p0 = split * per_split, p1 = min(p0 + per_split, L);   // p0 < p1: the plan has no empty split

    // queries: 16 heads x 64 channels per unit, split into LDS
    {
        constexpr int NU = (NS * NHT + kMlaWaves - 1) / kMlaWaves;
        f32x4 x[NU][4];
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int u = min(wave + kMlaWaves * i, NS * NHT - 1), s = u / NHT, ht = u % NHT;
            const float *base = s < NSL ? q_prime + 64 * s : q_pe;
            const int width = s < NSL ? R : P;
#pragma unroll
            for (int r = 0; r < 4; r++) x[i][r] = mla_load4(base + ((unsigned)min(h0 + 16 * ht + 4 * r + g, H - 1) * width + 4 * n));
        }
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int u = min(wave + kMlaWaves * i, NS * NHT - 1), s = u / NHT, ht = u % NHT;
            bf16x8 hi[2], lo[2];
#pragma unroll
            for (int r = 0; r < 4; r++) x[i][r] *= qscale;
            mla_operands(x[i], buf, lane, hi, lo);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                sq[2 * s + k][ht][0][lane] = __builtin_bit_cast(uint4, hi[k]);
                sq[2 * s + k][ht][1][lane] = __builtin_bit_cast(uint4, lo[k]);
            }
        }
    }

    f32x4 o[4][NHT];   // lane (channel slot n, g): heads 16 ht + 4 g + i, channel 64 wave + 4 n + j
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int ht = 0; ht < NHT; ht++) o[j][ht] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run[NHT], l_run[NHT];   // of head 16 ht + n: maximum over everything seen, this lane's part of the sum
#pragma unroll
    for (int ht = 0; ht < NHT; ht++) m_run[ht] = neg_inf(), l_run[ht] = 0.f;

    f32x4 kr[D][4];
    // step s of the keys of the round that starts at r0 (rows past the cache's end: its last one, masked below)
    auto fetch_k = [&](int r0, int s) __attribute__((always_inline)) {
        const float *base = s < NSL ? latent + (size_t)r0 * R + 64 * s : rope_k + (size_t)r0 * P;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const unsigned row = min(WPOS * wave + 4 * r + g, L - 1 - r0);
            kr[s % D][r] = mla_load4(base + (row * (s < NSL ? R : P) + 4 * n));
        }
    };
    f32x4 vr[2][8];
    auto fetch_v = [&](int r0, int ks, int slot) __attribute__((always_inline)) {
        const float *base = latent + (size_t)r0 * R;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const unsigned row = min(32 * ks + (e < 4 ? 4 * g + e : 12 + 4 * g + e), L - 1 - r0);
            vr[slot][e] = mla_load4(base + (row * R + 64 * wave + 4 * n));
        }
    };
    bool mine = p0 + WPOS * wave < p1;   // whether the wave has positions in the round
    if (mine) {
#pragma unroll
        for (int s = 0; s < D; s++) fetch_k(p0, s);
    }
    __syncthreads();

    for (int r0 = p0; r0 < p1; r0 += ROUND) {
        const int npos = min(p1 - r0, ROUND);
        const int pairs = (npos + 63) / 64;   // of 32-position steps of the values
        // ---- scores ---------------------------------------------------------------------------------------------
        f32x4 sc[NHT];   // rows = positions 4 g + i, column = head n (log2 units)
        if (mine) {
#pragma unroll
            for (int ht = 0; ht < NHT; ht++) sc[ht] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < NS; s++) {
                bf16x8 kh[2], kl[2];
                mla_operands(kr[s % D], buf, lane, kh, kl);
                if (s + D < NS) fetch_k(r0, s + D);
                if (s == NS - D) fetch_v(r0, 0, 0);
                if (s == NS - D + 1) fetch_v(r0, 1, 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < 2; k++)
#pragma unroll
                    for (int ht = 0; ht < NHT; ht++) {
                        const bf16x8 qh = as_bf16x8(sq[2 * s + k][ht][0][lane]), ql = as_bf16x8(sq[2 * s + k][ht][1][lane]);
                        sc[ht] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kl[k], qh, sc[ht], 0, 0, 0);
                        sc[ht] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh[k], ql, sc[ht], 0, 0, 0);
                        sc[ht] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh[k], qh, sc[ht], 0, 0, 0);
                    }
            }
#pragma unroll
            for (int ht = 0; ht < NHT; ht++) {
                float mb = neg_inf();
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (r0 + WPOS * wave + 4 * g + i >= p1) sc[ht][i] = neg_inf();
                    mb = fmaxf(mb, sc[ht][i]);
                }
                mb = rows_max(mb);
                if (g == 0) smax[16 * ht + n][wave] = mb;
            }
        } else {
            fetch_v(r0, 0, 0);
            fetch_v(r0, 1, 1);
#pragma unroll
            for (int ht = 0; ht < NHT; ht++) {
                sc[ht] = f32x4{neg_inf(), neg_inf(), neg_inf(), neg_inf()};
                if (g == 0) smax[16 * ht + n][wave] = neg_inf();
            }
        }
        __syncthreads();
        // ---- probabilities ----------------------------------------------------------------------------------------
        float alpha[NHT];
#pragma unroll
        for (int ht = 0; ht < NHT; ht++) {
            const f32x4 a = mla_load4(&smax[16 * ht + n][0]), b = mla_load4(&smax[16 * ht + n][4]);
            const float m = fmaxf(m_run[ht], fmaxf(fmaxf(fmaxf(a[0], a[1]), fmaxf(a[2], a[3])), fmaxf(fmaxf(b[0], b[1]), fmaxf(b[2], b[3]))));
            alpha[ht] = fast_exp2(m_run[ht] - m);   // 0 in the first round
            m_run[ht] = m;
            float p[4];
#pragma unroll
            for (int i = 0; i < 4; i++) p[i] = fast_exp2(sc[ht][i] - m);
            l_run[ht] = l_run[ht] * alpha[ht] + ((p[0] + p[1]) + (p[2] + p[3]));
            uint2 ph, pl;
            split_pair(p[0], p[1], ph.x, pl.x);
            split_pair(p[2], p[3], ph.y, pl.y);
            reinterpret_cast<uint2 *>(&sp[wave >> 1][ht][0][lane])[wave & 1] = ph;
            reinterpret_cast<uint2 *>(&sp[wave >> 1][ht][1][lane])[wave & 1] = pl;
        }
        if (r0 != p0) {
#pragma unroll
            for (int ht = 0; ht < NHT; ht++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float a = __shfl(alpha[ht], 4 * g + i, 64);
#pragma unroll
                    for (int j = 0; j < 4; j++) o[j][ht][i] *= a;
                }
        }
        __syncthreads();
        // ---- values -------------------------------------------------------------------------------------------------
        auto accumulate = [&](int ks, int slot) __attribute__((always_inline)) {
            bf16x8 vh[4], vl[4];
#pragma unroll
            for (int j = 0; j < 4; j++)
                mla_split8(f32x4{vr[slot][0][j], vr[slot][1][j], vr[slot][2][j], vr[slot][3][j]},
                           f32x4{vr[slot][4][j], vr[slot][5][j], vr[slot][6][j], vr[slot][7][j]}, vh[j], vl[j]);
            if (ks + 2 < 2 * pairs) fetch_v(r0, ks + 2, slot);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ht = 0; ht < NHT; ht++) {
                const bf16x8 ph = as_bf16x8(sp[ks][ht][0][lane]), pl = as_bf16x8(sp[ks][ht][1][lane]);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    o[j][ht] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl, vl[j], o[j][ht], 0, 0, 0);   // (without it the result is 5 % further off)
                    o[j][ht] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph, vl[j], o[j][ht], 0, 0, 0);
                    o[j][ht] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl, vh[j], o[j][ht], 0, 0, 0);
                    o[j][ht] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph, vh[j], o[j][ht], 0, 0, 0);
                }
            }
        };
        const int next = r0 + ROUND;
        for (int pr = 0; pr + 1 < pairs; pr++) {
            accumulate(2 * pr, 0);
            accumulate(2 * pr + 1, 1);
        }
        mine = next + WPOS * wave < p1;
        if (mine) {
#pragma unroll
            for (int s = 0; s < D; s++) fetch_k(next, s);
        }
        accumulate(2 * pairs - 2, 0);
        accumulate(2 * pairs - 1, 1);
    }

    // ---- partials ------------------------------------------------------------------------------------------------------
#pragma unroll
    for (int ht = 0; ht < NHT; ht++) {
        const float l = rows_sum(l_run[ht]);
        if (g == 0) ssum[wave][16 * ht + n] = l;
        if (h0 + 16 * ht < H) {
            const size_t pid = (size_t)(group * NHT + ht) * nsplit + split;
            float *po = part_o + (pid * 16 + 4 * g) * R + 64 * wave + 4 * n;
#pragma unroll
            for (int i = 0; i < 4; i++) *reinterpret_cast<f32x4 *>(po + i * R) = f32x4{o[0][ht][i], o[1][ht][i], o[2][ht][i], o[3][ht][i]};
            if (wave == 0 && g == 0) part_ml[pid * 32 + n] = m_run[ht];
        }
    }
    __syncthreads();
    if (tid < HW && h0 + (tid & ~15) < H) {
        float l = 0.f;
#pragma unroll
        for (int w = 0; w < kMlaWaves; w++) l += ssum[w][tid];
        part_ml[((size_t)(group * NHT + tid / 16) * nsplit + split) * 32 + 16 + (tid & 15)] = l;
    }
}

__device__ inline bf16x8 mla_lds8(const void *p) { return *reinterpret_cast<const bf16x8 *>(p); }

typedef short mla_i16x4 __attribute__((ext_vector_type(4)));
typedef short mla_i16x8 __attribute__((ext_vector_type(8)));
// Transposing 8-byte LDS read (see the layout note above).
__device__ inline mla_i16x4 mla_lds_tr(const unsigned char *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (mla_i16x4 __attribute__((address_space(3))) *)(__attribute__((address_space(3))) unsigned char *)p);
}

static constexpr int kMlaBlk = 16;    // positions per block
static constexpr int kMlaHG = 4;      // 16-head groups per workgroup
static constexpr float kMlaLazy = 8.f;
static constexpr int kMlaMayMove = 0x2 | 0x4 | 0x10 | 0x200;   // sched_barrier: vector and scalar ALU, memory and LDS writes may cross

template <int R, int P>
__global__ __launch_bounds__(kMlaHG * 128) void mla_stream_kernel(
    const float *__restrict__ q_prime, const float *__restrict__ q_pe, const float *__restrict__ latent,
    const float *__restrict__ rope_k, int H, int L, int blocks_per_split, float qscale,
    float *__restrict__ part_o, float *__restrict__ part_ml) {
    constexpr int HG = kMlaHG, NROLE = HG * 64;
    constexpr int DK = R + P;
    constexpr int KROW = DK + 16;         // row stride (bf16): 1184 bytes
    constexpr int NS = DK / 32;           // 32-wide steps of the score contraction
    constexpr int NT = R / 16;            // output tiles (16 channels each)
    static_assert(NROLE == 256 && R == 512 && P == 64, "the staging maps 256 threads per role onto a 16 x (512 + 64) block");
    constexpr int KPLANE = kMlaBlk * KROW * 2;           // bytes of one plane (hi or lo) of a block
    constexpr int KBUF = 2 * KPLANE;                     // one buffer
    constexpr int VPOS = 6;              // positions of a block whose latent rows the value waves stage; the score waves take the rest
    __shared__ __attribute__((aligned(16))) unsigned char smem[3 * KBUF];
    __shared__ __attribute__((aligned(16))) uint16_t pbuf[2][HG][2][16][kMlaBlk];  // weights [buffer][group][hi|lo][head][position]
    __shared__ float abuf[2][HG][16];                                             // rescale factor of a block, per head

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, g = lane >> 4;
    const bool score_role = wave < HG;
    const int hgl = wave % HG, rtid = tid % NROLE;
    const int split = blockIdx.x, nsplit = gridDim.x;
    const int nhg = (H + 15) / 16;
    const int hg = blockIdx.y * HG + hgl;
    const bool active = hg < nhg;  // a wave past the last head group repeats the last head and stores nothing

    const int nblk = (L + kMlaBlk - 1) / kMlaBlk;
    const int b0 = split * blocks_per_split;
    const int b1 = min(b0 + blocks_per_split, nblk);
    const size_t pid = (size_t)hg * nsplit + split;
    if (b0 >= b1) {
        if (active && score_role && g == 0) {
            part_ml[pid * 32 + n] = neg_inf();
            part_ml[pid * 32 + 16 + n] = 0.f;
        }
        return;
    }
    auto clampb =[&](int b) { return min(b, b1 - 1); };  // requests past the range repeat its last block; nobody reads them
    // block b lives in buffer (b - b0) % 3
    auto bufof =[&](int b) { return smem + ((b - b0) % 3) * KBUF; };
    // A block's rows are requested two blocks before they are written to LDS, in two sets of registers, and 16 bytes a lane: with
    // that and the operands read ahead of the products (below) 128 heads over 32768 positions take 43.7 us instead of 46.5.
    // (Neither by itself gains: a block's 3.9 k clocks are 1.9 k of matrix time at a clock that the matrix load pulls down, 1 k of
    // conversion and 1.4 k of LDS reads at least.  Tried and not kept: 32 heads a wave over half of the channels, half the LDS
    // reads but a barrier more a block (50.2 us), either role's waves ahead of the other's by priority, 4 or 8 rows staged by the value waves.)
    const int srow = rtid >> 7, scol = rtid & 127;   // 128 threads x 4 channels a latent row
    const std::integral_constant<int, 0> zero{};
    const std::integral_constant<int, 1> one{};
    auto put4 = [&](unsigned char *at, const f32x4 &x) __attribute__((always_inline)) {
        uint2 hi, lo;
        split_pair(x[0], x[1], hi.x, lo.x);
        split_pair(x[2], x[3], hi.y, lo.y);
        *reinterpret_cast<uint2 *>(at) = hi;
        *reinterpret_cast<uint2 *>(at + KPLANE) = lo;
    };

    if (score_role) {
        // ================= scores and softmax of head group hgl =================
        // staging: four channels of one rotary key, and of every second of the latent rows that the value waves leave
        constexpr int NR = (kMlaBlk - VPOS) / 2;
        f32x4 rraw[2], lraw[2][NR];   // [block % 2 from b0 + 1 on]
        auto fetch =[&](int b, auto slot) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
            rraw[S] = mla_load4(rope_k + (size_t)min(clampb(b) * kMlaBlk + (rtid >> 4), L - 1) * P + 4 * (rtid & 15));
#pragma unroll
            for (int j = 0; j < NR; j++)
                lraw[S][j] = mla_load4(latent + (size_t)min(clampb(b) * kMlaBlk + VPOS + 2 * j + srow, L - 1) * R + 4 * scol);
        };
        auto commit =[&](int b, auto slot) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
            unsigned char *base = bufof(b);
            put4(base + ((rtid >> 4) * KROW + R + 4 * (rtid & 15)) * 2, rraw[S]);
#pragma unroll
            for (int j = 0; j < NR; j++) put4(base + ((VPOS + 2 * j + srow) * KROW + 4 * scol) * 2, lraw[S][j]);
        };
        fetch(b0, zero);
        // the 16 queries as B operands: lane (n, g) holds head n, channels 32 s + 8 g .. + 7 of [q' | q_pe].  Read row by row in whole
        // lines and exchanged through LDS, three 64-channel steps at a time (requested in operand order they took 3 us of the launch).
        bf16x8 qh[NS], ql[NS];
        {
            static_assert(kMlaHG * 16 * kMlaRow * 4 <= KBUF, "the exchange buffers fit one block buffer");
            float *buf = reinterpret_cast<float *>(smem + 2 * KBUF) + hgl * 16 * kMlaRow;   // block b0 + 2 is written after the barriers below
            f32x4 x[3][4];
#pragma unroll
            for (int t = 0; t < DK / 64; t += 3) {
#pragma unroll
                for (int u = 0; u < 3; u++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const unsigned head = min(hg * 16 + 4 * r + g, H - 1);
                        x[u][r] = (64 * (t + u) < R ? mla_load4(q_prime + 64 * (t + u) + (head * R + 4 * n)) : mla_load4(q_pe + (head * P + 4 * n))) * qscale;
                    }
#pragma unroll
                for (int u = 0; u < 3; u++) {
                    bf16x8 hi[2], lo[2];
                    mla_operands(x[u], buf, lane, hi, lo);
#pragma unroll
                    for (int k = 0; k < 2; k++) qh[2 * (t + u) + k] = hi[k], ql[2 * (t + u) + k] = lo[k];
                }
            }
        }
        float m_ref = neg_inf(), l_sum = 0.f;
        const int kr_rd = (n * KROW + 8 * g) * 2;   // [hi][position n][8 g]; lo at + KPLANE; step s at + 64 s
        commit(b0, zero);
        fetch(b0 + 1, zero);
        fetch(b0 + 2, one);
        __syncthreads();
        // iteration b0 - 1: block b0 is scored, nothing is accumulated yet; then one iteration per block
        auto iteration = [&](int it, auto slot) __attribute__((always_inline)) {
            const int b = it + 1;   // the block scored in this iteration
            const unsigned char *base = bufof(b);
            f32x4 sc = {0.f, 0.f, 0.f, 0.f};  // rows = positions 4g + i, column = head n (log2 units)
            // operands two to four steps ahead of the products (left alone the compiler reads them one step ahead, and every step
            // waits for LDS); only matrix instructions and LDS reads keep their places
            constexpr int GS = 2;
            bf16x8 ah[2][GS], al[2][GS];
            auto read_keys = [&](int q) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < GS; i++) {
                    ah[q & 1][i] = mla_lds8(base + kr_rd + 64 * (GS * q + i));
                    al[q & 1][i] = mla_lds8(base + kr_rd + 64 * (GS * q + i) + KPLANE);
                }
            };
            static_assert(NS % GS == 0, "whole groups");
            read_keys(0);
#pragma unroll
            for (int q = 0; q < NS / GS; q++) {
                if (q + 1 < NS / GS) read_keys(q + 1);
                __builtin_amdgcn_sched_barrier(kMlaMayMove);
#pragma unroll
                for (int i = 0; i < GS; i++) {
                    sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[q & 1][i], qh[GS * q + i], sc, 0, 0, 0);
                    sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[q & 1][i], ql[GS * q + i], sc, 0, 0, 0);
                    sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[q & 1][i], qh[GS * q + i], sc, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(kMlaMayMove);
            }
            // block it + 2 (its buffer was accumulated from in the previous iteration); block it + 4 is requested
            commit(it + 2, slot);
            fetch(it + 4, slot);
            {
                const int pos0 = b * kMlaBlk + 4 * g;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (pos0 + i >= L) sc[i] = neg_inf();
                float mb = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
                mb = rows_max(mb);
                // Move the reference point only when some head's maximum has moved far: weights stay
                // below 2^kMlaLazy, and the reference point cancels in the merge.
                float alpha = 1.f;
                if (__any(mb > m_ref + kMlaLazy)) {
                    const float m_new = fmaxf(m_ref, mb);
                    alpha = fast_exp2(m_ref - m_new);
                    m_ref = m_new;
                    l_sum *= alpha;
                }
                float p[4];
#pragma unroll
                for (int i = 0; i < 4; i++) p[i] = fast_exp2(sc[i] - m_ref);
                l_sum += (p[0] + p[1]) + (p[2] + p[3]);
                uint2 ph, pl;
                split_pair(p[0], p[1], ph.x, pl.x);
                split_pair(p[2], p[3], ph.y, pl.y);
                *reinterpret_cast<uint2 *>(&pbuf[b & 1][hgl][0][n][4 * g]) = ph;
                *reinterpret_cast<uint2 *>(&pbuf[b & 1][hgl][1][n][4 * g]) = pl;
                if (g == 0) abuf[b & 1][hgl][n] = alpha;
            }
            __syncthreads();
        };
        for (int it = b0 - 1; it < b1 - 1; it += 2) {
            iteration(it, zero);
            if (it + 1 < b1 - 1) iteration(it + 1, one);
        }
        l_sum = rows_sum(l_sum);
        if (active && g == 0) {
            part_ml[pid * 32 + n] = m_ref;
            part_ml[pid * 32 + 16 + n] = l_sum;
        }
        __syncthreads();  // iteration b1 - 1: the value waves accumulate the last block
    } else {
        // ================= values of head group hgl =================
        // staging: four channels of every second of the block's first VPOS latent rows
        f32x4 raw[2][VPOS / 2];
        auto fetch =[&](int b, auto slot) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
#pragma unroll
            for (int j = 0; j < VPOS / 2; j++)
                raw[S][j] = mla_load4(latent + (size_t)min(clampb(b) * kMlaBlk + 2 * j + srow, L - 1) * R + 4 * scol);
        };
        auto commit =[&](int b, auto slot) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
            unsigned char *base = bufof(b);
#pragma unroll
            for (int j = 0; j < VPOS / 2; j++) put4(base + ((2 * j + srow) * KROW + 4 * scol) * 2, raw[S][j]);
        };
        f32x4 o[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        // A operand of tile t: lane (j, g) points at position 8 (g & 1) + j/4 [+ 4], channels 16 t + 4 (j % 4) .. + 3,
        // in the hi plane for g < 2 and the lo plane otherwise; the transposing read hands lane j channel 16 t + j
        // at positions 8 (g & 1) .. + 3 [+ 4]
        const bool hi_slots = g < 2;
        const int tr_rd = (hi_slots ? 0 : KPLANE) + ((8 * (g & 1) + (n >> 2)) * KROW + 4 * (n & 3)) * 2;
        fetch(b0, zero);
        commit(b0, zero);
        fetch(b0 + 1, zero);
        fetch(b0 + 2, one);
        __syncthreads();
        // iteration b0 - 1: no weights yet
        commit(b0 + 1, zero);
        fetch(b0 + 3, zero);
        __syncthreads();
        auto iteration = [&](int it, auto slot) __attribute__((always_inline)) {
            commit(it + 2, slot);    // its buffer held block it - 1
            fetch(it + 4, slot);
            const unsigned char *base = bufof(it) + tr_rd;
            // lane (n, g): weights of head n at positions 8 (g & 1) .. + 7
            const bf16x8 pb_h = mla_lds8(&pbuf[it & 1][hgl][0][n][8 * (g & 1)]);
            const bf16x8 pb_l = mla_lds8(&pbuf[it & 1][hgl][1][n][8 * (g & 1)]);
            const float alpha = abuf[it & 1][hgl][n];
            if (__any(alpha != 1.f)) {
#pragma unroll
                for (int t = 0; t < NT; t++) o[t] *= alpha;
            }
            // operands four tiles ahead of the products, as above
            constexpr int GT = 4;
            bf16x8 a[2][GT];
            auto read_values = [&](int q) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < GT; i++) {
                    const mla_i16x4 a0 = mla_lds_tr(base + 32 * (GT * q + i));
                    const mla_i16x4 a1 = mla_lds_tr(base + 32 * (GT * q + i) + 4 * KROW * 2);
                    const mla_i16x8 a8 = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
                    a[q & 1][i] = __builtin_bit_cast(bf16x8, a8);
                }
            };
            read_values(0);
#pragma unroll
            for (int q = 0; q < NT / GT; q++) {
                if (q + 1 < NT / GT) read_values(q + 1);
                __builtin_amdgcn_sched_barrier(kMlaMayMove);
#pragma unroll
                for (int i = 0; i < GT; i++) o[GT * q + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q & 1][i], pb_l, o[GT * q + i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < GT; i++) o[GT * q + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q & 1][i], pb_h, o[GT * q + i], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(kMlaMayMove);
            }
            __syncthreads();
        };
        for (int it = b0; it < b1; it += 2) {
            iteration(it, one);
            if (it + 1 < b1) iteration(it + 1, zero);
        }
        // o[t][i] is channel 16 t + 4g + i of head n
        if (active) {
            float *po = part_o + (pid * 16 + n) * R + 4 * g;
#pragma unroll
            for (int t = 0; t < NT; t++) *reinterpret_cast<f32x4 *>(po + 16 * t) = o[t];
        }
    }
}

bool mla_shape_supported(int kv_lora_rank, int qk_rope_head_dim) {
    return kv_lora_rank == 512 && qk_rope_head_dim == 64;
}

// Partition of the heads and of the cache over workgroups, a workgroup per CU.  Which kernel (us a layer, one call after the
// other / three sequences side by side, in brackets the streaming kernel with its queries read in operand order):
//   rounds, 16 heads  where one round of 128 positions is enough: 128 heads over 200 positions 11.5 / 7.6 (17.0 / 8.4), 1500
//                     14.8 / 11.1 (26.1 / 15.1), 4096 17.9 / 13.7, where 32 heads take 20.8 / 13.9 and at 4600 22.2 / 15.3 against 21.3 / 16.7;
//                     64 over 2000 14.5 / 10.8 (24.0 / 11.4), 8192 18.7 / 13.7
//                     (28.8 / 22.6).  17 to 32 heads, whose two groups share an L2: up to three rounds, 30 over 24576 21.7 / 20.3 (the
//                     present streaming kernel 29.1 / 24.4), 40000 29.2 / 30.6 (35.0 / 31.3), 49152 32.9 / 36.1 (39.4 / 35.0),
//                     but 55000 39.3 / 40.2 (41.1 / 38.2).  Up to 16 heads, where nobody shares the second read of
//                     the rows: up to 80 positions a CU, from where on it is a draw: 16 over 16384 19.3 / 15.3 (streaming 23.0 / 16.3), 18400 23.4 / 16.6 (23.6 /
//                     16.5), 20480 25.8 / 17.8 (25.3 / 18.3), 22500 25.1 / 19.1 (24.8 / 20.2), but 32768 32.0 / 24.8 (30.5 / 25.3)
//   rounds, 32 heads  up to two rounds: 128 over 8192 24.3 / 18.5 (28.6 / 24.4), 12000 26.6 / 23.2 (streaming 30.4 / 26.2), 16384 30.9 / 28.0 (31.7 / 31.0), 18000
//                     34.8 / 32.4 (34.8 / 32.5), but 24000 40.8 / 39.8 (41.5 / 39.4); 64 over 32768 33.8 / 31.3 (38.0 / 36.5)
//   streaming, 64     beyond: 128 over 32768 43.6 / 44.8 (47.9 / 48.7), 65536 76.5 / 74.7 (79.5 / 79.8)
MlaPlan mla_plan(int H, int L, int num_cus, int forced_splits) {
    MlaPlan p;
    p.nhg = (H + 15) / 16;
    auto rounds = [&](int tiles) {   // of a workgroup that serves `tiles` head groups
        const int64_t groups = (p.nhg + tiles - 1) / tiles;
        return (L * groups + 128 * (int64_t)num_cus - 1) / (128 * (int64_t)num_cus);
    };
    const bool few = p.nhg == 1 ? L <= 80 * (int64_t)num_cus : rounds(1) <= (p.nhg == 2 ? 3 : 1);
    p.head_tiles = few ? 1 : p.nhg > 2 && rounds(2) <= 2 ? 2 : kMlaHG;
    p.groups = (p.nhg + p.head_tiles - 1) / p.head_tiles;
    // (rounded down for the rounds kernel: with 48 heads' three groups one workgroup too many would run alone)
    int splits = forced_splits > 0 ? forced_splits : p.head_tiles == kMlaHG ? (num_cus + p.groups - 1) / p.groups : num_cus / p.groups;
    splits = std::max(1, std::min(splits, 1024));
    // whole blocks of 16 positions; a share of less than two leaves more partials than it saves time
    const int blocks = (L + 15) / 16;
    int per = (blocks + splits - 1) / splits;
    if (forced_splits <= 0 && p.head_tiles < kMlaHG) per = std::max(per, 2);
    p.per_split = 16 * per;
    p.splits = (blocks + per - 1) / per;
    return p;
}

size_t mla_workspace_o_elems(const MlaPlan &p, int R) { return (size_t)p.nhg * p.splits * 16 * R; }
size_t mla_workspace_ml_elems(const MlaPlan &p) { return (size_t)p.nhg * p.splits * 32; }

int launch_mla_sdpa_folded(hipStream_t stream, int H, int R, int P, int L, float softmax_scale,
                           const float *q_prime, const float *q_pe, const float *latent, const float *rope_k,
                           float *out, const SdpaWorkspace &ws, const MlaPlan &plan) {
    if (!mla_shape_supported(R, P))
        return fail(MFA_ERR_SHAPE, "latent attention: kv_lora_rank %d / qk_rope_head_dim %d not built (512 / 64)", R, P);
    if (H <= 0 || L <= 0) return fail(MFA_ERR_INVALID, "latent attention: num_heads %d, cache_len %d", H, L);
    if (ws.part_o_elems < mla_workspace_o_elems(plan, R) || ws.part_ml_elems < mla_workspace_ml_elems(plan))
        return fail(MFA_ERR_INVALID, "latent attention: workspace too small for %d splits", plan.splits);
    const float qscale = softmax_scale * 1.4426950408889634f;  // scores in log2 units
    if (plan.head_tiles == kMlaHG) {
        launch_kernel(mla_stream_kernel<512, 64>, dim3(plan.splits, plan.groups), dim3(kMlaHG * 128), stream, q_prime, q_pe, latent, rope_k, H, L, plan.per_split / kMlaBlk, qscale, ws.part_o, ws.part_ml);
    } else {
        const dim3 grid((unsigned)((plan.splits + 7) / 8 * 8 * plan.groups));   // see mla_rounds_kernel: a split's workgroups on one XCD
#define MFA_MLA(HT)                                                                                                \
    launch_kernel(mla_rounds_kernel<HT>, grid, dim3(kMlaWaves * 64), stream, q_prime, q_pe, latent, rope_k, \
                  H, L, plan.splits, plan.groups, plan.per_split, qscale, ws.part_o, ws.part_ml)
        if (plan.head_tiles == 1) MFA_MLA(1);
        else MFA_MLA(2);
#undef MFA_MLA
    }
    MFA_HIP(hipGetLastError());
    return launch_sdpa_merge(stream, ws, plan.splits, /*hpk=*/H, /*Hq=*/H, plan.nhg, R, /*n_tok=*/1,
                             /*gate=*/nullptr, out);
}

}  // namespace mfa
