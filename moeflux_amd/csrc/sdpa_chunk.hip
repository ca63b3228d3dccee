// Causal attention of a prompt chunk over a tiled bf16 KV cache, on 32x32 matrix tiles.
//
// The reference has no batched prefill: eval_prompt is a token loop
// (crates/moeflux/src/riir/mod.rs:1196-1214) whose every token runs the decode chain of
// crates/moeflux/src/riir/sdpa.rs:63-172.  Row t of the chunk equals that decode at
// kv_len = kv_len0 + t + 1.
//
// A wave owns 32 query rows (rows of one kv head: token-major, then the hpk query heads that share
// it); its query operands (a bf16 high and low part) and its output tiles stay in registers.  The
// cache is walked in blocks of 32 positions, copied to LDS by asynchronous loads (K and V lie in
// operand order in memory already, and the pieces of the 16-wide tiles are operands of the 32-wide
// ones as they are: a 16-byte unit is 8 channels of a key, or 8 positions of a value channel that are
// the score tile's own).  A KiB of LDS operand feeds two 32x32x16 products, 64 clocks of the matrix core; of
// 16-row groups it fed half as much, and the four SIMDs asked for all the LDS could give.  The scores of a
// block are formed beside the soft-max of the one before, two blocks to a barrier where LDS allows.
// Rows that leave CUs idle split the cache (sdpa_chunk_plan).
//
// What bounds it: behind a long cache the matrix cores at the rate they sustain.  512 tokens of 32 heads
// of 128 behind 32768 positions, three sequences side by side: 580 us with 16-row groups, 429 with this kernel, 384 with its
// soft-max left out (one call after the other, at a lower clock: 664 and 502) (both parts of query and probabilities are products, so 2.75e11 operations are 5.5e11 executed: 1.4 PFLOP/s).
// Over short caches launch, query, first block and epilogue: 512 tokens from an empty cache 17 us,
// of which the longest workgroup's eight blocks are 7.
#include <cmath>

#include "sdpa_wave.h"

namespace mfa {

typedef __attribute__((ext_vector_type(16))) float f32x16;

// One 1 KiB piece from memory to LDS without passing through registers: lane l's 16 bytes land at
// lds + 16 l.  As assembly, because the compiler waits for every such load in flight ahead of every LDS
// read; the kernel's own wait (wait_pieces) counts them.
// m0 is a clobber: a builtin that needs it then sets it again behind this.  (The compiler's warning is that it does
// not keep a reserved register's value across the statement, which is what is wanted.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ inline void copy_piece(const uint4 *src, unsigned lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "m0", "memory");
}
#pragma clang diagnostic pop
template <int N> __device__ inline void wait_pieces_and_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

struct ChunkArgs {
    const uint16_t *k, *v;
    size_t plane_elems;
    ChunkQuery in;
    int hpk, Hq, n_tok;
    int64_t kv_len0;
    float qscale;
    float *out;
    float *part_o, *part_ml;
    int nrt;             // row tiles per kv head
    int nsplit, bps;     // splits of the cache, blocks of 32 positions per split
    int ncombo;          // kv heads * splits
    int contiguous;      // 1: an XCD takes whole (kv head, split) pairs
};

// The query rows from their raw projection: RMS norm over the head and the rotation of its first quarter
// (full_attn_forward.rs:238-323), the arithmetic of attn_prologue.h.  Lane (n, h) holds channels 16 s + 8 h .. + 3 of
// its row in x[s] and the next four in y[s], lane (n, 1 - h) the rest of the row; the rotated quarter's pairs
// (i, i + D / 8) are D / 128 k-steps apart and so a lane's own.
template <int D> struct RowNorm {
    static constexpr int NS = D / 16, ROT = D / 128;   // k-steps of the row, and of one half of its rotated channels
    uint4 w[NS], cs[ROT][4];

    // asked for with the rows themselves: behind them they were 3 us of a 20 us launch
    __device__ __attribute__((always_inline)) inline void request(const ChunkQuery &in, int token, int h) {
#pragma unroll
        for (int s = 0; s < NS; s++) w[s] = vec_load((const uint4 *)(in.q_norm + 16 * s + 8 * h));
#pragma unroll
        for (int s = 0; s < ROT; s++)
#pragma unroll
            for (int i = 0; i < 4; i++) cs[s][i] = vec_load((const uint4 *)(in.table + ((size_t)token * (D / 8) + 16 * s + 8 * h + 2 * i)));
    }
    __device__ __attribute__((always_inline)) inline void apply(uint4 (&x)[NS], uint4 (&y)[NS], float eps) const {
        auto at = [&](int s, int e) -> unsigned & { return e < 4 ? (e == 0 ? x[s].x : e == 1 ? x[s].y : e == 2 ? x[s].z : x[s].w)
                                                                 : (e == 4 ? y[s].x : e == 5 ? y[s].y : e == 6 ? y[s].z : y[s].w); };
        auto part = [](const uint4 &u, int i) { return i == 0 ? u.x : i == 1 ? u.y : i == 2 ? u.z : u.w; };
        float ss = 0.f;
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float v = __builtin_bit_cast(float, at(s, e));
                ss += v * v;
            }
        float other = ss;
        rows_swap32(ss, other);
        ss += other;
        const float inv_rms = 1.0f / sqrtf(ss / (float)D + eps);
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const unsigned pair = part(w[s], e / 2);
                const float wt = __builtin_bit_cast(float, e % 2 ? pair & 0xffff0000u : pair << 16);
                at(s, e) = __builtin_bit_cast(unsigned, __builtin_bit_cast(float, at(s, e)) * inv_rms * wt);
            }
#pragma unroll
        for (int s = 0; s < ROT; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float c = __builtin_bit_cast(float, part(cs[s][e / 2], e % 2 * 2)), sn = __builtin_bit_cast(float, part(cs[s][e / 2], e % 2 * 2 + 1));
                const float a = __builtin_bit_cast(float, at(s, e)), b = __builtin_bit_cast(float, at(s + ROT, e));
                at(s, e) = __builtin_bit_cast(unsigned, a * c - b * sn);
                at(s + ROT, e) = __builtin_bit_cast(unsigned, a * sn + b * c);
            }
    }
};

template <int D, int RW, int KS, int G, bool SPLIT, bool RAW>
__global__ __launch_bounds__(64 * RW * KS, D == 256 ? 1 : 2) void sdpa_chunk_kernel(const ChunkArgs a) {
    constexpr int NS = D / 16;          // k-steps of the scores, 1 KiB pieces of a block's K and of its V
    constexpr int NT = D / 32;          // 32-wide output tiles
    constexpr int PIECES = NS / RW;     // pieces of K (and of V) a wave copies per block
    constexpr int NBUF = 2 * G;         // buffers of K and of V: G blocks in use, G on their way
    constexpr int BUF_U4 = NS * 64;
    static_assert(NS % RW == 0, "the waves of a set copy whole pieces");
    __shared__ uint4 lds[KS][2][NBUF][BUF_U4];
    __shared__ float s_m[KS][RW][32], s_l[KS][RW][32];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = wave % RW, ks = wave / RW;
    const int n = lane & 31, h = lane >> 5;
    int combo, rt;
    {
        const int bid = blockIdx.x, total = gridDim.x;
        if (a.contiguous) {
            const int x = bid & 7, per = total >> 3, rem = total & 7;
            const int l = x * per + (x < rem ? x : rem) + (bid >> 3);
            combo = l / a.nrt;
            rt = l % a.nrt;
        } else {
            combo = bid % a.ncombo;
            rt = a.nrt - 1 - bid / a.ncombo;
        }
    }
    const int kvh = combo / a.nsplit, split = combo % a.nsplit;
    const int nrows = a.n_tok * a.hpk;
    const int tile_row0 = rt * 32 * RW;
    // blocks of the tile's last row, and the share of this split
    int last = tile_row0 + 32 * RW - 1;
    if (last > nrows - 1) last = nrows - 1;
    const int nblk = (int)((a.kv_len0 + last / a.hpk + 1 + 31) / 32);
    const int b0 = split * a.bps;
    int b1 = SPLIT ? b0 + a.bps : nblk;
    if (b1 > nblk) b1 = nblk;
    // this lane's row
    const int row0 = tile_row0 + rw * 32, rr = row0 + n;
    const bool ok = rr < nrows;
    const size_t part = (((size_t)kvh * a.nrt + rt) * a.nsplit + split) * RW + rw;   // this wave's partial
    if (SPLIT && b0 >= b1) {
        if (ks == 0 && h == 0) {
            a.part_ml[part * 64 + n] = neg_inf();
            a.part_ml[part * 64 + 32 + n] = 0.f;
        }
        return;
    }
    const int nit = (b1 - b0 + KS - 1) / KS;

    const uint4 *kp = reinterpret_cast<const uint4 *>(a.k + (size_t)kvh * a.plane_elems) + lane;
    const uint4 *vp = reinterpret_cast<const uint4 *>(a.v + (size_t)kvh * a.plane_elems) + lane;
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)&lds[ks][0][0][0];
    constexpr unsigned KIND = NBUF * BUF_U4 * 16;
    auto block_of = [&](int it) {
        int b = b0 + it * KS + ks;
        b = b < b1 ? b : b1 - 1;
        return b;
    };
    // K of block it and V of block it - 1 into their buffers (block b's is b % NBUF)
    auto request = [&](int it) __attribute__((always_inline)) {
        const int bk = block_of(it), bv = block_of(it - 1);
        const unsigned kslot = it & (NBUF - 1), vslot = (it - 1) & (NBUF - 1);
        const uint4 *kb = kp + (int64_t)(bk >> 1) * (64 * D / 8) + (bk & 1) * 128;
        const uint4 *vb = vp + (int64_t)bv * (32 * D / 8);
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
            const int li = rw * PIECES + i;   // k-step li / 2 of 32 channels, sub-tile li % 2
            copy_piece(kb + (li >> 1) * 256 + (li & 1) * 64, lds0 + (kslot * NS + li) * 1024);
        }
        if (it == 0) return;
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
            const int li = rw * PIECES + i;
            copy_piece(vb + li * 64, lds0 + KIND + (vslot * NS + li) * 1024);
        }
    };

    // Query operands: lane (n, h) holds channels 16 s + 8 h .. + 7 of its row for every step s.  Rows are read in
    // runs of 32 channels (128 bytes, 8 rows a load) and change lanes through a piece of LDS of the wave's own, in
    // buffers that the first blocks leave free: read in operand order, 32 rows a load, a wave's query takes
    // D / 8 loads of 150 clocks each.
    uint4 *tr = G == 2 ? (rw < 2 ? lds[ks][0][2 + (rw & 1)] : lds[ks][1][1 + (rw & 1)]) : (rw == 0 ? lds[ks][0][1] : lds[ks][1][0]);
    const int tr_row = lane >> 3, tr_chunk = lane & 7;   // row tr_row + 8 j, 16-byte chunk tr_chunk of the run
    const auto tr_at = [](int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); };
    int64_t tr_q[4];
    bool tr_ok[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = row0 + tr_row + 8 * j;
        tr_ok[j] = r < nrows;
        tr_q[j] = tr_ok[j] ? (int64_t)(r / a.hpk) * a.Hq + kvh * a.hpk + r % a.hpk : 0;
    }
    uint4 qh[NS], ql[NS];
    {
        uint4 raw[NT][4];
        std::conditional_t<RAW, RowNorm<D>, int> norm;
        if constexpr (RAW) norm.request(a.in, ok ? rr / a.hpk : 0, h);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) raw[t][j] = vec_load((const uint4 *)(a.in.q + tr_q[j] * a.in.stride + 32 * t + 4 * tr_chunk));
#pragma unroll
        for (int g = 0; g < G; g++) request(g);
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
            for (int j = 0; j < 4; j++) tr[tr_at(tr_row + 8 * j, tr_chunk)] = raw[t][j];
            wave_lds_order();   // (with the one below a layer of 203 tokens behind 3001 takes 58.2 -> 58.7 us at 256 channels: four registers more in scratch)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                qh[2 * t + u] = tr[tr_at(n, 4 * u + 2 * h)];
                ql[2 * t + u] = tr[tr_at(n, 4 * u + 2 * h + 1)];
            }
            wave_lds_order();   // ahead of the next run's writes
        }
        if constexpr (RAW) norm.apply(qh, ql, a.in.eps);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const float4 x = __builtin_bit_cast(float4, qh[s]), y = __builtin_bit_cast(float4, ql[s]);
            split_pair(x.x, x.y, qh[s].x, ql[s].x);
            split_pair(x.z, x.w, qh[s].y, ql[s].y);
            split_pair(y.x, y.y, qh[s].z, ql[s].z);
            split_pair(y.z, y.w, qh[s].w, ql[s].w);
        }
        const unsigned keep = ok ? 0xffffffffu : 0u;   // a row past the chunk's last is all zero
#pragma unroll
        for (int s = 0; s < NS; s++) {
            qh[s].x &= keep; qh[s].y &= keep; qh[s].z &= keep; qh[s].w &= keep;
            ql[s].x &= keep; ql[s].y &= keep; ql[s].z &= keep; ql[s].w &= keep;
        }
    }
    bool q_exact;
    {
        unsigned any = 0;
#pragma unroll
        for (int s = 0; s < NS; s++) any |= (ql[s].x | ql[s].y | ql[s].z | ql[s].w) & 0x7fff7fffu;
        q_exact = __all(any == 0);
    }
    const int64_t limit = ok ? a.kv_len0 + rr / a.hpk + 1 : 0;
    const int64_t limit_min = (row0 + 31 < nrows) ? a.kv_len0 + row0 / a.hpk + 1 : 0;
    int64_t wave_max = 0;
    if (row0 < nrows) {
        const int wl = row0 + 31 < nrows ? row0 + 31 : nrows - 1;
        wave_max = a.kv_len0 + wl / a.hpk + 1;
    }
    // iterations some row of this wave sees: block b0 + it KS + ks begins below wave_max and the split's end
    int nl;
    {
        int64_t wb = (wave_max + 31) / 32;
        if (wb > b1) wb = b1;
        const int64_t left = wb - b0 - ks;
        nl = left > 0 ? (int)((left + KS - 1) / KS) : 0;
    }

    f32x16 o[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[t][i] = 0.f;
    float m_ref = neg_inf(), l_run = 0.f;
    float m_loc = neg_inf();
    const int lane_u4 = ((lane >> 4) & 1) * 64 + (lane >> 5) * 16 + (lane & 15);

    auto qk = [&](auto exact_tag, int slot, f32x16 &s_new) __attribute__((always_inline)) {
        const uint4 *cur = &lds[ks][0][slot][lane_u4];
#pragma unroll
        for (int i = 0; i < 16; i++) s_new[i] = 0.f;
        if constexpr (decltype(exact_tag)::value) {
#pragma unroll
            for (int s = 0; s < NS; s++)
                s_new = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(cur[(s >> 1) * 128 + (s & 1) * 32]), as_bf16x8(qh[s]), s_new, 0, 0, 0);
        } else {
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const bf16x8 kk = as_bf16x8(cur[(s >> 1) * 128 + (s & 1) * 32]);
                s_new = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kk, as_bf16x8(qh[s]), s_new, 0, 0, 0);
                s_new = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kk, as_bf16x8(ql[s]), s_new, 0, 0, 0);
            }
        }
    };
    auto softmax = [&](const f32x16 &x, uint4 (&ph)[2], uint4 (&pl)[2]) __attribute__((always_inline)) {
        const float ref = (m_ref == neg_inf()) ? 0.f : m_ref;
        float e[16];
#pragma unroll
        for (int i = 0; i < 16; i++) e[i] = fast_exp2(fmaf(x[i], a.qscale, -ref));
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            s0 += e[i];
            s1 += e[i + 1];
        }
        l_run += s0 + s1;
        // step j of the value product: slots 0..3 are registers 4 j .., slots 4..7 registers 4 (j + 2) ..
#pragma unroll
        for (int j = 0; j < 2; j++) {
            split_pair(e[4 * j], e[4 * j + 1], ph[j].x, pl[j].x);
            split_pair(e[4 * j + 2], e[4 * j + 3], ph[j].y, pl[j].y);
            split_pair(e[4 * j + 8], e[4 * j + 9], ph[j].z, pl[j].z);
            split_pair(e[4 * j + 10], e[4 * j + 11], ph[j].w, pl[j].w);
        }
    };
    auto pv = [&](int slot, const uint4 (&ph)[2], const uint4 (&pl)[2]) __attribute__((always_inline)) {
        const uint4 *cur = &lds[ks][1][slot][lane_u4];
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const bf16x8 vv = as_bf16x8(cur[t * 128 + j * 32]);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv, as_bf16x8(ph[j]), o[t], 0, 0, 0);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv, as_bf16x8(pl[j]), o[t], 0, 0, 0);
            }
        }
    };
    auto mask_max = [&](int it, f32x16 &x) __attribute__((always_inline)) {
        const int64_t p0 = (int64_t)(b0 + it * KS + ks) * 32;
        if (p0 + 32 > limit_min) {
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (p0 + 8 * (i >> 2) + 4 * h + (i & 3) >= limit) x[i] = neg_inf();
        }
        float m = x[0];
#pragma unroll
        for (int i = 1; i < 16; i++) m = fmaxf(m, x[i]);
        float b = m;
        rows_swap32(m, b);
        m_loc = fmaxf(m, b) * a.qscale;
    };
    // the row's reference follows its maximum lazily
    auto rescale = [&]() __attribute__((always_inline)) {
        const bool move = m_loc > m_ref + kLazyRescale;
        if (__any(move)) {
            float alpha = 1.0f;
            if (move) {
                alpha = fast_exp2(m_ref - m_loc);
                m_ref = m_loc;
            }
            l_run *= alpha;
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[t][i] *= alpha;
        }
    };

    // Block it's scores and block it - 1's soft-max and value product, independent of each other, side by side.
    int it = 0;
    auto next = [&]() __attribute__((always_inline)) {
        wait_pieces_and_barrier<0>();
#pragma unroll
        for (int g = 0; g < G; g++) request(it + G + g);
    };
    auto step = [&](auto exact_tag, int i, f32x16 &s_old, f32x16 &s_new) __attribute__((always_inline)) {
        rescale();
        uint4 ph[2], pl[2];
        qk(exact_tag, i & (NBUF - 1), s_new);
        softmax(s_old, ph, pl);
        pv((i - 1) & (NBUF - 1), ph, pl);
        mask_max(i, s_new);
    };
    auto walk = [&](auto exact_tag) __attribute__((always_inline)) {
        f32x16 sa, sb;   // scores of an even and of an odd block
        next();
        qk(exact_tag, 0, sa);
        mask_max(0, sa);
        if constexpr (G == 2) step(exact_tag, 1, sa, sb);
        it += G;
        while (it <= nl) {   // (the scores of block nl are of no block and dropped)
            next();
            if constexpr (G == 2) {
                step(exact_tag, it, sb, sa);
                if (it + 1 <= nl) step(exact_tag, it + 1, sa, sb);
            } else {
                step(exact_tag, it, sa, sb);
                sa = sb;
            }
            it += G;
        }
    };
    if (nl > 0) {
        if (q_exact) walk(std::true_type{});
        else walk(std::false_type{});
    }
    while (it <= nit) {
        next();
        it += G;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no piece may land after the workgroup has given its LDS back
    {
        float b = l_run;
        rows_swap32(l_run, b);
        l_run += b;
    }
    // ---- merge the sets -------------------------------------------------------------
    if constexpr (KS > 1) {
        static_assert(KS == 2 && RW * NT * 4 * 64 <= KS * 2 * NBUF * BUF_U4, "the merge reuses the staging buffers");
        wait_pieces_and_barrier<0>();
        float4 *xo = reinterpret_cast<float4 *>(&lds[0][0][0][0]);
        if (ks > 0) {
            if (h == 0) {
                s_m[ks][rw][n] = m_ref;
                s_l[ks][rw][n] = l_run;
            }
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    xo[((rw * NT + t) * 4 + i) * 64 + lane] = float4{o[t][4 * i], o[t][4 * i + 1], o[t][4 * i + 2], o[t][4 * i + 3]};
        }
        __syncthreads();
        if (ks > 0) return;
        const float m1 = s_m[1][rw][n], m_all = fmaxf(m_ref, m1);
        const float ref = (m_all == neg_inf()) ? 0.f : m_all;
        const float a0 = fast_exp2(m_ref - ref), a1 = fast_exp2(m1 - ref);
        l_run = l_run * a0 + s_l[1][rw][n] * a1;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4 v = xo[((rw * NT + t) * 4 + i) * 64 + lane];
                o[t][4 * i] = o[t][4 * i] * a0 + v.x * a1;
                o[t][4 * i + 1] = o[t][4 * i + 1] * a0 + v.y * a1;
                o[t][4 * i + 2] = o[t][4 * i + 2] * a0 + v.z * a1;
                o[t][4 * i + 3] = o[t][4 * i + 3] * a0 + v.w * a1;
            }
        m_ref = m_all;
    }
    if constexpr (SPLIT) {
        float4 *po = reinterpret_cast<float4 *>(a.part_o) + part * (NT * 4 * 64) + lane;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) po[(t * 4 + i) * 64] = float4{o[t][4 * i], o[t][4 * i + 1], o[t][4 * i + 2], o[t][4 * i + 3]};
        if (h == 0) {
            a.part_ml[part * 64 + n] = m_ref;
            a.part_ml[part * 64 + 32 + n] = l_run;
        }
    } else {
        // through LDS again, so that rows are written (and the gate read) in runs of 128 bytes
        if constexpr (KS == 1) wait_pieces_and_barrier<0>();   // every wave is done with the staging buffers
        uint4 *ow = KS == 1 ? &lds[0][0][0][0] + rw * 256 : &lds[0][0][0][0] + RW * NT * 4 * 64 + rw * 256;
        const float inv = 1.0f / l_run;
        uint4 gt[NT][4];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) gt[t][j] = vec_load((const uint4 *)(a.in.gate + tr_q[j] * a.in.stride + 32 * t + 4 * tr_chunk));
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                ow[tr_at(n, 2 * i + h)] = __builtin_bit_cast(uint4, float4{o[t][4 * i] * inv, o[t][4 * i + 1] * inv, o[t][4 * i + 2] * inv, o[t][4 * i + 3] * inv});
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float4 y = __builtin_bit_cast(float4, ow[tr_at(tr_row + 8 * j, tr_chunk)]);
                const float4 g = __builtin_bit_cast(float4, gt[t][j]);
                y = float4{y.x * fast_sigmoid(g.x), y.y * fast_sigmoid(g.y), y.z * fast_sigmoid(g.z), y.w * fast_sigmoid(g.w)};
                if (tr_ok[j]) *(float4 *)(a.out + tr_q[j] * D + 32 * t + 4 * tr_chunk) = y;
            }
        }
    }
}

// The log-sum-exp merge of a split chunk's partials, normalisation and gate: one wave per 32 rows and 32
// channels, in the order the partials lie (lane (n, h): row n, channels 8 i + 4 h .. + 3 of its 32).
template <int D>
__global__ __launch_bounds__(256) void sdpa_chunk_merge_kernel(const ChunkArgs a, int rw_count, int n_units) {
    constexpr int NT = D / 32;
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (unit >= n_units) return;
    const int t = unit % NT, w32 = unit / NT;
    const int per_head = a.nrt * rw_count, kvh = w32 / per_head, wt = w32 % per_head;
    const int nrows = a.n_tok * a.hpk;
    if (wt * 32 >= nrows) return;
    const size_t part0 = ((size_t)kvh * a.nrt + wt / rw_count) * a.nsplit * rw_count + wt % rw_count;
    float m[kMaxChunkSplits], l[kMaxChunkSplits];
#pragma unroll
    for (int s = 0; s < kMaxChunkSplits; s++) {
        const size_t p = part0 + (size_t)(s < a.nsplit ? s : a.nsplit - 1) * rw_count;
        m[s] = a.part_ml[p * 64 + n];
        l[s] = a.part_ml[p * 64 + 32 + n];
    }
    __shared__ uint4 s_tr[4][256];
    uint4 *tr = s_tr[threadIdx.x >> 6];
    const int tr_row = lane >> 3, tr_chunk = lane & 7;
    const auto tr_at = [](int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); };
    size_t at[4];
    bool ok[4];
    uint4 gt[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = wt * 32 + tr_row + 8 * j;
        ok[j] = r < nrows;
        const size_t row = ok[j] ? (size_t)(r / a.hpk) * a.Hq + kvh * a.hpk + r % a.hpk : 0;
        at[j] = row * D + 32 * t + 4 * tr_chunk;
        gt[j] = vec_load((const uint4 *)(a.in.gate + row * a.in.stride + 32 * t + 4 * tr_chunk));
    }
    float M = neg_inf();
#pragma unroll
    for (int s = 0; s < kMaxChunkSplits; s++) M = fmaxf(M, m[s]);
    float den = 0.f;
    float4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = float4{0.f, 0.f, 0.f, 0.f};
    const float4 *po = reinterpret_cast<const float4 *>(a.part_o) + part0 * (NT * 4 * 64) + t * 4 * 64 + lane;
#pragma unroll
    for (int s0 = 0; s0 < kMaxChunkSplits; s0 += 4) {
        if (s0 >= a.nsplit) break;
        uint4 v[4][4];
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                v[s][i] = vec_load((const uint4 *)(po + (size_t)(s0 + s < a.nsplit ? s0 + s : a.nsplit - 1) * rw_count * (NT * 4 * 64) + i * 64));
#pragma unroll
        for (int s = 0; s < 4; s++) {
            // a split that saw nothing of the row (sum 0) weighs nothing, whatever its part of the workspace holds; one
            // that saw nothing but NaN has no maximum either, and its sum carries them into the result
            const float none = l[s0 + s] == 0.f ? 0.f : l[s0 + s];
            const float w = s0 + s < a.nsplit ? (m[s0 + s] != neg_inf() ? fast_exp2(m[s0 + s] - M) : none) : 0.f;
            if (w != 0.f) {
                den += w * l[s0 + s];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float4 x = __builtin_bit_cast(float4, v[s][i]);
                    acc[i].x += w * x.x; acc[i].y += w * x.y; acc[i].z += w * x.z; acc[i].w += w * x.w;
                }
            }
        }
    }
    const float inv = 1.0f / den;
#pragma unroll
    for (int i = 0; i < 4; i++)
        tr[tr_at(n, 2 * i + h)] = __builtin_bit_cast(uint4, float4{acc[i].x * inv, acc[i].y * inv, acc[i].z * inv, acc[i].w * inv});
    wave_lds_order();
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float4 y = __builtin_bit_cast(float4, tr[tr_at(tr_row + 8 * j, tr_chunk)]), g = __builtin_bit_cast(float4, gt[j]);
        if (ok[j])
            *(float4 *)(a.out + at[j]) = float4{y.x * fast_sigmoid(g.x), y.y * fast_sigmoid(g.y), y.z * fast_sigmoid(g.z), y.w * fast_sigmoid(g.w)};
    }
}

// Whether the kernel can norm and rotate the query rows itself (RowNorm).
bool sdpa_chunk_takes_raw(int D, int rotary_dim) { return D >= 128 && rotary_dim * 4 == D; }

// Which kernel takes a chunk, and how it is cut up.  Estimates in microseconds, with the kernels' constants by width
// (64, 128, 256); `load` is workgroups per CU.
//
// On 32x32 tiles: the shape of a workgroup and the splits of the cache of the smallest cost, which is the call's own time and
// one and a half times the time of the whole device that it takes: a chunk's layers follow each other, but other sequences may
// run beside them.
//   workgroup  kFixed (launch, query, first block, epilogue) + blocks per wave set * kBlock; a CU that holds two
//              workgroups (head_dim <= 128) runs them 5 % faster than one after the other
//   partials   written at 4.5 TB/s, merged at 7.5 TB/s with the gate and the result; 12 for the second launch
// A split chunk's partials fit limits.ws_elems floats.
//
// That kernel's workgroups begin slowly (32 query rows a wave in 512 registers), so that a short cache, or few rows before a
// long one, are better served by 16-row groups: by sdpa_prefill (Rows) up to 2048 positions, by the split-K kernel beyond.  They
// are taken where one sequence after itself is estimated faster with them (sequences side by side are bound by the
// launches there, and so no slower).  The estimates are fitted to 800 chunks of 2 .. 1024 tokens behind 0 .. 16384 positions
// (32 and 16 heads over 2 of 256, 32 over 4 and over 32 of 128, 16 over 2 of 64), normed and raw, every route of
// every chunk measured: 8 % r.m.s. on a time, and of the routes they choose 29 of 1600 are more than 3 % slower than the
// 16-row groups for one sequence, one 14 %; without them 418 were, up to 62 %, most of them small (2 .. 64 tokens of 32 heads over 2
// of 256 from an empty cache 21 us a layer, 14 to 18 with 16-row groups).
static constexpr double kFixed[2][3] = {{6.0, 9.0, 12.0}, {7.0, 9.0, 14.0}}, kBlock[2][3] = {{0.5, 0.8, 1.58}, {0.55, 0.85, 1.85}};

struct ChunkShape {
    int w, Hq, Hkv, D, n_tok;
    int64_t rows, kv_len, nblk;
    double num_cus;
    bool causal() const { return kv_len - n_tok < n_tok; }   // most of the work is the triangle: tiles differ, the longest go first
    double seen() const { return causal() ? ((double)(kv_len - n_tok) + 0.5 * n_tok) / (double)kv_len : 1.0; }
    // the prologue of raw projections: all heads of a token, 16 bytes a q channel and fewer of k and v
    double prologue() const { return 0.5 + 3.6e-6 * n_tok * (double)(Hq + 2 * Hkv) * D; }
};

// One sequence's time of a layer, prologue included, behind another of its own.
static double tiles32_time(const ChunkShape &c, const ChunkPlan &p, ChunkQueryKind kind) {
    static constexpr double kStart[2][3] = {{9.0, 10.5, 16.0}, {10.0, 12.0, 18.0}}, kStep[2][3] = {{0.6, 1.0, 1.8}, {0.6, 1.05, 1.9}};
    static constexpr double kRawQuery[3] = {0.5, 1.4, 2.5};   // norm and rotation in the launch; k, v and table ahead of it
    const int shape = p.ks - 1, slots = c.D <= 128 ? 2 : 1;
    const double its = (p.bps + p.ks - 1) / p.ks, load = (double)p.nrt * c.Hkv * p.splits / c.num_cus, rounds = ceil(load / slots);
    const double step = kStep[shape][c.w] * (load > 1 && slots == 2 ? 0.95 : 1.0), start = kStart[shape][c.w];
    double t = c.causal() ? fmax(start + its * step, start * rounds + load * its * c.seen() * step) : start * rounds + ceil(load) * its * step;
    if (p.splits > 1) t += 4.0 + 4.0 * p.nrt * c.Hkv * p.splits * 32.0 * p.rw * c.D / 9e6;
    if (kind == ChunkQueryKind::Raw) t += kRawQuery[c.w] + 8e-6 * c.n_tok * (double)c.Hkv * c.D;
    if (kind == ChunkQueryKind::RawPrologue) t += c.prologue();
    return t;
}
static double rows_time(const ChunkShape &c, int64_t wgs, ChunkQueryKind kind) {
    static constexpr double kStart[3] = {8.2, 9.8, 11.5}, kStep[3] = {0.69, 1.0, 1.45};
    const double its = (double)(c.D <= 128 ? (c.nblk + 1) / 2 : c.nblk);   // two wave sets where there is room for them
    return kStart[c.w] + its * kStep[c.w] + 3.5 * (double)wgs / c.num_cus + 0.8e-6 * (double)c.kv_len * c.Hkv * c.D +
           (kind == ChunkQueryKind::Normed ? 0.0 : c.prologue());
}
// (a row group streams its kv head's cache by itself, from its XCD's L2 or from memory)
static double split_k_time(const ChunkShape &c, ChunkQueryKind kind) {
    static constexpr double kStream[3] = {0.005, 0.010, 0.0173};
    const int64_t nhg = (c.rows + 15) / 16, groups = nhg * c.Hkv;
    int64_t splits = (int64_t)c.num_cus / groups;
    if (splits > c.nblk / 4) splits = c.nblk / 4;
    if (splits < 1) splits = 1;
    const double load = (double)(groups * splits) / c.num_cus, kv = (double)c.kv_len;
    const double xcds = nhg < 8 ? (double)nhg : 8.0;
    return 12.0 + fmax(ceil(load) * kv / (double)splits * kStream[c.w], 4.0 * kv * c.Hkv * c.D * xcds / 6.5e6) +
           7e-6 * (double)c.rows * c.Hkv * c.D + (kind == ChunkQueryKind::Normed ? 0.0 : c.prologue());
}

ChunkPlan sdpa_chunk_plan(int kv_dtype, int Hq, int Hkv, int D, int n_tok, int64_t kv_len, int num_cus, ChunkQueryKind kind,
                          const ChunkLimits &limits) {
    ChunkPlan best;
    if (n_tok < 2 || !sdpa_shape_supported(kv_dtype, D)) return best;
    const int64_t rows = (int64_t)n_tok * (Hq / Hkv), row_wgs = ((rows + 15) / 16 + 3) / 4 * Hkv;
    if (kv_dtype != MFA_KV_BF16) {
        // a short cache (nothing to gain from splitting it), or rows that alone give half the CUs a workgroup
        if ((kv_len + 15) / 16 <= 64 || row_wgs >= num_cus / 2) best.route = ChunkRoute::Rows;
        return best;
    }
    const ChunkShape c{D == 64 ? 0 : D == 128 ? 1 : 2, Hq, Hkv, D, n_tok, rows, kv_len, (kv_len + 31) / 32, (double)num_cus};
    const int w = c.w, slots = D <= 128 ? 2 : 1;
    const int64_t nblk = c.nblk;
    if ((rows + 127) * Hkv > INT32_MAX / 2 || nblk > INT32_MAX / 2) return best;   // 32-bit row and block numbers
    static constexpr double kStream[3] = {0.007, 0.0108, 0.0175};
    static constexpr double kLaunch = 12.0, kEmpty = 2.5;   // of a workgroup's fixed time, what its CU is free in
    const double out_bytes = 8.0 * (double)rows * Hkv * D, seen = c.seen();
    const bool two_launches = limits.shifted && nblk > 64 && row_wgs < num_cus / 2;
    double best_cost = 0;
    for (int shape = 0; shape < 2; shape++) {
        const int rw = shape ? 2 : 4, ks = shape ? 2 : 1;
        const int64_t nrt = (rows + 32 * rw - 1) / (32 * rw);
        for (int64_t want = two_launches ? 2 : 1; want <= kMaxChunkSplits && want <= nblk; want++) {
            const int64_t bps = (nblk + want - 1) / want;
            if ((nblk + bps - 1) / bps != want) continue;
            const size_t elems = want > 1 ? (size_t)(nrt * Hkv * want) * 32 * rw * D : 0;
            if (elems > limits.ws_elems) break;
            const double its = (double)((bps + ks - 1) / ks), load = (double)(nrt * Hkv * want) / num_cus, fixed = kFixed[shape][w];
            const double block = kBlock[shape][w] * (load > 1 && slots == 2 ? 0.95 : 1.0), rounds = ceil(load / slots);
            double t = c.causal() ? fmax(fixed + its * block, fixed * rounds + load * its * seen * block) : fixed * rounds + ceil(load) * its * block;
            double busy = load * (fixed - kEmpty + its * seen * block);
            if (want > 1) {
                const double moved = 4.0 * elems / 4.5e6 + (4.0 * elems + out_bytes) / 7.5e6;
                t += moved + kLaunch;
                busy += moved;
            }
            if (best.route != ChunkRoute::Tiles32 || t + 1.5 * busy < best_cost) {
                best_cost = t + 1.5 * busy;
                best = ChunkPlan{ChunkRoute::Tiles32, rw, ks, (int)nrt, (int)want, (int)bps};
            }
        }
    }
    if (best.route != ChunkRoute::Tiles32) return best;
    const double own = tiles32_time(c, best, kind);
    if (nblk <= 64) {
        // (past a workgroup per CU the 32x32 tiles are faster at every length)
        if (row_wgs <= num_cus && rows_time(c, row_wgs, kind) <= own) best = ChunkPlan{ChunkRoute::Rows};
    } else if (limits.split_k && row_wgs < num_cus / 2) {
        const int64_t groups = (rows + 15) / 16 * Hkv;
        int64_t splits = num_cus / groups;
        if (splits > nblk / 4) splits = nblk / 4;
        if (splits < 1) splits = 1;
        const double load = (double)(groups * splits) / num_cus, stream = (double)kv_len / (double)splits * kStream[w], merge = out_bytes / 8 * 6.9e-6;
        if (3.0 + ceil(load) * stream + kLaunch + merge + 1.5 * (load * (stream + 1.0) + merge) < best_cost || split_k_time(c, kind) <= own)
            best = ChunkPlan{};
    }
    return best;
}

ChunkPlan sdpa_chunk_plan_of(int Hq, int Hkv, int n_tok, int64_t kv_len, int rw, int splits) {
    const int64_t rows = (int64_t)n_tok * (Hq / Hkv), nblk = (kv_len + 31) / 32, bps = (nblk + splits - 1) / splits;
    return ChunkPlan{ChunkRoute::Tiles32, rw, rw == 4 ? 1 : 2, (int)((rows + 32 * rw - 1) / (32 * rw)), (int)((nblk + bps - 1) / bps), (int)bps};
}

size_t sdpa_chunk_part_elems(const ChunkPlan &p, int Hkv, int D) {
    return p.splits > 1 ? (size_t)Hkv * p.nrt * p.splits * 32 * p.rw * D : 0;
}

int launch_sdpa_chunk(hipStream_t stream, const ChunkPlan &p, int Hq, int Hkv, int D, int n_tok, int64_t kv_len,
                      size_t plane_elems, const void *k_tiled, const void *v_tiled, const ChunkQuery &in,
                      float *out, float *ws, size_t ws_elems) {
    const size_t elems = sdpa_chunk_part_elems(p, Hkv, D);
    if (p.route != ChunkRoute::Tiles32 || elems > ws_elems) return fail(MFA_ERR_INVALID, "sdpa: chunk plan without its workspace");
    const int hpk = Hq / Hkv;
    ChunkArgs a{(const uint16_t *)k_tiled, (const uint16_t *)v_tiled, plane_elems, in, hpk, Hq, n_tok, kv_len - n_tok,
                (1.0f / sqrtf((float)D)) * kLog2e, out, ws, ws + elems, p.nrt, p.splits, p.bps, Hkv * p.splits,
                kv_len - n_tok >= n_tok};
    const dim3 grid((unsigned)(p.nrt * Hkv * p.splits));
    const bool raw = in.q_norm != nullptr;
    if (raw && D < 128) return fail(MFA_ERR_SHAPE, "sdpa: raw query rows of %d channels", D);
#define MFA_CHUNK(DD, RWW, KSS, GG, SP, RAWW) \
    hipLaunchKernelGGL((sdpa_chunk_kernel<DD, RWW, KSS, GG, SP, RAWW>), grid, dim3(64 * RWW * KSS), 0, stream, a)
#define MFA_CHUNK_R(DD, RWW, KSS, GG)                                    \
    do {                                                                 \
        if (p.splits > 1 && raw) MFA_CHUNK(DD, RWW, KSS, GG, true, (DD >= 128)); \
        else if (p.splits > 1) MFA_CHUNK(DD, RWW, KSS, GG, true, false); \
        else if (raw) MFA_CHUNK(DD, RWW, KSS, GG, false, (DD >= 128));   \
        else MFA_CHUNK(DD, RWW, KSS, GG, false, false);                  \
    } while (0)
    // (two wave sets at head_dim >= 128 leave room for one block of each in use and one on its way)
    if (D == 256) {
        if (p.ks == 1) MFA_CHUNK_R(256, 4, 1, 2);
        else MFA_CHUNK_R(256, 2, 2, 1);
    } else if (D == 128) {
        if (p.ks == 1) MFA_CHUNK_R(128, 4, 1, 2);
        else MFA_CHUNK_R(128, 2, 2, 1);
    } else {
        if (p.ks == 1) MFA_CHUNK_R(64, 4, 1, 2);
        else MFA_CHUNK_R(64, 2, 2, 2);
    }
#undef MFA_CHUNK_R
#undef MFA_CHUNK
    MFA_HIP(hipGetLastError());
    if (p.splits > 1) {
        const int n_units = Hkv * p.nrt * p.rw * (D / 32);
        const dim3 mgrid((n_units + 3) / 4);
        if (D == 256) hipLaunchKernelGGL(sdpa_chunk_merge_kernel<256>, mgrid, dim3(256), 0, stream, a, p.rw, n_units);
        else if (D == 128) hipLaunchKernelGGL(sdpa_chunk_merge_kernel<128>, mgrid, dim3(256), 0, stream, a, p.rw, n_units);
        else hipLaunchKernelGGL(sdpa_chunk_merge_kernel<64>, mgrid, dim3(256), 0, stream, a, p.rw, n_units);
        MFA_HIP(hipGetLastError());
    }
    return MFA_OK;
}

}  // namespace mfa
