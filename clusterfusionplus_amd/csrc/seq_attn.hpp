// Attention of a portion of the sequence models (device code; included by seq_kernels.hip).
#pragma once
#include <type_traits>

#include "seq_device.hpp"
#include "seq_plan.hpp"

namespace cfpp {

// The query columns of one key / value head are (token, head of the group), head fastest; a workgroup takes 4 C of them
// and walks the keys its tokens can see, first the cached ones (positions before k_split), then those in the buffer.  Behind a
// key's own row comes the part that all heads share, if there is one.  The softmax is online, the sink is added to the
// denominator at the end.
//
// Where a portion has too few columns to fill the chip, `splits` workgroups share the keys of the same columns; they leave their
// sums, maxima and denominators, and k_seq_attn_merge makes the outputs.
struct SeqAttn {
    const char *q, *k, *v, *kc, *vc;
    const char* kr;          // rows of the shared part, of position 0 on
    char* out;
    const float* sink;       // nullable
    const float* gate;       // nullable: [T][ldg], the outputs are multiplied by its sigmoid
    int T, H, R, G, qrow, krow, vrow, V, vtiles, pos0, chunk, cap, rows, ldo, k_split, runits, rrow, ldg;
    float scale_log2;
    int splits, up, swap;    // (of attn_block)
    float *part, *ml;        // splits > 1: [splits][T][H][16 vtiles], [splits][T][H][2]
};
template <int UN> __device__ __forceinline__ int swz_key(int row) { return UN % 16 ? (row >> 1) & 7 : row & 15; }

// Matrix products of a wave: blocks of C x C outputs (16 or 32), a lane has one column and the rows 8 j + 4 g .. + 3 of it (16: j = 0), where
// g = lane / C; an operand's unit of 16 bytes is the g-th of the product's k.
template <int C> struct AttnBlock;
template <> struct AttnBlock<16> { typedef f32x4 acc; };
template <> struct AttnBlock<32> { typedef float acc __attribute__((ext_vector_type(16))); };
template <typename T> __device__ __forceinline__ f32x4 attn_mma(u32x4 a, u32x4 b, f32x4 c) { return mma16<T>(a, b, c); }
template <typename T> __device__ __forceinline__ AttnBlock<32>::acc attn_mma(u32x4 a, u32x4 b, AttnBlock<32>::acc c) {
    static_assert(sizeof(T) == 2, "");
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
// maximum and sum of a column over the lanes that share it
template <int C> __device__ __forceinline__ float rows_max(float v) {
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    if constexpr (C == 32) return v;
    a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
template <int C> __device__ __forceinline__ float rows_sum(float v) {
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    if constexpr (C == 32) return v;
    a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// Tiles of KT keys in LDS: NK elements of a key, NT value columns.  Two buffers, filled by copies that go there directly: the next
// tile's are on their way while one is worked on.  Key rows are stored in units of 16 bytes, permuted by swz_key.  Value rows stay
// rows: their fragments, four keys of a column per lane, come from transposing reads (bf16) or element by element (fp32), and
// blocks of 16 columns are permuted so that the rows that a read takes together start in different banks.
template <typename T, int NK, int NT, int C> struct AttnTile {
    static constexpr int keys = sizeof(T) == 2 ? 64 : 32;
    static constexpr int kbytes = NK * (int)sizeof(T), ku = kbytes / 16;             // a key row and its units
    static constexpr int vbytes = NT * (int)sizeof(T), vu = vbytes / 16, block = 16 * (int)sizeof(T) / 16;   // ... of a value row; units of a block
    static constexpr int ksize = keys * kbytes, vsize = keys * vbytes, size = ksize + vsize;
    static constexpr int kcopies = ksize / 1024 / kSeqWaves, vcopies = vsize / 1024 / kSeqWaves;             // 1 KB copies of a wave
    static_assert(ksize % (1024 * kSeqWaves) == 0 && vsize % (1024 * kSeqWaves) == 0, "");
    // a lane's place in its row comes again after so many copies (a multiple of 16 rows on)
    static constexpr int period(int units) {
        int p = 1;
        while (p * 64 * kSeqWaves % units != 0 || p * 64 * kSeqWaves / units % 16 != 0) ++p;
        return p;
    }
    static constexpr int kp = period(ku), vp = period(vu), krows = kp * 64 * kSeqWaves / ku, vrows = vp * 64 * kSeqWaves / vu;
    static __device__ __forceinline__ int vswz(int row) {
        if (C == 32) return NT >= 128 ? (row & 3) * 2 : row & 2;           // (a read takes two blocks of four rows)
        return sizeof(T) == 4 ? (row >> 2) & 3 : NT >= 128 ? row & 7 : (row >> 1) & 3;
    }
};

// What bounds it: a SIMD's vector instructions and matrix products, which overlap in part only: a product of 16 x 16 x 32 takes 16 cycles of the
// matrix core and, measured beside another wave's fused multiply-adds, 9 of the other wave's issue; and the power that both draw (8000 tokens run
// at 1.8 GHz).  So: two workgroups per compute unit, one barrier per tile, nothing waited for but the tile itself, and few
// instructions per weight.  Columns in blocks of 32 where there are enough of them: a product of 32 x 32 x 16 does twice the work for the same issue,
// and a lane keeps the maximum of one column, shared with one other lane.  In us per layer, 8000 tokens with 32 heads of 192 and 128 / 2048 with 128 and
// 128: copies that the compiler knows of 1753 / 141, its waits taken out 1264 / 104, the longest walks first 945 / 85, blocks of 32 instead of
// 2 x 16 935 / 79, sums that are rescaled for maxima that move by 2^8 only and no value converted twice 895 / 73, addresses that are carried from
// tile to tile 887 / 70.
// 37 tokens at 1990, 32 / 8 heads: 85 -> 12 us and 5 for the merge (24 workgroups became 384).
// Tried and slower, on blocks of 16 with fragments read ahead, which took 875 us on that card (8000 tokens): two groups of four waves that take turns at
// products and softmax (1000), the scores of the next tile beside the softmax with tiles of 32 keys (1318).
// Reading ahead takes heads of up to 64 from 79 to 103 registers, four waves of a SIMD instead of five: 16 heads, 1500 tokens at 0 / at 1990 take 29.6 /
// 66.4 us without and 24.6 / 55.2 with it and the order of the workgroups, 100 tokens 6.5 and 6.5.
// (NK: elements of a key row in LDS, NT: value columns.  The products run over all of them, without branches between the reads
// of LDS: past the end of the query there are zeros, and of the columns past the end of a value nothing is stored.
// C: columns of a wave; SH: keys have a shared part)
template <typename T, int NK, int NT, int C, bool SH>
__global__ __launch_bounds__(kSeqThreads, (NT <= 128 ? 2 : 1)) void k_seq_attn(SeqAttn a) {
    using L = AttnTile<T, NK, NT, C>;
    using Acc = typename AttnBlock<C>::acc;
    constexpr int KT = L::keys, G = kWave / C, KS = L::ku / G, NE = C * C / kWave, kCols = C * kSeqWaves;      // lanes of a column, steps of a score, outputs of a lane
    extern __shared__ __align__(1024) char lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane % C, g = lane / C;
    // Workgroups go row by row, a row being the same columns of all key heads and splits, with the longest walks first (attn_block), so that the short
    // ones fill the chip's last moments (head by head, a quarter of the compute units' time was a tail: 8000 tokens, 32 heads of 192 and 128: 1264 -> 956 us;
    // 2048 tokens, 128 and 128: 104 -> 86 us).  Where the heads are a multiple of eight, all workgroups of a head are on one XCD and walk its keys
    // side by side.
    // (one split: the grid has one dimension, which is not limited to 65535)
    const int ncols = a.T * a.R, rows = (ncols + kCols - 1) / kCols, part = blockIdx.x / (unsigned)a.G, gq = blockIdx.x - part * a.G;
    const bool in_parts = C == 16 && a.splits > 1;       // (portions with blocks of 32 fill the chip)
    const int split = in_parts ? part : 0, c0 = attn_block(in_parts ? blockIdx.y : part, rows, a.up, a.swap) * kCols;

    // (its sign goes to the query; not zero, so that it keeps the scores of keys that are not seen at -infinity; NaN stays NaN)
    const float size = fabsf(a.scale_log2), scale = size < 1e-30f ? 1e-30f : size;
    const int cc = min(c0 + wave * C + col, ncols - 1), tok = cc / a.R, head = gq * a.R + (cc - tok * a.R);
    u32x4 qf[KS];
    float m = kNegBig, l = 0.0f;                         // running maximum (log2 domain), this lane's share of the denominator
    Acc acc[NT / C];
    {
        const char* qr = a.q + ((size_t)tok * a.H + head) * a.qrow + g * 16;
        const int units = a.qrow / 16;
        const uint32_t flip = a.scale_log2 < 0.0f ? (sizeof(T) == 2 ? 0x80008000u : 0x80000000u) : 0u;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            qf[s] = ld16(qr + min(s, units / G - 1) * (G * 16)) ^ u32x4{flip, flip, flip, flip};
            if (s >= units / G) qf[s] = u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < NT / C; ++i) acc[i] = Acc(0.0f);
    }
    // keys the workgroup needs, and those every column of this wave sees / any column sees
    const int t_first = c0 / a.R, t_last = min(a.T - 1, (c0 + kCols - 1) / a.R);
    const int k_first = chunk_start(a.pos0 + t_first, a.chunk), k_end = a.pos0 + t_last + 1;
    const int w_first = min(c0 + wave * C, ncols - 1) / a.R, w_last = min(c0 + (wave + 1) * C - 1, ncols - 1) / a.R;
    const int all_lo = chunk_start(a.pos0 + w_last, a.chunk), all_hi = a.pos0 + w_first;
    const int any_lo = chunk_start(a.pos0 + w_first, a.chunk), any_hi = a.pos0 + w_last;
    const int dunits = a.krow / 16, vunits = a.vrow / 16;

    // tiles: [k_first, k_split) in the cache, then [k_split, k_end) in the buffer; this split's are t0 .. t1 - 1
    const int in_cache = max(0, min(k_end, a.k_split) - k_first), n_cached = (in_cache + KT - 1) / KT, new_first = max(k_first, a.k_split);
    const int ntiles = n_cached + (max(0, k_end - new_first) + KT - 1) / KT;
    const int t0 = in_parts ? mul_div(ntiles, split, a.splits) : 0, t1 = in_parts ? mul_div(ntiles, split + 1, a.splits) : ntiles;
    struct Tile { int k0, hi; const char *k, *v; };      // first key, end of its part, its rows
    auto tile_at = [&](int i) {
        const bool cached = i < n_cached;
        const int k0 = cached ? k_first + i * KT : new_first + (i - n_cached) * KT;
        const ptrdiff_t row = (ptrdiff_t)gq * (cached ? a.rows : a.cap) + k0 - (cached ? chunk_start(a.pos0, a.chunk) : a.k_split);
        return Tile{k0, cached ? min(k_end, a.k_split) : k_end, (cached ? a.kc : a.k) + row * a.krow, (cached ? a.vc : a.v) + row * a.vrow};
    };
    // the lane's place in the copies: row of the tile, unit of its source row (the shared part comes from rows of its own)
    const uint32_t l0 = lds_address(lds);
    uint32_t koff[L::kp], voff[L::vp];
    const char* kfrom[L::kp];                         // SH: where the lane's next copies come from, and the way on to their next rows
    int64_t kstep[L::kp];
#pragma unroll
    for (int i = 0; i < L::kp; ++i) {
        const int p = (i * kSeqWaves + wave) * 64 + lane, r = p / L::ku, u = (p % L::ku) ^ swz_key<L::ku>(r);
        const bool sh = SH && u >= dunits && u < dunits + a.runits;
        koff[i] = sh ? r * a.rrow + (u - dunits) * 16 : r * a.krow + (u < dunits ? u : 0) * 16;
        kstep[i] = L::krows * (sh ? a.rrow : a.krow);
    }
#pragma unroll
    for (int i = 0; i < L::vp; ++i) {
        const int p = (i * kSeqWaves + wave) * 64 + lane, r = p / L::vu, u = (p % L::vu) ^ (L::vswz(r) * L::block);
        voff[i] = r * a.vrow + min(u, vunits - 1) * 16;
    }
    // tile i, and the tile i behind the one before it: nothing is multiplied but where the cached part ends
    auto begin_at = [&](int i) __attribute__((always_inline)) {
        const Tile t = tile_at(i);
        if constexpr (SH) {
            const char* const rows = a.kr + (ptrdiff_t)t.k0 * a.rrow;
#pragma unroll
            for (int j = 0; j < L::kp; ++j) {
                const int p = (j * kSeqWaves + wave) * 64 + lane, u = (p % L::ku) ^ swz_key<L::ku>(p / L::ku);
                kfrom[j] = (u >= dunits && u < dunits + a.runits ? rows : t.k) + koff[j];
            }
        }
        return t;
    };
    const ptrdiff_t ktile = (ptrdiff_t)KT * a.krow, vtile = (ptrdiff_t)KT * a.vrow, kgroup = (ptrdiff_t)L::krows * a.krow, vgroup = (ptrdiff_t)L::vrows * a.vrow;
    auto follow = [&](const Tile& t, int i) __attribute__((always_inline)) {
        return i == n_cached ? begin_at(i) : Tile{t.k0 + KT, t.hi, t.k + ktile, t.v + vtile};
    };
    auto fetch = [&](const Tile& t, int buf) __attribute__((always_inline)) {
        const uint32_t d = l0 + buf * L::size + wave * 1024;
        // rows past the end (`whole` false): the last one again
        auto copies = [&](auto whole) __attribute__((always_inline)) {
            constexpr bool W = decltype(whole)::value;
            const int last = t.hi - 1 - t.k0;
            const char *kb = t.k, *vb = t.v;
#pragma unroll
            for (int i = 0; i < L::kcopies; ++i) {
                const int j = i % L::kp, r = i / L::kp * L::krows + (j * kSeqWaves * 64 + wave * 64 + lane) / L::ku;
                const uint32_t to = d + i * (kSeqWaves * 1024);
                if constexpr (SH) {
                    if constexpr (W) copy_to_lds16_from(kfrom[j], to);
                    else copy_to_lds16_from(kfrom[j] - max(0, r - last) * ((int)kstep[j] / L::krows), to);
                    kfrom[j] += kstep[j];
                } else {
                    if (j == 0) kb = i == 0 ? uniform(kb) : uniform(kb + kgroup);
                    if constexpr (W) copy_to_lds16_at(koff[j], kb, to);
                    else copy_to_lds16_from(kb + (int)koff[j] - max(0, r - last) * a.krow, to);
                }
            }
#pragma unroll
            for (int i = 0; i < L::vcopies; ++i) {
                const int j = i % L::vp, r = i / L::vp * L::vrows + (j * kSeqWaves * 64 + wave * 64 + lane) / L::vu;
                const uint32_t to = d + L::ksize + i * (kSeqWaves * 1024);
                if (j == 0) vb = i == 0 ? uniform(vb) : uniform(vb + vgroup);
                if constexpr (W) copy_to_lds16_at(voff[j], vb, to);
                else copy_to_lds16_from(vb + (int)voff[j] - max(0, r - last) * a.vrow, to);
            }
        };
        if (t.k0 + KT <= t.hi) copies(std::true_type{});
        else copies(std::false_type{});
    };
    // key fragments: unit d G + g of row col (C rows on, and past the units that the permutation mixes, it is the same)
    constexpr int KD = (L::ku % 16 ? 8 : 16) / G;
    int kat[KD];
#pragma unroll
    for (int d = 0; d < KD; ++d) kat[d] = col * L::kbytes + ((d * G + g) ^ swz_key<L::ku>(col)) * 16;
    // value fragments: the lane's rows start at key 4 g (bf16: with the transposing read, lane i of a group of 16 reads 8 bytes of key
    // 4 g + i / 4 and receives four keys of column i; C = 32: every second group takes the next 16 columns).  Of the first block of
    // columns; block i: vat ^ i blocks
    const int vrow0 = 4 * g + (sizeof(T) == 2 ? (lane & 15) >> 2 : 0);
    const int vat = L::ksize + vrow0 * L::vbytes + (L::vswz(vrow0) ^ (C == 32 ? (lane >> 4) & 1 : 0)) * L::block * 16 + (sizeof(T) == 2 ? (col & 3) * 8 : col * 4);

    Tile t{};
    if (t0 < t1) {
        t = begin_at(t0);
        fetch(t, 0);
    }
    for (int it = t0, buf = 0; it < t1; ++it, buf ^= 1) {
        pipe_barrier<0>();                               // the tile is there, and nobody reads the other buffer any more
        Tile tn = t;
        if (it + 1 < t1) {
            tn = follow(t, it + 1);
            fetch(tn, buf ^ 1);
        }
        const char* const tile = lds + buf * L::size;
        if (t.k0 <= any_hi && min(t.k0 + KT, t.hi) > any_lo) {
            // Two blocks of keys side by side; their fragments are read two steps ahead.
            constexpr int KB = KT / C, KP = 2, kSteps = KB / KP * KS;
            Acc s[KB];
            u32x4 kf[3][KP];
            auto read_keys = [&](int i) __attribute__((always_inline)) {
                const int d = i % KS, kt = i / KS * KP;
#pragma unroll
                for (int j = 0; j < KP; ++j)
                    kf[i % 3][j] = *reinterpret_cast<const u32x4*>(tile + kat[d % KD] + ((kt + j) * C * L::kbytes + d / KD * KD * G * 16));
            };
            read_keys(0);
            read_keys(1);
#pragma unroll
            for (int i = 0; i < kSteps; ++i) {
                if (i + 2 < kSteps) read_keys(i + 2);
                __builtin_amdgcn_sched_barrier(0);
                const int d = i % KS, kt = i / KS * KP;
#pragma unroll
                for (int j = 0; j < KP; ++j) s[kt + j] = attn_mma<T>(kf[i % 3][j], qf[d], d == 0 ? Acc(0.0f) : s[kt + j]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!(t.k0 + KT <= t.hi && t.k0 >= all_lo && t.k0 + KT - 1 <= all_hi)) {
                int k0 = t.k0 + g * 4, pq = a.pos0 + tok;
                asm volatile("" : "+v"(k0), "+v"(pq));   // (what is for the comparisons stays inside the branch)
                const int end = min(pq, t.hi - 1) - k0, begin = chunk_start(pq, a.chunk) - k0;
#pragma unroll
                for (int kt = 0; kt < KB; ++kt)
#pragma unroll
                    for (int r = 0; r < NE; ++r) {
                        const int k = kt * C + (r >> 2) * 8 + (r & 3);
                        if (k > end || k < begin) s[kt][r] = -INFINITY;
                    }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < KB; ++kt)
#pragma unroll
                for (int r = 0; r < NE; ++r) mx = fmaxf(mx, s[kt][r]);
            // (a maximum that has moved by less than 2^8 stays as it is: weights up to 256 lose nothing, and the sums need not be rescaled)
            const float top = rows_max<C>(mx) * scale;
            if (__builtin_amdgcn_ballot_w64(top > m + 8.0f) != 0) {
                const float mn = fmaxf(m, top), c = fast_exp2(m - mn);
                l *= c;
#pragma unroll
                for (int i = 0; i < NT / C; ++i) acc[i] *= c;
                m = mn;
            }
            // (weights of four keys each)
            f32x4 w[KT / 4 / G];
#pragma unroll
            for (int i = 0; i < KT / 4 / G; ++i) {
#pragma unroll
                for (int r = 0; r < 4; ++r) w[i][r] = fast_exp2(fmadd(s[i / (NE / 4)][i % (NE / 4) * 4 + r], scale, -m));
                l += (w[i][0] + w[i][1]) + (w[i][2] + w[i][3]);
            }
            __builtin_amdgcn_sched_barrier(0);           // (values read ahead of the softmax would take its registers)
            if constexpr (sizeof(T) == 2) {
                // a product takes the weights of eight keys of a lane; two blocks of value columns are multiplied side by side while the next are read
                constexpr int KV = KT / 8 / G, VB = NT / C > 1 ? 2 : 1;
                u32x4 hi[KV], lo[KV];
#pragma unroll
                for (int h = 0; h < KV; ++h) split_weights(w[2 * h], w[2 * h + 1], hi[h], lo[h]);
                u32x4 f[2][VB][2];
                constexpr int kSteps = NT / C / VB * (KV / 2);
                auto read_values = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                    for (int k = 0; k < VB; ++k)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const char* b = tile + (vat ^ ((i / (KV / 2) * VB + k) * (C / 16) * L::block * 16)) + (i % (KV / 2) * 2 + h) * (8 * G) * L::vbytes;
                            const u32x2 x = read_transposed(b), y = read_transposed(b + 4 * G * L::vbytes);
                            f[i & 1][k][h] = u32x4{x.x, x.y, y.x, y.y};
                        }
                };
                read_values(0);
#pragma unroll
                for (int i = 0; i < kSteps; ++i) {
                    if (i + 1 < kSteps) read_values(i + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int part = 0; part < 2; ++part)
#pragma unroll
                            for (int k = 0; k < VB; ++k) {
                                const int n = i / (KV / 2) * VB + k, e = i % (KV / 2) * 2 + h;
                                acc[n] = attn_mma<T>(f[i & 1][k][h], part == 0 ? hi[e] : lo[e], acc[n]);
                            }
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                // Values of four keys are read two products ahead: left to the compiler, each pair of reads is waited for right where it is used (700
                // tokens at 1990, 16 / 4 heads of 128: 223 us with all reads hoisted, 232 with none, 207 two ahead).
                constexpr int KV = KT / C, kSteps = NT / C * KV;
                f32x4 f[3];
                auto read_values = [&](int i) __attribute__((always_inline)) {
                    const char* b = tile + (vat ^ (i / KV * L::block * 16)) + i % KV * C * L::vbytes;
#pragma unroll
                    for (int j = 0; j < 4; ++j) f[i % 3][j] = *reinterpret_cast<const float*>(b + j * L::vbytes);
                };
                read_values(0);
                read_values(1);
#pragma unroll
                for (int i = 0; i < kSteps; ++i) {
                    if (i + 2 < kSteps) read_values(i + 2);
                    __builtin_amdgcn_sched_barrier(0);
                    acc[i / KV] = attn_mma<T>(__builtin_bit_cast(u32x4, f[i % 3]), __builtin_bit_cast(u32x4, w[i % KV]), acc[i / KV]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        t = tn;
    }
    const float lw = rows_sum<C>(l);
    if (c0 + wave * C + col >= ncols) return;
    auto four = [&](int v) { return f32x4{acc[v / C][v % C / 8 * 4], acc[v / C][v % C / 8 * 4 + 1], acc[v / C][v % C / 8 * 4 + 2], acc[v / C][v % C / 8 * 4 + 3]}; };      // outputs v + 4 g ..
    constexpr int kOut = 4 * G;                          // outputs of a column from one of a lane's four to the next
    if (in_parts) {
        const size_t row = ((size_t)split * a.T + tok) * a.H + head;
        if (g == 0) *reinterpret_cast<float2*>(a.ml + row * 2) = make_float2(m, lw);
        float* p = a.part + row * (a.vtiles * 16) + g * 4;
#pragma unroll
        for (int v = 0; v < NT; v += kOut)
            if (v < a.vtiles * 16) *reinterpret_cast<f32x4*>(p + v) = four(v);
        return;
    }
    const float snk = a.sink != nullptr ? a.sink[head] * kLog2e : kNegBig, mm = fmaxf(m, snk), c = fast_exp2(m - mm);
    const float f = c / (lw * c + fast_exp2(snk - mm));                // (no sink: the last term is zero)
    T* o = reinterpret_cast<T*>(a.out + (size_t)tok * a.ldo) + head * a.V;
    const float* gate = a.gate + (size_t)tok * a.ldg + head * a.V;
    const bool fours = (a.V & 3) == 0;
#pragma unroll
    for (int v = 0; v < NT; v += kOut)
        if (v < a.vtiles * 16) {
            const int v0 = v + g * 4;
            const f32x4 x = four(v);
            f32x4 y;
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = a.gate != nullptr && v0 + r < a.V ? x[r] * f * sigmoid(gate[v0 + r]) : x[r] * f;
            if (fours) {
                if (v0 < a.V) store4<T>(o + v0, y);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (v0 + r < a.V) o[v0 + r] = from_f32<T>(y[r]);
            }
        }
}

// Workgroup (token, 256 groups of four output columns): the splits' sums, relative to the largest maximum, with the sink and the
// gate.  At most S splits, all of them requested before the first is used.
template <typename T, int S>
__global__ __launch_bounds__(kSeqThreads) void k_seq_attn_merge(SeqAttn a) {
    const int t = blockIdx.x, per = a.vtiles * 4, i = blockIdx.y * kSeqThreads + threadIdx.x, h = i / per, v0 = (i - h * per) * 4;
    if (h >= a.H) return;
    const size_t row0 = (size_t)t * a.H + h, step = (size_t)a.T * a.H;
    float2 ml[S];
    f32x4 p[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < a.splits) {
            ml[s] = *reinterpret_cast<const float2*>(a.ml + (row0 + s * step) * 2);
            p[s] = *reinterpret_cast<const f32x4*>(a.part + (row0 + s * step) * (a.vtiles * 16) + v0);
        }
    const float snk = a.sink != nullptr ? a.sink[h] * kLog2e : kNegBig;
    float m = snk;
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < a.splits) m = fmaxf(m, ml[s].x);
    float l = fast_exp2(snk - m);
    f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < a.splits) {
            const float c = fast_exp2(ml[s].x - m);
            l = fmadd(ml[s].y, c, l);
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = fmadd(p[s][r], c, y[r]);
        }
    T* o = reinterpret_cast<T*>(a.out + (size_t)t * a.ldo) + h * a.V;
    const float* gate = a.gate + (size_t)t * a.ldg + h * a.V;
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = a.gate != nullptr && v0 + r < a.V ? y[r] / l * sigmoid(gate[v0 + r]) : y[r] / l;
    if ((a.V & 3) == 0) {
        if (v0 < a.V) store4<T>(o + v0, y);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (v0 + r < a.V) o[v0 + r] = from_f32<T>(y[r]);
    }
}

}  // namespace cfpp
