// Attention of a portion of the sequence models (device code; included by seq_kernels.hip).
#pragma once
#include <type_traits>

#include "seq_device.hpp"

namespace cfpp {

// The query columns of one key / value head are (token, head of the group), head fastest; a workgroup takes 64 CT of them
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
    int T, H, R, dsteps, qrow, krow, vrow, V, vtiles, pos0, chunk, cap, rows, ldo, k_split, runits, rrow, ldg;
    float scale_log2;
    int splits;
    float *part, *ml;        // splits > 1: [splits][T][H][16 vtiles], [splits][T][H][2]
};
template <int UN> __device__ __forceinline__ int swz_key(int row) { return UN % 16 ? (row >> 1) & 7 : row & 15; }

// the other half of the wave, the other rows of 16 lanes of each half: maximum and sum over all four row groups of a column
__device__ __forceinline__ float rows_max(float v) {
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float rows_sum(float v) {
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// Tiles of KT keys in LDS: NK elements of a key, NT value columns.  Two buffers, filled by copies that go there directly: the next
// tile's are on their way while one is worked on.  Key rows are stored in units of 16 bytes, permuted by swz_key.  Value rows stay
// rows: their fragments, four keys of a column per lane, come from transposing reads (bf16) or element by element (fp32), and
// blocks of 16 columns are permuted so that the rows that a read takes together start in different banks.
template <typename T, int NK, int NT> struct AttnTile {
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
        return sizeof(T) == 4 ? (row >> 2) & 3 : NT >= 128 ? row & 7 : (row >> 1) & 3;
    }
};

// What bounds it: the matrix cores and the softmax's vector instructions, which take turns inside a wave and overlap with the other
// wave of the SIMD.  So two workgroups per compute unit, one barrier per tile, and nothing is waited for but the tile itself: with
// copies that the compiler knows of it waited for the next tile's before this tile's first read of LDS, and values took a detour
// through registers to be transposed.  8000 tokens, 32 heads of 192 and 128: 1753 -> 1237 us; 2048 tokens, 128 and 128: 141 -> 103 us
// (before the order of the workgroups was changed, below).
// 37 tokens at 1990, 32 / 8 heads: 85 -> 12 us and 5 for the merge (24 workgroups became 384).
// (NK: elements of a key row in LDS, NT: value columns.  The products run over all of them, without branches between the reads
// of LDS: past the end of the query there are zeros, and of the columns past the end of a value nothing is stored.
// SH: keys have a shared part)
template <typename T, int NK, int NT, int CT, bool SH>
__global__ __launch_bounds__(kSeqThreads, (NT <= 128 ? 2 : 1)) void k_seq_attn(SeqAttn a) {
    using L = AttnTile<T, NK, NT>;
    constexpr int KT = L::keys, KS = L::kbytes / 64;
    extern __shared__ __align__(1024) char lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 15, g = lane >> 4;
    // The longest walks of all key heads first, so that the short ones fill the chip's last moments (head by head, a quarter of the compute
    // units' time was a tail: 8000 tokens, 32 heads of 192 and 128: 1264 -> 956 us; 2048 tokens, 128 and 128: 104 -> 86 us); and where the heads are a
    // multiple of eight, all workgroups of a head are on one XCD and walk its keys side by side.
    const int ncols = a.T * a.R, gx = (ncols + 64 * CT - 1) / (64 * CT), G = a.H / a.R, bx = blockIdx.x / G, gq = blockIdx.x - bx * G;
    const int c0 = (gx - 1 - bx) * 64 * CT;

    // (its sign goes to the query; not zero, so that it keeps the scores of keys that are not seen at -infinity; NaN stays NaN)
    const float size = fabsf(a.scale_log2), scale = size < 1e-30f ? 1e-30f : size;
    int pq[CT], first[CT], tok[CT], head[CT];
    u32x4 qf[CT][KS];
    float m[CT], l[CT];                                  // running maximum (log2 domain), this lane's share of the denominator
    f32x4 acc[CT][NT / 16];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int cc = min(c0 + (wave * CT + ct) * 16 + col, ncols - 1);
        tok[ct] = cc / a.R;
        head[ct] = gq * a.R + (cc - tok[ct] * a.R);
        pq[ct] = a.pos0 + tok[ct];
        first[ct] = chunk_start(pq[ct], a.chunk);
        const char* qr = a.q + ((size_t)tok[ct] * a.H + head[ct]) * a.qrow + g * 16;
        const uint32_t flip = a.scale_log2 < 0.0f ? (sizeof(T) == 2 ? 0x80008000u : 0x80000000u) : 0u;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            qf[ct][s] = ld16(qr + min(s, a.dsteps - 1) * 64) ^ u32x4{flip, flip, flip, flip};
            if (s >= a.dsteps) qf[ct][s] = u32x4{0, 0, 0, 0};
        }
        m[ct] = kNegBig;
        l[ct] = 0.0f;
#pragma unroll
        for (int i = 0; i < NT / 16; ++i) acc[ct][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // keys the workgroup needs, and those every column of this wave sees / any column sees
    const int t_first = c0 / a.R, t_last = min(a.T - 1, (c0 + 64 * CT - 1) / a.R);
    const int k_first = chunk_start(a.pos0 + t_first, a.chunk), k_end = a.pos0 + t_last + 1;
    const int w_first = min(c0 + wave * CT * 16, ncols - 1) / a.R, w_last = min(c0 + (wave + 1) * CT * 16 - 1, ncols - 1) / a.R;
    const int all_lo = chunk_start(a.pos0 + w_last, a.chunk), all_hi = a.pos0 + w_first;
    const int any_lo = chunk_start(a.pos0 + w_first, a.chunk), any_hi = a.pos0 + w_last;
    const int dunits = a.krow / 16, vunits = a.vrow / 16;

    // tiles: [k_first, k_split) in the cache, then [k_split, k_end) in the buffer; this split's are t0 .. t1 - 1
    const int in_cache = max(0, min(k_end, a.k_split) - k_first), n_cached = (in_cache + KT - 1) / KT, new_first = max(k_first, a.k_split);
    const int ntiles = n_cached + (max(0, k_end - new_first) + KT - 1) / KT, split = blockIdx.y;
    const int t0 = mul_div(ntiles, split, a.splits), t1 = mul_div(ntiles, split + 1, a.splits);
    struct Tile { int k0, hi; const char *k, *v; };      // first key, end of its part, row of position 0
    auto tile_at = [&](int i) {
        const bool cached = i < n_cached;
        const int k0 = cached ? k_first + i * KT : new_first + (i - n_cached) * KT;
        const ptrdiff_t row0 = (ptrdiff_t)gq * (cached ? a.rows : a.cap) - (cached ? chunk_start(a.pos0, a.chunk) : a.k_split);
        return Tile{k0, cached ? min(k_end, a.k_split) : k_end, (cached ? a.kc : a.k) + row0 * a.krow, (cached ? a.vc : a.v) + row0 * a.vrow};
    };
    // the lane's place in the copies: row of the tile, unit of its source row (the shared part comes from rows of its own)
    const uint32_t l0 = lds_address(lds);
    uint32_t koff[L::kp], voff[L::vp], shared = 0;       // bit i of shared: copy i takes from the shared part
#pragma unroll
    for (int i = 0; i < L::kp; ++i) {
        const int p = (i * kSeqWaves + wave) * 64 + lane, r = p / L::ku, u = (p % L::ku) ^ swz_key<L::ku>(r);
        const bool sh = SH && u >= dunits && u < dunits + a.runits;
        shared |= (uint32_t)sh << i;
        koff[i] = sh ? r * a.rrow + (u - dunits) * 16 : r * a.krow + (u < dunits ? u : 0) * 16;
    }
#pragma unroll
    for (int i = 0; i < L::vp; ++i) {
        const int p = (i * kSeqWaves + wave) * 64 + lane, r = p / L::vu, u = (p % L::vu) ^ (L::vswz(r) * L::block);
        voff[i] = r * a.vrow + min(u, vunits - 1) * 16;
    }
    auto fetch = [&](const Tile& t, int buf) __attribute__((always_inline)) {
        const uint32_t d = l0 + buf * L::size + wave * 1024;
        // rows past the end (`whole` false): the last one again
        auto copies = [&](auto whole) __attribute__((always_inline)) {
            constexpr bool W = decltype(whole)::value;
            const int last = t.hi - 1 - t.k0;
#pragma unroll
            for (int i = 0; i < L::kcopies; ++i) {
                const int r0 = i / L::kp * L::krows, r = r0 + ((i % L::kp) * kSeqWaves * 64 + wave * 64 + lane) / L::ku;
                const bool sh = SH && ((shared >> (i % L::kp)) & 1);
                const char *kb = uniform(t.k + (ptrdiff_t)(t.k0 + r0) * a.krow), *rb = SH ? uniform(a.kr + (ptrdiff_t)(t.k0 + r0) * a.rrow) : nullptr;
                const uint32_t to = d + i * (kSeqWaves * 1024);
                int o = (int)koff[i % L::kp];
                if (!W) o -= max(0, r - last) * (sh ? a.rrow : a.krow);
                if constexpr (W && !SH) copy_to_lds16_at((uint32_t)o, kb, to);
                else copy_to_lds16_from((sh ? rb : kb) + o, to);
            }
#pragma unroll
            for (int i = 0; i < L::vcopies; ++i) {
                const int r0 = i / L::vp * L::vrows, r = r0 + ((i % L::vp) * kSeqWaves * 64 + wave * 64 + lane) / L::vu;
                const char* vb = uniform(t.v + (ptrdiff_t)(t.k0 + r0) * a.vrow);
                const uint32_t to = d + L::ksize + i * (kSeqWaves * 1024);
                if constexpr (W) copy_to_lds16_at(voff[i % L::vp], vb, to);
                else copy_to_lds16_from(vb + (int)voff[i % L::vp] - max(0, r - last) * a.vrow, to);
            }
        };
        if (t.k0 + KT <= t.hi) copies(std::true_type{});
        else copies(std::false_type{});
    };
    // value fragments: the lane's rows start at key 4 g (bf16: with the transposing read, lane col of a group of 16 reads 8 bytes of
    // key 4 g + col / 4 and receives four keys of column col)
    const int vrow0 = sizeof(T) == 2 ? 4 * g + (col >> 2) : 4 * g, vsw = L::vswz(vrow0);
    int vat[NT / 16];
#pragma unroll
    for (int i = 0; i < NT / 16; ++i)
        vat[i] = L::ksize + vrow0 * L::vbytes + (i ^ vsw) * L::block * 16 + (sizeof(T) == 2 ? (col & 3) * 8 : col * 4);

    Tile t{};
    if (t0 < t1) {
        t = tile_at(t0);
        fetch(t, 0);
    }
    for (int it = t0, buf = 0; it < t1; ++it, buf ^= 1) {
        pipe_barrier<0>();                               // the tile is there, and nobody reads the other buffer any more
        Tile tn = t;
        if (it + 1 < t1) {
            tn = tile_at(it + 1);
            fetch(tn, buf ^ 1);
        }
        const char* const tile = lds + buf * L::size;
        if (t.k0 <= any_hi && min(t.k0 + KT, t.hi) > any_lo) {
            // the fragments of the next 16 keys are read while these are multiplied
            f32x4 s[CT][KT / 16];
            u32x4 kf[2][KS];
            auto read = [&](int kt) __attribute__((always_inline)) {
                const int r = kt * 16 + col;
#pragma unroll
                for (int d = 0; d < KS; ++d)
                    kf[kt & 1][d] = *reinterpret_cast<const u32x4*>(tile + r * L::kbytes + ((d * 4 + g) ^ swz_key<L::ku>(r)) * 16);
            };
            read(0);
#pragma unroll
            for (int kt = 0; kt < KT / 16; ++kt) {
                if (kt + 1 < KT / 16) read(kt + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) s[ct][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int d = 0; d < KS; ++d)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) s[ct][kt] = mma16<T>(kf[kt & 1][d], qf[ct][d], s[ct][kt]);
            }
            __builtin_amdgcn_sched_barrier(0);
            const bool full = t.k0 + KT <= t.hi && t.k0 >= all_lo && t.k0 + KT - 1 <= all_hi;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                if (!full) {
                    int k0 = t.k0 + g * 4;
                    asm volatile("" : "+v"(k0));         // (the comparisons stay inside the branch)
                    const int hi = min(pq[ct], t.hi - 1) - k0, lo = first[ct] - k0;
#pragma unroll
                    for (int kt = 0; kt < KT / 16; ++kt)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (kt * 16 + r > hi || kt * 16 + r < lo) s[ct][kt][r] = -INFINITY;
                }
                float mx = -INFINITY;
#pragma unroll
                for (int kt = 0; kt < KT / 16; ++kt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[ct][kt][r]);
                const float mn = fmaxf(m[ct], rows_max(mx) * scale);
                if (__builtin_amdgcn_ballot_w64(mn != m[ct]) != 0) {
                    const float c = fast_exp2(m[ct] - mn);
                    l[ct] *= c;
#pragma unroll
                    for (int i = 0; i < NT / 16; ++i) acc[ct][i] *= c;
                    m[ct] = mn;
                }
#pragma unroll
                for (int kt = 0; kt < KT / 16; ++kt) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[ct][kt][r] = fast_exp2(fmadd(s[ct][kt][r], scale, -mn));
                    l[ct] += (s[ct][kt][0] + s[ct][kt][1]) + (s[ct][kt][2] + s[ct][kt][3]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);           // (values read ahead of the softmax would take its registers)
            if constexpr (sizeof(T) == 2) {
                u32x4 hi[CT][KT / 32], lo[CT][KT / 32];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int h = 0; h < KT / 32; ++h) split_weights(s[ct][2 * h], s[ct][2 * h + 1], hi[ct][h], lo[ct][h]);
#pragma unroll
                for (int i = 0; i < NT / 16; ++i)
#pragma unroll
                    for (int h = 0; h < KT / 32; ++h) {
                        const u32x2 x = read_transposed(tile + vat[i] + h * 32 * L::vbytes), y = read_transposed(tile + vat[i] + (h * 32 + 16) * L::vbytes);
                        const u32x4 f = {x.x, x.y, y.x, y.y};
#pragma unroll
                        for (int ct = 0; ct < CT; ++ct) acc[ct][i] = mma16<T>(f, hi[ct][h], acc[ct][i]);
#pragma unroll
                        for (int ct = 0; ct < CT; ++ct) acc[ct][i] = mma16<T>(f, lo[ct][h], acc[ct][i]);
                    }
            } else {
#pragma unroll
                for (int i = 0; i < NT / 16; ++i)
#pragma unroll
                    for (int h = 0; h < KT / 16; ++h) {
                        f32x4 f;
#pragma unroll
                        for (int j = 0; j < 4; ++j) f[j] = *reinterpret_cast<const float*>(tile + vat[i] + (h * 16 + j) * L::vbytes);
#pragma unroll
                        for (int ct = 0; ct < CT; ++ct) acc[ct][i] = mma16<T>(__builtin_bit_cast(u32x4, f), __builtin_bit_cast(u32x4, s[ct][h]), acc[ct][i]);
                    }
            }
        }
        t = tn;
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const float lw = rows_sum(l[ct]);
        if (c0 + (wave * CT + ct) * 16 + col >= ncols) continue;
        if (a.splits > 1) {
            const size_t row = ((size_t)split * a.T + tok[ct]) * a.H + head[ct];
            if (g == 0) *reinterpret_cast<float2*>(a.ml + row * 2) = make_float2(m[ct], lw);
            float* p = a.part + row * (a.vtiles * 16) + g * 4;
#pragma unroll
            for (int i = 0; i < NT / 16; ++i)
                if (i < a.vtiles) *reinterpret_cast<f32x4*>(p + i * 16) = acc[ct][i];
            continue;
        }
        const float snk = a.sink != nullptr ? a.sink[head[ct]] * kLog2e : kNegBig, mm = fmaxf(m[ct], snk), c = fast_exp2(m[ct] - mm);
        const float f = c / (lw * c + fast_exp2(snk - mm));            // (no sink: the last term is zero)
        T* o = reinterpret_cast<T*>(a.out + (size_t)tok[ct] * a.ldo) + head[ct] * a.V;
        const float* gate = a.gate + (size_t)tok[ct] * a.ldg + head[ct] * a.V;
        const bool fours = (a.V & 3) == 0;
#pragma unroll
        for (int i = 0; i < NT / 16; ++i)
            if (i < a.vtiles) {
                const int v0 = i * 16 + g * 4;
                f32x4 y;
#pragma unroll
                for (int r = 0; r < 4; ++r) y[r] = a.gate != nullptr && v0 + r < a.V ? acc[ct][i][r] * f * sigmoid(gate[v0 + r]) : acc[ct][i][r] * f;
                if (fours) {
                    if (v0 < a.V) store4<T>(o + v0, y);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (v0 + r < a.V) o[v0 + r] = from_f32<T>(y[r]);
                }
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
