// Latent attention and residual streams of the sequence models (device code; included by seq_kernels.hip).
//
// A latent mixer caches one row per position: the normed latent c (kv_rank values, padded to whole weight rows) and, behind
// it, the rotated key part that all heads share.
//   Portions: the plain keys and the values of all heads are made from the cached latents by one matrix product
//   (kEpiHeads) and attention runs over them head by head; the rotated part is read from the cache rows as it is.
//   Portions of few tokens behind many positions (plan_latent_turn): as in decode, for all columns (token, head) side by side (k_seq_latent_absorb,
//   k_seq_latent_block, k_seq_latent_turn_out).
//   Decode: the query is taken into the latent space instead, q' = W_uk^T q (k_seq_latent_q), all heads attend to the cache
//   rows themselves, as keys and as values (k_seq_latent_attn), and W_uv turns the weighted latents into the heads' outputs
//   (k_seq_latent_out, which also merges the splits).  A step reads the cache once instead of making keys and values.
#pragma once
#include <type_traits>

#include "seq_device.hpp"
#include "seq_plan.hpp"

namespace cfpp {

// (cos, sin) of pair j of a position; the pair is (j, j + R/2) or (2j, 2j + 1)
__device__ __forceinline__ int pair_first(int j, int R, int half) { return half ? j : 2 * j; }
__device__ __forceinline__ int pair_second(int j, int R, int half) { return half ? j + R / 2 : 2 * j + 1; }

// R rotated values of `row` to `out`, zeros up to `end` bytes; the workgroup's threads from `tid` on, `n` of them
template <typename T>
__device__ __forceinline__ void rotate_row(const float* __restrict__ row, char* out, int R, int end, int half, const float2* __restrict__ cs, int tid, int n) {
    T* o = reinterpret_cast<T*>(out);
    for (int j = tid; j < R / 2; j += n) {
        const float2 t = cs[j];
        const float u = row[pair_first(j, R, half)], v = row[pair_second(j, R, half)];
        o[pair_first(j, R, half)] = from_f32<T>(u * t.x - v * t.y);
        o[pair_second(j, R, half)] = from_f32<T>(v * t.x + u * t.y);
    }
    for (int j = R + tid; j < end / (int)sizeof(T); j += n) o[j] = from_f32<T>(0.0f);
}

// The latent row of one position: norm over the first `rank` values, rotation of the other R.
struct LatentRow {
    const float* w;          // [rank]
    int rank, R, rot_off, crow, half;
    float eps;
};
template <typename T>
__device__ __forceinline__ void latent_row(const LatentRow& a, const float* __restrict__ z, char* row, const float2* __restrict__ cs, float* red) {
    const float inv = inv_rms(block_sum(share_sq(z, a.rank, threadIdx.x), red), a.rank, a.eps);
    for (int i = threadIdx.x; i < a.rank; i += kSeqThreads) reinterpret_cast<T*>(row)[i] = from_f32<T>(z[i] * inv * a.w[i]);
    rotate_row<T>(z + a.rank, row + a.rot_off, a.R, a.crow - a.rot_off, a.half, cs, threadIdx.x, kSeqThreads);
}

// ---- portions ----------------------------------------------------------------------------------
// One workgroup per token: raw projection (fp32) -> queries [token][head][plain | rotated | zeros] and the cache row.
struct SeqLatentFinish {
    float* z;                // partial results of `parts` splits, part_stride floats apart; the first becomes their sum
    int ld, n, made, parts;  // values of a row that are read, those in front of its gates
    size_t part_stride;
    int own;                 // the layer makes cache rows
    LatentRow kv;
    const float2* cs;        // [positions][R / 2]
    int H, D, R, pos0, rot_at, qrow;      // rot_at: bytes in front of the rotated part of a query
    char *q, *kc;            // kc: cache row of position 0
};
template <typename T>
__global__ __launch_bounds__(kSeqThreads) void k_seq_latent_finish(SeqLatentFinish a) {
    __shared__ float red[kSeqWaves];
    const int t = blockIdx.x, n = a.D + a.R;
    merge_parts(a.z + (size_t)t * a.ld, a.n, a.parts, a.part_stride);
    const float* z = a.z + (size_t)t * a.ld;
    const float2* cs = a.cs + (size_t)(a.pos0 + t) * (a.R / 2);
    char* q = a.q + (size_t)t * a.H * a.qrow;
    if (a.own) latent_row<T>(a.kv, z + a.H * n, a.kc + (size_t)(a.pos0 + t) * a.kv.crow, cs, red);
    const int p4 = a.rot_at / (int)sizeof(T) / 4;        // groups of four plain values, padding included
    for (int i = threadIdx.x; i < a.H * p4; i += kSeqThreads) {
        const int h = i / p4, d = (i - h * p4) * 4;
        const float* row = z + h * n + d;
        f32x4 x;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = d + j < a.D ? row[j] : 0.0f;
        store4<T>(q + (size_t)h * a.qrow + d * sizeof(T), x);
    }
    const int end = a.qrow - a.rot_at, per = max(a.R / 2, end / (int)sizeof(T) - a.R);     // threads per head: pairs, zeros behind them
    for (int i = threadIdx.x; i < a.H * per; i += kSeqThreads) {
        const int h = i / per;
        rotate_row<T>(z + h * n + a.D, q + (size_t)h * a.qrow + a.rot_at, a.R, end, a.kv.half, cs, i - h * per, per);
    }
}

// The same where the row is whole groups of four values, up to 1024 U of them: everything is requested at once (of C parts together), and the
// row is read from LDS, where it took three or four round trips.  Gates are read only where they come in parts, and their sum goes back.
// 8000 tokens of 6720 values and 4096 gates: 100 -> 71 us for 330 MB.  U = 4 where the row fits, since places behind its end are requested like others:
// 150 tokens of 3648 in parts 6.4 us, with 8 groups 5.6, with 4 5.0; 100 of 1120 in parts 4.5, 5.6 and 4.7.  C = 0: a projection
// that is larger than the 256 MB cache is read from its end, and past the caches: 8000 tokens of 10816 values, of which 6720 are read, 71 -> 57 us (2048
// tokens 21.4 and 21.7, 4000 32 and 32; in rows of queries, keys and values 71 -> 67 for 8000 and 21.6 -> 22.4 for 2048, not done there).
template <typename T, int U, int C>
__global__ __launch_bounds__(kSeqThreads) void k_seq_latent_finish4(SeqLatentFinish a) {
    __shared__ float red[kSeqWaves];
    extern __shared__ __align__(16) char smem[];
    float* const row = reinterpret_cast<float*>(smem);   // [made], then the position's pairs
    float2* const pairs = reinterpret_cast<float2*>(row + a.made);
    const int t = C == 0 ? (int)(gridDim.x - 1 - blockIdx.x) : (int)blockIdx.x, tid = threadIdx.x, n = a.D + a.R, n4 = a.n / 4, kv0 = a.H * n;
    float* const z = a.z + (size_t)t * a.ld;
    f32x4 x[U];
#pragma unroll
    for (int j = 0; j < U; ++j) x[j] = load_row4<C == 0>(z, min(tid + j * kSeqThreads, n4 - 1));
    constexpr int kNorm = 2;                             // (a latent has 512 values at most)
    float w[kNorm];
#pragma unroll
    for (int j = 0; j < kNorm; ++j) w[j] = a.own ? a.kv.w[min(tid + j * kSeqThreads, a.kv.rank - 1)] : 0.0f;
    float2 pair = make_float2(0.0f, 0.0f);
    if (tid < a.R / 2) pair = a.cs[(size_t)(a.pos0 + t) * (a.R / 2) + tid];
    add_rows4<U, (C > 0 ? C : 1)>(x, z + a.part_stride, a.parts - 1, a.part_stride, n4);
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const int i = (tid + j * kSeqThreads) * 4;
        if (i < a.made) *reinterpret_cast<f32x4*>(row + i) = x[j];
        else if (i < a.n && a.parts > 1) *reinterpret_cast<f32x4*>(z + i) = x[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) ss = i + r >= kv0 && i + r < kv0 + a.kv.rank && i < a.made ? fmadd(x[j][r], x[j][r], ss) : ss;
    }
    if (tid < a.R / 2) pairs[tid] = pair;
    const float inv = inv_rms(block_sum(ss, red), a.kv.rank, a.kv.eps);         // (its barriers are behind the row's stores too)
    if (a.own) {
        char* const to = a.kc + (size_t)(a.pos0 + t) * a.kv.crow;
#pragma unroll
        for (int j = 0; j < kNorm; ++j) {
            const int i = tid + j * kSeqThreads;
            if (i < a.kv.rank) reinterpret_cast<T*>(to)[i] = from_f32<T>(row[kv0 + i] * inv * w[j]);
        }
        rotate_row<T>(row + kv0 + a.kv.rank, to + a.kv.rot_off, a.R, a.kv.crow - a.kv.rot_off, a.kv.half, pairs, tid, kSeqThreads);
    }
    char* const q = a.q + (size_t)t * a.H * a.qrow;
    const int p4 = a.rot_at / (int)sizeof(T) / 4;        // groups of four plain values, padding included
    for (int i = tid; i < a.H * p4; i += kSeqThreads) {
        const int h = i / p4, d = (i - h * p4) * 4;
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = d + j < a.D ? row[h * n + d + j] : 0.0f;
        store4<T>(q + (size_t)h * a.qrow + d * sizeof(T), v);
    }
    const int end = a.qrow - a.rot_at, per = max(a.R / 2, end / (int)sizeof(T) - a.R);     // threads per head: pairs, zeros behind them
    for (int i = tid; i < a.H * per; i += kSeqThreads) {
        const int h = i / per;
        rotate_row<T>(row + h * n + a.D, q + (size_t)h * a.qrow + a.rot_at, a.R, end, a.kv.half, pairs, i - h * per, per);
    }
}

// ---- one token ---------------------------------------------------------------------------------
// Workgroup (head, 128 bytes of latent columns): those columns of W_uk^T q, summed in fp32 over the head's plain dimensions.
// A thread owns one 16-byte unit of the columns and every 32nd dimension.  The first workgroup of a head also rotates the
// rest of its query; one more workgroup makes the position's cache row.
struct SeqLatentQ {
    const float* z;
    const int* state;
    const float2* cs;
    const char* w_uk;        // T [H * D][pitch bytes]
    int pitch, H, D, R, nrb, own;
    LatentRow kv;
    char* q;                 // T [H][kv.crow bytes]: q' padded to `pitch` bytes, then the rotated part
    char* kc;                // caches, slot 0
    size_t slot_bytes;
};
template <typename T>
__global__ __launch_bounds__(kSeqThreads) void k_seq_latent_q(SeqLatentQ a) {
    constexpr int U = Unit<T>::n, G = kSeqThreads / 8;   // elements per unit, dimension groups
    constexpr int kLoads = 4;
    __shared__ float red[kSeqWaves];
    __shared__ float part[kSeqWaves][8 * U];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = blockIdx.x / a.nrb, rb = blockIdx.x - h * a.nrb;
    const int pos = a.state[1];
    const float2* cs = a.cs + (size_t)pos * (a.R / 2);
    if (h == a.H) {
        latent_row<T>(a.kv, a.z + a.H * (a.D + a.R), a.kc + a.state[3] * a.slot_bytes + (size_t)pos * a.kv.crow, cs, red);
        return;
    }
    const float* z = a.z + h * (a.D + a.R);
    const char* w = a.w_uk + (size_t)h * a.D * a.pitch + rb * 128 + (tid & 7) * 16;
    float acc[U];
#pragma unroll
    for (int e = 0; e < U; ++e) acc[e] = 0.0f;
    for (int d0 = tid >> 3; d0 < a.D; d0 += G * kLoads) {
        u32x4 b[kLoads];
        float x[kLoads];
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int d = min(d0 + i * G, a.D - 1);
            b[i] = ld16(w + (size_t)d * a.pitch);
            x[i] = d0 + i * G < a.D ? z[d] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            float v[U];
            unpack16<T>(b[i], v);
#pragma unroll
            for (int e = 0; e < U; ++e) acc[e] = fmadd(v[e], x[i], acc[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < U; ++e) {                        // lanes of the same unit
        acc[e] += xor_shfl(acc[e], 8);
        acc[e] += xor_shfl(acc[e], 16);
        acc[e] += xor_shfl(acc[e], 32);
    }
    if (lane < 8) {
#pragma unroll
        for (int e = 0; e < U; ++e) part[wave][lane * U + e] = acc[e];
    }
    __syncthreads();
    char* q = a.q + (size_t)h * a.kv.crow;
    if (tid < 8 * U) reinterpret_cast<T*>(q + rb * 128)[tid] = from_f32<T>((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]));
    if (rb == 0) rotate_row<T>(z + a.D, q + a.kv.rot_off, a.R, a.kv.crow - a.kv.rot_off, a.kv.half, cs, tid, kSeqThreads);
}

// Tiles of keys of a decode step, and how many workgroups share them: a few tiles each while that keeps the number of partial
// results, which every workgroup of k_seq_latent_out reads for its head, small.
template <typename T> struct LatentTile { static constexpr int keys = sizeof(T) == 2 ? 32 : 16; };
template <typename T> __device__ __forceinline__ int latent_tiles(int pos) { return (pos + LatentTile<T>::keys) / LatentTile<T>::keys; }
__device__ __forceinline__ int latent_splits(int tiles, int most, int least) { return min(most, (tiles + least - 1) / least); }

// Column fragments of c^T for the second product, for eight (or two) sets of 16 latent columns: keys 4g .. 4g + 3 (x) and 16 + 4g .. (y) of
// column lane & 15, from a tile of cache rows in LDS; `p`, `q`: the lane's place in the rows of the one and the other.  The reads
// and their wait are written out: behind its own transposed reads the compiler would also wait for the copies to the other buffers.
struct TrCols { u32x2 x, y; };
__device__ __forceinline__ void tr_read8(TrCols (&f)[8], uint32_t p, uint32_t q) {
    asm volatile(
        "ds_read_b64_tr_b16 %0, %16\n\tds_read_b64_tr_b16 %1, %17\n\t"
        "ds_read_b64_tr_b16 %2, %16 offset:32\n\tds_read_b64_tr_b16 %3, %17 offset:32\n\t"
        "ds_read_b64_tr_b16 %4, %16 offset:64\n\tds_read_b64_tr_b16 %5, %17 offset:64\n\t"
        "ds_read_b64_tr_b16 %6, %16 offset:96\n\tds_read_b64_tr_b16 %7, %17 offset:96\n\t"
        "ds_read_b64_tr_b16 %8, %16 offset:128\n\tds_read_b64_tr_b16 %9, %17 offset:128\n\t"
        "ds_read_b64_tr_b16 %10, %16 offset:160\n\tds_read_b64_tr_b16 %11, %17 offset:160\n\t"
        "ds_read_b64_tr_b16 %12, %16 offset:192\n\tds_read_b64_tr_b16 %13, %17 offset:192\n\t"
        "ds_read_b64_tr_b16 %14, %16 offset:224\n\tds_read_b64_tr_b16 %15, %17 offset:224\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(f[0].x), "=&v"(f[0].y), "=&v"(f[1].x), "=&v"(f[1].y), "=&v"(f[2].x), "=&v"(f[2].y), "=&v"(f[3].x), "=&v"(f[3].y), "=&v"(f[4].x),
          "=&v"(f[4].y), "=&v"(f[5].x), "=&v"(f[5].y), "=&v"(f[6].x), "=&v"(f[6].y), "=&v"(f[7].x), "=&v"(f[7].y)
        : "v"(p), "v"(q)
        : "memory");
}
__device__ __forceinline__ void tr_read2(TrCols (&f)[2], uint32_t p, uint32_t q) {
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %1, %5\n\t"
        "ds_read_b64_tr_b16 %2, %4 offset:32\n\tds_read_b64_tr_b16 %3, %5 offset:32\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(f[0].x), "=&v"(f[0].y), "=&v"(f[1].x), "=&v"(f[1].y)
        : "v"(p), "v"(q)
        : "memory");
}

// Workgroup (split, group of heads).  Four waves: RW of them share 16 heads, each with its part of the scores' dimensions (the
// parts are added through LDS, in the same order by all of them) and of the output's latent columns; 4 / RW sets of 16 heads.
// Tiles of cache rows go through buffers in LDS, two ahead, and
// serve as keys (row fragments) and as values (transposed reads).  A row in LDS has room for NR latents and 128 rotated values
// and an odd number of 16-byte units; past the end of the cache row its last unit is repeated, which meets zeros in the query
// and columns that are not stored.
struct SeqLatentAttn {
    const char* q;           // T [H][crow bytes]
    const char* kc;          // caches, slot 0
    size_t slot_bytes;
    const int* state;
    float *acc, *ml;         // [ns][H][rp], [ns][H][2]
    float scale_log2;
    int H, crow, ns, least, rp;      // least: tiles of a split
};
template <typename T, int NR> struct LatentLds {
    static constexpr int ksteps = (NR + 128) * (int)sizeof(T) / 64, up = ksteps * 4 + 1;
    static constexpr int copies = (LatentTile<T>::keys * up + 255) / 256;            // 1 KB copies per wave and tile
    static constexpr int tile = copies * kSeqWaves * 1024, buffers = 3;
};

// 64 units of the tile per copy, the waves in turn
template <typename T, int NR>
__device__ __forceinline__ void latent_stage(char* __restrict__ tile, const char* __restrict__ kc, int crow, int kb, int last, int wave, int lane) {
    using L = LatentLds<T, NR>;
    const int units = crow / 16;
#pragma unroll
    for (int i = 0; i < L::copies; ++i) {
        const int c = i * kSeqWaves + wave, l = c * 64 + lane, r = l / L::up, u = l - r * L::up;
        copy_to_lds16(kc + (size_t)min(kb + r, last) * crow + min(u, units - 1) * 16, tile + c * 1024);
    }
}

// One tile: the copies of a later one, scores, softmax, second product.  `parts`: [wave][KF][lane].
template <typename T, int NR, int RW>
__device__ __forceinline__ void latent_tile(AttnState<NR / RW>& st, const u32x4 (&qf)[LatentLds<T, NR>::ksteps / RW], const char* __restrict__ tile,
                                            char* __restrict__ next, bool more, f32x4* __restrict__ parts, const char* __restrict__ kc, int crow, int kb, int kn,
                                            int k1, float scale_log2, int rw, int wave, int lane) {
    using L = LatentLds<T, NR>;
    constexpr int KT = LatentTile<T>::keys, KF = KT / 16, NW = NR / RW, KS = L::ksteps / RW;
    static_assert(L::ksteps % RW == 0, "");
    const int col = lane & 15, g = lane >> 4;
    if (more) latent_stage<T, NR>(next, kc, crow, kn, k1 - 1, wave, lane);
    f32x4 s[KF];
    u32x4 kf[KS][KF];
#pragma unroll
    for (int d = 0; d < KS; ++d)
#pragma unroll
        for (int kt = 0; kt < KF; ++kt) kf[d][kt] = *reinterpret_cast<const u32x4*>(tile + ((kt * 16 + col) * L::up + (rw * KS + d) * 4 + g) * 16);
    __builtin_amdgcn_sched_barrier(0);                   // (all reads are requested before the first product waits for one)
#pragma unroll
    for (int kt = 0; kt < KF; ++kt) {
        s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < KS; ++d) s[kt] = mma16<T>(kf[d][kt], qf[d], s[kt]);
    }
#pragma unroll
    for (int kt = 0; kt < KF; ++kt) parts[(wave * KF + kt) * kWave + lane] = s[kt];
    lds_barrier();
#pragma unroll
    for (int kt = 0; kt < KF; ++kt) {
        f32x4 p[RW];
#pragma unroll
        for (int w = 0; w < RW; ++w) p[w] = parts[((wave - rw + w) * KF + kt) * kWave + lane];
        s[kt] = p[0];
#pragma unroll
        for (int w = 1; w < RW; ++w) s[kt] += p[w];
    }
#pragma unroll
    for (int kt = 0; kt < KF; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[kt][r] = kb + kt * 16 + g * 4 + r < k1 ? s[kt][r] * scale_log2 : kMasked;
    attn_softmax<NW, KF>(st, s, NW / 16);
    if constexpr (sizeof(T) == 2) {
        u32x4 hi, lo;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            f32x4 rest;
#pragma unroll
            for (int r = 0; r < 4; ++r) rest[r] = s[kt][r] - (float)(bf16_t)s[kt][r];
            hi[2 * kt] = pack_bf16(s[kt][0], s[kt][1]);
            hi[2 * kt + 1] = pack_bf16(s[kt][2], s[kt][3]);
            lo[2 * kt] = pack_bf16(rest[0], rest[1]);
            lo[2 * kt + 1] = pack_bf16(rest[2], rest[3]);
        }
        constexpr int B = NW >= 128 ? 8 : 2;             // sets of 16 columns read together
        const uint32_t v = (uint32_t)(uintptr_t)(tile + (4 * g + (col >> 2)) * L::up * 16 + rw * NW * 2 + (col & 3) * 8);
#pragma unroll
        for (int i = 0; i < NW / 16; i += B) {
            TrCols c[B];
            if constexpr (B == 8) tr_read8(c, v + i * 32, v + i * 32 + 16 * L::up * 16);
            else tr_read2(c, v + i * 32, v + i * 32 + 16 * L::up * 16);
#pragma unroll
            for (int j = 0; j < B; ++j) {
                const u32x4 f = {c[j].x.x, c[j].x.y, c[j].y.x, c[j].y.y};
                st.acc[i + j] = mma16<T>(f, hi, st.acc[i + j]);
                st.acc[i + j] = mma16<T>(f, lo, st.acc[i + j]);
            }
        }
    } else {
        const char* v = tile + 4 * g * L::up * 16 + (rw * NW + col) * 4;
#pragma unroll
        for (int i = 0; i < NW / 16; ++i) {
            f32x4 f;
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] = *reinterpret_cast<const float*>(v + j * L::up * 16 + i * 64);
            st.acc[i] = mma16<T>(__builtin_bit_cast(u32x4, f), __builtin_bit_cast(u32x4, s[0]), st.acc[i]);
        }
    }
}

template <typename T, int NR, int RW>
__global__ __launch_bounds__(kSeqThreads, 1) void k_seq_latent_attn(SeqLatentAttn a) {
    using L = LatentLds<T, NR>;
    constexpr int KT = LatentTile<T>::keys, NW = NR / RW, KS = L::ksteps / RW;
    extern __shared__ __align__(1024) char tiles[];
    __shared__ f32x4 parts[kSeqWaves * (KT / 16) * kWave];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 15, g = lane >> 4;
    const int rw = wave % RW, h0 = ((int)blockIdx.y * (kSeqWaves / RW) + wave / RW) * 16;
    const int pos = a.state[1], ntiles = latent_tiles<T>(pos), nsplit = latent_splits(ntiles, a.ns, a.least), sp = blockIdx.x;
    if (sp >= nsplit) return;
    const int k0 = mul_div(ntiles, sp, nsplit) * KT, k1 = min(mul_div(ntiles, sp + 1, nsplit) * KT, pos + 1);
    const char* kc = a.kc + a.state[3] * a.slot_bytes;
    const int ksteps = a.crow / 64;
    const char* qr = a.q + (size_t)min(h0 + col, a.H - 1) * a.crow + g * 16;
    u32x4 qf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        qf[s] = ld16(qr + min(rw * KS + s, ksteps - 1) * 64);
        if (rw * KS + s >= ksteps) qf[s] = u32x4{0, 0, 0, 0};
    }
    latent_stage<T, NR>(tiles, kc, a.crow, k0, k1 - 1, wave, lane);
    if (k0 + KT < k1) latent_stage<T, NR>(tiles + L::tile, kc, a.crow, k0 + KT, k1 - 1, wave, lane);
    AttnState<NW> st;
    attn_reset(st);
    int buf = 0;
    for (int kb = k0; kb < k1; kb += KT) {
        // this wave's copies of the tile have arrived (the next tile's may be on their way), then everybody's; and nobody reads
        // the buffer of the tile before any more
        if (kb + KT < k1) wait_vm<L::copies>();
        else wait_vm<0>();
        lds_barrier();
        const int ahead = buf == 0 ? 2 : buf - 1;        // (buf + 2) % 3
        latent_tile<T, NR, RW>(st, qf, tiles + buf * L::tile, tiles + ahead * L::tile, kb + 2 * KT < k1, parts, kc, a.crow, kb, kb + 2 * KT, k1, a.scale_log2, rw,
                               wave, lane);
        buf = buf == 2 ? 0 : buf + 1;
    }
    if (h0 + col >= a.H) return;
    const size_t row = (size_t)sp * a.H + h0 + col;
    if (rw == 0 && g == 0) *reinterpret_cast<float2*>(a.ml + row * 2) = make_float2(st.m, st.l);
#pragma unroll
    for (int i = 0; i < NW / 16; ++i)
        if (rw * NW + i * 16 < a.rp) *reinterpret_cast<f32x4*>(a.acc + row * a.rp + rw * NW + i * 16 + g * 4) = st.acc[i];
}

// Workgroup (head, kLatentOut of its outputs; the head runs fastest, which keeps the workgroups of one head, who read the same
// partial results, on few XCDs): merges the splits of the head, then its rows of W_uv, four per wave, in fp32, and
// the output gate.
// It is bound by the partial results, which every workgroup of a head reads: 32 heads of 512 latents behind 4096 positions, 65 splits, 133 KB.  The splits'
// maxima go ahead of them: a step of 32 such layers 3049 -> 3027 us.  (kM: loads in flight per thread.  With 36, one round trip for 65 splits, 3022; over nine models
// and nine contexts between 2.5 % less, for 8 heads behind 8000 positions, and 4 % more, for 48 heads behind 4096: two workgroups per compute unit instead of four.)
constexpr int kLatentOut = 16;
constexpr int kLatentSplits = kSeqThreads;
struct SeqLatentOut {
    const float *acc, *ml;
    const int* state;
    const float* sink;       // nullable
    const float* gate;       // nullable: [H * V] before the sigmoid
    const char* w_uv;        // T [H * V][pitch bytes]
    char* out;               // T [H * V]
    int H, V, pitch, ns, least, rp;
};
template <typename T>
__global__ __launch_bounds__(kSeqThreads) void k_seq_latent_out(SeqLatentOut a) {
    constexpr int U = Unit<T>::n, RPW = kLatentOut / kSeqWaves, NC = sizeof(T) == 2 ? 1 : 2;     // rows per wave, 1 KB loads per row
    __shared__ float f[kLatentSplits], red[kSeqWaves];
    __shared__ __align__(16) float sum[kSeqThreads * 4];
    __shared__ __align__(16) float lat[NC * 64 * U];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = blockIdx.x, v0 = blockIdx.y * kLatentOut;
    // What is needed first is requested first: a thread's split's maximum and denominator (past the splits: unused), its rows of W_uv, and, once the
    // number of splits is known, the partial results.  A thread sums four latent columns over every nsg-th split; the first kM of these are
    // requested together, before their weights are known.
    float2 ml = *reinterpret_cast<const float2*>(a.ml + ((size_t)min(tid, a.ns - 1) * a.H + h) * 2);
    const float snk = a.sink != nullptr ? a.sink[h] * kLog2e : kNegBig;
    u32x4 b[RPW][NC];
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
        const int v = min(v0 + wave * RPW + i, a.V - 1);
#pragma unroll
        for (int c = 0; c < NC; ++c) b[i][c] = ld16(a.w_uv + ((size_t)h * a.V + v) * a.pitch + min(c * 1024 + lane * 16, a.pitch - 16));
    }
    const int nsplit = latent_splits(latent_tiles<T>(a.state[1]), a.ns, a.least);
    const int r4 = a.rp / 4, nsg = kSeqThreads / r4, sg = tid / r4, x = tid - sg * r4;
    const float* p = a.acc + (size_t)h * a.rp + x * 4;
    const size_t split_stride = (size_t)a.H * a.rp;
    constexpr int kM = 16;
    f32x4 t[kM];
    auto request = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kM; ++j) {
            if (j % 4 == 0 && s0 + j * nsg >= nsplit) break;         // (the same for the workgroup)
            t[j] = *reinterpret_cast<const f32x4*>(p + min(s0 + sg + j * nsg, nsplit - 1) * split_stride);
        }
    };
    request(0);
    __builtin_amdgcn_sched_barrier(0);
    if (tid >= nsplit) ml = make_float2(kNegBig, 0.0f);              // (at most one split per thread)
    const float wm = wave_max(ml.x);
    if (lane == 0) red[wave] = wm;
    __syncthreads();
    const float m = fmaxf(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])), snk), e = fast_exp2(ml.x - m);
    const float l = block_sum(ml.y * e, red) + (a.sink != nullptr ? fast_exp2(snk - m) : 0.0f);
    f[tid] = e / l;
    for (int i = tid; i < NC * 64 * U; i += kSeqThreads) lat[i] = 0.0f;
    __syncthreads();
    if (sg < nsg) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < nsplit; s0 += nsg * kM) {
            if (s0 > 0) request(s0);
#pragma unroll
            for (int j = 0; j < kM; ++j) {
                if (j % 4 == 0 && s0 + j * nsg >= nsplit) break;
                const int k = s0 + sg + j * nsg;
                const bool live = k < nsplit;            // (a split's values may be infinite: not times zero)
                const float w = f[min(k, nsplit - 1)];
#pragma unroll
                for (int c = 0; c < 4; ++c) s[c] = live ? fmadd(t[j][c], w, s[c]) : s[c];
            }
        }
        *reinterpret_cast<f32x4*>(sum + sg * a.rp + x * 4) = s;
    }
    __syncthreads();
    for (int i = tid; i < a.rp; i += kSeqThreads) {
        float s = 0.0f;
        for (int j = 0; j < nsg; ++j) s += sum[j * a.rp + i];
        lat[i] = s;
    }
    __syncthreads();
    float acc[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        float y[U];
        const bool in = c * 1024 + lane * 16 < a.pitch;
#pragma unroll
        for (int e = 0; e < U; ++e) y[e] = in ? lat[(c * 64 + lane) * U + e] : 0.0f;
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            float w[U];
            unpack16<T>(b[i][c], w);
#pragma unroll
            for (int e = 0; e < U; ++e) acc[i] = fmadd(w[e], y[e], acc[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < RPW; ++i) acc[i] = wave_sum(acc[i]);
    if (lane < RPW) {
        float o = 0.0f;
#pragma unroll
        for (int i = 0; i < RPW; ++i) o = lane == i ? acc[i] : o;
        const int v = v0 + wave * RPW + lane;
        if (v < a.V) {
            if (a.gate != nullptr) o *= sigmoid(a.gate[h * a.V + v]);
            reinterpret_cast<T*>(a.out)[h * a.V + v] = from_f32<T>(o);
        }
    }
}

// ---- portions of few tokens behind many positions ----------------------------------------------
// The same three passes as for one token, for the columns (token, head) of a portion, head fastest: the cache is read as it is, and no keys and
// values are made of it.  A column costs a portion's products of kv_rank instead of dim and vdim values for every key, so it is for few tokens (plan_latent_turn).  What it
// replaces at 3000 positions: 16 heads 20 us for the keys and values, 12 for the attention and 5 for its merge; 128 heads 90, 60 and 8.

// Queries into the latent space: workgroup (head, 64 latent columns, tokens), W_uk^T q from the rows that k_seq_latent_finish has made.  A wave owns 16
// of the columns; W_uk, whose rows are dimensions, is taken through LDS, where a product's operand is read down its columns.
struct SeqLatentAbsorb {
    const char* q;           // T [tokens][H][qrow bytes]: plain part, at `plain` bytes the rotated part
    const char* w_uk;        // T [H * D][pitch bytes]
    char* out;               // T [tokens][H][crow bytes]: q' padded to `pitch` bytes, then the rotated part
    int n, pitch, H, D, R, ncb, qrow, plain, crow;
};
constexpr int kAbsorbDims = 128, kAbsorbSets = 2;        // dimensions in LDS at a time, sets of 16 tokens of a workgroup
template <typename T>
__global__ __launch_bounds__(kSeqThreads) void k_seq_latent_absorb(SeqLatentAbsorb a) {
    constexpr int U = Unit<T>::n, kCols = 64, kUnits = kCols / U, P = kCols + 2 * U, KS = 4 * U;      // units of a row in LDS, its elements, dimensions of a product
    constexpr int kLoads = kAbsorbDims * kUnits / kSeqThreads, kSteps = kAbsorbDims / KS;
    __shared__ __align__(16) T w[kAbsorbDims * P];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 15, g = lane >> 4;
    const int h = blockIdx.x / a.ncb, c0 = (blockIdx.x - h * a.ncb) * kCols, t0 = blockIdx.y * 16 * kAbsorbSets, columns = a.pitch / (int)sizeof(T);
    const char* from = a.w_uk + (size_t)h * a.D * a.pitch + (size_t)c0 * sizeof(T);
    const int units = min(kUnits, (columns - c0) / U);
    f32x4 acc[kAbsorbSets];
#pragma unroll
    for (int s = 0; s < kAbsorbSets; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int d0 = 0; d0 < a.D; d0 += kAbsorbDims) {
        // one round trip for everything; behind the last dimension there are zeros (of a query others would begin there)
        u32x4 b[kLoads], x[kAbsorbSets][kSteps];
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int r = (tid + i * kSeqThreads) / kUnits, u = (tid + i * kSeqThreads) % kUnits;
            b[i] = ld16(from + (size_t)min(d0 + r, a.D - 1) * a.pitch + min(u, units - 1) * 16);
            if (d0 + r >= a.D || u >= units) b[i] = u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int s = 0; s < kAbsorbSets; ++s) {
            const char* q = a.q + ((size_t)min(t0 + s * 16 + col, a.n - 1) * a.H + h) * a.qrow;
#pragma unroll
            for (int k = 0; k < kSteps; ++k) {
                const int at = (d0 + k * KS + g * U) * (int)sizeof(T);
                x[s][k] = ld16(q + min(at, a.plain - 16));
                if (at >= a.plain) x[s][k] = u32x4{0, 0, 0, 0};
            }
        }
        if (d0 > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int r = (tid + i * kSeqThreads) / kUnits, u = (tid + i * kSeqThreads) % kUnits;
            *reinterpret_cast<u32x4*>(w + r * P + u * U) = b[i];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kSteps; ++k) {
            T f[U];
#pragma unroll
            for (int e = 0; e < U; ++e) f[e] = w[(k * KS + g * U + e) * P + wave * 16 + col];
            u32x4 fw;
            __builtin_memcpy(&fw, f, 16);
#pragma unroll
            for (int s = 0; s < kAbsorbSets; ++s) acc[s] = mma16<T>(fw, x[s][k], acc[s]);
        }
    }
    const int c = c0 + wave * 16 + g * 4;
#pragma unroll
    for (int s = 0; s < kAbsorbSets; ++s) {
        const int t = t0 + s * 16 + col;
        if (t < a.n && c < columns) store4<T>(a.out + ((size_t)t * a.H + h) * a.crow + (size_t)c * sizeof(T), acc[s]);
    }
    if (c0 != 0) return;
    const int tail = (a.crow - a.pitch) / (int)sizeof(T), tokens = min(16 * kAbsorbSets, a.n - t0);  // rotated values, zeros behind them
    for (int i = tid; i < tokens * tail; i += kSeqThreads) {
        const int t = i / tail, j = i - t * tail;
        const size_t row = (size_t)(t0 + t) * a.H + h;
        reinterpret_cast<T*>(a.out + row * a.crow + a.pitch)[j] = j < a.R ? reinterpret_cast<const T*>(a.q + row * a.qrow + a.plain)[j] : from_f32<T>(0.0f);
    }
}

// What weights and denominators are multiplied by, so that sums of a million latents stay within the range of the latents themselves: values made of latents
// of any size may be small, and have sums that are in range.  A power of two, so outputs are the same bits without it wherever sums are in range.
constexpr float kBlockWeight = 1.0f / (1 << 20);

// Workgroup (split, block of 16 S columns).  As k_seq_latent_attn, but every wave takes its part of S sets of columns at a time, so that a tile is read from
// LDS once for all of them: a tile is a chain of barrier, reads, products, exchange of scores and softmax, which takes 1.4 us for one set,
// 1.65 for two and 2.3 for four.  What bounds it is that chain.  128 heads, 40 tokens at 3000, 5120 columns: a workgroup of four waves per token and 32
// heads 141 us; blocks of four sets whose softmax every wave does for itself 139, each set's softmax in one wave, the weights through LDS, 107; eight waves, two
// on a SIMD, the score's products of different sets in turn and copies that the compiler does not wait for 79 (390 TFLOP/s with the weights' two parts).
// Two buffers: the next tile's copies have the whole of this one's time.
struct SeqLatentBlock {
    const char* q;           // T [columns][crow bytes]
    const char* kc;          // cache row of position 0
    float *acc, *ml;         // [ns][columns][rp], [ns][columns][2]: sums and denominators times kBlockWeight
    float scale_log2;
    int n, H, pos0, crow, ns, rp;
};
// Waves: KP of them share a score's dimensions, KG have keys of their own; each has NW latent columns of the sums.
template <typename T, int NR> struct BlockWaves {
    static constexpr int waves = NR >= 512 ? 8 : 4, kf = LatentTile<T>::keys / 16, groups = waves == 8 ? kf : 1, kp = waves / groups, keys = kf / groups;
    static constexpr int columns = NR / waves, steps = LatentLds<T, NR>::ksteps / kp;
    static_assert(LatentLds<T, NR>::ksteps % kp == 0 && columns % 32 == 0, "");
};
template <typename T, int NR, int S>
__global__ __launch_bounds__((kWave * BlockWaves<T, NR>::waves)) void k_seq_latent_block(SeqLatentBlock a) {
    using L = LatentLds<T, NR>;
    using B = BlockWaves<T, NR>;
    constexpr int KT = LatentTile<T>::keys, KF = B::kf, W = B::waves, KP = B::kp, KS = B::steps, KW = B::keys, NW = B::columns;
    constexpr int kWeights = sizeof(T) == 2 ? 2 : 1;     // 16-byte units of a lane's weights
    static_assert(S <= W, "");
    extern __shared__ __align__(1024) char tiles[];
    __shared__ f32x4 parts[S * KP * KF * kWave];         // scores of one part of the dimensions
    __shared__ u32x4 weights[S * kWeights * kWave];
    __shared__ float moved[S * 16];                      // what a column's sums are multiplied by
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 15, g = lane >> 4;
    const int kp = wave % KP, key0 = wave / KP * KW;     // the wave's dimensions, and its first set of 16 keys
    const int ncols = a.n * a.H, c0 = (int)blockIdx.y * 16 * S, sp = blockIdx.x;
    const int end = a.pos0 + min(c0 + 16 * S - 1, ncols - 1) / a.H + 1, ntiles = (end + KT - 1) / KT;      // keys that the block's last token sees
    const int k0 = mul_div(ntiles, sp, a.ns) * KT, k1 = min(mul_div(ntiles, sp + 1, a.ns) * KT, end);
    const int ksteps = a.crow / 64, units = a.crow / 16;
    auto stage = [&](uint32_t tile, int kb) __attribute__((always_inline)) {  // 64 units of the tile per copy, the waves in turn
        constexpr int kCopies = L::copies * kSeqWaves;
#pragma unroll
        for (int i = 0; i < (kCopies + W - 1) / W; ++i) {
            const int c = i * W + wave, l = c * 64 + lane, r = l / L::up, u = l - r * L::up;
            if (c < kCopies) copy_to_lds16_from(a.kc + (size_t)min(kb + r, k1 - 1) * a.crow + min(u, units - 1) * 16, tile + c * 1024);
        }
    };
    const uint32_t l0 = lds_address(tiles);
    if (k0 < k1) stage(l0, k0);
    u32x4 qf[S][KS];
    f32x4 acc[S][NW / 16];
    // wave s has the maxima and denominators of set s
    float m = kNegBig, l = 0.0f;
    const int seen = min(k1, a.pos0 + min(c0 + min(wave, S - 1) * 16 + col, ncols - 1) / a.H + 1);    // end of the keys that the column sees
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int c = min(c0 + s * 16 + col, ncols - 1);
        const char* qr = a.q + (size_t)c * a.crow + g * 16;
#pragma unroll
        for (int d = 0; d < KS; ++d) {
            qf[s][d] = ld16(qr + min(kp * KS + d, ksteps - 1) * 64);
            if (kp * KS + d >= ksteps) qf[s][d] = u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < NW / 16; ++i) acc[s][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    int buf = 0;
    for (int kb = k0; kb < k1; kb += KT, buf ^= 1) {
        // the tile is there, and nobody reads the other buffer any more
        wait_vm<0>();
        lds_barrier();
        const char* const tile = tiles + buf * L::tile;
        if (kb + KT < k1) stage(l0 + (buf ^ 1) * L::tile, kb + KT);
        u32x4 kf[KS][KW];
#pragma unroll
        for (int d = 0; d < KS; ++d)
#pragma unroll
            for (int kt = 0; kt < KW; ++kt)
                kf[d][kt] = *reinterpret_cast<const u32x4*>(tile + (((key0 + kt) * 16 + col) * L::up + (kp * KS + d) * 4 + g) * 16);
        __builtin_amdgcn_sched_barrier(0);               // (all reads are requested before the first product waits for one)
        f32x4 w[S][KW];
#pragma unroll
        for (int d = 0; d < KS; ++d)
#pragma unroll
            for (int kt = 0; kt < KW; ++kt)
#pragma unroll
                for (int s = 0; s < S; ++s) w[s][kt] = mma16<T>(kf[d][kt], qf[s][d], d == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : w[s][kt]);
        __builtin_amdgcn_sched_barrier(0);               // (chains side by side, not one behind the other)
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int kt = 0; kt < KW; ++kt) parts[((s * KP + kp) * KF + key0 + kt) * kWave + lane] = w[s][kt];
        lds_barrier();
        if (wave < S) {
            f32x4 x[KF], p[KF][KP];
            float top = kNegBig, sum = 0.0f;
#pragma unroll
            for (int kt = 0; kt < KF; ++kt)
#pragma unroll
                for (int v = 0; v < KP; ++v) p[kt][v] = parts[((wave * KP + v) * KF + kt) * kWave + lane];
#pragma unroll
            for (int kt = 0; kt < KF; ++kt) {
                x[kt] = p[kt][0];
#pragma unroll
                for (int v = 1; v < KP; ++v) x[kt] += p[kt][v];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x[kt][r] = kb + kt * 16 + g * 4 + r < seen ? x[kt][r] * a.scale_log2 : kMasked;
                    top = fmaxf(top, x[kt][r]);
                }
            }
            top = fmaxf(m, rows_max<16>(top));
            const float c = fast_exp2(m - top);
            m = top;
#pragma unroll
            for (int kt = 0; kt < KF; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x[kt][r] = fast_exp2(x[kt][r] - m) * kBlockWeight;
                    sum += x[kt][r];
                }
            l = l * c + rows_sum<16>(sum);
            if (g == 0) moved[wave * 16 + col] = c;
            u32x4* const to = weights + wave * kWeights * kWave + lane;
            if constexpr (sizeof(T) == 2) {
                u32x4 hi, lo;
                split_weights(x[0], x[1], hi, lo);
                to[0] = hi;
                to[kWave] = lo;
            } else {
                to[0] = __builtin_bit_cast(u32x4, x[0]);
            }
        }
        lds_barrier();
        u32x4 hi[S], lo[S];
        float c[S];
        bool any = false;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            c[s] = moved[s * 16 + col];
            hi[s] = weights[s * kWeights * kWave + lane];
            if constexpr (kWeights == 2) lo[s] = weights[(s * kWeights + 1) * kWave + lane];
        }
#pragma unroll
        for (int s = 0; s < S; ++s) any = any || c[s] != 1.0f;
        if (__builtin_amdgcn_ballot_w64(any) != 0) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < NW / 16; ++i) acc[s][i] *= c[s];
        }
        if constexpr (sizeof(T) == 2) {
            constexpr int R = NW / 16 >= 8 ? 8 : 2;      // sets of 16 columns read together
            const uint32_t v = (uint32_t)(uintptr_t)(tile + (4 * g + (col >> 2)) * L::up * 16 + wave * NW * 2 + (col & 3) * 8);
#pragma unroll
            for (int i = 0; i < NW / 16; i += R) {
                TrCols f[R];
                if constexpr (R == 8) tr_read8(f, v + i * 32, v + i * 32 + 16 * L::up * 16);
                else tr_read2(f, v + i * 32, v + i * 32 + 16 * L::up * 16);
#pragma unroll
                for (int part = 0; part < 2; ++part)
#pragma unroll
                    for (int j = 0; j < R; ++j)
#pragma unroll
                        for (int s = 0; s < S; ++s)
                            acc[s][i + j] = mma16<T>(u32x4{f[j].x.x, f[j].x.y, f[j].y.x, f[j].y.y}, part == 0 ? hi[s] : lo[s], acc[s][i + j]);
            }
        } else {
            const char* v = tile + 4 * g * L::up * 16 + (wave * NW + col) * 4;
#pragma unroll
            for (int i = 0; i < NW / 16; ++i) {
                f32x4 f;
#pragma unroll
                for (int j = 0; j < 4; ++j) f[j] = *reinterpret_cast<const float*>(v + j * L::up * 16 + i * 64);
#pragma unroll
                for (int s = 0; s < S; ++s) acc[s][i] = mma16<T>(__builtin_bit_cast(u32x4, f), hi[s], acc[s][i]);
            }
        }
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int c = c0 + s * 16 + col;
        if (c >= ncols) continue;
        const size_t row = (size_t)sp * ncols + c;
        if (wave == s && g == 0) *reinterpret_cast<float2*>(a.ml + row * 2) = make_float2(m, l);
#pragma unroll
        for (int i = 0; i < NW / 16; ++i)
            if (wave * NW + i * 16 < a.rp) *reinterpret_cast<f32x4*>(a.acc + row * a.rp + wave * NW + i * 16 + g * 4) = acc[s][i];
    }
}

// Workgroup (head, up to 16 tokens, kTurnRows of the head's outputs, 16 of a wave): merges the splits of these columns, then its rows of W_uv, and the output gate.  The
// latents lie in LDS as fp32 or as two bf16 parts, which keep 16 of their bits (they are finite unless a cached latent is not, and then its scores are
// no numbers either).  Bound by round trips and, with many columns, by the partial results, which
// the workgroups of a head read once each (half of V): 16 heads, 8 tokens in 64 splits 9 us, 128 heads, 40 tokens in 3 splits 23 us.  A workgroup for
// each token and 16 outputs, as for one token, took 22 and, with 128 heads, 149 us for 40 tokens.
static_assert(kTurnSplits <= kWave && kTurnRows == 16 * kSeqWaves, "a lane has a split, a wave 16 rows");
struct SeqLatentTurnOut {
    const float *acc, *ml;
    const float* sink;       // nullable
    const float* gate;       // nullable: [tokens][ldg] before the sigmoid
    const char* w_uv;        // T [H * V][pitch bytes]
    char* out;               // T [tokens][ldo bytes]
    int n, tokens, H, V, pitch, ns, rp, ldg, ldo;            // tokens: of a workgroup
};
template <typename T>
__global__ __launch_bounds__(kSeqThreads) void k_seq_latent_turn_out(SeqLatentTurnOut a) {
    constexpr int U = Unit<T>::n, kParts = sizeof(T) == 2 ? 2 : 1, kM = 16, kW = 16;
    __shared__ float f[16][kTurnSplits];
    extern __shared__ __align__(16) char lat[];          // [kParts][16][pitch + 16 bytes]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 15, g = lane >> 4, h = blockIdx.x;
    const int t0 = blockIdx.y * a.tokens, nt = min(a.tokens, a.n - t0), lrow = a.pitch + 16, ncols = a.n * a.H;
    const float snk = a.sink != nullptr ? a.sink[h] * kLog2e : kNegBig;
    // the wave's first rows of W_uv are on their way beside the merge
    const int steps = a.pitch / 64, v0 = (int)blockIdx.z * kTurnRows + wave * 16;
    u32x4 fw[kW];
    const char* const w = a.w_uv + ((size_t)h * a.V + min(v0 + col, a.V - 1)) * a.pitch + g * 16;
    auto request = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kW; ++i) fw[i] = ld16(w + min(k + i, steps - 1) * 64);
    };
    const int r4 = a.rp / 4, c4 = a.pitch / (int)sizeof(T) / 4;      // groups of four latents, of four columns of a row of W_uv
    f32x4 y[kM];
    auto ask = [&](int i, int s0) __attribute__((always_inline)) {
        const int t = i / c4, x = i - t * c4;
        const float* p = a.acc + ((size_t)(t0 + min(t, nt - 1)) * a.H + h) * a.rp + min(x, r4 - 1) * 4;
#pragma unroll
        for (int j = 0; j < kM; ++j) {
            if (j % 4 == 0 && s0 + j >= a.ns) break;     // (the same for the workgroup)
            y[j] = *reinterpret_cast<const f32x4*>(p + (size_t)min(s0 + j, a.ns - 1) * ncols * a.rp);
        }
    };
    // (a lane has a split)
    constexpr int kT = 16 / kSeqWaves;
    float2 ml[kT];
#pragma unroll
    for (int j = 0; j < kT; ++j)
        ml[j] = *reinterpret_cast<const float2*>(a.ml + ((size_t)min(lane, a.ns - 1) * ncols + (size_t)(t0 + min(wave + j * kSeqWaves, nt - 1)) * a.H + h) * 2);
    ask(tid, 0);
    request(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kT; ++j) {
        const int t = wave + j * kSeqWaves;
        if (t >= nt) break;
        const float2 z = lane < a.ns ? ml[j] : make_float2(kNegBig, 0.0f);
        const float m = wave_max(fmaxf(z.x, snk)), e = fast_exp2(z.x - m);
        const float l = wave_sum(z.y * e) + (a.sink != nullptr ? fast_exp2(snk - m) * kBlockWeight : 0.0f);
        f[t][lane] = e / l;
    }
    __syncthreads();
    for (int i = tid; i < nt * c4; i += kSeqThreads) {
        const int t = i / c4, x = i - t * c4;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        if (i != tid) ask(i, 0);
        for (int s0 = 0;;) {
#pragma unroll
            for (int j = 0; j < kM; ++j) {
                if (j % 4 == 0 && s0 + j >= a.ns) break;
                const bool live = s0 + j < a.ns && x < r4;           // (a split's values may be infinite: not times zero)
                const float w = f[t][min(s0 + j, a.ns - 1)];
#pragma unroll
                for (int c = 0; c < 4; ++c) s[c] = live ? fmadd(y[j][c], w, s[c]) : s[c];
            }
            s0 += kM;
            if (s0 >= a.ns) break;
            ask(i, s0);
        }
        char* to = lat + t * lrow + x * 4 * (int)sizeof(T);
        if constexpr (kParts == 2) {
            const u32x2 hi = {pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3])};
            *reinterpret_cast<u32x2*>(to) = hi;
            *reinterpret_cast<u32x2*>(to + 16 * lrow) = u32x2{pack_bf16(s[0] - __uint_as_float(hi.x << 16), s[1] - __uint_as_float(hi.x & 0xffff0000u)),
                                                             pack_bf16(s[2] - __uint_as_float(hi.y << 16), s[3] - __uint_as_float(hi.y & 0xffff0000u))};
        } else {
            *reinterpret_cast<f32x4*>(to) = s;
        }
    }
    __syncthreads();
    if (v0 >= a.V) return;
    const char* x = lat + min(col, nt - 1) * lrow + g * 16;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0;;) {
#pragma unroll
        for (int i = 0; i < kW; ++i) {
            if (k + i >= steps) break;
#pragma unroll
            for (int j = 0; j < kParts; ++j) acc = mma16<T>(fw[i], *reinterpret_cast<const u32x4*>(x + j * 16 * lrow + (k + i) * 64), acc);
        }
        k += kW;
        if (k >= steps) break;
        request(k);                                      // (at the end, not the beginning: from there the compiler takes each load to its product, 10.7 -> 12.6 us)
    }
    if (col >= nt) return;
    T* o = reinterpret_cast<T*>(a.out + (size_t)(t0 + col) * a.ldo) + (size_t)h * a.V;
    const float* gate = a.gate + (size_t)(t0 + col) * a.ldg + (size_t)h * a.V;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int v = v0 + g * 4 + r;
        if (v < a.V) o[v] = from_f32<T>(a.gate != nullptr ? acc[r] * sigmoid(gate[v]) : acc[r]);
    }
}

// ---- residual streams --------------------------------------------------------------------------
// One workgroup per token: the streams after a sublayer (or at the start: all equal to the embedding, or at the end: as they
// are), and the next sublayer's input norm(sum_t in[t] x_t).
struct SeqStreams {
    float* x;                // [tokens][streams][width]
    const float* y;          // the sublayer's output, nullable: the sum of `parts` rows, part_stride floats apart
    int parts;
    size_t part_stride;
    const float* ys;         // nullable: [tokens][top][width], outputs of the chosen experts
    int top;
    float slot_weight;
    const float *mix, *out;  // null: the streams stay as they are
    const float* in;         // null: all one
    const float* w;          // norm weight; null: no next input
    float noff, eps;
    int streams, width;
    char* xb;
    int pitch;
    float* copy;             // nullable: receives the sum of the streams
    const int* rows;         // nullable: take token rows[t], write input t
    int way;                 // k_seq_streams4: one of kStreams..
    const float *y0, *mix0, *out0;       // ... kStreamsAgain: the update that was not stored
    // the start
    const int* tokens;       // null: not the start
    const int* state;        // not null: one token, its position from here instead of pos0 + t
    const char *embed, *pos;
    int embed_pitch, pos0;
};
template <typename T, int S>
__global__ __launch_bounds__(kSeqThreads) void k_seq_streams(SeqStreams a) {
    __shared__ float red[kSeqWaves];
    extern __shared__ __align__(16) float us[];
    const int t = a.rows != nullptr ? a.rows[blockIdx.x] : (int)blockIdx.x;
    float* x = a.x + (size_t)t * a.streams * a.width;
    float mix[S][S], out[S], in[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const bool live = s < a.streams;
        in[s] = !live ? 0.0f : a.in != nullptr ? a.in[s] : 1.0f;
        out[s] = live && a.mix != nullptr ? a.out[s] : 0.0f;
#pragma unroll
        for (int j = 0; j < S; ++j) mix[s][j] = live && j < a.streams && a.mix != nullptr ? a.mix[s * a.streams + j] : 0.0f;
    }
    const T *e = nullptr, *ep = nullptr;
    if (a.tokens != nullptr) {
        e = reinterpret_cast<const T*>(a.embed + (size_t)a.tokens[t] * a.embed_pitch);
        if (a.pos != nullptr) ep = reinterpret_cast<const T*>(a.pos + (size_t)(a.state != nullptr ? a.state[1] : a.pos0 + t) * a.embed_pitch);
    }
    float ss = 0.0f;
    // N elements at a time (4 where the rows allow it); every thread reads back only what it has written
    auto sum = [&](auto n, int i) {
        constexpr int N = decltype(n)::value;
        float v[S][N];
        if (e != nullptr) {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const float z = to_f32(e[i + j]) + (ep != nullptr ? to_f32(ep[i + j]) : 0.0f);
#pragma unroll
                for (int s = 0; s < S; ++s) v[s][j] = z;
            }
        } else {
            float o[S][N], y[N];
#pragma unroll
            for (int s = 0; s < S; ++s) {
#pragma unroll
                for (int j = 0; j < N; ++j) o[s][j] = 0.0f;
                if (s < a.streams) add_n<N>(o[s], x + (size_t)s * a.width + i);
            }
#pragma unroll
            for (int j = 0; j < N; ++j) y[j] = 0.0f;
            if (a.ys != nullptr) {
                const float* ys = a.ys + (size_t)t * a.top * a.width + i;
                for (int k = 0; k < a.top; ++k) add_n<N>(y, ys + (size_t)k * a.width);
#pragma unroll
                for (int j = 0; j < N; ++j) y[j] *= a.slot_weight;
            }
            if (a.y != nullptr)
                for (int k = 0; k < a.parts; ++k) add_n<N>(y, a.y + k * a.part_stride + (size_t)t * a.width + i);
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    if (a.mix == nullptr) {
                        v[s][j] = o[s][j];
                    } else {
                        v[s][j] = out[s] * y[j];
#pragma unroll
                        for (int k = 0; k < S; ++k) v[s][j] = fmadd(mix[k][s], o[k][j], v[s][j]);
                    }
                }
        }
        if (a.rows == nullptr) {
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (s < a.streams) put_n<float, N>(x + (size_t)s * a.width + i, v[s]);
        }
        float u[N], all[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            u[j] = all[j] = 0.0f;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                u[j] = fmadd(in[s], v[s][j], u[j]);
                all[j] += s < a.streams ? v[s][j] : 0.0f;
            }
            us[i + j] = u[j];
            ss = fmadd(u[j], u[j], ss);
        }
        if (a.copy != nullptr) put_n<float, N>(a.copy + (size_t)t * a.width + i, all);
    };
    const int w4 = (a.width & 3) ? 0 : a.width;
    for (int i = threadIdx.x * 4; i < w4; i += kSeqThreads * 4) sum(std::integral_constant<int, 4>{}, i);
    for (int i = w4 + threadIdx.x; i < a.width; i += kSeqThreads) sum(std::integral_constant<int, 1>{}, i);
    if (a.w == nullptr) return;
    const float inv = inv_rms(block_sum(ss, red), a.width, a.eps);
    T* xb = reinterpret_cast<T*>(a.xb + (size_t)blockIdx.x * a.pitch);
    auto put = [&](auto n, int i) {
        constexpr int N = decltype(n)::value;
        float w[N], v[N];
#pragma unroll
        for (int j = 0; j < N; ++j) w[j] = a.noff;
        add_n<N>(w, a.w + i);
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = us[i + j] * inv * w[j];
        put_n<T, N>(xb + i, v);
    };
    for (int i = threadIdx.x * 4; i < w4; i += kSeqThreads * 4) put(std::integral_constant<int, 4>{}, i);
    for (int i = w4 + threadIdx.x; i < a.width; i += kSeqThreads) put(std::integral_constant<int, 1>{}, i);
}

// The same for rows of whole groups of four elements, up to 1024 U of them: the streams stay in registers, and everything is requested
// before anything is used.  That is for portions of few tokens, where a row is a chain of round trips; with many, both kernels are bound
// by their bytes.  Four streams of 4096 values, 37 tokens: 12.7 -> 9.8 us, 150: 15.4 -> 12.0, 512: 25.8 -> 20.4, 1000: 34.7 and 34.8, 8000:
// 220 and 213; two of 2048, 37 tokens: 7.9 -> 5.8 us, 512: 8.3 and 8.2, 8000: 57 and 59.
//
// Portions of many tokens are bound by their bytes, most of which are the streams (M: what the kernel does with them, kStreamsStay and kStreamsAgain where
// streams_later says so).  The update after a mixer is not stored: only the next input is needed of it.  The update after the feed-forward makes it again,
// from the same values in the same order, and reads one row more for that, where a row for each stream is not written.  The streams go past the caches,
// which leaves those to the sublayers' outputs.  Four streams of 4096 values, 8000 tokens: 220 + 220 us -> 140 + 269 (5.1 TB/s); without the latter 160 + 276.
enum : int { kStreamsKept = 0, kStreamsStay = 1, kStreamsAgain = 2 };
template <typename T, int S, int U, int M>
__global__ __launch_bounds__(kSeqThreads) void k_seq_streams4(SeqStreams a) {
    __shared__ float red[kSeqWaves];
    const int t = a.rows != nullptr ? a.rows[blockIdx.x] : (int)blockIdx.x, tid = threadIdx.x, n4 = a.width / 4;
    float* x = a.x + (size_t)t * a.streams * a.width;
    f32x4 o[S][U], w[U], y[U], z[M == kStreamsAgain ? U : 1];
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const int i = min(tid + j * kSeqThreads, n4 - 1);
        if (a.tokens == nullptr) {
#pragma unroll
            for (int s = 0; s < S; ++s) o[s][j] = load_row4<M != kStreamsKept>(x + (size_t)min(s, a.streams - 1) * a.width, i);
        } else {
            const T* e = reinterpret_cast<const T*>(a.embed + (size_t)a.tokens[t] * a.embed_pitch) + i * 4;
            const T* p = a.pos != nullptr ? reinterpret_cast<const T*>(a.pos + (size_t)(a.state != nullptr ? a.state[1] : a.pos0 + t) * a.embed_pitch) + i * 4 : nullptr;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[0][j][r] = to_f32(e[r]) + (p != nullptr ? to_f32(p[r]) : 0.0f);
#pragma unroll
            for (int s = 1; s < S; ++s) o[s][j] = o[0][j];
        }
        w[j] = a.w != nullptr ? reinterpret_cast<const f32x4*>(a.w)[i] : f32x4{0.f, 0.f, 0.f, 0.f};
        y[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (M == kStreamsAgain) z[j] = load_row4<true>(a.y0 + (size_t)t * a.width, i);
    }
    if (a.ys != nullptr) {
        add_rows4<U, 2>(y, a.ys + (size_t)t * a.top * a.width, a.top, a.width, n4);
#pragma unroll
        for (int j = 0; j < U; ++j) y[j] *= a.slot_weight;
    }
    if (a.y != nullptr) add_rows4<U, (U <= 2 ? 4 : 2)>(y, a.y + (size_t)t * a.width, a.parts, a.part_stride, n4);
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const int i = tid + j * kSeqThreads;
        auto update = [&](const float* mix, const float* out, f32x4 y) __attribute__((always_inline)) {
            f32x4 v[S];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const bool live = s < a.streams;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[s][r] = (live ? out[s] : 0.0f) * y[r];
#pragma unroll
                for (int k = 0; k < S; ++k) {
                    const float m = live && k < a.streams ? mix[k * a.streams + s] : 0.0f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[s][r] = fmadd(m, o[k][j][r], v[s][r]);
                }
            }
#pragma unroll
            for (int s = 0; s < S; ++s) o[s][j] = v[s];
        };
        if constexpr (M == kStreamsAgain) update(a.mix0, a.out0, z[j]);
        if (a.tokens == nullptr && a.mix != nullptr) update(a.mix, a.out, y[j]);
        f32x4 u = {0.f, 0.f, 0.f, 0.f}, all = u;
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (s < a.streams) {
                const float in = a.in != nullptr ? a.in[s] : 1.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) u[r] = fmadd(in, o[s][j][r], u[r]);
                all += o[s][j];
            }
        if (i < n4) {
            if (a.rows == nullptr && M != kStreamsStay) {
#pragma unroll
                for (int s = 0; s < S; ++s)
                    if (s < a.streams) {
                        if constexpr (M == kStreamsAgain) __builtin_nontemporal_store(o[s][j], reinterpret_cast<f32x4*>(x + (size_t)s * a.width) + i);
                        else reinterpret_cast<f32x4*>(x + (size_t)s * a.width)[i] = o[s][j];
                    }
            }
            if (a.copy != nullptr) reinterpret_cast<f32x4*>(a.copy + (size_t)t * a.width)[i] = all;
#pragma unroll
            for (int r = 0; r < 4; ++r) ss = fmadd(u[r], u[r], ss);
        }
        y[j] = u;
    }
    if (a.w == nullptr) return;
    const float inv = inv_rms(block_sum(ss, red), a.width, a.eps);
    T* xb = reinterpret_cast<T*>(a.xb + (size_t)blockIdx.x * a.pitch);
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const int i = tid + j * kSeqThreads;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[j][r] = y[j][r] * inv * (a.noff + w[j][r]);
        if (i < n4) store4<T>(xb + i * 4, y[j]);
    }
}

}  // namespace cfpp
