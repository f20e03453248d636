// Matrix products of a portion of the sequence models: out[token][row] = W[row] . a[token] (device code; included by
// seq_kernels.hip).
//
// Tiles of both operands go to LDS in steps of 128 bytes of k, copied there by the memory system itself (global_load_lds), and
// the copies of later steps stay in flight across the barriers: every wave waits for its own copies of the step that is due, by
// number, and the barrier behind that wait makes the whole step's tile visible.  Two kernels:
//   k_seq_gemm   any tile, a ring of NB buffers, one barrier per step.  Narrow tiles of tokens for portions of a few tokens, where
//                the product is a stream of weights and what counts is the number of bytes in flight;
//   k_seq_gemm8  256 x 256 tiles, bf16, for products that are bound by the matrix cores.
// Both can split k over workgroups (kEpiF32): each split writes its own partial result, the kernel that reads the product adds
// them up in order.
#pragma once
#include "seq_device.hpp"

namespace cfpp {

// kEpiHeads: rows of keys of all heads, then rows of values of all heads, each head's rows [position] in a buffer of its own.
// kEpiStreams (one token): the output row goes into the residual streams.
enum : int { kEpiF32 = 0, kEpiRelu2 = 1, kEpiGated = 2, kEpiHead = 3, kEpiHeads = 4, kEpiStreams = 5 };
struct SeqGemm {
    const char* w;           // [n rows][kbytes]
    const char* a;           // [tokens][lda bytes]
    int n, m, kbytes, lda;
    const float* bias;       // nullable (kEpiF32, kEpiGated)
    float* yf;               // kEpiF32 / kEpiHead: [tokens][ldy]
    int ldy;
    char* yt;                // kEpiRelu2 / kEpiGated: T, [tokens][ldyt bytes]; kEpiHeads: keys
    int ldyt;
    float mul, cap;          // kEpiHead
    char* yv;                // kEpiHeads: values; key rows of kd elements, kp bytes apart, heads kh bytes apart; values alike
    int nk, kd, kp, vd, vp;  // ... nk: rows of keys
    size_t kh, vh;
    // tiles of tokens sorted by expert (tile_off null: a plain product); their inputs lie in less than 4 GiB
    const int* tile_off;     // [experts + 1] prefix sums of tiles
    const int* row_off;      // [experts + 1] prefix sums of sorted slots
    const int* slots;        // sorted slots: token * top + j
    int experts, slot_div;   // input row of slot s: s / slot_div
    size_t w_stride;
    // (k_seq_gemm) The weights are read by one tile of tokens only, as a stream past the caches, in which the inputs stay: 37 tokens x 14336 x 4096
    // 27.1 -> 24.8 us, 64 experts of 2816 x 2048 with 66 tokens each 171 -> 159 us; with two token tiles it costs (36 -> 42 us).  Weights that
    // stay in the 256 MB cache from call to call would come faster from there: a product of 4096 x 4096 for 37 tokens, called over 200 MB of
    // such matrices, 7.9 -> 8.5 us, over 300 MB and more 8.9 -> 8.6.  In models this small the streams are too short to tell (199 MB of
    // weights, 37 tokens: 198 to 203 us with, 198 to 201 without; 502 MB: 610 to 633 and 646 to 658), so the model's size is not asked.
    int once;
    int splits;              // of k (kEpiF32); the s-th partial result lies s * split_stride floats behind yf
    size_t split_stride;
};

// rows of 128 bytes: units of row r are stored at unit ^ swz(r), which spreads 16 consecutive rows over all banks
__device__ __forceinline__ int swz128(int row) { return (row >> 1) & 7; }

// Which tile a workgroup works on.
struct GemmTile {
    const char* w;           // the matrix (of the expert)
    int tw, tt;              // tile of rows, tile of tokens
    int row0, m;             // experts: first sorted slot of the tile; tokens (experts: slots of the tile)
    int split;
};
template <int BW, int BT>
__device__ __forceinline__ bool gemm_tile(const SeqGemm& p, GemmTile& t) {
    // every XCD works on a contiguous range of tiles; inside it tiles go through groups of up to 8 token tiles, and the splits
    // of k come one after the other, so that the workgroups that run together share their inputs' part.  (Of expert tiles only
    // an upper bound is launched: the ranges divide those that there are.)
    const int tiles_w = (p.n + BW - 1) / BW, xcd = blockIdx.x % 8, i = blockIdx.x / 8;
    const int total = p.tile_off != nullptr ? p.tile_off[p.experts] * tiles_w : (int)gridDim.x, per = total / 8, rem = total % 8;
    if (i >= per + (xcd < rem ? 1 : 0)) return false;
    int id = xcd * per + min(xcd, rem) + i;
    t.w = p.w;
    t.row0 = t.split = 0;
    t.m = p.m;
    if (p.tile_off != nullptr) {
        t.tt = id / tiles_w;
        t.tw = id - t.tt * tiles_w;
        int lo = 0, hi = p.experts;                      // last expert whose first tile is <= tt
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (p.tile_off[mid] <= t.tt) lo = mid; else hi = mid;
        }
        // (experts without tokens have no tiles: skip to the one that owns the tile)
        while (p.tile_off[lo + 1] <= t.tt) ++lo;
        t.w += (size_t)lo * p.w_stride;
        t.row0 = p.row_off[lo] + (t.tt - p.tile_off[lo]) * BT;
        t.m = p.row_off[lo + 1] - t.row0;
        t.tt = 0;
    } else {
        const int tiles_t = (p.m + BT - 1) / BT, tiles = tiles_w * tiles_t;
        t.split = id / tiles;
        id -= t.split * tiles;
        const int group = 8 * tiles_w, gi = id / group, first = gi * 8;
        const int gs = min(8, tiles_t - first), r = id - gi * group;
        t.tt = first + r % gs;
        t.tw = r / gs;
    }
    return true;
}
// byte offset of token `tok` of the tile from its input base (the tile's first row; experts: the whole input)
template <int BT>
__device__ __forceinline__ uint32_t gemm_input_row(const SeqGemm& p, const GemmTile& t, int tok) {
    const int k = min(tok, t.m - 1 - t.tt * BT);
    return (uint32_t)(p.tile_off != nullptr ? p.slots[t.row0 + k] / p.slot_div : k) * (uint32_t)p.lda;
}

// The results of a wave: MI x NI tiles of 16 x 16, rows n0 + 16 i + 4 g + r of token c0 + 16 j + col.
template <typename T, int EPI, int MI, int NI>
__device__ __forceinline__ void gemm_store(const SeqGemm& p, const GemmTile& t, const f32x4 (&acc)[MI][NI], int nw0, int c0, int col, int g) {
    // kEpiHeads: where row n goes at position 0, and the bytes from one position to the next; `whole`: rows n0 .. n0 + 3 lie together
    auto head_row = [&](int n, int& rp) {
        const bool k = n < p.nk;
        const int d = k ? p.kd : p.vd, m = k ? n : n - p.nk, h = m / d;
        rp = k ? p.kp : p.vp;
        return (k ? p.yt + h * p.kh : p.yv + h * p.vh) + (m - h * d) * (int)sizeof(T);
    };
    // bf16 outputs leave in units of 16 bytes (gated, two tiles only: 8) where a wave has an even number of tiles of rows (64 x 16, 64 x 32, 96 x 128,
    // 96 x 160 and 192 x 160 have one or three, and store 4 or 8 bytes below): as a lane has them, 4 or 2 outputs of a token, a store of the wave takes 16
    // lines of memory for 512 or 256 bytes.  Lane group g of every two tiles' four (gated, four tiles: of all four) takes a row's next outputs from
    // the groups beside it.  256 x 256 tiles: keys and values from latents of 512 values, 3151 positions 24.6 -> 20.4 us, 8000 103 -> 82;
    // 16384 x 4096, 2048 tokens 238 -> 220; 22528 gated rows, 8000 tokens 1089 -> 1059.
    constexpr int kTiles = sizeof(T) != 2 || MI % 2 != 0 ? 1 : EPI == kEpiRelu2 || EPI == kEpiHeads ? 2 : EPI == kEpiGated ? (MI % 4 == 0 ? 4 : 2) : 1;
    if constexpr (kTiles > 1) {
        if (nw0 + MI * 16 <= p.n && (EPI != kEpiHeads || ((p.kd | p.vd) & 7) == 0)) {
            constexpr int N = MI / kTiles;
            const int at = kTiles == 4 ? g * 16 : (g & 1) * 16 + (g >> 1) * 8;         // the lane's first row among those of the tiles
            char* to[N];
            int step[N];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int n0 = nw0 + i * kTiles * 16 + at;
                if constexpr (EPI == kEpiHeads) {
                    to[i] = head_row(n0, step[i]);
                } else {
                    to[i] = p.yt + (size_t)(EPI == kEpiGated ? n0 / 2 : n0) * sizeof(T);
                    step[i] = p.ldyt;
                }
            }
            f32x4 b[MI];
#pragma unroll
            for (int i = 0; i < MI; ++i)
                b[i] = EPI == kEpiGated && p.bias != nullptr ? *reinterpret_cast<const f32x4*>(p.bias + nw0 + i * 16 + g * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
            auto swap16 = [](uint32_t& x, uint32_t& y) {
                const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
                x = r[0];
                y = r[1];
            };
            auto swap32 = [](uint32_t& x, uint32_t& y) {
                const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
                x = r[0];
                y = r[1];
            };
            auto gate = [&](int i, int j) {
                const f32x4 v = acc[i][j] + b[i];
                return pack_bf16(silu(v[0]) * v[1], silu(v[2]) * v[3]);
            };
            int rows[NI];
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int tl = min(c0 + j * 16 + col, t.m - 1);
                rows[j] = p.tile_off != nullptr ? p.slots[t.row0 + tl] : tl;
            }
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                if (c0 + j * 16 >= t.m) break;           // (the same for the wave: its lanes exchange)
                const bool live = c0 + j * 16 + col < t.m;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    char* const y = to[i] + (size_t)rows[j] * step[i];
                    if constexpr (EPI == kEpiGated) {
                        uint32_t d[kTiles];
#pragma unroll
                        for (int k = 0; k < kTiles; ++k) d[k] = gate(i * kTiles + k, j);
                        swap16(d[0], d[1]);
                        if constexpr (kTiles == 4) {
                            swap16(d[2], d[3]);
                            swap32(d[0], d[2]);
                            swap32(d[1], d[3]);
                            if (live) *reinterpret_cast<u32x4*>(y) = u32x4{d[0], d[1], d[2], d[3]};
                        } else {
                            if (live) *reinterpret_cast<u32x2*>(y) = u32x2{d[0], d[1]};
                        }
                    } else {
                        f32x4 u = acc[2 * i][j], v = acc[2 * i + 1][j];
                        if constexpr (EPI == kEpiRelu2) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                u[r] = relu2(u[r]);
                                v[r] = relu2(v[r]);
                            }
                        }
                        uint32_t u0 = pack_bf16(u[0], u[1]), u1 = pack_bf16(u[2], u[3]), v0 = pack_bf16(v[0], v[1]), v1 = pack_bf16(v[2], v[3]);
                        swap16(u0, v0);
                        swap16(u1, v1);
                        if (live) *reinterpret_cast<u32x4*>(y) = u32x4{u0, u1, v0, v1};
                    }
                }
            }
            return;
        }
    }
    char* dst[MI];
    int pitch[MI];
    bool whole[MI];
    if constexpr (EPI == kEpiHeads) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int n0 = min(nw0 + i * 16 + g * 4, p.n - 1);
            dst[i] = head_row(n0, pitch[i]);
            whole[i] = ((p.kd | p.vd) & 3) == 0 && n0 + 3 < p.n;       // (n0, the keys' rows and the heads' rows are multiples of four)
        }
    }
    float* const yf = p.yf + (EPI == kEpiF32 ? t.split * p.split_stride : 0);
    // Everything that is read is requested here: the biases of a lane's rows, the slots of its tokens.  (Where they are used, each is a round
    // trip: 21888 gated rows x 2048 with biases, 150 tokens: 6.8 us of 30 were fifteen of them; 256 x 256 tiles have 32.)
    int row[NI];
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        const int tl = c0 + j * 16 + col;
        row[j] = p.tile_off != nullptr ? p.slots[t.row0 + min(tl, t.m - 1)] : tl;
    }
    f32x4 bias[MI];
    if constexpr (EPI == kEpiF32 || EPI == kEpiGated) {
        const bool with_bias = p.bias != nullptr && t.split == 0;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int n0 = nw0 + i * 16 + g * 4;
            bias[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (!with_bias) continue;
            if (n0 + 3 < p.n) {
                bias[i] = *reinterpret_cast<const f32x4*>(p.bias + n0);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n0 + r < p.n) bias[i][r] = p.bias[n0 + r];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        if (c0 + j * 16 + col >= t.m) continue;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int n0 = nw0 + i * 16 + g * 4;
            const f32x4 v = acc[i][j];
            if constexpr (EPI == kEpiF32 || EPI == kEpiHead) {
                float* y = yf + (size_t)row[j] * p.ldy + n0;
                f32x4 o = v;
                if (EPI == kEpiF32) o += bias[i];
                if (EPI == kEpiHead) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] = soft_cap(o[r] * p.mul, p.cap);
                }
                if (n0 + 3 < p.n && (p.ldy & 3) == 0) {
                    *reinterpret_cast<f32x4*>(y) = o;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n0 + r < p.n) y[r] = o[r];
                }
            } else if constexpr (EPI == kEpiRelu2) {
                T* y = reinterpret_cast<T*>(p.yt + (size_t)row[j] * p.ldyt) + n0;
                if (n0 + 3 < p.n) {                      // (rows are padded to 128 bytes and n0 is a multiple of four)
                    store4<T>(y, f32x4{relu2(v[0]), relu2(v[1]), relu2(v[2]), relu2(v[3])});
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n0 + r < p.n) y[r] = from_f32<T>(relu2(v[r]));
                }
            } else if constexpr (EPI == kEpiHeads) {
                if (whole[i]) {
                    store4<T>(dst[i] + (size_t)row[j] * pitch[i], v);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n0 + r < p.n) {
                            int rp;
                            char* b = head_row(n0 + r, rp);
                            *reinterpret_cast<T*>(b + (size_t)row[j] * rp) = from_f32<T>(v[r]);
                        }
                }
            } else {
                T* y = reinterpret_cast<T*>(p.yt + (size_t)row[j] * p.ldyt) + n0 / 2;
                float o[2];
#pragma unroll
                for (int r = 0; r < 4; r += 2) o[r / 2] = silu(v[r] + bias[i][r]) * (v[r + 1] + bias[i][r + 1]);
                if (n0 + 3 < p.n) {
                    store2<T>(y, o[0], o[1]);
                } else if (n0 < p.n) {
                    y[0] = from_f32<T>(o[0]);
                }
            }
        }
    }
}

// BW rows x BT tokens, WR x WC waves, a ring of NB buffers (NB - 1 steps in flight).
template <typename T, int BW, int BT, int WR, int WC, int NB, int EPI>
__global__ __launch_bounds__(kWave* WR* WC) void k_seq_gemm(SeqGemm p) {
    constexpr int NW = WR * WC, MI = BW / WR / 16, NI = BT / WC / 16;
    constexpr int WI = BW / 8 / NW, AC = BT / 8, AI = (AC + NW - 1) / NW;      // 1 KB copies of a wave and step; copies of the input
    constexpr int kStep = (BW + BT) * kRowBytes;
    static_assert(BW % (8 * NW) == 0 && BW % (16 * WR) == 0 && BT % (16 * WC) == 0, "");
    extern __shared__ __align__(1024) char lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wr = wave / WC, wc = wave % WC;
    GemmTile t;
    if (!gemm_tile<BW, BT>(p, t)) return;
    const int nk = p.kbytes / kRowBytes, kb = mul_div(nk, t.split, p.splits), n = mul_div(nk, t.split + 1, p.splits) - kb;
    // Tiles of a weight stream begin at different steps and go round (steps of 5 apart: of n steps every one is a start, or n / 5 of them where n
    // is a multiple of 5).  Workgroups that run side by side would otherwise ask for the same 128 bytes of rows that are 4 KB apart, or a multiple of
    // it; the copies in flight cover (NB - 1) x 128 <= 640 bytes of a row.  That these lie in few of the memory's channels is supposed, from the
    // times alone: 64 experts of 2816 x 2048, 66 tokens each: 154 -> 140 us; 21888 gated rows x 2048, 150 tokens: 31.2 -> 28.1; 14336 x 4096, 37
    // tokens: 24.7 -> 24.2.  Not where several tiles of tokens share a weight's copy in the caches or the splits of k are apart by themselves (2 to 5 %
    // slower), nor for a head, whose eight rounds of workgroups drift apart (1 % slower), nor in fp32 (14336 x 4096, 2 tokens 46 and 43 us, but 17
    // tokens 56 and 58, 12 experts' 2816 x 2048 43 and 47).
    constexpr bool kTurns = sizeof(T) == 2 && EPI != kEpiHead;
    const int first = kTurns && p.once && p.splits == 1 ? t.tw * 5 % n : 0;
    const char* bw = uniform(t.w + (size_t)t.tw * BW * p.kbytes + (size_t)(kb + first) * kRowBytes);
    const char* ba = uniform(p.a + (p.tile_off != nullptr ? (size_t)0 : (size_t)t.tt * BT * p.lda) + (size_t)(kb + first) * kRowBytes);
    uint32_t vw[WI], va[AI];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int r = (wave + i * NW) * 8 + (lane >> 3);
        vw[i] = (uint32_t)min(r, p.n - 1 - t.tw * BW) * (uint32_t)p.kbytes + ((lane & 7) ^ swz128(r)) * 16;
    }
#pragma unroll
    for (int i = 0; i < AI; ++i) {                       // (where the waves' shares differ, the last copy is made twice)
        const int r = min(wave + i * NW, AC - 1) * 8 + (lane >> 3);
        va[i] = gemm_input_row<BT>(p, t, r) + ((lane & 7) ^ swz128(r)) * 16;
    }
    const uint32_t l0 = lds_address(lds);
    int fill = 0, issued = 0, use = 0;                   // buffer of the next copies, steps requested, buffer in use
    auto next = [&](int b) __attribute__((always_inline)) { return b + 1 == NB ? 0 : b + 1; };
    auto request = [&]() __attribute__((always_inline)) {
        const uint32_t b = l0 + fill * kStep;
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            if (p.once) copy_to_lds16_once(vw[i], bw, b + (wave + i * NW) * 1024);
            else copy_to_lds16_at(vw[i], bw, b + (wave + i * NW) * 1024);
        }
#pragma unroll
        for (int i = 0; i < AI; ++i) copy_to_lds16_at(va[i], ba, b + BW * kRowBytes + min(wave + i * NW, AC - 1) * 1024);
        ++issued;
        // (No branch: a step of a narrow tile takes 0.2 us, and a jump out of the loop's line costs 4 to 11 % of it.  Head of 4000 x 4096, one token:
        // 16.5 us, with the jump 18.2; 1024 x 2048 in bf16, 300 tokens: 10.8 and 12.0; 14336 x 4096 in fp32, 17 tokens: 55.7 and 58.9.)
        const int64_t on = kRowBytes - (kTurns && issued == n - first ? (int64_t)n * kRowBytes : 0);
        bw += on;
        ba += on;
        fill = next(fill);
    };
    f32x4 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int col = lane & 15, g = lane >> 4;
    while (issued < min(NB - 1, n)) request();
    for (int k = 0; k < n; ++k) {
        // this step's tile has arrived, and nobody reads the buffer of the step before any more
        if (issued - k >= NB - 1) pipe_barrier<(NB - 2) * (WI + AI)>(); else pipe_barrier<0>();
        if (issued < n) request();
        const char* lw = lds + use * kStep;
        const char* la = lw + BW * kRowBytes;
        use = next(use);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u32x4 fw[MI], fa[NI];
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int r = wr * (BW / WR) + i * 16 + col;
                fw[i] = *reinterpret_cast<const u32x4*>(lw + r * kRowBytes + ((s * 4 + g) ^ swz128(r)) * 16);
            }
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int r = wc * (BT / WC) + j * 16 + col;
                fa[j] = *reinterpret_cast<const u32x4*>(la + r * kRowBytes + ((s * 4 + g) ^ swz128(r)) * 16);
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) acc[i][j] = mma16<T>(fw[i], fa[j], acc[i][j]);
        }
    }
    gemm_store<T, EPI, MI, NI>(p, t, acc, t.tw * BW + wr * (BW / WR), t.tt * BT + wc * (BT / WC), col, g);
}

// 256 rows x 256 tokens, eight waves of 128 x 64 in two groups of four (waves i and i + 4 share a SIMD) that take turns: while one
// group multiplies a quarter of its step's products, the other reads operands from LDS and requests copies.  Group 1 runs one
// barrier behind.  The quarters of step k are (W half 0, A half 0), (W0, A1), (W1, A1), (W1, A0); their reads are spread evenly, 8, 8, 4 and 4 per
// wave: A0 and the second part of W0; A1 and the first part of W1; the rest of W1; the first part of the next W0 (12, 4, 8 and 0, as the
// products need them, is 2 to 4 % slower: the longest turn decides).  The copies of a half two steps on go to its place one quarter after its
// last read, when both groups have it; four or five halves stay in flight behind each wait.
template <int EPI>
__global__ __launch_bounds__(512, 2) void k_seq_gemm8(SeqGemm p) {
    constexpr int B = 256, kHalf = 128 * kRowBytes, kStep = 4 * kHalf;         // W0, W1, A0, A1
    extern __shared__ __align__(1024) char lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wr = wave >> 2, wc = wave & 3;
    GemmTile t;
    if (!gemm_tile<B, B>(p, t)) return;
    const int nk = p.kbytes / kRowBytes, kb = mul_div(nk, t.split, p.splits), n = mul_div(nk, t.split + 1, p.splits) - kb;
    const char* bw = uniform(t.w + (size_t)t.tw * B * p.kbytes + (size_t)kb * kRowBytes);
    const char* ba = uniform(p.a + (p.tile_off != nullptr ? (size_t)0 : (size_t)t.tt * B * p.lda) + (size_t)kb * kRowBytes);
    // half h of W: rows wr * 128 + h * 64 + 0 .. 63 of both groups; half h of A: tokens wc * 64 + h * 32 + 0 .. 31 of the four columns
    uint32_t vw[2][2], va[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int q = (wave + i * 8) * 8 + (lane >> 3), u = ((lane & 7) ^ swz128(q)) * 16;       // row of the half in LDS
            vw[h][i] = (uint32_t)min((q >> 6) * 128 + h * 64 + (q & 63), p.n - 1 - t.tw * B) * (uint32_t)p.kbytes + u;
            va[h][i] = gemm_input_row<B>(p, t, (q >> 5) * 64 + h * 32 + (q & 31)) + u;
        }
    const uint32_t l0 = lds_address(lds);
    enum { W0, W1, A0, A1 };
    // (past the last step its bytes are copied again, to places that nobody reads)
    auto request = [&](int what, int k) __attribute__((always_inline)) {
        const char* s = (what < A0 ? bw : ba) + (size_t)min(k, n - 1) * kRowBytes;
        const uint32_t d = l0 + (k & 1) * kStep + what * kHalf;
#pragma unroll
        for (int i = 0; i < 2; ++i) copy_to_lds16_at(what < A0 ? vw[what & 1][i] : va[what & 1][i], s, d + (wave + i * 8) * 1024);
    };
    f32x4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int col = lane & 15, g = lane >> 4;
    u32x4 fw0[4][2], fw1[4][2], fa0[2][2], fa1[2][2];
    const int u0 = (g ^ swz128(col)) * 16, u1 = ((4 + g) ^ swz128(col)) * 16;  // (16 rows on, the swizzle is the same)
    const char* lw = lds + (wr * 64 + col) * kRowBytes;
    const char* la = lds + A0 * kHalf + (wc * 32 + col) * kRowBytes;
    auto read_w = [&](u32x4 (&f)[4][2], int k, int h, int i0) __attribute__((always_inline)) {
        const char* b = lw + (k & 1) * kStep + h * kHalf;
#pragma unroll
        for (int i = i0; i < i0 + 2; ++i) {
            f[i][0] = *reinterpret_cast<const u32x4*>(b + i * 16 * kRowBytes + u0);
            f[i][1] = *reinterpret_cast<const u32x4*>(b + i * 16 * kRowBytes + u1);
        }
    };
    auto read_a = [&](u32x4 (&f)[2][2], int k, int h) __attribute__((always_inline)) {
        const char* b = la + (k & 1) * kStep + h * kHalf;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            f[j][0] = *reinterpret_cast<const u32x4*>(b + j * 16 * kRowBytes + u0);
            f[j][1] = *reinterpret_cast<const u32x4*>(b + j * 16 * kRowBytes + u1);
        }
    };
    auto turn = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // the end of a quarter's reads, its products, and the end of its turn at the matrix cores
    auto multiply = [&](int wh, const u32x4 (&w)[4][2], const u32x4 (&f)[2][2], int ah) __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        turn();
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[wh * 4 + i][ah * 2 + j] = mma16<bf16_t>(w[i][s], f[j][s], acc[wh * 4 + i][ah * 2 + j]);
        __builtin_amdgcn_s_setprio(0);
        turn();
    };
    request(W0, 0);
    request(A0, 0);
    request(A1, 0);
    request(W1, 0);
    request(W0, 1);
    request(A0, 1);
    request(A1, 1);
    wait_vm<10>();                                       // W0 and A0 of the first step
    turn();
    if (wr == 1) turn();
    read_w(fw0, 0, 0, 0);
    for (int k = 0; k < n; ++k) {
        read_a(fa0, k, 0);
        read_w(fw0, k, 0, 2);
        request(W1, k + 1);
        wait_vm<8>();                                    // (behind A1 and W1 of this step: W0, A0, A1, W1 of the next ones)
        multiply(0, fw0, fa0, 0);
        read_a(fa1, k, 1);
        read_w(fw1, k, 1, 0);
        request(W0, k + 2);
        multiply(0, fw0, fa1, 1);
        read_w(fw1, k, 1, 2);
        request(A0, k + 2);
        wait_vm<10>();                                   // (behind the next W0: A0, A1, W1, and W0, A0 of the step after it)
        multiply(1, fw1, fa1, 1);
        read_w(fw0, k + 1, 0, 0);
        request(A1, k + 2);
        wait_vm<10>();                                   // (behind the next A0)
        multiply(1, fw1, fa0, 0);
    }
    if (wr == 0) turn();
    wait_vm<0>();                                        // (no copy is in flight when the workgroup's LDS goes to another)
    gemm_store<bf16_t, EPI, 8, 4>(p, t, acc, t.tw * B + wr * 128, t.tt * B + wc * 64, col, g);
}

}  // namespace cfpp
