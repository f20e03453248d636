// What the kernels of a portion of the sequence models are launched with, from sizes alone.  Plain C++ without the device's headers, so
// that the choices can be looked at on the host.
#pragma once
#include <math.h>
#include <stddef.h>

#include <algorithm>

namespace cfpp {

inline int up_to(int a, int b) { return (a + b - 1) / b * b; }
inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// The tiles of the matrix products and what they cost, in us, as measured on an MI355X over 2 to 4000 tokens, 1500 to 50432
// rows and k of 1408 to 14336 (bf16; fp32: 17 to 1500 tokens): a step of 128 bytes of k when a compute unit has one workgroup, the
// share of a step when it has `resident` of them (the more of them, the more bytes in flight; past that they take turns), and
// what a workgroup costs beside its steps.  (bf16: with all waves copying.  Since four waves do, steps are up to 17 % shorter in all tiles but those of
// weight streams; a table fitted to that chose tiles that are 0.7 % better on their own and up to 2 % worse in a model, so it stays.)
// The estimate below is there to compare tiles: a product takes longer than it says, 10 % on average for the tile chosen (root mean
// square 16 %; fp32 15 and 20 %), most where it is a stream of weights: 22528 x 4096 estimated and measured 36 / 35 us for 66 tokens, 36 / 38
// for 100, 40 / 44 for 150, 58 / 63 for 300, 84 / 87 for 512, 253 / 272 for 2048.  What it chooses is 1.7 % slower than the best tile and split
// measured, on average over 15 products and 14 numbers of tokens, 22 % at worst (10816 x 4096 for 17 tokens); fp32, over 5 products, 8 numbers of tokens
// and two sizes of k, 1.9 and 28 % (4100 x 4128 for 301 tokens).  The fp32 tiles of 64 tokens and more multiply parts in bf16 (k_seq_gemm_split).
// A tile is in the table because it is missed where it is chosen; without it the next choice takes longer, on average and at most:
// 64 x 16 2 / 24 %, 64 x 32 7 / 29, 64 x 64 6 / 13, 64 x 96 11 / 34, 256 x 96 0 / 9, 256 x 128 19 / 34,
// 256 x 256 11 / 27, 128 x 64 3 / 11, 96 x 128 11 / 31, 128 x 128 alone on a compute unit 16 / 48, 128 x 192 10 / 21, 192 x 160 8 / 31, 96 x 160 10 / 17.
// (256 x 96, which a product alone can do without, is for the experts' rows: see plan_experts.)  128 x 128 with two workgroups per compute unit is for few steps of k (keys and values from latents of 200 values, 4000 positions) and for 128256 rows of
// a head.
// The tiles from the ninth on are for 50 to 700 tokens, where a product is still a stream of weights, which tiles of few tokens read
// two or three times: they hold the tokens in one tile or two, and their rings fill a compute unit's LDS.
struct GemmShape { int rows, tokens, resident; float step, share, fixed; };
constexpr GemmShape kShapes16[] = {{64, 16, 2, 0.213f, 0.180f, 1.7f}, {64, 32, 2, 0.228f, 0.204f, 1.9f}, {64, 64, 2, 0.269f, 0.241f, 2.4f},
                                   {64, 96, 2, 0.304f, 0.282f, 2.9f}, {256, 96, 1, 0.804f, 0.804f, 5.5f}, {128, 128, 2, 0.618f, 0.618f, 5.3f},
                                   {256, 128, 1, 0.919f, 0.919f, 6.9f}, {256, 256, 1, 1.098f, 1.098f, 13.9f},
                                   {128, 64, 2, 0.414f, 0.396f, 3.0f}, {96, 128, 1, 0.496f, 0.496f, 4.1f}, {128, 128, 1, 0.549f, 0.549f, 4.6f},
                                   {128, 192, 1, 0.693f, 0.693f, 5.7f}, {192, 160, 1, 0.807f, 0.807f, 6.4f}, {96, 160, 1, 0.557f, 0.557f, 4.7f}};
constexpr GemmShape kShapes32[] = {{64, 16, 2, 0.285f, 0.215f, 1.7f}, {64, 32, 2, 0.393f, 0.320f, 2.0f}, {64, 64, 2, 0.489f, 0.450f, 4.4f},
                                   {128, 128, 1, 1.000f, 1.000f, 6.5f}, {128, 64, 1, 0.630f, 0.630f, 5.3f}};
struct GemmShapes {
    const GemmShape* first;
    int count;
    const GemmShape& operator[](int i) const { return first[i]; }
};
inline GemmShapes shapes_of(bool bf16) {
    if (bf16) return {kShapes16, (int)(sizeof(kShapes16) / sizeof(kShapes16[0]))};
    return {kShapes32, (int)(sizeof(kShapes32) / sizeof(kShapes32[0]))};
}

// `tiles` tiles of `steps` steps on `cus` compute units
inline float gemm_tiles_cost(const GemmShape& c, double tiles, float steps, int cus) {
    const int load = (int)ceil(tiles / cus), full = load / c.resident, rest = load % c.resident;
    float t = full * (steps * std::max(c.step, c.resident * c.share) + c.fixed);
    if (rest > 0) t += steps * std::max(c.step, rest * c.share) + c.fixed;
    return t;
}
// what a stream of so many bytes takes at 5.8 TB/s
inline float stream_cost(double bytes) { return (float)(bytes / 5.8e6); }

// A plain product: n rows of kbytes bytes, m tokens; `room` floats for partial results of rows of ldy floats (0: k is not split).
struct GemmSizes {
    int n, m, kbytes, ldy;
    size_t room;
    int steps() const { return kbytes / 128; }
};
// Its time with one tile and one number of splits.  Reading a partial result costs its bytes at 5 TB/s, and 0.3 us.
inline float gemm_cost(const GemmSizes& g, const GemmShape& c, int splits, int cus) {
    const double tiles = (double)ceil_div(g.n, c.rows) * ceil_div(g.m, c.tokens) * splits;
    float t = std::max(gemm_tiles_cost(c, tiles, (float)g.steps() / splits, cus), stream_cost((double)g.n * g.kbytes));
    if (splits > 1) t += 0.3f + 4e-6f * splits * g.m * g.n / 5.0f;
    return t;
}
// The cheapest tile, and with room for partial results the cheapest number of splits of k as well.  No split has fewer than three steps.
struct GemmPlan { int shape, splits; };
inline GemmPlan plan_gemm(const GemmSizes& g, bool bf16, int cus) {
    const GemmShapes shapes = shapes_of(bf16);
    GemmPlan best{0, 1};
    float least = INFINITY;
    for (int i = 0; i < shapes.count; ++i)
        for (int sp : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (sp > 1 && (g.room == 0 || g.steps() / sp < 3 || (size_t)sp * g.m * g.ldy > g.room)) break;
            const float t = gemm_cost(g, shapes[i], sp, cus);
            if (t < least) {
                least = t;
                best = {i, sp};
            }
        }
    return best;
}

// Tile of the expert products of a portion of n tokens (both use it).  An expert has avg +- sqrt(avg) of them; where that fits a
// tile, it has one (`once`), and the product is a stream of weights.  A stream hides the tiles' own time only in part: with 66 tokens
// per expert, 64 experts of 2816 x 2048 take 159 us in tiles of 64 x 96, estimated at 118, and 151 us in tiles of 256 x 96, at 94.
struct ExpertSizes { int n, top, experts, ff, xbytes; };     // tokens, experts of a token, experts, their inner size, bytes of an input row
struct ExpertPlan { int shape, tokens, once; };
struct ExpertCost { float stream, tiles; };
// of `rows` rows of `kbytes` bytes of each expert
inline ExpertCost expert_cost(const ExpertSizes& e, const GemmShape& c, int rows, int kbytes, int cus) {
    const double avg = (double)e.n * e.top / e.experts, live = e.experts * std::min(1.0, avg);
    const bool one = avg + 1.5 * sqrt(avg) <= c.tokens;
    const double per = one ? 1.0 : std::max(1.0, avg / c.tokens + 0.5);
    return {stream_cost(live * rows * kbytes), gemm_tiles_cost(c, live * per * ceil_div(rows, c.rows), (float)kbytes / 128, cus)};
}
inline float expert_time(const ExpertCost& c) { return std::max(c.tiles, c.stream) + 0.3f * std::min(c.tiles, c.stream); }
inline ExpertPlan plan_experts(const ExpertSizes& e, bool bf16, int cus) {
    const GemmShapes shapes = shapes_of(bf16);
    const double avg = (double)e.n * e.top / e.experts;
    ExpertPlan best{};
    float least = INFINITY;
    for (int i = 0; i < shapes.count; ++i) {
        const float cost = expert_time(expert_cost(e, shapes[i], 2 * e.ff, e.xbytes, cus));
        if (cost < least) {
            least = cost;
            best = {i, shapes[i].tokens, avg + 1.5 * sqrt(avg) <= shapes[i].tokens};
        }
    }
    return best;
}
// Whether the shared expert's product g goes into the launch of the experts' (`rows` rows of `kbytes` bytes each), in their tile: where
// both together are estimated to take less than one after the other with a launch of 1.5 us in between, and no tile of it outlasts the experts'
// product.  Only tiles of 64 rows, two of which share a compute unit: one works while the other waits for weights.  (A compute unit that has one tile at
// a time does one after the other: 700 tokens, tiles of 256 x 96, 137 + 25 us in two launches, 162 in one.)  Five layers of 64 experts of 1408 x 2048 with
// six of them and a shared one of 2816 for each token, two launches and one: 2 tokens 562 -> 527 us, 10 947 -> 896, 40 1218 -> 1182, 150 1400 -> 1385, 300 and 500 equal to 1 %.
inline bool plan_beside(const ExpertSizes& e, const ExpertPlan& plan, int rows, int kbytes, const GemmSizes& g, bool bf16, int cus) {
    const GemmShape& c = shapes_of(bf16)[plan.shape];
    if (c.rows != 64 || (!bf16 && c.tokens >= 64)) return false;     // (fp32: a kernel of another kind)
    const float own = g.steps() * c.step + c.fixed, tiles = (float)(ceil_div(g.n, c.rows) * ceil_div(g.m, c.tokens));
    const ExpertCost alone = expert_cost(e, c, rows, kbytes, cus);
    const ExpertCost both = {alone.stream + stream_cost((double)g.n * g.kbytes), alone.tiles + tiles / cus * (g.steps() * std::max(c.share, c.step / c.resident) + c.fixed / c.resident)};
    const GemmPlan own_plan = plan_gemm(g, bf16, cus);
    return own <= std::max(alone.stream, alone.tiles) && expert_time(both) < expert_time(alone) + 1.5f + gemm_cost(g, shapes_of(bf16)[own_plan.shape], own_plan.splits, cus);
}

// Attention of a portion of T tokens at positions pos0 and on: R query heads for each of G key / value heads, `keys` of them in a tile.
struct AttnSizes {
    int T, R, G, pos0, chunk, keys;
    bool pairs;              // bf16: waves of 32 columns are possible
    int per_cu;              // workgroups that share a compute unit
    size_t floats;           // of a split's partial results
};
// Columns of a workgroup and splits of the keys.  bf16: waves of 32 columns take fewer instructions per weight, those of 16 balance better
// where there are few workgroups.  The line is at two workgroups of four such waves per compute unit, which is where it belongs for 32 heads of 128
// (us with 16 / 32 columns: 1500 tokens, 384 workgroups 43 / 52, 2048 tokens, 512 workgroups 67 / 68, 3000 122 / 126; behind 1990 positions 114 / 122,
// 156 / 150, 262 / 248).  Of keys of 192 it is early for prompts (2048 tokens 74 / 76, 2300 88 / 95, 3000 140 / 133; at 1990 183 / 171), of heads of
// 64 more so (2048 39 / 45, 3000 69 / 71; at 1990 96 / 89), and of 256 late for 32 heads (1500 110 / 93, 2048 167 / 143; at 1990 421 / 333).
// Splits fill the chip: two workgroups per compute unit, with two tiles at least in each split of the longest walk, which begins at the chunk of the
// portion's first token (that chunk counts and not the context: 37 tokens just behind a chunk of 8192 see one tile; shared by 16 splits, eight layers
// of 32 / 8 heads of 128 took 1005 us, and take 957).
//
// The order of the workgroups.  A row of them is the same columns of all key heads and splits; rows go from the last block of columns, which walks
// the most keys, to the first.  Where all are resident, two per compute unit, workgroups i and i + `cus` share one (the hardware places them in turn:
// read from its registers, 512 workgroups of 64 KB), so the rows behind the first `cus` workgroups go upwards, and a long walk has a short one beside
// it.  In us, head by head / downwards only / so, in fp32: 16 heads of 192 and 128, 1000 tokens 101 / 94 / 63; 32 / 8 heads of 128, 1000 tokens 129 /
// 107 / 85; 10 / 5 heads of 64, 1500 tokens in two splits 52 / 57 / 43; 12 / 4 heads of 96 and 80, 700 tokens in three 38 / 43 / 31; bf16, where
// a walk of so few workgroups is short: equal to 1 %.  With more workgroups the longest come first, since what is left over goes where a walk has
// ended.  Two that share a compute unit should not end together: then two that are left over go there, and other units stay idle.  The older one
// of the two is served first, so a somewhat longer one ends with the younger (768 workgroups, 1500 tokens at 1990, fp32: on 128 units within 10 us,
// and four workgroups on each of these, two on the others).  So where there is less than one left over per unit, and the walks are alike, the
// younger are the longer ones: 32 heads of 192 and 128, 1150 tokens at 1990, fp32 731 -> 585 us, 1500 tokens 848 -> 701 (610 and 729 when reads
// of values were waited for and the older one ended first), bf16 133 -> 116 and 153 -> 139.  Alike: at least half as many keys in front of the portion
// as in it, and no chunk that begins inside (2100 tokens at 0 in bf16 would take 83 us instead of 73).
struct AttnPlan { bool two; int splits, up, swap; };         // rows that go down; so many rows come behind as many that follow them
constexpr int attn_block(int row, int rows, int up, int swap) {
    return row >= up ? row - up : rows - 1 - (row < swap ? row + swap : row < 2 * swap ? row - swap : row);
}
inline AttnPlan plan_attn(const AttnSizes& a, int cus, size_t room) {
    const int cols = a.T * a.R, behind = a.pos0 + a.T - (a.chunk > 0 ? a.pos0 / a.chunk * a.chunk : 0);
    const int tiles = ceil_div(a.chunk > 0 ? std::min(behind, a.chunk) : behind, a.keys);
    const bool two = a.pairs && ceil_div(cols, 128) * a.G >= 2 * cus;
    const int wgs = ceil_div(cols, two ? 128 : 64) * a.G;
    const int splits = std::max(1, (int)std::min<size_t>({(size_t)16, (size_t)(a.per_cu * cus / wgs), (size_t)(tiles / 2), room / a.floats}));
    const int rows = wgs / a.G, some = std::max(1, cus / (a.G * splits)), total = wgs * splits;
    if (a.per_cu >= 2 && total <= 2 * cus) return {two, splits, some, 0};
    const bool alike = 2 * (behind - a.T) >= a.T && (a.chunk == 0 || behind <= a.chunk);
    return {two, splits, rows, a.per_cu >= 2 && total <= 3 * cus && alike ? std::min(some, rows / 2) : 0};
}

// A portion of few tokens behind many positions: latent attention may read the cached latents themselves instead of the keys and values that are
// made of them.  A column (token, head) then takes products of `rank` values with every key instead of dim and vdim of them, and leaves sums of `rank` values
// for each split; keys and values cost the same for one token as for a hundred.  Where the line is follows from an estimate of both, with
// coefficients fitted to the difference measured over latent_2b, latent_6b9, latent_wide and a small uneven model (16, 32, 128 and 12 heads), 2 to 150 tokens at
// 200, 1000, 3000 and 4000 (bf16: 128 differences, 6 us off on average; fp32: the uneven model alone).  In us per layer, made and read: 16 heads at 3000,
// 2 tokens 108 / 91, 20 110 / 104, 40 113 / 112, 64 118 / 124; 128 heads at 3000, 2 tokens 411 / 282, 20 429 / 342, 64 480 / 469, 100 514 / 588; at 1000,
// 20 333 / 319, 64 406 / 409; at 200, 10 300 / 302; 12 heads in fp32 at 3000, 2 tokens 111 / 85, 20 121 / 110, 64 139 / 164.  Not chosen within 4 us, which
// is what the estimate misses small models by.
// Held against both ways over 11 models (12 to 128 heads of 64 to 192 dimensions, ranks of 64 to 512), 2 to 250 tokens at 150 to 64000, 1666 sizes in bf16 and
// 1645 in fp32: layers take 25 and 35 % less on average where the latents are read (617 and 866 sizes); 8 and 6 of these are more than 0.6 % slower, 2.8 % at
// most (fp32, 32 heads of rank 256, which takes the kernel for 512: 64 tokens at 6000 417 / 429).  Ranks of up to 128, whose kernel takes less than the estimate
// says, are among them (353 sizes, 6 % faster and more); 382 sizes that would gain over 3 % are left to keys and values.  With more tokens the choice may come
// back: the product that makes keys takes another row of tiles (64 heads at 2000: 48 tokens 173 / 178 us, 49 208 / 178; 32 heads at 1000: 24 159 / 165, 25
// 164 / 164), or attention another block of columns.
// n tokens at pos and on; dim, rot, vdim: values of a head's key (plain, rotated) and value; bytes of a latent row, latents of it.
struct LatentSizes {
    int n, pos, heads, dim, rot, vdim, kbytes, rank;
    bool bf16;
    size_t room;             // floats for partial results
};
// splits 0: keys and values are made.  sets: of 16 columns in a block; tokens: of a workgroup that merges kTurnSplits splits at most and multiplies kTurnRows
// rows of W_uv by them.
struct LatentTurn { int splits, sets, tokens; };
constexpr int kTurnSplits = 64, kTurnRows = 64;
inline LatentTurn plan_latent_turn(const LatentSizes& z, int cus) {
    if (z.n > 256) return {};                            // (not measured)
    const int keys = z.bf16 ? 32 : 16, cols = z.n * z.heads, ctx = z.pos + z.n, tiles = ceil_div(ctx, keys), esize = z.bf16 ? 2 : 4;
    const GemmSizes g{z.heads * (z.dim + z.vdim), ctx, z.kbytes, 0, 0};
    const GemmPlan made = plan_gemm(g, z.bf16, cus);
    const float gemm = gemm_cost(g, shapes_of(z.bf16)[made.shape], made.splits, cus);
    const float mb = 1e-6f * ctx * g.n * esize, gflop = 2e-9f * ctx * cols * (z.dim + z.rot + z.vdim);
    const float least = z.bf16 ? 14.0f + 0.86f * gemm + 0.067f * mb + 1.3f * gflop : 1.0f + 0.7f * gemm + 0.26f * mb + 0.3f * gflop;
    LatentTurn best{};
    float cost = least - 4.0f;                           // (of what is chosen: a round of workgroups, its tiles, partial results, columns)
    const int most = (int)std::min<size_t>({(size_t)kTurnSplits, z.room / ((size_t)cols * (z.rank + 2)), (size_t)ceil_div(tiles, 2)});
    for (int sets : {1, 2, 4}) {
        const float tile = sets == 1 ? 1.4f : sets == 2 ? 1.65f : 2.3f;
        for (int splits = 1; splits <= most; ++splits) {
            const float rounds = (float)ceil_div(ceil_div(cols, 16 * sets) * splits, cus), walk = rounds * ceil_div(tiles, splits) * tile;
            const float parts = 4e-6f * cols * splits * z.rank;
            const float t = z.bf16 ? 16.0f * rounds + 0.83f * walk + 0.44f * parts + 3.2e-3f * cols : 0.6f * rounds + 1.3f * walk + 0.6f * parts + 4e-3f * cols;
            if (t < cost) {
                cost = t;
                best = {splits, sets, 16};
            }
        }
    }
    while (best.tokens > 2 && z.heads * ceil_div(z.vdim, kTurnRows) * ceil_div(z.n, best.tokens) < cus) best.tokens /= 2;
    return best;
}

}  // namespace cfpp
