// Choice and launch of the weight-streaming GEMM's tile (gemm_stream.hpp).
#include "h3q_kernels.hpp"

#include "gemm_stream.hpp"

namespace h3q {

namespace {

struct StreamTile {
    int id, bm, bn;  // id: the case of launch_stream_op
};
constexpr StreamTile kTiles[] = {{42, 64, 64},   {44, 64, 128},  {54, 80, 128}, {64, 96, 128},  {74, 112, 128},
                                 {84, 128, 128}, {58, 80, 256},  {68, 96, 256}, {78, 112, 256}, {88, 128, 256}};
constexpr int64_t kCus = 256;
// Predicted time of a split call over that of the four-wave kernel alone, at most.
constexpr double kSplitGain = 0.98;

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Microseconds of a call with one tile size: per round of 256 tiles a launch,
// the first memory round trip and the epilogue, and per 128-byte k-tile the
// bytes a CU pulls ((BM + BN) * 128) and its matrix instructions (BM * BN).
// Fitted to 84 measured calls (N x K of the H3 and benchmark projections, M =
// 40 .. 3200, tiled operands); it picks the fastest of the ten tiles or one
// within 6% of it in 80 of them.
double stream_cost(const StreamTile& t, int64_t m, int64_t n, int64_t k) {
    const double per_ktile = 8e-4 * (t.bm + t.bn) + 1.3e-5 * t.bm * t.bn;
    const int64_t rounds = ceil_div(ceil_div(m, t.bm) * ceil_div(n, t.bn), kCus);
    return 2.0 + rounds * (3.5 + k / 128.0 * per_ktile);
}

struct StreamChoice {
    int tile;
    double cost;
};
StreamChoice best_stream_tile(int64_t m, int64_t n, int64_t k) {
    StreamChoice best{0, 0.0};
    for (const StreamTile& t : kTiles) {
        const double c = stream_cost(t, m, n, k);
        if (best.tile == 0 || c < best.cost) best = {t.id, c};
    }
    return best;
}

// The forms and offsets that gemm_stream_kernel takes.
bool stream_takes(const GemmArgs& a) {
    // 16-byte output pieces and 32-bit block-relative offsets.
    if (a.n % 8 || a.ldo % 8 || (uintptr_t)a.out % 16 || a.k < 128) return false;
    // The bias comes in by LDS copies of whole dwords.  The per-tile kernels, whose
    // calls with a K tail, binary16 output or few rows and an adapter come here, read
    // it element by element and keep those with a bias at an odd element.
    if ((uintptr_t)a.bias % 4) return false;
    if (a.lora_t && (a.out_f16 || a.lora_rank > 128)) return false;
    return 256 * a.k < (int64_t(1) << 30);
}

// The same of the four-wave kernel: 64-byte k-steps of 0.68 us in a full round
// of 256 x 256 tiles, 0.62 us in a last round more than half full, 0.51 us in
// one whose tiles run as halves.
double four_wave_cost(const GemmArgs& a) {
    const int64_t tiles = ceil_div(a.m, 256) * ceil_div(a.n, 256);
    const int64_t rounds = tiles / kCus, rem = tiles % kCus;
    const double last = rem == 0 ? 0.0 : (2 * rem <= kCus ? 0.51 : 0.62);
    return 8.0 + a.k / 64.0 * (0.68 * rounds + last);
}

// The same of the sixteen-wave kernels (gemm.hip), which take a K that is not a
// multiple of 128: 128-byte k-tiles of 1.75 us in a full round of 256 x 256 tiles,
// 1.13 us plus up to 0.8 by its tiles in the last one.
double sixteen_wave_cost(const GemmArgs& a) {
    const int64_t tiles = ceil_div(a.m, 256) * ceil_div(a.n, 256), ktiles = ceil_div(a.k, 128);
    const int64_t rounds = tiles / kCus, rem = tiles % kCus;
    const double last = rem == 0 ? 0.0 : 1.13 + 0.8 * rem / kCus;
    return 11.0 * ceil_div(tiles, kCus) + ktiles * (1.75 * rounds + last);
}

// The streaming kernel with such a K, over its cost with tiled operands: against the
// persistent sixteen-wave kernel, its binary16 form and its form with an adapter.
// Measured on 1668 calls (192 .. 16384 rows, N 256 .. 5376, K 144 .. 4112): of 567 that
// go to the sixteen-wave kernels almost all are faster there, up to 30% (3500 x 3520 x
// 4112 binary16 65.6 against 80.9 us, with an adapter 65.1 / 84.2, 16384 x 4096 x 624 bf16
// 84.0 / 103.5); those left are up to 3.8 times faster here (600 x 3520 x 1040 21.3 / 11.0,
// 2600 x 256 x 4112 49.7 / 14.1), and 27 of them up to 10% slower.
double tail_factor(const GemmArgs& a) { return a.lora_t ? 1.72 : (a.out_f16 ? 1.68 : 1.54); }

// Whether the streaming tiles are the faster ones for M <= 128 rows, decided on
// weights that come from HBM, as a step reads those of each layer (measured on
// about 900 calls, N 512 .. 16384, K 256 .. 13824, both weight states; below, HBM
// and in parentheses Infinity Cache, us, gemm_skinny.hip / these tiles).
//
// Tiled weights: there a workgroup takes 32 columns and all of A.  Up to 8192
// columns these are one round, and at 65 .. 128 rows the streaming tiles gain from
// the cache only (128 x 5120 x 5120 14.3 / 15.3 (12.9 / 10.6), 128 x 2048 x 2048
// 7.0 / 8.7 (5.5 / 7.2)) until K is long (128 x 5120 x 13824 35.2 / 33.6 (34.8 /
// 22.6)).  Above, they gain at every K (128 x 10752 x 5376 30.1 / 23.4).  At 33 ..
// 64 rows a workgroup does half the work and its second round hides more (40 x
// 10752 x 5376 20.5 / 17.7, 40 x 8208 x 5120 2-6% slower, 40 x 16384 x 4096 3%).
bool beats_skinny_tiled(int64_t m, int64_t n, int64_t k) {
    if (m > 64) return n > 8192 || k >= 12288;
    return m > 32 && n > 10240 && k >= 5120;
}

// Row-major weights: there a workgroup takes 16 columns and its time grows with
// the rows; up to 4096 columns each CU gets one, up to 8192 two.  A K that is not a
// multiple of 128 costs these tiles 10-25%.  32 x 1024 x 3072 6.8 / 9.6, 64 x 2048
// x 2048 7.5 / 8.5, 64 x 4096 x 5120 18.0 / 17.8 (14.4 / 12.1), 65 x 2048 x 2048 8.6 /
// 8.4, 65 x 2048 x 3088 10.3 / 11.1, 96 x 2048 x 3088 12.9 / 11.1, 17 x 5120 x 5120
// 16.6 / 16.1, 17 x 8192 x 5120 17.7 / 18.9, 24 x 5120 x 3072 12.1 / 11.6, 32 x 5120 x
// 3088 15.3 / 14.4 (9.2 / 10.0), 128 x 5120 x 5120 51 / 18.
bool beats_skinny_rows(int64_t m, int64_t n, int64_t k) {
    const bool tail = k % 128 != 0;
    if (n <= 4096) {
        if (m > 64) return k >= (!tail ? 2048 : m > 80 ? 3072 : 4096);
        return m > 56 && k >= 5120;
    }
    if (m > 64) return k >= 2048;
    if (m > 32) return k >= 3072;
    if (m > 24) return k >= (tail ? 4096 : 3072);
    if (m <= 16) return false;
    if (n > 8192) return k >= 3072;
    return !tail && k >= (n > 6144 ? 7168 : 5120);
}

}  // namespace

// Above 128 rows, and with an adapter at any count, the rule looks at sizes and at
// the output's alignment, never at the layouts, so there a call gives the same bits
// whatever layout its operands have.  Up to 128 rows without one the layout of the
// weights decides, and e4m3 sums may differ in their order between layouts.
int stream_tile(const GemmArgs& a) {
    if (!stream_takes(a)) return 0;
    const StreamChoice best = best_stream_tile(a.m, a.n, a.k);
    if (a.m > kSkinnyMaxM) {
        if (a.k % 128) return tail_factor(a) * best.cost - 2.0 < sixteen_wave_cost(a) ? best.tile : 0;
        // Against the four-wave kernel: 0.78 keeps the calls that gain in both weight
        // states (Infinity Cache, HBM) and both layouts; of those left out the
        // best gained 8% in one state and lost 3% in the other.
        return best.cost < 0.78 * four_wave_cost(a) ? best.tile : 0;
    }
    // M <= 128: against the kernels of gemm_skinny.hip, which take no adapter
    // (M = 40, 10752 x 5376, rank 64: 61 us by the per-tile kernel) and read tiled
    // activations beside tiled weights only.
    if (a.lora_t || (a.a_tiled && !a.b_tiled) || (a.b_tiled ? beats_skinny_tiled(a.m, a.n, a.k) : beats_skinny_rows(a.m, a.n, a.k))) return best.tile;
    return 0;
}

// A last round of a few 256 x 256 tiles costs the four-wave kernel 0.51 us per
// 64-byte step on an otherwise idle chip.  Here full rounds keep that kernel (the
// first columns or rows of the output) and what is left is spread over all CUs by
// smaller weight-streaming tiles, in a second launch.  The candidates are the
// largest first part of all full rounds and of one fewer, by columns and by rows.
// Sizes only, as above.  Measured on 44 calls (1223 .. 19873 rows, H3 and
// benchmark projections, with the quantizer): predicted below 0.8 of one launch
// 10-15% faster (3179 x 5376 x 7168 154 -> 133 us, 6411 x 5120 x 13824 444 -> 389),
// 0.8-0.9 3-8%, 0.9-0.98 0-3% (one of 20 0.1% slower), above it -0.3 .. +1.3%.
GemmSplit gemm_split(const GemmArgs& a) {
    GemmSplit split{false, 0, 0};
    if (!stream_takes(a)) return split;
    const int64_t tiles_m = ceil_div(a.m, 256), tiles_n = ceil_div(a.n, 256);
    const int64_t rounds = tiles_m * tiles_n / kCus;
    if (rounds == 0 || tiles_m * tiles_n % kCus == 0) return split;
    double cost = kSplitGain * four_wave_cost(a);
    for (int64_t full = rounds; full > 0 && full >= rounds - 1; --full) {
        const double main = 8.0 + a.k / 64.0 * 0.68 * full;
        const int64_t n0 = full * kCus / tiles_m * 256, m0 = full * kCus / tiles_n * 256;
        if (n0 > 0 && n0 < a.n) {
            const StreamChoice rest = best_stream_tile(a.m, a.n - n0, a.k);
            if (main + rest.cost < cost) {
                split = {true, n0, rest.tile};
                cost = main + rest.cost;
            }
        }
        if (m0 > 0 && m0 < a.m) {
            const StreamChoice rest = best_stream_tile(a.m - m0, a.n, a.k);
            if (main + rest.cost < cost) {
                split = {false, m0, rest.tile};
                cost = main + rest.cost;
            }
        }
    }
    return split;
}

hipError_t launch_gemm_split(int kind, const GemmSplit& split, const GemmArgs& a, hipStream_t st) {
    GemmArgs head = a, rest = a;
    if (split.columns) {
        const int64_t n0 = split.at;
        head.n = n0;
        rest.n = a.n - n0;
        rest.b = (const uint8_t*)a.b + (a.b_tiled ? n0 / 16 * (a.k / 128) * 2048 : n0 * a.ldb);
        if (a.b_scale_per_col) rest.b_scale = a.b_scale + n0;
        if (a.bias) rest.bias = a.bias + n0;
        if (a.lora_t) rest.lora_b = a.lora_b + n0 * a.ldlb;
        rest.out = (uint16_t*)a.out + n0;
    } else {
        const int64_t m0 = split.at;
        head.m = m0;
        rest.m = a.m - m0;
        rest.a = (const uint8_t*)a.a + (a.a_tiled ? m0 / 16 * (a.k / 128) * 2048 : m0 * a.lda);
        if (a.a_scale_per_row) rest.a_scale = a.a_scale + m0;
        if (a.lora_t) rest.lora_t = a.lora_t + m0 * a.ldt;
        rest.out = (uint16_t*)a.out + m0 * a.ldo;
    }
    const hipError_t e = launch_gemm_w4(kind, head, st);
    return e != hipSuccess ? e : launch_gemm_stream(kind, split.tile, rest, st);
}

void stream_tile_shape(int tile, int64_t* rows, int64_t* columns) {
    for (const StreamTile& t : kTiles)
        if (t.id == tile) *rows = t.bm, *columns = t.bn;
}

hipError_t launch_gemm_stream(int kind, int tile, const GemmArgs& a, hipStream_t st) {
    if (kind == kOpE4M3) return a.b_tiled ? launch_stream_e4m3_tiled(tile, a, st) : launch_stream_e4m3_rows(tile, a, st);
    return a.b_tiled ? launch_stream_int8_tiled(tile, a, st) : launch_stream_int8_rows(tile, a, st);
}

}  // namespace h3q
