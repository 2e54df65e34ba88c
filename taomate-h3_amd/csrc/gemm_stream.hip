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

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Microseconds of a call with one tile size: per round of 256 tiles a launch,
// the first memory round trip and the epilogue, and per 128-byte k-tile the
// bytes a CU pulls ((BM + BN) * 128) and its matrix instructions (BM * BN).
// Fitted to 84 measured calls (N x K of the H3 and benchmark projections, M =
// 40 .. 3200, tiled operands); it picks the fastest of the ten tiles or one
// within 6% of it in 80 of them.
double stream_cost(const StreamTile& t, const GemmArgs& a) {
    const double per_ktile = 8e-4 * (t.bm + t.bn) + 1.3e-5 * t.bm * t.bn;
    const int64_t rounds = ceil_div(ceil_div(a.m, t.bm) * ceil_div(a.n, t.bn), kCus);
    return 2.0 + rounds * (3.5 + a.k / 128.0 * per_ktile);
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

}  // namespace

// The rule looks at sizes only (never at the layouts when an adapter is
// present), so a call gives the same bits whatever layout its operands have.
int stream_tile(const GemmArgs& a) {
    // 16-byte output pieces and 32-bit block-relative offsets.
    if (a.n % 8 || a.ldo % 8 || (uintptr_t)a.out % 16 || a.k < 128) return 0;
    if (a.lora_t && (a.out_f16 || a.lora_rank > 128)) return 0;
    if (256 * a.k >= (int64_t(1) << 30)) return 0;
    const StreamTile* best = nullptr;
    double cost = 0.0;
    for (const StreamTile& t : kTiles) {
        const double c = stream_cost(t, a);
        if (best == nullptr || c < cost) {
            best = &t;
            cost = c;
        }
    }
    if (a.m > kSkinnyMaxM) {
        // Against the four-wave kernel (or the 16-wave one where K is not a
        // multiple of 128): 0.78 keeps the calls that gain in both weight
        // states (Infinity Cache, HBM) and both layouts; of those left out the
        // best gained 8% in one state and lost 3% in the other.
        return cost < 0.78 * four_wave_cost(a) ? best->id : 0;
    }
    // Against the weight-streaming kernels of M <= 128, which take no adapter.
    if (a.lora_t) return best->id;  // M = 40, 10752 x 5376, rank 64: 61 us by the per-tile kernel
    if (a.b_tiled) {
        // They give every CU 32 columns and all of A: 14.8 against 11.8 us at
        // 128 x 5120 x 5120, but 10.8 against 11.8 us at M = 64; above 8192
        // columns their 32-column workgroups no longer fit one round (M = 40,
        // N = 10752: 20.6 against 14.5 us; N = 5120: 10.2 against 11.3 us).
        return a.m > 64 || (a.m > 32 && a.n > 8192) ? best->id : 0;
    }
    // Row-major weights: 20 x 5120 x 5120 14.0 against 13.2 us, 100 x 5120 x
    // 5120 38 against 14 us; short K the other way (64 x 2048 x 2048 7.4 against
    // 8.1 us, 64 x 1024 x 1040 5.0 against 7.1 us).
    return (a.m > 16 && a.k >= 3072) || (a.m > 64 && a.k >= 2048) ? best->id : 0;
}

hipError_t launch_gemm_stream(int kind, int tile, const GemmArgs& a, hipStream_t st) {
    if (kind == kOpE4M3) return a.b_tiled ? launch_stream_e4m3_tiled(tile, a, st) : launch_stream_e4m3_rows(tile, a, st);
    return a.b_tiled ? launch_stream_int8_tiled(tile, a, st) : launch_stream_int8_rows(tile, a, st);
}

}  // namespace h3q
