// Weight-streaming scaled GEMM for a few dozen to a few thousand rows, gfx950.
//
//   out[m, n] = round( s_a[m] * (s_w[n] * float(sum_k A[m, k] * W[n, k])) [+ bias[n]]
//                      [+ lora_scale * (t[m, :] . lora_b[n, :])] )
//
// What bounds it.  At these row counts the 256 x 256 tiles of the four-wave
// kernel leave most of the 256 CUs idle, and its ring of four 64-byte k-steps
// waits for memory: about 0.51 us per step whatever the tile count (47 us for
// any M from 129 to 1376 at N = K = 5120).  Here every CU gets one tile of a
// size chosen so that the tiles come to at most 256 where they can (stream_tile), and
// the loop is bound by what one CU can pull: measured on MI355X, 8 waves
// reading with 16-byte loads get 130 KB/us from the L2, 89 KB/us when the lines
// come from the Infinity Cache and 55 KB/us from HBM (a CU has about 25 KB of
// line fills in flight, and more loads in flight or prefetches by the same CU
// do not raise it).  So a tile's cost is (BM + BN) * K bytes, plus the matrix
// instructions, which run at a power-limited clock once every CU issues them.
//
// Work split.  A workgroup of 8 waves owns BM = 16 MT rows and BN = 32 WN
// columns; wave (kg, wn) takes columns 32 wn .. 32 wn + 31 and every WK-th
// 128-byte k-tile (WK = 8 / WN groups), so the weights go from memory straight
// into the registers of the one wave that uses them, D = 4 k-tiles ahead.  The
// activations of a k-tile are read by WN waves: they come into an LDS ring of
// SA stages (WK k-tiles each) by LDS-DMA.  Each wave reads a 16-row fragment
// two slots ahead of its two MFMAs (v_mfma_f32_16x16x128_f8f6f4 or two
// v_mfma_i32_16x16x64_i8 each); one barrier per stage, in the middle of the
// stage, both publishes the next one and frees the previous one, so no
// fragment read waits behind it.  After the last k-tile the WK partial sums are
// added in group order through LDS (each group finishes its share of the row
// blocks), scaled, staged as a 2-byte tile and stored as whole rows.
//
// Operand layouts.  Tiled operands are copied or loaded in place: a 16-row
// block of a k-tile is 2 KiB in fragment order.  Row-major ones are read as
// whole 128-byte lines, 8 rows per 1 KiB instruction, with 16-byte chunk c of
// row r placed at chunk c ^ swz(r) so that the fragment reads of 16 rows hit
// distinct banks; row-major weights pass through 2 KiB of LDS per wave to get
// into fragment order.  Rows past M / N and chunks past K read as zeros.
//
// Measured (random codes, tiled operands, us; four-wave kernel -> this one;
// weights in the Infinity Cache / from HBM):
//   M x N x K              four-wave      this kernel
//   160 x 5120 x 5120      45.4 / 46.2    11.8 / 13.9
//   592 x 10752 x 5376     48.9 / 50.3    32.8 / 37.9
//   1043 x 5120 x 5120     46.6 / 47.0    27.0 / 33.5
//   1376 x 5120 x 13824    112  / 114     88.2 / 91.4
// and against the weight-streaming kernel of M <= 128 (gemm_skinny.hip), which keeps
// the second of these (gemm_stream.hip):
//   112 x 10752 x 5376     28.9 / 29.4    15.9 / 22.9
//   128 x 5120 x 5120      12.9 / 14.3    10.6 / 15.3
#pragma once

#include <stdint.h>

#include <type_traits>

#include "gemm_tiles.hpp"
#include "h3q_common.hpp"
#include "h3q_kernels.hpp"

namespace h3q {

template <int OP>
struct StreamMfma;
template <>
struct StreamMfma<kOpE4M3> {
    using acc_t = v4f;
    static __device__ __forceinline__ acc_t run(v8i a, v8i b, acc_t c) {
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
    }
};
template <>
struct StreamMfma<kOpInt8> {
    using acc_t = v4i;
    static __device__ __forceinline__ acc_t run(v8i a, v8i b, acc_t c) {
        const v4i alo = {a[0], a[1], a[2], a[3]}, ahi = {a[4], a[5], a[6], a[7]};
        const v4i blo = {b[0], b[1], b[2], b[3]}, bhi = {b[4], b[5], b[6], b[7]};
        c = __builtin_amdgcn_mfma_i32_16x16x64_i8(alo, blo, c, 0, 0, 0);
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(ahi, bhi, c, 0, 0, 0);
    }
};

template <int MT_, int WN_, bool TB_, bool LORA_>
struct StreamCfg {
    static constexpr bool TB = TB_, LORA = LORA_;          // tiled weights, adapter in the epilogue
    static constexpr int MT = MT_, WN = WN_, WK = 8 / WN_;
    static constexpr int BM = 16 * MT, BN = 32 * WN;
    static constexpr int D = 4;                            // weight k-tiles in registers
    static constexpr int PF = 2;                           // row-block fragments read ahead
    static constexpr int STAGE = WK * MT * 2048;           // activations: one k-tile of 128 bytes per K group
    static constexpr int OTHER = 3 * 1024 + (LORA ? MT * 4096 : 16) + (TB ? 16 : 8 * 2048);  // LDS besides the ring
    static constexpr int SA = 4 * STAGE + OTHER <= 160 * 1024 ? 4 : 3;  // ring stages
    static constexpr int PIECES = WK * MT * 2;             // 1 KiB copies per stage
    static constexpr int CA = (PIECES + 7) / 8;            // copies per wave, at most
    static constexpr int CA_MIN = PIECES / 8;              // and at least
    // Loads a wave has issued after the copies of stage s + 1 when it waits for
    // them in the middle of stage s, at least: vmcnt at or below it means they
    // have landed (loads complete in order).
    static constexpr int WAIT = (SA - 2) * 4 + (SA - 3) * CA_MIN;
    static constexpr int WAIT_TAIL = (SA - 3) * CA_MIN;    // the copies alone
    static constexpr int RSLOT = (MT + WK - 1) / WK * (WK - 1);  // row blocks a wave hands to the other K groups
    static constexpr int RED = 8 * RSLOT * 2048;
    static constexpr int OUT = BM * BN * 2;
    static constexpr int RING = SA * STAGE;
    static constexpr int LDS = (RING > RED ? RING : RED) > OUT ? (RING > RED ? RING : RED) : OUT;
    static_assert(MT >= 4 && MT <= 8 && D >= SA - 2, "fragment ring and wait counts");
    static_assert(D * 4 + SA * CA + 4 < 63, "vmcnt range");
};

template <int OP, class C>
__global__ __launch_bounds__(512, 2) void gemm_stream_kernel(GemmArgs p, int tiles_m, int tiles_n, int stream_out) {
    using acc_t = typename StreamMfma<OP>::acc_t;
    constexpr bool TB = C::TB, LORA = C::LORA;
    constexpr int MT = C::MT, WN = C::WN, WK = C::WK, D = C::D, SA = C::SA, BM = C::BM, BN = C::BN, PF = C::PF;
    constexpr uint32_t kOob = 0x80000000u;  // beyond every descriptor's range: loads return 0, stores drop
    constexpr int kNonTemporal = 2;         // cache policy of large outputs (see gemm_w4.hip)
    __shared__ __attribute__((aligned(1024))) uint8_t lds_ring[C::LDS];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_vec[3 * 1024];  // row scales | column scales | bias
    __shared__ __attribute__((aligned(1024))) uint8_t lds_t[LORA ? MT * 4096 : 16];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_w[TB ? 16 : 8 * 2048];
    H3Q_LDS uint8_t* const ring = (H3Q_LDS uint8_t*)lds_ring;
    H3Q_LDS uint8_t* const vec = (H3Q_LDS uint8_t*)lds_vec;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, kg = wave / WN;
    const int r16 = lane & 15, kq = lane >> 4;
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int rows = (int)(p.m - m0 < BM ? p.m - m0 : BM);
    const int cols = (int)(p.n - n0 < BN ? p.n - n0 : BN);
    const int kbytes = (int)p.k;
    const int steps = (kbytes + 127) >> 7;
    const int iters = (steps + WK - 1) / WK;
    const bool ta = p.a_tiled != 0;

    // Row-major 1 KiB pieces: lane l holds row 8 half + l / 8, 16-byte chunk
    // (l % 8) ^ swz(row) of the row's 128 bytes; the fragment of (row r16,
    // bytes 32 kq ..) is then read at `row_lo`, `row_hi`.
    auto swz = [](int r) __attribute__((always_inline)) { return (r ^ (r >> 3)) & 7; };
    const int lo_row = lane >> 3, lo_chunk = (lane & 7) ^ swz(lo_row), hi_chunk = (lane & 7) ^ swz(8 + lo_row);
    const uint32_t row_base = (uint32_t)((r16 >> 3) * 1024 + (r16 & 7) * 128);
    const uint32_t row_lo = row_base + (uint32_t)(((2 * kq) ^ swz(r16)) << 4);
    const uint32_t row_hi = row_base + (uint32_t)(((2 * kq + 1) ^ swz(r16)) << 4);

    // Activation pieces of this wave: c = wave + 8 i is half c % 2 of row block
    // (c / 2) % MT of K group (c / 2) / MT.
    const uint32_t a_bytes = ta ? (uint32_t)((rows + 15) / 16 * steps * 2048) : (uint32_t)rows * (uint32_t)p.lda;
    const CopySrc ra((const uint8_t*)p.a + (ta ? (m0 / 16) * steps * 2048 : m0 * p.lda), a_bytes);
    const uint32_t a_kstep = ta ? 2048u : 128u;
    const int a_half = wave & 1;
    const int a_byte = ta ? 0 : 16 * (a_half ? hi_chunk : lo_chunk);  // of the k-tile's 128 (tiled: whole k-tiles only)
    uint32_t aoff[C::CA];
#pragma unroll
    for (int i = 0; i < C::CA; ++i) {
        const int blk = ((wave + 8 * i) >> 1) % MT;
        if (ta) {
            aoff[i] = 16 * blk < rows ? (uint32_t)(blk * steps * 2048 + a_half * 1024 + lane * 16) : kOob;
        } else {
            const int row = 16 * blk + 8 * a_half + lo_row;
            aoff[i] = row < rows ? (uint32_t)(row * (int)p.lda + a_byte) : kOob;
        }
    }
    auto copy_a = [&](int s, int st) __attribute__((always_inline)) {  // super-step s into ring slot st
        const uint32_t base = (uint32_t)(uintptr_t)(ring + st * C::STAGE);
#pragma unroll
        for (int i = 0; i < C::CA; ++i) {
            const int c = wave + 8 * i;
            if (C::PIECES % 8 != 0 && c >= C::PIECES) break;
            const int kt = s * WK + (c >> 1) / MT;
            uint32_t off = a_byte < kbytes - kt * 128 ? aoff[i] + (uint32_t)kt * a_kstep : kOob;
            asm volatile("" : "+v"(off));
            copy16(ra, base + (uint32_t)(c * 1024), off);
        }
    };

    // Weights of this wave: column blocks 2 wn, 2 wn + 1, two 1 KiB loads each
    // per k-tile (tiled: the halves of the block; row-major: rows 0..7, 8..15).
    const uint32_t b_bytes = TB ? (uint32_t)((cols + 15) / 16 * steps * 2048) : (uint32_t)cols * (uint32_t)p.ldb;
    const __amdgpu_buffer_rsrc_t rb =
        make_rsrc((const uint8_t*)p.b + (TB ? (n0 / 16) * steps * 2048 : n0 * p.ldb), b_bytes);
    uint32_t boff[2][TB ? 1 : 2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int blk = 2 * wn + j;
        if constexpr (TB) {
            boff[j][0] = 16 * blk < cols ? (uint32_t)(blk * steps * 2048 + lane * 16) : kOob;
        } else {
            const int row = 16 * blk + lo_row;
            boff[j][0] = row < cols ? (uint32_t)(row * (int)p.ldb + 16 * lo_chunk) : kOob;
            boff[j][1] = row + 8 < cols ? (uint32_t)((row + 8) * (int)p.ldb + 16 * hi_chunk) : kOob;
        }
    }
    auto load_b = [&](int s, v8i (&w)[2]) __attribute__((always_inline)) {
        const int kt = s * WK + kg;
        const int left = kbytes - kt * 128;  // bytes of K from this k-tile on
        // Past K: an offset beyond the descriptor (below 2^30 bytes) for every
        // lane (the wait counts need every load issued, so no branch; the
        // empty asm keeps the compiler from making one, or one load of two).
        uint32_t k0 = left > 0 ? (uint32_t)kt * (TB ? 2048u : 128u) : 0x40000000u;
        asm volatile("" : "+s"(k0));
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t o_lo = boff[j][0] + k0;
            uint32_t o_hi = TB ? boff[j][0] + k0 + 1024u : boff[j][TB ? 0 : 1] + k0;
            if constexpr (!TB) {
                o_lo = 16 * lo_chunk < left ? o_lo : kOob;
                o_hi = 16 * hi_chunk < left ? o_hi : kOob;
                asm volatile("" : "+v"(o_lo), "+v"(o_hi));
            }
            const v4u lo = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rb, o_lo, 0, 0));
            const v4u hi = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rb, o_hi, 0, 0));
            w[j] = v8i{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
        }
    };
    // The loaded pieces of one column block as an MFMA fragment.
    auto weight_frag = [&](const v8i& w) __attribute__((always_inline)) -> v8i {
        if constexpr (TB) return w;
        H3Q_LDS uint8_t* const q = (H3Q_LDS uint8_t*)lds_w + wave * 2048;
        *(H3Q_LDS v4i*)(q + lane * 16) = v4i{w[0], w[1], w[2], w[3]};
        *(H3Q_LDS v4i*)(q + 1024 + lane * 16) = v4i{w[4], w[5], w[6], w[7]};
        const v4i lo = *(const H3Q_LDS v4i*)(q + row_lo), hi = *(const H3Q_LDS v4i*)(q + row_hi);
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    const uint32_t frag_lo = ta ? (uint32_t)(lane * 16) : row_lo, frag_hi = ta ? 1024u + (uint32_t)(lane * 16) : row_hi;
    auto frag = [&](int st, int t) __attribute__((always_inline)) -> v8i {
        const H3Q_LDS uint8_t* q = ring + st * C::STAGE + (kg * MT + t) * 2048;
        const v4i lo = *(const H3Q_LDS v4i*)(q + frag_lo);
        const v4i hi = *(const H3Q_LDS v4i*)(q + frag_hi);
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };

    acc_t acc[2][MT];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[j][t] = acc_t{};

    // Prologue: epilogue vectors and adapter rows, activation stages
    // 0 .. SA - 2, weight k-tiles 0 .. D - 1.
    if (wave == 0)
        copy16(CopySrc(p.a_scale + (p.a_scale_per_row ? m0 : 0), (uint32_t)(p.a_scale_per_row ? rows : 1) * 4u),
               (uint32_t)(uintptr_t)vec, 16u * lane);
    if (wave == 1)
        copy16(CopySrc(p.b_scale + (p.b_scale_per_col ? n0 : 0), (uint32_t)(p.b_scale_per_col ? cols : 1) * 4u),
               (uint32_t)(uintptr_t)(vec + 1024), 16u * lane);
    if (wave == 2 && p.bias)
        copy16(CopySrc(p.bias + n0, (uint32_t)cols * 2u), (uint32_t)(uintptr_t)(vec + 2048),
               lane < 32 ? 16u * lane : kOob);
    if constexpr (LORA) {  // piece c: row block c / 4, ranks 32 (c % 4) .. + 31, in bf16 fragment order
        const CopySrc rt((const uint8_t*)p.lora_t + m0 * p.ldt * 2, (uint32_t)rows * (uint32_t)p.ldt * 2u);
        for (int c = wave; c < MT * 4; c += 8) {
            const int row = 16 * (c >> 2) + r16, k = 32 * (c & 3) + 8 * kq;
            copy16(rt, (uint32_t)(uintptr_t)((H3Q_LDS uint8_t*)lds_t + c * 1024),
                   row < rows && k < p.lora_rank ? (uint32_t)((row * (int)p.ldt + k) * 2) : kOob);
        }
    }
#pragma unroll
    for (int s = 0; s < SA - 1; ++s) copy_a(s, s);
    v8i wb[D][2];
#pragma unroll
    for (int d = 0; d < D; ++d) load_b(d, wb[d]);
    wait_vmcnt<(SA - 2) * C::CA_MIN + 4 * D>();  // stage 0 has landed
    asm volatile("s_barrier" ::: "memory");

    int st = 0;  // ring slot of the running super-step
    // Row-block fragments in a register ring of four, read PF slots ahead of
    // their MFMAs, across super-steps (D * MT is a multiple of four, so the
    // ring position is a constant of the unrolled step).
    v8i xf[4];
#pragma unroll
    for (int t = 0; t < PF; ++t) xf[t] = frag(0, t);
    // The last steps (tail) load no more weights, so only the copies count
    // behind the ones they wait for.
    auto step = [&](int s, auto phase, auto tail, v8i (&w)[2]) __attribute__((always_inline)) {
        constexpr int P0 = decltype(phase)::value;
        constexpr bool TAIL = decltype(tail)::value;
        constexpr int MID = MT / 2 - 1;  // MID + 1 + PF <= MT: the next stage is published before its first read
        const int nst = st + 1 == SA ? 0 : st + 1, pst = st == 0 ? SA - 1 : st - 1;
        const v8i w0 = weight_frag(w[0]), w1 = weight_frag(w[1]);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            xf[(P0 + t + PF) & 3] = t + PF < MT ? frag(st, t + PF) : frag(nst, t + PF - MT);
            __builtin_amdgcn_sched_barrier(0);
            acc[0][t] = StreamMfma<OP>::run(w0, xf[(P0 + t) & 3], acc[0][t]);
            acc[1][t] = StreamMfma<OP>::run(w1, xf[(P0 + t) & 3], acc[1][t]);
            if (t == MID) {
                // Every wave is past super-step s - 1 (its MFMAs hold what
                // they read), so that slot takes stage s - 1 + SA; stage
                // s + 1 has landed in every wave.
                wait_vmcnt<TAIL ? C::WAIT_TAIL : C::WAIT>();
                asm volatile("s_barrier" ::: "memory");
                copy_a(s - 1 + SA, pst);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!TAIL) load_b(s + D, w);
        __builtin_amdgcn_sched_barrier(0);
        st = nst;
    };
    const std::integral_constant<int, 0> p0;
    const std::integral_constant<int, MT & 3> p1;
    const std::integral_constant<int, (2 * MT) & 3> p2;
    const std::integral_constant<int, (3 * MT) & 3> p3;
    const std::false_type body;
    const std::true_type tail;
    int s = 0;
    for (; s + D <= iters; s += D) {
        step(s, p0, body, wb[0]);
        step(s + 1, p1, body, wb[1]);
        step(s + 2, p2, body, wb[2]);
        step(s + 3, p3, body, wb[3]);
    }
    if (s < iters) step(s, p0, tail, wb[0]);
    if (s + 1 < iters) step(s + 1, p1, tail, wb[1]);
    if (s + 2 < iters) step(s + 2, p2, tail, wb[2]);
    // All copies have landed (the trailing ones read zeros past K) and every
    // wave is done with the ring.
    wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // Sum of the K groups in group order: group g finishes row blocks t with
    // t % WK == g and hands the others over through LDS.
    if constexpr (WK > 1) {
        H3Q_LDS acc_t* const red = (H3Q_LDS acc_t*)ring;
        auto slot = [&](int g, int j, int t) __attribute__((always_inline)) -> int {  // t % WK != g
            const int x = t / WK * (WK - 1) + t % WK - (t % WK > g ? 1 : 0);
            return (((g * WN + wn) * 2 + j) * C::RSLOT + x) * 64 + lane;
        };
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t)
                if (t % WK != kg) red[slot(kg, j, t)] = acc[j][t];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                if (t % WK != kg) continue;
                acc_t sum = kg == 0 ? acc[j][t] : red[slot(0, j, t)];
#pragma unroll
                for (int g = 1; g < WK; ++g) {
                    if (g == kg) sum += acc[j][t];
                    else sum += red[slot(g, j, t)];
                }
                acc[j][t] = sum;
            }
        __syncthreads();
    }

    // Epilogue: the scaled rows are staged as a [BM, BN] tile of 2-byte
    // outputs (16-byte chunk c of row r at c ^ (r % 8)), then stored by rows.
    const bool f16 = p.out_f16 != 0, has_bias = p.bias != nullptr;
    v4i lb[2][4];
    if constexpr (LORA) {
        const __amdgpu_buffer_rsrc_t rl =
            make_rsrc((const uint8_t*)p.lora_b + n0 * p.ldlb * 2, (uint32_t)cols * (uint32_t)p.ldlb * 2u);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = 32 * wn + 16 * j + r16, k = 32 * q + 8 * kq;
                lb[j][q] = __builtin_bit_cast(
                    v4i, __builtin_amdgcn_raw_buffer_load_b128(
                             rl, row < cols && k < p.lora_rank ? (uint32_t)((row * (int)p.ldlb + k) * 2) : kOob, 0, 0));
            }
    }
    const H3Q_LDS float* vsa = (const H3Q_LDS float*)vec;
    const H3Q_LDS float* vsw = (const H3Q_LDS float*)(vec + 1024);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int nl = 32 * wn + 16 * j + 4 * kq;  // first of this lane's four columns
        v4f sw;
        if (p.b_scale_per_col) sw = *(const H3Q_LDS v4f*)(vsw + nl);
        else sw = v4f{vsw[0], vsw[0], vsw[0], vsw[0]};
        v2u b2 = {0u, 0u};
        if (has_bias) b2 = *(const H3Q_LDS v2u*)(vec + 2048 + 2 * nl);
        const float bias[4] = {out_lo(b2[0], f16), out_hi(b2[0], f16), out_lo(b2[1], f16), out_hi(b2[1], f16)};
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            if (WK > 1 && t % WK != kg) continue;
            const int ml = 16 * t + r16;
            const float sa = vsa[p.a_scale_per_row ? ml : 0];
            v4f l = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (LORA) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v4i tf = *(const H3Q_LDS v4i*)((const H3Q_LDS uint8_t*)lds_t + (t * 4 + q) * 1024 + lane * 16);
                    l = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, lb[j][q]),
                                                                __builtin_bit_cast(v8bf, tf), l, 0, 0, 0);
                }
            }
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = __fmul_rn(sw[e], (float)acc[j][t][e]);
                y[e] = has_bias ? __builtin_fmaf(sa, v, bias[e]) : __fmul_rn(sa, v);
                if constexpr (LORA) y[e] = __builtin_fmaf(p.lora_scale, l[e], y[e]);
            }
            *(H3Q_LDS v2u*)(ring + ml * (BN * 2) + (((nl >> 3) ^ (ml & 7)) << 4) + (nl & 4) * 2) =
                v2u{pack_out2(y[0], y[1], f16), pack_out2(y[2], y[3], f16)};
        }
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t ro = make_rsrc((uint8_t*)p.out + m0 * p.ldo * 2, (uint32_t)rows * (uint32_t)p.ldo * 2u);
    constexpr int CH = BN / 8;  // 16-byte chunks per row
    for (int i = threadIdx.x; i < BM * CH; i += 512) {
        const int r = i / CH, c = i % CH;
        const v4u v = *(const H3Q_LDS v4u*)(ring + r * (BN * 2) + ((c ^ (r & 7)) << 4));
        const uint32_t off = 8 * c < cols && r < rows ? (uint32_t)(r * (int)p.ldo + (int)n0 + 8 * c) * 2u : 0xFFFFFFF0u;
        if (stream_out) __builtin_amdgcn_raw_buffer_store_b128(v, ro, off, 0, kNonTemporal);
        else __builtin_amdgcn_raw_buffer_store_b128(v, ro, off, 0, 0);
    }
}

template <int OP, int MT, int WN, bool TB>
hipError_t launch_stream_cfg(const GemmArgs& a, hipStream_t st) {
    using Plain = StreamCfg<MT, WN, TB, false>;
    using Lora = StreamCfg<MT, WN, TB, true>;
    const int tiles_m = (int)((a.m + Plain::BM - 1) / Plain::BM), tiles_n = (int)((a.n + Plain::BN - 1) / Plain::BN);
    const int stream_out = a.m * a.ldo * 2 >= (int64_t(64) << 20);
    const dim3 grid((unsigned)(tiles_m * tiles_n));
    if (a.lora_t)
        hipLaunchKernelGGL((gemm_stream_kernel<OP, Lora>), grid, dim3(512), 0, st, a, tiles_m, tiles_n, stream_out);
    else
        hipLaunchKernelGGL((gemm_stream_kernel<OP, Plain>), grid, dim3(512), 0, st, a, tiles_m, tiles_n, stream_out);
    return hipGetLastError();
}

template <int OP, bool TB>
hipError_t launch_stream_op(int tile, const GemmArgs& a, hipStream_t st) {
    switch (tile) {
        case 42: return launch_stream_cfg<OP, 4, 2, TB>(a, st);
        case 44: return launch_stream_cfg<OP, 4, 4, TB>(a, st);
        case 54: return launch_stream_cfg<OP, 5, 4, TB>(a, st);
        case 64: return launch_stream_cfg<OP, 6, 4, TB>(a, st);
        case 74: return launch_stream_cfg<OP, 7, 4, TB>(a, st);
        case 84: return launch_stream_cfg<OP, 8, 4, TB>(a, st);
        case 58: return launch_stream_cfg<OP, 5, 8, TB>(a, st);
        case 68: return launch_stream_cfg<OP, 6, 8, TB>(a, st);
        case 78: return launch_stream_cfg<OP, 7, 8, TB>(a, st);
        case 88: return launch_stream_cfg<OP, 8, 8, TB>(a, st);
        default: return hipErrorInvalidValue;
    }
}

// One instance per operand kind and weight layout, each in its own source file.
hipError_t launch_stream_e4m3_tiled(int tile, const GemmArgs& a, hipStream_t st);
hipError_t launch_stream_e4m3_rows(int tile, const GemmArgs& a, hipStream_t st);
hipError_t launch_stream_int8_tiled(int tile, const GemmArgs& a, hipStream_t st);
hipError_t launch_stream_int8_rows(int tile, const GemmArgs& a, hipStream_t st);

}  // namespace h3q
