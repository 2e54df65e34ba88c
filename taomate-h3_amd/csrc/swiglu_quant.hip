// Fused SwiGLU + per-token quantization, gfx950: the producer of the fc2 input
// of a DiT MLP (H3/model/layers.py:469-479: F.silu(gate) * up, or the Triton
// fused_swiglu of H3/inference/fused_kernels.py:240-261, 663-677), with the
// activation quantizer of the following W8A8 linear folded in.  For a row
// [gate (F) | up (F)] of bf16:
//
//   e = exp(-gate)
//   s = bf16(gate / (1 + e))           (IEEE binary32 sum and division: torch's
//                                       silu, x / (1 + exp(-x)), rounded to bf16)
//   y = bf16(s * up)                   (stored if out)
//   codes, s_row = per-token quantization of y   (if codes)
//
// s depends on gate alone, through 65536 possible bf16 values.  The
// definition of e is exp_f32 of the CPU restatement (Cody and Waite reduction
// and a degree-7 polynomial from IEEE operations only, within 1 ulp of a
// correctly rounded exp); the kernel evaluates e with the hardware exp2
// (v_exp_f32 of -gate * RN(1/ln 2)), and s comes out bit-identical to the
// restatement's for every one of the 65536 bf16 gate values (checked
// exhaustively on MI355X, tests/test_gpu_swiglu.py), at 2 instructions instead
// of about 15 and two branches.  The sum, the division and the products are
// single IEEE operations in the order written, so the CPU restatement
// reproduces y bit for bit.  The reference's results differ from these only
// where its own exp (the library's, or Triton's) moves the binary32 silu
// across a bf16 rounding boundary.
//
// A row is shared by as many waves as it fills, y kept in VGPRs (8-element vectors)
// for the quantizer, so that even a few long rows spread over the chip.
// Per row 4F bytes in, F bytes of codes + 4 bytes of scale out (+ 2F with out).
//
// Table form (swiglu_quant_lut_kernel, from a row count that depends on the row's
// length, see launch_sq_fmt).
// Because s is a function of the 16-bit gate pattern alone, the library
// evaluates it once per device for all 65536 patterns (silu_table_kernel,
// the same instructions as above) into a 128 KiB table in device memory.
// Each workgroup copies the table into LDS when it starts and looks s up
// there (one LDS read per element instead of the exp, the sum and the IEEE
// division), so the outputs are the same bits and the kernel sheds about
// half of its vector instructions.  The first call on a device fills the
// table and waits for it (once); a call made while its stream is being
// captured into a graph before that has happened runs the form above.
#include <mutex>

#include "h3q_common.hpp"
#include "h3q_kernels.hpp"
#include "row_quant.hpp"

#pragma clang fp contract(off)

namespace h3q {

namespace {

__device__ __forceinline__ float silu_f32(float g) {
    const float e = __builtin_amdgcn_exp2f(-g * 0x1.715476p+0f);  // exp(-g)
    return g / (1.0f + e);
}

// Two gate and two up values (packed bf16) -> two y values (packed bf16).
__device__ __forceinline__ uint32_t swiglu2(uint32_t g, uint32_t u) {
    const uint32_t s = pack_bf16x2(silu_f32(bf16_lo(g)), silu_f32(bf16_hi(g)));
    return pack_bf16x2(bf16_lo(s) * bf16_lo(u), bf16_hi(s) * bf16_hi(u));
}

// The same with s read from the LDS table (indexed by the gate's bits).
__device__ __forceinline__ uint32_t swiglu2_lut(const H3Q_LDS uint16_t* t, uint32_t g, uint32_t u) {
    const uint32_t s = (uint32_t)t[g & 0xFFFFu] | ((uint32_t)t[g >> 16] << 16);
    return pack_bf16x2(bf16_lo(s) * bf16_lo(u), bf16_hi(s) * bf16_hi(u));
}

}  // namespace

// bf16(silu(g)) for every 16-bit pattern g, one per device (see above).
__device__ __align__(256) uint16_t silu_table[65536];

__global__ __launch_bounds__(256) void silu_table_kernel(uint16_t* __restrict__ table) {
    const uint32_t g = (blockIdx.x * 256 + threadIdx.x) * 2;
    // the pair (g, g + 1) as one packed word, rounded exactly as swiglu2 does
    const uint32_t w = g | ((g + 1) << 16);
    reinterpret_cast<uint32_t*>(table)[g >> 1] = pack_bf16x2(silu_f32(bf16_lo(w)), silu_f32(bf16_hi(w)));
}

// Direct form: workgroups of four waves, SPLIT waves to a row, NV vectors per lane
// each: wave `part` of a row takes vectors (SPLIT i + part) * 64 + lane, and the row's
// maximum is exchanged through LDS (double-buffered by parity, so one barrier a
// group of rows; a wave of its own needs none).
template <int FMT, int ROUND, int NV, int SPLIT>
__global__ __launch_bounds__(256) void swiglu_quant_kernel(SwigluQuantArgs p) {
    __shared__ uint32_t red[2][4];
    constexpr int kRows = 4 / SPLIT;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int part = wave % SPLIT, sub = wave / SPLIT;
    const int nvec = p.half >> 3;
    int parity = 0;
    const int64_t groups = (p.rows + kRows - 1) / kRows;
    for (int64_t group = blockIdx.x; group < groups; group += gridDim.x) {
        const int64_t row = group * kRows + sub;
        const bool live = row < p.rows;
        const uint4* gr = reinterpret_cast<const uint4*>(p.x + row * p.ldx);
        const uint4* ur = reinterpret_cast<const uint4*>(p.x + row * p.ldx + p.half);
        uint4 y[NV];
        uint32_t m = 0;
        constexpr int B = NV < 4 ? NV : 4;
#pragma unroll
        for (int i0 = 0; i0 < NV; i0 += B) {
            uint4 g[B], u[B];
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int vec = ((i0 + b) * SPLIT + part) * 64 + lane;
                const bool in = live && i0 + b < NV && vec < nvec;
                g[b] = in ? gr[vec] : make_uint4(0, 0, 0, 0);
                u[b] = in ? ur[vec] : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int b = 0; b < B; ++b) {
                if (i0 + b >= NV) break;
                y[i0 + b] = make_uint4(swiglu2(g[b].x, u[b].x), swiglu2(g[b].y, u[b].y), swiglu2(g[b].z, u[b].z),
                                       swiglu2(g[b].w, u[b].w));
                // Materialize the packed result here: without it the compiler
                // interleaves the exp sequences of several vectors and runs
                // out of registers.
                asm volatile("" : "+v"(y[i0 + b].x), "+v"(y[i0 + b].y), "+v"(y[i0 + b].z), "+v"(y[i0 + b].w));
                m = pk_abs_max(m, y[i0 + b].x);
                m = pk_abs_max(m, y[i0 + b].y);
                m = pk_abs_max(m, y[i0 + b].z);
                m = pk_abs_max(m, y[i0 + b].w);
            }
        }
        if (p.out && live) {
            uint4* orow = reinterpret_cast<uint4*>(p.out + row * p.ldo);
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int vec = (SPLIT * i + part) * 64 + lane;
                if (vec < nvec) orow[vec] = y[i];
            }
        }
        if (p.codes == nullptr) continue;
        float amax = wave_max(amax_from_packed(m));
        if constexpr (SPLIT > 1) {
            if (lane == 0) red[parity][wave] = __float_as_uint(amax);
            __syncthreads();
            amax = 0.0f;
#pragma unroll
            for (int w = 0; w < SPLIT; ++w) amax = mag_max(amax, __uint_as_float(red[parity][sub * SPLIT + w]));
            parity ^= 1;
        }
        if (!live) continue;
        RowQuant<FMT, ROUND> rq;
        rq.init(amax);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int vec = (SPLIT * i + part) * 64 + lane;
            if (vec < nvec) {
                uint2 o;
                o.x = rq.pack4(y[i].x, y[i].y);
                o.y = rq.pack4(y[i].z, y[i].w);
                *reinterpret_cast<uint2*>(p.codes + row * p.ldq + 8 * (int64_t)vec) = o;
            }
        }
        if (lane == 0 && part == 0) p.scales[row] = rq.s;
    }
}

// Table form: one workgroup of 16 waves per CU (the 128 KiB table fills most of
// the LDS), SPLIT waves to a row, so a workgroup takes groups of 16 / SPLIT rows
// blockIdx.x, blockIdx.x + grid, ...  The next group's gate and up are requested
// before the barrier that exchanges this group's maxima, so reads and stores
// overlap.  Measured on MI355X (int8 codes, inputs rotated, us; a wave per row of any
// length -> this): 2640 x 7168 26.4 -> 22.3, 8192 x 7168 59.6 -> 53.9, 8192 x 13824
// 119.4 -> 108.4 (5.2 TB/s, the rate of a large copy), 4000 x 14336 58.9 -> 54.5.
constexpr int kLutWaves = 16;
template <int FMT, int ROUND, int NV, int SPLIT>
__global__ __launch_bounds__(kLutWaves * 64) void swiglu_quant_lut_kernel(SwigluQuantArgs p,
                                                                         const uint16_t* __restrict__ table) {
    __shared__ __attribute__((aligned(1024))) uint16_t lds_table[65536];
    __shared__ uint32_t red[2][kLutWaves];
    constexpr int kRows = kLutWaves / SPLIT;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = wave % SPLIT, sub = wave / SPLIT;
    const int nvec = p.half >> 3;
    const int64_t groups = (p.rows + kRows - 1) / kRows;
    uint4 g[NV], u[NV];
    auto load = [&](int64_t group) __attribute__((always_inline)) {
        const int64_t row = group * kRows + sub;
        if (row >= p.rows) return;
        const uint4* gr = reinterpret_cast<const uint4*>(p.x + row * p.ldx);
        const uint4* ur = reinterpret_cast<const uint4*>(p.x + row * p.ldx + p.half);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int vec = (i * SPLIT + part) * 64 + lane;
            if (vec < nvec) {
                g[i] = gr[vec];
                u[i] = ur[vec];
            }
        }
    };
#pragma unroll
    for (int i = 0; i < NV; ++i) g[i] = u[i] = make_uint4(0, 0, 0, 0);  // lanes past the row: y = 0
    {
        // 128 KiB by LDS-DMA: 128 wave copies of 1 KiB.
        const CopySrc src(table, 65536u * 2u);
        const uint32_t base = (uint32_t)(uintptr_t)(H3Q_LDS uint16_t*)lds_table;
#pragma unroll
        for (int i = 0; i < 128 / kLutWaves; ++i) {
            const int c = wave + kLutWaves * i;
            copy16(src, base + (uint32_t)(c * 1024), (uint32_t)(c * 1024 + 16 * lane));
        }
        load(blockIdx.x);
        wait_vmcnt0();
        __syncthreads();
    }
    const H3Q_LDS uint16_t* t = (const H3Q_LDS uint16_t*)lds_table;
    int parity = 0;
    for (int64_t group = blockIdx.x; group < groups; group += gridDim.x) {
        const int64_t row = group * kRows + sub;
        uint4 y[NV];
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            y[i] = make_uint4(swiglu2_lut(t, g[i].x, u[i].x), swiglu2_lut(t, g[i].y, u[i].y),
                              swiglu2_lut(t, g[i].z, u[i].z), swiglu2_lut(t, g[i].w, u[i].w));
            // keeps the compiler from holding many vectors' lookups live at once
            asm volatile("" : "+v"(y[i].x), "+v"(y[i].y), "+v"(y[i].z), "+v"(y[i].w));
            m = pk_abs_max(m, y[i].x);
            m = pk_abs_max(m, y[i].y);
            m = pk_abs_max(m, y[i].z);
            m = pk_abs_max(m, y[i].w);
        }
        load(group + gridDim.x);
        float amax = wave_max(amax_from_packed(m));
        if constexpr (SPLIT > 1) {
            if (lane == 0) red[parity][wave] = __float_as_uint(amax);
            // (not __syncthreads: the next group's loads stay in flight)
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            amax = 0.0f;
#pragma unroll
            for (int w = 0; w < SPLIT; ++w) amax = mag_max(amax, __uint_as_float(red[parity][sub * SPLIT + w]));
            parity ^= 1;
        }
        if (row >= p.rows) continue;
        if (p.out) {
            uint4* orow = reinterpret_cast<uint4*>(p.out + row * p.ldo);
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int vec = (i * SPLIT + part) * 64 + lane;
                if (vec < nvec) orow[vec] = y[i];
            }
        }
        if (p.codes == nullptr) continue;
        RowQuant<FMT, ROUND> rq;
        rq.init(amax);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int vec = (i * SPLIT + part) * 64 + lane;
            if (vec < nvec) {
                uint2 o;
                o.x = rq.pack4(y[i].x, y[i].y);
                o.y = rq.pack4(y[i].z, y[i].w);
                *reinterpret_cast<uint2*>(p.codes + row * p.ldq + 8 * (int64_t)vec) = o;
            }
        }
        if (lane == 0 && part == 0) p.scales[row] = rq.s;
    }
}

namespace {

// The current device's table, filled on first use (launch + wait, once per
// device), and its CU count; null while a graph is being captured on st and
// the table does not exist yet.
hipError_t silu_table_for(hipStream_t st, const uint16_t** out, int* cus) {
    constexpr int kMaxDevices = 64;
    static std::mutex lock;
    static const uint16_t* tables[kMaxDevices] = {};
    static int cu_count[kMaxDevices] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> guard(lock);
    if (!tables[dev]) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        e = hipStreamIsCapturing(st, &status);
        if (e != hipSuccess) return e;
        if (status != hipStreamCaptureStatusNone) {
            *out = nullptr;
            return hipSuccess;
        }
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(silu_table));  // the current device's copy
        if (e != hipSuccess) return e;
        e = hipDeviceGetAttribute(&cu_count[dev], hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) return e;
        // The wait below is legal even while another stream of this thread
        // is being captured in global mode: relaxed mode for the fill only.
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        e = hipThreadExchangeStreamCaptureMode(&mode);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(silu_table_kernel, dim3(65536 / 512), dim3(256), 0, st, (uint16_t*)ptr);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        const hipError_t restore = hipThreadExchangeStreamCaptureMode(&mode);
        if (e == hipSuccess) e = restore;
        if (e != hipSuccess) return e;
        tables[dev] = (const uint16_t*)ptr;
    }
    *out = tables[dev];
    *cus = cu_count[dev] > 0 ? cu_count[dev] : 256;
    return hipSuccess;
}

// ND, SD: vectors per lane and waves per row of the direct form; NT, ST: those of the
// table form, which takes calls of at least `table_rows` rows.
template <int FMT, int ROUND, int ND, int SD, int NT, int ST>
hipError_t launch_sq_nv(const SwigluQuantArgs& a, int64_t table_rows, hipStream_t st) {
    if (a.rows >= table_rows) {
        const uint16_t* table = nullptr;
        int cus = 0;
        const hipError_t e = silu_table_for(st, &table, &cus);
        if (e != hipSuccess) return e;
        if (table) {
            constexpr int kRows = kLutWaves / ST;
            const int64_t groups = (a.rows + kRows - 1) / kRows;
            const int64_t blocks = groups < cus ? groups : cus;
            hipLaunchKernelGGL((swiglu_quant_lut_kernel<FMT, ROUND, NT, ST>), dim3((unsigned)blocks),
                               dim3(kLutWaves * 64), 0, st, a, table);
            return hipGetLastError();
        }
    }
    constexpr int64_t kBlocks = 8192;
    constexpr int kRows = 4 / SD;
    const int64_t groups = (a.rows + kRows - 1) / kRows;
    const int64_t blocks = groups < kBlocks ? groups : kBlocks;
    hipLaunchKernelGGL((swiglu_quant_kernel<FMT, ROUND, ND, SD>), dim3((unsigned)blocks), dim3(256), 0, st, a);
    return hipGetLastError();
}

// By the row's length: as many waves to a row as it fills, and the row count from
// which the table is paid back.  Its copy into every workgroup's LDS takes 2-3 us, so
// short rows, whose direct form runs at the same rate, need many (us, direct / table):
// F = 512 2640 rows 4.9 / 5.8, 8192 8.0 / 8.0, 20000 14.2 / 13.2; F = 1024 2640 6.7 / 7.5,
// 8192 12.3 / 11.4; F = 2048 2640 9.4 / 10.3, 8192 21.9 / 19.2; F = 3584 800 7.5 / 7.6, 1043 8.5 /
// 9.6 (a second round of 1024 rows), 2640 14.1 / 13.4; F = 7168 128 4.7 / 5.5, 300 7.1 / 6.2;
// F = 14336 6.8 / 7.7 and 10.8 / 9.0.  Four waves to every row took 15.7 us at 8192 x 512
// directly and 16.4 by the table, 17.0 and 17.5 at 8192 x 1024.
template <int FMT, int ROUND>
hipError_t launch_sq_fmt(const SwigluQuantArgs& a, hipStream_t st) {
    const int nvec = a.half / 8;
    if (nvec <= 64) return launch_sq_nv<FMT, ROUND, 1, 1, 1, 1>(a, 8192, st);
    if (nvec <= 128) return launch_sq_nv<FMT, ROUND, 1, 2, 2, 1>(a, 5120, st);
    if (nvec <= 256) return launch_sq_nv<FMT, ROUND, 1, 4, 2, 2>(a, 4096, st);
    if (nvec <= 512) return launch_sq_nv<FMT, ROUND, 2, 4, 2, 4>(a, 1100, st);
    if (nvec <= 1024) return launch_sq_nv<FMT, ROUND, 4, 4, 2, 8>(a, 192, st);
    if (nvec <= 1536) return launch_sq_nv<FMT, ROUND, 6, 4, 3, 8>(a, 192, st);
    if (nvec <= 1792) return launch_sq_nv<FMT, ROUND, 7, 4, 4, 8>(a, 192, st);
    return launch_sq_nv<FMT, ROUND, 8, 4, 4, 8>(a, 192, st);
}

}  // namespace

hipError_t launch_swiglu_quant(const SwigluQuantArgs& a, int fmt, int rounding, hipStream_t st) {
    if (fmt == kFmtInt8)
        return rounding == kRoundRcpMul ? launch_sq_fmt<kFmtInt8, kRoundRcpMul>(a, st)
                                        : launch_sq_fmt<kFmtInt8, kRoundDiv>(a, st);
    return launch_sq_fmt<kFmtE4M3, kRoundDiv>(a, st);
}

}  // namespace h3q
