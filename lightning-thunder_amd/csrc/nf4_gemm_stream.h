// Fused NF4 matmul for bf16 or fp16 x of up to 128 rows, and more while the chip is filled once at most, exact weights (the
// kernel; launcher, time model and rules: nf4_gemm_stream.hip).
//
// Replaces the dequantize_4bit + F.linear route of bitsandbytes.matmul_4bit (MatMul4Bit.forward, reached from
// thunder/transforms/quantization.py:39) between a decode step and a prompt.  What such a call has to move is the weight,
// so the kernel is built around that stream: one workgroup of 8 consumer and 4 producer waves per CU.
//
// * Consumer wave w owns 32 weight rows and a share of K: WN waves side by side cover the R = 32 WN rows of the tile, WK =
//   8 / WN groups of them share K (and `splits` workgroups share it further), dealt in units of 256 k so that what a tile's
//   waves read at one time is one stretch of a row.  Lane l holds weight row l % 32; its 16 bytes of a 64-k step are 32 codes
//   (k = 32 (l / 32) ..), each dword of which becomes one B fragment of v_mfma_f32_32x32x16: rne(lut16[code] * absmax) in
//   x's type, the value nf4hip_dequantize writes.  The lookup is one ds_read_b64 per byte of codes in a table of fp32 pairs.
// * Codes go from memory into the wave's own 4 KB slot of LDS and from there into registers, a set of four steps at a time.
//   Loaded into registers directly, in the layout the fragments need (32 rows x 32 bytes per request instead of 8 rows x
//   128), they cost the CU's address unit twice the time, and a wave that waits to place a request multiplies nothing:
//   [8192, 28672], M = 16, fp32 absmax 51 us then, 45 this way, 38 with a set's requests placed one behind each slice and K
//   dealt in units instead of ranges.
// * Producer wave p moves a quarter of x, memory -> LDS, three stages.  Requests of one wave complete in order, so a wave
//   that fetched both x (from L2) and codes (from HBM) would turn every wait for x into one for the codes before it.
// * One barrier per stage of x.  The WK partial sums of a tile meet in LDS, in a fixed order; with splits they meet in
//   the workspace (protocol of nf4_common.h), again in a fixed order.
//
// What bounds it (counters, [8192, 28672], M = 16; share of the kernel's cycles): no unit is busy throughout -- address unit 60 % (in 27 % held
// by the cache), VALU 48 %, LDS 34 %, MFMA 20 %; [14336, 4096], M = 64: 39, 25, 20, 16 %; [4096, 14336], M = 512 (128 x 256 tiles): 44, 36, 38,
// 47 %.  Two consumer waves per SIMD that meet at a barrier add up the times of fetch (~12 us of the first), expansion (~12) and
// multiplication with its LDS reads (~16; the parts from variants with the others taken out of an earlier form) more than they overlap
// them.  Book (64 KB), code slots (32 KB) and x leave no LDS for more waves.  With M <= 16 half of every MFMA and x read is duplicate rows.
// Measured against what served these calls before (graph replay, cold weights, us): M = 32 [4096, 4096] 18.0 -> 9.7,
// [14336, 4096] 24.7 -> 14.5, [28672, 4096] 33.2 -> 21.4, lm_head [128256, 4096] 112.7 -> 77.8; M = 64 [4096, 4096] 18.7 -> 14.2,
// [14336, 4096] 27.3 -> 20.0, lm_head 124.8 -> 98.7; fp16 (dequantize + library GEMM before) [14336, 4096] M = 4 47 -> 13.
#pragma once

#include "nf4_gemv.h"

namespace nf4 {
namespace stream {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr int CONSUMERS = 8, PRODUCERS = 4;
constexpr int THREADS = 64 * (CONSUMERS + PRODUCERS);
constexpr int BOOK_BYTES = 256 * 256;  // byte -> (fp32, fp32) of its two codes, 32 copies: 256 B per byte value
constexpr int STEP_K = 64;

template <bool NESTED, int BM, int WN>
struct Shape {
    static constexpr int WK = CONSUMERS / WN;
    static constexpr int R = 32 * WN;
    static constexpr int TI = (BM + 31) / 32;
    static constexpr int STEP_BYTES = BM * STEP_K * 2;  // x of one step of one k group
    static constexpr int LIMIT = 16 * 1024;
    // k steps per stage
    static constexpr int SPS = 4 * WK * STEP_BYTES <= LIMIT ? 4 : 2 * WK * STEP_BYTES <= LIMIT ? 2 : 1;
    static constexpr int STAGE_BYTES = WK * SPS * STEP_BYTES;
    static constexpr int CHUNKS = STAGE_BYTES / 1024;
    static constexpr int XL = CHUNKS / PRODUCERS;  // LDS-direct loads per producer and stage
    static constexpr int CODES = BOOK_BYTES + 3 * STAGE_BYTES;  // per consumer: 32 rows x 128 bytes of codes (four steps)
    static constexpr int SCALES = CODES + CONSUMERS * 4096;     // per consumer: 32 rows x 4 absmax (nested: their 8-bit codes)
    static constexpr int SCALE_BYTES = NESTED ? 128 : 512;
    static constexpr int MAP = SCALES + CONSUMERS * SCALE_BYTES;
    static constexpr int SMEM_BYTES = MAP + (NESTED ? 1024 : 0);
    static constexpr bool FITS = SMEM_BYTES <= 160 * 1024;
    static_assert(!FITS || (WK - 1) * WN * TI * 4096 <= MAP - BOOK_BYTES, "partial sums of the k groups");
};

__device__ __forceinline__ float2_t lds_f32x2(uint32_t addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) float2_t*>(addr);
}
__device__ __forceinline__ float lds_f32(uint32_t addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) float*>(addr);
}
__device__ __forceinline__ u32x4v lds_u128(uint32_t addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) u32x4v*>(addr);
}

// Codes and scales of four k steps of one weight row
template <bool NESTED, bool ABS4>
struct CodeSet {
    u32x4v w[4];
    float s[4];
    // nested absmax, from which s is made: 8-bit codes (four in a dword with ABS4) and second-level absmax
    uint32_t q[NESTED ? (ABS4 ? 1 : 4) : 1];
    float second[NESTED ? (ABS4 ? 1 : 4) : 1];
};

#if defined(__HIP_DEVICE_COMPILE__)
// four book reads of one dword of codes ...
struct Pairs {
    float2_t v[4];
};
__device__ __forceinline__ Pairs look_up(uint32_t d, uint32_t book_lane) {
    Pairs p;
#pragma unroll
    for (int c = 0; c < 4; ++c) p.v[c] = lds_f32x2(__builtin_amdgcn_perm(d, book_lane, 0x0c0c0400u | ((uint32_t)c << 8)));
    return p;
}
// ... scaled and rounded: one B fragment
template <bool F16>
__device__ __forceinline__ u32x4v scale_round(const Pairs& p, float scale) {
    u32x4v o;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float2_t f = {__fmul_rn(p.v[c].x, scale), __fmul_rn(p.v[c].y, scale)};
        o[c] = F16 ? __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2_t))
                   : __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
    }
    return o;
}

template <bool F16>
__device__ __forceinline__ f32x16 mfma(u32x4v a, u32x4v b, f32x16 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
#endif

// ABS4: blocksize 64 and K % 256 == 0, so the four absmax of a code set are one aligned 16-byte (nested: 4-byte) load.
template <bool F16, bool NESTED, bool ABS4, int BM, int WN>
__global__ __launch_bounds__(THREADS) void stream_kernel(MatmulArgs a, int splits, int per, int extra, uint32_t* counters,
                                                           float* partials) {
#if defined(__HIP_DEVICE_COMPILE__)
    using T = Shape<NESTED, BM, WN>;
    constexpr int WK = T::WK, R = T::R, TI = T::TI, SPS = T::SPS;
    extern __shared__ __attribute__((aligned(4096))) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * R, m0 = blockIdx.z * BM;
    const int tile = blockIdx.z * gridDim.x + blockIdx.x;
    const int ksteps = a.K / STEP_K;
    // K in units of four steps, dealt to the k groups of all splits in turn: what a tile's waves read at one time lies next to
    // each other in memory.  Every group has `per` units, the first `extra` one more.
    const int units = (ksteps + 3) >> 2, groups = splits * WK;
    auto count_of = [&](int g) {  // k steps of group g of this workgroup
        const int all = (int)blockIdx.y * WK + g;
        const int n = per + (all < extra ? 1 : 0);
        const bool has_last = all == (extra ? extra : groups) - 1;
        return 4 * n - (has_last ? 4 * units - ksteps : 0);
    };
    int longest = 0;
#pragma unroll
    for (int g = 0; g < WK; ++g) longest = max(longest, count_of(g));
    const int stages = (longest + SPS - 1) / SPS;

    if (wave >= CONSUMERS) {
        // ---- producer: chunk c = 8 rows x 128 bytes of x of (group, step of the stage, row octet).  Row rr of a chunk sits
        // in 128-byte slot rr ^ (c & 1), its 16-byte piece p at position p ^ rr: the lanes that a 128-bit fragment read
        // serves together hit different banks.
        const int p = wave - CONSUMERS;
        const __amdgpu_buffer_rsrc_t xrsrc =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.x), 0, (int)(uint32_t)((int64_t)a.M * a.K * 2), 0x00020000);
        uint32_t xoff[T::XL];
        int group[T::XL], last[T::XL], sub[T::XL];
#pragma unroll
        for (int i = 0; i < T::XL; ++i) {
            const int c = p + PRODUCERS * i;
            const int octet = c % (BM / 8), js = c / (BM / 8);
            const int g = js / SPS;
            const int rr = (lane >> 3) ^ (c & 1);
            const int row = min(m0 + octet * 8 + rr, a.M - 1);
            xoff[i] = (uint32_t)row * (uint32_t)(a.K * 2) + (uint32_t)(((lane & 7) ^ rr) << 4);
            sub[i] = js % SPS;
            group[i] = (int)blockIdx.y * WK + g;
            last[i] = max(count_of(g) - 1, 0);  // steps past a group's end repeat its last one and are not used
        }
        auto load_stage = [&](int t, int slot) {
#pragma unroll
            for (int i = 0; i < T::XL; ++i) {
                const int s = min(t * SPS + sub[i], last[i]);  // of the group
                const int step = min((group[i] + (s >> 2) * groups) * 4 + (s & 3), ksteps - 1);
                const uint32_t lds = BOOK_BYTES + slot * T::STAGE_BYTES + (p + PRODUCERS * i) * 1024;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(xrsrc, (lds_void_ptr)(uintptr_t)lds, 16, xoff[i], step * (STEP_K * 2), 0, 0);
            }
        };
        // Barrier t stands before the last slice of stage t: the stage's fragments have all been read by then, so its slot
        // takes stage t + 3, and stage t + 1 has to be there.
        for (int t = 0; t < 3; ++t)
            if (t < stages) load_stage(t, t);
        if (stages > 2)
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * T::XL) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        int slot = 0;
        for (int t = 0; t < stages; ++t) {
            if (t + 2 < stages)
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(T::XL) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            if (t + 3 < stages) load_stage(t + 3, slot);
            slot = slot == 2 ? 0 : slot + 1;
        }
        return;
    }

    // ---- consumer ----
    const int kg = wave / WN, ng = wave % WN;
    const int count = count_of(kg);
    const int unit0 = (int)blockIdx.y * WK + kg;  // set u is unit unit0 + u * groups
    const int rows = min(R, a.N - n0);
    const int row = min(ng * 32 + (lane & 31), rows - 1);  // inside the tile
    // buffers that begin at the tile's first row and end with its last: offsets fit 32 bits, and a request with an offset
    // past the end (a code set that does not exist) returns zeros without touching memory
    const uint32_t row_codes = (uint32_t)a.K / 2;
    const uint32_t row_blocks = (uint32_t)a.K >> a.block_log2;
    const __amdgpu_buffer_rsrc_t crsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(a.packed) + (int64_t)n0 * row_codes, 0, (int)(rows * row_codes), 0x00020000);
    const void* abs_base = NESTED ? (const void*)(a.nested.q + (int64_t)n0 * row_blocks) : (const void*)(a.absmax + (int64_t)n0 * row_blocks);
    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(abs_base), 0, (int)(rows * row_blocks * (NESTED ? 1 : 4)), 0x00020000);
    const __amdgpu_buffer_rsrc_t a2rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(NESTED ? a.nested.absmax2 : a.lut16), 0,
        NESTED ? (int)((((uint32_t)a.N * row_blocks - 1) >> a.nested.nested_log2) * 4 + 4) : 0, 0x00020000);

    const float second = a.lut16[tid >> 5];
    const float map_entry = NESTED ? a.nested.map256[tid & 255] : 0.0f;

    // Codes: request i of a set moves rows 8 i .. + 7 of this wave, 128 bytes each, into its slot (laid out as x's chunks).
    uint32_t code_off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int rr = (lane >> 3) ^ (i & 1);
        code_off[i] = (uint32_t)min(ng * 32 + 8 * i + rr, rows - 1) * row_codes + (uint32_t)(((lane & 7) ^ rr) << 4);
    }
    const uint32_t code_slot = T::CODES + wave * 4096;
    auto fetch_codes = [&](int u, int i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(crsrc, (lds_void_ptr)(uintptr_t)(code_slot + i * 1024), 16, code_off[i] + (uint32_t)(unit0 + u * groups) * 128u, 0, 0, 2);
    };
    const uint32_t blk0 = (uint32_t)row * row_blocks;
    // Scales: four absmax of each of the 32 rows
    const uint32_t scale_slot = T::SCALES + wave * T::SCALE_BYTES;
    auto fetch_scales = [&](int u) {
        const uint32_t step = (uint32_t)(unit0 + u * groups) * 4u;
        if constexpr (ABS4) {
            if (lane < 32) {
                const uint32_t b = blk0 + step;
                if constexpr (NESTED)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(arsrc, (lds_void_ptr)(uintptr_t)scale_slot, 4, b, 0, 0, 0);
                else
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(arsrc, (lds_void_ptr)(uintptr_t)scale_slot, 16, b * 4u, 0, 0, 0);
            }
        } else if constexpr (!NESTED) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {  // lane: row l / 4, the absmax of one step
                const uint32_t r = (uint32_t)min(ng * 32 + 16 * i + (lane >> 2), rows - 1);
                const uint32_t b = r * row_blocks + ((step + (lane & 3)) * STEP_K >> a.block_log2);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(arsrc, (lds_void_ptr)(uintptr_t)(scale_slot + i * 256), 4, b * 4u, 0, 0, 0);
            }
        }
    };
    const uint32_t code_read = code_slot + ((lane & 31) >> 3) * 1024 + (((lane & 7) ^ ((lane >> 3) & 1)) << 7);
    using Set = CodeSet<NESTED, ABS4>;
    // A set out of its slot, all landed
    auto read_set = [&](Set& c) {
#pragma unroll
        for (int j = 0; j < 4; ++j) c.w[j] = lds_u128(code_read + (((2 * j + (lane >> 5)) ^ (lane & 7)) << 4));
        if constexpr (!NESTED) {
            const float4_t v = __builtin_bit_cast(float4_t, lds_u128(scale_slot + (lane & 31) * 16));
#pragma unroll
            for (int i = 0; i < 4; ++i) c.s[i] = v[i];
        } else if constexpr (ABS4) {
            c.q[0] = __float_as_uint(lds_f32(scale_slot + (lane & 31) * 4));
        }
    };
    auto tie_scales = [&](Set& c) {  // wait for the scales read_set has asked for
        if constexpr (!NESTED)
            asm volatile("" : "+v"(c.s[0]), "+v"(c.s[1]), "+v"(c.s[2]), "+v"(c.s[3])::"memory");
        else if constexpr (ABS4)
            asm volatile("" : "+v"(c.q[0])::"memory");
    };
    // The compiler's own wait for what load_second requested belongs here, where it costs nothing: behind the next requests, some
    // of them under a branch, it would be a wait for those as well.
    auto tie_second = [&](Set& c) {
        if constexpr (NESTED) {
#pragma unroll
            for (int j = 0; j < (ABS4 ? 1 : 4); ++j) asm volatile("" : "+v"(c.second[j])::"memory");
            if constexpr (!ABS4) asm volatile("" : "+v"(c.q[0]), "+v"(c.q[ABS4 ? 0 : 1]), "+v"(c.q[ABS4 ? 0 : 2]), "+v"(c.q[ABS4 ? 0 : 3])::"memory");
        }
    };
    auto load_second = [&](Set& c, int u) {  // what a nested set reads from memory itself, requested with the set's codes
        if constexpr (NESTED && ABS4) {
            c.second[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                a2rsrc, ((((uint32_t)n0 * row_blocks + blk0 + (uint32_t)(unit0 + u * groups) * 4u) >> a.nested.nested_log2) << 2), 0, 0));
        } else if constexpr (NESTED) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t b = blk0 + (((uint32_t)(unit0 + u * groups) * 4u + i) * STEP_K >> a.block_log2);
                c.q[i] = __builtin_amdgcn_raw_buffer_load_b8(arsrc, b, 0, 0);
                c.second[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(a2rsrc, ((((uint32_t)n0 * row_blocks + b) >> a.nested.nested_log2) << 2), 0, 0));
            }
        }
    };
    auto look_up_scales = [&](Set& c) {
        if constexpr (NESTED) {
#pragma unroll
            for (int j = 0; j < 4; ++j) c.s[j] = lds_f32(T::MAP + (ABS4 ? (c.q[0] >> (8 * j)) & 255u : c.q[ABS4 ? 0 : j]) * 4);
        }
    };
    auto finish_scales = [&](Set& c) {
        if constexpr (NESTED) {
#pragma unroll
            for (int j = 0; j < 4; ++j) c.s[j] = __fadd_rn(__fmul_rn(c.s[j], c.second[ABS4 ? 0 : j]), a.nested.offset);
        }
    };

    const int nsets = (count + 3) >> 2;
    Set sa, sb;
    if (nsets > 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fetch_codes(0, i);
        fetch_scales(0);
    }
    load_second(sa, 0);
    // pair book: thread tid writes copy tid % 32 of the 16 byte values (it << 4) | (tid / 32)
#pragma unroll
    for (int it = 0; it < 16; ++it) {
        const float2_t pair = {a.lut16[it], second};
        *reinterpret_cast<__attribute__((address_space(3))) float2_t*>((uint32_t)((((it << 4) | (tid >> 5)) << 8) + ((tid & 31) << 3))) = pair;
    }
    if (NESTED && tid < 256) *reinterpret_cast<__attribute__((address_space(3))) float*>((uint32_t)(T::MAP + tid * 4)) = map_entry;

    f32x16 acc[TI];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[i][q] = 0.0f;

    const uint32_t book_lane = (lane & 31) * 8;
    // x fragment of tile i, slice s: row r = 32 i + l % 32 (l % 16 with 16 rows), piece 4 (l / 32) + s
    const int fr = lane & (BM < 32 ? 15 : 31);
    const uint32_t frag_row = (uint32_t)((fr >> 3) * 1024 + (((fr & 7) ^ ((fr >> 3) & 1)) << 7));
    uint32_t frag[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
        frag[s] = BOOK_BYTES + kg * SPS * T::STEP_BYTES + frag_row + (uint32_t)(((((lane >> 5) << 2) | s) ^ (fr & 7)) << 4);

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // set 0
    read_set(sa);
    asm volatile("" : "+v"(sa.w[0]), "+v"(sa.w[1]), "+v"(sa.w[2]), "+v"(sa.w[3])::"memory");
    tie_scales(sa);
    if (nsets > 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fetch_codes(1, i);
        fetch_scales(1);
    }
    load_second(sb, 1);
    lds_barrier();  // code book, map and x of stage 0

    uint32_t st = 0;  // offset of the current stage
    int done = 0;
    look_up_scales(sa);
    finish_scales(sa);
    float scale = sa.s[0];
    u32x4v fb = scale_round<F16>(look_up(sa.w[0][0], book_lane), scale);
    Pairs ahead = look_up(sa.w[0][1], book_lane);
    u32x4v fa[TI];
#pragma unroll
    for (int i = 0; i < TI; ++i) fa[i] = lds_u128(frag[0] + i * 4096);
    // Step j of set `cur`; nw0, nw1, next_scale: the first two dwords and the scale of the step behind it.  While slice s is
    // multiplied, the fragments of slice s + 1 and the book entries of slice s + 2 are read and those of s + 1 scaled.
    auto step = [&](const Set& cur, int j, uint32_t nw0, uint32_t nw1, const float& next_scale, auto request) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t base = st + (j % SPS) * T::STEP_BYTES;
            if (s == 3) {
                if (j % SPS == SPS - 1) {
                    // this stage's fragments have arrived (their registers are operands here), the next stage has landed
                    if constexpr (TI == 1)
                        asm volatile("s_barrier" : "+v"(fa[0])::"memory");
                    else if constexpr (TI == 2)
                        asm volatile("s_barrier" : "+v"(fa[0]), "+v"(fa[1])::"memory");
                    else
                        asm volatile("s_barrier" : "+v"(fa[0]), "+v"(fa[1]), "+v"(fa[2]), "+v"(fa[3])::"memory");
                    st = st == 2 * T::STAGE_BYTES ? 0 : st + T::STAGE_BYTES;
                }
                base = st + ((j + 1) % SPS) * T::STEP_BYTES;
            }
            u32x4v fan[TI];
#pragma unroll
            for (int i = 0; i < TI; ++i) fan[i] = lds_u128(frag[(s + 1) & 3] + base + i * 4096);
            const Pairs next = look_up(s == 0 ? cur.w[j][2] : s == 1 ? cur.w[j][3] : s == 2 ? nw0 : nw1, book_lane);
#pragma unroll
            for (int i = 0; i < TI; ++i) acc[i] = mfma<F16>(fa[i], fb, acc[i]);
            fb = scale_round<F16>(ahead, s < 3 ? scale : next_scale);
            request(s);
            ahead = next;
#pragma unroll
            for (int i = 0; i < TI; ++i) fa[i] = fan[i];
            __builtin_amdgcn_sched_barrier(0);
        }
        scale = next_scale;
        ++done;
    };
    // The four steps of set u (`cur`).  Ahead of the last one set u + 1, requested four steps ago, is read out of its slot (the
    // wait is for everything: nothing else of this wave is under way); behind its slices the slot takes set u + 2, one
    // request at a time: eight waves that issue four each at once stall, and with them the barrier, until the address unit
    // has taken them all.
    auto four = [&](Set& cur, Set& nxt, int u) {
        auto none = [](int) {};
#pragma unroll
        for (int j = 0; j < 3; ++j) step(cur, j, cur.w[j + 1][0], cur.w[j + 1][1], cur.s[j + 1], none);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        tie_second(nxt);
        read_set(nxt);
        const bool more = u + 2 < nsets;
        step(cur, 3, nxt.w[0][0], nxt.w[0][1], nxt.s[0], [&](int i) {
            if (i == 0) {  // the slot has been read
                asm volatile("" : "+v"(nxt.w[0]), "+v"(nxt.w[1]), "+v"(nxt.w[2]), "+v"(nxt.w[3])::"memory");
                tie_scales(nxt);
            }
            if (i == 1) look_up_scales(nxt);
            if (i == 2) finish_scales(nxt);
            if (more) {
                fetch_codes(u + 2, i);
                if (i == 3) fetch_scales(u + 2);
            }
        });
        load_second(cur, u + 2);
    };
    const int sets = count >> 2;
    int u = 0;
    for (; u + 2 <= sets; u += 2) {
        four(sa, sb, u);
        four(sb, sa, u + 1);
    }
    if (u < sets) four(sa, sb, u);
    if constexpr (!ABS4) {  // the last one to three steps of K
        if (u < sets) sa = sb;
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (j < (count & 3)) step(sa, j, sa.w[j + 1][0], sa.w[j + 1][1], sa.s[j + 1], [](int) {});
    }
    for (int t = done / SPS; t < stages; ++t) lds_barrier();

    // ---- the k groups of the tile meet in LDS (the stages are free), added in order by the waves of group 0
    if (WK > 1) {
        const uint32_t red = BOOK_BYTES + lane * 16;
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4_t v = {acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]};
                    *reinterpret_cast<__attribute__((address_space(3))) float4_t*>(red + ((((kg - 1) * WN + ng) * TI + i) * 4 + q) * 1024) = v;
                }
        }
        lds_barrier();
        if (kg == 0) {
#pragma unroll
            for (int g = 0; g < WK - 1; ++g)
#pragma unroll
                for (int i = 0; i < TI; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const u32x4v v = lds_u128(red + (((g * WN + ng) * TI + i) * 4 + q) * 1024);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][4 * q + e] += __uint_as_float(v[e]);
                    }
        }
    }
    if (splits > 1) {
        // this workgroup's sums in register order (coalesced); the last to arrive for the tile adds all in split order
        constexpr int SLOT = WN * TI * 16 * 64;
        float* tile_part = partials + (int64_t)tile * splits * SLOT + (ng * TI * 16) * 64 + lane;
        if (kg == 0) {
            float* mine = tile_part + (int64_t)blockIdx.y * SLOT;
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    __hip_atomic_store(mine + (i * 16 + q) * 64, acc[i][q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            publish_partials();
        }
        lds_barrier();
        typedef __attribute__((address_space(3))) uint32_t* lds_u32_ptr;
        if (tid == 0)
            *reinterpret_cast<lds_u32_ptr>(256u) = __hip_atomic_fetch_add(&counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        lds_barrier();
        acquire_partials();
        if (*reinterpret_cast<lds_u32_ptr>(256u) != (uint32_t)(splits - 1)) return;
        if (kg == 0) {
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                float sum[16];
#pragma unroll
                for (int q = 0; q < 16; ++q) sum[q] = 0.0f;
                constexpr int G = 4;  // splits whose loads are under way together
                for (int sp0 = 0; sp0 < splits; sp0 += G) {
                    float v[G][16];
#pragma unroll
                    for (int g = 0; g < G; ++g)
#pragma unroll
                        for (int q = 0; q < 16; ++q)
                            v[g][q] = __hip_atomic_load(tile_part + (int64_t)min(sp0 + g, splits - 1) * SLOT + (i * 16 + q) * 64,
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int g = 0; g < G; ++g)
                        if (sp0 + g < splits) {
#pragma unroll
                            for (int q = 0; q < 16; ++q) sum[q] += v[g][q];
                        }
                }
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[i][q] = sum[q];
            }
        }
        if (tid == 0) __hip_atomic_store(&counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (kg > 0) return;
    // acc[i][q] = out[m][n], n = lane & 31, m = 8 (q / 4) + 4 (lane / 32) + q % 4 inside the 32 x 32 tile
    const int n = n0 + ng * 32 + (lane & 31);
    if (n >= a.N) return;
    float b = 0.0f;
    if (a.bias) b = F16 ? (float)__builtin_bit_cast(_Float16, a.bias[n]) : bf16_bits_to_f32(a.bias[n]);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int q = 0; q < (BM < 32 ? 8 : 16); ++q) {
            const int m = m0 + i * 32 + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
            const float v = acc[i][q] + b;
            if (m < a.M)
                a.out[(int64_t)m * a.N + n] = F16 ? __builtin_bit_cast(uint16_t, (_Float16)v) : (uint16_t)f32_to_bf16_bits(v);
        }
#endif
}

}  // namespace stream
}  // namespace nf4
