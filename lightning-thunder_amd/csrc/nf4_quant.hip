// NF4 blockwise quantize / dequantize kernels for gfx950 (bit-exact contract, HBM-bound).
//
// quantize  : bitsandbytes.functional.quantize_4bit(w, quant_type="nf4"), the call made at
//             thunder/transforms/quantization.py:63
// dequantize: bitsandbytes.functional.dequantize_4bit, reached through matmul_4bit from
//             thunder/transforms/quantization.py:39
//
// Data layout.  The weight is a flat row-major array of n elements.  Every lane owns 8
// consecutive elements: one 128-bit load of bf16/f16 input (two for fp32), one 32-bit word of
// packed codes, one 128-bit store of bf16/f16 output.  A quantisation block of B elements is
// therefore B/8 adjacent lanes, and the block maximum is a butterfly over those lanes.
//
// This file is compiled with -ffp-contract=off: every product and sum below is rounded once.
#include <hip/hip_fp16.h>

#include "nf4_common.h"

namespace nf4 {
namespace {

// The decision thresholds of the NF4 code (midpoints of adjacent code values) appear below as the
// exact fp32 bit patterns a C compiler produces for the literals -0.8480964004993439f ...
// 0.8614784181118011f (four of the midpoints are exact ties in fp32).
// code = number of thresholds strictly below s (NaN -> 0).
//
// [-1, 1] is cut into 32 cells of width 1/16; adjacent thresholds are at least 0.08 apart, so a cell
// holds at most one of them, and code = (thresholds below the cell) + (s > the cell's threshold).
// Both numbers of a cell are one 64-bit LDS word; 32 words are one word per bank, so a wave's reads
// never conflict.  The cell's byte offset comes out of two additions: fma(s, 0.5, 0.5 - 2^-9) clamped
// to [0, 1] (NaN and negatives 0), plus 2^15, whose last bit is 2^-8: the low mantissa bits then hold
// floor(128 s + 128) and the cell is that without its last three bits.  s = 1 may round up into word
// 32, which is the last cell once more (the words behind it only pad the mask's range).  A value within
// rounding distance of a cell boundary may land in the neighbouring cell, which gives the same code
// because no threshold is closer than 1.6e-3 to a boundary.
__device__ __constant__ const uint32_t CELL_THR[32] = {
    0x7F800000u, 0x7F800000u, 0xBF591CD9u, 0x7F800000u, 0x7F800000u, 0x7F800000u, 0xBF1C5270u, 0x7F800000u,
    0xBEEB8480u, 0x7F800000u, 0xBEADEA76u, 0x7F800000u, 0xBE703CECu, 0xBE0D38BCu, 0x7F800000u, 0xBD3A7871u,
    0x3D22FAFFu, 0x3DF64863u, 0x7F800000u, 0x3E5067E0u, 0x3E9582D4u, 0x7F800000u, 0x3EC753F9u, 0x7F800000u,
    0x3F006D03u, 0x7F800000u, 0x3F248DAFu, 0x7F800000u, 0x7F800000u, 0x3F5C89D9u, 0x7F800000u, 0x7F800000u};
__device__ __constant__ const uint32_t CELL_BASE[32] = {0, 0, 0,  1,  1,  1,  1,  2,  2,  3,  3,  4,  4,  5,  6,  6,
                                                        7, 8, 9,  9,  10, 11, 11, 12, 12, 13, 13, 14, 14, 14, 15, 15};

constexpr int CODE_CELLS = 64;

// Appends the code of s to the codes in `word`.
__device__ __forceinline__ uint32_t append_code(uint32_t word, float s, const uint2* cells) {
    const float u = __builtin_amdgcn_fmed3f(__builtin_fmaf(s, 0.5f, 0.5f - 0x1p-9f), 0.0f, 1.0f) + 0x1p15f;
    const uint2 cell = cells[(__float_as_uint(u) >> 3) & (CODE_CELLS - 1)];
    return (word << 4) + cell.y + (s > __uint_as_float(cell.x) ? 1u : 0u);
}

// 8 elements as they lie in memory
template <int DTYPE>
struct Raw8 {
    uint32_t d[DTYPE == F32 ? 8 : 4];
};

template <int DTYPE>
__device__ __forceinline__ Raw8<DTYPE> load8(const void* w, int64_t e0) {
    Raw8<DTYPE> r;
    const uint4* p = reinterpret_cast<const uint4*>(static_cast<const char*>(w) + e0 * (DTYPE == F32 ? 4 : 2));
    const uint4 a = load16_stream(p);
    r.d[0] = a.x; r.d[1] = a.y; r.d[2] = a.z; r.d[3] = a.w;
    if (DTYPE == F32) {
        const uint4 b = load16_stream(p + 1);
        r.d[4] = b.x; r.d[5] = b.y; r.d[6] = b.z; r.d[7] = b.w;
    }
    return r;
}

// the same where the array may end inside: elements at or beyond n read as 0
template <int DTYPE>
__device__ __forceinline__ Raw8<DTYPE> load8_edge(const void* w, int64_t e0, int64_t n) {
    if (e0 + 8 <= n) return load8<DTYPE>(w, e0);
    Raw8<DTYPE> r = {};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if (e0 + j >= n) continue;
        if (DTYPE == F32)
            r.d[j] = static_cast<const uint32_t*>(w)[e0 + j];
        else
            r.d[j / 2] |= (uint32_t)static_cast<const uint16_t*>(w)[e0 + j] << (16 * (j & 1));
    }
    return r;
}

template <int DTYPE>
__device__ __forceinline__ float element(const Raw8<DTYPE>& r, int j) {
    if (DTYPE == F32) return __uint_as_float(r.d[j]);
    if (DTYPE == BF16) return __uint_as_float(j & 1 ? r.d[j / 2] & 0xffff0000u : r.d[j / 2] << 16);
    return __half2float(__ushort_as_half((unsigned short)(r.d[j / 2] >> (16 * (j & 1)))));
}

template <int CTRL>
__device__ __forceinline__ float max_dpp(float m) {
    return fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m), CTRL, 0xf, 0xf, true)));
}

// Maximum over `lanes` (a power of two, 64 at most) adjacent lanes: within 16 by DPP, an operand modifier of the maximum
// itself, where a shuffle is an LDS round trip.
__device__ __forceinline__ float group_max(float m, int lanes) {
    if (lanes > 1) m = max_dpp<0xB1>(m);   // quad_perm [1, 0, 3, 2]
    if (lanes > 2) m = max_dpp<0x4E>(m);   // quad_perm [2, 3, 0, 1]
    if (lanes > 4) m = max_dpp<0x141>(m);  // row_half_mirror
    if (lanes > 8) m = max_dpp<0x140>(m);  // row_mirror
    for (int off = 16; off < lanes; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    return m;
}

// A workgroup covers Q_SLOTS consecutive spans of THREADS * 8 elements (a span holds whole
// quantisation blocks); a thread owns 8 consecutive elements of each span.
//
// Bound by HBM (the weight read once, a quarter of it written) once the loads of all spans are in flight before the first
// is used: they are taken as raw words, behind one branch for the whole workgroup, and converted afterwards.  With the
// bounds check and the conversion around each load a span waited for the one before it, and with the cells fetched by
// two ds_bpermute each span's arithmetic came on top: [28672, 8192] bf16 took
// 126 us, now 92-96 (602 MB: 6.3-6.5 TB/s).
// Spans per workgroup (same shape): 1 / 2 / 4 / 8 took 110 / 97 / 92-96 / 101 us.
// The weight is read past the last-level cache, whatever its size: it is read once, and where kernels have left the cache full of
// lines to be written back, taking it in waits for those.  Past the cache / through it, us a weight, quantising 1 GB of weights one after
// the other: [4096, 4096] bf16 13.2 / 14.8, [14336, 4096] 29.2 / 34.1, [28672, 4096] 49.7 / 55.7, just written by a copy 13.9 / 13.8, 28.1 / 28.5,
// 49.5 / 63.5; behind 512 MB of writes to another buffer 14.1 / 18.6, 30.6 / 48, 54.7 / 83.  Only the same weight over and over gains by the
// cache (12.5 / 12.6, 29.3 / 26.9, 50.2 / 47.3; [8192, 4096] 18.1 / 16.8), and a weight is quantised once.
constexpr int Q_SLOTS = 4;

template <int THREADS, int DTYPE>
__global__ __launch_bounds__(THREADS) void quantize_kernel(const void* __restrict__ w, int64_t n, int block_log2,
                                                           uint8_t* __restrict__ packed, float* __restrict__ absmax) {
    __shared__ float wave_max[Q_SLOTS][THREADS / 64];
    __shared__ uint2 cells[CODE_CELLS];
    const int tid = threadIdx.x;
    const int group = 1 << (block_log2 - 3);  // lanes per quantisation block
    const int64_t first = (int64_t)blockIdx.x * (Q_SLOTS * THREADS * 8) + tid * 8;
    const bool whole = ((int64_t)blockIdx.x + 1) * (Q_SLOTS * THREADS * 8) <= n;
    Raw8<DTYPE> raw[Q_SLOTS];
    if (whole) {
#pragma unroll
        for (int c = 0; c < Q_SLOTS; ++c) raw[c] = load8<DTYPE>(w, first + c * (THREADS * 8));
    } else {
#pragma unroll
        for (int c = 0; c < Q_SLOTS; ++c) raw[c] = load8_edge<DTYPE>(w, first + c * (THREADS * 8), n);
    }
    if (tid < CODE_CELLS)
        cells[tid] = tid < 32 ? make_uint2(CELL_THR[tid], CELL_BASE[tid]) : make_uint2(0x7F800000u, 15u);
    // all loads are waited for here: a later wait for one of them would be for the stores of the span before it as well (97 us for
    // [28672, 8192] instead of 94)
#pragma unroll
    for (int c = 0; c < Q_SLOTS; ++c)
#pragma unroll
        for (uint32_t& d : raw[c].d) asm volatile("" : "+v"(d));
    __syncthreads();
#pragma unroll
    for (int c = 0; c < Q_SLOTS; ++c) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = element<DTYPE>(raw[c], j);
        float m = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(v[j]));
        m = group_max(m, group < 64 ? group : 64);
        if (group > 64) {  // uniform branch: blocks of 1024, 2048 or 4096 elements span several waves
            if ((tid & 63) == 0) wave_max[c][tid >> 6] = m;
            __syncthreads();
            const int waves = group >> 6;
            const int w0 = (tid >> 6) & ~(waves - 1);
            for (int j = 0; j < waves; ++j) m = fmaxf(m, wave_max[c][w0 + j]);
        }
        const float inv = __fdiv_rn(1.0f, m);
        uint32_t word = 0;
#pragma unroll
        for (int j = 3; j >= 0; --j) {  // byte j: element 2j in the high half
            word = append_code(word, __fmul_rn(v[2 * j], inv), cells);
            word = append_code(word, __fmul_rn(v[2 * j + 1], inv), cells);
        }
        const int64_t e0 = first + c * (THREADS * 8);
        if (whole || e0 < n) {
            if ((tid & (group - 1)) == 0) absmax[e0 >> block_log2] = m;
            if (whole || e0 + 8 <= n) {
                reinterpret_cast<uint32_t*>(packed)[e0 / 8] = word;
            } else {
                const int64_t nbytes = (n + 1) / 2;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (e0 / 2 + j < nbytes) packed[e0 / 2 + j] = (uint8_t)(word >> (8 * j));
            }
        }
    }
}

// Two values as bf16, rounded to nearest even, in one instruction.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}

// Eight elements of output from one 32-bit word of codes.
template <bool STREAM, int OUT>
__device__ __forceinline__ void dequant8_store(uint32_t word, float s, const float* lut, void* out, int64_t e0,
                                               bool full, int64_t n) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t byte = (word >> (8 * j)) & 0xffu;
        v[2 * j] = __fmul_rn(lut[byte >> 4], s);
        v[2 * j + 1] = __fmul_rn(lut[byte & 15u], s);
    }
    if (OUT == F32) {
        float* o = reinterpret_cast<float*>(out);
        if (full) {
            store16<STREAM>(o + e0, __float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3]));
            store16<STREAM>(o + e0 + 4, __float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7]));
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (e0 + j < n) o[e0 + j] = v[j];
        }
    } else {
        uint32_t h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (OUT == BF16) {
                h[j] = pack_bf16(v[2 * j], v[2 * j + 1]);
            } else {
                // the product is rounded to fp32 first: without this a mixed-precision multiply-add would do both at once
                asm("" : "+v"(v[2 * j]), "+v"(v[2 * j + 1]));
                h[j] = (uint32_t)__half_as_ushort(__float2half_rn(v[2 * j])) |
                       (uint32_t)__half_as_ushort(__float2half_rn(v[2 * j + 1])) << 16;
            }
        }
        uint16_t* o = reinterpret_cast<uint16_t*>(out);
        if (full) {
            store16<STREAM>(o + e0, h[0], h[1], h[2], h[3]);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (e0 + j < n) o[e0 + j] = (uint16_t)(h[j / 2] >> (16 * (j & 1)));
        }
    }
}

// A workgroup covers DQ_SLOTS consecutive spans of 2048 elements; a thread owns 8 consecutive
// elements of each span, so every load and store of a wave is contiguous.  Bound by HBM, mostly by the writes.
//
// The loads of all spans are in flight before the first is used: codes first (they come from the farthest), then the
// statistics, with one branch for the whole workgroup instead of one around each load.
// 16-bit outputs are packed by one conversion per two values.
// A streamed output's (DQ_STREAM) first store waits for the last load (lm_head 213 -> 210 us; nested 215 -> 209).
// us, with a check around every load -> now: nested [28672, 8192] bf16 99 -> 95 back to back.  Statistics first: 106.
// Spans per workgroup 1 / 2 / 4 / 8: 132 / 134 / 115 / 120.
// Nested absmax: the map is copied into LDS meanwhile, so that no load waits for another.  With the map looked up in
// global memory (code -> map entry -> value, two dependent loads per span) the kernel took 175 us for that weight.
constexpr int DQ_SLOTS = 4;

// How a weight's codes are read and its output written: both through the last-level cache; codes past it; output streamed as well.
enum : int { DQ_NEAR = 0, DQ_FAR = 1, DQ_STREAM = 2 };

template <bool NESTED, int WAY, int OUT>
__global__ __launch_bounds__(256) void dequantize_kernel(const uint8_t* __restrict__ packed,
                                                         const float* __restrict__ absmax, NestedAbsmax nq,
                                                         const float* __restrict__ lut16, int64_t n, int block_log2,
                                                         void* __restrict__ out) {
    __shared__ float lut[16];
    __shared__ float map[NESTED ? 256 : 1];
    constexpr bool STREAM = WAY == DQ_STREAM;
    const int tid = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * (DQ_SLOTS * 2048) + tid * 8;
    const bool whole = ((int64_t)blockIdx.x + 1) * (DQ_SLOTS * 2048) <= n;
    const float lut_entry = lut16[tid & 15], map_entry = NESTED ? nq.map256[tid] : 0.0f;
    uint32_t word[DQ_SLOTS], q[DQ_SLOTS];
    float s[DQ_SLOTS];  // absmax, or with nested absmax the second-level value
    if (whole) {
#pragma unroll
        for (int c = 0; c < DQ_SLOTS; ++c) {
            const uint32_t* const at = reinterpret_cast<const uint32_t*>(packed) + ((first + c * 2048) >> 3);
            word[c] = WAY == DQ_NEAR ? *at : __builtin_nontemporal_load(at);
        }
    } else {
        const int64_t nbytes = (n + 1) / 2;
#pragma unroll
        for (int c = 0; c < DQ_SLOTS; ++c) {
            const int64_t e0 = first + c * 2048;
            word[c] = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (e0 / 2 + j < nbytes) word[c] |= (uint32_t)packed[e0 / 2 + j] << (8 * j);
        }
    }
#pragma unroll
    for (int c = 0; c < DQ_SLOTS; ++c) {
        // lanes past the end read the last block's statistics, which they do not use
        const int64_t e0 = first + c * 2048, blk = (whole || e0 < n ? e0 : n - 1) >> block_log2;
        if (NESTED) {
            q[c] = nq.q[blk];
            s[c] = nq.absmax2[blk >> nq.nested_log2];
        } else {
            q[c] = 0;
            s[c] = absmax[blk];
        }
    }
    if (tid < 16) lut[tid] = lut_entry;
    if (NESTED) map[tid] = map_entry;
    if (STREAM) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no store ahead of the last load
    __syncthreads();
#pragma unroll
    for (int c = 0; c < DQ_SLOTS; ++c) {
        const int64_t e0 = first + c * 2048;
        const float scale = NESTED ? __fadd_rn(__fmul_rn(map[q[c]], s[c]), nq.offset) : s[c];  // as nested_absmax
        if (whole || e0 < n) dequant8_store<STREAM, OUT>(word[c], scale, lut, out, e0, whole || e0 + 8 <= n, n);
    }
}

// offset = mean of absmax, float64 sum rounded to fp32 once: up to DQ_SUMS workgroups add a contiguous range each (absmax
// was just written and comes from the caches), and whoever needs the offset adds their sums (dq_offset below).  A thread
// adds its values in the order in which they lie; full rounds of 1024 values are loaded DQ_ROUNDS at a time.
// [28672, 8192]: 5.3 us; loaded a round at a time, with a second kernel for the offset, 11.  The same sum taken inside the quantize kernel made that kernel 16-25 us longer (float64
// registers).
constexpr int DQ_ROUNDS = 8;

__global__ __launch_bounds__(256) void dq_sum_kernel(const float* __restrict__ absmax, int64_t nblocks, int64_t per,
                                                     double* __restrict__ sums) {
    __shared__ double wave_sum[4];
    const int tid = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * per, last = min(first + per, nblocks);
    const int rounds = (int)((last - first) / 1024);
    double t = 0.0;
    const float4* p = reinterpret_cast<const float4*>(absmax + first) + tid;
    for (int r = 0; r < rounds; r += DQ_ROUNDS) {
        float4 f[DQ_ROUNDS];
#pragma unroll
        for (int c = 0; c < DQ_ROUNDS; ++c)
            if (r + c < rounds) f[c] = p[(r + c) * 256];
#pragma unroll
        for (int c = 0; c < DQ_ROUNDS; ++c)
            if (r + c < rounds) t += ((double)f[c].x + (double)f[c].y) + ((double)f[c].z + (double)f[c].w);
    }
    const int64_t i = first + (int64_t)rounds * 1024 + tid * 4;
    if (i + 4 <= last) {
        const float4 f = *reinterpret_cast<const float4*>(absmax + i);
        t += ((double)f.x + (double)f.y) + ((double)f.z + (double)f.w);
    } else {
        for (int64_t k = i; k < last; ++k) t += (double)absmax[k];
    }
    for (int off = 1; off < 64; off <<= 1) t += __shfl_xor(t, off, 64);
    if ((tid & 63) == 0) wave_sum[tid >> 6] = t;
    __syncthreads();
    if (tid == 0) sums[blockIdx.x] = (wave_sum[0] + wave_sum[1]) + (wave_sum[2] + wave_sum[3]);
}

__device__ __constant__ const uint32_t NF4_CODE_BITS[16] = {
    0xBF800000u, 0xBF3239B1u, 0xBF066B30u, 0xBECA32A0u, 0xBE91A24Du, 0xBE3D353Fu, 0xBDBA7871u, 0x00000000u,
    0x3DA2FAFFu, 0x3E24CAE3u, 0x3E7C04DDu, 0x3EAD033Au, 0x3EE1A4B8u, 0x3F1007ABu, 0x3F3913B3u, 0x3F800000u};
// What the offset of a compressed absmax comes from and where it and the two tables that a double-quantised weight
// carries go (the tables NULL: not wanted).  `sums` NULL: the offset is `value` and nothing is written.
struct DqOffset {
    const double* sums;
    float* out;
    float* map_out;
    float* code_out;
    int count;
    float value;
};

// Adds the workgroups' sums, in the same order in every workgroup: butterflies over 64 of them, then those one by one.
template <int THREADS>
__device__ __forceinline__ void dq_wave_sums(const DqOffset& o, double* wave_sum) {
    const int tid = threadIdx.x;
    if (tid >= DQ_SUMS) return;
    constexpr int EACH = THREADS < DQ_SUMS ? DQ_SUMS / THREADS : 1;
    double t[EACH];
#pragma unroll
    for (int i = 0; i < EACH; ++i) t[i] = tid + i * THREADS < o.count ? o.sums[tid + i * THREADS] : 0.0;
    for (int off = 1; off < 64; off <<= 1)
#pragma unroll
        for (int i = 0; i < EACH; ++i) t[i] += __shfl_xor(t[i], off, 64);
#pragma unroll
    for (int i = 0; i < EACH; ++i)
        if ((tid & 63) == 0) wave_sum[(tid + i * THREADS) >> 6] = t[i];
}

__device__ __forceinline__ float dq_offset(const double* wave_sum, int64_t nblocks) {
    double t = wave_sum[0];
#pragma unroll
    for (int j = 1; j < DQ_SUMS / 64; ++j) t += wave_sum[j];
    return (float)(t / (double)nblocks);
}

// r = absmax - offset; absmax2 = max|r| over a nested block; then the nearest entry of the 256-entry map (lowest index on
// ties) for every r * (1/absmax2).  A lane owns four consecutive values (one 128-bit load, one 32-bit word of codes), a
// nested block is a power of two of adjacent lanes.
//
// The nearest entry of an ascending map is found by bisection: rounded distances fl(s - map[j]) fall towards s from
// either side (rounding is monotonic), so the minimum lies at the last entry <= s or the first one > s.  Equal rounded
// distances are settled as the scan over all entries would: the left candidate wins a tie, and from there the index
// goes down while the distance stays the same.  A map that is not ascending and finite takes that scan.  The
// bisection walks a tree in level order (node n's children are 2n and 2n + 1), in which a level's entries lie side by
// side: the upper seven levels read without bank conflicts, and a step is a compare, an add with its carry and a shift.
// 11 LDS reads per value instead of 256 reads, subtractions and compares (93 us for the 3.7 M values of [28672, 8192]).
//
// The offset is added up by every workgroup itself from the DQ_SUMS partial sums (4 KB from a cache), which saves a launch
// between the sums and this kernel; the first workgroup writes it and the tables out.  DQ_SPANS spans of THREADS * 4
// values per workgroup, so that the map, its check and the offset are paid once for all of them and the values' loads are
// in flight meanwhile, and the searches of DQ_SPANS * 4 values go down their tree together: [28672, 8192] 14 us (15.6 with
// four spans); [4096, 4096] 6 us, where a search after the other took 8.6.
constexpr int DQ_SPANS = 2;

template <int THREADS>
__global__ __launch_bounds__(THREADS) void dq_compress_kernel(const float* __restrict__ absmax, int64_t nblocks,
                                                              int nested_log2, const float* __restrict__ map256,
                                                              DqOffset o, uint8_t* __restrict__ q,
                                                              float* __restrict__ absmax2) {
    __shared__ float map[256];
    __shared__ float tree[256];
    __shared__ float wave_max[DQ_SPANS][THREADS / 64];
    __shared__ double wave_sum[DQ_SUMS / 64];
    __shared__ int wave_zero[4], wave_rising[4];
    const int tid = threadIdx.x;
    const int64_t first = ((int64_t)blockIdx.x * (DQ_SPANS * THREADS) + tid) * 4;
    float v[DQ_SPANS][4];
    if (((int64_t)blockIdx.x + 1) * (DQ_SPANS * THREADS * 4) <= nblocks) {
#pragma unroll
        for (int c = 0; c < DQ_SPANS; ++c) {
            const float4 f = *reinterpret_cast<const float4*>(absmax + first + c * (THREADS * 4));
            v[c][0] = f.x; v[c][1] = f.y; v[c][2] = f.z; v[c][3] = f.w;
        }
    } else {
#pragma unroll
        for (int c = 0; c < DQ_SPANS; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int64_t i = first + c * (THREADS * 4) + k;
                v[c][k] = i < nblocks ? absmax[i] : 0.0f;
            }
    }
    if (tid < 256) {  // whole waves
        const int node = max(tid, 1);  // node n of level l is entry (2 (n - 2^l) + 1) 2^(7 - l) - 1
        const float entry = map256[tid], next = map256[min(tid + 1, 255)];
        tree[tid] = map256[((2 * node + 1) << (7 - (31 - __clz(node)))) - 257];
        map[tid] = entry;
        const uint64_t zeros = __ballot(entry == 0.0f);
        const bool rising = entry <= next && (isfinite(entry) || (tid != 0 && tid != 255));
        const bool all_rising = __ballot(rising) == ~0ull;
        if ((tid & 63) == 0) {
            wave_zero[tid >> 6] = zeros ? tid + __ffsll((unsigned long long)zeros) - 1 : 256;
            wave_rising[tid >> 6] = all_rising;
        }
    }
    if (o.sums) dq_wave_sums<THREADS>(o, wave_sum);
    __syncthreads();
    const bool ascending = wave_rising[0] & wave_rising[1] & wave_rising[2] & wave_rising[3];
    // the map may hold no 0.0: then an all-zero block stores code 0
    const int first_zero = min(min(wave_zero[0], wave_zero[1]), min(wave_zero[2], wave_zero[3]));
    const int zero = first_zero == 256 ? 0 : first_zero;
    const float offset = o.sums ? dq_offset(wave_sum, nblocks) : o.value;
    if (o.sums && blockIdx.x == 0) {
        if (tid == 0) *o.out = offset;
        if (o.map_out && tid < 256) o.map_out[tid] = map[tid];
        if (o.code_out && tid < 16) o.code_out[tid] = __uint_as_float(NF4_CODE_BITS[tid]);
    }

    const int group = 1 << (nested_log2 - 2);  // lanes per nested block
    float m[DQ_SPANS];
#pragma unroll
    for (int c = 0; c < DQ_SPANS; ++c) {
        const int64_t i0 = first + c * (THREADS * 4);
        m[c] = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[c][k] = __fsub_rn(v[c][k], offset);
            if (i0 + k < nblocks) m[c] = fmaxf(m[c], fabsf(v[c][k]));
        }
        m[c] = group_max(m[c], group < 64 ? group : 64);
        if (group > 64) {  // uniform branch: the nested block spans several waves
            if ((tid & 63) == 0) wave_max[c][tid >> 6] = m[c];
            __syncthreads();
            const int waves = group >> 6, w0 = (tid >> 6) & ~(waves - 1);
            for (int j = 0; j < waves; ++j) m[c] = fmaxf(m[c], wave_max[c][w0 + j]);
        }
        if (i0 < nblocks && (tid & (group - 1)) == 0) absmax2[i0 >> nested_log2] = m[c];
        const float inv = __fdiv_rn(1.0f, m[c]);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[c][k] = __fmul_rn(v[c][k], inv);
    }

    int best[DQ_SPANS][4] = {};
    if (ascending) {  // the same for the whole workgroup
        // entries <= s (255 at most; 0 for NaN), the searches of all values side by side: each level is an LDS round trip
#pragma unroll
        for (int c = 0; c < DQ_SPANS; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) best[c][k] = 1;
#pragma unroll
        for (int level = 0; level < 8; ++level)
#pragma unroll
            for (int c = 0; c < DQ_SPANS; ++c)
#pragma unroll
                for (int k = 0; k < 4; ++k) best[c][k] = 2 * best[c][k] + (tree[best[c][k]] <= v[c][k] ? 1 : 0);
#pragma unroll
        for (int c = 0; c < DQ_SPANS; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) best[c][k] -= 256;
        float left[DQ_SPANS][4];
#pragma unroll
        for (int c = 0; c < DQ_SPANS; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int pos = best[c][k], before = pos > 0 ? pos - 1 : 0;
                const float right = fabsf(__fsub_rn(v[c][k], map[pos]));
                left[c][k] = fabsf(__fsub_rn(v[c][k], map[before]));
                if (left[c][k] <= right) best[c][k] = before;
                else left[c][k] = -1.0f;  // no distance: nothing further to the left is as near
            }
        bool tied = false;  // an entry further to the left is as near: duplicates, or entries closer than fp32 tells apart
#pragma unroll
        for (int c = 0; c < DQ_SPANS; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                tied |= best[c][k] > 0 && fabsf(__fsub_rn(v[c][k], map[max(best[c][k], 1) - 1])) == left[c][k];
        if (tied) {
#pragma unroll
            for (int c = 0; c < DQ_SPANS; ++c)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    while (best[c][k] > 0 && fabsf(__fsub_rn(v[c][k], map[best[c][k] - 1])) == left[c][k]) --best[c][k];
        }
    } else {
#pragma unroll
        for (int c = 0; c < DQ_SPANS; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float bestd = INFINITY;
                for (int j = 0; j < 256; ++j) {
                    const float d = fabsf(__fsub_rn(v[c][k], map[j]));
                    if (d < bestd) {
                        bestd = d;
                        best[c][k] = j;
                    }
                }
            }
    }

#pragma unroll
    for (int c = 0; c < DQ_SPANS; ++c) {
        const int64_t i0 = first + c * (THREADS * 4);
        uint32_t code[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)  // infinity and NaN: no distance is below infinity, the code stays 0
            code[k] = m[c] == 0.0f ? zero : isfinite(v[c][k]) ? best[c][k] : 0;
        if (i0 + 4 <= nblocks) {
            *reinterpret_cast<uint32_t*>(q + i0) = code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (i0 + k < nblocks) q[i0 + k] = (uint8_t)code[k];
        }
    }
}

__global__ __launch_bounds__(256) void dq_reconstruct_kernel(NestedAbsmax nq, int64_t nblocks,
                                                             float* __restrict__ absmax) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < nblocks) absmax[i] = nested_absmax(nq, i);
}

}  // namespace

namespace {

template <int DTYPE>
void enqueue_quantize(const void* w, int64_t n, int block_log2, uint8_t* packed, float* absmax, hipStream_t stream) {
    const int threads = block_log2 == 12 ? 512 : 256;  // a span holds a whole block
    const int64_t per = (int64_t)threads * 8 * Q_SLOTS;
    const dim3 grid((unsigned)((n + per - 1) / per));
    if (threads == 512)
        hipLaunchKernelGGL((quantize_kernel<512, DTYPE>), grid, dim3(512), 0, stream, w, n, block_log2, packed, absmax);
    else
        hipLaunchKernelGGL((quantize_kernel<256, DTYPE>), grid, dim3(256), 0, stream, w, n, block_log2, packed, absmax);
}

hipError_t enqueue_compress(const float* absmax, int64_t nblocks, int nested_log2, const float* map256, const DqOffset& o,
                            uint8_t* q, float* absmax2, hipStream_t stream) {
    // a span holds whole nested blocks: 1024 values, or 4096 for the two largest nested block sizes
    const int threads = nested_log2 <= 10 ? 256 : 1024;
    const int64_t per = (int64_t)threads * 4 * DQ_SPANS;
    const dim3 grid((unsigned)((nblocks + per - 1) / per));
    if (threads == 256)
        hipLaunchKernelGGL(dq_compress_kernel<256>, grid, dim3(256), 0, stream, absmax, nblocks, nested_log2, map256, o, q, absmax2);
    else
        hipLaunchKernelGGL(dq_compress_kernel<1024>, grid, dim3(1024), 0, stream, absmax, nblocks, nested_log2, map256, o, q, absmax2);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_quantize(const void* w, int w_dtype, int64_t n, int block_log2, uint8_t* packed, float* absmax,
                           hipStream_t stream) {
    if (n == 0) return hipSuccess;
    if (w_dtype == BF16)
        enqueue_quantize<BF16>(w, n, block_log2, packed, absmax, stream);
    else if (w_dtype == F16)
        enqueue_quantize<F16>(w, n, block_log2, packed, absmax, stream);
    else
        enqueue_quantize<F32>(w, n, block_log2, packed, absmax, stream);
    return hipGetLastError();
}

hipError_t launch_dq_statistics(const float* absmax, int64_t nblocks, int nested_log2, const float* map256, double* sums,
                                float* offset, uint8_t* q, float* absmax2, float* map_out, float* code_out, hipStream_t stream) {
    if (nblocks == 0) return hipSuccess;
    // a workgroup of the sum takes at least 4096 values
    const int64_t per = max((int64_t)4096, ((nblocks + DQ_SUMS - 1) / DQ_SUMS + 3) & ~(int64_t)3);
    const int count = (int)((nblocks + per - 1) / per);
    hipLaunchKernelGGL(dq_sum_kernel, dim3((unsigned)count), dim3(256), 0, stream, absmax, nblocks, per, sums);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return enqueue_compress(absmax, nblocks, nested_log2, map256, {sums, offset, map_out, code_out, count, 0.0f}, q, absmax2, stream);
}

namespace {

template <int WAY, int OUT>
void enqueue_dequantize(const uint8_t* packed, const float* absmax, const NestedAbsmax& nested, const float* lut16,
                        int64_t n, int block_log2, void* out, hipStream_t stream) {
    const dim3 grid((unsigned)((n + 2048 * DQ_SLOTS - 1) / (2048 * DQ_SLOTS))), threads(256);
    if (nested.q)
        hipLaunchKernelGGL((dequantize_kernel<true, WAY, OUT>), grid, threads, 0, stream, packed, absmax, nested, lut16, n, block_log2, out);
    else
        hipLaunchKernelGGL((dequantize_kernel<false, WAY, OUT>), grid, threads, 0, stream, packed, absmax, nested, lut16, n, block_log2, out);
}

}  // namespace

hipError_t launch_dequantize(const uint8_t* packed, const float* absmax, const NestedAbsmax& nested,
                             const float* lut16, int64_t n, int block_log2, void* out, int out_dtype,
                             hipStream_t stream) {
    if (n == 0) return hipSuccess;
    // An output that fits in the 256 MB last-level cache is written with ordinary stores, so that the
    // GEMM that usually follows finds it there; a larger one cannot stay anyway and is streamed
    // (non-temporal stores: 20 % faster on their own, 5 % slower for that GEMM).
    // Codes are read through that cache where two or three such weights fit it with their outputs, and may be found there again.  Through it /
    // past it, us a weight to bf16, the same one over and over; 0.4 to 0.5 GB of weights in turn; behind 512 MB of writes: [4096, 4096] 8.7 / 10.1,
    // 10.9 / 10.0, 14.2 / 14.0; [8192, 4096], 64 MB, 13.5 / 16.1, 18.4 / 17.5, 23.2 / 21.1; [10240, 4096] 16.7 / 18.7, 21.9 / 20.7, 27.6 / 25.2;
    // [14336, 4096] 22.8 / 25.0, 29.4 / 28.0, 35.6 / 32.0; [22528, 4096] 34.6 / 36.7, 43.5 / 41.6, 52.2 / 46.6: 3 us against 1 up to 64 MB, 2 against
    // 1 to 6 beyond.  (Three in turn: [8192, 4096] 14.0 / 16.8, [14336, 4096] 26.6 / 25.5.)
    const int64_t out_bytes = n * (out_dtype == F32 ? 4 : 2);
    const int way = out_bytes > ((int64_t)192 << 20) ? DQ_STREAM : out_bytes > ((int64_t)64 << 20) ? DQ_FAR : DQ_NEAR;
    const auto pick = [way](auto near, auto far, auto stream_out) { return way == DQ_NEAR ? near : way == DQ_FAR ? far : stream_out; };
    const auto enqueue = out_dtype == F32    ? pick(enqueue_dequantize<DQ_NEAR, F32>, enqueue_dequantize<DQ_FAR, F32>, enqueue_dequantize<DQ_STREAM, F32>)
                         : out_dtype == BF16 ? pick(enqueue_dequantize<DQ_NEAR, BF16>, enqueue_dequantize<DQ_FAR, BF16>, enqueue_dequantize<DQ_STREAM, BF16>)
                                             : pick(enqueue_dequantize<DQ_NEAR, F16>, enqueue_dequantize<DQ_FAR, F16>, enqueue_dequantize<DQ_STREAM, F16>);
    enqueue(packed, absmax, nested, lut16, n, block_log2, out, stream);
    return hipGetLastError();
}

hipError_t launch_dq_compress(const float* absmax, int64_t nblocks, int nested_log2, const float* map256,
                              float offset, uint8_t* q, float* absmax2, hipStream_t stream) {
    if (nblocks == 0) return hipSuccess;
    return enqueue_compress(absmax, nblocks, nested_log2, map256, {nullptr, nullptr, nullptr, nullptr, 0, offset}, q, absmax2, stream);
}

hipError_t launch_dq_reconstruct(const NestedAbsmax& nested, int64_t nblocks, float* absmax, hipStream_t stream) {
    if (nblocks == 0) return hipSuccess;
    const int64_t grid = (nblocks + 255) / 256;
    hipLaunchKernelGGL(dq_reconstruct_kernel, dim3((unsigned)grid), dim3(256), 0, stream, nested, nblocks, absmax);
    return hipGetLastError();
}

}  // namespace nf4
