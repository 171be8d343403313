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
// Lane c of a wave keeps cell c & 31 in two registers and every lane fetches its cell with
// ds_bpermute: 6 VALU operations per element instead of a 4-level tree of compares and selects.
// The cell index comes from fma(s, 16, 16) rounded to fp32; a value within rounding distance of a
// cell boundary may land in the neighbouring cell, which gives the same code because no threshold
// is closer than 1.6e-3 to a boundary.
__device__ __constant__ const uint32_t CELL_THR[32] = {
    0x7F800000u, 0x7F800000u, 0xBF591CD9u, 0x7F800000u, 0x7F800000u, 0x7F800000u, 0xBF1C5270u, 0x7F800000u,
    0xBEEB8480u, 0x7F800000u, 0xBEADEA76u, 0x7F800000u, 0xBE703CECu, 0xBE0D38BCu, 0x7F800000u, 0xBD3A7871u,
    0x3D22FAFFu, 0x3DF64863u, 0x7F800000u, 0x3E5067E0u, 0x3E9582D4u, 0x7F800000u, 0x3EC753F9u, 0x7F800000u,
    0x3F006D03u, 0x7F800000u, 0x3F248DAFu, 0x7F800000u, 0x7F800000u, 0x3F5C89D9u, 0x7F800000u, 0x7F800000u};
__device__ __constant__ const uint32_t CELL_BASE[32] = {0, 0, 0,  1,  1,  1,  1,  2,  2,  3,  3,  4,  4,  5,  6,  6,
                                                        7, 8, 9,  9,  10, 11, 11, 12, 12, 13, 13, 14, 14, 14, 15, 15};

struct CodeCells {
    uint32_t thr;   // CELL_THR[lane & 31]
    uint32_t base;  // CELL_BASE[lane & 31]
};

__device__ __forceinline__ uint32_t nf4_code(float s, const CodeCells& cc) {
    // NaN and negatives convert to 0, values above 31 are clamped
    const uint32_t cell = min((uint32_t)__builtin_fmaf(s, 16.0f, 16.0f), 31u);
    const float t = __uint_as_float((uint32_t)__builtin_amdgcn_ds_bpermute((int)(cell << 2), (int)cc.thr));
    const uint32_t b = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(cell << 2), (int)cc.base);
    return b + (s > t ? 1u : 0u);
}

__device__ __forceinline__ float load_elem(const void* w, int dtype, int64_t i) {
    if (dtype == BF16) return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(w)[i]);
    if (dtype == F16) return __half2float(reinterpret_cast<const __half*>(w)[i]);
    return reinterpret_cast<const float*>(w)[i];
}

// Load the 8 elements [e0, e0+8) as fp32; elements at or beyond n read as 0.
__device__ __forceinline__ void load8(const void* w, int dtype, int64_t e0, int64_t n, float v[8]) {
    if (e0 + 8 <= n) {
        if (dtype == F32) {
            const float4 a = reinterpret_cast<const float4*>(w)[e0 / 4];
            const float4 b = reinterpret_cast<const float4*>(w)[e0 / 4 + 1];
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
            v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
            const uint4 q = reinterpret_cast<const uint4*>(w)[e0 / 8];
            const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (dtype == BF16) {
                    v[2 * j] = __uint_as_float(d[j] << 16);
                    v[2 * j + 1] = __uint_as_float(d[j] & 0xffff0000u);
                } else {
                    v[2 * j] = __half2float(__ushort_as_half((unsigned short)(d[j] & 0xffffu)));
                    v[2 * j + 1] = __half2float(__ushort_as_half((unsigned short)(d[j] >> 16)));
                }
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (e0 + j < n) ? load_elem(w, dtype, e0 + j) : 0.0f;
    }
}

// A workgroup covers Q_SLOTS consecutive spans of THREADS * 8 elements (a span holds whole
// quantisation blocks); a thread owns 8 consecutive elements of each span.  The loads of all spans
// are in flight before the first reduction.
constexpr int Q_SLOTS = 4;

template <int THREADS>
__global__ __launch_bounds__(THREADS) void quantize_kernel(const void* __restrict__ w, int dtype, int64_t n,
                                                           int block_log2, uint8_t* __restrict__ packed,
                                                           float* __restrict__ absmax) {
    __shared__ float wave_max[Q_SLOTS][THREADS / 64];
    const int tid = threadIdx.x;
    const int group = 1 << (block_log2 - 3);  // lanes per quantisation block
    const CodeCells cc = {CELL_THR[tid & 31], CELL_BASE[tid & 31]};
    float v[Q_SLOTS][8];
    float m[Q_SLOTS];
#pragma unroll
    for (int c = 0; c < Q_SLOTS; ++c) {
        const int64_t e0 = (((int64_t)blockIdx.x * Q_SLOTS + c) * THREADS + tid) * 8;
        load8(w, dtype, e0, n, v[c]);
    }
    const int in_wave = group < 64 ? group : 64;
#pragma unroll
    for (int c = 0; c < Q_SLOTS; ++c) {
        float mm = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) mm = fmaxf(mm, fabsf(v[c][j]));
        // max over the lanes of one quantisation block
        for (int off = 1; off < in_wave; off <<= 1) mm = fmaxf(mm, __shfl_xor(mm, off, 64));
        m[c] = mm;
    }
    if (group > 64) {  // uniform branch: blocks of 1024, 2048 or 4096 elements span several waves
#pragma unroll
        for (int c = 0; c < Q_SLOTS; ++c)
            if ((tid & 63) == 0) wave_max[c][tid >> 6] = m[c];
        __syncthreads();
        const int waves = group >> 6;
        const int first = (tid >> 6) & ~(waves - 1);
#pragma unroll
        for (int c = 0; c < Q_SLOTS; ++c)
            for (int j = 0; j < waves; ++j) m[c] = fmaxf(m[c], wave_max[c][first + j]);
    }
#pragma unroll
    for (int c = 0; c < Q_SLOTS; ++c) {
        const int64_t e0 = (((int64_t)blockIdx.x * Q_SLOTS + c) * THREADS + tid) * 8;
        // every lane computes its codes (the cell lookup reads other lanes' registers, so no lane
        // may drop out before it); lanes past the end hold zeros and store nothing
        const float inv = __fdiv_rn(1.0f, m[c]);
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t hi = nf4_code(__fmul_rn(v[c][2 * j], inv), cc);
            const uint32_t lo = nf4_code(__fmul_rn(v[c][2 * j + 1], inv), cc);
            word |= ((hi << 4) | lo) << (8 * j);
        }
        if (e0 >= n) continue;
        if ((tid & (group - 1)) == 0) absmax[e0 >> block_log2] = m[c];
        if (e0 + 8 <= n) {
            reinterpret_cast<uint32_t*>(packed)[e0 / 8] = word;
        } else {
            const int64_t nbytes = (n + 1) / 2;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (e0 / 2 + j < nbytes) packed[e0 / 2 + j] = (uint8_t)(word >> (8 * j));
        }
    }
}

// Eight elements of output from one 32-bit word of codes.
template <bool STREAM>
__device__ __forceinline__ void dequant8_store(uint32_t word, float s, const float* lut, void* out, int out_dtype,
                                               int64_t e0, int64_t n) {
    const bool full = e0 + 8 <= n;
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t byte = (word >> (8 * j)) & 0xffu;
        v[2 * j] = __fmul_rn(lut[byte >> 4], s);
        v[2 * j + 1] = __fmul_rn(lut[byte & 15u], s);
    }
    if (out_dtype == F32) {
        float* o = reinterpret_cast<float*>(out);
        if (full) {
            store16<STREAM>(o + e0, __float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3]));
            store16<STREAM>(o + e0 + 4, __float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7]));
        } else {
            for (int j = 0; j < 8; ++j)
                if (e0 + j < n) o[e0 + j] = v[j];
        }
    } else {
        uint32_t h[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            h[j] = out_dtype == BF16 ? f32_to_bf16_bits(v[j]) : (uint32_t)__half_as_ushort(__float2half_rn(v[j]));
        uint16_t* o = reinterpret_cast<uint16_t*>(out);
        if (full) {
            store16<STREAM>(o + e0, h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
        } else {
            for (int j = 0; j < 8; ++j)
                if (e0 + j < n) o[e0 + j] = (uint16_t)h[j];
        }
    }
}

// A workgroup covers DQ_SLOTS consecutive spans of 2048 elements; a thread owns 8 consecutive
// elements of each span, so every load and store of a wave is contiguous, and the loads of all
// spans are in flight before the first store.
// Nested absmax: the 8-bit code and the second-level absmax of every span are requested together with the codes and the
// map is copied into LDS meanwhile, so that no load waits for another.  With the map looked up in global memory
// (code -> map entry -> value, two dependent loads per span) the kernel took 175 us for the 592 MB of a [28672, 8192]
// weight (3.4 TB/s); now 101 us (5.9 TB/s).
constexpr int DQ_SLOTS = 4;

template <bool NESTED, bool STREAM>
__global__ __launch_bounds__(256) void dequantize_kernel(const uint8_t* __restrict__ packed,
                                                         const float* __restrict__ absmax, NestedAbsmax nq,
                                                         const float* __restrict__ lut16, int64_t n, int block_log2,
                                                         void* __restrict__ out, int out_dtype) {
    __shared__ float lut[16];
    __shared__ float map[NESTED ? 256 : 1];
    const int tid = threadIdx.x;
    const float lut_entry = lut16[tid & 15], map_entry = NESTED ? nq.map256[tid] : 0.0f;
    uint32_t word[DQ_SLOTS], q[DQ_SLOTS];
    float s[DQ_SLOTS];  // absmax, or with nested absmax the second-level value
#pragma unroll
    for (int c = 0; c < DQ_SLOTS; ++c) {
        const int64_t e0 = (((int64_t)blockIdx.x * DQ_SLOTS + c) * 256 + tid) * 8;
        word[c] = q[c] = 0;
        s[c] = 0.0f;
        if (e0 >= n) continue;
        const int64_t blk = e0 >> block_log2;
        if (NESTED) {
            q[c] = nq.q[blk];
            s[c] = nq.absmax2[blk >> nq.nested_log2];
        } else {
            s[c] = absmax[blk];
        }
        if (e0 + 8 <= n) {
            word[c] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(packed) + e0 / 8);
        } else {
            const int64_t nbytes = (n + 1) / 2;
            for (int j = 0; j < 4; ++j)
                if (e0 / 2 + j < nbytes) word[c] |= (uint32_t)packed[e0 / 2 + j] << (8 * j);
        }
    }
    if (tid < 16) lut[tid] = lut_entry;
    if (NESTED) map[tid] = map_entry;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < DQ_SLOTS; ++c) {
        const int64_t e0 = (((int64_t)blockIdx.x * DQ_SLOTS + c) * 256 + tid) * 8;
        const float scale = NESTED ? __fadd_rn(__fmul_rn(map[q[c]], s[c]), nq.offset) : s[c];  // as nested_absmax
        if (e0 < n) dequant8_store<STREAM>(word[c], scale, lut, out, out_dtype, e0, n);
    }
}

// offset = mean of absmax, float64 sum rounded to fp32 once: up to DQ_SUMS workgroups add a contiguous range each (absmax
// was just written and comes from the caches), one adds their sums.  The second kernel also writes the two tables a
// double-quantised weight carries (NULL: not wanted), which saves their copies a launch each.  [28672, 8192]: 11 us for
// both; the same sum taken inside the quantize kernel made that kernel 16-25 us longer (float64 registers).
__global__ __launch_bounds__(256) void dq_sum_kernel(const float* __restrict__ absmax, int64_t nblocks, int64_t per,
                                                     double* __restrict__ sums) {
    __shared__ double wave_sum[4];
    const int tid = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * per, last = min(first + per, nblocks);
    double t = 0.0;
#pragma unroll 4
    for (int64_t i = first + tid * 4; i < last; i += 1024) {
        if (i + 4 <= last) {
            const float4 f = *reinterpret_cast<const float4*>(absmax + i);
            t += ((double)f.x + (double)f.y) + ((double)f.z + (double)f.w);
        } else {
            for (int64_t k = i; k < last; ++k) t += (double)absmax[k];
        }
    }
    for (int off = 1; off < 64; off <<= 1) t += __shfl_xor(t, off, 64);
    if ((tid & 63) == 0) wave_sum[tid >> 6] = t;
    __syncthreads();
    if (tid == 0) sums[blockIdx.x] = (wave_sum[0] + wave_sum[1]) + (wave_sum[2] + wave_sum[3]);
}

__device__ __constant__ const uint32_t NF4_CODE_BITS[16] = {
    0xBF800000u, 0xBF3239B1u, 0xBF066B30u, 0xBECA32A0u, 0xBE91A24Du, 0xBE3D353Fu, 0xBDBA7871u, 0x00000000u,
    0x3DA2FAFFu, 0x3E24CAE3u, 0x3E7C04DDu, 0x3EAD033Au, 0x3EE1A4B8u, 0x3F1007ABu, 0x3F3913B3u, 0x3F800000u};
__global__ __launch_bounds__(DQ_SUMS) void dq_offset_kernel(const double* __restrict__ sums, int count, int64_t nblocks,
                                                            float* __restrict__ offset, const float* __restrict__ map256,
                                                            float* __restrict__ map_out, float* __restrict__ code_out) {
    __shared__ double wave_sum[DQ_SUMS / 64];
    const int tid = threadIdx.x;
    double t = tid < count ? sums[tid] : 0.0;
    if (map_out && tid < 256) map_out[tid] = map256[tid];
    if (code_out && tid < 16) code_out[tid] = __uint_as_float(NF4_CODE_BITS[tid]);
    for (int off = 1; off < 64; off <<= 1) t += __shfl_xor(t, off, 64);
    if ((tid & 63) == 0) wave_sum[tid >> 6] = t;
    __syncthreads();
    if (tid == 0) {
        for (int j = 1; j < DQ_SUMS / 64; ++j) t += wave_sum[j];
        *offset = (float)(t / (double)nblocks);
    }
}

// r = absmax - offset; absmax2 = max|r| over a nested block; then the nearest entry of the 256-entry map (lowest index on
// ties) for every r * (1/absmax2).  A lane owns four consecutive values (one 128-bit load, one 32-bit word of codes), a
// nested block is a power of two of adjacent lanes.
//
// The nearest entry of an ascending map is found by bisection: rounded distances fl(s - map[j]) fall towards s from
// either side (rounding is monotonic), so the minimum lies at the last entry <= s or the first one > s.  Equal rounded
// distances are settled as the scan over all entries would: the left candidate wins a tie, and from there the index
// goes down while the distance stays the same.  A map that is not ascending and finite takes that scan.  Bisection: 9
// LDS reads per value instead of 256 reads, subtractions and compares; [28672, 8192] (3.7 M values) 93 us before, now 14.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void dq_compress_kernel(const float* __restrict__ absmax, int64_t nblocks,
                                                              int nested_log2, const float* __restrict__ map256,
                                                              float offset_value, const float* __restrict__ offset_ptr,
                                                              uint8_t* __restrict__ q, float* __restrict__ absmax2) {
    __shared__ float map[256];
    __shared__ float wave_max[THREADS / 64];
    __shared__ int zero_code;
    const int tid = threadIdx.x;
    const int64_t i0 = ((int64_t)blockIdx.x * THREADS + tid) * 4;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (i0 + 4 <= nblocks) {
        const float4 f = *reinterpret_cast<const float4*>(absmax + i0);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (i0 + c < nblocks) v[c] = absmax[i0 + c];
    }
    const float offset = offset_ptr ? *offset_ptr : offset_value;
    if (tid < 256) map[tid] = map256[tid];
    if (tid == 0) zero_code = 256;  // sentinel: the map holds no 0.0 (then an all-zero block stores code 0)
    __syncthreads();
    if (tid < 256 && map[tid] == 0.0f) atomicMin(&zero_code, tid);
    const bool ascending =
        __syncthreads_and(tid >= 255 ? isfinite(map[0]) && isfinite(map[255]) : map[tid] <= map[tid + 1]);

    float m = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        v[c] = __fsub_rn(v[c], offset);
        if (i0 + c < nblocks) m = fmaxf(m, fabsf(v[c]));
    }
    const int group = 1 << (nested_log2 - 2);  // lanes per nested block
    for (int off = 1; off < (group < 64 ? group : 64); off <<= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if (group > 64) {  // uniform branch: the nested block spans several waves
        if ((tid & 63) == 0) wave_max[tid >> 6] = m;
        __syncthreads();
        const int waves = group >> 6, first = (tid >> 6) & ~(waves - 1);
        for (int j = 0; j < waves; ++j) m = fmaxf(m, wave_max[first + j]);
    }
    if (i0 >= nblocks) return;
    if ((tid & (group - 1)) == 0) absmax2[i0 >> nested_log2] = m;

    const float inv = __fdiv_rn(1.0f, m);
    uint32_t code[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float s = __fmul_rn(v[c], inv);
        if (m == 0.0f) {
            code[c] = zero_code == 256 ? 0 : zero_code;
        } else if (!isfinite(s)) {
            code[c] = 0;  // no distance is below infinity
        } else if (ascending) {
            int pos = 0;  // entries <= s (255 at most)
#pragma unroll
            for (int step = 128; step; step >>= 1)
                if (map[pos + step - 1] <= s) pos += step;
            const float right = fabsf(__fsub_rn(s, map[pos]));
            int best = pos;
            if (pos > 0) {
                const float left = fabsf(__fsub_rn(s, map[pos - 1]));
                if (left <= right) {
                    best = pos - 1;
                    while (best > 0 && fabsf(__fsub_rn(s, map[best - 1])) == left) --best;
                }
            }
            code[c] = best;
        } else {
            float bestd = INFINITY;
            int best = 0;
            for (int j = 0; j < 256; ++j) {
                const float d = fabsf(__fsub_rn(s, map[j]));
                if (d < bestd) {
                    bestd = d;
                    best = j;
                }
            }
            code[c] = best;
        }
    }
    if (i0 + 4 <= nblocks) {
        *reinterpret_cast<uint32_t*>(q + i0) = code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (i0 + c < nblocks) q[i0 + c] = (uint8_t)code[c];
    }
}

__global__ __launch_bounds__(256) void dq_reconstruct_kernel(NestedAbsmax nq, int64_t nblocks,
                                                             float* __restrict__ absmax) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < nblocks) absmax[i] = nested_absmax(nq, i);
}

}  // namespace

hipError_t launch_quantize(const void* w, int w_dtype, int64_t n, int block_log2, uint8_t* packed, float* absmax,
                           hipStream_t stream) {
    if (n == 0) return hipSuccess;
    if (block_log2 == 12) {
        const int64_t grid = (n + 4096 * Q_SLOTS - 1) / (4096 * Q_SLOTS);
        hipLaunchKernelGGL(quantize_kernel<512>, dim3((unsigned)grid), dim3(512), 0, stream, w, w_dtype, n, block_log2,
                           packed, absmax);
    } else {
        const int64_t grid = (n + 2048 * Q_SLOTS - 1) / (2048 * Q_SLOTS);
        hipLaunchKernelGGL(quantize_kernel<256>, dim3((unsigned)grid), dim3(256), 0, stream, w, w_dtype, n, block_log2,
                           packed, absmax);
    }
    return hipGetLastError();
}

hipError_t launch_quantize_dq(const void* w, int w_dtype, int64_t n, int block_log2, int nested_log2, const float* map256,
                              uint8_t* packed, float* absmax, double* sums, float* offset, uint8_t* q, float* absmax2,
                              float* map_out, float* code_out, hipStream_t stream) {
    const int64_t nblocks = (n + (1 << block_log2) - 1) >> block_log2;
    hipError_t e = launch_quantize(w, w_dtype, n, block_log2, packed, absmax, stream);
    if (e != hipSuccess) return e;
    // a workgroup of the sum takes at least 4096 values
    const int64_t per = max((int64_t)4096, ((nblocks + DQ_SUMS - 1) / DQ_SUMS + 3) & ~(int64_t)3);
    const int count = (int)((nblocks + per - 1) / per);
    hipLaunchKernelGGL(dq_sum_kernel, dim3((unsigned)count), dim3(256), 0, stream, absmax, nblocks, per, sums);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(dq_offset_kernel, dim3(1), dim3(DQ_SUMS), 0, stream, sums, count, nblocks, offset, map256, map_out, code_out);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return launch_dq_compress(absmax, nblocks, nested_log2, map256, 0.0f, offset, q, absmax2, stream);
}

hipError_t launch_dequantize(const uint8_t* packed, const float* absmax, const NestedAbsmax& nested,
                             const float* lut16, int64_t n, int block_log2, void* out, int out_dtype,
                             hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const int64_t grid = (n + 2048 * DQ_SLOTS - 1) / (2048 * DQ_SLOTS);
    // An output that fits in the 256 MB last-level cache is written with ordinary stores, so that the
    // GEMM that usually follows finds it there; a larger one cannot stay anyway and is streamed
    // (non-temporal stores: 20 % faster on their own, 5 % slower for that GEMM).
    const int64_t out_bytes = n * (out_dtype == F32 ? 4 : 2);
    const bool stream_out = out_bytes > ((int64_t)192 << 20);
    const dim3 g((unsigned)grid), b(256);
    if (nested.q) {
        if (stream_out)
            hipLaunchKernelGGL((dequantize_kernel<true, true>), g, b, 0, stream, packed, absmax, nested, lut16, n, block_log2, out, out_dtype);
        else
            hipLaunchKernelGGL((dequantize_kernel<true, false>), g, b, 0, stream, packed, absmax, nested, lut16, n, block_log2, out, out_dtype);
    } else {
        if (stream_out)
            hipLaunchKernelGGL((dequantize_kernel<false, true>), g, b, 0, stream, packed, absmax, nested, lut16, n, block_log2, out, out_dtype);
        else
            hipLaunchKernelGGL((dequantize_kernel<false, false>), g, b, 0, stream, packed, absmax, nested, lut16, n, block_log2, out, out_dtype);
    }
    return hipGetLastError();
}

hipError_t launch_dq_compress(const float* absmax, int64_t nblocks, int nested_log2, const float* map256,
                              float offset, const float* offset_ptr, uint8_t* q, float* absmax2, hipStream_t stream) {
    if (nblocks == 0) return hipSuccess;
    // a workgroup holds whole nested blocks: 1024 values, or 4096 for the two largest nested block sizes
    const int threads = nested_log2 <= 10 ? 256 : 1024;
    const dim3 grid((unsigned)((nblocks + 4 * threads - 1) / (4 * threads)));
    if (threads == 256)
        hipLaunchKernelGGL(dq_compress_kernel<256>, grid, dim3(256), 0, stream, absmax, nblocks, nested_log2, map256, offset,
                           offset_ptr, q, absmax2);
    else
        hipLaunchKernelGGL(dq_compress_kernel<1024>, grid, dim3(1024), 0, stream, absmax, nblocks, nested_log2, map256, offset,
                           offset_ptr, q, absmax2);
    return hipGetLastError();
}

hipError_t launch_dq_reconstruct(const NestedAbsmax& nested, int64_t nblocks, float* absmax, hipStream_t stream) {
    if (nblocks == 0) return hipSuccess;
    const int64_t grid = (nblocks + 255) / 256;
    hipLaunchKernelGGL(dq_reconstruct_kernel, dim3((unsigned)grid), dim3(256), 0, stream, nested, nblocks, absmax);
    return hipGetLastError();
}

}  // namespace nf4
