// The whole single-token step of a Llama decoder in one launch: per layer the four 4-bit linears (fp32 absmax, blocksize 64),
// RMSNorm, rotary embedding, KV-cache update, grouped-query attention (head size 128, four query heads per kv head),
// SiLU(gate) * up and the residual adds, then the 4-bit output head, for 1..16 sequences (rows of x).  C ABI: nf4hip_decode_chain.h.
//
// What bounded the step before (one launch per linear and one for the attention, 164 in a graph): not the 3.9 GB of weights,
// which take 0.6 ms, but what stands between two streams of them -- the launch, the first requests' way to memory, the code-book
// table, the tail: 6..9 us of every launch of 6..16.  Here one workgroup per CU stays for the whole step:
// * Its share of every weight is one stream.  Requests run two tiles (16 weight rows x 4096 k) ahead and do not stop where a
//   linear ends: while the workgroups exchange activations, the next linear's first two tiles arrive.
// * Activations go from workgroup to workgroup through memory, words that say themselves whether they have been written:
//   bf16 pairs into scratch filled with NOT_YET ahead of the step (a pair of that value becomes another NaN), fp32 sums with
//   the layer beside them in one 64-bit word.  No flag, so no store waits for another to be acknowledged and no load follows a
//   load: 1.2 us from store to use, six or seven exchanges per layer.  Every such access is an agent-scope one (see nf4_common.h).  Scratch
//   of tagged words is used again by the next layer: a workgroup writes it only when all that read the last layer's have
//   left something that it has read since.
// * Nobody waits for a workgroup that does not run: each counts itself in, and when all of the grid are there -- or 50 us
//   have passed -- those that are, share the work.  Every phase (a linear; the attention goes with the output projection) is dealt in
//   tasks by the shape alone, a workgroup takes task me, me + members, .., and leaves the results of all its tasks of a phase
//   ahead of its first wait in the next, so any number of members ends with the same bits.  (A wait that lasts seconds all the
//   same gives NaN.)
//   While some are missing, the first that comes to the next layer (the next phase, where few are there) settles how many share it, and the
//   late ones join there: a workgroup needs a CU to itself, and kernels of other streams may hold most of them when a step
//   begins.  One sequence, 64 / 192 / 240 / 255 CUs held for another 0.42 ms: 1.6 / 1.6 / 1.6 / 2.1 ms (late ones gone for good 2.3 / 3.6 / 13.5 / 205;
//   by launches 1.75 / 1.9 / 2.05 / 2.05); with none held it costs 0..1 %.
// * Every sum is taken in the order of the kernel that the launch-by-launch step runs at Llama-3-8B's shapes (1, 5..16 sequences: the two
//   steps give the same bits; other batches and widths: the same roundings of stored tensors, sums in another order).
//   Through 32 layers any other order would move the logits by 0.05 of their norm, as two correct bf16 evaluations differ.
//   - CHAIN_SLICES, nf4_gemv_stage.hip's tile: wave w has 256 k of the workgroup's K range, x as MFMA operands in 32 registers,
//     sixteen waves' sums added through LDS.  The down projection (K > 4096) is split over up to four workgroups, each of which
//     finishes every fourth row of x.
//   - CHAIN_ROWS, one row of x (QKV, output and down projection), nf4_gemv_rows.hip's: 2048 k of a row per wave, one barrier per linear,
//     K up to 16384 in the workgroup.
//   - CHAIN_QUADS, five to eight rows of x (QKV), nf4_gemv_quad.hip's: four rows of 512 k per wave.
//   All take codes and absmax through the wave's ring in LDS and the byte -> two code-book values table there.
// * Attention: a (sequence, kv head, range of cached keys) per workgroup, sums as in decode_glue.hip; the first keys and values are
//   under way before the queries are known.
//
// Measured (graph replay, Llama-3-8B, 512 / 576 positions, MI355X, from box to box): 1 sequence 1584..1612 -> 1190..1215 us, 8 sequences 2025 -> 1620..1670.
// What bounds it now, per layer and for one sequence (38 us; stamps of the 100 MHz clock): tiles 22 us (1.1 us each in the gate-up
// projection while their data is there, 1.3 where HBM sets the pace, 1.6 in the others, whose 4x4x4 MFMAs fill the matrix
// pipe), six exchanges 9, attention's own work 4, the rest waits for the slowest workgroup.  Tried and not kept: a third tile
// ahead in registers (the exchange's loads return behind it), batches of tiles between two barriers (absmax then has to arrive a
// tile earlier), absmax fetched by each wave for itself (16 lines per request: gate-up 9.3 -> 10.3 us), every wave asking for
// the sums of squares (a few lines that all ask for delay the stores to them: 1255 -> 1511 us in all), a pause ahead of the
// first look at x (only behind the down projection with more than two rows of x, where it keeps the early ones out of the others' way).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "../../include/nf4hip_decode_chain.h"
#include "decode_chain.h"
#include "decode_math.h"
#include "nf4_gemv.h"

namespace {

using nf4::absmax_bits;
using nf4::absmax_of_bf16_pair;
using nf4::bf16_pair_to_f16;
using nf4::F16Scale;
using nf4::f16_scale_for;
using nf4::u16x2_t;
using nf4x::bf16_to_f32;
using nf4x::f32_to_bf16;
using nf4x::round_bf16;

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4;
typedef __attribute__((__vector_size__(4 * sizeof(_Float16)))) _Float16 f16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4e __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr int WAVES = 16;
constexpr int THREADS = WAVES * 64;
constexpr int SLICE_K = 256;
constexpr int SLOT_BYTES = 1024;
constexpr int RING_BYTES = 4 * SLOT_BYTES;  // of a wave: two tiles
constexpr int HD = 128;    // head size
constexpr int REP = 4;     // query heads of a kv head
constexpr int MAX_SLOTS = 512;  // partial sums of squares of a row of x

// ---- LDS map ----
constexpr int TABLE_SPAN = 256 * 256;  // 256-byte rows: 32 copies of an entry, then 128 bytes of the reduction buffers
constexpr int RING_OFF = TABLE_SPAN;
constexpr int ABS_OFF = RING_OFF + WAVES * RING_BYTES;
constexpr int ABS_BYTES = 16 * WAVES * 16;
constexpr int ABS_BUFS = 3;
constexpr int DONE_OFF = ABS_OFF + ABS_BUFS * ABS_BYTES;  // per row of x: the words a task leaves
constexpr int DONE_WORDS = 256;
constexpr int PTR_OFF = DONE_OFF + WAVES * DONE_WORDS * 4;  // codes and absmax of every linear: 16 bytes each
constexpr int ROPE_OFF = PTR_OFF + (4 * CHAIN_LAYERS + 1) * 16;  // cos, sin of the position
constexpr int ML_OFF = ROPE_OFF + 2 * HD * 4;            // of the attention: maxima of (wave, two heads), sums of (head, four waves)
constexpr int RSTD_OFF = ML_OFF + WAVES * 8 + REP * 16;  // 1 / rms of a row of x
constexpr int CTL_OFF = RSTD_OFF + WAVES * 4;
constexpr int SMEM_BYTES = 160 * 1024;
static_assert(CTL_OFF + 16 <= SMEM_BYTES, "LDS of one CU");
constexpr int RED_BUF_BYTES = WAVES * 1024;
[[maybe_unused]] constexpr uint32_t RED_PLANE = (1024u >> 7) << 8;
[[maybe_unused]] constexpr uint32_t RED_FLIP = ((uint32_t)RED_BUF_BYTES >> 7) << 8;
__device__ __forceinline__ uint32_t red_addr(uint32_t o) { return ((o >> 7) << 8) | 0x80u | (o & 127u); }

// scratch of the attention: four queries (scaled), the new key, the new value in fp32 at DONE_OFF; scores, then probabilities of
// the keys (four heads each) in the reduction buffers and, from key PS_KEYS on, behind the queries
[[maybe_unused]] constexpr int QS_BYTES = (REP + 2) * HD * 4;
constexpr int PS_KEYS = 2048;
constexpr int PS_MAX = PS_KEYS + (WAVES * DONE_WORDS * 4 - QS_BYTES) / 16;
__device__ __forceinline__ uint32_t ps_addr(int key) {
    return key < PS_KEYS ? red_addr((uint32_t)key * 16u) : (uint32_t)(DONE_OFF + QS_BYTES + (key - PS_KEYS) * 16);
}

template <typename T>
__device__ __forceinline__ T lds_read(uint32_t addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) T*>((uintptr_t)addr);
}
template <typename T>
__device__ __forceinline__ void lds_write(uint32_t addr, T v) {
    *reinterpret_cast<__attribute__((address_space(3))) T*>((uintptr_t)addr) = v;
}

#if defined(__HIP_DEVICE_COMPILE__)
typedef const __attribute__((address_space(4))) ChainArgs* args_ptr;
constexpr int SC1 = 16;  // cache policy of an agent-scope access: served from memory, not from this XCD's caches
constexpr uint32_t NOT_YET = 0xffffffffu;
constexpr uint32_t NOWHERE = 0x7ffffff0u;  // a buffer offset past every end: reads as zero, touches nothing

template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ const uint8_t* uniform_ptr(uint32_t lo, uint32_t hi) {
    return reinterpret_cast<const uint8_t*>((uint64_t)(uint32_t)uniform((int)lo) | ((uint64_t)(uint32_t)uniform((int)hi) << 32));
}
// a word that other workgroups wait for
__device__ __forceinline__ void publish(void* base, uint32_t word, uint32_t v) {
    __hip_atomic_store(static_cast<uint32_t*>(base) + word, v == NOT_YET ? NOT_YET - 1 : v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a 32-bit value that carries its layer
__device__ __forceinline__ void publish_tagged(void* base, uint32_t at, float v, uint32_t tag) {
    __hip_atomic_store(static_cast<uint64_t*>(base) + at, (uint64_t)__float_as_uint(v) | ((uint64_t)tag << 32), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
constexpr int QUAD_X1 = 0xB1, QUAD_X2 = 0x4E, HALF_MIRROR = 0x141, MIRROR = 0x140;
// over the 16 lanes of a row, in every one of them
template <typename OP>
__device__ __forceinline__ float row16(float v, OP op) {
    v = op(v, __uint_as_float(dpp<QUAD_X1>(__float_as_uint(v))));
    v = op(v, __uint_as_float(dpp<QUAD_X2>(__float_as_uint(v))));
    v = op(v, __uint_as_float(dpp<HALF_MIRROR>(__float_as_uint(v))));
    return op(v, __uint_as_float(dpp<MIRROR>(__float_as_uint(v))));
}
// lanes l and l ^ 16, l and l ^ 32
template <typename OP>
__device__ __forceinline__ float across16(float v, OP op) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <typename OP>
__device__ __forceinline__ float across32(float v, OP op) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float add(float x, float y) { return x + y; }
// Sums over lanes, in every one of them: lanes l and l ^ 8, 4, 2, 1 of a row of sixteen, in this order (what is equal in lanes l and
// l ^ 8 may be rotated by 4 for l ^ 4)
__device__ __forceinline__ float row16_down(float v) {
    v += __uint_as_float(dpp<0x128>(__float_as_uint(v)));
    v += __uint_as_float(dpp<0x124>(__float_as_uint(v)));
    v += __uint_as_float(dpp<0x122>(__float_as_uint(v)));
    return v + __uint_as_float(dpp<0x121>(__float_as_uint(v)));
}
// ... and halves first: __shfl_xor by 32, 16, .. 1
__device__ __forceinline__ float sum_down(float v) { return row16_down(across16(across32(v, add), add)); }
// lane l ^ 4 (a shift by four either way inside the row)
__device__ __forceinline__ float lane_xor4(float v) {
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp((int)__float_as_uint(v), (int)__float_as_uint(v), 0x104, 0xf, 0x5, false);
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp((int)o, (int)__float_as_uint(v), 0x114, 0xf, 0xa, false));
}
__device__ __forceinline__ float add_xor4(float v) { return v + lane_xor4(v); }
// over eight neighbouring lanes: l ^ 4, 2, 1
__device__ __forceinline__ float sum8_down(float v) {
    v = add_xor4(v);
    v += __uint_as_float(dpp<QUAD_X2>(__float_as_uint(v)));
    return v + __uint_as_float(dpp<QUAD_X1>(__float_as_uint(v)));
}
__device__ __forceinline__ uint32_t max4(const u32x4& v) { return max(max(v.x, v.y), max(v.z, v.w)); }

#endif

// One kernel per way of multiplying QKV (CHAIN_ROWS: one sequence; CHAIN_QUADS: five to eight; CHAIN_SLICES): with all three in one, 137
// scalar registers were spilled instead of 61..67, 32 layers of the 8B shapes took 1214 us with one sequence and 1657 with eight (now 1198,
// 1629), four layers of d 2048 with six 167 (163).
template <int QKV_MODE>
__global__ __launch_bounds__(THREADS, 1) void chain_kernel(ChainArgs) {
#if defined(__HIP_DEVICE_COMPILE__)
    // What a part of the step derives from the thread's number and the arguments it derives again: kept across parts they
    // would take more registers than there are.
    args_ptr ap = (args_ptr)__builtin_amdgcn_kernarg_segment_ptr();
    const int wave = uniform((int)threadIdx.x >> 6);
    auto thread_id = [&]() {
        int t = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(t));
        return t + wave * 64;
    };
    auto arguments = [&]() {
        args_ptr q = ap;
        asm volatile("" : "+s"(q));
        return q;
    };
#define ARGS const __attribute__((address_space(4))) ChainArgs& a = *arguments()
    ARGS;
    const int tid = thread_id();
    const int64_t pos64 = *a.pos;
    if (pos64 < 0 || pos64 >= a.max_seq) return;  // uniform: a position outside the cache touches nothing
    const int p = (int)pos64;

    const int head_phase = 4 * a.n_layer, last_phase = head_phase - (a.with_head ? 0 : 1);
    // ---- who takes part
    if (wave == 0) {
        uint32_t* const ctl = reinterpret_cast<uint32_t*>(a.ws + a.ctl_off);
        uint32_t r = 0, members = 0;
        if (tid == 0) {
            r = __hip_atomic_fetch_add(&ctl[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            auto decide = [&](uint32_t count) {
                uint32_t none = 0;
                __hip_atomic_compare_exchange_strong(&ctl[CHAIN_CTL_MEMBERS], &none, count, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            };
            const uint32_t most = (uint32_t)min(a.workgroups, a.first_members);
            if (r == most - 1) decide(most);
            const uint64_t t0 = wall_clock64();
            while ((members = __hip_atomic_load(&ctl[CHAIN_CTL_MEMBERS], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0)
                if (wall_clock64() - t0 > CHAIN_MUSTER_TICKS)
                    decide(min(__hip_atomic_load(&ctl[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), most));
        }
        r = (uint32_t)uniform((int)r);
        members = (uint32_t)uniform((int)members);
        // Late: it joins at the first phase that is dealt to more than its number, once that is settled.  (Phases are settled in order, and each
        // by who has seen the one before and counts afterwards: never for fewer.)
        int first = 0;
        for (int tries = 0; members <= r; ++tries) {
            first = last_phase + 1;
            members = 0;
#pragma unroll
            for (int i = 2; i >= 0; --i) {
                const int phase = tid + 64 * i;
                uint32_t v = ~0u;
                if (phase <= last_phase) v = __hip_atomic_load(&ctl[CHAIN_CTL_MEMBERS + phase], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint64_t mine = __ballot(phase <= last_phase && (v == 0 || v > r));
                if (mine) {
                    first = 64 * i + __ffsll((unsigned long long)mine) - 1;
                    members = (uint32_t)__builtin_amdgcn_readlane((int)v, first - 64 * i);
                }
            }
            if (first > last_phase) break;  // all of the step is dealt to others
            if (members == 0) {
                if (tries > CHAIN_MAX_POLLS) {
                    first = last_phase + 1;
                    break;
                }
                __builtin_amdgcn_s_sleep(64);  // 2 us
            }
        }
        if (tid == 0) {
            lds_write<uint32_t>(CTL_OFF, r);
            lds_write<uint32_t>(CTL_OFF + 4, members);
            lds_write<uint32_t>(CTL_OFF + 8, (uint32_t)first);
        }
    }
    // pointers of the stream and the rotary tables' row, while the others arrive
    if (tid < 4 * a.n_layer + 1) {
        const bool head = tid == 4 * a.n_layer;
        lds_write<uint64_t>(PTR_OFF + tid * 16, (uint64_t)(head ? a.head.codes : a.layers[tid >> 2].lin[tid & 3].codes));
        lds_write<uint64_t>(PTR_OFF + tid * 16 + 8, (uint64_t)(head ? a.head.absmax : a.layers[tid >> 2].lin[tid & 3].absmax));
    } else if (tid >= 512 && tid < 512 + HD) {
        lds_write<float>(ROPE_OFF + (tid - 512) * 4, a.cos_t[(int64_t)p * HD + tid - 512]);
    } else if (tid >= 768 && tid < 768 + HD) {
        lds_write<float>(ROPE_OFF + HD * 4 + (tid - 768) * 4, a.sin_t[(int64_t)p * HD + tid - 768]);
    }
    barrier();
    int phase = uniform((int)lds_read<uint32_t>(CTL_OFF + 8));
    if (phase > last_phase) return;
    // Those who share the phases up to `stop`, and this workgroup's number among them: of its arrival, while some are missing.
    int G = uniform((int)lds_read<uint32_t>(CTL_OFF + 4)), me = 0, stop = 0;
    auto settled = [&]() {
        ARGS;
        const int last = 4 * a.n_layer - (a.with_head ? 0 : 1);  // (again: see above)
        const bool all = G == a.workgroups;
        me = all ? (int)blockIdx.x : uniform((int)lds_read<uint32_t>(CTL_OFF));
        // It stops the stream of weights, 4 us: once a layer, or with less than a quarter of the workgroups, which take longer for a phase, once
        // a phase.  The late ones read it from the words of all the phases that it covers.
        stop = all ? last : 4 * G < a.workgroups ? phase : min(phase | 3, last);
        uint32_t* const members = reinterpret_cast<uint32_t*>(a.ws + a.ctl_off) + CHAIN_CTL_MEMBERS;
        if (!all && wave == 0 && thread_id() < stop - phase)
            __hip_atomic_store(&members[phase + 1 + thread_id()], (uint32_t)G, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    settled();

    // ---- the stream of weights
    // where it stands: a tile of one task of one linear
    const uint8_t *st_codes = nullptr, *st_absmax = nullptr;
    uint32_t st_left = 0;   // bytes of the task's codes from here on
    uint32_t st_tile = 0;   // codes of a tile
    int st_task = me, st_phase = phase, st_mode = CHAIN_SLICES;
    uint32_t st_even = 0, st_odd = 0, st_scales = 0;  // lane constants of the requests
    auto enter = [&]() {
        ARGS;
        // (called with nothing left of the last task)
        int kind = 0;
        while (st_phase <= stop) {
            kind = st_phase == head_phase ? CHAIN_HEAD : st_phase & 3;
            if (st_task < a.shape[kind].row_tasks * a.shape[kind].ksplits) break;
            ++st_phase;
            st_task = me;
        }
        if (st_phase > stop) return;
        const auto& s = a.shape[kind];
        const u32x4 ptr = lds_read<u32x4>(PTR_OFF + st_phase * 16);
        const int q = s.ksplits == 1 ? 0 : st_task % s.ksplits, r0 = (s.ksplits == 1 ? st_task : st_task / s.ksplits) * s.rows_per_task;
        const int row_bytes = s.K >> 1;
        st_left = (uint32_t)uniform(min(s.rows_per_task, s.N - r0) * row_bytes);
        st_codes = uniform_ptr(ptr.x, ptr.y) + (int64_t)r0 * row_bytes;
        st_absmax = uniform_ptr(ptr.z, ptr.w) + (int64_t)r0 * (row_bytes >> 3);
        st_mode = s.mode;
        st_tile = (uint32_t)(s.tile_rows * row_bytes);
        const int lane = thread_id() & 63;
        if (s.mode == CHAIN_SLICES) {
            // codes: lane i takes row i / 8 of the half tile, 16-byte piece (i % 8) ^ (row of the tile) / 2 of the wave's slice;
            // absmax: wave r fetches row r of a tile for all, lane i the four of slice i ^ r
            const int slice0 = q * s.slices_per_split, slices = min(s.slices_per_split, (s.K >> 8) - slice0);
            const int lrow = lane >> 3, apiece = (lane & 15) ^ wave;
            const uint32_t slice = (uint32_t)(slice0 + wave) * 128u, piece = (uint32_t)((lane & 7) ^ (lrow >> 1)) << 4;
            st_even = wave < slices ? (uint32_t)(lrow * row_bytes) + slice + piece : NOWHERE;
            st_odd = wave < slices ? (uint32_t)((lrow + 8) * row_bytes) + slice + (piece ^ 64u) : NOWHERE;
            st_scales = apiece < slices ? (uint32_t)(wave * (row_bytes >> 3)) + (uint32_t)(slice0 + apiece) * 16u : NOWHERE;
        } else {
            // `parts` waves side by side along K, `lanes` of them one above the other.  Rows: half a tile is one row per wave, lane i has
            // 32 k of its 2048; quads: four rows per wave of 512 k each, row i / 16, its 16-byte pieces in another order per row.
            // absmax: of the even half's rows in lanes 0..31, of the odd half's in the others.
            const int part = wave % s.parts, rl = wave / s.parts;
            const bool rows = s.mode == CHAIN_ROWS, on = rl < s.lanes;
            const int half = lane >> 5, l5 = lane & 31;
            const int row = rows ? rl : 4 * rl + (lane >> 4), up = (rows ? 1 : 4) * s.lanes;
            const int piece = rows ? lane : (lane & 15) ^ (4 * (lane >> 4));
            const uint32_t k16 = (uint32_t)part * (rows ? 1024u : 256u) + (uint32_t)piece * 16u;
            const bool inside = on && (int)k16 < row_bytes;
            st_even = inside ? (uint32_t)(row * row_bytes) + k16 : NOWHERE;
            st_odd = inside ? (uint32_t)((row + up) * row_bytes) + k16 : NOWHERE;
            const int arow = (rows ? rl : 4 * rl + (l5 >> 3)) + half * up, block = rows ? part * 32 + l5 : part * 8 + (l5 & 7);
            st_scales = on && block < (row_bytes >> 5) ? (uint32_t)(arow * (row_bytes >> 3)) + (uint32_t)block * 4u : NOWHERE;
        }
    };
    auto advance = [&]() {
        const bool more = st_left > st_tile;
        st_left = more ? st_left - st_tile : 0u;
        st_codes += st_tile;
        st_absmax += st_tile >> 3;
        if (!more) {
            st_task += G;
            enter();
        }
    };
    // The three requests of a tile: absmax, even half, odd half.
    auto request = [&](uint32_t slots, uint32_t abs_buf) {
        const uint32_t left = (uint32_t)uniform((int)st_left);
        const uint32_t ring = RING_OFF + wave * RING_BYTES + slots;
        const __amdgpu_buffer_rsrc_t cr = rsrc(st_codes, (int)left), ar = rsrc(st_absmax, (int)(left >> 3));
        if (st_mode != CHAIN_SLICES)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (lds_void_ptr)(uintptr_t)(ABS_OFF + abs_buf + wave * 256), 4, st_scales, 0, 0, 2);
        else if ((thread_id() & 63) < 16)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (lds_void_ptr)(uintptr_t)(ABS_OFF + abs_buf + wave * 256), 16, st_scales, 0, 0, 2);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(cr, (lds_void_ptr)(uintptr_t)ring, 16, st_even, 0, 0, 2);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(cr, (lds_void_ptr)(uintptr_t)(ring + SLOT_BYTES), 16, st_odd, 0, 0, 2);
    };
    uint32_t slots = 0, abs_now = 0;  // where the current tile's codes and absmax are
    auto prime = [&]() {  // the first two tiles of what begins at st_task (and nothing is left of what was before)
        st_left = 0;
        st_task -= G;
#pragma unroll 1
        for (int i = 0; i < 3; ++i) {
            if (i) request(slots ^ (i == 2 ? 2 * SLOT_BYTES : 0), i == 1 ? abs_now : abs_now == 2 * ABS_BYTES ? 0 : abs_now + ABS_BYTES);
            advance();
        }
    };
    prime();
    uint32_t parity = 0;              // which reduction buffer the next tile writes
    bool dead = false;  // a wait ran out: nothing is waited for any more, the step's answer is NaN

    // code book of the next linear: two values per thread
    float lut_hi, lut_lo;
    auto request_lut = [&](const float* lut, int tid) {
        lut_hi = lut[tid >> 6];
        lut_lo = lut[(tid >> 2) & 15];
    };
    request_lut(phase == head_phase ? a.head.lut : a.layers[phase >> 2].lin[phase & 3].lut, tid);

    auto spin = [&](auto&& attempt) {  // attempt(): does this lane still miss something?
        int tries = 0;
        while (__ballot(attempt()) != 0) {
            if (dead || ++tries > CHAIN_MAX_POLLS) {
                dead = true;
                break;
            }
            asm volatile("" ::: "memory");
        }
    };

    // (the first layer's input lies behind the others: it is written ahead of this launch)
    auto input_set = [&](const auto& a, int l) { return a.ws + a.in_off + (int64_t)(l == 0 ? a.model_layers : l - 1) * a.in_stride; };
    auto layer_set = [&](const auto& a, int l) { return a.ws + a.layer_off + (int64_t)l * a.layer_stride; };

    // One linear of one layer.
    auto linear = [&](auto kind_tag, auto mode_tag, int l, const float* next_lut) {
        constexpr int KIND = decltype(kind_tag)::value, MODE = decltype(mode_tag)::value;
        ARGS;
        const int tid = thread_id(), lane = tid & 63, n = lane & 15, g = lane >> 4;
        const int M = a.batch;
        const uint32_t d_words = (uint32_t)a.d_model >> 1;
        // as in nf4_gemv_stage.hip
        const uint32_t col4 = (uint32_t)(lane & 31) * 4u;
        const uint32_t c0 = RING_OFF + wave * RING_BYTES + (n < 8 ? 0u : (uint32_t)SLOT_BYTES) + (uint32_t)(n & 7) * 128u + ((uint32_t)((g >> 1) ^ (n >> 1)) << 4) + (uint32_t)(g & 1) * 8u;
        const uint32_t aread = ABS_OFF + (uint32_t)(n * 16 + (wave ^ n)) * 16u;
        const uint32_t red_w = red_addr((uint32_t)(4 * g) * 1024u + (uint32_t)((16 * wave + n) ^ ((g & 1) << 4)) * 4u);
        const uint32_t red_r = red_addr((uint32_t)wave * 1024u + (uint32_t)((16 * g + n) ^ (((wave >> 2) & 1) << 4)) * 4u);
        const bool reducer = wave < M;
        const bool writes_sums = 4 * g < M;
        constexpr bool F16 = KIND == CHAIN_DOWN;
        constexpr bool SCALED = KIND == CHAIN_QKV || KIND == CHAIN_GATE_UP || KIND == CHAIN_HEAD;
        const auto& s = a.shape[KIND];
        const int N = s.N, K = s.K, ntasks = s.row_tasks * s.ksplits;
        const int layer = a.layer0 + l;
        uint8_t* const in = input_set(a, layer);
        uint8_t* const mid = layer_set(a, layer);
        // what this linear reads, what it leaves
        const uint8_t* const x_src = KIND == CHAIN_QKV || KIND == CHAIN_HEAD ? in
                                     : KIND == CHAIN_OUT                     ? mid + a.y_off
                                     : KIND == CHAIN_GATE_UP                 ? mid + a.xo_off
                                                                             : mid + a.h_off;
        const uint8_t* const ss_src = KIND == CHAIN_GATE_UP ? mid + a.sso_off : in + a.ss_off;
        const int ss_slots = a.shape[KIND == CHAIN_GATE_UP ? CHAIN_OUT : CHAIN_DOWN].sums;
        const bool scaled = SCALED && (KIND != CHAIN_QKV || layer > 0);  // (the first layer's input is normalised ahead of this launch)
        // Row m's sums of squares, of wave m: eight per lane, added as the epilogue of the kernel that this mode follows adds them.
        float ssp[8];
        auto ask_sums = [&](int m) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                ssp[j] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rsrc(ss_src + m * MAX_SLOTS * 4, ss_slots * 4), lane * 4 + 256 * j, 0, SC1));
        };
        auto sums_missing = [&]() {
            uint32_t mx = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) mx = max(mx, __float_as_uint(ssp[j]));
            return mx;
        };
        auto rstd_of_sums = [&]() {
            float t;
            if constexpr (MODE == CHAIN_SLICES) {
                t = ssp[0];
#pragma unroll
                for (int j = 1; j < 8; ++j) t += ssp[j];
                t = sum_down(t);
            } else if constexpr (MODE == CHAIN_QUADS) {
                t = sum_down(((ssp[0] + ssp[1]) + (ssp[2] + ssp[3])) + ((ssp[4] + ssp[5]) + (ssp[6] + ssp[7])));
            } else {
                t = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; ++j) t += sum_down(ssp[j]);
            }
            return rsqrtf(t / (float)K + a.eps);
        };

        // byte -> two code-book values: every wave is past the barrier behind the last use of the table
        {
            const uint32_t vb = F16 ? (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)lut_hi) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)lut_lo) << 16)
                                    : f32_to_bf16(lut_hi) | (f32_to_bf16(lut_lo) << 16);
            const u32x4 v = {vb, vb, vb, vb};
            const uint32_t dst = (uint32_t)(tid >> 2) * 256u + (uint32_t)(tid & 3) * 32u;
            lds_write(dst, v);
            lds_write(dst + 16, v);
        }
        if (next_lut) request_lut(next_lut, tid);

        // The workgroups that are done first would ask for x while the others still wait for each other's sums.
        if (KIND == CHAIN_QKV && M > 2) __builtin_amdgcn_s_sleep(40);
        if constexpr (MODE == CHAIN_ROWS) {
            // One row of x, as nf4_gemv_rows.hip adds: a lane has 32 k of a weight row (v_mfma 4x4x4, of whose sixteen products per lane
            // quad the diagonal is wanted), lanes by a butterfly, the parts of K in order.  No sums of sixteen waves to meet after
            // every tile, and K up to 16384 within the workgroup.
            const int part = wave % s.parts, rl = wave / s.parts;
            const bool k_on = rl < s.lanes && part * 2048 + 32 * lane < K;
            const uint32_t mine = RING_OFF + wave * RING_BYTES + (uint32_t)lane * 16u;
            const uint32_t scales = ABS_OFF + (uint32_t)wave * 256u + (uint32_t)(lane >> 1) * 4u;
            for (int task = me; task < ntasks; task += G) {
                const int r0 = task * s.rows_per_task, r1 = min(N, r0 + s.rows_per_task), nrows = r1 - r0;
                // what the rows' finishing needs: lane r of wave 0
                const int my_row = min(r0 + lane, r1 - 1);
                uint32_t resid_w = 0, norm_w = 0;
                if constexpr (!SCALED) {
                    if (wave == 0) norm_w = (KIND == CHAIN_OUT ? a.layers[l].norm_mid : a.layers[l].norm_next)[my_row];
                }
                // x: 16-byte pieces tid and tid + 1024 of the row
                const __amdgpu_buffer_rsrc_t xr = rsrc(x_src, K * 2);
                u32x4 v[2];
                v[1] = u32x4{0, 0, 0, 0};
                spin([&]() {
                    v[0] = __builtin_amdgcn_raw_buffer_load_b128(xr, tid * 16, 0, SC1);
                    if (wave * 512 + 8192 < K) v[1] = __builtin_amdgcn_raw_buffer_load_b128(xr, tid * 16 + 16384, 0, SC1);
                    uint32_t mx = max(max4(v[0]), max4(v[1]));
                    if (wave == 0) {
                        if constexpr (SCALED) {
                            if (scaled) {
                                ask_sums(0);
                                mx = max(mx, sums_missing());
                            }
                        } else {
                            resid_w = __builtin_amdgcn_raw_buffer_load_b32(rsrc(KIND == CHAIN_OUT ? in + a.r_off : mid + a.ro_off, N * 2), (my_row >> 1) * 4, 0, SC1);
                            mx = max(mx, resid_w);
                        }
                    }
                    return mx == NOT_YET;
                });
                asm volatile("" ::"v"(lut_hi), "v"(lut_lo), "v"(norm_w));  // (arrived ahead of x)
                float rstd = 1.0f;
                if constexpr (SCALED) {
                    if (wave == 0 && scaled) rstd = rstd_of_sums();
                }
                barrier();  // the reduction buffers are free
                // piece q of a lane's four at q ^ (lane / 2) % 4
                auto piece_at = [&](int block, int q) { return red_addr((uint32_t)block * 64u + (uint32_t)((q ^ (block >> 1)) & 3) * 16u); };
                if (tid * 8 < K) lds_write<u32x4>(piece_at(tid >> 2, tid & 3), v[0]);
                if (tid * 8 + 8192 < K) lds_write<u32x4>(piece_at((tid >> 2) + 256, tid & 3), v[1]);
                barrier();  // x, the table
                u32x4 xv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    xv[j] = u32x4{0, 0, 0, 0};
                    if (k_on) xv[j] = lds_read<u32x4>(piece_at(part * 64 + lane, j));
                }
                float unscale = 1.0f;
                if constexpr (F16) {
                    u16x2_t mx = {0, 0};
#pragma unroll
                    for (int j = 0; j < 16; ++j) mx = absmax_of_bf16_pair(xv[j >> 2][j & 3], mx);
                    const F16Scale fs = f16_scale_for(absmax_bits(mx));
#pragma unroll
                    for (int j = 0; j < 16; ++j) xv[j >> 2][j & 3] = bf16_pair_to_f16(xv[j >> 2][j & 3], fs.to_f16);
                    unscale = fs.from_f16;
                }
                const int tiles = (nrows + s.tile_rows - 1) / s.tile_rows;
                for (int t = 0; t < tiles; ++t) {
                    wait_vm<3>();  // (as below)
                    u32x4 cd[2];
                    float sc[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        cd[h] = lds_read<u32x4>(mine + slots + h * SLOT_BYTES);
                        sc[h] = lds_read<float>(scales + abs_now + h * 128);
                    }
                    asm volatile("" ::"v"(cd[0]), "v"(cd[1]), "v"(sc[0]), "v"(sc[1]));
                    request(slots, abs_now == 0 ? 2 * ABS_BYTES : abs_now - ABS_BYTES);
                    advance();
                    float part_sum[2] = {0.0f, 0.0f};
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (t * s.tile_rows + h * s.lanes >= nrows) break;  // (uniform: the odd half of a task's last tile)
                        f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            uint2 w;
                            const uint32_t d = cd[h][i >> 1];
                            w.x = lds_read<uint32_t>(__builtin_amdgcn_perm(d, col4, 0x0c0c0400u | ((uint32_t)(2 * (i & 1)) << 8)));
                            w.y = lds_read<uint32_t>(__builtin_amdgcn_perm(d, col4, 0x0c0c0400u | ((uint32_t)(2 * (i & 1) + 1) << 8)));
                            const uint2 xb = make_uint2(xv[i >> 1][2 * (i & 1)], xv[i >> 1][2 * (i & 1) + 1]);
                            if constexpr (F16)
                                c = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, w), __builtin_bit_cast(f16x4, xb), c, 0, 0, 0);
                            else
                                c = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, w), __builtin_bit_cast(s16x4, xb), c, 0, 0, 0);
                        }
                        const float c01 = (lane & 1) ? c[1] : c[0], c23 = (lane & 1) ? c[3] : c[2];
                        const float diag = (lane & 2) ? c23 : c01;
                        part_sum[h] = diag * ((k_on ? sc[h] : 0.0f) * unscale);
                    }
                    // both rows over the wave, lane bit 0 choosing the row from the first step on
                    const uint32_t keep = __float_as_uint((lane & 1) ? part_sum[1] : part_sum[0]), send = __float_as_uint((lane & 1) ? part_sum[0] : part_sum[1]);
                    float sum = __uint_as_float(keep) + __uint_as_float(dpp<QUAD_X1>(send));
                    sum += __uint_as_float(dpp<QUAD_X2>(__float_as_uint(sum)));
                    sum = add_xor4(sum);
                    sum += __uint_as_float(dpp<0x128>(__float_as_uint(sum)));
                    sum = across32(across16(sum, add), add);
                    const int row = t * s.tile_rows + (lane & 1) * s.lanes + rl;
                    if (lane < 2 && rl < s.lanes && row < nrows) lds_write<float>(DONE_OFF + (uint32_t)(row * s.parts + part) * 4u, sum);
                    slots ^= 2 * SLOT_BYTES;
                    abs_now = abs_now == 2 * ABS_BYTES ? 0 : abs_now + ABS_BYTES;
                }
                barrier();  // all parts of all rows; the table is done with
                if (wave == 0) {
                    float sum = 0.0f;
                    for (int c = 0; c < s.parts; ++c) sum += lds_read<float>(DONE_OFF + (uint32_t)(min(lane, nrows - 1) * s.parts + c) * 4u);
                    const uint32_t word = (uint32_t)(r0 + lane) >> 1;
                    const bool writes = lane < nrows && !(lane & 1);
                    if constexpr (SCALED) {
                        const uint32_t b = f32_to_bf16(sum * rstd), o = dpp<QUAD_X1>(b);
                        if (writes) publish(mid + a.qkv_off, word, b | (o << 16));
                    } else {
                        const uint32_t rw = (lane & 1) ? resid_w >> 16 : resid_w & 0xffffu;
                        const float r = nf4x::resid_add(bf16_to_f32(rw), round_bf16(dead ? __uint_as_float(0x7fc00000u) : sum));
                        const uint32_t rb = f32_to_bf16(r), xb = f32_to_bf16(r * bf16_to_f32(norm_w));
                        const uint32_t ro = dpp<QUAD_X1>(rb), xo = dpp<QUAD_X1>(xb);
                        uint8_t* const next = KIND == CHAIN_OUT ? mid + a.xo_off : input_set(a, layer + 1);
                        uint8_t* const next_r = KIND == CHAIN_OUT ? mid + a.ro_off : next + a.r_off;
                        uint8_t* const next_ss = KIND == CHAIN_OUT ? mid + a.sso_off : next + a.ss_off;
                        if (writes) {
                            publish(next, word, xb | (xo << 16));
                            publish(next_r, word, rb | (ro << 16));
                        }
                        const float ss = sum8_down(lane < nrows ? r * r : 0.0f);  // a sum of squares per eight rows
                        if (lane < nrows && !(lane & 7)) publish(next_ss, (uint32_t)(r0 + lane) >> 3, __float_as_uint(ss));
                    }
                }
            }
        } else if constexpr (MODE == CHAIN_QUADS) {
            // Five to eight rows of x, as nf4_gemv_quad.hip adds: lane 4 s + r has 32 k (segment s of 512) of weight row r of a group
            // of four and of rows r and r + 4 of x; the sixteen products of a lane quad are four weight rows times four rows of x.
            const int part = wave % s.parts, rl = wave / s.parts, r = lane & 3, seg = lane >> 2;
            const bool on = rl < s.lanes;
            const uint32_t mine = RING_OFF + wave * RING_BYTES + (uint32_t)(r * 16 + (seg ^ (4 * r))) * 16u;
            const uint32_t scales = ABS_OFF + (uint32_t)wave * 256u + (uint32_t)(r * 8 + (seg >> 1)) * 4u;
            for (int task = me; task < ntasks; task += G) {
                const int r0 = task * s.rows_per_task, r1 = min(N, r0 + s.rows_per_task), nrows = r1 - r0;
                const __amdgpu_buffer_rsrc_t xr = rsrc(x_src, M * K * 2);
                const uint32_t at = on ? (uint32_t)part * 1024u + (uint32_t)lane * 16u : NOWHERE;
                spin([&]() {
                    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(xr, on ? at + (uint32_t)(wave % M) * (uint32_t)(K * 2) : NOWHERE, 0, SC1);
                    uint32_t mx = max4(v);
                    if (wave < M && scaled) {
                        ask_sums(wave);
                        mx = max(mx, sums_missing());
                    }
                    return mx == NOT_YET;
                });
                u32x4 raw[8];  // (through this XCD's cache: see below)
#pragma unroll
                for (int j = 0; j < 8; ++j) raw[j] = __builtin_amdgcn_raw_buffer_load_b128(xr, on && j < M ? at + (uint32_t)j * (uint32_t)(K * 2) : NOWHERE, 0, 0);
                uint32_t missing = 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) missing |= __ballot(max4(raw[j]) == NOT_YET) != 0 ? 1u << j : 0u;
                if (missing) {
                    spin([&]() {
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            if (missing >> j & 1) raw[j] = __builtin_amdgcn_raw_buffer_load_b128(xr, on && j < M ? at + (uint32_t)j * (uint32_t)(K * 2) : NOWHERE, 0, SC1);
                        missing = 0;
#pragma unroll
                        for (int j = 0; j < 8; ++j) missing |= __ballot(max4(raw[j]) == NOT_YET) != 0 ? 1u << j : 0u;
                        return missing != 0;
                    });
                }
                asm volatile("" ::"v"(lut_hi), "v"(lut_lo));  // (arrived ahead of x)
                if (wave < M && scaled) {
                    const float rstd = rstd_of_sums();
                    if (lane == 0) lds_write<float>(RSTD_OFF + wave * 4, rstd);
                }
                // raw[j]: 8 k of row j; a transposition inside every lane quad gives lane r the quad's 32 k of rows r and r + 4
                u32x4 xv[2][4];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        uint32_t w[4] = {raw[4 * h][e], raw[4 * h + 1][e], raw[4 * h + 2][e], raw[4 * h + 3][e]};
                        nf4::transpose_quad(w[0], w[1], w[2], w[3], lane & 1, lane & 2);
#pragma unroll
                        for (int j = 0; j < 4; ++j) xv[h][j][e] = w[j];
                    }
                }
                barrier();  // the table
                const int tiles = (nrows + s.tile_rows - 1) / s.tile_rows;
                for (int t = 0; t < tiles; ++t) {
                    wait_vm<3>();  // (as below)
                    u32x4 cd[2];
                    float sc[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        cd[h] = lds_read<u32x4>(mine + slots + h * SLOT_BYTES);
                        sc[h] = lds_read<float>(scales + abs_now + h * 128);
                    }
                    asm volatile("" ::"v"(cd[0]), "v"(cd[1]), "v"(sc[0]), "v"(sc[1]));
                    request(slots, abs_now == 0 ? 2 * ABS_BYTES : abs_now - ABS_BYTES);
                    advance();
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (t * s.tile_rows + 4 * h * s.lanes >= nrows) break;  // (uniform: the odd half of a task's last tile)
                        f32x4 c[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            uint2 w;
                            const uint32_t d = cd[h][i >> 1];
                            w.x = lds_read<uint32_t>(__builtin_amdgcn_perm(d, col4, 0x0c0c0400u | ((uint32_t)(2 * (i & 1)) << 8)));
                            w.y = lds_read<uint32_t>(__builtin_amdgcn_perm(d, col4, 0x0c0c0400u | ((uint32_t)(2 * (i & 1) + 1) << 8)));
#pragma unroll
                            for (int m4 = 0; m4 < 2; ++m4) {
                                const uint2 xb = make_uint2(xv[m4][i >> 1][2 * (i & 1)], xv[m4][i >> 1][2 * (i & 1) + 1]);
                                c[m4] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, w), __builtin_bit_cast(s16x4, xb), c[m4], 0, 0, 0);
                            }
                        }
                        const uint32_t sb = __float_as_uint(sc[h]);
                        const float s4[4] = {__uint_as_float(dpp<0x00>(sb)), __uint_as_float(dpp<0x55>(sb)), __uint_as_float(dpp<0xAA>(sb)), __uint_as_float(dpp<0xFF>(sb))};
#pragma unroll
                        for (int m4 = 0; m4 < 2; ++m4) {
                            // over lanes l ^ 4, 8, 16, 32, the sixteen segments; lane bits 2 and 3 choose the weight row from the first steps on
                            float tot[4];
#pragma unroll
                            for (int i = 0; i < 4; ++i) tot[i] = fmaf(s4[i], c[m4][i], 0.0f);
                            const bool b2 = lane & 4, b3 = lane & 8;
                            const float w0 = (b2 ? tot[1] : tot[0]) + lane_xor4(b2 ? tot[0] : tot[1]);
                            const float w1 = (b2 ? tot[3] : tot[2]) + lane_xor4(b2 ? tot[2] : tot[3]);
                            float v = (b3 ? w1 : w0) + __uint_as_float(dpp<0x128>(__float_as_uint(b3 ? w0 : w1)));
                            v = across32(across16(v, add), add);
                            const int row = t * s.tile_rows + 4 * (h * s.lanes + rl) + seg;  // lanes 0..15: weight row seg of the group
                            if (lane < 16 && on && row < nrows) lds_write<float>(DONE_OFF + (uint32_t)((row * s.parts + part) * 8 + 4 * m4 + r) * 4u, v);
                        }
                    }
                    slots ^= 2 * SLOT_BYTES;
                    abs_now = abs_now == 2 * ABS_BYTES ? 0 : abs_now + ABS_BYTES;
                }
                barrier();  // all parts of all rows; the table is done with
                for (int i = tid; i < (nrows >> 1) * 8; i += THREADS) {
                    const int m = i & 7, row = (i >> 3) * 2;
                    float s0 = 0.0f, s1 = 0.0f;
                    for (int c = 0; c < s.parts; ++c) {
                        s0 += lds_read<float>(DONE_OFF + (uint32_t)((row * s.parts + c) * 8 + m) * 4u);
                        s1 += lds_read<float>(DONE_OFF + (uint32_t)(((row + 1) * s.parts + c) * 8 + m) * 4u);
                    }
                    if (scaled) {
                        const float rstd = lds_read<float>(RSTD_OFF + m * 4);
                        s0 *= rstd;
                        s1 *= rstd;
                    }
                    if (m < M) publish(mid + a.qkv_off, (uint32_t)m * (uint32_t)(N >> 1) + (uint32_t)((r0 + row) >> 1), f32_to_bf16(s0) | (f32_to_bf16(s1) << 16));
                }
                if (task + G < ntasks) barrier();  // (the next task's sums go where these were)
            }
        } else
        for (int task = me; task < ntasks; task += G) {
            const int ksplits = KIND == CHAIN_DOWN ? s.ksplits : 1;
            const int q = ksplits == 1 ? 0 : task % ksplits, r0 = (ksplits == 1 ? task : task / ksplits) * s.rows_per_task, r1 = min(N, r0 + s.rows_per_task);
            const int tiles = (r1 - r0 + 15) >> 4;
            const int slice0 = q * s.slices_per_split, slices = min(s.slices_per_split, (K >> 8) - slice0);
            const bool on = wave < slices;

            // ---- x, and what the wave's finishing needs
            uint32_t resid_w = 0, norm_w = 0;  // CHAIN_OUT (one tile)
            const uint32_t norm_row = (uint32_t)min(r0 + n, N - 1);
            if constexpr (KIND == CHAIN_OUT) {
                if (reducer) norm_w = a.layers[l].norm_mid[norm_row];
            }
            u32x4 xv[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) ssp[j] = 0.0f;
            const __amdgpu_buffer_rsrc_t xr = rsrc(x_src, M * K * 2);
            const uint32_t x_slice = (uint32_t)(slice0 + wave) * 512u;
            auto ask_rest = [&]() {  // (a few lines that every workgroup asks for: by the waves that use them only)
                if (!reducer) return;
                if (scaled) ask_sums(wave);
                if constexpr (KIND == CHAIN_OUT)
                    resid_w = __builtin_amdgcn_raw_buffer_load_b32(rsrc(in + a.r_off, M * (int)d_words * 4), ((uint32_t)wave * d_words + (norm_row >> 1)) * 4u, 0, SC1);
            };
            auto rest_missing = [&]() { return KIND == CHAIN_OUT ? resid_w : SCALED ? sums_missing() : 0u; };
            float unscale[4] = {1.0f, 1.0f, 1.0f, 1.0f};
            auto larger = [](float x, float y) { return __uint_as_float(max(__float_as_uint(x), __float_as_uint(y))); };  // (of bits)
            if (M <= 2) {
                // two rows: a wave's slice in one request, into operand order through LDS (the buffer that the next tile writes)
                const int row = lane >> 5;
                const uint32_t at = on ? (uint32_t)min(row, M - 1) * (uint32_t)(K * 2) + x_slice + (uint32_t)(lane & 31) * 16u : NOWHERE;
                u32x4 v;
                spin([&]() {
                    v = __builtin_amdgcn_raw_buffer_load_b128(xr, at, 0, SC1);
                    ask_rest();
                    return max(max4(v), rest_missing()) == NOT_YET;
                });
                if constexpr (F16) {
                    u16x2_t mx = {0, 0};
#pragma unroll
                    for (int e = 0; e < 4; ++e) mx = absmax_of_bf16_pair(v[e], mx);
                    const float mb = across16(row16(__uint_as_float(absmax_bits(mx)), larger), larger);
                    const F16Scale fs = f16_scale_for(__float_as_uint(mb));
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = bf16_pair_to_f16(v[e], fs.to_f16);
                    unscale[0] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fs.from_f16), 0));
                    unscale[1] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fs.from_f16), 32));
                }
                lds_write<u32x4>(red_addr((uint32_t)wave * 1024u + (uint32_t)lane * 16u) ^ parity, v);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    xv[j] = lds_read<u32x4>(red_addr((uint32_t)wave * 1024u + (uint32_t)(n & 1) * 512u + (uint32_t)g * 32u + (uint32_t)(j >> 1) * 128u + (uint32_t)(j & 1) * 16u) ^ parity);
            } else {
                const uint32_t at = on ? (uint32_t)min(n, M - 1) * (uint32_t)(K * 2) + x_slice + (uint32_t)g * 32u : NOWHERE;
                // More: one row of the slice is waited for, and then all rows are read through this XCD's cache, where one of its 32
                // workgroups finds them absent and the others present (each address is read for the first time in this launch,
                // so no older line can be there).  What is not complete yet after all is asked for from memory.
                spin([&]() {
                    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(xr, on ? (uint32_t)(wave % M) * (uint32_t)(K * 2) + x_slice + (uint32_t)(lane & 31) * 16u : NOWHERE, 0, SC1);
                    ask_rest();
                    return max(max4(v), rest_missing()) == NOT_YET;
                });
#pragma unroll
                for (int j = 0; j < 8; ++j) xv[j] = u32x4{0, 0, 0, 0};
                if (n < M) {  // (rows past M hold anything)
#pragma unroll
                    for (int j = 0; j < 8; ++j) xv[j] = __builtin_amdgcn_raw_buffer_load_b128(xr, at + (uint32_t)(j >> 1) * 128u + (uint32_t)(j & 1) * 16u, 0, 0);
                }
                uint32_t missing = 0;  // of the eight requests
#pragma unroll
                for (int j = 0; j < 8; ++j) missing |= __ballot(max4(xv[j]) == NOT_YET) != 0 ? 1u << j : 0u;
                if (missing) {
                    spin([&]() {
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            if (missing >> j & 1) xv[j] = __builtin_amdgcn_raw_buffer_load_b128(xr, at + (uint32_t)(j >> 1) * 128u + (uint32_t)(j & 1) * 16u, 0, SC1);
                        missing = 0;
#pragma unroll
                        for (int j = 0; j < 8; ++j) missing |= __ballot(max4(xv[j]) == NOT_YET) != 0 ? 1u << j : 0u;
                        return missing != 0;
                    });
                }
                if constexpr (F16) {
                    u16x2_t mx = {0, 0};
#pragma unroll
                    for (int j = 0; j < 8; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) mx = absmax_of_bf16_pair(xv[j][e], mx);
                    const float mb = __uint_as_float(absmax_bits(mx));
                    const F16Scale fs = f16_scale_for(__float_as_uint(across32(across16(mb, larger), larger)));
#pragma unroll
                    for (int j = 0; j < 8; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) xv[j][e] = bf16_pair_to_f16(xv[j][e], fs.to_f16);
#pragma unroll
                    for (int i = 0; i < 4; ++i) unscale[i] = __int_as_float(__builtin_amdgcn_ds_bpermute((4 * g + i) * 4, __float_as_int(fs.from_f16)));
                }
            }
            asm volatile("" ::"v"(lut_hi), "v"(lut_lo));  // (arrived ahead of x)
            if constexpr (KIND == CHAIN_OUT) asm volatile("" ::"v"(norm_w));
            float rstd = 1.0f;
            if constexpr (SCALED) {
                if (reducer && scaled) rstd = rstd_of_sums();
            }
            barrier();  // the table; the reduction buffers are free

            float resid_ss = 0.0f;
            auto finish_tile = [&](int t, const float (&pt)[4]) {
                float sum = across32(across16(((pt[0] + pt[1]) + pt[2]) + pt[3], add), add);
                const int row = r0 + 16 * t + n;
                const bool mine = g == 0 && row < r1;
                if constexpr (SCALED) sum *= rstd;
                // what the row of x is left with goes to LDS, word by word, and on from there behind the last tile: a store in
                // the loop would be waited for by the counts below
                const uint32_t done = DONE_OFF + (uint32_t)(wave * DONE_WORDS) * 4u;
                if constexpr (KIND == CHAIN_QKV || KIND == CHAIN_HEAD) {
                    const uint32_t v = f32_to_bf16(sum), o = dpp<QUAD_X1>(v);
                    if (mine && !(n & 1)) lds_write<uint32_t>(done + (uint32_t)(16 * t + n) * 2u, v | (o << 16));
                } else if constexpr (KIND == CHAIN_OUT) {
                    const uint32_t rw = (n & 1) ? resid_w >> 16 : resid_w & 0xffffu;
                    const float r = nf4x::resid_add(bf16_to_f32(rw), round_bf16(sum));
                    const uint32_t rb = f32_to_bf16(r), xb = f32_to_bf16(r * bf16_to_f32(norm_w));
                    const uint32_t ro = dpp<QUAD_X1>(rb), xo = dpp<QUAD_X1>(xb);
                    if (mine) {
                        resid_ss = fmaf(r, r, resid_ss);
                        if (!(n & 1)) {
                            lds_write<uint32_t>(done + (uint32_t)(16 * t + n) * 2u, xb | (xo << 16));
                            lds_write<uint32_t>(done + (uint32_t)(32 + 16 * t + n) * 2u, rb | (ro << 16));
                        }
                    }
                } else if constexpr (KIND == CHAIN_GATE_UP) {
                    const float v = round_bf16(sum), o = __uint_as_float(dpp<QUAD_X1>(__float_as_uint(v)));
                    const uint32_t h = nf4x::silu_mul_bf16(v, o), h2 = dpp<QUAD_X2>(h);
                    if (mine && !(n & 3)) lds_write<uint32_t>(done + (uint32_t)(16 * t + n), h | (h2 << 16));
                } else {
                    if (mine) lds_write<float>(done + (uint32_t)(16 * t + n) * 4u, sum);
                }
            };
            auto leave = [&]() {  // the task's words, to whoever waits for them
                const uint32_t done = DONE_OFF + (uint32_t)(wave * DONE_WORDS) * 4u;
                const int words = (r1 - r0) >> (KIND == CHAIN_DOWN ? 0 : KIND == CHAIN_GATE_UP ? 2 : 1);
                for (int i = lane; i < words; i += 64) {
                    const uint32_t v = lds_read<uint32_t>(done + (uint32_t)i * 4u);
                    if constexpr (KIND == CHAIN_QKV) {
                        publish(mid + a.qkv_off, (uint32_t)wave * (uint32_t)(N >> 1) + (uint32_t)(r0 >> 1) + (uint32_t)i, v);
                    } else if constexpr (KIND == CHAIN_OUT) {
                        const uint32_t w = (uint32_t)wave * d_words + (uint32_t)(r0 >> 1) + (uint32_t)i;
                        publish(mid + a.xo_off, w, v);
                        publish(mid + a.ro_off, w, lds_read<uint32_t>(done + (uint32_t)(16 + i) * 4u));
                    } else if constexpr (KIND == CHAIN_GATE_UP) {
                        publish(mid + a.h_off, (uint32_t)wave * (uint32_t)(N >> 2) + (uint32_t)(r0 >> 2) + (uint32_t)i, v);
                    } else if constexpr (KIND == CHAIN_DOWN) {
                        publish_tagged(a.ws + a.dpart_off, (uint32_t)(q * M + wave) * (uint32_t)N + (uint32_t)(r0 + i), __uint_as_float(v), (uint32_t)layer + 1u);
                    } else {
                        reinterpret_cast<uint32_t*>(a.out)[(((int64_t)wave * N + r0) >> 1) + i] = dead ? 0x7fff7fffu : v;
                    }
                }
            };
            auto read_sums = [&](float (&pt)[4]) {
#pragma unroll
                for (int i = 0; i < 4; ++i) pt[i] = lds_read<float>((red_r ^ parity ^ RED_FLIP) + (uint32_t)i * 512u);
            };
            auto two_blocks = [&](const u32x2& ca, const u32x2& cb, const u32x4* xa, float sa, float sb, f32x4& acc) {
                f32x4 c0v = {0.f, 0.f, 0.f, 0.f}, c1v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    u32x4 w0, w1;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t sel = 0x0c0c0400u | ((uint32_t)j << 8);
                        w0[j] = lds_read<uint32_t>(__builtin_amdgcn_perm(ca[h], col4, sel));
                        w1[j] = lds_read<uint32_t>(__builtin_amdgcn_perm(cb[h], col4, sel));
                    }
                    if constexpr (F16) {
                        c0v = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, xa[h]), __builtin_bit_cast(f16x8, w0), c0v, 0, 0, 0);
                        c1v = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, xa[2 + h]), __builtin_bit_cast(f16x8, w1), c1v, 0, 0, 0);
                    } else {
                        c0v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xa[h]), __builtin_bit_cast(bf16x8, w0), c0v, 0, 0, 0);
                        c1v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xa[2 + h]), __builtin_bit_cast(bf16x8, w1), c1v, 0, 0, 0);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = fmaf(c0v[i], sa, acc[i]);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = fmaf(c1v[i], sb, acc[i]);
            };

            for (int t = 0; t < tiles; ++t) {
                // This tile's codes were requested two tiles ago; the three requests of the tile before this one are younger.
                // Anything else under way only makes the wait longer.
                wait_vm<3>();
                u32x2 cd[4];
                const uint32_t at = c0 ^ slots;
#pragma unroll
                for (int b = 0; b < 4; ++b) cd[b] = lds_read<u32x2>(at ^ (uint32_t)(b << 5));
                const f32x4e am = lds_read<f32x4e>(aread + abs_now);
                float pt[4];
                if (t > 0 && reducer) read_sums(pt);
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                if (on) two_blocks(cd[0], cd[1], xv, am.x, am.y, acc);
                asm volatile("" ::"v"(cd[0]), "v"(cd[1]), "v"(cd[2]), "v"(cd[3]), "v"(am));
                request(slots, abs_now == 0 ? 2 * ABS_BYTES : abs_now - ABS_BYTES);
                advance();
                if (t > 0 && reducer) finish_tile(t - 1, pt);
                if (on) {
                    two_blocks(cd[2], cd[3], xv + 4, am.z, am.w, acc);
                    if constexpr (F16) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[i] *= unscale[i];
                    }
                }
                if (writes_sums) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) lds_write<float>((red_w ^ parity) + (uint32_t)i * RED_PLANE, acc[i]);
                }
                parity ^= RED_FLIP;
                slots ^= 2 * SLOT_BYTES;
                abs_now = abs_now == 2 * ABS_BYTES ? 0 : abs_now + ABS_BYTES;
                // the next tile's absmax, requested one tile ago (behind the last tile the wait for the next task's x sees to that)
                if (t + 1 < tiles) wait_vm<5>();
                barrier();
            }

            if (reducer) {
                float pt[4];
                read_sums(pt);
                finish_tile(tiles - 1, pt);
                leave();
            }

            if constexpr (KIND == CHAIN_OUT) {
                if (reducer) {
                    resid_ss = row16_down(lane < 16 ? resid_ss : 0.0f);
                    if (lane == 0) publish(mid + a.sso_off, (uint32_t)(wave * MAX_SLOTS + task), __float_as_uint(resid_ss));
                }
            }
        }
        if constexpr (KIND == CHAIN_DOWN) {
            // The K ranges of a task's rows meet, once every task of this workgroup has left its sums: each of their workgroups
            // finishes every ksplits-th row of x, a wave each.
            if constexpr (MODE == CHAIN_SLICES)
                for (int task = me; task < ntasks; task += G) {
                    const int ksplits = s.ksplits, q = ksplits == 1 ? 0 : task % ksplits, rt = ksplits == 1 ? task : task / ksplits;
                    const int r0 = rt * s.rows_per_task, r1 = min(N, r0 + s.rows_per_task);
                    const int m = q + wave * ksplits;
                    if (m >= M) continue;
                    uint8_t* const next = input_set(a, layer + 1);
                    const uint32_t tag = (uint32_t)layer + 1u;
                    const __amdgpu_buffer_rsrc_t pr = rsrc(a.ws + a.dpart_off, ksplits * M * N * 8);
                    const __amdgpu_buffer_rsrc_t rr = rsrc(mid + a.ro_off, M * (int)d_words * 4);
                    float ss = 0.0f;
                    for (int i = r0; i < r1; i += 64) {
                        const bool mine = i + lane < r1;
                        const int row = min(i + lane, r1 - 1);
                        const uint32_t nw = a.layers[l].norm_next[row];
                        u32x2 v[CHAIN_MAX_KSPLITS];
                        uint32_t rw;
                        spin([&]() {
                            bool missing = false;
#pragma unroll
                            for (int k = 0; k < CHAIN_MAX_KSPLITS; ++k)
                                v[k] = __builtin_amdgcn_raw_buffer_load_b64(pr, (uint32_t)((min(k, ksplits - 1) * M + m) * N + row) * 8u, 0, SC1);
                            rw = __builtin_amdgcn_raw_buffer_load_b32(rr, ((uint32_t)m * d_words + (uint32_t)(row >> 1)) * 4u, 0, SC1);
#pragma unroll
                            for (int k = 0; k < CHAIN_MAX_KSPLITS; ++k) missing = missing || v[k].y != tag;
                            return missing || rw == NOT_YET;
                        });
                        float sum = 0.0f;
#pragma unroll
                        for (int k = 0; k < CHAIN_MAX_KSPLITS; ++k)
                            if (k < ksplits) sum += __uint_as_float(v[k].x);
                        if (dead) sum = __uint_as_float(0x7fc00000u);
                        rw = (row & 1) ? rw >> 16 : rw & 0xffffu;
                        const float r = nf4x::resid_add(bf16_to_f32(rw), round_bf16(sum));
                        const uint32_t rb = f32_to_bf16(r), xb = f32_to_bf16(r * bf16_to_f32(nw));
                        const uint32_t ro = dpp<QUAD_X1>(rb), xo = dpp<QUAD_X1>(xb);
                        if (mine) {
                            const uint32_t w = (uint32_t)m * d_words + (uint32_t)(row >> 1);
                            if (!(lane & 1)) {
                                publish(next, w, xb | (xo << 16));
                                publish(next + a.r_off, w, rb | (ro << 16));
                            }
                            ss = fmaf(r, r, ss);
                        }
                    }
                    ss = sum_down(ss);
                    if (lane == 0) publish(next + a.ss_off, (uint32_t)(m * MAX_SLOTS + rt), __float_as_uint(ss));
                }
        }
        if (me >= ntasks) {
            asm volatile("" ::"v"(lut_hi), "v"(lut_lo));
            barrier();
        }
    };

    // Attention of one layer.  Task = (sequence, kv head, range of the cached keys): the four query heads of the group over those keys,
    // every sum taken in the order of decode_glue.hip's kernels; then each range merges a share of the columns.
    auto attention = [&](int l) {
        int splits, ntasks;
        {
            ARGS;
            splits = a.max_splits;
            ntasks = a.batch * a.n_kv * splits;
        }
        for (int task = me; task < ntasks; task += G) {
            ARGS;
            const int M = a.batch;
            const int layer = a.layer0 + l;
            uint8_t* const mid = layer_set(a, layer);
            const uint32_t tag = (uint32_t)layer + 1u;
            const int chunk = (p + splits - 1) / splits;
            const int split = task % splits, bh = task / splits, b = bh / a.n_kv, hk = bh % a.n_kv;
            const int lo = min(split * chunk, p), hi = min(lo + chunk, p), keys = hi - lo;
            const bool has_new = split == splits - 1;
            const int64_t cache_row0 = ((int64_t)b * a.n_kv + hk) * a.max_seq;
            uint16_t* const kc = a.kcache + (int64_t)l * a.cache_stride + cache_row0 * HD;
            uint16_t* const vc = a.vcache + (int64_t)l * a.cache_stride + cache_row0 * HD;
            const __amdgpu_buffer_rsrc_t kr = rsrc(kc + (int64_t)lo * HD, keys * HD * 2), vr = rsrc(vc + (int64_t)lo * HD, keys * HD * 2);
            // Two heads per half of the workgroup.  Keys: elements 16 sub .. + 15 of keys kslot, kslot + 64, ..; values: columns c4 .. + 3 of
            // rows vslot, vslot + 16, ..
            constexpr int KU = 3, VU = 10;
            u32x4 ka[KU], kb[KU];
            u32x2 vv[VU];
            auto load_keys = [&](int k0, int t9) {
#pragma unroll
                for (int u = 0; u < KU; ++u) {
                    if (k0 + u * 64 >= keys) break;  // uniform
                    const uint32_t at = (uint32_t)(k0 + u * 64 + (t9 >> 3)) * (HD * 2) + (uint32_t)(t9 & 7) * 32u;  // (past the range: zeros)
                    ka[u] = __builtin_amdgcn_raw_buffer_load_b128(kr, at, 0, 0);
                    kb[u] = __builtin_amdgcn_raw_buffer_load_b128(kr, at + 16, 0, 0);
                }
            };
            auto load_values = [&](int k0, int t9) {
#pragma unroll
                for (int u = 0; u < VU; ++u)
                    if (k0 + u * 16 < keys) vv[u] = __builtin_amdgcn_raw_buffer_load_b64(vr, (uint32_t)(k0 + u * 16 + (t9 >> 5)) * (HD * 2) + (uint32_t)(t9 & 31) * 8u, 0, 0);
            };
            {
                const int t9 = thread_id() & 511;
                load_keys(0, t9);
                load_values(0, t9);
            }
            // queries (and the new key and value) of this group: rotated into LDS
            const int tid1 = thread_id(), part = tid1 >> 7, j = tid1 & 127;
            if (part < (has_new ? 6 : 4)) {
                const __amdgpu_buffer_rsrc_t qr = rsrc(mid + a.qkv_off, M * a.shape[CHAIN_QKV].N * 2);
                const uint32_t qkv_words = (uint32_t)a.shape[CHAIN_QKV].N >> 1;
                const uint32_t head = part < 4 ? (uint32_t)(hk * REP + part) : (uint32_t)(a.n_head + hk + (part == 5 ? a.n_kv : 0));
                const uint32_t w = ((uint32_t)b * qkv_words + head * (HD / 2)) * 4u;
                uint32_t mine, other;
                spin([&]() {
                    mine = __builtin_amdgcn_raw_buffer_load_b32(qr, w + (uint32_t)(j >> 1) * 4u, 0, SC1);
                    other = __builtin_amdgcn_raw_buffer_load_b32(qr, w + (uint32_t)((j ^ (HD / 2)) >> 1) * 4u, 0, SC1);
                    return max(mine, other) == NOT_YET;
                });
                mine = (j & 1) ? mine >> 16 : mine & 0xffffu;
                other = (j & 1) ? other >> 16 : other & 0xffffu;
                uint32_t v = mine;
                if (part < 5) {
                    const float c = lds_read<float>(ROPE_OFF + j * 4), sn = lds_read<float>(ROPE_OFF + HD * 4 + j * 4);
                    const float sgn = j < HD / 2 ? -1.0f : 1.0f;
                    v = f32_to_bf16(bf16_to_f32(mine) * c + sgn * bf16_to_f32(other) * sn);
                }
                const float f = bf16_to_f32(v);
                lds_write<float>(DONE_OFF + part * (HD * 4) + j * 4, part < 4 ? f * rsqrtf((float)HD) : f);
                if (part == 4) kc[(int64_t)p * HD + j] = (uint16_t)v;
                if (part == 5) vc[(int64_t)p * HD + j] = (uint16_t)v;
            }
            barrier();

            {
                const int t9 = thread_id() & 511, sub = t9 & 7, kslot = t9 >> 3, pair = wave >> 3;
                float qv[2][16], top[2] = {-INFINITY, -INFINITY};
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const f32x4e v = lds_read<f32x4e>(DONE_OFF + (2 * pair + h) * (HD * 4) + sub * 64 + i * 16);
#pragma unroll
                        for (int e = 0; e < 4; ++e) qv[h][4 * i + e] = v[e];
                    }
                auto dots = [&](const float (&k16)[16], float (&dot)[2]) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        float d = 0.0f;
#pragma unroll
                        for (int i = 0; i < 16; ++i) d = fmaf(qv[h][i], k16[i], d);
                        d += __uint_as_float(dpp<QUAD_X1>(__float_as_uint(d)));
                        d += __uint_as_float(dpp<QUAD_X2>(__float_as_uint(d)));
                        dot[h] = d + __uint_as_float(dpp<HALF_MIRROR>(__float_as_uint(d)));
                    }
                };
                for (int k0 = 0; k0 < keys; k0 += KU * 64) {
#pragma unroll
                    for (int u = 0; u < KU; ++u) {
                        if (k0 + u * 64 >= keys) break;  // uniform
                        float k16[16], dot[2];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            k16[2 * e] = __uint_as_float(ka[u][e] << 16);
                            k16[2 * e + 1] = __uint_as_float(ka[u][e] & 0xffff0000u);
                            k16[8 + 2 * e] = __uint_as_float(kb[u][e] << 16);
                            k16[8 + 2 * e + 1] = __uint_as_float(kb[u][e] & 0xffff0000u);
                        }
                        dots(k16, dot);
                        const int key = k0 + u * 64 + kslot;
                        if (key < keys) {
                            const u32x2 v = {__float_as_uint(dot[0]), __float_as_uint(dot[1])};
                            if (sub == 0) lds_write<u32x2>(ps_addr(key) + pair * 8, v);
                            top[0] = fmaxf(top[0], dot[0]);
                            top[1] = fmaxf(top[1], dot[1]);
                        }
                    }
                    if (k0 + KU * 64 < keys) load_keys(k0 + KU * 64, t9);
                }
                if (has_new) {  // all lanes compute it, one stores it
                    float k16[16], dot[2];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const f32x4e v = lds_read<f32x4e>(DONE_OFF + REP * (HD * 4) + sub * 64 + i * 16);
#pragma unroll
                        for (int e = 0; e < 4; ++e) k16[4 * i + e] = v[e];
                    }
                    dots(k16, dot);
                    const u32x2 v = {__float_as_uint(dot[0]), __float_as_uint(dot[1])};
                    if (t9 == 0) lds_write<u32x2>(ps_addr(keys) + pair * 8, v);
                    top[0] = fmaxf(top[0], dot[0]);
                    top[1] = fmaxf(top[1], dot[1]);
                }
                auto larger_of = [](float x, float y) { return fmaxf(x, y); };
#pragma unroll
                for (int h = 0; h < 2; ++h) top[h] = across32(across16(row16(top[h], larger_of), larger_of), larger_of);
                const u32x2 v = {__float_as_uint(top[0]), __float_as_uint(top[1])};
                if ((t9 & 63) == 0) lds_write<u32x2>(ML_OFF + wave * 8, v);
            }
            barrier();
            // probabilities: head wave / 4, 256 threads a head
            const int all_keys = keys + (has_new ? 1 : 0);
            float top = -INFINITY;
            {
                const int tid2 = thread_id(), h = wave >> 2;
#pragma unroll
                for (int w = 0; w < 8; ++w) top = fmaxf(top, lds_read<float>(ML_OFF + ((h >> 1) * 8 + w) * 8 + (h & 1) * 4));
                float sum = 0.0f;
                for (int i = tid2 & 255; i < all_keys; i += 256) {
                    const float e = __expf(lds_read<float>(ps_addr(i) + h * 4) - top);
                    lds_write<float>(ps_addr(i) + h * 4, e);
                    sum += e;
                }
                sum = sum_down(sum);
                if ((tid2 & 63) == 0) lds_write<float>(ML_OFF + WAVES * 8 + wave * 4, sum);
            }
            barrier();
            {
                const int t9 = thread_id() & 511, c4 = (t9 & 31) * 4, vslot = t9 >> 5, pair = wave >> 3;
                float o[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                auto accumulate = [&](const float (&v4)[4], u32x2 w) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        o[0][i] = fmaf(__uint_as_float(w.x), v4[i], o[0][i]);
                        o[1][i] = fmaf(__uint_as_float(w.y), v4[i], o[1][i]);
                    }
                };
                for (int k0 = 0; k0 < keys; k0 += VU * 16) {
#pragma unroll
                    for (int u = 0; u < VU; ++u) {
                        const int key = k0 + u * 16 + vslot;
                        if (key < keys) {
                            const float v4[4] = {__uint_as_float(vv[u].x << 16), __uint_as_float(vv[u].x & 0xffff0000u), __uint_as_float(vv[u].y << 16),
                                                 __uint_as_float(vv[u].y & 0xffff0000u)};
                            accumulate(v4, lds_read<u32x2>(ps_addr(key) + pair * 8));
                        }
                    }
                    if (k0 + VU * 16 < keys) load_values(k0 + VU * 16, t9);
                }
                if (has_new && vslot == 0) {
                    const f32x4e v = lds_read<f32x4e>(DONE_OFF + (REP + 1) * (HD * 4) + c4 * 4);
                    const float v4[4] = {v[0], v[1], v[2], v[3]};
                    accumulate(v4, lds_read<u32x2>(ps_addr(keys) + pair * 8));
                }
                barrier();  // the probabilities are done with
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const f32x4e v = {o[h][0], o[h][1], o[h][2], o[h][3]};
                    lds_write<f32x4e>(red_addr((uint32_t)((vslot * REP + 2 * pair + h) * (HD * 4) + c4 * 4)), v);
                }
            }
            barrier();
            const int tid3 = thread_id();
            if (tid3 < REP * HD) {
                const int h = tid3 >> 7, col = tid3 & 127;
                const uint32_t slot = (uint32_t)((bh * splits + split) * CHAIN_ATTN_SLOT);
                float t = 0.0f;
#pragma unroll
                for (int v = 0; v < 16; ++v) t += lds_read<float>(red_addr((uint32_t)((v * REP + h) * (HD * 4) + col * 4)));
                publish_tagged(a.ws + a.apart_off, slot + (uint32_t)tid3, t, tag);
                if (col == 0) {
                    float mx = -INFINITY;
#pragma unroll
                    for (int w = 0; w < 8; ++w) mx = fmaxf(mx, lds_read<float>(ML_OFF + ((h >> 1) * 8 + w) * 8 + (h & 1) * 4));
                    const f32x4e su = lds_read<f32x4e>(ML_OFF + WAVES * 8 + h * 16);
                    publish_tagged(a.ws + a.apart_off, slot + REP * HD + 2 * h, mx, tag);
                    publish_tagged(a.ws + a.apart_off, slot + REP * HD + 2 * h + 1, ((su[0] + su[1]) + su[2]) + su[3], tag);
                }
            }
            if (task + G < ntasks) barrier();  // (the next task's queries go where the sums were)
        }
        for (int task = me; task < ntasks; task += G) {
            ARGS;
            const int tid = thread_id();
            const int M = a.batch;
            const uint32_t d_words = (uint32_t)a.d_model >> 1;
            const int layer = a.layer0 + l;
            uint8_t* const mid = layer_set(a, layer);
            const uint32_t tag = (uint32_t)layer + 1u;
            const int split = task % splits, bh = task / splits, b = bh / a.n_kv, hk = bh % a.n_kv;
            constexpr int PAIRS = REP * HD / 2;
            const int p0 = PAIRS * split / splits, p1 = PAIRS * (split + 1) / splits;
            if (p0 + wave * 64 >= p1) continue;
            const int pair = min(p0 + tid, p1 - 1);
            const __amdgpu_buffer_rsrc_t pr = rsrc(a.ws + a.apart_off, M * a.n_kv * splits * CHAIN_ATTN_SLOT * 8);
            u32x4 ov[CHAIN_MAX_SPLITS], ml[CHAIN_MAX_SPLITS];
            spin([&]() {
                bool missing = false;
#pragma unroll
                for (int i = 0; i < CHAIN_MAX_SPLITS; ++i) {
                    const uint32_t at = (uint32_t)((bh * splits + min(i, splits - 1)) * CHAIN_ATTN_SLOT) * 8u;
                    ov[i] = __builtin_amdgcn_raw_buffer_load_b128(pr, at + (uint32_t)pair * 16u, 0, SC1);
                    ml[i] = __builtin_amdgcn_raw_buffer_load_b128(pr, at + (uint32_t)(REP * HD + 2 * (pair >> 6)) * 8u, 0, SC1);
                }
#pragma unroll
                for (int i = 0; i < CHAIN_MAX_SPLITS; ++i) missing = missing || ov[i].y != tag || ov[i].w != tag || ml[i].y != tag || ml[i].w != tag;
                return missing;
            });
            float m = -INFINITY, den = 0.0f, na = 0.0f, nb = 0.0f;
#pragma unroll
            for (int i = 0; i < CHAIN_MAX_SPLITS; ++i)
                if (i < splits) m = fmaxf(m, __uint_as_float(ml[i].x));
#pragma unroll
            for (int i = 0; i < CHAIN_MAX_SPLITS; ++i)
                if (i < splits) {
                    const float mi = __uint_as_float(ml[i].x), w = mi == -INFINITY ? 0.0f : __expf(mi - m);
                    den = fmaf(w, __uint_as_float(ml[i].z), den);
                    na = fmaf(w, __uint_as_float(ov[i].x), na);
                    nb = fmaf(w, __uint_as_float(ov[i].z), nb);
                }
            if (dead) na = __uint_as_float(0x7fc00000u);
            if (p0 + tid < p1)
                publish(mid + a.y_off, (uint32_t)b * d_words + (uint32_t)(hk * REP) * (HD / 2) + (uint32_t)pair, f32_to_bf16(na / den) | (f32_to_bf16(nb / den) << 16));
        }
    };

    using Qkv = std::integral_constant<int, CHAIN_QKV>;
    using Out = std::integral_constant<int, CHAIN_OUT>;
    using GateUp = std::integral_constant<int, CHAIN_GATE_UP>;
    using Down = std::integral_constant<int, CHAIN_DOWN>;
    using Head = std::integral_constant<int, CHAIN_HEAD>;
    using Slices = std::integral_constant<int, CHAIN_SLICES>;
    using Rows = std::integral_constant<int, CHAIN_ROWS>;
    using Quads = std::integral_constant<int, CHAIN_QUADS>;
    asm volatile("" ::"v"(lut_hi), "v"(lut_lo));
    // Some were missing: the first that comes here settles how many share the next phases, and the stream goes on.  (Its requests past
    // the stop, of no bytes, name the same LDS.)
    auto settle = [&]() {
        ARGS;
        uint32_t v = 0;
        if ((thread_id() & 63) == 0) {
            uint32_t* const ctl = reinterpret_cast<uint32_t*>(a.ws + a.ctl_off);
            v = __hip_atomic_load(&ctl[CHAIN_CTL_MEMBERS + phase], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (v == 0) {
                const uint32_t here = __hip_atomic_load(&ctl[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint32_t count = min(here, (uint32_t)min(a.workgroups, a.first_members + phase * a.more_members));
                if (__hip_atomic_compare_exchange_strong(&ctl[CHAIN_CTL_MEMBERS + phase], &v, count, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                    v = count;
            }
        }
        G = uniform((int)v);
        settled();
        wait_vm<0>();
        st_phase = phase;
        st_task = me;
        prime();
    };
    const int n_layer = a.n_layer;
    const int from = phase;
    auto takes_part = [&](int this_phase) {
        if (this_phase < from) return false;  // (a late workgroup may begin in the middle of a layer)
        if (this_phase > stop) {
            phase = uniform(this_phase);
            settle();
        }
        return true;
    };
    for (int l = phase >> 2; l < n_layer; ++l) {
        ARGS;
        if (takes_part(4 * l)) {
            const float* const lut1 = a.layers[l].lin[1].lut;
            if constexpr (QKV_MODE == CHAIN_ROWS)
                linear(Qkv{}, Rows{}, l, lut1);
            else if constexpr (QKV_MODE == CHAIN_QUADS)
                linear(Qkv{}, Quads{}, l, lut1);
            else
                linear(Qkv{}, Slices{}, l, lut1);
            barrier();  // the attention's scratch is where the last sums were
        }
        if (takes_part(4 * l + 1)) {
            attention(l);
            barrier();  // ... and the other way round
            const float* const lut2 = a.layers[l].lin[2].lut;
            if constexpr (QKV_MODE == CHAIN_ROWS)
                linear(Out{}, Rows{}, l, lut2);
            else
                linear(Out{}, Slices{}, l, lut2);
        }
        if (takes_part(4 * l + 2)) linear(GateUp{}, Slices{}, l, a.layers[l].lin[3].lut);
        takes_part(4 * l + 3);
        const float* const next = l + 1 < a.n_layer ? a.layers[l + 1].lin[0].lut : a.with_head ? a.head.lut : nullptr;
        if constexpr (QKV_MODE == CHAIN_ROWS)
            linear(Down{}, Rows{}, l, next);
        else
            linear(Down{}, Slices{}, l, next);
    }
    if (a.with_head) {
        takes_part(head_phase);
        linear(Head{}, Slices{}, n_layer, nullptr);
    }
    wait_vm<0>();  // requests past the end of the stream still name this workgroup's LDS
#endif
}

// Ahead of the step: scratch that nothing has been written to yet reads as NOT_YET (tagged values: layer 0, control words: 0), and
// the first layer's input is there: r = x and its RMSNorm (the sums of decode_glue.hip's add_rmsnorm_kernel).
constexpr int BEGIN_THREADS = 512;
__global__ __launch_bounds__(BEGIN_THREADS) void chain_begin_kernel(const uint16_t* x, const uint16_t* norm, float eps, int d, int batch, uint8_t* ws,
                                                                     int64_t zero_bytes, int64_t unset_bytes, int64_t r_off) {
    const int tid = threadIdx.x;
    if ((int)blockIdx.x < batch) {
        __shared__ float part[BEGIN_THREADS / 64];
        uint8_t* const in = ws + zero_bytes + unset_bytes;
        const int row = blockIdx.x;
        const bool on = tid * 8 < d;
        float ss = 0.0f;
        u32x4 xv = {0, 0, 0, 0}, wv = {0, 0, 0, 0};
        if (on) {
            xv = *reinterpret_cast<const u32x4*>(x + (int64_t)row * d + tid * 8);
            wv = *reinterpret_cast<const u32x4*>(norm + tid * 8);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float r0 = __uint_as_float(xv[e] << 16), r1 = __uint_as_float(xv[e] & 0xffff0000u);
                ss = fmaf(r0, r0, ss);
                ss = fmaf(r1, r1, ss);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
        if ((tid & 63) == 0) part[tid >> 6] = ss;
        __syncthreads();
        float tot = 0.0f;
#pragma unroll
        for (int w = 0; w < BEGIN_THREADS / 64; ++w) tot += part[w];
        const float rstd = rsqrtf(tot / (float)d + eps);
        if (on) {
            u32x4 ov, rv;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float r0 = __uint_as_float(xv[e] << 16), r1 = __uint_as_float(xv[e] & 0xffff0000u);
                ov[e] = f32_to_bf16(r0 * rstd * __uint_as_float(wv[e] << 16)) | (f32_to_bf16(r1 * rstd * __uint_as_float(wv[e] & 0xffff0000u)) << 16);
                if (ov[e] == 0xffffffffu) ov[e] = 0xfffffffeu;
                rv[e] = xv[e] == 0xffffffffu ? 0xfffffffeu : xv[e];
            }
            *reinterpret_cast<u32x4*>(in + ((int64_t)row * d + tid * 8) * 2) = ov;
            *reinterpret_cast<u32x4*>(in + r_off + ((int64_t)row * d + tid * 8) * 2) = rv;
        }
        return;
    }
    const int64_t step = (int64_t)(gridDim.x - batch) * BEGIN_THREADS * 16;
    for (int64_t i = ((int64_t)(blockIdx.x - batch) * BEGIN_THREADS + tid) * 16; i < zero_bytes + unset_bytes; i += step) {
        const uint32_t v = i < zero_bytes ? 0u : 0xffffffffu;
        *reinterpret_cast<u32x4*>(ws + i) = u32x4{v, v, v, v};
    }
}

int chip_cus() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) {
        (void)hipGetLastError();
        return 256;
    }
    return cus < MAX_SLOTS ? cus : MAX_SLOTS;
}

bool deal(ChainShape& s, int mode, int64_t N, int64_t K, int workgroups) {
    if (N <= 0 || N % 8 || K <= 0 || K % SLICE_K || K > CHAIN_MAX_KSPLITS * WAVES * SLICE_K || N * K / 2 >= INT32_MAX) return false;
    const int slices = (int)(K / SLICE_K);
    s.N = (int)N;
    s.K = (int)K;
    s.mode = mode;
    s.ksplits = mode == CHAIN_SLICES ? (slices + WAVES - 1) / WAVES : 1;
    s.slices_per_split = (slices + s.ksplits - 1) / s.ksplits;
    const int part_k = mode == CHAIN_ROWS ? 2048 : 512;
    s.parts = mode == CHAIN_SLICES ? WAVES : (int)((K + part_k - 1) / part_k);
    s.lanes = WAVES / s.parts;
    s.tile_rows = mode == CHAIN_SLICES ? 16 : (mode == CHAIN_ROWS ? 2 : 8) * s.lanes;
    const int shares = workgroups / s.ksplits, eights = (int)(N / 8);
    if (shares < 1 || s.lanes < 1) return false;
    s.rows_per_task = (eights + shares - 1) / shares * 8;
    s.row_tasks = ((int)N + s.rows_per_task - 1) / s.rows_per_task;
    s.sums = mode == CHAIN_ROWS ? eights : s.row_tasks;
    // rows: a lane of one wave finishes a row; quads: (row, part of K, row of x) in LDS
    return mode == CHAIN_SLICES || s.rows_per_task <= 64;
}

// Everything but the pointers; false: not served
bool plan(ChainArgs& a, size_t& bytes, int64_t batch, int64_t n_layer, int64_t d_model, int n_head, int n_kv_head, int64_t d_ff, int64_t vocab,
          int64_t max_seq, int workgroups) {
    if (batch < 1 || batch > WAVES || n_layer < 1 || n_layer > 1024 || max_seq < 1 || max_seq > 32768) return false;
    if (n_head < 1 || n_kv_head < 1 || n_head != REP * n_kv_head || d_model != (int64_t)n_head * HD || d_model > WAVES * SLICE_K) return false;
    if (d_ff < 1 || d_ff > (1 << 20) || vocab < 1 || vocab > (1 << 24)) return false;
    // (modes: what the launch-by-launch step runs at Llama-3-8B's shapes, so that the two give the same bits there)
    const int one = batch == 1 ? CHAIN_ROWS : CHAIN_SLICES;
    const int qkv = batch >= 5 && batch <= 8 && d_model % 512 == 0 ? CHAIN_QUADS : one;
    if (!deal(a.shape[CHAIN_QKV], qkv, (int64_t)(n_head + 2 * n_kv_head) * HD, d_model, workgroups) || !deal(a.shape[CHAIN_OUT], one, d_model, d_model, workgroups) ||
        !deal(a.shape[CHAIN_GATE_UP], CHAIN_SLICES, 2 * d_ff, d_model, workgroups) || !deal(a.shape[CHAIN_DOWN], one, d_model, d_ff, workgroups) ||
        !deal(a.shape[CHAIN_HEAD], CHAIN_SLICES, vocab, d_model, workgroups))
        return false;
    if (a.shape[CHAIN_OUT].sums > MAX_SLOTS || a.shape[CHAIN_DOWN].sums > MAX_SLOTS) return false;
    // a wave keeps the residual of one tile of the output projection, and LDS DONE_WORDS words of a task
    if (a.shape[CHAIN_OUT].rows_per_task > 16 || a.shape[CHAIN_QKV].rows_per_task > 2 * DONE_WORDS || a.shape[CHAIN_GATE_UP].rows_per_task > 4 * DONE_WORDS ||
        a.shape[CHAIN_DOWN].rows_per_task > DONE_WORDS || a.shape[CHAIN_HEAD].rows_per_task > 2 * DONE_WORDS)
        return false;
    const int64_t M = batch;
    a.batch = (int)batch;
    a.model_layers = (int)n_layer;
    a.n_head = n_head;
    a.n_kv = n_kv_head;
    a.max_seq = (int)max_seq;
    a.d_model = (int)d_model;
    const int64_t groups = M * n_kv_head;
    // ranges of keys: decode_glue.hip's
    a.max_splits = (int)(1024 / (M * n_head));
    if (a.max_splits < 2) return false;
    if (a.max_splits > CHAIN_MAX_SPLITS) a.max_splits = CHAIN_MAX_SPLITS;
    if ((max_seq + a.max_splits - 2) / a.max_splits + 1 > PS_MAX) return false;  // LDS holds the scores of a range
    int64_t at = 0;
    auto take = [&](int64_t n) {
        const int64_t r = at;
        at += (n + 255) & ~(int64_t)255;
        return r;
    };
    a.ctl_off = (int)take((n_layer + CHAIN_LAYERS - 1) / CHAIN_LAYERS * CHAIN_CTL_BYTES);
    a.apart_off = (int)take(groups * a.max_splits * CHAIN_ATTN_SLOT * 8);
    a.dpart_off = (int)take(a.shape[CHAIN_DOWN].ksplits * M * d_model * 8);
    a.layer_off = at;
    at = 0;
    a.qkv_off = (int)take(M * a.shape[CHAIN_QKV].N * 2);
    a.y_off = (int)take(M * d_model * 2);
    a.xo_off = (int)take(M * d_model * 2);
    a.ro_off = (int)take(M * d_model * 2);
    a.sso_off = (int)take(M * MAX_SLOTS * 4);
    a.h_off = (int)take(M * d_ff * 2);
    a.layer_stride = at;
    at = 0;
    take(M * d_model * 2);
    a.r_off = (int)take(M * d_model * 2);
    a.ss_off = (int)take(M * MAX_SLOTS * 4);
    a.in_stride = at;
    a.in_off = a.layer_off + n_layer * a.layer_stride;
    bytes = (size_t)(a.in_off + (n_layer + 1) * a.in_stride);
    return true;
}

}  // namespace

// (the error text lives with the other entry points)
extern "C" int nf4hip_decode_fail(const char* text);

extern "C" {

__attribute__((visibility("default"))) size_t nf4hip_decode_chain_workspace_bytes(int64_t batch, int64_t n_layer, int64_t d_model, int n_head,
                                                                                 int n_kv_head, int64_t d_ff, int64_t vocab, int64_t max_seq) {
    ChainArgs a;
    size_t bytes = 0;
    return plan(a, bytes, batch, n_layer, d_model, n_head, n_kv_head, d_ff, vocab, max_seq, chip_cus()) ? bytes : 0;
}

__attribute__((visibility("default"))) int nf4hip_decode_chain_joined(const void* x, const void* const* layers, const void* const* head, const void* norm_first,
                                                              float eps, const int64_t* pos, const float* cos_t, const float* sin_t, void* kcache,
                                                              void* vcache, int64_t batch, int64_t n_layer, int64_t d_model, int n_head, int n_kv_head,
                                                              int64_t d_ff, int64_t vocab, int64_t max_seq, int max_workgroups, int first_members,
                                                              int more_members, void* out, void* workspace, size_t workspace_bytes, void* stream) {
    if (first_members < 0 || more_members < 0 || more_members > (1 << 16)) return nf4hip_decode_fail("nf4hip_decode_chain: a negative or too large number of workgroups");
    if (!x || !layers || !head || !norm_first || !pos || !cos_t || !sin_t || !kcache || !vcache || !out) return nf4hip_decode_fail("nf4hip_decode_chain: null pointer");
    ChainArgs a;
    size_t need = 0;
    const int workgroups = chip_cus();
    if (!plan(a, need, batch, n_layer, d_model, n_head, n_kv_head, d_ff, vocab, max_seq, workgroups))
        return nf4hip_decode_fail("nf4hip_decode_chain: a shape that is not served (nf4hip_decode_chain_workspace_bytes answers 0)");
    if (!workspace || workspace_bytes < need) return nf4hip_decode_fail("nf4hip_decode_chain: a workspace of nf4hip_decode_chain_workspace_bytes() bytes is required");
    auto misaligned = [](const void* p) { return p == nullptr || (reinterpret_cast<uintptr_t>(p) & 15u) != 0; };
    bool bad = misaligned(x) || misaligned(norm_first) || misaligned(kcache) || misaligned(vcache) || misaligned(out) || misaligned(workspace);
    for (int64_t i = 0; i < n_layer * 14; ++i) bad = bad || misaligned(layers[i]);
    for (int i = 0; i < 3; ++i) bad = bad || misaligned(head[i]);
    if (bad) return nf4hip_decode_fail("nf4hip_decode_chain: a pointer is null or not 16-byte aligned");
    // allow the whole 160 KB of LDS once per device
    static bool ready[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nf4hip_decode_fail("nf4hip_decode_chain: no current device");
    if (!ready[dev]) {
        for (const auto kernel : {chain_kernel<CHAIN_SLICES>, chain_kernel<CHAIN_ROWS>, chain_kernel<CHAIN_QUADS>})
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, SMEM_BYTES) != hipSuccess)
                return nf4hip_decode_fail("nf4hip_decode_chain: LDS size");
        ready[dev] = true;
    }
    const int mode = a.shape[CHAIN_QKV].mode;
    const auto kernel = mode == CHAIN_ROWS ? chain_kernel<CHAIN_ROWS> : mode == CHAIN_QUADS ? chain_kernel<CHAIN_QUADS> : chain_kernel<CHAIN_SLICES>;
    a.eps = eps;
    a.pos = pos;
    a.cos_t = cos_t;
    a.sin_t = sin_t;
    a.cache_stride = batch * n_kv_head * max_seq * HD;
    a.out = static_cast<uint16_t*>(out);
    a.ws = static_cast<uint8_t*>(workspace);
    auto linear = [](const void* const* p) {
        return ChainLinear{static_cast<const uint8_t*>(p[0]), static_cast<const float*>(p[1]), static_cast<const float*>(p[2])};
    };
    a.head = linear(head);
    a.workgroups = max_workgroups > 0 && max_workgroups < workgroups ? max_workgroups : workgroups;
    a.first_members = first_members > 0 && first_members < a.workgroups ? first_members : a.workgroups;
    a.more_members = more_members;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t zero_bytes = a.layer_off, unset_bytes = (int64_t)need - a.in_stride - zero_bytes;
    const int64_t fill_wgs = (zero_bytes + unset_bytes + BEGIN_THREADS * 64 - 1) / (BEGIN_THREADS * 64);
    hipLaunchKernelGGL(chain_begin_kernel, dim3((unsigned)(batch + (fill_wgs < 1024 ? fill_wgs : 1024))), dim3(BEGIN_THREADS), 0, s, static_cast<const uint16_t*>(x),
                       static_cast<const uint16_t*>(norm_first), eps, (int)d_model, (int)batch, a.ws, zero_bytes, unset_bytes, (int64_t)a.r_off);
    for (int64_t l0 = 0; l0 < n_layer; l0 += CHAIN_LAYERS) {
        a.layer0 = (int)l0;
        a.n_layer = (int)(n_layer - l0 < CHAIN_LAYERS ? n_layer - l0 : CHAIN_LAYERS);
        a.with_head = l0 + a.n_layer == n_layer;
        a.ctl_off = (int)(l0 / CHAIN_LAYERS * CHAIN_CTL_BYTES);
        a.kcache = static_cast<uint16_t*>(kcache) + l0 * a.cache_stride;
        a.vcache = static_cast<uint16_t*>(vcache) + l0 * a.cache_stride;
        for (int i = 0; i < a.n_layer; ++i) {
            const void* const* p = layers + (l0 + i) * 14;
            for (int j = 0; j < 4; ++j) a.layers[i].lin[j] = linear(p + 3 * j);
            a.layers[i].norm_mid = static_cast<const uint16_t*>(p[12]);
            a.layers[i].norm_next = static_cast<const uint16_t*>(p[13]);
        }
        hipLaunchKernelGGL(kernel, dim3((unsigned)a.workgroups), dim3(THREADS), SMEM_BYTES, s, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : nf4hip_decode_fail("nf4hip_decode_chain: launch failed");
}

__attribute__((visibility("default"))) int nf4hip_decode_chain(const void* x, const void* const* layers, const void* const* head, const void* norm_first,
                                                              float eps, const int64_t* pos, const float* cos_t, const float* sin_t, void* kcache,
                                                              void* vcache, int64_t batch, int64_t n_layer, int64_t d_model, int n_head, int n_kv_head,
                                                              int64_t d_ff, int64_t vocab, int64_t max_seq, int max_workgroups, void* out,
                                                              void* workspace, size_t workspace_bytes, void* stream) {
    return nf4hip_decode_chain_joined(x, layers, head, norm_first, eps, pos, cos_t, sin_t, kcache, vcache, batch, n_layer, d_model, n_head, n_kv_head, d_ff,
                                      vocab, max_seq, max_workgroups, 0, 0, out, workspace, workspace_bytes, stream);
}

}  // extern "C"
