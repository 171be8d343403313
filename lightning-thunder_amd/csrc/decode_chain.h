// Plan of the one-launch decode step (decode_chain.hip): what its host side hands to its kernels.
#pragma once

#include <stdint.h>

enum : int { CHAIN_QKV = 0, CHAIN_OUT = 1, CHAIN_GATE_UP = 2, CHAIN_DOWN = 3, CHAIN_HEAD = 4, CHAIN_KINDS = 5 };

// How a tile is multiplied: sixteen waves with 256 k each of sixteen rows (nf4_gemv_stage.hip); with one row of x, a lane per 32 k of a
// row (nf4_gemv_rows.hip); four rows per lane quad (nf4_gemv_quad.hip)
enum : int { CHAIN_SLICES = 0, CHAIN_ROWS = 1, CHAIN_QUADS = 2 };

constexpr int CHAIN_LAYERS = 32;      // layers of one launch: their pointers fit the 4 KB of kernel arguments
constexpr int CHAIN_MAX_KSPLITS = 4;  // K ranges of the down projection: sixteen waves of 256 k each
constexpr int CHAIN_MAX_SPLITS = 8;   // ranges of cached keys
constexpr int CHAIN_ATTN_SLOT = 4 * 128 + 8;  // tagged values one range of keys leaves: output, (maximum, sum) of four heads
constexpr int CHAIN_MAX_POLLS = 1 << 21;      // seconds: what is waited for comes from workgroups that are running
constexpr uint64_t CHAIN_MUSTER_TICKS = 5000;  // of the 100 MHz clock
constexpr int CHAIN_CTL_BYTES = 1024;           // control words of a launch: arrivals, then members of each phase
constexpr int CHAIN_CTL_MEMBERS = 32;           // first of those
static_assert((CHAIN_CTL_MEMBERS + 4 * CHAIN_LAYERS + 1) * 4 <= CHAIN_CTL_BYTES, "a word per phase");

struct ChainLinear {
    const uint8_t* codes;
    const float* absmax;
    const float* lut;
};
struct ChainLayer {
    ChainLinear lin[4];
    const uint16_t* norm_mid;   // of the norm between attention and MLP
    const uint16_t* norm_next;  // of the next layer's first norm, or the final one
};
// A linear [N, K] is dealt to the workgroups in tasks: `rows_per_task` weight rows (a multiple of 8) of one of `ksplits` K
// ranges, each of `slices_per_split` 256-k slices (<= 16; the last range may hold fewer).
struct ChainShape {
    int N, K, rows_per_task, row_tasks, ksplits, slices_per_split;
    int mode, tile_rows;  // how a tile is multiplied, and how many rows it has
    int parts, lanes;     // CHAIN_ROWS, CHAIN_QUADS: waves along K, groups of them
    int sums;             // partial sums of squares of a row of x that its tasks leave
};
struct ChainArgs {
    ChainLayer layers[CHAIN_LAYERS];
    ChainLinear head;
    const int64_t* pos;
    const float* cos_t;
    const float* sin_t;
    uint16_t* kcache;  // of the launch's first layer
    uint16_t* vcache;
    int64_t cache_stride;  // elements of a layer's cache
    uint16_t* out;
    uint8_t* ws;
    ChainShape shape[CHAIN_KINDS];
    int workgroups;                  // of the launch
    int first_members, more_members;  // at most first_members + phase * more_members of them take part in a phase
    int batch, n_layer, layer0, model_layers, with_head, n_head, n_kv, max_seq, d_model, max_splits;
    float eps;
    // byte offsets in the workspace; *_off of sets: inside the set of a layer
    int ctl_off, apart_off, dpart_off;
    int64_t in_off, in_stride, layer_off, layer_stride;
    int r_off, ss_off;                                     // of an input set; it begins with bf16(r * norm weight)
    int qkv_off, y_off, xo_off, ro_off, sso_off, h_off;    // of a layer's set
};
static_assert(sizeof(ChainArgs) <= 4096, "kernel arguments");
