// FP8 block-scaled projections of nine or more activation rows
// (fp8_batch.hip), launched by the entry points of fp8_gemv.hip.
#pragma once

#include <cstdint>

#include "common.h"
#include "fp8_plan.h"

namespace plm {

constexpr int kBatchOuts = 8;     // weights with outputs of their own in one call
constexpr int kBatchGroups = 64;  // weights per launch (their addresses travel as kernel arguments)

// Where the tokens of a grouped launch are, on the device (all indexed by
// the launch's first group + its group): group g has count[g] tokens, its
// t-th is activation row list[g * list_ld + t], and its results start at
// output row base[g].
struct BatchGroups {
    const int* count = nullptr;  // null: every group has every activation row, in order
    const int* base = nullptr;
    const int* list = nullptr;   // null: activation row base[g] + t
    int64_t list_ld = 0;
};

// out[g][t][row] = W_g[row] . x_t (or silu(gate) * up as bf16 hi / lo planes).
// Dense (groups.count null): group g's results are output rows g * m + t.
struct BatchRows {
    const uint8_t* w[2][kBatchGroups];  // w[1]: the up weights of a SiLU launch
    const float* s[2][kBatchGroups];
    const float* x = nullptr;           // activations, one of: fp32,
    const uint16_t* xb = nullptr;       //   bf16,
    const uint16_t* xhi = nullptr;      //   the hi / lo planes of a SiLU launch (its output rows)
    const uint16_t* xlo = nullptr;
    int64_t x_stride = 0;
    float* out = nullptr;               // element (output row, row) at output row * rows + row, or
    uint16_t* hhi = nullptr;            //   SiLU: the planes, same layout
    uint16_t* hlo = nullptr;
    int64_t rows = 0;
    int64_t K = 0;
    int64_t scale_cols = 0;
    int64_t m = 0;                      // activation rows (grouped: of the whole call)
    int ngroups = 0;
    int waves = 0;                      // K blocks b = w, w + waves, ... are wave w's
    bool tiled = false;                 // weights in 8-row tiles
    BatchGroups groups;
    // outs[0] set: ngroups weights w[0][g] of out_rows[g] rows each (rows: the
    // most), every activation row of each to outs[g][m][out_rows[g]]
    float* outs[kBatchOuts] = {};
    int64_t out_rows[kBatchOuts] = {};
};

int fp8_batch_rows(const BatchRows& p, hipStream_t st);

// Prompt chunks (fp8_panel_kernel), the same bits: the linears of p.outs over
// one packed copy of the activations, and the SwiGLU MLP (gate_up's two
// weights, then down's).
int fp8_panel_linear(const BatchRows& p, hipStream_t st);
int fp8_panel_mlp(const BatchRows& gate_up, const BatchRows& down, hipStream_t st);

// Waves of the down phase over nb K blocks (one group's): see fp8_down_kernel.
constexpr int kBatchDownWaves = 16;

// The routed experts on the (expert, row, weight) pairs of a prompt chunk:
// out[r] = sum over r's experts of weight * expert(x_r).  Weights 16-byte
// aligned, inter and hid multiples of 16.
struct PairProblem {
    const uint8_t* const* w[3];  // gate, up, down: one address per expert
    const float* const* s[3];
    const float* x = nullptr;    // activations [batch][hid], fp32 or
    const uint16_t* xb = nullptr;
    const int64_t* items = nullptr;
    const int64_t* rows = nullptr;
    const float* weights = nullptr;
    float* out = nullptr;
    int* bad = nullptr;  // pairs with an index out of range are left out and, when not null, counted here
    int64_t experts = 0, pairs = 0, batch = 0, inter = 0, hid = 0, gsc = 0, dsc = 0;
    int gate_waves = 0;
};

int fp8_batch_pairs(const PairProblem& p, hipStream_t st);

}  // namespace plm
