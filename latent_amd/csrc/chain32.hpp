// Host interface of the fp32 matrix-core chain over the row layout (chain32.hip).
#pragma once

#include <stddef.h>

#include "common.hpp"

namespace latent {
namespace chain32 {

constexpr int64_t kMinPairs = 32, kMaxPairs = 512;  // routed pairs of a call
constexpr int64_t kMaxExpert = 512;

constexpr int kUnitPairs = 4;  // pairs of one expert a workgroup multiplies together

// Written by the prep kernel: units of at most kUnitPairs pairs of one expert.
struct Grouping {
  const int* meta;        // [4] units
  const int4* unit_info;  // {expert, first pair, pairs, 0}
  const int* unit_tok;    // [units][kUnitPairs] token of each unit row (0 past the unit's pairs)
  const int* pos_of;      // [T*K] grouped position of each routed slot
  const float* pair_w;
};

// Scratch inside the caller's workspace, after the grouping.
struct Layout {
  size_t units, pos_of, part_a, part_c, y, total;
  int a_rows, n_a;  // rows of d per phase A item, items per unit and factor
  int n_c, n_d;     // column chunks of ff and of d
};

bool supported(const latent_moe_args& a);
int64_t max_units(const latent_moe_args& a);
Layout layout_for(const latent_moe_args& a);
// Runs after the prep kernel on the same stream.
int forward(const latent_moe_args& a, const Factor* fac, const Grouping& g, char* scratch, hipStream_t s);

}  // namespace chain32
}  // namespace latent
