// Gate of the filter kernels that come in two forms: on the pairs themselves,
// and through a table of the filter over the distance (filter_table.hip).
//
// The table's check (table_check_kernel) leaves eight words per block: for
// W, dW/dd, H, dH/dd (H = act(W1 g + b1) times the CFConv envelope) the
// largest error of interpolating every second node from its neighbours at
// twice the spacing, and the largest magnitude, as the bits of non-negative
// floats (a NaN is larger than every number and fails the comparison), and
// one word for the largest change of a first-layer pre-activation between
// neighbouring nodes.  The interpolation used has half that spacing, so its
// error is 2^-4 of the measured one: at the bounds below 2.5e-7 of the largest
// value and 1e-6 of the largest derivative -- the rounding of the fp32
// evaluation itself (3.4e-7 and 6e-7; the split-fp16 kernels' derivative:
// 4.7e-6).  The cutoff distance, up to 1/8 of a cell past the last node, has
// its error measured as it is used: of the truncation of the cells beside the
// ends, and compared with the same bounds.
//
// Basis functions narrower than the spacing, which could lie between two nodes
// unseen, set the last word to infinity; of wider ones the nodes see every
// feature, and a pre-activation that changes by less than 1/4 per node leaves
// the activation none of its own.  So do weights of 65504 or more, which the
// split kernels report.
#pragma once

#include "common.h"

constexpr int kGateWords = 12;
constexpr float kGateValueTol = 4e-6f;
constexpr float kGateDerivTol = 1.6e-5f;
constexpr float kGateSlope = 0.25f;

struct FilterGate {
  const unsigned* words;  // nullptr: the kernel always runs
  int want;               // run when the table serves (1) or does not (0)
};

__device__ __forceinline__ bool filter_table_serves(const unsigned* __restrict__ g) {
  // & and not &&: the words are read together, not one after the other
  return (__uint_as_float(g[0]) <= kGateValueTol * __uint_as_float(g[4])) &
         (__uint_as_float(g[1]) <= kGateDerivTol * __uint_as_float(g[5])) &
         (__uint_as_float(g[2]) <= kGateValueTol * __uint_as_float(g[6])) &
         (__uint_as_float(g[3]) <= kGateDerivTol * __uint_as_float(g[7])) &
         (__uint_as_float(g[8]) <= kGateSlope);
}

__device__ __forceinline__ bool gate_closed(const FilterGate& gate) {
  return gate.words != nullptr && filter_table_serves(gate.words) != (gate.want != 0);
}
