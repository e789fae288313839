// Batched contraction of a tree network at many points, vertex by vertex
// (tree.hip; used by the evaluate of trees and wide chains).
#pragma once
#include "qtt_internal.h"

// Evaluate float64 networks of any tree (nv >= 1, any coordinates): device
// points and values, queued on the context's stream.
int launch_eval_tree(qtt_ctx* ctx, qtt_net* net, const double* xs, int64_t npts, double* out);

// Gradient of sum_m ybar_m f(x_m) with respect to the cores of a float64 chain
// with bonds of at most 64 (device pointers; waits for the result).  *inf_weight
// is set if a weight is infinite: the caller then takes a kernel that multiplies
// by the weight last (see grad_weight_kernel).
int launch_grad_chain(qtt_ctx* ctx, qtt_net* net, const double* xs, const double* ybar, int64_t npts, double* grad,
                      bool* inf_weight);
