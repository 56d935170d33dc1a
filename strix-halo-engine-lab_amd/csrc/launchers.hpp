// Launches whose kernels live in translation units of their own (they compile in parallel).
#pragma once
#include "route_wave.hpp"

namespace strix950 {

// route.hip: logits of a batch past the decode sizes into a.scores; softmax, selection and weights of every row of a.scores
void launch_route_batch_logits(const RouteArgs& a, hipStream_t st);
void launch_route_select(const RouteArgs& a, hipStream_t st);

}  // namespace strix950
