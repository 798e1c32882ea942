// norm_route.hip for the entry points that make rows (sublayer_ops.hip, stream_ops.hip): 0, or the error; what the rows themselves need has been checked
#pragma once
#include "common.hpp"

int m40_norm_add_route(hipStream_t stream, const M40llmNormAdd& n);
int m40_stream_update_route(hipStream_t stream, const M40llmStreamUpdate& u);
// experts.hip: whether a route is refused (its logits aside)
bool m40_route_refused(const M40llmRoute& r);
