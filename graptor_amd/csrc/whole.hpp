// whole.hpp -- BFSLVLv and CCv runs of small graphs without the host between
// their steps (whole.hip).
#pragma once
#include "../../include/gpr.h"
#include <stddef.h>

namespace gpr {

// Bytes of pinned memory that a run reports its progress in (gpr_graph::wline).
constexpr size_t WHOLE_LINE = 128;

// Whether a run with these options takes that form: the benchmark's default
// schedule, nothing traced or profiled, a graph of at most whole_edges edges
// (symmetric for CC).
bool whole_run(const gpr_graph *g, const gpr_run_opts &o, bool cc);
// levels / labels: n results in original IDs, or null to leave them on the
// device.
int whole_bfs(gpr_graph *g, uint32_t start, float threshold_pct, uint32_t *levels, gpr_run_info *info);
int whole_cc(gpr_graph *g, uint32_t *labels, gpr_run_info *info);

} // namespace gpr
