// mc_advance_kernel for replicas with 33 to 68 k-vectors per thread (K up to 17408), but for
// the FP32 form without a cell list (compiled with mc_batch.hip's flags).
#include "mc_advance.hpp"

namespace fmc {

void launch_wide(bool cells, bool f32, int grid, size_t lds, hipStream_t st, ReplicaState* s, const long long* m,
                 TraceEntry* tr, int cap, const LadderRun* lr, const ReplicaMap& map) {
    if (cells && f32) launch_advance<68, true, true>(grid, lds, st, s, m, tr, cap, lr, map);
    else if (cells) launch_advance<68, true, false>(grid, lds, st, s, m, tr, cap, lr, map);
    else launch_advance<68, false, false>(grid, lds, st, s, m, tr, cap, lr, map);
}

} // namespace fmc
