// Level-scheduled segment scan kernels for bf16_t activations.
#include "segment_level.hpp"

namespace ramnet {

hipError_t launch_level_bf16(const SegmentJob &job, const LevelGeom &geo, int vec, int km, bool full, hipStream_t stream) {
    return level_dispatch<bf16_t>(job, geo, vec, km, full, stream);
}

}  // namespace ramnet
