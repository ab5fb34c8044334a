// Level-scheduled segment scan kernels for float activations.
#include "segment_level.hpp"

namespace ramnet {

hipError_t launch_level_f32(const SegmentJob &job, const LevelGeom &geo, int vec, int km, bool full, hipStream_t stream) {
    return level_dispatch<float>(job, geo, vec, km, full, stream);
}

}  // namespace ramnet
