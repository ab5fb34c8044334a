// Level-scheduled segment scan kernels for _Float16 activations.
#include "segment_level.hpp"

namespace ramnet {

hipError_t launch_level_f16(const SegmentJob &job, const LevelGeom &geo, int vec, int km, bool full, hipStream_t stream) {
    return level_dispatch<_Float16>(job, geo, vec, km, full, stream);
}

}  // namespace ramnet
