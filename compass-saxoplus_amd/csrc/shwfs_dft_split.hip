// MFMA spot kernels, split-FP16 operands, windows of up to 16 points.
#include "shwfs_image_dft.hpp"

namespace shwfs {
template int32_t launch_dft_pq<kSplitFp16, 1>(const ImageParams&, int, hipStream_t, const void*,
                                              const BgParams&);
template int32_t launch_dft_tasks_pq<kSplitFp16, 1>(int, bool, int, bool, const BatchTask*,
                                                    const TaskStarts&, const TaskArgs&, int, int,
                                                    int, size_t, const uint32_t*, uint32_t, int,
                                                    hipStream_t);
}  // namespace shwfs
