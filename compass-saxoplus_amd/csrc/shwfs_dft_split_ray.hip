// Split-FP16 spot kernels with the guide-star raytrace in the field stage.
#include "shwfs_image_dft.hpp"

namespace shwfs {

int32_t launch_split_ray(const ImageParams& p, const RayParams& r, int nfft, hipStream_t st) {
  if (p.nvalid <= 0) return SHWFS_OK;
  switch (nfft) {
    case 16: return launch_dft_ray_n<16, 1>(p, r, st);
    case 32: return launch_dft_ray_n<32, 1>(p, r, st);
    default: return fail(SHWFS_ERR_UNSUPPORTED, "traced spot kernel: needs nfft 16 or 32");
  }
}

}  // namespace shwfs
