// Priority order of the kernel variants (fastest first, generic last).
#include "variants.h"

namespace tvx {

const std::vector<ConvSetupFn>& ConvVariants() {
  static const std::vector<ConvSetupFn> v = {DwRegSetup, DwManyPlanesSetup, DwConv3x3Setup, DwPlanesSetup, PwRegSetup, PwRegF16Setup, PwConvSetup, ConvIm2colSetup, ConvBandSetup, ConvIgemmF16Setup, ConvTileSetup, ConvIm2colRestSetup, ConvIgemmSetup, ConvGemmSetup, ConvGenericSetup};
  return v;
}

const std::vector<FcSetupFn>& FcVariants() {
  static const std::vector<FcSetupFn> v = {FcRowsSetup, FcMfmaSetup, FcGenericSetup};
  return v;
}

const std::vector<SimpleSetupFn>& PoolVariants() {
  static const std::vector<SimpleSetupFn> v = {PoolStencilSetup, PoolRowsSetup, PoolRegSetup, PoolGenericSetup};
  return v;
}

}  // namespace tvx
