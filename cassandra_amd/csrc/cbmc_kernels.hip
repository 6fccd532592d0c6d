// cbmc_kernels.hip -- the growth kernels of cbmc_grow.h for one precision and
// pair style: built once per (CASS_P, CASS_LJ), the accessor named CASS_NAME.
#include "cbmc_grow.h"

namespace cass {

CbmcKernels CASS_NAME() {
  using P = CASS_P;
  constexpr bool LJ = CASS_LJ != 0;
  return CbmcKernels{
      k_widom_cbmc<P, 256, LJ>,
      k_widom_cbmc<P, 512, LJ>,
      {k_gcmc_chain<P, 128, LJ>, k_gcmc_chain<P, 256, LJ>, k_gcmc_chain<P, 512, LJ>, k_gcmc_chain<P, 1024, LJ>},
      k_gemc_chain<P, 512, LJ>,
      k_regrow_chain<P, 512, LJ>};
}

}  // namespace cass
