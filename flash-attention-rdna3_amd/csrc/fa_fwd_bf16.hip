// Instantiates the fwd kernels for bf16.
#include "fa_fwd_impl.hpp"

namespace fa {
template hipError_t fwd_by_mods<bf16_t>(const fa_fwd_params& p, const FwdScratch& w, hipStream_t s);
}  // namespace fa
