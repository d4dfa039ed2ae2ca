// Chunked root walk for the leaf-mode TTM.
#include "walk_kernel.hpp"

namespace mmcsf {
template void walk_launch<kTtm>(int, const Factors &, const WalkArgs &, hipStream_t);
template void walk_preload<kTtm>();
template void walk_launch<kTtmStream>(int, const Factors &, const WalkArgs &, hipStream_t);
}  // namespace mmcsf
