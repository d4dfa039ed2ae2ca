// Chunked walk over sorted COO (root-mode MTTKRP of the COO type).
#include "walk_kernel.hpp"

namespace mmcsf {
template void walk_launch<kMttkrp, kCoo>(int, const Factors &, const WalkArgs &, hipStream_t);
template void walk_preload<kMttkrp, kCoo>();
}  // namespace mmcsf
