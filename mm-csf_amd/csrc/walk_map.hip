// Chunked walk over a tree's nonzeros in the order of a level below its root.
#include "walk_kernel.hpp"

namespace mmcsf {
template void walk_launch<kMttkrp, kMap>(int, const Factors &, const WalkArgs &, hipStream_t);
template void walk_preload<kMttkrp, kMap>();
}  // namespace mmcsf
