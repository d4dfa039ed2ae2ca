// Chunked root walks of several modes in one launch (all-mode MTTKRP).
#include "walk_kernel.hpp"

namespace mmcsf {
template bool walk_launch_set<kMttkrp>(int, const Factors &, WalkSet &, int, const uint64_t *, bool, hipStream_t);
template void walk_preload_set<kMttkrp>();
}  // namespace mmcsf
