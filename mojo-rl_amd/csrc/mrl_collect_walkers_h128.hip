// The walkers' fused collection kernels (collect_walkers.hpp) at hidden width 128.
#include "collect_walkers.hpp"

namespace mrl {
template int launch_collect_walker_t<128, 1>(mrl_ctx *, const mrl_rollout *, const CollectArgs &);
template int launch_collect_walker_t<128, 2>(mrl_ctx *, const mrl_rollout *, const CollectArgs &);
}  // namespace mrl
