// The 16-envs-per-workgroup collection kernels (collect16.hpp) at hidden width 128.
#include "collect16.hpp"

namespace mrl {
template int launch_collect16_t<128, 1>(mrl_ctx *, const mrl_rollout *, const CollectArgs &, int32_t *);
template int launch_collect16_t<128, 2>(mrl_ctx *, const mrl_rollout *, const CollectArgs &, int32_t *);
}  // namespace mrl
