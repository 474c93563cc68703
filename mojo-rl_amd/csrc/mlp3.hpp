// Host-side interface of the fused three-layer MLP kernels (mrl_mlp3.hip, mrl_rows.hip, mrl_fb.hip).
#pragma once
#include "mrl_host.hpp"

namespace mrl {

// one net's buffers for the fused kernels; fields a call does not need stay null
struct Mlp3Net {
    const float *x;          // forward: input [B, IN]
    const float *params;
    float *out;              // forward: [B, A] or [B, 2A]
    float *cache;            // forward: written when non-null; backward: read
    const float *grad_out;   // backward
    float *grad_in;          // backward: written when non-null
    float *ls_part, *db_part, *thin_part;            // workspace: the row tiles' pieces (set by the host function)
    // for the weight-gradient launch: h1 and g1 split, as operands contracted over the batch rows
    // (mlp_split.hpp: k-step = 32 batch rows, the other index = column)
    unsigned short *h1q, *g1q;
    const unsigned short *wf, *wb;                   // fused update: the hidden layer's weights split (mlp_split.hpp), forward / W^T
    int A, gauss;            // set by the host function from the description
    int thin_stride;         // floats per row tile in thin_part: IN H + H A, + H H where the tiles carry dW1 too
};
struct Mlp3Nets { Mlp3Net n[2]; };

// split operand copies of the nets' hidden-layer weights (mlp_split.hpp)
struct SplitNets {
    const float *w1[2];
    unsigned short *wf[2], *wb[2];
};

// The PPO part of the fused update (net 0 = actor, net 1 = critic) over minibatch rows that are still
// where the rollout left them: the forward reads its input rows through `idx`, and every row tile
// goes straight on to its loss gradients (deep_agents/ppo/ppo.mojo:285-378, 538-633;
// kernels.mojo:230-486) and to its share of the KL early-stop test, so that neither a gather nor a
// loss launch is needed.
struct FwdLoss {
    const int32_t *idx;                                   // [mb] rollout rows of the minibatch
    const float *r_obs, *r_act, *r_adv, *r_ret, *r_logp, *r_val;
    const float *adv_stats;                               // {mean, std} of the minibatch's advantages; null: as they are
    float *g_actor_out, *g_values, *kl;                   // [mb, head], [mb], [mb]
    float *kl_part;                                       // [row tiles] sums of the tiles' KL estimates, for the test
    int32_t *kl_flag;                                     // null: no test (nothing is left in kl_part)
    const int32_t *skip;                                  // *skip != 0: nothing of this minibatch is needed
    // (The kernels request the word first, always, and test it behind their first requests.  0.6 us of a minibatch's 51 at
    // H = 256 and 4096 rows, for the 45 of one behind the stop.)
    uint64_t *posts; int n_posts;                         // words to clear for the kernel that applies the update
    int dw_in_tiles;                                      // forward + backward: the row tiles leave their dW1 as well
    int mb, A, continuous, clip_value;                    // A = actions (discrete) or action width (continuous)
    float clip_eps, ent_coef, value_coef;
};

bool mlp3_fusable(const mrl_mlp_desc &d, int *H, int *act, bool *gauss);
bool mlp3_pair_fusable(const mrl_mlp_desc &a, const mrl_mlp_desc &b);
int mlp3_forward(mrl_ctx *ctx, const mrl_mlp_desc &d, int batch, const float *in, const float *params,
                 float *out, float *cache);
int mlp3_backward(mrl_ctx *ctx, const mrl_mlp_desc &d, int batch, const float *grad_out, const float *params,
                  const float *cache, float *grads, float *grad_in);

// The fused update of two nets: one kernel per row tile runs forward (inputs read through loss.idx, io.n[i].out
// written), loss gradients and the way back (mrl_fb.hip), then the H x H weight gradients and the sums over the tiles.
// Workspace: UpdateWs, carved from the context's; the backward of one net (mrl_rows.hip) uses it as well.
struct UpdateWs {
    int rows, tiles;          // batch rows per tile
    bool dw_in_tiles;
    SplitNets split;          // copies of the hidden layers' weights that io.n[i].wf / wb read
    Mlp3Net net[2];           // h1q, g1q, ls_part, db_part, thin_part, thin_stride
    float *partial;
    int splits, steps_per;    // batch splits of the weight-gradient launch, k-steps of 32 rows each
};
int mlp3_update_ws(mrl_ctx *ctx, const mrl_mlp_desc *const *descs, int n_nets, int batch, const float *const *params, UpdateWs *out);
int launch_split_weights(mrl_ctx *ctx, int H, const SplitNets &s, int n_nets);
// the tiles and, where they do not leave it themselves, the hidden layers' weight gradient: pieces, not yet added up
int mlp3_update_n(mrl_ctx *ctx, const mrl_mlp_desc *const *descs, int batch, Mlp3Nets io, const UpdateWs &ws, const FwdLoss &loss);
struct SumNets;   // tile_sums.hpp
SumNets mlp3_sum_nets(const mrl_mlp_desc *const *descs, int n_nets, const UpdateWs &ws, float *const *grads, const int32_t *skip);
// sq_part (nullable): receives per-block sums of squares of the gradients, [net * 1024 + block];
// *sq_blocks = number of blocks written (0 when none were)
int mlp3_sum_tiles(mrl_ctx *ctx, const SumNets &sn, int tile_rows, float *sq_part, int *sq_blocks);
int launch_fwd16(mrl_ctx *ctx, int H, int act, int batch, int IN, const Mlp3Net &nn);
int launch_bwd(mrl_ctx *ctx, int H, int act, int batch, int IN, int rows, const Mlp3Net &nn, bool dw_in_tiles);
int launch_dw_frag(mrl_ctx *ctx, int H, int n_nets, int batch, const UpdateWs &ws, int P0, int Ptot, int w1_off, const int32_t *skip);
int launch_fb(mrl_ctx *ctx, int H, int act, int batch, int IN, int rows, const Mlp3Nets &nets, const FwdLoss &fl);
// grows the context's MLP workspace to at least `floats`
int mlp_ensure_ws(mrl_ctx *ctx, size_t floats, float **out);

}  // namespace mrl
