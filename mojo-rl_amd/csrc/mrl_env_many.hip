// BipedalWalker's and HalfCheetah's stand-alone step for batches that give every SIMD several wavefronts.
//
// The workgroups of mrl_env.hip are built for the shortest step of ONE round of them: BipedalWalker's rows (128 terrain
// edges each) and contact lists fill a CU's LDS with 16 envs, whose solver keeps two of eight wavefronts busy, and
// HalfCheetah's kernel carries the one-lane form for rows of foreign wiring and with it 302 registers, one wavefront per
// SIMD.  A batch of several rounds ran them one after the other.  Here a workgroup is ONE wavefront with eight envs, eight
// lanes each, through every phase of the step, and as many of them share a SIMD as registers and LDS allow:
//   * terrain stays in global memory; a phase stages the few edges near the env in LDS;
//   * contacts go straight to their place in the env's list: the eight lanes take eight (body, vertex) pairs at a time,
//     count first, then write behind the counts of the lanes before them;
//   * rows of foreign wiring are left alone and stepped by a second launch, which ends at once where there are none
//     (4.5 us of launch and of one word read, counted below).  No reset of this library makes such rows: a caller's own
//     joint table does.  One lane steps such a row, from global memory, behind the other rows instead of beside them: us per
//     step, workgroup form -> this one, one such row / every ninth / all:  BipedalWalker  8200 envs 85 -> 184 / 230 -> 233 /
//     200 -> 242,  65536 envs 469 -> 340 / 1306 -> 922 / 1158 -> 1020;  HalfCheetah  8200 envs 212 -> 270 / 300 -> 321 / 374 -> 229,
//     65536 envs 544 -> 468 / 1746 -> 1171 / 2121 -> 907.
// Same operations on the same values as the workgroup forms: identical results bit for bit.
//
// What bounds it: the vector units' instruction stream, two to four wavefronts of dependent chains per SIMD
// (BipedalWalker: 168 registers and 14.6 KB of LDS, eleven wavefronts per CU; HalfCheetah: 128 registers, four wavefronts
// per SIMD).
// us per step, workgroup form -> this one:
//   BipedalWalker  4096: 33 -> 56   5000: 56 -> 56   8192: 64 -> 58   16384: 125 -> 70   65536: 446 -> 182
//   HalfCheetah    8192: 42 -> 49  10000: 80 -> 60                   16384: 82 -> 64   65536: 317 -> 177
#include <cmath>
#include "mrl_host.hpp"
#include "env_block.hpp"
#include "env_cheetah_lanes.hpp"

namespace mrl {

constexpr int MANY_EPB = 8, GROUP = 8;   // envs per wavefront, lanes per env

// or over the eight lanes of an env: neighbours, pairs, then the mirrored half row
MRL_DEV unsigned group_or(unsigned v) {
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false);    // quad_perm 1 0 3 2
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false);    // quad_perm 2 3 0 1
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false);   // row_half_mirror
    return v;
}

// ---------------------------------------------------------------- BipedalWalker

struct BipedalMany {
    using L = bw::L;
    // a row without its edges: everything up to them, then the edge count and the metadata
    static constexpr int HEAD = L::EDGES_OFF, META = HEAD + 1, STRIDE = (META + L::META_SIZE) | 1;
    static constexpr int CTS = (L::MAX_CONTACTS * CONTACT_SCRATCH) | 1;
    static constexpr int TASKS = 21, MAX_STAGED_LIDAR = CTS / 6;
    // edges staged behind the records of the contact list while the list is being made
    static constexpr int MAX_STAGED = 24, STAGED_AT = CTS - 6 * MAX_STAGED;
    static_assert(MANY_EPB * CTS >= L::STATE_SIZE, "a finished row is rebuilt in the contact scratch");
    static_assert(L::MAX_EDGES == 128 && EdgeMask<L>::WORDS == 4, "sixteen edges per lane");
};

// The edges of an env near an x interval: the mask (edges_near_bits), their number, and -- if they are at most `room` --
// their coordinates in LDS in ascending order.
struct NearEdges {
    unsigned w[4];
    int n;
    bool staged;
    // place of edge e among them
    MRL_DEV int rank(int e) const {
        const int q = e >> 5;
        int at = __popc((q == 0 ? w[0] : q == 1 ? w[1] : q == 2 ? w[2] : w[3]) & ((1u << (e & 31)) - 1u));
        at += q > 0 ? __popc(w[0]) : 0;
        at += q > 1 ? __popc(w[1]) : 0;
        at += q > 2 ? __popc(w[2]) : 0;
        return at;
    }
};
MRL_DEV NearEdges near_edges(const float *edges, int n_edges, float xlo, float xhi, float widen, int b, float *stage, int room) {
    float x0[16], x1[16];   // this lane's edges: b, 8 + b, ...
#pragma unroll
    for (int k = 0; k < 16; ++k) { x0[k] = edges[(8 * k + b) * 6]; x1[k] = edges[(8 * k + b) * 6 + 2]; }
    NearEdges m;
    unsigned mine = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const float E[3] = {x0[k], 0.0f, x1[k]};
        mine |= (unsigned)(8 * k + b < n_edges && edge_near(E, xlo, xhi, widen)) << k;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        unsigned v = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) v |= ((mine >> (4 * q + k)) & 1u) << (8 * k + b);
        m.w[q] = group_or(v);
    }
    m.n = __popc(m.w[0]) + __popc(m.w[1]) + __popc(m.w[2]) + __popc(m.w[3]);
    m.staged = m.n <= room;
    if (m.staged) {
        for (unsigned left = mine; left; left &= left - 1) {
            const int e = 8 * (__ffs((int)left) - 1) + b, at = m.rank(e);
            float v[6];
#pragma unroll
            for (int f = 0; f < 6; ++f) v[f] = edges[e * 6 + f];
#pragma unroll
            for (int f = 0; f < 6; ++f) stage[at * 6 + f] = v[f];
        }
    }
    return m;
}
// edge e, the r-th near one (r is looked at only where it is staged)
MRL_DEV void near_edge(const float *edges, const float *stage, bool staged, int e, int r, float (&E)[6]) {
    if (staged) {
#pragma unroll
        for (int f = 0; f < 6; ++f) E[f] = stage[6 * r + f];
    } else {
#pragma unroll
        for (int f = 0; f < 6; ++f) E[f] = edges[6 * e + f];
    }
}

// The contact list of an env (edge_detect: (body, vertex) order, edges in ascending order, cut at MAX_CONTACTS) by its
// eight lanes, eight pairs at a time; returns the number of records.  sin_b / cos_b: of the angle of body b.
MRL_DEV int detect_group(const float *row, const float *edges, const float *shapes, int n_edges, float sin_b, float cos_b,
                         float *contacts, int b, int lane) {
    using L = bw::L;
    float xlo, xhi;
    bodies_x_interval<L>(row, shapes, xlo, xhi);
    float *stage = contacts + BipedalMany::STAGED_AT;
    NearEdges near = near_edges(edges, n_edges, xlo, xhi, 0.0f, b, stage, BipedalMany::MAX_STAGED);
    bw::wave_sync();
    int total = 0;
#pragma unroll 1
    for (int k0 = 0; k0 < BipedalMany::TASKS; k0 += GROUP) {
        const int k = k0 + b;
        int body, vertex, max_verts;
        BipedalWalker::detect_task(k < BipedalMany::TASKS ? k : 0, body, vertex, max_verts);
        const float *B = row + L::BODIES_OFF + body * BODY_SIZE;
        const float *S = shapes + (int)B[IDX_SHAPE] * SHAPE_SIZE;
        const float sin_a = __shfl(sin_b, (lane & ~7) + body, 64), cos_a = __shfl(cos_b, (lane & ~7) + body, 64);
        const float local_x = S[2 + vertex * 2], local_y = S[3 + vertex * 2];
        const float world_x = B[IDX_X] + local_x * cos_a - local_y * sin_a;
        const float world_y = B[IDX_Y] + local_x * sin_a + local_y * cos_a;
        const bool task = k < BipedalMany::TASKS && vertex < (int)S[1];
        // which edges it touches
        unsigned hit[4] = {0u, 0u, 0u, 0u};
        int r = 0, count = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            for (unsigned cand = near.w[q]; cand; cand &= cand - 1, ++r) {
                const int e = __ffs((int)cand) - 1;
                float E[6], rec[CONTACT_SIZE];
                near_edge(edges, stage, near.staged, 32 * q + e, r, E);
                int c = 0;
                if (task && edge_x_pass(E[0], E[2], world_x)) vertex_edge_test(E, body, world_x, world_y, rec, c, 1);
                hit[q] |= (unsigned)c << e;
            }
            count += __popc(hit[q]);
        }
        int before = count;
#pragma unroll
        for (int off = 1; off < GROUP; off <<= 1) {
            const int o = __shfl_up(before, off, GROUP);
            before += b >= off ? o : 0;
        }
        const int all = __shfl(before, lane | 7, 64);
        int at = total + before - count;
        total += all;
        // (the staged edges lie behind the first STAGED_AT / CONTACT_SIZE records: beyond them they are gone)
        near.staged = near.staged && total <= BipedalMany::STAGED_AT / CONTACT_SIZE;
        bw::wave_sync();
#pragma unroll
        for (int q = 0; q < 4; ++q)
            for (unsigned cand = hit[q]; cand; cand &= cand - 1) {
                const int e = 32 * q + __ffs((int)cand) - 1;
                float E[6];
                near_edge(edges, stage, near.staged, e, near.rank(e), E);
                vertex_edge_test(E, body, world_x, world_y, contacts, at, L::MAX_CONTACTS);
            }
        bw::wave_sync();
    }
    return total < L::MAX_CONTACTS ? total : L::MAX_CONTACTS;
}

// Lidar ray i against the near edges whose place is `part` modulo `parts` (bw::lidar_value_part, lidar_ray_picked)
MRL_DEV float lidar_group(const float *row, const float *grow, const NearEdges &near, const float *stage, int i, int part, int parts) {
    using L = bw::L;
    const float *B = row + L::BODIES_OFF;
    const float hull_x = B[IDX_X], hull_y = B[IDX_Y];
    const float lidar_range = (float)bw::LIDAR_RANGE;
    const float local_angle = (float)i * 1.5f / (float)9;
    const float world_angle = B[IDX_ANGLE] - local_angle - (float)(3.14159265358979323846 / 2.0);
    float sn, cs;
    sincos32(world_angle, sn, cs);
    const float rdx = cs * lidar_range, rdy = sn * lidar_range, end_x = hull_x + rdx;
    if (!(hull_x == hull_x) || !(end_x == end_x)) return part == 0 ? lidar_ray<L>(grow, hull_x, hull_y, rdx, rdy) : 1.0f;
    if (!near.staged) {
        EdgeMask<L> m;
#pragma unroll
        for (int q = 0; q < 4; ++q) m.w[q] = near.w[q];
        return part == 0 ? lidar_ray_near<L>(grow, m, hull_x, hull_y, rdx, rdy) : 1.0f;
    }
    const float rlo = (hull_x < end_x ? hull_x : end_x) - 0.01f, rhi = (hull_x > end_x ? hull_x : end_x) + 0.01f;
    static_assert(BipedalMany::MAX_STAGED_LIDAR <= 64, "a bit per staged edge");
    unsigned long long picked = 0;
    for (int r = part; r < near.n; r += parts) {
        const float x0 = stage[6 * r], x1 = stage[6 * r + 2];
        const float elo = x0 < x1 ? x0 : x1, ehi = x0 < x1 ? x1 : x0;
        picked |= (unsigned long long)!(ehi < rlo || elo > rhi) << r;
    }
    float min_t = 1.0f;
    for (; picked; picked &= picked - 1)
        lidar_edge(stage + 6 * (__ffsll((long long)picked) - 1), hull_x, hull_y, rdx, rdy, min_t);
    return min_t;
}

// a row that the eight-lane forms step: the walker's own joints, bodies with no more vertices than detect_task plans
MRL_DEV bool bipedal_row_ok(const float *row, const float *shapes) {
    bool ok = bw::lanes_row_ok(row);
#pragma unroll
    for (int b = 0; b < bw::L::NUM_BODIES; ++b) {
        const float *S = shapes + (int)row[bw::L::BODIES_OFF + b * BODY_SIZE + IDX_SHAPE] * SHAPE_SIZE;
        ok = ok && (int)S[0] == SHAPE_POLYGON && (int)S[1] <= (b == 0 ? 5 : 4);
    }
    return ok;
}

template <bool AUTORESET>
__global__ __launch_bounds__(64, 3) void bipedal_many_kernel(float *states, const float *actions, float *rewards, float *dones,
                                                          float *obs, const float *shapes_g, int batch, uint64_t reset_seed,
                                                          Accounting acc, int *foreign, int call) {
    using M = BipedalMany;
    using L = bw::L;
    __shared__ float rows[MANY_EPB * M::STRIDE];
    __shared__ float cts[MANY_EPB * M::CTS];
    __shared__ float shapes[bw::NSHAPE_FLOATS];
    const int lane = threadIdx.x, slot = lane >> 3, b = lane & 7;
    const int env0 = blockIdx.x * MANY_EPB, nenv = min(MANY_EPB, batch - env0);
    float *gbase = states + (size_t)env0 * L::STATE_SIZE;
    constexpr int IN = M::HEAD - L::BODIES_OFF, TAIL = L::META_SIZE + 1;   // (the observation is written anew)
    static_assert(IN <= 192 && IN > 128 && TAIL <= 64, "three loads per lane and row, one for the tail");
    {
        float v[MANY_EPB][3], q[2];
#pragma unroll
        for (int e = 0; e < MANY_EPB; ++e)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (e < nenv && lane + 64 * k < IN) v[e][k] = gbase[(size_t)e * L::STATE_SIZE + L::BODIES_OFF + lane + 64 * k];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int e = (lane + 64 * k) >> 4, c = lane & 15;
            if (e < nenv && c < TAIL) q[k] = gbase[(size_t)e * L::STATE_SIZE + L::EDGE_COUNT_OFF + c];
        }
        for (int i = lane; i < bw::NSHAPE_FLOATS; i += 64) shapes[i] = shapes_g[i];
#pragma unroll
        for (int e = 0; e < MANY_EPB; ++e)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (e < nenv && lane + 64 * k < IN) rows[e * M::STRIDE + L::BODIES_OFF + lane + 64 * k] = v[e][k];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int e = (lane + 64 * k) >> 4, c = lane & 15;
            if (e < nenv && c < TAIL) rows[e * M::STRIDE + M::HEAD + c] = q[k];
        }
    }
    __syncthreads();

    const bool live = slot < nenv;
    const int mine = live ? slot : 0;
    float *row = rows + slot * M::STRIDE, *contacts = cts + slot * M::CTS, *meta = row + M::META;
    const float *grow = gbase + (size_t)mine * L::STATE_SIZE, *edges = grow + L::EDGES_OFF;
    const bool ok = live && bipedal_row_ok(row, shapes);
    if (live && !ok && b == 0) *foreign = call;
    bool finished = false;
    NearEdges near{};
    if (ok) {
        float act[bw::ACT];
        EpisodeSums sums{0.0f, 0.0f};
        if (b == 0) {
            sums = account_before(acc, env0 + slot);
            bw::step_motors(row, actions + (size_t)(env0 + slot) * bw::ACT, act);
        }
        int n_edges = (int)row[M::HEAD];
        n_edges = n_edges < L::MAX_EDGES ? n_edges : L::MAX_EDGES;
        int n;
        {
            float sin_b, cos_b;
            sincos32(row[L::BODIES_OFF + (b < L::NUM_BODIES ? b : 0) * BODY_SIZE + IDX_ANGLE], sin_b, cos_b);
            n = detect_group(row, edges, shapes, n_edges, sin_b, cos_b, contacts, b, lane);
        }
        bw::physics_lanes(row, contacts, n, lane);
        bw::wave_sync();
        if (b == 0) {
            float r, d;
            bw::step_tail<false, false>(row, contacts, n, act, r, d, meta);
            rewards[env0 + slot] = r;
            dones[env0 + slot] = d;
            account(acc, env0 + slot, r, d, sums);
            finished = d > 0.5f;
        }
        bw::wave_sync();
        // the ten rays: eight side by side, then four lanes for each of the other two
        const float hull_x = row[L::BODIES_OFF + IDX_X], lidar_range = (float)bw::LIDAR_RANGE;
        near = near_edges(edges, n_edges, hull_x - lidar_range, hull_x + lidar_range, 0.02f, b, contacts, M::MAX_STAGED_LIDAR);
        bw::wave_sync();
        row[14 + b] = lidar_group(row, grow, near, contacts, b, 0, 1);
        float t = lidar_group(row, grow, near, contacts, 8 + (b >> 2), b & 3, 4);
#pragma unroll
        for (int off = 1; off <= 2; off <<= 1) {
            const float other = __shfl_xor(t, off, 64);
            t = other < t ? other : t;
        }
        if ((b & 3) == 0) row[22 + (b >> 2)] = t;
    }
    const unsigned long long fin = AUTORESET ? __ballot(finished) : 0ull, good = __ballot(ok);
    __syncthreads();
    // the changed parts of the rows out, and the observations
    for (int e = 0; e < nenv; ++e) {
        if (!((good >> (8 * e)) & 1ull) || ((fin >> (8 * e)) & 1ull)) continue;
        float *g = gbase + (size_t)e * L::STATE_SIZE;
        const float *src = rows + e * M::STRIDE;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (lane + 64 * k < M::HEAD) g[lane + 64 * k] = src[lane + 64 * k];
        if (lane < L::META_SIZE) g[L::META_OFF + lane] = src[M::META + lane];
        if (lane < bw::OBS) obs[(size_t)(env0 + e) * bw::OBS + lane] = src[lane];
    }
    // finished rows are rebuilt one after the other in the contact scratch
    for (unsigned long long left = fin; left; left &= left - 1) {
        const int e = (__ffsll((long long)left) - 1) >> 3;
        BipedalWalker::reset_wave(cts, reset_seed, env0 + e, lane);
        __syncthreads();
        float *g = gbase + (size_t)e * L::STATE_SIZE;
        for (int i = lane; i < L::STATE_SIZE; i += 64) g[i] = cts[i];
        if (lane < bw::OBS) obs[(size_t)(env0 + e) * bw::OBS + lane] = cts[lane];
        __syncthreads();
    }
}

// ---------------------------------------------------------------- HalfCheetah

struct HalfCheetahMany : HalfCheetah {
    static constexpr int EPB = MANY_EPB, THREADS = 64;
};

template <bool AUTORESET>
__global__ __launch_bounds__(64, 4) void halfcheetah_many_kernel(float *states, const float *actions, float *rewards, float *dones,
                                                              float *obs, const float *shapes_g, int batch, uint64_t reset_seed,
                                                              Accounting acc, int *foreign, int call) {
    using E = HalfCheetahMany;
    using S = Stage<E>;
    __shared__ float rows[E::EPB * S::STRIDE];
    __shared__ float shapes[E::NSHAPE];
    const int lane = threadIdx.x, slot = lane >> 3, b = lane & 7;
    const int env0 = blockIdx.x * E::EPB, nenv = min(E::EPB, batch - env0);
    float *gbase = states + (size_t)env0 * E::STATE;
    S::in(rows, gbase, nenv, lane);
    for (int i = lane; i < E::NSHAPE; i += E::THREADS) shapes[i] = shapes_g[i];
    __syncthreads();

    const bool live = slot < nenv;
    float *row = rows + slot * S::STRIDE;
    const int env = env0 + (live ? slot : 0);
    const bool ok = live && hc::lanes_row_ok(row, shapes);
    if (live && !ok && b == 0) *foreign = call;
    bool finished = false;
    if (ok) {
        float r = 0.0f, d = 0.0f;
        hc::step_lanes(row, shapes, actions + (size_t)env * E::ACT_W, lane, r, d);
        if (b == 0) {
            rewards[env] = r;
            dones[env] = d;
            account(acc, env, r, d);
            finished = d > 0.5f;
            if (AUTORESET && finished) E::reset(row, reset_seed, env);
        }
    }
    const unsigned long long fin = AUTORESET ? __ballot(finished) : 0ull, good = __ballot(ok);
    unsigned long long was_reset = 0, stepped = 0;
#pragma unroll
    for (int k = 0; k < E::EPB; ++k) {
        was_reset |= ((fin >> (8 * k)) & 1ull) << k;
        stepped |= ((good >> (8 * k)) & 1ull) << k;
    }
    __syncthreads();
    for (int i = lane; i < nenv * E::OBS; i += E::THREADS) {
        const int r = i / E::OBS, c = i - r * E::OBS;
        if ((stepped >> r) & 1ull) obs[(size_t)env0 * E::OBS + i] = rows[r * S::STRIDE + c];
    }
    S::out(rows, gbase, nenv, lane, 0, E::DYN_END, stepped);
    S::out(rows, gbase, nenv, lane, E::L::META_OFF, E::STATE, stepped);
    if (AUTORESET) S::out_rows(rows, gbase, nenv, was_reset, lane, E::DYN_END, E::L::META_OFF);
}

// ---------------------------------------------------------------- rows of foreign wiring

struct BipedalForeign : BipedalWalker {
    static MRL_DEV bool ok(const float *row, const float *shapes) { return bipedal_row_ok(row, shapes); }
    static MRL_DEV void step(float *row, float *cts, const float *shapes, int env, const float *a, float &r, float &d) {
        bw::step_row<true>(row, cts, shapes, env, a, r, d);
    }
};
struct HalfCheetahForeign : HalfCheetah {
    static MRL_DEV bool ok(const float *row, const float *shapes) { return hc::lanes_row_ok(row, shapes); }
};

// One lane per env over the whole batch, in global memory; nothing to do unless the launch before it met such a row
// (*foreign == call), which it left as it was.
template <class E, bool AUTORESET>
__global__ __launch_bounds__(64) void foreign_rows_kernel(float *states, const float *actions, float *rewards, float *dones,
                                                          float *obs, const float *shapes_g, int batch, uint64_t reset_seed,
                                                          Accounting acc, const int *foreign, int call) {
    using S = Stage<E>;
    __shared__ float cts[WAVE * S::CSTRIDE];
    __shared__ float shapes[E::NSHAPE];
    if (*foreign != call) return;
    const int lane = threadIdx.x;
    for (int i = lane; i < E::NSHAPE; i += WAVE) shapes[i] = shapes_g[i];
    __syncthreads();
    for (int env = blockIdx.x * WAVE + lane; env < batch; env += gridDim.x * WAVE) {
        float *row = states + (size_t)env * E::STATE;
        if (E::ok(row, shapes)) continue;
        const EpisodeSums sums = account_before(acc, env);
        float r, d;
        E::step(row, cts + lane * S::CSTRIDE, shapes, env, actions + (size_t)env * E::ACT_W, r, d);
        rewards[env] = r;
        dones[env] = d;
        account(acc, env, r, d, sums);
        if (AUTORESET && d > 0.5f) E::reset(row, reset_seed, env);
        for (int k = 0; k < E::OBS; ++k) obs[(size_t)env * E::OBS + k] = row[k];
    }
}

template <class E, bool AUTORESET>
static void launch_foreign(mrl_ctx *ctx, int batch, float *states, const float *actions, float *rewards, float *dones,
                           float *obs, const float *shapes, uint64_t reset_seed, const Accounting &acc, int *foreign) {
    hipLaunchKernelGGL((foreign_rows_kernel<E, AUTORESET>), dim3(std::min(grid_for(batch, WAVE), ctx->n_cus)), dim3(WAVE), 0,
                       ctx->stream, states, actions, rewards, dones, obs, shapes, batch, reset_seed, acc, foreign,
                       ctx->foreign_call);
}

template <bool AUTORESET>
static void launch_many(mrl_ctx *ctx, int env_id, int batch, float *states, const float *actions, float *rewards,
                        float *dones, float *obs, uint64_t reset_seed, const Accounting &acc, int *foreign) {
    const dim3 grid(grid_for(batch, MANY_EPB)), block(64);
    if (env_id == MRL_ENV_BIPEDAL) {
        hipLaunchKernelGGL(bipedal_many_kernel<AUTORESET>, grid, block, 0, ctx->stream, states, actions, rewards, dones, obs,
                           ctx->bw_shapes, batch, reset_seed, acc, foreign, ctx->foreign_call);
        launch_foreign<BipedalForeign, AUTORESET>(ctx, batch, states, actions, rewards, dones, obs, ctx->bw_shapes, reset_seed, acc, foreign);
    } else {
        hipLaunchKernelGGL(halfcheetah_many_kernel<AUTORESET>, grid, block, 0, ctx->stream, states, actions, rewards, dones, obs,
                           ctx->hc_shapes, batch, reset_seed, acc, foreign, ctx->foreign_call);
        launch_foreign<HalfCheetahForeign, AUTORESET>(ctx, batch, states, actions, rewards, dones, obs, ctx->hc_shapes, reset_seed, acc, foreign);
    }
}

// From the batch on at which the workgroup forms need a second round: one 16-env workgroup per CU, one eight-env wavefront
// per SIMD (4096 and 8192 envs on 256 CUs; up to there they are faster, table at the head of the file).
bool env_step_many_pays(const mrl_ctx *ctx, int env_id, int batch) {
    if (env_id == MRL_ENV_BIPEDAL) return batch > BipedalWalker::EPB * ctx->n_cus;
    return env_id == MRL_ENV_HALFCHEETAH && batch > MANY_EPB * 4 * ctx->n_cus;
}

void env_step_many(mrl_ctx *ctx, int env_id, int batch, float *states, const float *actions, float *rewards, float *dones,
                   float *obs, bool autoreset, uint64_t reset_seed, const Accounting &acc) {
    int *foreign = reinterpret_cast<int *>(ctx->upd_scratch + FOREIGN_WORD);
    ctx->foreign_call += 1;
    if (autoreset) launch_many<true>(ctx, env_id, batch, states, actions, rewards, dones, obs, reset_seed, acc, foreign);
    else launch_many<false>(ctx, env_id, batch, states, actions, rewards, dones, obs, reset_seed, acc, foreign);
}

}  // namespace mrl
