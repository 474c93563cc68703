// HalfCheetah's env step with one lane per BODY (body_lanes.hpp): eight lanes per env (seven bodies, one idle), eight
// envs per wavefront.
//
// The bodies form a path, back foot - shin - thigh - torso - front thigh - shin - foot.  The joint sweep visits joints
// 0 .. 5 in order, but after joint 0 (torso - back thigh) the back leg's joints 1, 2 touch bodies 1, 2, 3 only and the
// front leg's joints 3, 4, 5 bodies 0, 4, 5, 6: two chains without a body in common, which run side by side -- four joint
// slots per sweep instead of six.  Each slot pairs lane l with l ^ 1, 7 - l, l ^ 2, 7 - l.
//
// The wiring is HalfCheetah's (cheetah_planar_v2.mojo: torso 0; back thigh / shin / foot 1, 2, 3;
// front 4, 5, 6; joint j joins body j + 1 to its parent).  A row whose joint table or shapes differ
// from that is stepped by the one-lane form instead (lanes_row_ok, tested by the caller).
#pragma once
#include "env_walkers.hpp"
#include "body_lanes.hpp"

namespace mrl {
namespace hc {

constexpr int LANES_PER_ENV = 8;

struct Wiring {
    static constexpr int LANES = 8, SLOTS = 4;
    static constexpr uint32_t BODY = 0x4253F610u;          // lanes 0 .. 7: torso, back thigh, front foot, -, back foot, front shin, back shin, front thigh
    static constexpr int LANE_OF[7] = {0, 1, 6, 4, 7, 5, 2};
    static constexpr int CTRL[4] = {0xB1, 0x141, 0x4E, 0x141};   // l ^ 1, 7 - l, l ^ 2, 7 - l
    static constexpr uint32_t IN[4] = {0x03u, 0xC3u, 0xF0u, 0x24u}, CHILD[2] = {0x32u, 0xC4u};
    static constexpr uint32_t JOINT[2] = {0x42420000u, 0x31500513u};
    static constexpr bool SPRING = false, MOTOR = true, ANGLES_AFTER = true, LAST_TURNS_FIRST = false;
};

// LDS writes of this wavefront's lanes become visible to its other lanes
MRL_DEV void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// lanes of one env sit side by side: value of lane `src` of my group
template <class V>
MRL_DEV V group_get(V v, int base, int src) { return __shfl(v, base + src, 64); }

// true when the row has the wiring and shapes this form assumes
MRL_DEV bool lanes_row_ok(const float *row, const float *shapes) {
    bool ok = body_lanes_row_ok<L, Topology, Wiring>(row);
    for (int b = 0; b < 7; ++b) {
        const float *S = shapes + (int)row[L::BODIES_OFF + b * BODY_SIZE + IDX_SHAPE] * SHAPE_SIZE;
        ok = ok && (int)S[0] == SHAPE_POLYGON && (int)S[1] <= 4;
    }
    return ok;
}

// everything after the physics of an env step but the observation (cheetah_planar_v2.mojo:790-846): reward
// and metadata; `a` = the clamped action, (x_after, torso_z) = the torso's position after the physics,
// `penalised` = ground contacts of the last sub-step on bodies other than the two feet
MRL_DEV void step_tail(float *row, const double *a, double x_before, double x_after, double torso_z, int penalised,
                       float &reward, float &done) {
    const double forward_velocity = (x_after - x_before) / (0.01 * (double)5);
    const double forward_reward = 1.0 * forward_velocity;
    double ctrl_cost = 0.0;
#pragma unroll
    for (int i = 0; i < ACT; ++i) {
        double c = a[i] < 1.0 ? a[i] : 1.0;
        c = c > -1.0 ? c : -1.0;
        ctrl_cost += c * c;
    }
    ctrl_cost *= 0.1;
    double height_bonus = 0.0;
    if (torso_z > 0.1) height_bonus = 1.0 * (torso_z < 0.5 ? torso_z : 0.5);
    const double penalty = 0.5 * (double)penalised;   // 0.5 per contact, summed in Float64: exact in any order
    const double r = forward_reward - ctrl_cost + height_bonus - penalty;
    float *M = row + L::META_OFF;
    const int step_count = (int)M[META_STEP] + 1;
    M[META_STEP] = (float)step_count;
    M[META_PREV_X] = (float)x_after;
    M[META_TOTAL] = (float)((double)M[META_TOTAL] + r);
    const bool d = step_count >= 1000;
    M[META_DONE] = d ? 1.0f : 0.0f;
    reward = (float)r;
    done = d ? 1.0f : 0.0f;
}

// the lane's own ground contacts (collision/flat_terrain.mojo:69-204), at most one per vertex, in vertex order
struct GroundContacts {
    LaneContact c[4];
    int kept;
    MRL_DEV void velocity(LaneBody &B, float friction, float restitution) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (!any_lane(k < kept)) return;
            contact_velocity<OneBody>(B, 0, c[k].f, c[k].jn, c[k].jt, friction, restitution, k < kept);
        }
    }
    MRL_DEV void position(LaneBody &B, float) const {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (!any_lane(k < kept)) return;
            c[k].position(B);
        }
    }
};

// The env step of hc::step_row by the eight lanes of an env's group (all lanes of the wavefront call
// it together; `lane` = lane in the wavefront, `row` = the group's env row in LDS, `action` = its six
// action components).  Lane 0 of the group returns reward / done.
MRL_DEV void step_lanes(float *row, const float *shapes, const float *action, int lane, float &reward, float &done) {
    const int l = lane & 7, base = lane & ~7, body = lane_body<Wiring>(l);
    const bool has = body < 7;
    const int b = has ? body : 0;

    const float gx = (float)0.0, gy = (float)-9.81, dt = (float)0.01, friction = (float)0.9, restitution = (float)0.0;
    const float baumgarte = (float)0.2;

    // ---- the action into the joint motors (the child's lane of joint body - 1), as hc::step_row does
    if (has && body > 0) {
        float v = action[body - 1];
        v = v < 1.0f ? v : 1.0f;
        v = v > -1.0f ? v : -1.0f;
        const double av = (double)v;
        float *J = row + L::JOINTS_OFF + (body - 1) * JOINT_SIZE;
        J[J_MOTOR_SPEED] = (av >= 0.0 ? 1.0f : -1.0f) * 1000.0f;
        J[J_MAX_TORQUE] = (float)(1.0 * ::fabs(av));
    }
    wave_sync_lds();

    LaneBody B;
    lane_body_load<L>(B, row, b);
    const float *F = row + L::FORCES_OFF + b * 3;
    float fx = F[0], fy = F[1], tau = F[2];
    LaneJoints<Wiring, false> usual(l);
    usual.load<L>(row, l, B, dt);
    const float *S = shapes + (int)row[L::BODIES_OFF + b * BODY_SIZE + IDX_SHAPE] * SHAPE_SIZE;
    const int n_verts = has ? (int)S[1] : 0;
    float lvx[4], lvy[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) { lvx[v] = S[2 + v * 2]; lvy[v] = S[3 + v * 2]; }
    const double x_before = (double)B.x[0];   // meaningful on lane 0 (the torso)

    float sn, cs;
    sincos32(B.ang[0], sn, cs);
    GroundContacts contacts;
    contacts.kept = 0;
    with_joints<L>(usual, row, l, B, dt, !usual.usual<L>(row, l, B), [&](auto &J) {
#pragma unroll 1
        for (int sub = 0; sub < 5; ++sub) {
            lane_integrate_velocity(B, fx, fy, tau, gx, gy, dt);
            fx = fy = tau = 0.0f;   // the forces are cleared at the end of every sub-step
            // ---- contacts, compacted in vertex order
            float px[4] = {0.0f, 0.0f, 0.0f, 0.0f}, py[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            int found = 0;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float world_x = B.x[0] + lvx[v] * cs - lvy[v] * sn;
                const float world_y = B.y[0] + lvx[v] * sn + lvy[v] * cs;
                const bool hit = v < n_verts && 0.0f - world_y > 0.0f;
#pragma unroll
                for (int c = 0; c <= v; ++c) {
                    px[c] = hit && found == c ? world_x : px[c];
                    py[c] = hit && found == c ? world_y : py[c];
                }
                found += hit ? 1 : 0;
            }
            // the list of an env is cut at MAX_CONTACTS in (body, vertex) order: contacts before mine are counted, where the
            // list can be that long
            contacts.kept = found;
            if (any_lane(found > L::MAX_CONTACTS / 7)) {
                int before = 0;
#pragma unroll
                for (int o = 0; o < 7; ++o) {
                    const int c = group_get(found, base, Wiring::LANE_OF[o]);
                    before += o < body ? c : 0;
                }
                const int left = L::MAX_CONTACTS - before;
                contacts.kept = left < 0 ? 0 : (left > found ? found : left);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (!any_lane(c < contacts.kept)) break;
                contacts.c[c].prepare(B, c < contacts.kept, px[c], py[c], 0.0f, 1.0f, 0.0f - py[c], baumgarte);
            }
            body_lanes_solve<Wiring, std::decay_t<decltype(J)>::ALL, 4, 2>(B, J, contacts, sn, cs, dt, friction, restitution, baumgarte);
        }
    });
    // ---- bodies and forces back into the row, then the rest of the step on the torso's lane
    if (has) lane_body_store<L>(B, row, b);
    int penalised = 0;   // contacts of the last sub-step on anything but the feet (bodies 3 and 6)
#pragma unroll
    for (int o = 0; o < 7; ++o) {
        const int c = group_get(contacts.kept, base, Wiring::LANE_OF[o]);
        penalised += (o != 3 && o != 6) ? c : 0;
    }
    // ---- the observation (hc::observe: the same expressions on the same values), every body's lane its own
    // entries: the torso its height, angle and velocity, a leg segment its angle and angular velocity
    // against its parent's
    {
        const LaneSlots<Wiring> slots(l);
        const double p_ang = (double)slots.parent(B.ang[0], B.ang[0]), p_w = (double)slots.parent(B.w[0], B.w[0]);
        if (body == 0) {
            row[0] = B.y[0]; row[1] = B.ang[0]; row[8] = B.vx[0]; row[9] = B.vy[0]; row[10] = B.w[0];
        } else if (has) {
            row[1 + body] = (float)((double)B.ang[0] - p_ang);
            row[10 + body] = (float)((double)B.w[0] - p_w);
        }
    }
    if (body == 0) {
        double a[ACT];
#pragma unroll
        for (int k = 0; k < ACT; ++k) {
            float v = action[k];
            v = v < 1.0f ? v : 1.0f;
            v = v > -1.0f ? v : -1.0f;
            a[k] = (double)v;
        }
        step_tail(row, a, x_before, (double)B.x[0], (double)B.y[0], penalised, reward, done);
    }
    wave_sync_lds();   // the row is complete for whoever reads it next
}

}  // namespace hc
}  // namespace mrl
