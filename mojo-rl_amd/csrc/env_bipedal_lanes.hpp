// BipedalWalker's physics step with one lane per BODY (body_lanes.hpp): eight lanes per env (five bodies, three idle).
//
// The joint sweep visits joints 0 .. 3 in order -- hull - upper leg 1, upper leg 1 - lower leg 1, hull - upper leg 2, upper
// leg 2 - lower leg 2 -- and joints 1 and 2 have no body in common: three joint slots per sweep instead of four, which
// pair lane l with l ^ 1, l ^ 2 and 7 - l.
//
// The contacts are the env's merged list in LDS (the records the per-vertex detection tasks left, in
// (body, vertex) order, cut at MAX_CONTACTS).  A row whose joint table differs from the walker's own is stepped by the
// one-lane form instead (lanes_row_ok, tested by the caller).
#pragma once
#include "env_walkers.hpp"
#include "body_lanes.hpp"

namespace mrl {
namespace bw {

constexpr int LANES_PER_ENV = 8;

struct Wiring {
    static constexpr int LANES = 8, SLOTS = 3;
    static constexpr uint32_t BODY = 0xFF4F2310u;          // lanes 0 .. 7: hull, upper leg 1, upper leg 2, lower leg 1, -, lower leg 2, -, -
    static constexpr int CTRL[3] = {0xB1, 0x4E, 0x141};    // l ^ 1, l ^ 2, 7 - l
    static constexpr uint32_t IN[3] = {0x03u, 0x0Fu, 0x24u}, CHILD[2] = {0x22u, 0x0Cu};
    static constexpr uint32_t JOINT[2] = {0x00300300u, 0x00001212u};
    static constexpr bool SPRING = false, MOTOR = true, ANGLES_AFTER = false, LAST_TURNS_FIRST = false;
};

// true when the row has the wiring this form assumes
MRL_DEV bool lanes_row_ok(const float *row) { return body_lanes_row_ok<L, Topology, Wiring>(row); }

// The physics of bw::step_finish (one sub-step: 6 velocity and 2 position sweeps) by the eight lanes of
// an env's group; all lanes of the group call it together.  `lane` = lane in the wavefront, `row` = the
// group's env row in LDS (motors already set by step_motors), `contacts` = the env's merged contact list
// with n >= 0 records.  Leaves the bodies and the cleared forces in the row.
MRL_DEV void physics_lanes(float *row, float *contacts, int n, int lane) {
    const int l = lane & 7, body = lane_body<Wiring>(l);
    const bool has = body < L::NUM_BODIES;
    const int b = has ? body : 0;
    const float gx = (float)0.0, gy = (float)-10.0, dt = (float)(1.0 / FPS), friction = (float)2.5, restitution = (float)0.0;
    const float baumgarte = (float)0.2;

    LaneBody B;
    lane_body_load<L>(B, row, b);
    const float *F = row + L::FORCES_OFF + b * 3;
    lane_integrate_velocity(B, F[0], F[1], F[2], gx, gy, dt);
    LaneJoints<Wiring, false> usual(l);
    usual.load<L>(row, l, B, dt);
    LaneListContacts<L, 2> list;
    list.load(B, contacts, n, body, baumgarte);
    float sn, cs;
    sincos32(B.ang[0], sn, cs);
    with_joints<L>(usual, row, l, B, dt, !usual.usual<L>(row, l, B), [&](auto &J) {
        body_lanes_solve<Wiring, std::decay_t<decltype(J)>::ALL, 6, 2>(B, J, list, sn, cs, dt, friction, restitution, baumgarte);
    });
    if (has) lane_body_store<L>(B, row, b);
    // ---- observation entries 0 .. 7 and 9 .. 12 (observe_state: the same expressions on the same values), every
    // body's lane its own: the hull 0 .. 3, a leg segment its angle and angular velocity against its parent's.
    // The contact flags (8, 13) and the lidar are left to what follows (step_tail<false, false>).
    {
        const LaneSlots<Wiring> slots(l);
        const double p_ang = (double)slots.parent(B.ang[0], B.ang[0]), p_w = (double)slots.parent(B.w[0], B.w[0]);
        if (body == 0) {
            const double hull_angle = B.ang[0], hull_omega = B.w[0], hull_vx = B.vx[0], hull_vy = B.vy[0];
            row[0] = (float)hull_angle;
            row[1] = (float)(hull_omega / 5.0);
            row[2] = (float)(hull_vx * (600.0 / SCALE) / FPS);
            row[3] = (float)(hull_vy * (400.0 / SCALE) / FPS);
        } else if (has) {
            const int leg = (body - 1) >> 1, at = 4 + 5 * leg + (((body - 1) & 1) ? 2 : 0);
            row[at] = (float)(((double)B.ang[0] - p_ang) / 1.0);
            row[at + 1] = (float)(((double)B.w[0] - p_w) / 10.0);
        }
    }
}

}  // namespace bw
}  // namespace mrl
