// The solver of an articulated env with one lane per BODY: LANES lanes side by side per env, in registers what
// physics2d_reg.hpp holds per env.
//
// What bounds it: a physics step is a chain of Gauss-Seidel sweeps on one wavefront, which issues an instruction every six
// cycles whether it depends on the last one or not (a branch costs five of them, taken or not).  So the fewest
// instructions win, and the lanes of an env share them:
//   * integration, sines and cosines, ground contacts (the other party is the ground, so contacts of different bodies
//     commute exactly) run on every body's own lane;
//   * joints without a body in common run side by side: the wiring's slots, in the order of the joint table;
//   * in a slot both bodies of a joint do their own half.  Written from a lane's own side -- d = mine - partner's -- the
//     child's and the parent's half are one formula: the parent's relative velocities, impulses, limits and motor speeds
//     are the child's negated, and a negation commutes with rounding;
//   * the lanes are laid out so that in every slot each lane finds its partner by one DPP pattern, which is an operand of
//     the subtraction that uses it;
//   * no lane branches on its own flags: a lane that a term does not concern computes it and keeps its value.
// Same operations on the same values as the one-lane form, in an order the arithmetic cannot tell from it: identical
// results bit for bit (but for the sign of a zero velocity that starts as -0).
//
// A wiring R has
//   LANES, BODIES (body b is listed in BODY as the nibble of its lane, 15: no body), SLOTS <= 4
//   CTRL[s]   DPP pattern that exchanges the partners of slot s
//   IN[s]     bit l: lane l takes part in slot s;  slots s and s + 2 have no lane in common
//   CHILD[e]  bit l: lane l is the child in its slot of parity e
//   JOINT[e]  nibble l: the joint of lane l's slot of parity e (0 where it has none)
//   SPRING, MOTOR: whether every joint has that term (all have a limit)
// These are the terms that the env's reset gives its joints.  A caller may have changed a row's: where a joint of the
// wavefront's has others (or a limit the wrong way round, or nothing to turn), the step runs on a second instance that decides
// every term lane by lane (ANY).
#pragma once
#include "physics2d_reg.hpp"

namespace mrl {

template <int CTRL>
MRL_DEV float dpp_xchg(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

template <class R>
MRL_DEV int lane_body(int l) { return (int)((R::BODY >> (4 * l)) & 15u); }
template <class R>
MRL_DEV int lane_joint(int e, int l) { return (int)(((e ? R::JOINT[1] : R::JOINT[0]) >> (4 * l)) & 15u); }

// true when the row's joints are wired as the lanes assume.  (A motor that no step sets keeps the caller's torque, and a
// negative one turns both bodies the same way, which the halves do not.)
template <class L, class T, class R>
MRL_DEV bool body_lanes_row_ok(const float *row) {
    if ((int)row[L::JOINT_COUNT_OFF] != L::MAX_JOINTS) return false;
    bool ok = true;
#pragma unroll
    for (int j = 0; j < L::MAX_JOINTS; ++j) {
        const float *J = row + L::JOINTS_OFF + j * JOINT_SIZE;
        ok = ok && (int)J[J_TYPE] == 0 && (int)J[J_BODY_A] == T::a(j) && (int)J[J_BODY_B] == T::b(j);
        if (!R::MOTOR) ok = ok && (((int)J[J_FLAGS] & JF_MOTOR) == 0 || J[J_MAX_TORQUE] >= 0.0f);
    }
    return ok;
}

// true when the joints of such a row have the terms that R names, limits in order and something to turn
template <class L, class T, class R>
MRL_DEV bool body_lanes_row_usual(const float *row) {
    constexpr int FLAGS = JF_LIMIT | (R::SPRING ? JF_SPRING : 0) | (R::MOTOR ? JF_MOTOR : 0);
    bool usual = true;
#pragma unroll
    for (int j = 0; j < L::MAX_JOINTS; ++j) {
        const float *J = row + L::JOINTS_OFF + j * JOINT_SIZE;
        const float ia = row[L::BODIES_OFF + T::a(j) * BODY_SIZE + IDX_INV_INERTIA];
        const float ib = row[L::BODIES_OFF + T::b(j) * BODY_SIZE + IDX_INV_INERTIA];
        usual = usual && ((int)J[J_FLAGS] & (JF_LIMIT | JF_SPRING | JF_MOTOR)) == FLAGS && J[J_LO] <= J[J_HI] && ia + ib > 1e-10f;
    }
    return usual;
}

// the velocities of the lane's body are B.vx[0] .., its place B.x[0] ..
typedef RegBodies<OneBody> LaneBody;

template <class L>
MRL_DEV void lane_body_load(LaneBody &B, const float *row, int body) {
    const float *P = row + L::BODIES_OFF + body * BODY_SIZE;
    B.x[0] = P[IDX_X]; B.y[0] = P[IDX_Y]; B.ang[0] = P[IDX_ANGLE];
    B.vx[0] = P[IDX_VX]; B.vy[0] = P[IDX_VY]; B.w[0] = P[IDX_OMEGA];
    B.im[0] = P[IDX_INV_MASS]; B.ii[0] = P[IDX_INV_INERTIA];
}
// bodies back and forces cleared (lanes with a body)
template <class L>
MRL_DEV void lane_body_store(const LaneBody &B, float *row, int body) {
    float *P = row + L::BODIES_OFF + body * BODY_SIZE, *F = row + L::FORCES_OFF + body * 3;
    P[IDX_X] = B.x[0]; P[IDX_Y] = B.y[0]; P[IDX_ANGLE] = B.ang[0];
    P[IDX_VX] = B.vx[0]; P[IDX_VY] = B.vy[0]; P[IDX_OMEGA] = B.w[0];
    F[0] = 0.0f; F[1] = 0.0f; F[2] = 0.0f;
}

// integrators/euler.mojo:82-130, :132-183
MRL_DEV void lane_integrate_velocity(LaneBody &B, float fx, float fy, float tau, float gx, float gy, float dt) {
    const bool moves = B.im[0] != 0.0f;
    const float vx = B.vx[0] + (fx * B.im[0] + gx) * dt, vy = B.vy[0] + (fy * B.im[0] + gy) * dt;
    const float w = B.w[0] + tau * B.ii[0] * dt;
    B.vx[0] = moves ? vx : B.vx[0];
    B.vy[0] = moves ? vy : B.vy[0];
    B.w[0] = moves ? w : B.w[0];
}
MRL_DEV void lane_integrate_position(LaneBody &B, float dt) {
    const float pi_val = (float)3.14159265358979323846;
    const float two_pi = (float)(2.0 * 3.14159265358979323846);
    const bool moves = B.im[0] != 0.0f;
    const float x = B.x[0] + B.vx[0] * dt, y = B.y[0] + B.vy[0] * dt;
    const float angle = B.ang[0] + B.w[0] * dt;
    const float d1 = angle - two_pi, d2 = d1 - two_pi, u1 = angle + two_pi, u2 = u1 + two_pi;
    float a = angle > pi_val ? (d1 > pi_val ? d2 : d1) : angle;
    a = angle < -pi_val ? (u1 < -pi_val ? u2 : u1) : a;
    a = (angle > 100.0f || angle < -100.0f) ? 0.0f : a;
    B.x[0] = moves ? x : B.x[0];
    B.y[0] = moves ? y : B.y[0];
    B.ang[0] = moves ? a : B.ang[0];
}

// ---------------------------------------------------------------- contacts of the lane's body

struct LaneContact {
    ContactFixed f;
    float jn, jt;
    float push_x, push_y;   // what a position sweep moves the body by (solvers/impulse.mojo:333-402; the depth stays as detected)
    float push;             // 1: it does (a flag in a vector register: lane masks are short)

    MRL_DEV void prepare(const LaneBody &B, bool live, float px, float py, float nx, float ny, float depth, float baumgarte) {
        f = contact_prepare<OneBody>(B, 0, px, py, nx, ny);
        jn = jt = 0.0f;
        const float correction = depth - SOLVER_SLOP, total = B.im[0] + 0.0f;
        push = live && !(correction <= 0.0f) && total != 0.0f ? 1.0f : 0.0f;
        const float by = baumgarte * correction * B.im[0] / total;
        push_x = nx * by;
        push_y = ny * by;
    }
    MRL_DEV void position(LaneBody &B) const {
        const float x = B.x[0] + push_x, y = B.y[0] + push_y;
        B.x[0] = push != 0.0f ? x : B.x[0];
        B.y[0] = push != 0.0f ? y : B.y[0];
    }
};

// The records of an env's merged contact list (in LDS) that are of this lane's body, in list order: the first REG in
// registers, any others in their records, as LdsContacts keeps them.
template <class L, int REG>
struct LaneListContacts {
    LaneContact c[REG];
    int count;
    unsigned rest;
    float *cts;

    static MRL_DEV LaneListContacts none() {
        LaneListContacts l;
        l.count = 0;
        l.rest = 0;
        l.cts = nullptr;
        return l;
    }
    MRL_DEV float *masses(int i) const { return cts + L::MAX_CONTACTS * CONTACT_SIZE + 4 * i; }

    MRL_DEV void load(const LaneBody &B, float *contacts, int n, int body, float baumgarte) {
        cts = contacts;
        unsigned mine = 0;   // (every slot is read, the count cuts afterwards)
#pragma unroll
        for (int i = 0; i < L::MAX_CONTACTS; ++i) mine |= (unsigned)((int)cts[i * CONTACT_SIZE + C_BODY_A] == body) << i;
        mine &= n >= 32 ? 0xFFFFFFFFu : ((1u << n) - 1u);
        count = __popc(mine);
        rest = mine;
#pragma unroll
        for (int r = 0; r < REG; ++r) {
            if (!any_lane(r < count)) break;
            const int i = r < count ? __ffs((int)rest) - 1 : 0;
            rest &= rest - 1u;
            const float *C = cts + i * CONTACT_SIZE;
            c[r].prepare(B, r < count, C[C_PX], C[C_PY], C[C_NX], C[C_NY], C[C_DEPTH], baumgarte);
        }
        if (!any_lane(rest != 0)) return;
        for (unsigned m = rest; m; m &= m - 1) {
            const int i = __ffs((int)m) - 1;
            float *C = cts + i * CONTACT_SIZE, *K = masses(i);
            const ContactFixed f = contact_prepare<OneBody>(B, 0, C[C_PX], C[C_PY], C[C_NX], C[C_NY]);
            C[C_PX] = f.ra_x; C[C_PY] = f.ra_y;
            K[0] = f.k; K[1] = f.k_t; K[2] = f.rk; K[3] = f.rk_t;
        }
    }
    MRL_DEV void velocity(LaneBody &B, float friction, float restitution) {
#pragma unroll
        for (int r = 0; r < REG; ++r) {
            if (!any_lane(r < count)) return;
            contact_velocity<OneBody>(B, 0, c[r].f, c[r].jn, c[r].jt, friction, restitution, r < count);
        }
        if (!any_lane(rest != 0)) return;
        for (unsigned m = rest; m; m &= m - 1) {
            const int i = __ffs((int)m) - 1;
            float *C = cts + i * CONTACT_SIZE;
            const float *K = masses(i);
            ContactFixed f;
            f.nx = C[C_NX]; f.ny = C[C_NY]; f.ra_x = C[C_PX]; f.ra_y = C[C_PY];
            f.inv_mass_a = B.im[0]; f.inv_inertia_a = B.ii[0];
            f.k = K[0]; f.k_t = K[1]; f.rk = K[2]; f.rk_t = K[3];
            float jn = C[C_JN], jt = C[C_JT];
            contact_velocity<OneBody>(B, 0, f, jn, jt, friction, restitution);
            C[C_JN] = jn; C[C_JT] = jt;
        }
    }
    MRL_DEV void position(LaneBody &B, float baumgarte) const {
#pragma unroll
        for (int r = 0; r < REG; ++r) {
            if (!any_lane(r < count)) return;
            c[r].position(B);
        }
        if (!any_lane(rest != 0)) return;
        for (unsigned m = rest; m; m &= m - 1) {
            const int i = __ffs((int)m) - 1;
            const float *C = cts + i * CONTACT_SIZE;
            contact_position<OneBody>(B, 0, C[C_NX], C[C_NY], C[C_DEPTH], baumgarte);
        }
    }
};

// ---------------------------------------------------------------- joints

// a lane's place in the wiring, l: lane in the env's group
template <class R>
struct LaneSlots {
    static constexpr int S = R::SLOTS;
    bool in[S], child[2];

    MRL_DEV explicit LaneSlots(int l) {
#pragma unroll
        for (int s = 0; s < S; ++s) in[s] = ((R::IN[s] >> l) & 1u) != 0;
        child[0] = ((R::CHILD[0] >> l) & 1u) != 0;
        child[1] = ((R::CHILD[1] >> l) & 1u) != 0;
    }

    // the value that my partner holds, in my slot of parity E
    template <int E>
    MRL_DEV float partner(float v) const {
        const float a = dpp_xchg<R::CTRL[E]>(v);
        if constexpr (E + 2 < S) {
            if constexpr (R::CTRL[E + 2] != R::CTRL[E]) {
                const float b = dpp_xchg<R::CTRL[E + 2]>(v);
                return in[E + 2] ? b : a;
            }
        }
        return a;
    }
    // ... and my parent's, of a value that each lane holds per parity
    MRL_DEV float parent(float v0, float v1) const {
        const float a = partner<0>(v0), b = partner<1>(v1);
        return child[0] ? a : b;
    }
};

template <class R, bool ANY>
struct LaneJoints : LaneSlots<R> {
    using Slots = LaneSlots<R>;
    using Slots::S;
    using Slots::in;
    using Slots::child;
    using Slots::parent;
    static constexpr bool SPRING = R::SPRING || ANY, MOTOR = R::MOTOR || ANY, ALL = ANY;
    // by parity of the slot, from the lane's own side (the parent's are the child's negated, its bounds swapped)
    float ax[2], ay[2];                  // my anchor
    float eff[2], reff[2];
    float lo[2], hi[2], ref[2], speed[2], max_impulse[2], damp[2];
    bool springs[2], motors[2];          // (ANY)
    // of the joint whose child I am
    float p_im, p_ii, c_ref, c_lo, c_hi, c_stiff;
    // fixed during a velocity phase
    float rx[2], ry[2], k11[2], k12[2], k22[2], below[2], above[2], spring[2];

    MRL_DEV explicit LaneJoints(int l) : Slots(l) {}

    // whether the joint whose child I am, if there is one, has the terms R names
    template <class L>
    MRL_DEV bool usual(const float *row, int l, const LaneBody &B) const {
        constexpr int FLAGS = JF_LIMIT | (R::SPRING ? JF_SPRING : 0) | (R::MOTOR ? JF_MOTOR : 0);
        const int flags = (int)row[L::JOINTS_OFF + lane_joint<R>(child[0] ? 0 : 1, l) * JOINT_SIZE + J_FLAGS];
        return !(child[0] || child[1]) || ((flags & (JF_LIMIT | JF_SPRING | JF_MOTOR)) == FLAGS && c_lo <= c_hi && p_ii + B.ii[0] > 1e-10f);
    }

    // the constants of a step
    template <class L>
    MRL_DEV void load(const float *row, int l, const LaneBody &B, float dt) {
        p_im = parent(B.im[0], B.im[0]); p_ii = parent(B.ii[0], B.ii[0]);
        eff[0] = this->template partner<0>(B.ii[0]) + B.ii[0];
        eff[1] = this->template partner<1>(B.ii[0]) + B.ii[0];
        // (a limit that is not there: bounds that no angle is beyond)
        const float none = __builtin_nanf("");
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float *J = row + L::JOINTS_OFF + lane_joint<R>(e, l) * JOINT_SIZE;
            ax[e] = J[child[e] ? J_BX : J_AX]; ay[e] = J[child[e] ? J_BY : J_AY];
            const float l0 = J[J_LO], h0 = J[J_HI], r0 = J[J_REF];
            lo[e] = child[e] ? l0 : -h0; hi[e] = child[e] ? h0 : -l0; ref[e] = child[e] ? r0 : -r0;
            if (MOTOR) {
                const float v0 = J[J_MOTOR_SPEED];
                speed[e] = child[e] ? v0 : -v0;
                max_impulse[e] = J[J_MAX_TORQUE] * dt;
            }
            if (SPRING) damp[e] = J[J_DAMP];
            if (ANY) {
                const int flags = (int)J[J_FLAGS];
                const bool turns = eff[e] > 1e-10f, limited = turns && (flags & JF_LIMIT) != 0;
                springs[e] = turns && (flags & JF_SPRING) != 0;
                motors[e] = turns && (flags & JF_MOTOR) != 0;
                lo[e] = limited ? lo[e] : none;
                hi[e] = limited ? hi[e] : none;
                eff[e] = turns ? eff[e] : 1.0f;
            }
        }
        const float *J = row + L::JOINTS_OFF + lane_joint<R>(child[0] ? 0 : 1, l) * JOINT_SIZE;
        c_ref = J[J_REF]; c_lo = J[J_LO]; c_hi = J[J_HI];
        if (SPRING) c_stiff = J[J_STIFF];
        if (ANY) {
            const bool limited = ((int)J[J_FLAGS] & JF_LIMIT) != 0 && p_ii + B.ii[0] > 1e-10f;
            c_lo = limited ? c_lo : none;
            c_hi = limited ? c_hi : none;
        }
        reff[0] = 1.0f / eff[0];
        reff[1] = 1.0f / eff[1];
    }

    // lever arms, K^-1 and the angle-dependent spring / limit terms for the velocity phase (joints/revolute.mojo:90-200):
    // each joint's by its child, which hands them to its parent
    MRL_DEV void prepare(const LaneBody &B, float sn, float cs) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            rx[e] = ax[e] * cs - ay[e] * sn;
            ry[e] = ax[e] * sn + ay[e] * cs;
        }
        const float prx = parent(rx[0], rx[1]), pry = parent(ry[0], ry[1]), p_ang = parent(B.ang[0], B.ang[0]);
        float c11, c12, c22;
        joint_inverse(p_im, p_ii, B.im[0], B.ii[0], prx, pry, child[0] ? rx[0] : rx[1], child[0] ? ry[0] : ry[1], c11, c12, c22);
        const float rel_angle = B.ang[0] - p_ang - c_ref, inf = __builtin_inff();
        const float c_below = rel_angle <= c_lo ? 0.0f : -inf;
        const float c_above = !(rel_angle <= c_lo) && rel_angle >= c_hi ? 0.0f : inf;
        const float c_spring = SPRING ? -c_stiff * rel_angle : 0.0f;
        hand<0>(c11, c12, c22, c_below, c_above, c_spring);
        hand<1>(c11, c12, c22, c_below, c_above, c_spring);
    }
    template <int E>
    MRL_DEV void hand(float c11, float c12, float c22, float c_below, float c_above, float c_spring) {
        auto partner = [&](float v) { return Slots::template partner<E>(v); };
        const float h11 = partner(c11), h12 = partner(c12), h22 = partner(c22);
        const float hb = partner(c_below), ha = partner(c_above);
        k11[E] = child[E] ? c11 : h11; k12[E] = child[E] ? c12 : h12; k22[E] = child[E] ? c22 : h22;
        below[E] = child[E] ? c_below : -ha;
        above[E] = child[E] ? c_above : -hb;
        if (SPRING) {
            const float hs = partner(c_spring);
            spring[E] = child[E] ? c_spring : -hs;
        }
    }

    // slot SL of a velocity sweep (joints/revolute.mojo:100-320)
    template <int SL>
    MRL_DEV void velocity_slot(LaneBody &B, float dt) const {
        constexpr int e = SL & 1, ctrl = R::CTRL[SL];
        const float im = B.im[0], ii = B.ii[0], w = B.w[0];
        const float px = B.vx[0] - w * ry[e], py = B.vy[0] + w * rx[e];
        const float dx = px - dpp_xchg<ctrl>(px), dy = py - dpp_xchg<ctrl>(py);
        const float jx = k11[e] * dx + k12[e] * dy, jy = k12[e] * dx + k22[e] * dy;
        const float vx = B.vx[0] - im * jx, vy = B.vy[0] - im * jy;
        float cw = w - ii * (rx[e] * jy - ry[e] * jx);
        if (SPRING) {
            const float torque = spring[e] - damp[e] * (w - dpp_xchg<ctrl>(w));   // (velocities from before the point impulse)
            const float to = cw + div_by(ii * (torque * dt), eff[e], reff[e]);
            cw = !ANY || springs[e] ? to : cw;
        }
        {
            const float d = cw - dpp_xchg<ctrl>(cw);
            const float q = div_by(d, eff[e], reff[e]);
            const bool acts = (d < below[e] || d > above[e]) && q != 0.0f;
            const float to = cw - ii * q;
            cw = acts ? to : cw;
        }
        if (MOTOR) {
            const float d = cw - dpp_xchg<ctrl>(cw);
            float q = div_by(speed[e] - d, eff[e], reff[e]);
            q = q > max_impulse[e] ? max_impulse[e] : q;
            q = q < -max_impulse[e] ? -max_impulse[e] : q;
            const float to = cw + ii * q;
            cw = !ANY || motors[e] ? to : cw;
        }
        B.vx[0] = in[SL] ? vx : B.vx[0];
        B.vy[0] = in[SL] ? vy : B.vy[0];
        B.w[0] = in[SL] ? cw : B.w[0];
    }
    MRL_DEV void velocity_sweep(LaneBody &B, float dt) const {
        velocity_slot<0>(B, dt);
        velocity_slot<1>(B, dt);
        if constexpr (S > 2) velocity_slot<2>(B, dt);
        if constexpr (S > 3) velocity_slot<3>(B, dt);
    }

    // slot SL of a position sweep (joints/revolute.mojo:323-495); the lanes that moved: zero when no joint of the
    // wavefront's is off by more than the slop
    template <int SL>
    MRL_DEV uint64_t position_slot(LaneBody &B, float sn, float cs, float baumgarte) const {
        constexpr int e = SL & 1, ctrl = R::CTRL[SL];
        const float im = B.im[0], ii = B.ii[0];
        const float qx = ax[e] * cs - ay[e] * sn, qy = ax[e] * sn + ay[e] * cs;
        const float px = B.x[0] + qx, py = B.y[0] + qy;
        const float dx = px - dpp_xchg<ctrl>(px), dy = py - dpp_xchg<ctrl>(py);
        const bool off = in[SL] && !(dx * dx + dy * dy < SOLVER_SLOP_SQ);
        const uint64_t moved = __builtin_amdgcn_ballot_w64(off);
        if (moved == 0) return 0;
        // K^-1 and the correction by the child
        float i11, i12, i22;
        joint_inverse(p_im, p_ii, im, ii, dpp_xchg<ctrl>(qx), dpp_xchg<ctrl>(qy), qx, qy, i11, i12, i22);
        const float cgx = baumgarte * (i11 * dx + i12 * dy), cgy = baumgarte * (i12 * dx + i22 * dy);
        const float hgx = dpp_xchg<ctrl>(cgx), hgy = dpp_xchg<ctrl>(cgy);
        const float gx = child[e] ? cgx : -hgx, gy = child[e] ? cgy : -hgy;
        const float x = B.x[0] - im * gx, y = B.y[0] - im * gy;
        float a = B.ang[0] - ii * (qx * gy - qy * gx);
        {
            const float rel = a - dpp_xchg<ctrl>(a) - ref[e];
            const bool low = rel < lo[e], high = rel > hi[e];
            // (beyond both: of limits the wrong way round, where the child's lower one counts)
            const bool to_lo = ANY && !child[e] ? !high : low;
            const float c = baumgarte * ((to_lo ? lo[e] : hi[e]) - rel);
            const float to = a + div_by(ii * c, eff[e], reff[e]);
            a = (low || high) && c != 0.0f ? to : a;
        }
        B.x[0] = off ? x : B.x[0];
        B.y[0] = off ? y : B.y[0];
        B.ang[0] = off ? a : B.ang[0];
        return moved;
    }

    // The position sweeps from (B, sn, cs), which keep in step but for the last slot's turn where nothing reads it.
    // NEAR: angles are taken to be within 2^20; returns false when one was not, and the results are void.
    template <bool NEAR, int ITERS, class Contacts>
    MRL_DEV bool position_sweeps(LaneBody &B, float &sn, float &cs, const Contacts &contacts, float baumgarte,
                                 const SinCosK &K) const {
        float widest = 0.0f;
        uint64_t stale = 0;   // not zero: a body has turned since its sine and cosine were taken
        auto turn = [&]() {
            if (NEAR) sincos32_near(B.ang[0], sn, cs, K);
            else sincos32(B.ang[0], sn, cs, K);
            widest = fmaxf(widest, fabsf(B.ang[0]));
        };
#pragma unroll 1
        for (int it = 0; it < ITERS; ++it) {
            contacts.position(B, baumgarte);
            auto slot = [&](auto sl) {
                constexpr int SL = decltype(sl)::value;
                const uint64_t moved = position_slot<SL>(B, sn, cs, baumgarte);
                if (SL == S - 1 && !R::LAST_TURNS_FIRST) {
                    // (the bodies of the last slot are next read behind another turn, if at all)
                    if (it + 1 < ITERS || !R::ANGLES_AFTER) { stale = stale | moved; return; }
                } else if (SL == S - 1 && it + 1 == ITERS && !R::ANGLES_AFTER) {
                    return;
                }
                if ((moved | stale) != 0) turn();
                stale = 0;
            };
            slot(std::integral_constant<int, 0>{});
            slot(std::integral_constant<int, 1>{});
            if constexpr (S > 2) slot(std::integral_constant<int, 2>{});
            if constexpr (S > 3) slot(std::integral_constant<int, 3>{});
        }
        return !NEAR || !any_lane(widest > 0x1p20f);
    }
};

// One physics step (sub-step): velocity sweeps, integration, position sweeps.  In: velocities with the forces applied,
// (sn, cs) of the angles, contacts loaded; out: (sn, cs) of the new angles where R::ANGLES_AFTER.
template <class R, bool ANY, int VEL, int POS, class Contacts>
MRL_DEV void body_lanes_solve(LaneBody &B, LaneJoints<R, ANY> &J, Contacts &contacts, float &sn, float &cs, float dt, float friction,
                              float restitution, float baumgarte) {
    J.prepare(B, sn, cs);
#pragma unroll 1
    for (int it = 0; it < VEL; ++it) {
        contacts.velocity(B, friction, restitution);
        J.velocity_sweep(B, dt);
    }
    lane_integrate_position(B, dt);
    const SinCosK K = SinCosK::held();
    sincos32(B.ang[0], sn, cs, K);
    const float x = B.x[0], y = B.y[0], ang = B.ang[0], s0 = sn, c0 = cs;
    if (__builtin_expect(J.template position_sweeps<true, POS>(B, sn, cs, contacts, baumgarte, K), 1)) return;
    B.x[0] = x; B.y[0] = y; B.ang[0] = ang;
    sn = s0; cs = c0;
    J.template position_sweeps<false, POS>(B, sn, cs, contacts, baumgarte, K);
}

// f(the lane's joints): J as loaded, or with every term decided lane by lane where one of the wavefront's lanes is `odd`.
// us where every row is, such rows in the one-lane form : now: HalfCheetah step of 1000 / 65536 envs 190 : 42, 788 : 206,
// rollout of 4096 envs (H = 64, 32 steps) 7659 : 1350; BipedalWalker 82 : 25, 798 : 178, 2048 envs 2661 : 845.
template <class L, class R, class F>
MRL_DEV void with_joints(LaneJoints<R, false> &J, const float *row, int l, const LaneBody &B, float dt, bool odd, F &&f) {
    if (__builtin_expect(any_lane(odd), 0)) {
        LaneJoints<R, true> A(l);
        A.template load<L>(row, l, B, dt);
        f(A);
    } else {
        f(J);
    }
}

}  // namespace mrl
