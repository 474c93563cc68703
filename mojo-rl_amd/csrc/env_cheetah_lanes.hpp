// HalfCheetah's env step with one lane per BODY: eight lanes per env (seven bodies, one idle), eight
// envs per wavefront.
//
// With one lane per env the step is one long instruction stream per wavefront (5 sub-steps x 6
// Gauss-Seidel sweeps over 6 joints and up to 14 contacts, each body picked with a 7-way select
// chain).  Much of that stream is work on different bodies that does not interact:
//   * integration, ground detection and the contact sweeps touch only the contact's own body (the
//     ground is the other party), so contacts of different bodies commute exactly: every lane runs
//     the contacts of its own body, in vertex order, at the place in the sweep where the one-lane
//     form runs all contacts;
//   * the joint sweep visits joints 0 .. 5 in order, but after joint 0 (torso - back thigh) the back
//     leg's joints 1, 2 touch bodies 1, 2, 3 only and the front leg's joints 3, 4, 5 bodies 0, 4, 5, 6:
//     two chains without a body in common, which run side by side -- four joint slots per sweep
//     instead of six.  In a slot the CHILD body's lane does the joint (parent state fetched from the
//     parent's lane, parent result handed back), so every lane holds its body in plain registers.
// Same operations on the same values in an order the arithmetic cannot tell from the one-lane form's:
// the results are identical bit for bit (the parity tests compare both with the oracle).
//
// The wiring is HalfCheetah's (cheetah_planar_v2.mojo: torso 0; back thigh / shin / foot 1, 2, 3;
// front 4, 5, 6; joint j joins body j + 1 to its parent).  A row whose joint table or shapes differ
// from that is stepped by the one-lane form instead (lanes_row_ok, tested by the caller).
#pragma once
#include "env_walkers.hpp"

namespace mrl {
namespace hc {

constexpr int LANES_PER_ENV = 8;

// LDS writes of this wavefront's lanes become visible to its other lanes
MRL_DEV void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// lanes of one env sit side by side: value of lane `src` of my group
template <class V>
MRL_DEV V group_get(V v, int base, int src) { return __shfl(v, base + src, 64); }

// The two exchanges of a joint slot as DPP row shifts (register to register, no trip through the LDS
// crossbar).  Rows are 16 lanes, so the two groups of a row shift side by side; a lane at a group's
// edge picks up a neighbour group's value that it never uses.
//   from_parent: every child's parent is the body before it, except the front thigh (4), whose
//                parent is the torso four lanes down;
//   from_kid<S>: the parent's lane takes the result of its child in slot S -- the next lane, except
//                the torso in slot 1, whose child is the front thigh four lanes up.
MRL_DEV float dpp_row_shr1(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x111, 0xF, 0xF, false)); }
MRL_DEV float dpp_row_shr4(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x114, 0xF, 0xF, false)); }
MRL_DEV float dpp_row_shl1(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x101, 0xF, 0xF, false)); }
MRL_DEV float dpp_row_shl4(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x104, 0xF, 0xF, false)); }
MRL_DEV float from_parent(float v, int b) {
    const float one = dpp_row_shr1(v), four = dpp_row_shr4(v);
    return b == 4 ? four : one;
}
template <int S>
MRL_DEV float from_kid(float v, int b) {
    const float one = dpp_row_shl1(v);
    if (S == 1) {
        const float four = dpp_row_shl4(v);
        return b == 0 ? four : one;
    }
    return one;
}

MRL_DEV float from_kid_slot(int s, float v, int b) {
    const float one = dpp_row_shl1(v), four = dpp_row_shl4(v);
    return (s == 1 && b == 0) ? four : one;
}

// true when the row has the wiring and shapes this form assumes
MRL_DEV bool lanes_row_ok(const float *row, const float *shapes) {
    if ((int)row[L::JOINT_COUNT_OFF] != 6) return false;
    bool ok = true;
    for (int j = 0; j < 6; ++j) {
        const float *J = row + L::JOINTS_OFF + j * JOINT_SIZE;
        ok = ok && (int)J[J_TYPE] == 0 && (int)J[J_BODY_A] == Topology::a(j) && (int)J[J_BODY_B] == Topology::b(j);
    }
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

// The env step of hc::step_row by the eight lanes of an env's group (all lanes of the wavefront call
// it together; `lane` = lane in the wavefront, `row` = the group's env row in LDS, `action` = its six
// action components).  Lane 0 of the group returns reward / done.
MRL_DEV void step_lanes(float *row, const float *shapes, const float *action, int lane, float &reward, float &done) {
    const int b = lane & 7, base = lane & ~7;
    const bool body = b < 7;
    // ---- wiring seen from this lane: as the child of joint b - 1 (bodies 1 .. 6) ...
    const bool child = b >= 1 && b <= 6;
    const int j = child ? b - 1 : 0;
    const int par = (b == 1 || b == 4) ? 0 : (child ? b - 1 : 0);
    const int myslot = b == 1 ? 0 : (b == 2 || b == 4) ? 1 : (b == 3 || b == 5) ? 2 : b == 6 ? 3 : -1;
    // ... and as the parent of the joint that runs in slot s: bit s of kidmask (the torso has a child in
    // slots 0 and 1, the front thigh in slot 1 being the one that sits four lanes up)
    const int kidmask = b == 0 ? 3 : b == 1 ? 2 : (b == 2 || b == 4) ? 4 : b == 5 ? 8 : 0;

    const float gx = (float)0.0, gy = (float)-9.81, dt = (float)0.01, friction = (float)0.9, restitution = (float)0.0;
    const float baumgarte = (float)0.2;

    // ---- the action into the joint motors (child lane of joint j), as hc::step_row does
    float *J = row + L::JOINTS_OFF + j * JOINT_SIZE;
    float motor_speed = 0.0f, max_torque = 0.0f;
    if (child) {
        float v = action[j];
        v = v < 1.0f ? v : 1.0f;
        v = v > -1.0f ? v : -1.0f;
        const double av = (double)v;
        motor_speed = (av >= 0.0 ? 1.0f : -1.0f) * 1000.0f;
        max_torque = (float)(1.0 * ::fabs(av));
        J[J_MOTOR_SPEED] = motor_speed;
        J[J_MAX_TORQUE] = max_torque;
    }
    const float lax = J[J_AX], lay = J[J_AY], lbx = J[J_BX], lby = J[J_BY];
    const float jref = J[J_REF], jlo = J[J_LO], jhi = J[J_HI], jstiff = J[J_STIFF], jdamp = J[J_DAMP];
    const int jflags = (int)J[J_FLAGS];

    // ---- my body
    float *Bp = row + L::BODIES_OFF + (body ? b : 0) * BODY_SIZE;
    float x = Bp[IDX_X], y = Bp[IDX_Y], ang = Bp[IDX_ANGLE], vx = Bp[IDX_VX], vy = Bp[IDX_VY], w = Bp[IDX_OMEGA];
    const float im = Bp[IDX_INV_MASS], ii = Bp[IDX_INV_INERTIA];
    float fx = row[L::FORCES_OFF + (body ? b : 0) * 3], fy = row[L::FORCES_OFF + (body ? b : 0) * 3 + 1],
          tau = row[L::FORCES_OFF + (body ? b : 0) * 3 + 2];
    const float *S = shapes + (int)Bp[IDX_SHAPE] * SHAPE_SIZE;
    const int n_verts = (int)S[1];
    float lvx[4], lvy[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) { lvx[v] = S[2 + v * 2]; lvy[v] = S[3 + v * 2]; }
    const float p_im = from_parent(im, b), p_ii = from_parent(ii, b);
    JointSweep q;   // the joint whose child I am
    q.ima = p_im; q.iia = p_ii; q.imb = im; q.iib = ii;
    q.eff = p_ii + ii;
    q.reff = 1.0f / q.eff;
    const bool turns = q.eff > 1e-10f, limited = turns && (jflags & JF_LIMIT) != 0;
    q.spring = turns && (jflags & JF_SPRING) != 0;
    q.motor = turns && (jflags & JF_MOTOR) != 0;
    q.damp = jdamp;
    q.motor_speed = motor_speed;
    q.max_impulse = max_torque * dt;
    const double x_before = (double)x;   // meaningful on lane 0 (the torso)

    // sine and cosine of my body's angle, kept in step with it (recomputed whenever the angle may have
    // changed): the same values that the one-lane form recomputes at every use
    float sin_a, cos_a;
    sincos32(ang, sin_a, cos_a);
    int kept = 0;   // my body's contacts of the current sub-step that made the list
    for (int sub = 0; sub < 5; ++sub) {
        // ---- integrate velocities (integrators/euler.mojo:82-130)
        if (im != 0.0f) {
            vx = vx + (fx * im + gx) * dt;
            vy = vy + (fy * im + gy) * dt;
            w = w + tau * ii * dt;
        }
        fx = fy = tau = 0.0f;   // the forces are cleared at the end of every sub-step
        // ---- ground contacts of my body, vertex order (collision/flat_terrain.mojo:69-204); the list
        // of an env is cut at MAX_CONTACTS in (body, vertex) order: contacts before mine are counted
        float cpx[4] = {0.0f, 0.0f, 0.0f, 0.0f}, cpy[4] = {0.0f, 0.0f, 0.0f, 0.0f}, cdepth[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        int found = 0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float world_x = x + lvx[v] * cos_a - lvy[v] * sin_a;
            const float world_y = y + lvx[v] * sin_a + lvy[v] * cos_a;
            const float penetration = 0.0f - world_y;
            const bool hit = body && v < n_verts && penetration > 0.0f;
            // compacted in vertex order
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (hit && found == c) { cpx[c] = world_x; cpy[c] = world_y; cdepth[c] = penetration; }
            }
            found += hit ? 1 : 0;
        }
        int before = 0;   // contacts of the bodies before mine
#pragma unroll
        for (int o = 0; o < 7; ++o) {
            const int c = group_get(found, base, o);
            before += o < b ? c : 0;
        }
        kept = L::MAX_CONTACTS - before;
        kept = kept < 0 ? 0 : (kept > found ? found : kept);
        // ---- what stays fixed during the velocity phase: contact lever arms and effective masses
        // (solvers/impulse.mojo:115-190) ...
        const float nx = 0.0f, ny = 1.0f;
        ContactFixed cf[4];
        float jn[4], jt[4], push_out[4];
        RegBodies<OneBody> B1;
        B1.x[0] = x; B1.y[0] = y; B1.im[0] = im; B1.ii[0] = ii;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            jn[c] = jt[c] = push_out[c] = 0.0f;
            cf[c] = ContactFixed{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f, 1.0f, 1.0f, 1.0f};
            if (!__any(c < kept)) continue;
            cf[c] = contact_prepare<OneBody>(B1, 0, cpx[c], cpy[c], nx, ny);
            // what each position sweep moves the body up by (solvers/impulse.mojo:333-402): the depth stays as detected
            const float total = im + 0.0f;
            const float correction = cdepth[c] - SOLVER_SLOP;
            if (c < kept && correction > 0.0f && total != 0.0f) push_out[c] = baumgarte * correction * im / total;
        }
        // ... and the joint's lever arms, K^-1 and limit angle (joints/revolute.mojo:90-200), by the child
        const float p_sin = from_parent(sin_a, b), p_cos = from_parent(cos_a, b);
        const float p_ang = from_parent(ang, b);
        const float rax = lax * p_cos - lay * p_sin, ray = lax * p_sin + lay * p_cos;
        const float rbx = lbx * cos_a - lby * sin_a, rby = lbx * sin_a + lby * cos_a;
        q.rax = rax; q.ray = ray; q.rbx = rbx; q.rby = rby;
        joint_inverse(p_im, p_ii, im, ii, rax, ray, rbx, rby, q.inv_k11, q.inv_k12, q.inv_k22);
        const float angle_error = (ang - p_ang) - jref;
        q.spring_term = -jstiff * angle_error;
        joint_limits(q, limited, ang - p_ang - jref, jlo, jhi);
        JointTerms any{false, false, false};
        any.add(q, child);

        // ---- velocity iterations: my contacts, then the joints slot by slot
        for (int it = 0; it < 4; ++it) {
            B1.vx[0] = vx; B1.vy[0] = vy; B1.w[0] = w;
#pragma unroll
            for (int c = 0; c < 4; ++c) {   // solvers/impulse.mojo:192-331
                if (!__any(c < kept)) break;
                contact_velocity<OneBody>(B1, 0, cf[c], jn[c], jt[c], friction, restitution, c < kept);
            }
            vx = B1.vx[0]; vy = B1.vy[0]; w = B1.w[0];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                // the joint whose child I am, when its slot is s (in any other slot its result is not used)
                float vxa = from_parent(vx, b), vya = from_parent(vy, b), wa = from_parent(w, b);
                float vxb = vx, vyb = vy, wb = w;
                joint_velocity(q, any, dt, vxa, vya, wa, vxb, vyb, wb);
                // the parent takes its new velocity from the child of this slot, the child keeps its own
                const float g_vx = from_kid_slot(s, vxa, b), g_vy = from_kid_slot(s, vya, b), g_w = from_kid_slot(s, wa, b);
                if ((kidmask >> s) & 1) { vx = g_vx; vy = g_vy; w = g_w; }
                if (myslot == s) { vx = vxb; vy = vyb; w = wb; }
            }
        }
        // ---- integrate positions (integrators/euler.mojo:132-183)
        if (im != 0.0f) {
            const float pi_val = (float)3.14159265358979323846;
            const float two_pi = (float)(2.0 * 3.14159265358979323846);
            x = x + vx * dt;
            y = y + vy * dt;
            float angle = ang + w * dt;
            if (angle > 100.0f || angle < -100.0f) {
                angle = 0.0f;
            } else if (angle > pi_val) {
                angle = angle - two_pi;
                if (angle > pi_val) angle = angle - two_pi;
            } else if (angle < -pi_val) {
                angle = angle + two_pi;
                if (angle < -pi_val) angle = angle + two_pi;
            }
            ang = angle;
        }
        sincos32(ang, sin_a, cos_a);
        // ---- position iterations: my contacts (solvers/impulse.mojo:333-402), then the joints
        // (joints/revolute.mojo:323-495) slot by slot
        bool stale = false;   // my body has turned since its sine and cosine were taken
        for (int it = 0; it < 2; ++it) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (!__any(c < kept)) break;
                if (push_out[c] > 0.0f) {
                    x = x + nx * push_out[c];
                    y = y + ny * push_out[c];
                }
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                float xa = from_parent(x, b), ya = from_parent(y, b), angle_a = from_parent(ang, b);
                const float s_a = from_parent(sin_a, b), c_a = from_parent(cos_a, b);
                float xb = x, yb = y, angle_b = ang;
                const float r_ax = lax * c_a - lay * s_a, r_ay = lax * s_a + lay * c_a;
                const float r_bx = lbx * cos_a - lby * sin_a, r_by = lbx * sin_a + lby * cos_a;
                bool moved = false;
                if (myslot == s)
                    moved = joint_position(p_im, p_ii, im, ii, q.eff, q.reff, r_ax, r_ay, r_bx, r_by, limited, jlo, jhi, jref, baumgarte,
                                           xa, ya, angle_a, xb, yb, angle_b);
                const bool any_moved = __any(moved);   // (a joint within the slop hands back what it was given)
                if (any_moved) {
                    const float g_x = from_kid_slot(s, xa, b), g_y = from_kid_slot(s, ya, b);
                    const float g_a = from_kid_slot(s, angle_a, b);
                    if ((kidmask >> s) & 1) { x = g_x; y = g_y; ang = g_a; }
                    if (myslot == s) { x = xb; y = yb; ang = angle_b; }
                }
                // (the last slot moves the front shin and foot only, which the second iteration reads in its
                // last two slots, behind two more of these; after the second iteration the next sub-step reads all)
                if (it == 0 && s == 3) {
                    stale = any_moved;
                } else if (any_moved || stale) {
                    sincos32(ang, sin_a, cos_a);
                    stale = false;
                }
            }
        }
    }
    // ---- bodies and forces back into the row, then the rest of the step on the torso's lane
    if (body) {
        Bp[IDX_X] = x; Bp[IDX_Y] = y; Bp[IDX_ANGLE] = ang; Bp[IDX_VX] = vx; Bp[IDX_VY] = vy; Bp[IDX_OMEGA] = w;
        row[L::FORCES_OFF + b * 3] = 0.0f; row[L::FORCES_OFF + b * 3 + 1] = 0.0f; row[L::FORCES_OFF + b * 3 + 2] = 0.0f;
    }
    int penalised = 0;   // contacts of the last sub-step on anything but the feet (bodies 3 and 6)
#pragma unroll
    for (int o = 0; o < 7; ++o) {
        const int c = group_get(kept, base, o);
        penalised += (o != 3 && o != 6) ? c : 0;
    }
    // ---- the observation (hc::observe: the same expressions on the same values), every body's lane its own
    // entries: the torso its height, angle and velocity, a leg segment its angle and angular velocity
    // against its parent's
    {
        const double p_ang = (double)from_parent(ang, b), p_w = (double)from_parent(w, b);
        if (b == 0) {
            row[0] = y; row[1] = ang; row[8] = vx; row[9] = vy; row[10] = w;
        } else if (child) {
            row[2 + j] = (float)((double)ang - p_ang);
            row[11 + j] = (float)((double)w - p_w);
        }
    }
    if (b == 0) {
        double a[ACT];
#pragma unroll
        for (int k = 0; k < ACT; ++k) {
            float v = action[k];
            v = v < 1.0f ? v : 1.0f;
            v = v > -1.0f ? v : -1.0f;
            a[k] = (double)v;
        }
        step_tail(row, a, x_before, (double)x, (double)y, penalised, reward, done);
    }
    wave_sync_lds();   // the row is complete for whoever reads it next
}

}  // namespace hc
}  // namespace mrl
