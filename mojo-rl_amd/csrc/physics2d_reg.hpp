// Register-resident form of the physics2d solver sweeps.
//
// The Gauss-Seidel sweeps touch the same few bodies over and over (4-6 velocity + 2 position
// iterations, each over every contact and joint).  Running them out of LDS makes every sweep a
// chain of dependent LDS round trips; here the dynamic body state and the joint table (and, for
// short contact lists, the contacts) are loaded into registers once per step, all sweeps run on
// registers, and the bodies are written back once.  A body is picked by its (runtime) index with
// a select chain over the NUM_BODIES register copies; joints (and register-resident contacts) are
// walked with fully unrolled, predicated loops so that every array index is a compile-time
// constant.
//
// Two further reductions, both value-preserving:
//   * whatever a velocity sweep recomputes from quantities that cannot change during the velocity
//     phase (positions, angles, masses: lever arms, effective masses, the joints' K^-1, spring
//     and limit terms) is computed once per step with the same expressions;
//   * an env whose joints always connect the same bodies passes that wiring as a compile-time
//     topology; the select chains then fold away.  The row's joint table is compared against it
//     first and the generic path is taken if any lane disagrees.
//
// The arithmetic is that of physics2d.hpp statement for statement (same operations, same order),
// so both forms give identical results.  Contacts are body-vs-ground only (body B = -1), which is
// all the terrain detectors ever emit.
#pragma once
#include <type_traits>
#include <utility>
#include "physics2d.hpp"

namespace mrl {

// floats of LDS scratch per contact: the 9-float record plus four slots for the two effective masses
// and their reciprocals
constexpr int CONTACT_SCRATCH = CONTACT_SIZE + 4;

// Per-body quantities of an env live in short vector values (ext_vector_type), not in arrays:
// reading or replacing one element of a vector is an operation on the whole value, so the
// compiler keeps it in registers from the first pass on.  (Arrays indexed inside a loop only get
// constant indices after unrolling; by then selects of loads have been merged into loads from a
// computed address, and the whole struct stays in memory.)
template <int N>
struct BodyVec {
    static constexpr int W = N <= 2 ? 2 : N <= 4 ? 4 : N <= 8 ? 8 : 16;
    typedef float type __attribute__((ext_vector_type(W)));
};

// element i (runtime) of the first N lanes of a body vector, as a select chain
template <int N, class V, int... K>
MRL_DEV float sel_impl(const V &a, int i, std::integer_sequence<int, K...>) {
    float r = a[0];
    ((r = (i == K + 1) ? a[K + 1] : r), ...);
    return r;
}
template <int N, class V>
MRL_DEV float sel(const V &a, int i) {
    return sel_impl<N>(a, i, std::make_integer_sequence<int, N - 1>{});
}

// a[i] = v for runtime i < N
template <int N, class V, int... K>
MRL_DEV void put_impl(V &a, int i, float v, std::integer_sequence<int, K...>) {
    ((a[K] = (i == K) ? v : a[K]), ...);
}
template <int N, class V>
MRL_DEV void put(V &a, int i, float v) {
    put_impl<N>(a, i, v, std::make_integer_sequence<int, N>{});
}

// joint j connects bodies a(j) -> b(j); DynamicTopology reads them from the row
struct DynamicTopology {
    static constexpr bool STATIC = false;
    static constexpr MRL_DEV int a(int) { return 0; }
    static constexpr MRL_DEV int b(int) { return 0; }
};

template <class L>
struct RegBodies {
    static constexpr int NB = L::NUM_BODIES;
    typename BodyVec<NB>::type x, y, ang, vx, vy, w, im, ii;

    MRL_DEV void load(const float *row) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const float *B = row + L::BODIES_OFF + b * BODY_SIZE;
            x[b] = B[IDX_X]; y[b] = B[IDX_Y]; ang[b] = B[IDX_ANGLE];
            vx[b] = B[IDX_VX]; vy[b] = B[IDX_VY]; w[b] = B[IDX_OMEGA];
            im[b] = B[IDX_INV_MASS]; ii[b] = B[IDX_INV_INERTIA];
        }
    }
    MRL_DEV void store(float *row) const {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float *B = row + L::BODIES_OFF + b * BODY_SIZE;
            B[IDX_X] = x[b]; B[IDX_Y] = y[b]; B[IDX_ANGLE] = ang[b];
            B[IDX_VX] = vx[b]; B[IDX_VY] = vy[b]; B[IDX_OMEGA] = w[b];
        }
    }
};

// a single body behind the register forms below (the forms with one lane per body)
struct OneBody { static constexpr int NUM_BODIES = 1; };

template <class L>
MRL_DEV void reg_integrate_velocities(RegBodies<L> &B, const float *row, float gx, float gy, float dt) {
#pragma unroll
    for (int b = 0; b < L::NUM_BODIES; ++b) {
        if (B.im[b] == 0.0f) continue;
        const float *F = row + L::FORCES_OFF + b * 3;
        B.vx[b] = B.vx[b] + (F[0] * B.im[b] + gx) * dt;
        B.vy[b] = B.vy[b] + (F[1] * B.im[b] + gy) * dt;
        B.w[b] = B.w[b] + F[2] * B.ii[b] * dt;
    }
}

template <class L>
MRL_DEV void reg_integrate_positions(RegBodies<L> &B, float dt) {
    const float pi_val = (float)3.14159265358979323846;
    const float two_pi = (float)(2.0 * 3.14159265358979323846);
#pragma unroll
    for (int b = 0; b < L::NUM_BODIES; ++b) {
        if (B.im[b] == 0.0f) continue;
        float x = B.x[b] + B.vx[b] * dt;
        float y = B.y[b] + B.vy[b] * dt;
        float angle = B.ang[b] + B.w[b] * dt;
        if (angle > 100.0f || angle < -100.0f) {
            angle = 0.0f;
        } else if (angle > pi_val) {
            angle = angle - two_pi;
            if (angle > pi_val) angle = angle - two_pi;
        } else if (angle < -pi_val) {
            angle = angle + two_pi;
            if (angle < -pi_val) angle = angle + two_pi;
        }
        B.x[b] = x; B.y[b] = y; B.ang[b] = angle;
    }
}

// ---------------------------------------------------------------- contacts

// Everything about one contact that stays fixed during the velocity phase.
struct ContactFixed {
    float nx, ny, ra_x, ra_y, inv_mass_a, inv_inertia_a, k, k_t;
    float rk, rk_t;   // 1 / k and 1 / k_t: every sweep divides by the effective masses (div_by)
};

template <class L>
MRL_DEV ContactFixed contact_prepare(const RegBodies<L> &B, int ia, float point_x, float point_y,
                                     float normal_x, float normal_y) {
    ContactFixed f;
    f.nx = normal_x; f.ny = normal_y;
    f.inv_mass_a = sel<L::NUM_BODIES>(B.im, ia); f.inv_inertia_a = sel<L::NUM_BODIES>(B.ii, ia);
    const float inv_mass_b = 0.0f, inv_inertia_b = 0.0f;
    f.ra_x = point_x - sel<L::NUM_BODIES>(B.x, ia); f.ra_y = point_y - sel<L::NUM_BODIES>(B.y, ia);
    const float rb_x = point_x - point_x, rb_y = point_y - point_y;
    const float ra_cross_n = f.ra_x * normal_y - f.ra_y * normal_x;
    const float rb_cross_n = rb_x * normal_y - rb_y * normal_x;
    float k = f.inv_mass_a + inv_mass_b;
    k = k + f.inv_inertia_a * ra_cross_n * ra_cross_n;
    k = k + inv_inertia_b * rb_cross_n * rb_cross_n;
    f.k = k;
    const float tangent_x = -normal_y, tangent_y = normal_x;
    const float ra_cross_t = f.ra_x * tangent_y - f.ra_y * tangent_x;
    const float rb_cross_t = rb_x * tangent_y - rb_y * tangent_x;
    float k_t = f.inv_mass_a + inv_mass_b;
    k_t = k_t + f.inv_inertia_a * ra_cross_t * ra_cross_t;
    k_t = k_t + inv_inertia_b * rb_cross_t * rb_cross_t;
    f.k_t = k_t;
    f.rk = 1.0f / k;
    f.rk_t = 1.0f / k_t;
    return f;
}

// One contact of one velocity sweep; jn / jt are the accumulated impulses.  `live`: the lane has such a contact.  Lanes
// that have none, or whose contact separates, take part and keep what they had (see joint_velocity below).
template <class L>
MRL_DEV void contact_velocity(RegBodies<L> &B, int ia, const ContactFixed &f, float &jn, float &jt,
                              float friction, float restitution, bool live = true) {
    const float normal_x = f.nx, normal_y = f.ny, ra_x = f.ra_x, ra_y = f.ra_y;
    const float inv_mass_a = f.inv_mass_a, inv_inertia_a = f.inv_inertia_a;
    const float vx0 = sel<L::NUM_BODIES>(B.vx, ia), vy0 = sel<L::NUM_BODIES>(B.vy, ia), w0 = sel<L::NUM_BODIES>(B.w, ia);
    float vel_a_x = vx0, vel_a_y = vy0, omega_a = w0;
    const float vel_b_x = 0.0f, vel_b_y = 0.0f, omega_b = 0.0f, rb_x = 0.0f, rb_y = 0.0f;
    float vel_at_a_x = vel_a_x - omega_a * ra_y, vel_at_a_y = vel_a_y + omega_a * ra_x;
    float vel_at_b_x = vel_b_x - omega_b * rb_y, vel_at_b_y = vel_b_y + omega_b * rb_x;
    float rel_vel_x = vel_at_a_x - vel_at_b_x, rel_vel_y = vel_at_a_y - vel_at_b_y;
    const float vel_normal = rel_vel_x * normal_x + rel_vel_y * normal_y;
    const bool push = live && vel_normal < 0.0f;
    if (!any_lane(push)) return;

    float j_normal = div_by(-(1.0f + restitution) * vel_normal, f.k, f.rk);
    const float old_impulse = jn;
    float new_impulse = old_impulse + j_normal;
    new_impulse = new_impulse < 0.0f ? 0.0f : new_impulse;
    jn = push ? new_impulse : jn;
    j_normal = new_impulse - old_impulse;
    const float impulse_x = j_normal * normal_x, impulse_y = j_normal * normal_y;
    vel_a_x = vel_a_x + impulse_x * inv_mass_a;
    vel_a_y = vel_a_y + impulse_y * inv_mass_a;
    omega_a = omega_a + (ra_x * impulse_y - ra_y * impulse_x) * inv_inertia_a;
    vel_at_a_x = vel_a_x - omega_a * ra_y; vel_at_a_y = vel_a_y + omega_a * ra_x;
    vel_at_b_x = vel_b_x - omega_b * rb_y; vel_at_b_y = vel_b_y + omega_b * rb_x;
    rel_vel_x = vel_at_a_x - vel_at_b_x; rel_vel_y = vel_at_a_y - vel_at_b_y;

    const float tangent_x = -normal_y, tangent_y = normal_x;
    const float vel_tangent = rel_vel_x * tangent_x + rel_vel_y * tangent_y;
    float j_tangent = div_by(-vel_tangent, f.k_t, f.rk_t);
    const float max_friction = friction * new_impulse;
    const float old_tangent = jt;
    const float sum_tangent = old_tangent + j_tangent;
    float new_tangent = sum_tangent < -max_friction ? -max_friction : sum_tangent;
    new_tangent = sum_tangent > max_friction ? max_friction : new_tangent;
    jt = push ? new_tangent : jt;
    j_tangent = new_tangent - old_tangent;
    const float friction_x = j_tangent * tangent_x, friction_y = j_tangent * tangent_y;
    vel_a_x = vel_a_x + friction_x * inv_mass_a;
    vel_a_y = vel_a_y + friction_y * inv_mass_a;
    omega_a = omega_a + (ra_x * friction_y - ra_y * friction_x) * inv_inertia_a;
    put<L::NUM_BODIES>(B.vx, ia, push ? vel_a_x : vx0);
    put<L::NUM_BODIES>(B.vy, ia, push ? vel_a_y : vy0);
    put<L::NUM_BODIES>(B.w, ia, push ? omega_a : w0);
}

// The solvers' slop, and sqrtf(s) < slop without the root: the root is rounded correctly and grows with s, so it is below
// the slop exactly for s below the smallest float whose root is not
constexpr float SOLVER_SLOP = 0.005f, SOLVER_SLOP_SQ = 0x1.a36e2cp-16f;

template <class L>
MRL_DEV void contact_position(RegBodies<L> &B, int ia, float normal_x, float normal_y, float depth,
                              float baumgarte) {
    float correction = depth - SOLVER_SLOP;
    if (correction <= 0.0f) return;
    correction = baumgarte * correction;
    const float inv_mass_a = sel<L::NUM_BODIES>(B.im, ia);
    const float inv_mass_b = 0.0f;
    const float total = inv_mass_a + inv_mass_b;
    if (total == 0.0f) return;
    const float correction_a = correction * inv_mass_a / total;
    put<L::NUM_BODIES>(B.x, ia, sel<L::NUM_BODIES>(B.x, ia) + normal_x * correction_a);
    put<L::NUM_BODIES>(B.y, ia, sel<L::NUM_BODIES>(B.y, ia) + normal_y * correction_a);
}

// contact list held in registers (short MAX_CONTACTS)
template <class L>
struct RegContacts {
    static constexpr int MC = L::MAX_CONTACTS;
    int n;
    int body[MC];
    float depth[MC], jn[MC], jt[MC];
    ContactFixed f[MC];

    MRL_DEV void load(const RegBodies<L> &B, float *contacts, int count) {
        n = count;
#pragma unroll
        for (int c = 0; c < MC; ++c) {
            body[c] = 0;
            depth[c] = jn[c] = jt[c] = 0.0f;
            f[c] = ContactFixed{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f, 1.0f, 1.0f, 1.0f};
            if (c < count) {
                const float *C = contacts + c * CONTACT_SIZE;
                body[c] = (int)C[C_BODY_A];
                depth[c] = C[C_DEPTH]; jn[c] = C[C_JN]; jt[c] = C[C_JT];
                f[c] = contact_prepare<L>(B, body[c], C[C_PX], C[C_PY], C[C_NX], C[C_NY]);
            }
        }
    }
    MRL_DEV void velocity_sweep(RegBodies<L> &B, float friction, float restitution) {
#pragma unroll
        for (int c = 0; c < MC; ++c) {
            if (!any_lane(c < n)) break;
            contact_velocity<L>(B, body[c], f[c], jn[c], jt[c], friction, restitution, c < n);
        }
    }
    MRL_DEV void position_sweep(RegBodies<L> &B, float baumgarte) const {
#pragma unroll
        for (int c = 0; c < MC; ++c) {
            if (!any_lane(c < n)) break;
            if (c < n) contact_position<L>(B, body[c], f[c].nx, f[c].ny, depth[c], baumgarte);
        }
    }
};

// Contact list left in the lane's LDS scratch (long lists).  After load() the record's contact
// point slots hold the lever arm (the only way the point enters a sweep) and four slots behind
// the MAX_CONTACTS records hold each contact's effective masses and their reciprocals; body indices, normals, depth
// and accumulated impulses stay where the detector put them.
template <class L>
struct LdsContacts {
    int n;
    float *cts;

    MRL_DEV float &k_slot(int c, int which) { return cts[L::MAX_CONTACTS * CONTACT_SIZE + 4 * c + which]; }

    MRL_DEV void load(const RegBodies<L> &B, float *contacts, int count) {
        n = count;
        cts = contacts;
        for (int c = 0; c < n; ++c) {
            float *C = cts + c * CONTACT_SIZE;
            const ContactFixed f = contact_prepare<L>(B, (int)C[C_BODY_A], C[C_PX], C[C_PY], C[C_NX], C[C_NY]);
            C[C_PX] = f.ra_x; C[C_PY] = f.ra_y;
            k_slot(c, 0) = f.k;
            k_slot(c, 1) = f.k_t;
            k_slot(c, 2) = f.rk;
            k_slot(c, 3) = f.rk_t;
        }
    }
    MRL_DEV void velocity_sweep(RegBodies<L> &B, float friction, float restitution) {
        for (int c = 0; c < n; ++c) {
            float *C = cts + c * CONTACT_SIZE;
            const int ia = (int)C[C_BODY_A];
            ContactFixed f;
            f.nx = C[C_NX]; f.ny = C[C_NY]; f.ra_x = C[C_PX]; f.ra_y = C[C_PY];
            f.inv_mass_a = sel<L::NUM_BODIES>(B.im, ia); f.inv_inertia_a = sel<L::NUM_BODIES>(B.ii, ia);
            f.k = k_slot(c, 0); f.k_t = k_slot(c, 1); f.rk = k_slot(c, 2); f.rk_t = k_slot(c, 3);
            float jn = C[C_JN], jt = C[C_JT];
            contact_velocity<L>(B, ia, f, jn, jt, friction, restitution);
            C[C_JN] = jn; C[C_JT] = jt;
        }
    }
    MRL_DEV void position_sweep(RegBodies<L> &B, float baumgarte) const {
        for (int c = 0; c < n; ++c) {
            const float *C = cts + c * CONTACT_SIZE;
            contact_position<L>(B, (int)C[C_BODY_A], C[C_NX], C[C_NY], C[C_DEPTH], baumgarte);
        }
    }
};

// ---------------------------------------------------------------- joints

// What one joint's velocity sweeps use; nothing of it changes during the velocity phase.
struct JointSweep {
    float rax, ray, rbx, rby, inv_k11, inv_k12, inv_k22;
    float ima, iia, imb, iib;         // the bodies' inverse masses and inertias
    float eff, reff;                  // iia + iib and its reciprocal: spring, limit and motor all divide by it (div_by)
    float spring_term, damp;
    float below, above;               // the limit stops a relative angular velocity < below or > above
    float motor_speed, max_impulse;
    bool spring, motor;
};

// The limit's test as two bounds: at its lower (upper) stop a joint's limit acts on a negative (positive) relative
// angular velocity, anywhere else, or without a limit, on none.
MRL_DEV void joint_limits(JointSweep &q, bool limited, float rel_angle, float lo, float hi) {
    const float inf = __builtin_inff();
    const bool at_lo = limited && rel_angle <= lo, at_hi = limited && !(rel_angle <= lo) && rel_angle >= hi;
    q.below = at_lo ? 0.0f : -inf;
    q.above = at_hi ? 0.0f : inf;
}

// Which terms any lane of the wavefront needs: a term that none does is stepped over by a scalar branch
struct JointTerms {
    bool spring, limit, motor;
    MRL_DEV void add(const JointSweep &q, bool active = true) {
        const bool s = any_lane(active && q.spring), l = any_lane(active && (q.below == 0.0f || q.above == 0.0f));
        const bool m = any_lane(active && q.motor);
        spring = spring | s;
        limit = limit | l;
        motor = motor | m;
    }
};

// One joint of one velocity sweep (joints/revolute.mojo:100-320): (vxa, vya, wa) and (vxb, vyb, wb) are the bodies'
// velocities before and after.
// What bounds it: the instructions of the one wavefront that runs the solver -- it issues one every five to six cycles,
// whether it waits for the one before or not, and a branch on a lane's own flag is a compare, a saved mask and a jump.  So
// there are none: what stays the same over the sweeps is decided ahead, a lane that a term does not concern computes it and
// keeps its value.  (LunarLander rollout of 777 envs, H = 64: 19.8 -> 19.4 us a step with the position sweep
// likewise; HalfCheetah, 4096 envs: 70.2 -> 67.2.)
MRL_DEV void joint_velocity(const JointSweep &q, const JointTerms &any, float dt, float &vxa, float &vya, float &wa,
                            float &vxb, float &vyb, float &wb) {
    const float va_anchor_x = vxa - wa * q.ray, va_anchor_y = vya + wa * q.rax;
    const float vb_anchor_x = vxb - wb * q.rby, vb_anchor_y = vyb + wb * q.rbx;
    const float cdot_x = vb_anchor_x - va_anchor_x, cdot_y = vb_anchor_y - va_anchor_y;
    const float impulse_x = -(q.inv_k11 * cdot_x + q.inv_k12 * cdot_y);
    const float impulse_y = -(q.inv_k12 * cdot_x + q.inv_k22 * cdot_y);
    float cur_wa = wa - q.iia * (q.rax * impulse_y - q.ray * impulse_x);
    float cur_wb = wb + q.iib * (q.rbx * impulse_y - q.rby * impulse_x);
    if (any.spring) {
        const float rel_omega = wb - wa;  // angular velocities from before the point impulse
        const float spring_torque = q.spring_term - q.damp * rel_omega;
        const float angular_impulse = spring_torque * dt;
        const float to_a = cur_wa - div_by(q.iia * angular_impulse, q.eff, q.reff);
        const float to_b = cur_wb + div_by(q.iib * angular_impulse, q.eff, q.reff);
        cur_wa = q.spring ? to_a : cur_wa;
        cur_wb = q.spring ? to_b : cur_wb;
    }
    if (any.limit) {
        const float rel_omega = cur_wb - cur_wa;
        const float stop = div_by(-rel_omega, q.eff, q.reff);
        const bool acts = (rel_omega < q.below || rel_omega > q.above) && stop != 0.0f;
        const float to_a = cur_wa - q.iia * stop, to_b = cur_wb + q.iib * stop;
        cur_wa = acts ? to_a : cur_wa;
        cur_wb = acts ? to_b : cur_wb;
    }
    if (any.motor) {
        const float rel_omega = cur_wb - cur_wa;
        const float speed_error = q.motor_speed - rel_omega;
        float motor_impulse = div_by(speed_error, q.eff, q.reff);
        motor_impulse = motor_impulse > q.max_impulse ? q.max_impulse : motor_impulse;
        motor_impulse = motor_impulse < -q.max_impulse ? -q.max_impulse : motor_impulse;
        const float to_a = cur_wa - q.iia * motor_impulse, to_b = cur_wb + q.iib * motor_impulse;
        cur_wa = q.motor ? to_a : cur_wa;
        cur_wb = q.motor ? to_b : cur_wb;
    }
    vxa = vxa - q.ima * impulse_x;
    vya = vya - q.ima * impulse_y;
    vxb = vxb + q.imb * impulse_x;
    vyb = vyb + q.imb * impulse_y;
    wa = cur_wa;
    wb = cur_wb;
}

// K^-1 of a joint's point constraint from its lever arms
MRL_DEV void joint_inverse(float ima, float iia, float imb, float iib, float rax, float ray, float rbx, float rby,
                           float &inv_k11, float &inv_k12, float &inv_k22) {
    const float k11 = ima + imb + iia * ray * ray + iib * rby * rby;
    const float k12 = -iia * rax * ray - iib * rbx * rby;
    const float k22 = ima + imb + iia * rax * rax + iib * rbx * rbx;
    float det = k11 * k22 - k12 * k12;
    det = det < 1e-10f ? 1e-10f : det;
    const float inv_det = 1.0f / det;
    inv_k11 = k22 * inv_det; inv_k12 = -k12 * inv_det; inv_k22 = k11 * inv_det;
}

// One joint of one position sweep (joints/revolute.mojo:323-495) for bodies at (xa, ya, angle_a) and (xb, yb, angle_b):
// the same places after the correction; false when there is none.  (r_ax, r_ay), (r_bx, r_by): the lever arms; lim: the joint
// has a limit.
MRL_DEV bool joint_position(float ima, float iia, float imb, float iib, float eff, float reff, float r_ax, float r_ay,
                            float r_bx, float r_by, bool lim, float lo, float hi, float ref, float baumgarte, float &xa,
                            float &ya, float &angle_a, float &xb, float &yb, float &angle_b) {
    const float anchor_ax = xa + r_ax, anchor_ay = ya + r_ay;
    const float anchor_bx = xb + r_bx, anchor_by = yb + r_by;
    const float cx = anchor_bx - anchor_ax, cy = anchor_by - anchor_ay;
    if (cx * cx + cy * cy < SOLVER_SLOP_SQ) return false;
    float ik11, ik12, ik22;
    joint_inverse(ima, iia, imb, iib, r_ax, r_ay, r_bx, r_by, ik11, ik12, ik22);
    const float correction_x = -baumgarte * (ik11 * cx + ik12 * cy);
    const float correction_y = -baumgarte * (ik12 * cx + ik22 * cy);
    xa = xa - ima * correction_x;
    ya = ya - ima * correction_y;
    xb = xb + imb * correction_x;
    yb = yb + imb * correction_y;
    float cur_a = angle_a - iia * (r_ax * correction_y - r_ay * correction_x);
    float cur_b = angle_b + iib * (r_bx * correction_y - r_by * correction_x);
    const float relative_angle = cur_b - cur_a - ref;
    const bool low = relative_angle < lo, high = relative_angle > hi;
    if (lim && (low || high)) {
        const float angle_correction = baumgarte * ((low ? lo : hi) - relative_angle);
        if (angle_correction != 0.0f) {
            cur_a = cur_a - div_by(iia * angle_correction, eff, reff);
            cur_b = cur_b + div_by(iib * angle_correction, eff, reff);
        }
    }
    angle_a = cur_a;
    angle_b = cur_b;
    return true;
}

// Joint table of one env.  Only what the velocity sweeps need is held in registers (filled by
// prepare_velocity); the two position sweeps read their few parameters from the row as they go.
template <class L, class T>
struct RegJoints {
    static constexpr int MJ = L::MAX_JOINTS, NB = L::NUM_BODIES;
    bool active[MJ];
    int ba_[MJ], bb_[MJ];
    JointSweep q[MJ];
    JointTerms any;

    MRL_DEV int ba(int j) const { return T::STATIC ? T::a(j) : ba_[j]; }
    MRL_DEV int bb(int j) const { return T::STATIC ? T::b(j) : bb_[j]; }

    static MRL_DEV void anchor(const float *J, float sin_a, float cos_a, float sin_b, float cos_b, float &ax, float &ay,
                               float &bx, float &by) {
        const float lax = J[J_AX], lay = J[J_AY], lbx = J[J_BX], lby = J[J_BY];
        ax = lax * cos_a - lay * sin_a; ay = lax * sin_a + lay * cos_a;
        bx = lbx * cos_b - lby * sin_b; by = lbx * sin_b + lby * cos_b;
    }

    // lever arms, K^-1 and the angle-dependent spring / limit terms for the velocity phase
    MRL_DEV void prepare_velocity(const RegBodies<L> &B, const float *row, float dt) {
        const int n = (int)row[L::JOINT_COUNT_OFF];
        typename BodyVec<NB>::type sn, cs;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float s, c;
            sincos32(B.ang[b], s, c);
            sn[b] = s; cs[b] = c;
        }
        any = JointTerms{false, false, false};
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
            const float *J = row + L::JOINTS_OFF + j * JOINT_SIZE;
            active[j] = (j < n) && ((int)J[J_TYPE] == 0);
            ba_[j] = (int)J[J_BODY_A]; bb_[j] = (int)J[J_BODY_B];
            const int a = ba(j), b = bb(j), flags = (int)J[J_FLAGS];
            JointSweep &k = q[j];
            anchor(J, sel<NB>(sn, a), sel<NB>(cs, a), sel<NB>(sn, b), sel<NB>(cs, b), k.rax, k.ray, k.rbx, k.rby);
            k.ima = sel<NB>(B.im, a); k.iia = sel<NB>(B.ii, a);
            k.imb = sel<NB>(B.im, b); k.iib = sel<NB>(B.ii, b);
            joint_inverse(k.ima, k.iia, k.imb, k.iib, k.rax, k.ray, k.rbx, k.rby, k.inv_k11, k.inv_k12, k.inv_k22);
            k.eff = k.iia + k.iib;
            k.reff = 1.0f / k.eff;
            const float angle_a = sel<NB>(B.ang, a), angle_b = sel<NB>(B.ang, b);
            const float ref = J[J_REF];
            const float angle_error = (angle_b - angle_a) - ref;
            k.spring_term = -J[J_STIFF] * angle_error;
            k.damp = J[J_DAMP];
            const bool turns = k.eff > 1e-10f;
            k.spring = turns && (flags & JF_SPRING) != 0;
            joint_limits(k, turns && (flags & JF_LIMIT) != 0, angle_b - angle_a - ref, J[J_LO], J[J_HI]);
            k.motor = turns && (flags & JF_MOTOR) != 0;
            k.motor_speed = J[J_MOTOR_SPEED];
            k.max_impulse = J[J_MAX_TORQUE] * dt;
            any.add(k, active[j]);
        }
    }

    MRL_DEV void velocity_sweep(RegBodies<L> &B, float dt) const {
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
            if (!active[j]) continue;
            const int a = ba(j), b = bb(j);
            float vxa = sel<NB>(B.vx, a), vya = sel<NB>(B.vy, a), wa = sel<NB>(B.w, a);
            float vxb = sel<NB>(B.vx, b), vyb = sel<NB>(B.vy, b), wb = sel<NB>(B.w, b);
            joint_velocity(q[j], any, dt, vxa, vya, wa, vxb, vyb, wb);
            put<NB>(B.vx, a, vxa); put<NB>(B.vy, a, vya);
            put<NB>(B.vx, b, vxb); put<NB>(B.vy, b, vyb);
            put<NB>(B.w, a, wa); put<NB>(B.w, b, wb);
        }
    }

    MRL_DEV void position_sweep(RegBodies<L> &B, const float *row, float baumgarte) const {
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
            if (!active[j]) continue;
            const float *J = row + L::JOINTS_OFF + j * JOINT_SIZE;
            const int a = ba(j), b = bb(j);
            float xa = sel<NB>(B.x, a), ya = sel<NB>(B.y, a), angle_a = sel<NB>(B.ang, a);
            float xb = sel<NB>(B.x, b), yb = sel<NB>(B.y, b), angle_b = sel<NB>(B.ang, b);
            float sin_a, cos_a, sin_b, cos_b, r_ax, r_ay, r_bx, r_by;
            sincos32(angle_a, sin_a, cos_a);
            sincos32(angle_b, sin_b, cos_b);
            anchor(J, sin_a, cos_a, sin_b, cos_b, r_ax, r_ay, r_bx, r_by);
            joint_position(q[j].ima, q[j].iia, q[j].imb, q[j].iib, q[j].eff, q[j].reff, r_ax, r_ay, r_bx, r_by,
                           ((int)J[J_FLAGS] & JF_LIMIT) != 0 && q[j].eff > 1e-10f, J[J_LO], J[J_HI], J[J_REF], baumgarte,
                           xa, ya, angle_a, xb, yb, angle_b);
            put<NB>(B.x, a, xa); put<NB>(B.y, a, ya);
            put<NB>(B.x, b, xb); put<NB>(B.y, b, yb);
            put<NB>(B.ang, a, angle_a); put<NB>(B.ang, b, angle_b);
        }
    }
};

// true when every joint of the row connects the bodies that the static topology T names
template <class L, class T>
MRL_DEV bool topology_matches(const float *row) {
    bool ok = true;
    const int n = (int)row[L::JOINT_COUNT_OFF];
#pragma unroll
    for (int j = 0; j < L::MAX_JOINTS; ++j) {
        if (j >= n) break;
        const float *J = row + L::JOINTS_OFF + j * JOINT_SIZE;
        ok = ok && (int)J[J_BODY_A] == T::a(j) && (int)J[J_BODY_B] == T::b(j);
    }
    return ok;
}

template <class L, class T, bool FLAT, bool REG_CONTACTS>
MRL_DEV int reg_physics_substep_impl(float *row, const float *shapes, float *contacts, float gx, float gy,
                                     float dt, float friction, float restitution, float baumgarte,
                                     int vel_iters, int pos_iters, int n_given) {
    RegBodies<L> B;
    B.load(row);
    reg_integrate_velocities<L>(B, row, gx, gy, dt);
    // the detectors read positions and angles only, which the velocity update has not touched
    const int n = n_given >= 0 ? n_given
                  : (FLAT ? flat_detect<L>(row, shapes, 0.0f, contacts) : edge_detect<L>(row, shapes, contacts));
    typename std::conditional<REG_CONTACTS, RegContacts<L>, LdsContacts<L>>::type C;
    C.load(B, contacts, n);
    RegJoints<L, T> J;
    J.prepare_velocity(B, row, dt);
    for (int it = 0; it < vel_iters; ++it) {
        C.velocity_sweep(B, friction, restitution);
        J.velocity_sweep(B, dt);
    }
    reg_integrate_positions<L>(B, dt);
    for (int it = 0; it < pos_iters; ++it) {
        C.position_sweep(B, baumgarte);
        J.position_sweep(B, row, baumgarte);
    }
    B.store(row);
#pragma unroll
    for (int k = 0; k < L::NUM_BODIES * 3; ++k) row[L::FORCES_OFF + k] = 0.0f;
    return n;
}

// One physics step (or sub-step) of an env row with the sweeps on registers.  `row` must hold the
// current bodies / joints; contacts are detected into the lane's LDS scratch, which holds
// MAX_CONTACTS * CONTACT_SCRATCH floats (detection order and the MAX_CONTACTS cut-off unchanged;
// afterwards the body indices of the contacts are still readable at
// contacts[c * CONTACT_SIZE + C_BODY_A / C_BODY_B], the contact-point slots are not), then
// everything iterative runs on registers.  n_given >= 0: `contacts` already holds that many
// contacts detected from the row's current positions (detection is skipped).
template <class L, class T, bool FLAT, bool REG_CONTACTS>
MRL_DEV int reg_physics_substep(float *row, const float *shapes, float *contacts, float gx, float gy,
                                float dt, float friction, float restitution, float baumgarte,
                                int vel_iters, int pos_iters, int n_given = -1) {
    if (T::STATIC && __all(topology_matches<L, T>(row) ? 1 : 0))
        return reg_physics_substep_impl<L, T, FLAT, REG_CONTACTS>(row, shapes, contacts, gx, gy, dt, friction,
                                                                  restitution, baumgarte, vel_iters,
                                                                  pos_iters, n_given);
    return reg_physics_substep_impl<L, DynamicTopology, FLAT, REG_CONTACTS>(
        row, shapes, contacts, gx, gy, dt, friction, restitution, baumgarte, vel_iters, pos_iters,
        n_given);
}

}  // namespace mrl
