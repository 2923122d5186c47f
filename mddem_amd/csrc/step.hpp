// The integrators' arguments and per-particle arithmetic, shared by the
// integration kernels and by the force kernels that go on to the next step's
// first half (integrate.hip, forces.hip).
#pragma once

#include "ctx.hpp"

namespace mdd {

struct IntArgs {
    int64_t n, npad;
    double dt;
    double4* pos;
    double4* vel;
    double4* omega;
    double4* quat;
    const double* mass;
    const double4* build_pos;
    const double* f64;
    const float* f32;
    const double* t64;
    const float* t32;
    int rot;         // apply rotation half-steps
    int vv;          // apply Verlet translational half-steps
    int check;       // evaluate the rebuild decision
    int paired;      // StepArgs: the first half of the step before was such a pass too, and
                     // nothing has written an orientation since, so spheres that it did not
                     // turn have the same one in both buffers
    double thr2;     // ((skin_fraction - 1) * min_skin)^2
    BoxP box;
    int box_exit;
    Status* st;
    int step;
    double* partial;
    int nparts;      // KE partials left by the last post kernel
    int q_in, q_out; // thermostat slots read / written
    double ndof, temp, q_mass;
    const SysP* sysp;       // batched ensemble: per-system box and threshold, or null
    const uint32_t* psys;
    const WallsP* walls;    // walls (device copy) and their state, or null: scheduled
    WallsDyn* wdyn;         // steps move them (PreInitialIntegration) and clear the sums
    int4* xq;               // fixed-point copy of the positions to keep current, or null
    double qs[3];           // its scale 2^32 / L per axis
    const int4* bxq;        // with xq on a periodic box: fixed-point build positions, or null
    double qu[3];           // L / 2^32 per axis
    double thr_band;        // |d2 - thr2| up to this: the double4 build position decides
};

__device__ inline int4 quantize_pos(const IntArgs& a, const double4& p) {
    return make_int4(quantize_axis(p.x, a.qs[0]), quantize_axis(p.y, a.qs[1]),
                     quantize_axis(p.z, a.qs[2]), 0);
}

__device__ inline void store_xq(const IntArgs& a, int64_t i, const double4& p) {
    a.xq[i] = quantize_pos(a, p);
}

template <typename F>
__device__ inline void load_f(const IntArgs& a, int64_t i, double& fx, double& fy, double& fz) {
    if constexpr (sizeof(F) == 8) {
        fx = a.f64[i];
        fy = a.f64[a.npad + i];
        fz = a.f64[2 * a.npad + i];
    } else {
        fx = double(a.f32[i]);
        fy = double(a.f32[a.npad + i]);
        fz = double(a.f32[2 * a.npad + i]);
    }
}

template <typename F>
__device__ inline void load_t(const IntArgs& a, int64_t i, double& tx, double& ty, double& tz) {
    if constexpr (sizeof(F) == 8) {
        tx = a.t64[i];
        ty = a.t64[a.npad + i];
        tz = a.t64[2 * a.npad + i];
    } else {
        tx = double(a.t32[i]);
        ty = double(a.t32[a.npad + i]);
        tz = double(a.t32[2 * a.npad + i]);
    }
}

// displacement_exceeded (neighbor.rs:564-601) + periodic box exit (651-666)
// for position p and the position b at the last build
__device__ inline void rebuild_check(const IntArgs& a, int64_t i, const double4& p,
                                     const double4& b) {
    const BoxP* box = &a.box;
    double thr2 = a.thr2;
    if (a.sysp) {
        const SysP& S = a.sysp[a.psys[i]];
        box = &S.box;
        thr2 = S.thr2;
    }
    double d[3] = {p.x - b.x, p.y - b.y, p.z - b.z};
    const double x[3] = {p.x, p.y, p.z};
    bool out = false;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (box->periodic[k]) {
            const double L = box->L[k], h = L * 0.5;
            if (d[k] > h)
                d[k] -= L;
            else if (d[k] < -h)
                d[k] += L;
            if (a.box_exit && (x[k] < box->lo[k] || x[k] >= box->hi[k])) out = true;
        }
    }
    if (d[0] * d[0] + d[1] * d[1] + d[2] * d[2] > thr2 || out)
        atomicMin(&a.st->abort_step, a.step);
}

// rebuild_check from the fixed-point position and build position (every
// axis periodic). The int32 differences are the minimum image, and each
// coordinate is within one quantum of its double value, so d2 is within
// thr_band of rebuild_check's d2 near the threshold; outside the band both
// decide alike, inside it rebuild_check decides from the double4.
__device__ inline void rebuild_check_fixed(const IntArgs& a, int64_t i, const double4& p,
                                           const int4& bq) {
    const int4 q = quantize_pos(a, p);
    const double dx = double(int(uint32_t(q.x) - uint32_t(bq.x))) * a.qu[0];
    const double dy = double(int(uint32_t(q.y) - uint32_t(bq.y))) * a.qu[1];
    const double dz = double(int(uint32_t(q.z) - uint32_t(bq.z))) * a.qu[2];
    const double d2 = dx * dx + dy * dy + dz * dz;
    if (fabs(d2 - a.thr2) <= a.thr_band) {
        rebuild_check(a, i, p, a.build_pos[i]);
        return;
    }
    bool out = false;
    if (a.box_exit) {
        const double x[3] = {p.x, p.y, p.z};
#pragma unroll
        for (int k = 0; k < 3; k++)
            if (x[k] < a.box.lo[k] || x[k] >= a.box.hi[k]) out = true;
    }
    if (d2 > a.thr2 || out) atomicMin(&a.st->abort_step, a.step);
}

// orientation update of initial_rotation with the kicked omega w
// (rotational.rs:70-83) into quat[i]; `keep`: the orientation goes there also
// where the spin is too slow to turn it
__device__ inline void rotate_quat(const IntArgs& a, int64_t i, const double4& w, double4* quat,
                                   bool keep) {
    const double dt = a.dt;
    const double omega_mag = sqrt(w.x * w.x + w.y * w.y + w.z * w.z);
    const double angle = omega_mag * dt;
    const bool turns = angle > 1e-14;
    if (!turns && !keep) return;
    const double4 b = a.quat[i];
    double4 q = b;
    if (turns) {
        const double inv = 1.0 / omega_mag;
        const double ax = w.x * inv, ay = w.y * inv, az = w.z * inv;
        const double half = angle * 0.5;
        const double s = sin(half);
        const double a0 = cos(half), a1 = ax * s, a2 = ay * s, a3 = az * s;
        q.x = a0 * b.x - a1 * b.y - a2 * b.z - a3 * b.w;
        q.y = a0 * b.y + a1 * b.x + a2 * b.w - a3 * b.z;
        q.z = a0 * b.z - a1 * b.w + a2 * b.x + a3 * b.y;
        q.w = a0 * b.w + a1 * b.z - a2 * b.y + a3 * b.x;
    }
    quat[i] = q;
}

__device__ inline void kick_drift(const IntArgs& a, double4& v, double4& p, double fx, double fy,
                                  double fz) {
    const double dt = a.dt;
    const double h = 0.5 * dt * v.w;
    v.x += h * fx;
    v.y += h * fy;
    v.z += h * fz;
    p.x += v.x * dt;
    p.y += v.y * dt;
    p.z += v.z * dt;
}

// Where a force pass that integrates writes the new state: buffers other
// than the ones it reads (neighbors' positions, velocities and spins are
// read while others already advance, and a pass that the overlap limit stops
// midway leaves the old state whole), exchanged by the host after the launch.
// (the orientations' own buffer: 0.1 us of 12.5 at 200,000 gas spheres, 0.3 of
// 19.1 on a bed of 62,500, against turning them in place)
// wdyn is the coming step's wall state.
struct StepArgs {
    IntArgs in;  // of the coming step
    double4 *pos, *vel, *omega, *quat;
    WallsDyn* wdyn;
};
struct NoStep {};

// Once per launch (one thread): what the coming step's first-half kernel does
// for the whole system. Its overlap count and wall state are other words than
// this step's, which the other blocks are still using. Only for walls at
// rest: moving ones may need this step's complete force sums.
__device__ inline void step_begin(const StepArgs& s, const WallsDyn* now) {
    s.in.st->overlap_count[s.in.step & 1] = 0;
    if (!s.in.walls) return;
    for (int k = 0; k < s.in.walls->count; k++) {
        for (int q = 0; q < 3; q++) {
            s.wdyn->w[k].p[q] = now->w[k].p[q];
            s.wdyn->w[k].v[q] = now->w[k].v[q];
        }
        s.wdyn->w[k].acc = 0ull;
    }
    s.wdyn->time = now->time + s.in.dt;
}

// One particle's inputs to step_advance besides its position and force,
// loaded before its row is walked so that their latency is not added to it.
struct StepIn {
    double4 v, w, b;
    int4 bq;
    bool stale;  // the other buffer may hold another orientation than this one
};

__device__ inline StepIn step_load(const StepArgs& s, int64_t i) {
    const IntArgs& a = s.in;
    StepIn x;
    x.v = a.vel[i];
    x.w = s.omega ? a.omega[i] : make_double4(0.0, 0.0, 0.0, 0.0);
    // (w is the spin that the last first half turned the orientation with)
    x.stale = !a.paired || x.w.x != 0.0 || x.w.y != 0.0 || x.w.z != 0.0;
    x.b = make_double4(0.0, 0.0, 0.0, 0.0);
    x.bq = make_int4(0, 0, 0, 0);
    if (a.check) {
        if (a.bxq)
            x.bq = a.bxq[i];
        else
            x.b = a.build_pos[i];
    }
    return x;
}

// The final half of this step and the first half of the coming one for one
// particle with force f and torque t: k_post_pre's arithmetic.
__device__ inline void step_advance(const StepArgs& s, int64_t i, double4 p, const StepIn& x,
                                    double fx, double fy, double fz, double tx, double ty,
                                    double tz) {
    const IntArgs& a = s.in;
    double4 v = x.v;
    const double h = 0.5 * a.dt * v.w;
    v.x += h * fx;
    v.y += h * fy;
    v.z += h * fz;
    kick_drift(a, v, p, fx, fy, fz);
    s.vel[i] = v;
    s.pos[i] = p;
    if (a.xq) store_xq(a, i, p);
    if (s.omega) {
        double4 w = x.w;
        const double ii = w.w;
        if (a.rot && ii != 0.0) {
            const double dt = a.dt;
            if (tx != 0.0 || ty != 0.0 || tz != 0.0) {
                w.x += 0.5 * dt * tx * ii;  // final_rotation of this step
                w.y += 0.5 * dt * ty * ii;
                w.z += 0.5 * dt * tz * ii;
                w.x += 0.5 * dt * tx * ii;  // initial_rotation of the coming one
                w.y += 0.5 * dt * ty * ii;
                w.z += 0.5 * dt * tz * ii;
            }
            rotate_quat(a, i, w, s.quat, x.stale);
        } else if (x.stale) {
            s.quat[i] = a.quat[i];
        }
        s.omega[i] = w;
    }
    if (a.check) {
        if (a.bxq)
            rebuild_check_fixed(a, i, p, x.bq);
        else
            rebuild_check(a, i, p, x.b);
    }
}

// integrate.hip: the arguments of a step's integration kernels, and of a
// force pass of step `step` that integrates (the new state goes to the
// third buffers; swap_step_buffers exchanges them after the launch, or back
// for a pass that the device did not run)
IntArgs integrate_args(Ctx& c, int step, bool check);
StepArgs step_args(Ctx& c, int step, bool paired);

}  // namespace mdd
