// Rosenbrock-W step (ROS3P, RODAS3P, Rosenbrock 2(3)).
//
// Follows the reference's GenericRosenbrockWStep.step (integrators/
// algorithms/generic_rosenbrock_w.py:470-740): the Jacobian is taken once at
// the step start (y_n, drivers at t_n), the time derivative
// dt * (df/dt + df/dd * dd/dt) is formed at t_n, and each stage solves
//   (I - gamma h J) K_i = gamma h (f(Y_i) + sum_j C_ij K_j / h + gamma_i dt f_t)
// with Y_i = y_n + sum_j a_ij K_j, by the matrix-free linear solver (no
// Newton iteration). The Krylov norm is referenced to y_n. Stage 0 starts
// from the previous step's last K (kept across steps); stage i starts from
// K_{i-1}. The operator is the cached form of codegen/linear_operators.py:
// 256-335 with a_ij = 1 and beta = 1; the Neumann series uses h_eff = h gamma
// and the Jacobi preconditioner the diagonal of I - gamma h J. Small systems
// keep the dense Jacobian in registers; larger ones re-evaluate J v at the
// step-start state. The linear solves run in Cfg::lin_real (FP32 in the
// mixed-precision mode, with right-hand sides and stage sums in FP64). Like
// the reference, the step reports no Newton / Krylov counts to the loop.
#pragma once

namespace cubie {

template <typename Cfg, typename Sys>
struct RosenbrockProblem {
    using L = typename Cfg::lin_real;
    static constexpr int n = Cfg::n;
    static constexpr int W = n;
    static constexpr bool cache_jac = Cfg::cache_jac;
    // matrix-free systems: the sparse Jacobian's nonzeros at (t_n, y_n),
    // evaluated once per step (the reference's cached auxiliaries)
    static constexpr bool sparse = Cfg::cache_sparse_jac && !cache_jac;
    const L* state;     // y_n, in the linear-solve precision
    const L* params;
    const L* drivers;
    const L* J;         // dense row-major Jacobian when cache_jac, else the
                        // sparse nonzeros when sparse
    const L* Jd;        // Jacobian diagonal
    const L* kw;        // 1 / Krylov tolerance weights (fixed per step)
    real t, h;

    __device__ __forceinline__ void prepare_linear() {}   // J is taken once per step
    __device__ __forceinline__ void jv(const L* v, L* out) const {
        if constexpr (cache_jac) {
            dense_jv<Sys, n>(J, v, out);
        } else if constexpr (sparse) {
            sparse_jv<Sys, n>(J, v, out);
        } else {
            Sys::jvp(state, params, drivers, v, out, L(t));
        }
    }
    __device__ __forceinline__ void op(const L* v, L* out) const {
        L tmp[n];
        jv(v, tmp);
        const L gh = L(Cfg::gamma * h);
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) out[i] = v[i] - gh * tmp[i];
    }
    __device__ __forceinline__ void neumann(const L* v, L* out) const {
        const L h_eff = L(h * Cfg::gamma);
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) out[i] = v[i];
        for (int k = 0; k < Cfg::preconditioner_order; ++k) {
            L tmp[n];
            jv(out, tmp);
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) out[i] = v[i] + h_eff * tmp[i];
        }
    }
    __device__ __forceinline__ void jacobi(const L* v, L* out) const {
        const L scale = L(Cfg::gamma * h);
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) out[i] = jacobi_divide(v[i], scale, Jd[i]);
    }
    __device__ __forceinline__ L krylov_norm2(const L* vals) const {
        L nrm2 = L(0);
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) {
            const L r = dabs(vals[i]) * kw[i];
            nrm2 += r * r;
        }
        return nrm2 * L(Cfg::inv_n);
    }
};

template <typename Cfg, typename Sys>
struct RosenbrockStep {
    static constexpr int n = Cfg::n;
    static constexpr int s = Cfg::stages;
    static constexpr int nd = Cfg::n_drivers;
    using Prob = RosenbrockProblem<Cfg, Sys>;
    Vec<real, n> stage_increment;   // last stage's K, the next step's first guess

    __device__ __forceinline__ void init() {
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) stage_increment[i] = real(0);
    }

    // (I - gamma h J) x = rhs from the guess in x, in the linear-solve precision.
    __device__ __forceinline__ int solve(Prob& P, real* rhs, real* x, int& it) {
        using L = typename Cfg::lin_real;
        if constexpr (same_type<L, real>::value) {
            return linear_solve<Cfg, L>(P, rhs, x, false, it);
        } else {
            L rl[n], xl[n];
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) { rl[i] = L(rhs[i]); xl[i] = L(x[i]); }
            const int st = linear_solve<Cfg, L>(P, rl, xl, false, it);
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) x[i] = real(xl[i]);
            return st;
        }
    }

    template <typename Ctx>
    __device__ __forceinline__ int step(Ctx& ctx, const Vec<real, n>& state, Vec<real, n>& proposed,
                                        Vec<real, Cfg::n_error>& error, real dt, real time,
                                        double /*t64*/, bool /*first_step*/, bool /*prev_accepted*/,
                                        int* counters) {
        const real current_time = time;
        const real end_time = current_time + dt;
        const real inv_dt = sdiv<Cfg>(real(1), dt);
        const real* params = ctx.params.data();

        // Jacobian at the step start, in the linear-solve precision
        using L = typename Cfg::lin_real;
        LinInputs<Cfg> li;
        li.bind(params, ctx.drivers.data());
        Vec<L, n> state_l;
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) state_l[i] = L(state[i]);
        const L t_l = L(current_time);
        Vec<L, (Prob::cache_jac ? n * n : (Prob::sparse ? Sys::jac_nnz : 1))> J;
        Vec<L, n> Jd;
        if constexpr (Prob::cache_jac) {
            Sys::jac(state_l.data(), li.params, li.drivers, J.data(), t_l);
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) Jd[i] = J[i * n + i];
        } else {
            if constexpr (Prob::sparse)
                Sys::jac_sparse(state_l.data(), li.params, li.drivers, J.data(), t_l);
            Sys::jac_diag(state_l.data(), li.params, li.drivers, Jd.data(), t_l);
        }

        // dt * total time derivative at (t_n, y_n)
        Vec<real, n> dfdt;
        {
            Vec<real, (nd > 0 ? nd : 1)> ddt;
CUBIE_UNROLL
            for (int q = 0; q < (nd > 0 ? nd : 1); ++q) ddt[q] = real(0);
            if constexpr (nd > 0) ctx.drv.eval_dt(current_time, ddt.data());
            Sys::dfdt(state.data(), params, ctx.drivers.data(), ddt.data(), dfdt.data(), current_time);
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) dfdt[i] *= dt;
        }
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) {
            proposed[i] = state[i];
            if constexpr (Cfg::has_error) error[i] = real(0);
        }

        Vec<L, n> kw;
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) {
            const L tol = L(Cfg::krylov_atol[i]) + L(Cfg::krylov_rtol[i]) * dabs(state_l[i]);
            kw[i] = sdiv<Cfg>(L(1), pmax(tol, L(1e-16)));
        }
        Prob P;
        P.kw = kw.data();
        P.state = state_l.data();
        P.params = li.params;
        P.drivers = li.drivers;
        P.J = J.data();
        P.Jd = Jd.data();
        P.t = current_time;
        P.h = dt;

        int status = ST_SUCCESS;
        Vec<real, s * n> store;
        real rhs[n];
        real obs_scratch[Cfg::n_obs > 0 ? Cfg::n_obs : 1];

        // stage 0 at the step start
        Sys::dxdt(state.data(), params, ctx.drivers.data(), obs_scratch, rhs, current_time);
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) {
            const real v = (rhs[i] + Cfg::gamma_stages[0] * dfdt[i]) * dt;
            rhs[i] = v * Cfg::gamma;
        }
        int it = 0;
        status |= solve(P, rhs, stage_increment.data(), it);
        counters[3] += it;
CUBIE_UNROLL
        for (int i = 0; i < n; ++i) {
            store[i] = stage_increment[i];
            if constexpr (Cfg::accumulates_output) proposed[i] += stage_increment[i] * Cfg::b[0];
            if constexpr (Cfg::has_error && Cfg::accumulates_error) error[i] += stage_increment[i] * Cfg::d[0];
        }

CUBIE_UNROLL
        for (int si = 1; si < s; ++si) {
            const real stage_time = current_time + dt * Cfg::c[si];
            real Y[n];
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) {
                real v = state[i];
CUBIE_UNROLL
                for (int j = 0; j < s - 1; ++j)
                    if (j < si) v += Cfg::A[si][j] * store[j * n + i];
                Y[i] = v;
            }
            if constexpr (nd > 0) ctx.drv.eval(stage_time, ctx.proposed_drivers.data());
            if constexpr (Cfg::n_obs > 0)
                Sys::observables(Y, params, ctx.proposed_drivers.data(), ctx.proposed_observables.data(),
                                 stage_time);
            Sys::dxdt(Y, params, ctx.proposed_drivers.data(), obs_scratch, rhs, stage_time);
            if (Cfg::b_row == si) {
CUBIE_UNROLL
                for (int i = 0; i < n; ++i) proposed[i] = Y[i];
            }
            if constexpr (Cfg::has_error) {
                if (Cfg::b_hat_row == si) {
CUBIE_UNROLL
                    for (int i = 0; i < n; ++i) error[i] = Y[i];
                }
            }
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) {
                real corr = real(0);
CUBIE_UNROLL
                for (int j = 0; j < s - 1; ++j)
                    if (j < si) corr += Cfg::rbC[si][j] * store[j * n + i];
                const real v = rhs[i] + corr * inv_dt + Cfg::gamma_stages[si] * dfdt[i];
                rhs[i] = v * dt * Cfg::gamma;
            }
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) stage_increment[i] = store[(si - 1) * n + i];
            status |= solve(P, rhs, stage_increment.data(), it);
            counters[3] += it;
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) {
                store[si * n + i] = stage_increment[i];
                if constexpr (Cfg::accumulates_output) proposed[i] += Cfg::b[si] * stage_increment[i];
                if constexpr (Cfg::has_error && Cfg::accumulates_error)
                    error[i] += Cfg::d[si] * stage_increment[i];
            }
        }
        if constexpr (Cfg::has_error && !Cfg::accumulates_error) {
CUBIE_UNROLL
            for (int i = 0; i < n; ++i) error[i] = proposed[i] - error[i];
        }
        if constexpr (nd > 0) ctx.drv.eval(end_time, ctx.proposed_drivers.data());
        if constexpr (Cfg::n_obs > 0)
            Sys::observables(proposed.data(), params, ctx.proposed_drivers.data(),
                             ctx.proposed_observables.data(), end_time);
        return status;
    }
};

}  // namespace cubie
