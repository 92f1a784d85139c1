// Fully implicit Runge-Kutta step (Gauss-Legendre, Radau IIA).
//
// Follows the reference's FIRKStep.step (integrators/algorithms/
// generic_firk.py:527-704): all s stages form one Newton problem of width
// s*n whose unknown holds the stage increments z_i, with stage states
// Y_i = y_n + sum_j a_ij z_j at times t + h c_i and one driver vector per
// stage. The coupled residual, operator and Neumann / Jacobi
// preconditioners are the n-stage forms of codegen/nonlinear_residuals.py:
// 193-362, linear_operators.py:599-755 and preconditioners.py:344-399,
// 927-1036; the Krylov norm tiles the step-start state over the stages
// (norms.py:275-324) and the Newton norm measures each stage against its
// own stage state (norms.py:377-432). The solution and error are the
// compensated (Kahan) sums y_n + sum b_i z_i and sum d_i z_i, or copies of a
// stage state when b / b_hat equals a row of A. The increments persist
// between steps as the next Newton starting guess, read ahead by the dense
// predictor when enabled. Tolerance vectors are indexed by state (entry e of
// the coupled vector uses state e mod n).
#pragma once

namespace cubie {

template <typename Cfg, typename Sys>
struct FirkProblem {
    using L = typename Cfg::lin_real;
    static constexpr int n = Cfg::n;
    static constexpr int s = Cfg::stages;
    static constexpr int W = s * n;
    static constexpr int nd = Cfg::n_drivers;
    real* u;                 // coupled increments, stage-major
    const real* base;        // y_n
    const real* params;
    const real* drivers;     // s stacked driver vectors
    const L* params_l;       // the same two, in the linear-solve precision
    const L* drivers_l;
    real t, h;

    __device__ __forceinline__ real stage_time(int i) const { return t + h * Cfg::c[i]; }

    // out = (with_base ? y_n : 0) + sum_j a_ij vec_j, skipping zero couplings.
    template <bool with_base, typename T, typename V>
    __device__ __forceinline__ void combine(int i, const V* vec, T* out) const {
CUBIE_UNROLL
        for (int k = 0; k < n; ++k) {
            T acc = with_base ? T(base[k]) : T(0);
CUBIE_UNROLL
            for (int j = 0; j < s; ++j)
                if (Cfg::A[i][j] != 0.0) acc += T(Cfg::A[i][j]) * T(vec[j * n + k]);
            out[k] = acc;
        }
    }
    // Stage state in the linear-solve precision (rounded once from `real`).
    __device__ __forceinline__ void stage_state_l(int i, L* Y) const {
        real Yr[n];
        combine<true>(i, u, Yr);
CUBIE_UNROLL
        for (int k = 0; k < n; ++k) Y[k] = L(Yr[k]);
    }

    static constexpr bool cache = Cfg::cache_jac;
    static constexpr bool direct_capable = false;   // FP64 Krylov in the mixed mode
    Vec<L, (cache ? s * n * n : 1)> J;   // J(Y_i) per stage, refreshed per linear solve
    // matrix-free systems: the sparse Jacobians' nonzeros at the stage states
    static constexpr bool sparse = Cfg::cache_sparse_jac && !cache;
    Vec<L, (sparse ? s * Sys::jac_nnz : 1)> Js;
    Vec<L, n> kw;                        // 1 / Krylov tolerance weights (per state)

    // Residual, then the per-stage Jacobians at the same iterate (fixed
    // during the Krylov solve that follows).
    __device__ __forceinline__ void residual_prepare(real* out) {
        residual(out);
        prepare_linear();
    }
    __device__ __forceinline__ void prepare_linear() {
        if constexpr (cache) {
CUBIE_UNROLL
            for (int i = 0; i < s; ++i) {
                L Y[n];
                stage_state_l(i, Y);
                Sys::jac(Y, params_l, drivers_l + i * nd, J.data() + i * n * n, L(stage_time(i)));
            }
        } else if constexpr (sparse) {
CUBIE_UNROLL
            for (int i = 0; i < s; ++i) {
                L Y[n];
                stage_state_l(i, Y);
                Sys::jac_sparse(Y, params_l, drivers_l + i * nd, Js.data() + i * Sys::jac_nnz,
                                L(stage_time(i)));
            }
        }
CUBIE_UNROLL
        for (int k = 0; k < n; ++k) {
            L tol = L(Cfg::krylov_atol[k]) + L(Cfg::krylov_rtol[k]) * dabs(L(base[k]));
            kw[k] = sdiv<Cfg>(L(1), pmax(tol, L(1e-16)));
        }
    }
    // J(Y_i) dir for stage i
    __device__ __forceinline__ void stage_jv(int i, const L* dir, L* out) const {
        if constexpr (cache) {
            dense_jv<Sys, n>(J.data() + i * n * n, dir, out);
        } else if constexpr (sparse) {
            sparse_jv<Sys, n>(Js.data() + i * Sys::jac_nnz, dir, out);
        } else {
            L Y[n];
            stage_state_l(i, Y);
            Sys::jvp(Y, params_l, drivers_l + i * nd, dir, out, L(stage_time(i)));
        }
    }

    __device__ __forceinline__ void op(const L* v, L* out) const {
CUBIE_UNROLL
        for (int i = 0; i < s; ++i) {
            L dir[n], jv[n];
            combine<false>(i, v, dir);
            stage_jv(i, dir, jv);
            const L hl = L(h);
CUBIE_UNROLL
            for (int k = 0; k < n; ++k) out[i * n + k] = v[i * n + k] - hl * jv[k];
        }
    }
    __device__ __forceinline__ void neumann(const L* v, L* out) const {
        const L hl = L(h);
CUBIE_UNROLL
        for (int e = 0; e < W; ++e) out[e] = v[e];
        for (int it = 0; it < Cfg::preconditioner_order; ++it) {
            L jvp[W];
CUBIE_UNROLL
            for (int i = 0; i < s; ++i) {
                L dir[n];
                combine<false>(i, out, dir);
                stage_jv(i, dir, jvp + i * n);
            }
CUBIE_UNROLL
            for (int e = 0; e < W; ++e) out[e] = v[e] + hl * jvp[e];
        }
    }
    __device__ __forceinline__ void jacobi(const L* v, L* out) const {
CUBIE_UNROLL
        for (int i = 0; i < s; ++i) {
            L jd[n];
            if constexpr (cache) {
CUBIE_UNROLL
                for (int k = 0; k < n; ++k) jd[k] = J[i * n * n + k * n + k];
            } else {
                L Y[n];
                stage_state_l(i, Y);
                Sys::jac_diag(Y, params_l, drivers_l + i * nd, jd, L(stage_time(i)));
            }
            const L scale = L(h * Cfg::A[i][i]);
CUBIE_UNROLL
            for (int k = 0; k < n; ++k) out[i * n + k] = jacobi_divide(v[i * n + k], scale, jd[k]);
        }
    }
    __device__ __forceinline__ void residual(real* out) const {
CUBIE_UNROLL
        for (int i = 0; i < s; ++i) {
            real Y[n], f[n], obs[Cfg::n_obs > 0 ? Cfg::n_obs : 1];
            combine<true>(i, u, Y);
            Sys::dxdt(Y, params, drivers + i * nd, obs, f, stage_time(i));
CUBIE_UNROLL
            for (int k = 0; k < n; ++k) out[i * n + k] = u[i * n + k] - h * f[k];
        }
    }
    __device__ __forceinline__ L krylov_norm2(const L* vals) const {
        L nrm2 = L(0);
CUBIE_UNROLL
        for (int e = 0; e < W; ++e) {
            const L r = dabs(vals[e]) * kw[e % n];
            nrm2 += r * r;
        }
        return nrm2 * L(1.0 / double(W));
    }
    __device__ __forceinline__ real correction_norm2(const real* vals) const {
        real nrm2 = real(0);
CUBIE_UNROLL
        for (int e = 0; e < W; ++e) {
            const int i = e / n, k = e % n;
            real sv = base[k];
CUBIE_UNROLL
            for (int j = 0; j < s; ++j) sv += Cfg::A[i][j] * u[j * n + k];
            const real ref = pmax(dabs(sv), dabs(base[k]));
            real tol = Cfg::newton_atol[k] + Cfg::newton_rtol[k] * ref;
            tol = pmax(tol, real(1e-16));
            const real r = sdiv<Cfg>(vals[e], tol);
            nrm2 += r * r;
        }
        return nrm2 * real(1.0 / double(W));
    }
};

template <typename Cfg, typename Sys>
struct FIRKStep {
    static constexpr int n = Cfg::n;
    static constexpr int s = Cfg::stages;
    static constexpr int W = s * n;
    static constexpr int nd = Cfg::n_drivers;
    Vec<real, W> stage_increment;   // persists across steps
    real previous_step_size;
    real theta;

    __device__ __forceinline__ void init() {
CUBIE_UNROLL
        for (int e = 0; e < W; ++e) stage_increment[e] = real(0);
        previous_step_size = real(0);
        theta = real(0);
    }

    // Dense read-ahead of the previous step's increments, in place
    // (stage_predictors.py:492-548).
    __device__ __forceinline__ void predict(real step_ratio, bool apply) {
        if constexpr (Cfg::dense_prediction) {
            constexpr int P = Cfg::pred_powers;
            constexpr int R = Cfg::pred_rows;
            constexpr int F = Cfg::pred_first;
            real transform[R * s];
CUBIE_UNROLL
            for (int e = 0; e < R * s; ++e) {
                real acc = real(0);
CUBIE_UNROLL
                for (int p = P - 1; p >= 0; --p) acc = acc * step_ratio + Cfg::pred_coeffs[p][e];
                transform[e] = acc * step_ratio;
            }
CUBIE_UNROLL
            for (int k = 0; k < n; ++k) {
                real prev[s];
CUBIE_UNROLL
                for (int j = 0; j < s; ++j) prev[j] = stage_increment[j * n + k];
CUBIE_UNROLL
                for (int r = 0; r < R; ++r) {
                    real acc = real(0);
CUBIE_UNROLL
                    for (int j = 0; j < s; ++j) acc += transform[r * s + j] * prev[j];
                    const int target = (F + r) * n + k;
                    stage_increment[target] = apply ? acc : stage_increment[target];
                }
            }
        }
    }

    template <typename Ctx>
    __device__ __forceinline__ int step(Ctx& ctx, const Vec<real, n>& state, Vec<real, n>& proposed,
                                        Vec<real, Cfg::n_error>& error, real dt, real time,
                                        double /*t64*/, bool first_step, bool prev_accepted,
                                        int* counters) {
        const real current_time = time;
        const real end_time = current_time + dt;
        int status = ST_SUCCESS;
        if constexpr (Cfg::dense_prediction) {
            const real previous_dt = previous_step_size;
            previous_step_size = dt;
            const real safe_prev = previous_dt > real(0) ? previous_dt : dt;
            const real step_ratio = dt / safe_prev;
            const bool apply = (!first_step) && prev_accepted && (step_ratio <= Cfg::pred_max_ratio);
            predict(step_ratio, apply);
        }
CUBIE_UNROLL
        for (int k = 0; k < n; ++k) {
            if constexpr (Cfg::accumulates_output) proposed[k] = state[k];
            if constexpr (Cfg::has_error && Cfg::accumulates_error) error[k] = real(0);
        }
        Vec<real, (nd > 0 ? s * nd : 1)> stack;
        if constexpr (nd > 0) {
CUBIE_UNROLL
            for (int i = 0; i < s; ++i) ctx.drv.eval(current_time + dt * Cfg::c[i], stack.data() + i * nd);
        }

        FirkProblem<Cfg, Sys> P;
        LinInputs<Cfg, (nd > 0 ? s * nd : 1)> li;
        li.bind(ctx.params.data(), stack.data());
        P.u = stage_increment.data();
        P.base = state.data();
        P.params = ctx.params.data();
        P.drivers = stack.data();
        P.params_l = li.params;
        P.drivers_l = li.drivers;
        P.t = current_time;
        P.h = dt;
        status |= newton_solve<Cfg>(P, theta, counters);

CUBIE_UNROLL
        for (int i = 0; i < s; ++i) {
            if constexpr (nd > 0) {
CUBIE_UNROLL
                for (int q = 0; q < nd; ++q) ctx.proposed_drivers[q] = stack[i * nd + q];
            }
            const bool out_row = !Cfg::accumulates_output && Cfg::b_row == i;
            const bool err_row = Cfg::has_error && !Cfg::accumulates_error && Cfg::b_hat_row == i;
            if (out_row || err_row) {
                real Y[n];
                P.template combine<true>(i, stage_increment.data(), Y);
CUBIE_UNROLL
                for (int k = 0; k < n; ++k) {
                    if (out_row) proposed[k] = Y[k];
                    if constexpr (Cfg::has_error && !Cfg::accumulates_error) {
                        if (err_row) error[k] = Y[k];
                    }
                }
            }
        }
        if constexpr (Cfg::accumulates_output) {
CUBIE_UNROLL
            for (int k = 0; k < n; ++k) {
                real acc = real(0), comp = real(0);
CUBIE_UNROLL
                for (int i = 0; i < s; ++i) {
                    const real term = Cfg::b[i] * stage_increment[i * n + k] - comp;
                    const real next = acc + term;
                    comp = (next - acc) - term;
                    acc = next;
                }
                proposed[k] = state[k] + acc;
            }
        }
        if constexpr (Cfg::has_error && Cfg::accumulates_error) {
CUBIE_UNROLL
            for (int k = 0; k < n; ++k) {
                real acc = real(0), comp = real(0);
CUBIE_UNROLL
                for (int i = 0; i < s; ++i) {
                    const real term = Cfg::d[i] * stage_increment[i * n + k] - comp;
                    const real next = acc + term;
                    comp = (next - acc) - term;
                    acc = next;
                }
                error[k] = acc;
            }
        }
        if constexpr (Cfg::c[s - 1] != 1.0) ctx.drv.eval(end_time, ctx.proposed_drivers.data());
        if constexpr (Cfg::n_obs > 0)
            Sys::observables(proposed.data(), ctx.params.data(), ctx.proposed_drivers.data(),
                             ctx.proposed_observables.data(), end_time);
        if constexpr (Cfg::has_error && !Cfg::accumulates_error) {
CUBIE_UNROLL
            for (int k = 0; k < n; ++k) error[k] = proposed[k] - error[k];
        }
        return status;
    }
};

}  // namespace cubie
