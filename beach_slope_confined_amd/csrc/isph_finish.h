// isph_finish.h -- the scalar part of a BiCGSTAB reduction: the sums t0, t1 of
// a row kernel's block partials become the iteration's scalars and stop flags.
// Shared by the one-block reduction kernel (k_finish) and the solves that
// stay on the chip (k_bicg_resident), so that both take the same decisions
// from the same bits.
#pragma once
#include "isph_kernels.h"

namespace isph {

__device__ __forceinline__ void finish_update(int kind, double t0, double t1, SolverScalars& s,
                                              const SolveCtl& ctl) {
    switch (kind) {
        case FIN_INIT: {
            s.bb = t0;
            s.nb = sqrt(t0);
            s.rr = t1;
            s.prevr = t1;
            s.iters = 0;
            s.total = 0;
            s.first = 1;
            s.status = 0;
            s.nupd = 0;
            s.rh2 = t1;
            s.brk = 0;
            if (t0 == 0.0) {
                s.done = DONE_ZERO_RHS;
                s.relres = 0.0;
            } else if (sqrt(t1) <= ctl.tol * s.nb) {
                s.done = DONE_CONVERGED;
                s.relres = sqrt(t1) / s.nb;
            } else {
                s.done = 0;
            }
            break;
        }
        // breakdown ((rhat, v) = 0, or (t, t) = 0 / (t, s) = 0): the step
        // degenerates to a minimal-residual step (alpha = 0) or to the half
        // step x + alpha p (omega = 0) and ends in a restart
        case FIN_ALPHA: {
            double a = s.prevr / t0;
            if (!isfinite(a)) {
                a = 0.0;
                s.brk = 1;
            }
            s.alpha = a;
            break;
        }
        case FIN_OMEGA: {
            double w = t0 / t1;
            if (!isfinite(w) || w == 0.0) {
                w = 0.0;
                s.brk = 1;
            }
            s.wi = w;
            break;
        }
        case FIN_BETA: {
            const double betas = (t0 / s.prevr) * (s.alpha / s.wi);
            s.betas = betas;
            s.prevr_prev = s.prevr;
            s.prevr = t0;
            s.rr = t1;
            s.iters = s.iters + 1;
            s.total = s.total + 1;
            s.first = 0;
            const double nr = sqrt(t1);
            if (!(fabs(t0) > BRK_COS * sqrt(t1 * s.rh2))) s.brk = 1;
            if (s.brk) {
                // FP64: true residual + restart; mixed: flush + full restart
                // (the flag stays set for the host until FIN_START)
                if (!ctl.mixed) {
                    s.brk = 0;
                    s.done = DONE_RECURRENCE;
                } else {
                    s.done = DONE_UPDATE;
                }
            } else if (!isfinite(betas) || !isfinite(t1)) {
                s.done = DONE_FAILED;
                s.status = ERR_NOCONV;
                s.relres = nr / s.nb;
            } else if (!ctl.mixed && nr <= ctl.tol * s.nb) {
                s.done = DONE_RECURRENCE;
            } else if (ctl.mixed && (nr <= ctl.tol * s.nb || nr <= ctl.delta * s.rupd)) {
                s.done = DONE_UPDATE;
            } else if (s.total >= ctl.maxit) {
                s.done = DONE_FAILED;
                s.status = ERR_NOCONV;
                s.relres = nr / s.nb;
            }
            break;
        }
        case FIN_TRUE: {
            const double nr = sqrt(t1);
            if (nr <= ctl.tol * s.nb) {
                s.done = DONE_CONVERGED;
                s.relres = nr / s.nb;
            } else if (!isfinite(nr)) {
                s.done = DONE_FAILED;
                s.status = ERR_NOCONV;
                s.relres = nr;
            } else {
                s.rr = t1;
                s.prevr = t1;
                s.rh2 = t1;
                s.first = 1;
                s.done = 0;
                if (s.total >= ctl.maxit) {
                    s.done = DONE_FAILED;
                    s.status = ERR_NOCONV;
                    s.relres = nr / s.nb;
                }
            }
            break;
        }
        case FIN_RESID: {
            // mixed outer residual; nupd counts the flushes (ctl.mixed == 2 after a flush)
            s.bb = t0;
            s.nb = sqrt(t0);
            s.nr = sqrt(t1);
            if (ctl.mixed == 2) s.nupd = s.nupd + 1;
            if (t0 == 0.0) {
                s.done = DONE_ZERO_RHS;
                s.relres = 0.0;
                break;
            }
            s.relres = s.nr / s.nb;
            if (s.nr <= ctl.tol * s.nb) {
                s.done = DONE_CONVERGED;
            } else if (ctl.mixed == 2 &&
                       (s.nupd >= ctl.maxupd || s.total >= ctl.maxit || !isfinite(s.nr))) {
                s.done = DONE_FAILED;
                s.status = ERR_NOCONV;
            } else {
                s.done = 0;
            }
            break;
        }
        case FIN_START:
            s.prevr = t0;
            s.prevr_prev = t0;
            s.rh2 = t0;
            s.brk = 0;
            s.rupd = s.nr;
            s.first = 1;
            s.iters = 0;
            s.done = 0;
            break;
        case FIN_REPLACE: {
            s.betas = (t0 / s.prevr_prev) * (s.alpha / s.wi);
            s.prevr = t0;
            s.rupd = s.nr;
            s.done = 0;
            break;
        }
        default:
            break;
    }
}

}  // namespace isph
