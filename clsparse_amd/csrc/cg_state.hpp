// Device state of one CG solve, shared by the launch-per-step iteration
// (cg.hip) and the persistent ones (cg_persist_kernel.hpp, fsai_persist.hip).
// Plain C++ (host and device): the host tests compile this header with g++.
#pragma once

#include "persist_plan.hpp"

namespace {

constexpr int kHist = 64;   // residual history ring (VERBOSE printing)
constexpr int kChunk = 32;  // iterations between two looks of the host at most (even: both parities)

enum Crit : int { kCritL1Ref = 0, kCritL2 = 1 };
enum Prec : int { kPrecNone = 0, kPrecJacobi = 1, kPrecFsai = 2 };

}  // namespace

struct CgDevState
{
    double norm_ref;   // denominator of the residual (||b||_1 or ||b||_2)
    double init_res;
    double rel_tol;
    double abs_tol;
    double cur_res;
    int max_iters;
    int done;
    int n_iters;
    int iter;
    int converged;
    int crit;
    // Copy of done taken by the x / r update of each iteration: the p update
    // skips on it, since its own workgroup 0 may set done while other
    // workgroups of the same launch have yet to start (they would skip their
    // rows of p, which a residual replacement still uses).
    int stop;
    // The p update fused into the next iteration (Jacobi / no preconditioner
    // with A in diagonal storage): the SpMV kernel forms p' = fma(beta_f, p, z)
    // on the fly and publishes beta_f for the x / r update, which stores p'
    // and clears `first`. `first` = 1 while p already holds the search
    // direction (after set-up or a residual replacement): then beta_f = 0 and
    // z holds p, so p' = p. `pending` = 1 from an x / r update to its
    // convergence test.
    int first;
    int pending;
    // Persistent iteration: grid-wide reductions so far (the slots of the
    // next one go by it), and 1 when a launch gave up waiting for another
    // workgroup (its iterations are lost).
    uint32_t epoch;
    int failed;
    double beta_f;
    double best_res;  // persistent learned-FSAI iteration: fsai_persist.hpp
    double hist[kHist];
};

// After a launch that gave up and a set-up from the x it left: the state of a
// solve after `iter` iterations (those before that launch). Some workgroups may
// have come to the launch's end all the same, with the sums of the one that gave
// up: the state then says done, and x is theirs and older rows mixed.
PP_HD inline void cg_recover(CgDevState& st, double init_res, int iter)
{
    st.failed = 0;
    st.done = 0;
    st.stop = 0;
    st.converged = 0;
    st.n_iters = 0;
    st.pending = 0;
    st.first = 1;
    st.iter = iter;
    st.init_res = init_res;
}
