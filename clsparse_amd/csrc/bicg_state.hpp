// Device state of one BiCGStab solve. Plain C++ (host and device): the host tests
// compile this header with g++.
#pragma once

#include "persist_plan.hpp"

struct BiDevState
{
    double norm_b;
    double rel_tol;
    double abs_tol;
    double init_res;
    double cur_res;
    double alpha_stop;  // alpha of the iteration that stopped at the first check
    int max_iters;
    int n_prior;        // the solver control's nIters before the call
    int iter;           // iterations completed
    int done;
    int stop_kind;      // 1: at the first check (x += alpha Mp pending), 2: at the second
    int n_iters;
    int converged;
    int precond;
    // Persistent iteration: grid-wide sums so far; 1 when a launch gave up
    // waiting for another workgroup.
    uint32_t epoch;
    int failed;
};

namespace {

PP_HD inline bool bi_finished(const BiDevState* st, double res, int it)
{
    const int n = (it == 0) ? st->n_prior : it;
    return res <= st->rel_tol || res <= st->abs_tol * st->init_res || n >= st->max_iters;
}

}  // namespace

// As cg_recover (cg_state.hpp).
PP_HD inline void bi_recover(BiDevState& st, double init_res, int iter)
{
    st.failed = 0;
    st.done = 0;
    st.stop_kind = 0;
    st.converged = 0;
    st.n_iters = 0;
    st.iter = iter;
    st.init_res = init_res;
}
