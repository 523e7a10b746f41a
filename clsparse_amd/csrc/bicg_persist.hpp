// The persistent BiCGStab iteration as the solver calls it (kernel in
// bicg_persist_kernel.hpp, one source per precision).
#pragma once

#include "bicg_state.hpp"
#include "common.hpp"
#include "persist_host.hpp"
#include "persist_plan.hpp"

// One launch: iterations from the state (x, r, r*, p, Mp = M p, <r*, r>) until
// the device state says done (x complete, also after a stop at the first
// check) or max_run iterations have run.
template <typename T>
struct BiPersistArgs
{
    uint32_t n;
    PersistPlan plan;
    const T* vals;   // diagonal storage, plan.ndiag * n
    int sym;         // the upper half may be read from the lower
    T* x;
    T* r;
    const T* rs;
    T* p;
    T* Mp;
    T* Ms;
    const T* invD;   // null: no preconditioner
    double* rr;      // g_in partials of <r*, r>, in and out
    uint32_t g_in;
    BiDevState* st;
    unsigned long long* slots;
    int max_run;
    int spin_limit;
};

// rows = 0 when the system does not run in one workgroup per CU.
PersistPlan bicg_persist_plan(size_t n, int ndiag, const int32_t* off, size_t value_size, int num_cus);
template <typename T>
clsparseStatus launch_bicg_persist(BiPersistArgs<T> a, hipStream_t s);
