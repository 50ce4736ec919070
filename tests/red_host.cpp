// Follows the step control (bdf_core.h) with the solve kernel's reduction buffers (ucg_reduce.h)
// and barriers, and counts the uses of a buffer that no barrier separates from its last reads.
// Built by tests/test_reductions_host.py with g++.
//
// Recorder computes as HostOps does and logs what the kernel's Ops does in the same call: a
// reduction is a write to its buffer, a barrier, and reads of it; the other calls have the barriers
// listed here at least (a barrier more in the kernel would only separate uses further).
#include <pthread.h>

#include <atomic>
#include <thread>

#include "bdf_host.cpp"

#include "../uclchem_amd/csrc/ucg_reduce.h"

namespace {

struct Recorder : HostOps {
    using HostOps::HostOps;
    bool open[ucg::RED_NBUF] = {};   // read since the last barrier
    int hazards = 0, reductions = 0, order_after_correction = 0, last = -1;
    void barrier()
    {
        for (bool &o : open) o = false;
        last = -1;
    }
    void reduce(int id)
    {
        reductions++;
        if (open[id]) hazards++;
        if (id == ucg::OpsBuffers::order && last == ucg::OpsBuffers::correction) order_after_correction++;
        barrier();
        open[id] = true;
        last = id;
    }
    bool set_ewt(double rtol)
    {
        reduce(ucg::OpsBuffers::weights);
        return HostOps::set_ewt(rtol);
    }
    double wrms(int v)
    {
        if (v != bdf::Z0) reduce(v == bdf::ACOR ? ucg::OpsBuffers::acor : ucg::OpsBuffers::history);
        return HostOps::wrms(v);
    }
    double wrms_acor_minus(double c, int zj)
    {
        reduce(ucg::OpsBuffers::order);
        return HostOps::wrms_acor_minus(c, zj);
    }
    double apply_correction(double scale)
    {
        reduce(ucg::OpsBuffers::correction);
        return HostOps::apply_correction(scale);
    }
    double hub_inverse(double fac)
    {
        reduce(ucg::OpsBuffers::first_step);
        return HostOps::hub_inverse(fac);
    }
    double ydd_norm(double t0, double hg)
    {
        barrier();
        reduce(ucg::OpsBuffers::ydd);
        return HostOps::ydd_norm(t0, hg);
    }
    void start_corrector()
    {
        HostOps::start_corrector();
        barrier();
    }
    void rhs()
    {
        HostOps::rhs();
        barrier();
    }
    void form_residual(double gamma, double rl1)
    {
        HostOps::form_residual(gamma, rl1);
        barrier();
    }
    int setup(double gamma, bool j)
    {
        barrier();
        return HostOps::setup(gamma, j);
    }
    void solve()
    {
        HostOps::solve();
        barrier();
    }
};

}  // namespace

extern "C" {

// Consecutive integrate() calls from t = 0 to each of tout[0..ncalls), as a point's intervals.
// out: hazards, reductions, order decisions that follow a correction without a barrier.
int red_host_run(int problem, int ncalls, const double *tout, double rtol, double atol, const double *y0, int mxstep,
                 int *out)
{
    if (problem < 0 || problem > 2) return -100;
    Recorder o(PROBLEMS[problem].n);
    o.P = &PROBLEMS[problem];
    for (int i = 0; i < o.n; i++) {
        o.z[0][i] = y0[i];
        o.atol[i] = atol;
    }
    double t = 0.0;
    int r = 0;
    for (int c = 0; c < ncalls; c++) {
        bdf::Stats st;
        o.barrier();   // the rates before every call end in one
        r = bdf::integrate(o, t, tout[c], rtol, mxstep, st);
    }
    out[0] = o.hazards;
    out[1] = o.reductions;
    out[2] = o.order_after_correction;
    return r;
}

// `threads` threads poll a cancel word that answers 1 from its `raised`-th reading on, `calls`
// times each, every `every`-th call.  seen [threads][calls]: what each poll returned; returns the
// number of readings of the word.
int red_host_cancel(int threads, int calls, int every, int raised, int *seen)
{
    pthread_barrier_t bar;
    pthread_barrier_init(&bar, nullptr, threads);
    std::atomic<int> readings{0};
    double flag = 0.0;
    std::vector<std::thread> team;
    for (int w = 0; w < threads; w++)
        team.emplace_back([&, w] {
            int n = 0;
            for (int c = 0; c < calls; c++) {
                seen[w * calls + c] = ucg::cancel_poll(
                    n, every, w == 0, flag, [&] { return ++readings >= raised; },
                    [&] { pthread_barrier_wait(&bar); });
                pthread_barrier_wait(&bar);   // a step has barriers
            }
        });
    for (auto &t : team) t.join();
    pthread_barrier_destroy(&bar);
    return readings;
}
}
