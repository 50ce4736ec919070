// Host build of the device-program planner (uclchem_amd/csrc/ucg_plan.h) for the tests that look
// at its programs.  Test infrastructure: built by tests/test_plan_host.py with g++.
#include <cstddef>
#include <cstdint>

#include "../include/uclchem_gpu.h"
#include "../uclchem_amd/csrc/ucg_plan.h"

extern "C" {

// Programs for `nwave` waves and at most `max_tail` tail rows (twice that as a wide tail).
// out: ok, wide, presum, sparse rows, tail rows, working slots, then {row, first, end} of the three
// sums, then the most slices a wave has in the entry and in the elimination program.  Returns 0, or
// -1 if the planner threw.
int plan_host(const ucg_network_desc *d, int nwave, int max_tail, int *out)
{
    std::vector<int> off((size_t)d->nreac + 1, 0);
    for (int k = 0; k < d->nreac; k++) off[k + 1] = off[k] + d->nfac[k];
    try {
        const ucg::SparsePrograms S = ucg::build_sparse_programs(d, nwave, max_tail, off, off.back());
        const int head[6] = {S.ok, S.wide, S.presum, S.ns, S.t, S.n_slots};
        for (int k = 0; k < 6; k++) out[k] = head[k];
        for (int k = 0; k < 9; k++) out[6 + k] = k < (int)S.sum_rows.size() ? S.sum_rows[k] : -1;
        const ucg::Program *list[2] = {&S.entries, &S.elim};
        for (int k = 0; k < 2; k++) {
            out[15 + k] = 0;
            for (size_t w = 1; w < list[k]->list_ptr.size(); w++)
                out[15 + k] = std::max(out[15 + k], list[k]->list_ptr[w] - list[k]->list_ptr[w - 1]);
        }
    } catch (const std::exception &) {
        return -1;
    }
    return 0;
}
}
