// kmc_transfer.h -- internal interface of the exact transfer rate used by the KMC context.
#pragma once
#include <cstdint>

#include "../../include/cntkmc.h"

namespace cntkmc {

// kmc_transfer_rates_device in two halves, so that the transfers of several chirality classes
// can run side by side, each on its own stream: transfer_launch queues the work and returns,
// transfer_wait waits for all that was queued.  The inputs must be ready (no stream waits on
// another) and stay untouched until the wait.
int transfer_launch(kmc_transfer* t, int64_t n, const double* d_theta, const double* d_z,
                    const double* d_a1, const double* d_a2, const int64_t* d_sel, double* d_rate);
int transfer_wait(kmc_transfer* t);

}  // namespace cntkmc
