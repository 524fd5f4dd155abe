// workspace.h -- device and pinned host memory of a plan, from a pool shared
// by all threads (workspace.cpp).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "spm_kernels.h"

namespace spm {

// One plan's memory: a device block and a pinned host block that holds the
// staged matrix and the run's result.  Owned by one plan at a time.
struct Workspace {
    int device = 0;
    char* dev = nullptr;
    size_t dev_bytes = 0;
    char* host = nullptr;         // staging area, and its device address
    char* host_dev = nullptr;
    size_t host_bytes = 0;
    RunResult* result_host = nullptr;  // in the same pinned block, by host and
    RunResult* result = nullptr;       // by device address
    unsigned int seq = 0;         // last run's flag value
};

// A workspace of at least these sizes on the calling thread's current device
// (= device), or SPM_ENOMEM.
int workspace_get(int device, size_t dev_bytes, size_t host_bytes, Workspace** out);
// Back to the pool, when nothing on the device uses it any more, or (idle
// false, or the pool is full) freed after the device's work.
void workspace_put(Workspace* w, bool idle);

}  // namespace spm
