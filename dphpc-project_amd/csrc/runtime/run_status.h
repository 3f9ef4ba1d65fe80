// What the host reads after a run, in pinned memory that the run's last kernel writes.
#pragma once

#include "common.h"

namespace gpumpi {

struct RunStatus {
    int32_t abort_flag, exit_code;
    ErrorRecord err;
};

// Before the launch: no run reports this flag, so an earlier run's status cannot pass for this
// one's if the kernel that writes it never ran.
constexpr int32_t kStatusPending = -1;
inline void status_arm(RunStatus* s) { s->abort_flag = kStatusPending; }

// After the wait: false if the run left no status.
inline bool status_read(const RunStatus* s, RunStatus* out) {
    *out = *s;
    return out->abort_flag != kStatusPending;
}

}  // namespace gpumpi
