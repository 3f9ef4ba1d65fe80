// A run's status is read only if the run wrote it: what an earlier run left does not count.
#include "runtime/run_status.h"

#include <cstdio>

using namespace gpumpi;

int main() {
    RunStatus s{}, got;
    for (int flag = 0; flag < 2; flag++) {
        s.abort_flag = flag;       // as the run before left it
        s.exit_code = 0;
        status_arm(&s);
        if (status_read(&s, &got)) {
            std::printf("the status of the run before (abort %d) passed for this one's\n", flag);
            return 1;
        }
        s.abort_flag = 1 - flag;   // as this run's last kernel writes it
        s.exit_code = 7;
        if (!status_read(&s, &got) || got.abort_flag != 1 - flag || got.exit_code != 7) {
            std::printf("the status written by the run is not read\n");
            return 1;
        }
    }
    return 0;
}
