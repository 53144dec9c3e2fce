// Places for teams of workgroups on the device's XCDs (team.h).
#include "team.h"

#include <hip/hip_runtime.h>
#include <sched.h>
#include <unistd.h>

#include <algorithm>
#include <mutex>

#include "jet_types.h"
#include "tuning.h"

namespace jet {

namespace {
constexpr int XCDS = 8;
std::mutex g_slot_mu;
int32_t g_slot_load[64][XCDS];
thread_local bool t_batch_thread = false;
thread_local bool t_abandoned = false;
int g_first_xcd = 0;  // taken when all are equally loaded
}  // namespace

void set_batch_thread(bool on) { t_batch_thread = on; }

int64_t team_max_n() {
    if (t_abandoned) return 0;
    return std::min<int64_t>(tuning().wg_max_n, t_batch_thread ? TEAM_BATCH_N : TEAM_MAX_N);
}

void team_abandoned() {
    t_abandoned = true;
    // another process may hold the XCD: processes that meet on one move on by
    // different steps
    std::lock_guard<std::mutex> lk(g_slot_mu);
    g_first_xcd = (g_first_xcd + 1 + (int)(getpid() % (XCDS - 1))) % XCDS;
}
void team_call_begins() { t_abandoned = false; }

TeamSlot::TeamSlot(int32_t team) : team_(team) {
    int dev = 0;
    JET_HIP(hipGetDevice(&dev));
    dev_ = dev & 63;
    if (team_ <= 1) {  // waits for nobody
        team_ = 0;
        return;
    }
    for (;;) {
        {
            std::lock_guard<std::mutex> lk(g_slot_mu);
            int best = g_first_xcd;
            for (int q = 1; q < XCDS; q++) {
                const int x = (g_first_xcd + q) % XCDS;
                if (g_slot_load[dev_][x] < g_slot_load[dev_][best]) best = x;
            }
            if (g_slot_load[dev_][best] + team_ <= TEAM_MAX) {
                g_slot_load[dev_][best] += team_;
                xcd_ = best;
                return;
            }
        }
        sched_yield();
    }
}

TeamSlot::~TeamSlot() {
    std::lock_guard<std::mutex> lk(g_slot_mu);
    g_slot_load[dev_][xcd_] -= team_;
}

}  // namespace jet
