// Teams of workgroups on one XCD (host side).
#pragma once
#include <cstdint>

namespace jet {

constexpr int TEAM_MAX = 32;        // workgroups of a team: one per CU of an XCD
constexpr int32_t TEAM_OWN = 2048;  // vertices a workgroup owns at most
constexpr int32_t TEAM_MAX_N = TEAM_MAX * TEAM_OWN;

// Device words of a team, zero at its launch: start-up and the barrier. Each
// word that is polled or added to has a 128-byte line.
struct TeamCtl {
    int32_t arrived, pad0[31];
    int32_t members, pad1[31];
    int32_t state, pad2[31];  // 0 undecided, the team's size, or -1 (abandoned)
    uint32_t bar, pad3[31];
    int32_t fail, pad4[31];
};

// Jobs of contexts of many workers use teams on levels of up to this many
// vertices: a team kernel holds one of the process's four hardware queues for
// the whole level, and the workgroups of its launch that fall on an XCD where
// another team runs wait for a free CU. 60 mixed graphs on 16 workers: 298-312
// ms without teams, 284 up to 512 vertices, 275 up to 2048, 268-273 up to
// 4096, 287 up to 8192, 342 up to 65,536.
constexpr int32_t TEAM_BATCH_N = 4096;
// Marks the calling thread as a worker of such a context.
void set_batch_thread(bool on);
// Levels of up to this many vertices may take a team on the calling thread (0
// after an abandoned start).
int64_t team_max_n();
// An abandoned start costs the bound of its wait: something else holds the
// XCD's CUs, and is likely to hold them for the next level too. The calling
// thread therefore starts no further team until its entry point returns
// (team_call_begins: the next one begins).
void team_abandoned();
void team_call_begins();

// A place for `team` workgroups on an XCD of the device, held from the launch
// of a team kernel until its result is read: the teams that this process has
// running on an XCD ask for no more CUs than it has. A team that has published
// its result may still be storing for some microseconds, and other kernels and
// other processes are not counted: a team then waits for a CU within the bound
// of its start. Waits until a place is free. A team of one waits for no other
// workgroup and takes no place.
class TeamSlot {
  public:
    explicit TeamSlot(int32_t team);
    ~TeamSlot();
    TeamSlot(const TeamSlot&) = delete;
    TeamSlot& operator=(const TeamSlot&) = delete;
    int32_t xcd() const { return xcd_; }

  private:
    int32_t dev_ = 0, xcd_ = 0, team_ = 0;
};

}  // namespace jet
