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
    int32_t state, pad2[31];  // 0 undecided, 1 go, 2 abandoned
    uint32_t bar, pad3[31];
    int32_t fail, pad4[31];
};

// A place for `team` workgroups on an XCD of the device, held while a team
// kernel runs there: the teams in flight on an XCD never need more CUs than
// it has, so that every team finds room for all of its workgroups. Waits
// until one is free. A team of one waits for no other workgroup and takes no
// place.
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
