// Flag words of the ePIE team's barriers (ptyk_epie.hip), apart from how they are loaded and stored, so
// that the protocol can be checked on the host over every order of its steps
// (tests/seam/team_barrier.cpp).
#pragma once

#ifdef __HIPCC__
#define PTYK_TEAM_FN __host__ __device__ constexpr
#else
#define PTYK_TEAM_FN constexpr
#endif

namespace ptyk {

constexpr int PTYK_EPIE_TEAM_MAX = 128;    // workgroups of the largest team
constexpr int PTYK_EPIE_FLAG_STRIDE = 16;  // 64-bit words of one workgroup: a 128-byte line, two in use

// A workgroup announces barrier `epoch` by one store of (epoch, value) to its word for that barrier, and
// waits until every workgroup's word for it holds that epoch; the values read then are the barrier's.
// Words alternate between barriers.  A workgroup that is past barrier e may announce e + 1 while a slower
// one still reads the words of e: those are other words.  It overwrites its word of e when it announces
// e + 2, which it does after its wait for e + 1, which needs everyone's announcement of e + 1, which each
// makes after its own wait for e: by then nobody reads the words of e any more.  (With one word a
// workgroup, a slow reader took the next barrier's value for this one's.)
PTYK_TEAM_FN int team_word(int w, unsigned epoch) { return w * PTYK_EPIE_FLAG_STRIDE + (int)(epoch & 1u); }
PTYK_TEAM_FN unsigned long long team_flag(unsigned epoch, unsigned value) {
  return ((unsigned long long)epoch << 32) | value;
}
PTYK_TEAM_FN bool team_here(unsigned long long flag, unsigned epoch) { return (unsigned)(flag >> 32) == epoch; }
PTYK_TEAM_FN unsigned team_value(unsigned long long flag) { return (unsigned)flag; }

}  // namespace ptyk
