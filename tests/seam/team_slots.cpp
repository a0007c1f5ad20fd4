// Order in which iterations get their workgroups out of a device's budget: one that wants all of it comes
// while another holds a part, and one that wants a little comes behind it.  Prints the order.
#include <chrono>
#include <cstdio>
#include <memory>
#include <string>
#include <thread>

#include "ptyk_team_slots.h"

using ptyk::TeamBudget;
using ptyk::TeamSlots;

int main() {
  TeamBudget b;
  std::mutex mu;
  std::string order;
  auto note = [&](char c) {
    std::lock_guard<std::mutex> l(mu);
    order += c;
  };
  auto waiting = [&](unsigned long n) {  // until n have come
    for (;;) {
      {
        std::lock_guard<std::mutex> l(b.mu);
        if (b.came == n) return;
      }
      std::this_thread::sleep_for(std::chrono::milliseconds(1));
    }
  };
  auto first = std::make_unique<TeamSlots>(&b, 4, 1);
  note('a');
  std::thread large([&] {
    TeamSlots s(&b, 4, 4);
    note('b');
  });
  waiting(2);
  std::thread small([&] {
    TeamSlots s(&b, 4, 1);
    note('c');
  });
  waiting(3);
  std::this_thread::sleep_for(std::chrono::milliseconds(100));  // time to be let in out of turn
  first.reset();
  large.join();
  small.join();
  { TeamSlots none(nullptr, 4, 4), nothing(&b, 4, 0); }
  TeamSlots all(&b, 4, 4);
  std::printf("%s %d\n", order.c_str(), b.left);
  return order == "abc" && b.left == 0 ? 0 : 1;
}
