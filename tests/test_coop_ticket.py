"""Tickets of the one-launch inner solves (csrc/ticket.h), on the host: the
work-groups in flight on a device never exceed its compute units, also in
whole rounds over the eight XCDs, whatever the device's size; devices do not
count against each other; a ticket is given back."""
import os
import subprocess


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "ticket.h"
#include <cstdio>
#include <memory>
#include <thread>
#include <vector>
using cloth::CoopTicket;
static int bad = 0;
static void check(bool ok, const char* what) { if (!ok) { bad = 1; std::printf("wrong: %s\n", what); } }
// how many launches of `blocks` work-groups a device of `cus` units takes
static unsigned granted(int device, unsigned blocks, unsigned cus) {
  std::vector<std::unique_ptr<CoopTicket>> held;
  for (;;) {
    std::unique_ptr<CoopTicket> t(new CoopTicket(device, blocks, cus));
    if (!*t) return (unsigned)held.size();
    held.push_back(std::move(t));
  }
}
int main() {
  check(granted(0, 64, 256) == 4, "four solves of 64 on 256 units");
  check(granted(0, 64, 64) == 1, "one on 64");
  check(granted(0, 64, 32) == 0, "none on 32");
  check(granted(0, 32, 32) == 1, "32 on 32");
  check(granted(0, 2, 256) == 32, "two work-groups take a round of eight");
  check(granted(0, 57, 256) == 4 && granted(0, 56, 256) == 4 && granted(0, 48, 256) == 5, "whole rounds");
  check(granted(0, 1, 0) == 0 && granted(-1, 1, 256) == 0 && granted(CoopTicket::kMaxDevices, 1, 256) == 0, "no device");
  {
    CoopTicket a(1, 200, 256), b(1, 64, 256), c(2, 200, 256), d(1, 56, 256);
    check(a && !b && c && d, "devices apart, the rest is free");
  }
  check(granted(1, 64, 256) == 4, "given back");
  // never more in flight than units, from several threads
  std::atomic<unsigned> now{0}, most{0}, taken{0};
  std::vector<std::thread> th;
  for (int k = 0; k < 8; k++)
    th.emplace_back([&, k] {
      const unsigned blocks = 8u * (1 + k);
      for (int i = 0; i < 20000; i++) {
        CoopTicket t(3, blocks, 96);
        if (!t) continue;
        taken++;
        const unsigned n = now.fetch_add(blocks) + blocks;
        unsigned m = most.load();
        while (m < n && !most.compare_exchange_weak(m, n)) {}
        now.fetch_sub(blocks);
      }
    });
  for (auto& t : th) t.join();
  check(most.load() <= 96 && taken.load() > 0, "threads");
  check(granted(3, 96, 96) == 1, "all given back");
  return bad;
}
"""


def test_work_groups_in_flight_fit_the_device(tmp_path):
    src, exe = str(tmp_path / "t.cpp"), str(tmp_path / "t")
    with open(src, "w") as f:
        f.write(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", os.path.join(ROOT, "closim_amd", "csrc"), src, "-o",
                    exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
