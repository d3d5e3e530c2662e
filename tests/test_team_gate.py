"""The decision that the four waves of a team workgroup take together before an
item (csrc/team_gate.hpp), on the CPU: whichever wave lags, reading its words only
after the leader has waited and gone on to the barrier, all waves come to the same
answer by the same number of barriers."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "adtomo.jl_amd", "csrc")

MAIN = r"""
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <thread>
#include "team_gate.hpp"

constexpr int kWaves = 4;
std::mutex mu;
std::condition_variable cv;
int arrived, round_no;
bool leader_done;  // the leader has reached the gate's barrier, or is through

bool barrier() {  // false: another wave never came
  std::unique_lock<std::mutex> lk(mu);
  const int r = round_no;
  if (++arrived == kWaves) {
    arrived = 0;
    ++round_no;
    cv.notify_all();
    return true;
  }
  return cv.wait_for(lk, std::chrono::seconds(1), [&] { return round_no != r; });
}

int main(int argc, char** argv) {
  const int lag = atoi(argv[1]);
  int bad = 0;
  for (int c = 0; c < 16; ++c) {
    const bool quit = c & 1, end = c & 2, waits = c & 4, gone = c & 8;
    adt::TDraw d{0, 0, quit ? 1 : 0, 0};
    arrived = round_no = 0;
    leader_done = false;
    int answer[kWaves], syncs[kWaves] = {};
    bool alone[kWaves] = {};
    auto wave = [&](int w) {
      bool first = true;
      auto leader_through = [&] {
        if (w != 0) return;
        std::lock_guard<std::mutex> lk(mu);
        leader_done = true;
        cv.notify_all();
      };
      answer[w] = adt::team_gate(
          d, end, waits, w == 0,
          [&](const int& x) {
            if (w == lag && first) {
              std::unique_lock<std::mutex> lk(mu);
              cv.wait(lk, [] { return leader_done; });
            }
            first = false;
            std::lock_guard<std::mutex> lk(mu);
            return x;
          },
          [&] { return gone; },
          [&] {
            ++syncs[w];
            leader_through();
            if (!barrier()) alone[w] = true;
          });
      leader_through();
    };
    std::thread t[kWaves];
    for (int w = 0; w < kWaves; ++w) t[w] = std::thread(wave, w);
    for (auto& x : t) x.join();
    const bool want = quit || end || (waits && gone);
    for (int w = 0; w < kWaves; ++w)
      if (answer[w] != want || syncs[w] != syncs[0] || alone[w]) {
        printf("quit %d end %d waits %d gone %d: wave %d answers %d after %d barriers\n", quit, end,
               waits, gone, w, answer[w], syncs[w]);
        bad = 1;
      }
  }
  return bad;
}
"""


@pytest.mark.parametrize("lag", [1, 2, 3])
def test_waves_agree_whichever_lags(tmp_path, lag):
    cxx = shutil.which("g++") or shutil.which("clang++")
    assert cxx, "needs a host C++ compiler"
    src, exe = tmp_path / "gate.cpp", tmp_path / "gate"
    src.write_text(MAIN)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe), str(lag)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
