"""Admission of one-launch solves to a device (fe_resident_gate.h), compiled for
the host: small launches of several threads are inside together, never more
than fit, and one that needs the whole device gets its turn."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "feng_amd" / "csrc"

PROGRAM = r"""
#include "fe_resident_gate.h"
#include <atomic>
#include <cassert>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
using namespace std::chrono;
static bool until(const std::function<bool()> &f)
{
  const auto end = steady_clock::now() + seconds(20);
  while(!f())
    if(steady_clock::now() > end) return false;
    else std::this_thread::sleep_for(microseconds(50));
  return true;
}
int main()
{
  // a workgroup an engine up to 32 on 256 CUs, the whole device at 256 and above
  assert(feGateNeed(1, 256) == 1 && feGateNeed(32, 256) == 1 && feGateNeed(33, 256) == 2 && feGateNeed(256, 256) == 8);
  assert(feGateNeed(225, 256) == 8 && feGateNeed(300, 256) == 8 && feGateNeed(3, 4) == 3 && feGateNeed(5, 0) == 5);
  {  // four of two units are inside together, a fifth is not
    FeResidentGate g;
    std::atomic<int> inside{0}, done{0};
    std::atomic<bool> go{false};
    std::vector<std::thread> ts;
    for(int i = 0; i < 5; ++i)
      ts.emplace_back([&] {
        g.enter(2, kGateCus);
        ++inside;
        const bool ok = until([&] { return go.load(); });
        assert(ok);
        --inside;
        g.leave(2);
        ++done;
      });
    assert(until([&] { return inside == 4; }));
    std::this_thread::sleep_for(milliseconds(50));
    assert(inside == 4 && g.busy());
    go = true;
    for(auto &t : ts) t.join();
    assert(done == 5 && !g.busy());
  }
  {  // a stream of small launches does not keep out one that needs the device
    FeResidentGate g;
    std::atomic<int> used{0}, turns{0};
    std::atomic<bool> stop{false};
    std::vector<std::thread> ts;
    for(int i = 0; i < 6; ++i)
      ts.emplace_back([&, i] {
        while(!stop) {
          const int need = 1 + i % 3;
          g.enter(need, kGateCus);
          const int now = used += need;
          assert(now <= kGateCus);
          std::this_thread::sleep_for(microseconds(100));
          used -= need;
          g.leave(need);
        }
      });
    ts.emplace_back([&] {
      for(int k = 0; k < 50; ++k) {
        g.enter(kGateCus, kGateCus);
        const int now = used += kGateCus;
        assert(now == kGateCus);
        std::this_thread::sleep_for(microseconds(100));
        used -= kGateCus;
        g.leave(kGateCus);
        ++turns;
      }
    });
    const bool ok = until([&] { return turns == 50; });
    stop = true;
    assert(ok);
    for(auto &t : ts) t.join();
    assert(!g.busy());
  }
  puts("ok");
}
"""


def test_gate(tmp_path):
    src = tmp_path / "gate.cpp"
    src.write_text("#undef NDEBUG\n#include <functional>\n" + PROGRAM)
    exe = tmp_path / "gate"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr
