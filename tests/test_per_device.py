"""No-GPU checks of what the library keeps per device: a kernel's dynamic LDS limit belongs to a device, so it is raised once on each
one, whichever threads the contexts run in."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pooled_amd", "csrc")

PROGRAM = r"""
#include "pa_per_device.h"
#include <cstdio>
#include <thread>
#include <vector>
enum Err { OK = 0, BAD = 7 };
static PaPerDevice flag;
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
  int calls = 0;
  auto good = [&] { calls++; return OK; };
  CHECK(flag.once(0, good) == OK && calls == 1);
  CHECK(flag.once(0, good) == OK && calls == 1);                        // done on this device
  CHECK(flag.once(3, good) == OK && calls == 2);                        // another device has a limit of its own
  CHECK(flag.once(5, [] { return BAD; }) == BAD);
  CHECK(flag.once(5, good) == OK && calls == 3);                        // a failure is not remembered as done
  CHECK(flag.once(PA_MAX_DEVICES - 1, good) == OK && calls == 4);
  for (int d : { -1, PA_MAX_DEVICES }) for (int i = 0; i < 2; i++) CHECK(flag.once(d, good) == OK);   // outside the table: every time
  CHECK(calls == 8);
  std::atomic<int> n[PA_MAX_DEVICES] = {};
  static PaPerDevice shared;
  std::vector<std::thread> ts;
  std::atomic<bool> early{false};
  for (int t = 0; t < 8; t++)
    ts.emplace_back([&, t] {
      for (int i = 0; i < 2000; i++) {
        const int d = (i + t) % PA_MAX_DEVICES;
        shared.once(d, [&] { n[d]++; return OK; });
        if (n[d] == 0) early = true;                                    // returned before anyone had done it
      }
    });
  for (auto& t : ts) t.join();
  CHECK(!early);
  for (int d = 0; d < PA_MAX_DEVICES; d++) CHECK(n[d] >= 1 && n[d] <= 8);
  puts("ok");
}
"""


def test_once_on_every_device(tmp_path):
    src, exe = tmp_path / "t.cc", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", CSRC, str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_every_kernel_attribute_is_set_per_device():
    """hipFuncSetAttribute is called by the per-device helper alone, each of whose callers hands in a flag of its own kernel."""
    sites, uses, flags = [], 0, 0
    for name in sorted(os.listdir(CSRC)):
        text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, name)).read())
        sites += [name] * len(re.findall(r"\bhipFuncSetAttribute\s*\(", text))
        if name.endswith(".hip"):
            uses += len(re.findall(r"\bpa_lds_limit\s*\(", text))
            flags += len(re.findall(r"\bstatic\s+PaPerDevice\b", text))
    assert sites == ["pa_internal.h"]
    assert uses == flags >= 4
