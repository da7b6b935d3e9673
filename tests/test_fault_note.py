"""csrc/fault_note.h: a thread's line goes to stderr where the process ends in
a fault, and the fault ends it as it would have without."""

import shutil
import signal
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "vllm_amd" / "csrc"

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <thread>
#include "fault_note.h"
using vllm_amd::FaultNote;
static void mine(int) { (void)!write(2, "mine\n", 5); _exit(7); }
static volatile int* nowhere = nullptr;
static volatile int zero = 0;
int main(int, char** argv) {
  const std::string what = argv[1];
  if (what == "handler") signal(SIGSEGV, mine);
  if (what == "after") {
    { FaultNote n; n.say("gone"); }
    return *nowhere;
  }
  if (what == "other thread") {
    FaultNote n;
    n.say("the one that waits");
    std::thread([] { FaultNote m; m.say("the one that ends"); *nowhere = 1; })
        .join();
  }
  if (what == "many") {
    // More than there is room for, and one within another.
    FaultNote n[12];
    n[0].say("%s", std::string(1000, 'x').c_str());
    *nowhere = 1;
  }
  if (what == "replaced") {
    { FaultNote n; n.say("gone"); signal(SIGSEGV, mine); }
    return *nowhere;
  }
  FaultNote n;
  n.say("step %d of %s", 3, "race");
  n.say("step %d of %s", 4, "race");
  if (what == "abort") abort();
  if (what == "divide") return 1 / zero;
  *nowhere = 1;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("fault_note")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    "-pthread", f"-I{CSRC}", str(d / "main.cpp"), "-o",
                    str(d / "main")], check=True)
    return d / "main"


@pytest.mark.parametrize("what,code,said", [
    ("fault", -signal.SIGSEGV, "[vllm_amd] ended in: step 4 of race\n"),
    ("abort", -signal.SIGABRT, "[vllm_amd] ended in: step 4 of race\n"),
    ("divide", -signal.SIGFPE, "[vllm_amd] ended in: step 4 of race\n"),
    ("handler", 7, "[vllm_amd] ended in: step 4 of race\nmine\n"),
    ("after", -signal.SIGSEGV, ""),
    ("other thread", -signal.SIGSEGV,
     "[vllm_amd] ended in: the one that ends\n"),
    ("many", -signal.SIGSEGV, "[vllm_amd] ended in: " + "x" * 238 + "\n"),
    ("replaced", 7, "mine\n")])
def test_note(program, what, code, said):
    r = subprocess.run([str(program), what], capture_output=True, text=True,
                       timeout=60)
    assert (r.returncode, r.stderr) == (code, said)
