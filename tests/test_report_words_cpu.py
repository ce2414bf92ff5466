"""The host words that launches report a wait that gave up to, compiled against stand-ins for the runtime: memory that cannot be had is
asked for again by the next call instead of failing every later one, and until it is there only launches that are waited for (and
have a status word to copy) may have workgroups that wait for each other."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ttt-tk_amd", "csrc")

PROGRAM = r"""
#include "ttt_mlp_report.hpp"
#include <cassert>
#include <cstdio>
#include <cstdlib>
static int fail = 0, asked = 0, errors = 0, mode_now = 0;
extern "C" hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  assert(mode_now == hipStreamCaptureModeRelaxed);
  asked++;
  if (fail > 0) { fail--; errors++; return hipErrorOutOfMemory; }
  *p = malloc(n);
  return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { const hipError_t e = errors ? hipErrorOutOfMemory : hipSuccess; errors = 0; return e; }
extern "C" hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
  const int old = mode_now; mode_now = *m; *m = static_cast<hipStreamCaptureMode>(old); return hipSuccess;
}
int main() {
  ReportWords r;
  mode_now = hipStreamCaptureModeGlobal;
  fail = 3;
  assert(!r.serves(false));                       // nobody waits and there is no word: one workgroup per pair
  assert(r.take() == nullptr && r.serves(true));  // a waiting call copies the status word
  assert(!r.serves(false) && asked == 3 && errors == 0);
  assert(r.serves(false) && asked == 4);          // there is room again
  assert(r.collecting() != nullptr && asked == 4 && mode_now == hipStreamCaptureModeGlobal);
  int* words[ReportWords::WORDS];
  int n = 0;
  while ((words[n] = r.take()) != nullptr) { assert(*words[n] == 0 && words[n] != r.collecting()); *words[n++] = 1; }
  assert(n == ReportWords::WORDS - 1);
  r.give(words[5]);
  int* w = r.take();
  assert(w == words[5] && *w == 0 && asked == 4);  // cleared for the next call
  puts("ok");
}
"""


def test_words_are_asked_for_again_and_launches_that_nobody_waits_for_need_one(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", f"-I{CSRC}", f"-I{rocm}/include", str(src), "-o", str(exe), "-pthread"], check=True)
    assert subprocess.run([str(exe)], stdout=subprocess.PIPE, check=True).stdout == b"ok\n"
