"""Copies of host memory with helper threads (csrc/hip/fe_host_copy.h), in a C++ program of its own:
a process forked after the helpers have started, asleep or polling, copies right and ends, and so
does its parent; copies of sizes about the chunk length, alone and from two threads at once, arrive whole.
"""
import os
import subprocess

import pytest

SOURCE = r"""
#include "fe_host_copy.h"
#include <signal.h>
#include <stdio.h>
#include <stdlib.h>
#include <sys/wait.h>
#include <time.h>
#include <vector>

static void nap(int ms) { timespec t{ms / 1000, (ms % 1000) * 1000000L}; nanosleep(&t, nullptr); }

static bool copies(unsigned seed) {
  const size_t C = HostCopy::CHUNK, sizes[] = {0, 1, C - 1, C, C + 1, 3 * C - 5, 16 * C, 33 * C + 7};
  for (size_t n : sizes) {
    std::vector<unsigned char> a(n), b(n + 1, 0xa5);
    for (size_t i = 0; i < n; ++i) a[i] = (unsigned char)(i * 2654435761u >> 13) ^ (unsigned char)seed;
    g_copy.copy(b.data(), a.data(), n);
    if (memcmp(a.data(), b.data(), n) != 0 || b[n] != 0xa5) return false;
  }
  return true;
}

int main(int argc, char **argv) {
  const char *mode = argv[1];
  g_copy.begin();
  if (!copies(1)) return 3;
  if (!strcmp(mode, "threads")) {
    bool ok[2] = {true, true};
    std::thread t([&] { for (int i = 0; i < 40; ++i) ok[1] = copies(100 + i) && ok[1]; });
    for (int i = 0; i < 40; ++i) ok[0] = copies(200 + i) && ok[0];
    t.join();
    g_copy.end();
    return ok[0] && ok[1] ? 0 : 3;
  }
  if (!strcmp(mode, "asleep")) {
    g_copy.end();
    nap(50);                                   /* the helpers go to sleep */
  }
  const pid_t child = fork();
  if (child == 0) {
    g_copy.begin();
    const bool ok = copies(2);
    g_copy.end();
    exit(ok ? 0 : 3);                          /* runs the destructors */
  }
  int st = 0;
  for (int i = 0; waitpid(child, &st, WNOHANG) == 0; ++i) {
    if (i == 200) {                            /* 10 s */
      kill(child, SIGKILL);
      waitpid(child, &st, 0);
      fprintf(stderr, "the forked child did not end\n");
      return 4;
    }
    nap(50);
  }
  if (!WIFEXITED(st) || WEXITSTATUS(st) != 0) return 5;
  return copies(3) ? 0 : 3;
}
"""


@pytest.fixture(scope="module")
def program(repo, tmp_path_factory):
    d = tmp_path_factory.mktemp("host_copy")
    (d / "main.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-variable", "-pthread",
                    "-I" + os.path.join(repo, "fasteddy-model_amd", "csrc", "hip"), str(d / "main.cpp"), "-o", str(d / "main")],
                   check=True)
    return str(d / "main")


@pytest.mark.parametrize("mode", ["threads", "asleep", "polling"])
def test_copies_and_forked_children(program, mode):
    r = subprocess.run([program, mode], timeout=60, capture_output=True, text=True)
    assert r.returncode == 0, (mode, r.returncode, r.stderr)
