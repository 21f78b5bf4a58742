"""The host copy that other threads help with (no GPU needed: the header is compiled here):
every byte at sizes around the blocks' edges and from several callers at once, pages touched
without a change, helpers that cannot be started, and a child process without them."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <sys/resource.h>
#include <sys/wait.h>
#include <unistd.h>
#include <cstdio>
#include <vector>
#include "qed_hostcopy.hpp"
using bytes = std::vector<unsigned char>;
static int run(size_t len, int times = 1) {
  bytes src(len + 1), dst(len + 1, 0);
  for (size_t i = 0; i < len; ++i) src[i] = (unsigned char)(1 + i * 2654435761u % 255);
  int bad = 0;
  for (int t = 0; t < times; ++t) {
    if (len) src[len / 2] ^= 0x40;
    qed::CopyHelpers::get().copy(dst.data(), src.data(), len);
    bad += dst != src;
  }
  qed::touch_pages(src.data(), len);
  return bad + (dst != src);
}
int main(int argc, char**) {
  int bad = 0;
  if (argc > 1) {  // room for the buffers, not for a helper's stack
    size_t pages = 0;
    FILE* f = fopen("/proc/self/statm", "r");
    if (!f || fscanf(f, "%zu", &pages) != 1) return 2;
    fclose(f);
    const size_t room = pages * sysconf(_SC_PAGESIZE) + (size_t(100) << 20);
    rlimit as{room, room};
    setrlimit(RLIMIT_AS, &as);
    bad += run(size_t(16) << 20, 3);
  } else {
    for (size_t len : {size_t(0), size_t(1), size_t(4097), size_t(8) << 20, (size_t(8) << 20) + 1,
                       (size_t(9) << 20) + 12345, size_t(16) << 20})
      bad += run(len, 3);
    std::vector<std::thread> callers;
    std::vector<int> res(4, 1);
    for (int c = 0; c < 4; ++c) callers.emplace_back([&res, c] { res[c] = run((size_t(8) << 20) + c * 1000, 20); });
    for (auto& t : callers) t.join();
    for (int r : res) bad += r;
    const pid_t child = fork();
    if (child == 0) _exit(run(size_t(16) << 20, 2));
    int status = 1;
    waitpid(child, &status, 0);
    bad += status != 0;
  }
  printf("bad %d\n", bad);
  return bad != 0;
}
"""


@pytest.mark.parametrize("limited", [False, True])
def test_copy_with_and_without_helpers(tmp_path, limited):
    src, exe = tmp_path / "copy.cpp", tmp_path / "copy"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "pyqcm_amd", "csrc"),
                           str(src), "-o", str(exe)])
    # a new thread's stack is as large as this limit when the program starts
    cmd = "ulimit -s 131072; exec %s limited" % exe if limited else str(exe)
    r = subprocess.run(["bash", "-c", cmd], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
