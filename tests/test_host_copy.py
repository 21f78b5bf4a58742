"""The host copy by several threads (no GPU needed: the header is compiled here): every byte
at sizes around the pieces' edges, and with threads that cannot be started."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <sys/resource.h>
#include <unistd.h>
#include <cstdio>
#include "qed_hostcopy.hpp"
using bytes = std::vector<unsigned char>;
static int run(size_t len, int nt) {
  bytes src(len + 1), dst(len + 1, 0);
  for (size_t i = 0; i < len; ++i) src[i] = (unsigned char)(1 + i * 2654435761u % 255);
  qed::copy_parallel(dst.data(), src.data(), len, nt);
  return dst == src ? 0 : 1;
}
int main() {
  int bad = 0;
  for (int nt : {1, 2, 7, 8})
    for (size_t len : {size_t(0), size_t(1), size_t(4095), size_t(4096), size_t(4097), size_t(8 * 4096),
                       size_t(8 * 4096 + 1), size_t(16) << 20})
      bad += run(len, nt);
  if (qed::copy_threads(1) != 1 || qed::copy_threads(size_t(16) << 20) < 1) ++bad;
  // room for the buffers and at most one thread's stack of 64 MB more
  size_t pages = 0;
  FILE* f = fopen("/proc/self/statm", "r");
  if (!f || fscanf(f, "%zu", &pages) != 1) return 2;
  fclose(f);
  rlimit stack{size_t(64) << 20, size_t(64) << 20};
  setrlimit(RLIMIT_STACK, &stack);
  const size_t room = pages * sysconf(_SC_PAGESIZE) + (size_t(100) << 20);
  rlimit as{room, room};
  setrlimit(RLIMIT_AS, &as);
  bad += run(size_t(16) << 20, 8);
  printf("bad %d\n", bad);
  return bad != 0;
}
"""


def test_copy_with_threads_that_do_not_start(tmp_path):
    src, exe = tmp_path / "copy.cpp", tmp_path / "copy"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "pyqcm_amd", "csrc"),
                           str(src), "-o", str(exe)])
    # the limit on a new thread's stack is read when the program starts
    r = subprocess.run(["bash", "-c", "ulimit -s 65536; exec " + str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
