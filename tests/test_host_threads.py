"""Host copies on the library's worker threads (copy_threads), without a GPU:
a small program linked against the library, whose pthread_create fails after
a given number of threads, as it does where a process may start no more."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "lammps-tensormd_amd", "lib")

PROGRAM = r"""
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <cstdio>
#include <cstdlib>
#include <vector>
namespace tmd {
struct HostCopy {
  void *dst;
  const void *src;
  size_t bytes;
};
void copy_threads(const HostCopy *c, int n);
}
static int allowed = 0, started = 0;
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg)
{
  using F = int (*)(pthread_t *, const pthread_attr_t *, void *(*) (void *), void *);
  static F real = (F) dlsym(RTLD_NEXT, "pthread_create");
  if (started >= allowed) return EAGAIN;
  started++;
  return real(t, a, f, arg);
}
int main(int argc, char **argv)
{
  allowed = std::atoi(argv[1]);
  // below and above the line from which the threads share a copy, odd sizes,
  // pieces that span two of the copies
  for (size_t scale : {1ul, 40ul, 400ul}) {
    size_t len[3] = {33000 * scale + 1, 7 * scale, 65536 * scale + 13};
    std::vector<unsigned char> src[3], dst[3];
    tmd::HostCopy c[3];
    for (int k = 0; k < 3; k++) {
      src[k].resize(len[k]);
      for (size_t i = 0; i < len[k]; i++) src[k][i] = (unsigned char) (i * 31 + i / 255 + k);
      dst[k].assign(len[k] + 1, 0xEE);
      c[k] = {dst[k].data(), src[k].data(), len[k]};
    }
    tmd::copy_threads(c, 3);
    for (int k = 0; k < 3; k++) {
      for (size_t i = 0; i < len[k]; i++)
        if (dst[k][i] != src[k][i]) return std::printf("copy %d differs at %zu\n", k, i), 1;
      if (dst[k][len[k]] != 0xEE) return std::printf("copy %d runs over\n", k), 1;
    }
  }
  std::printf("ok, %d threads started\n", started);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists(os.path.join(LIB, "libtensormd_amd.so")),
                    reason="needs g++ and the built library")
@pytest.mark.parametrize("threads", [0, 2, 64])
def test_copies_with_few_threads(tmp_path, threads):
    src, exe = tmp_path / "copies.cpp", tmp_path / "copies"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", str(src), "-o", str(exe), "-rdynamic", "-L" + LIB, "-ltensormd_amd",
                    "-Wl,-rpath," + LIB + ":/opt/rocm/lib", "-Wl,--allow-shlib-undefined", "-ldl", "-lpthread"],
                   check=True)
    r = subprocess.run([str(exe), str(threads)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-500:])
    assert r.stdout.startswith("ok")
