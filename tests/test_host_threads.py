"""Host passes on threads (csrc/host_threads.hpp) where the system gives fewer
threads than asked for, or none: every item of the pass is still visited once,
under chunk numbers that index the callers' per-thread slots.  And the row
windows (csrc/rowbuild.hpp) of a caller that is one of several threads start
none of their own."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r'''
#include "host_threads.hpp"
#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <dlfcn.h>
#include <pthread.h>
static std::atomic<int> left{0};
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Create create = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
  return left.fetch_sub(1) > 0 ? create(t, a, f, arg) : EAGAIN;
}
int main(int, char** argv) {
  left = std::atoi(argv[1]);
  constexpr int64_t kItems = 1003;
  std::atomic<int> seen[kItems] = {}, chunks[lbamd::kMaxHostThreads] = {};
  lbamd::parallel_ranges(kItems, [&](int64_t b, int64_t e, int t) {
    for (int64_t k = b; k < e; ++k) ++seen[k];
    ++chunks[t];
  }, 1);
  int bad = 0, ran = 0;
  for (auto& s : seen) bad += s != 1;
  for (auto& c : chunks) { bad += c > 1; ran += c; }
  std::printf("bad %d chunks %d of %d\n", bad, ran, lbamd::host_threads());
  return bad != 0 || ran != lbamd::host_threads();
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
@pytest.mark.parametrize("threads", [0, 1, 3, 64])
def test_passes_run_on_the_threads_there_are(tmp_path, threads):
    src, exe = tmp_path / "t.cpp", str(tmp_path / "t")
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "badchimp-cpp_amd", "csrc"),
                    str(src), "-o", exe, "-ldl"], check=True, capture_output=True)
    out = subprocess.run([exe, str(threads)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith("bad 0"), out.stdout + out.stderr


WINDOWS = r'''
#include "rowbuild.hpp"
#include <cstdio>
#include <dlfcn.h>
#include <pthread.h>
static std::atomic<int> started{0};
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Create create = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
  ++started;
  return create(t, a, f, arg);
}
int main() {
  using namespace lbamd;
  const int32_t dims[3] = {96, 128, 128};  // 210 k words: more than one thread's share
  std::vector<int32_t> geo(96 * 128 * 128);
  for (size_t k = 0; k < geo.size(); ++k) geo[k] = k * 2654435761u >> 31;
  RowBuild rb;
  WinBuild own, many;
  std::string why;
  if (!rows_from_geometry(LB_D3Q19, dims, geo.data(), 1, rb, why)) return 2;
  started = 0;
  if (!build_windows(rb, false, own, why, false, false) || started != 0) return 3;
  if (!build_windows(rb, false, many, why) || (started == 0) != (host_threads() == 1)) return 4;
  return own.win != many.win || own.plane != many.plane || own.count != many.count;
}
'''


def test_windows_of_one_of_several_threads(tmp_path):
    src, exe = tmp_path / "w.hip", str(tmp_path / "w")
    src.write_text(WINDOWS)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "badchimp-cpp_amd", "csrc"), str(src), "-o", exe, "-ldl"], check=True,
                   capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr)
