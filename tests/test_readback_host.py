"""The chunked device-to-host read (yee_readback.cpp) built for the host against a small stand-in of
the HIP calls it makes, which keeps device memory in host memory and can be told to fail: what it
does when threads or pinned memory cannot be had is not a matter of the GPU.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "fdtd3d_amd", "csrc")

HIP = r"""
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>
typedef int hipError_t;
typedef struct stream { int device; } *hipStream_t;
typedef struct event { int device; } *hipEvent_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101, hipErrorInvalidHandle = 400 };
enum { hipMemcpyDeviceToHost, hipEventDisableTiming, hipHostMallocDefault };
inline thread_local int cur_dev = 0;
inline thread_local hipError_t last = hipSuccess;
inline bool no_pinned = false;
inline std::atomic<int> pinned { 0 };
inline hipError_t ret (hipError_t e) { return e ? last = e : e; }
inline hipError_t hipGetLastError () { hipError_t e = last; last = hipSuccess; return e; }
inline hipError_t hipSetDevice (int d) { cur_dev = d; return hipSuccess; }
inline hipError_t hipGetDevice (int *d) { *d = cur_dev; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags (hipEvent_t *e, int) { *e = new event { cur_dev }; return hipSuccess; }
inline hipError_t hipEventDestroy (hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventSynchronize (hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord (hipEvent_t e, hipStream_t s) { return ret (e->device == s->device ? hipSuccess : hipErrorInvalidHandle); }
inline hipError_t hipStreamSynchronize (hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpy (void *d, const void *s, size_t n, int) { std::memcpy (d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync (void *d, const void *s, size_t n, int, hipStream_t) { std::memcpy (d, s, n); return hipSuccess; }
inline hipError_t hipHostMalloc (void **p, size_t n, int)
{
  if (no_pinned) return ret (hipErrorOutOfMemory);
  ++pinned;
  *p = std::malloc (n);
  return hipSuccess;
}
inline hipError_t hipHostFree (void *p) { --pinned; std::free (p); return hipSuccess; }
"""

MAIN = r"""
#include <hip/hip_runtime.h>
#include "yee_readback.h"
#include <cerrno>
#include <cstdint>
#include <cstdio>
#include <dlfcn.h>
#include <pthread.h>
#include <string>
#include <vector>

// threads that may still start (negative: any number)
static int threads_left = -1, threads_started = 0;
extern "C" int pthread_create (pthread_t *t, const pthread_attr_t *a, void *(*f) (void *), void *x)
{
  typedef int (*fn) (pthread_t *, const pthread_attr_t *, void *(*) (void *), void *);
  static fn real = (fn) dlsym (RTLD_NEXT, "pthread_create");
  if (threads_left == 0) return EAGAIN;
  if (threads_left > 0) --threads_left;
  ++threads_started;
  return real (t, a, f, x);
}

// Reads n FP32 values of a ramp on device `dev`, as they are and widened; 0 if both are right.
static int read_ramp (int dev, int64_t n)
{
  stream st { dev };
  std::vector<float> src ((size_t) n), raw ((size_t) n, -1.0f);
  std::vector<double> wide ((size_t) n, -1.0);
  for (int64_t q = 0; q < n; ++q) src[(size_t) q] = (float) (q % 16777216);
  if (yee::read_back (dev, &st, src.data (), n, 4, raw.data (), false) != hipSuccess) return 1;
  if (yee::read_back (dev, &st, src.data (), n, 4, wide.data (), true) != hipSuccess) return 2;
  for (int64_t q = 0; q < n; ++q)
    if (raw[(size_t) q] != src[(size_t) q] || wide[(size_t) q] != (double) src[(size_t) q]) return 3;
  return 0;
}

#define CHECK(x) do { if (!(x)) { std::printf ("failed: %s\n", #x); return 1; } } while (0)

int main (int argc, char **argv)
{
  const std::string what = argc > 1 ? argv[1] : "";
  const int64_t large = 16 << 20;   // 64 MB of FP32
  yee::readback_ref ();
  if (what == "threads")
  {
    threads_left = std::atoi (argv[2]);
    CHECK (read_ramp (0, large + 3) == 0);
    threads_left = -1;
    CHECK (read_ramp (0, large + 3) == 0);
  }
  else if (what == "pinned")
  {
    no_pinned = true;
    CHECK (read_ramp (0, large + 3) == 0);
    CHECK (hipGetLastError () == hipSuccess);
  }
  else if (what == "device")
  {
    hipSetDevice (1);   // another one than the handle's
    CHECK (read_ramp (0, large + 3) == 0);
    CHECK (cur_dev == 1);
    CHECK (hipGetLastError () == hipSuccess);
  }
  else if (what == "few")
  {
    // 4 MB and 8 MB of output a call: the fourth reaches 48
    for (int k = 0; k < 3; ++k)
    {
      CHECK (read_ramp (0, 1 << 20) == 0);
      CHECK (pinned == 0 && threads_started == 0);
    }
    CHECK (read_ramp (0, 1 << 20) == 0);
    CHECK (pinned == 1 && threads_started > 0);
    yee::readback_unref ();
    CHECK (pinned == 0);
    yee::readback_ref ();
    CHECK (read_ramp (0, 1 << 20) == 0);   // counted from the start again
    CHECK (pinned == 0);
    CHECK (read_ramp (0, large) == 0);     // one large read is enough
    CHECK (pinned == 1);
  }
  else CHECK (!"a known case");
  yee::readback_unref ();
  CHECK (pinned == 0);
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("readback")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "main.cpp").write_text(MAIN)
    exe = d / "readback"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(d), "-I", CSRC, str(d / "main.cpp"),
                    os.path.join(CSRC, "yee_readback.cpp"), "-o", str(exe), "-ldl"], check=True)
    return str(exe)


def run(program, *args):
    r = subprocess.run([program, *args], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


@pytest.mark.parametrize("allowed", [0, 1, 2])
def test_read_with_fewer_threads_than_asked_for(program, allowed):
    """std::thread throws where the process may start no more threads: the read goes on with those
    that started, none at worst, and leaves no exception for a C caller."""
    run(program, "threads", str(allowed))


def test_no_error_left_where_pinned_memory_cannot_be_had(program):
    """The read then takes plain copies, and the error of the attempt is not left for the next
    check of a kernel launch."""
    run(program, "pinned")


def test_handle_of_another_device_than_the_current_one(program):
    """The events belong to the handle's device, as its stream does, and the caller's current
    device stays as it was."""
    run(program, "device")


def test_a_few_small_reads_open_no_pool(program):
    """Pinned buffers and threads cost more than they gain until 48 MB have been read: a run that
    reads a few small fields takes plain copies."""
    run(program, "few")
