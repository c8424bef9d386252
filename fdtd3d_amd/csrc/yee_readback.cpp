// Device-to-host copies of whole fields.
//
// hipMemcpy into ordinary memory passes through the runtime's own staging on one host thread,
// which also takes the page faults of a fresh array: 10.5 GB/s here (17 GB/s into touched pages)
// where the link gives 57 GB/s.  Large reads therefore go in chunks through pinned buffers, with
// several host threads copying (or widening) chunks to their place while the next ones arrive:
// the six fields of 512^3 FP32 (3.2 GB, fresh arrays) take 82 ms in place of 310.
#include "yee_readback.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace yee {

namespace {

// 16 buffers of 2 MiB: two for each of up to 8 threads.  A full chunk is 36 us of the link, long
// against the 5 us of queueing a copy and an event; a smaller field takes chunks of an eighth of
// itself, down to 256 KiB, so that the threads still share its page faults and its widening.
constexpr int64_t kChunk = 2 << 20;
constexpr int64_t kLeastChunk = 256 << 10;
constexpr int kThreads = 8;
// Below this one hipMemcpy is as fast (3.2 MB into pages in use: 175 us, 184 in chunks; 5.5 MB 304
// and 226; into fresh pages 3.2 MB 749 and 299).
constexpr int64_t kLeast = 3 << 20;
// Opening and closing the pool (pinning 32 MB, starting threads) costs 1 to 2.5 ms, chunks gain 25 us
// a MB in pages in use and 75 us in fresh ones.  So the first reads after the pool was closed are plain
// copies until this much has been read: a run that reads 8 MB once takes 0.47 ms of 1.37, one
// that reads 24 MB 1.4 of 3.9, and 48 MB at once take 4.2 ms through the pool, 4.6 plain.
constexpr int64_t kOpen = 48 << 20;

// Threads that wait for a read between reads (starting eight takes 100 us, as long as 1 MB takes
// to arrive on the plain path).
struct Pool
{
  std::vector<std::thread> threads;
  std::mutex mu;
  std::condition_variable wake, done;
  const std::function<void (int)> *job = nullptr;
  int round = 0, want = 0, left = 0;
  bool stop = false;

  // Up to n - 1 threads: where the process may start no more, run goes on with fewer.
  void start (int n)
  {
    stop = false;
    try
    {
      threads.reserve ((size_t) n);
      for (int t = 1; t < n; ++t) threads.emplace_back ([this, t, seen = round] { serve (t, seen); });
    }
    catch (const std::exception &)
    {
    }
  }

  void serve (int t, int seen)
  {
    std::unique_lock<std::mutex> lock (mu);
    for (;;)
    {
      wake.wait (lock, [&] { return stop || round != seen; });
      if (stop) return;
      seen = round;
      if (t >= want) continue;
      const std::function<void (int)> *f = job;
      lock.unlock ();
      (*f) (t);
      lock.lock ();
      if (--left == 0) done.notify_one ();
    }
  }

  // f (0) .. f (n - 1), f (0) on the calling thread; returns when all are done.
  void run (int n, const std::function<void (int)> &f)
  {
    n = std::min (n, (int) threads.size () + 1);
    {
      std::lock_guard<std::mutex> lock (mu);
      job = &f;
      want = n;
      left = n - 1;
      ++round;
    }
    wake.notify_all ();
    f (0);
    std::unique_lock<std::mutex> lock (mu);
    done.wait (lock, [&] { return left == 0; });
  }

  void join ()
  {
    {
      std::lock_guard<std::mutex> lock (mu);
      stop = true;
    }
    wake.notify_all ();
    for (std::thread &th : threads) th.join ();
    threads.clear ();
  }
};

// The current device of the thread is `device` while this lives.
struct OnDevice
{
  int before = -1;
  bool ok;
  explicit OnDevice (int device)
  {
    ok = hipGetDevice (&before) == hipSuccess && (before == device || hipSetDevice (device) == hipSuccess);
  }
  ~OnDevice ()
  {
    if (before >= 0) (void) hipSetDevice (before);
  }
};

struct Staging
{
  std::mutex mu;   // held by the one read that uses the buffers and threads
  char *buf = nullptr;
  int64_t plain = 0;   // bytes that plain copies of kLeast or more have put in place since the last close
  int device = -1;
  hipEvent_t ev[2 * kThreads] = {};
  Pool pool;

  // Whether a read that puts `bytes` in place goes through the buffers.
  bool wanted (int64_t bytes)
  {
    if (buf || plain + bytes >= kOpen) return true;
    plain += bytes;
    return false;
  }

  // Buffers, events and threads for reads on `dev`, the current device; false if they are another
  // device's or cannot be had (the next check of a launch must not find that error).
  bool open (int dev)
  {
    if (buf) return dev == device;
    bool ok = true;
    for (hipEvent_t &e : ev) ok = ok && (e || hipEventCreateWithFlags (&e, hipEventDisableTiming) == hipSuccess);
    if (!ok || hipHostMalloc ((void **) &buf, 2 * kThreads * kChunk, hipHostMallocDefault) != hipSuccess)
    {
      buf = nullptr;
      close ();   // (events made before the failure are of this device)
      (void) hipGetLastError ();
      return false;
    }
    device = dev;
    pool.start ((int) std::min<unsigned> (kThreads, std::max (2u, std::thread::hardware_concurrency ()) / 2));
    return true;
  }

  void close ()
  {
    pool.join ();
    plain = 0;
    if (buf) (void) hipHostFree (buf);
    buf = nullptr;
    for (hipEvent_t &e : ev)
    {
      if (e) (void) hipEventDestroy (e);
      e = nullptr;
    }
  }
};

// Never destroyed: a program may end with handles alive, whose threads end with it.
Staging &g_staging = *new Staging;
std::mutex g_refs_mu;
int g_refs = 0;

void place (char *out, const char *in, int64_t bytes, bool widen)
{
  if (!widen)
  {
    std::memcpy (out, in, (size_t) bytes);
    return;
  }
  const float *f = (const float *) in;
  double *d = (double *) out;
  for (int64_t q = 0; q < bytes / 4; ++q) d[q] = f[q];
}

}  // namespace

void readback_ref ()
{
  std::lock_guard<std::mutex> lock (g_refs_mu);
  ++g_refs;
}

void readback_unref ()
{
  std::lock_guard<std::mutex> lock (g_refs_mu);
  if (--g_refs > 0) return;
  std::lock_guard<std::mutex> use (g_staging.mu);
  g_staging.close ();
}

hipError_t read_back (int device, hipStream_t stream, const void *src, int64_t n, size_t wsize, void *out, bool widen)
{
  const int64_t bytes = n * (int64_t) wsize;
  const int64_t grow = widen ? 2 : 1;
  const OnDevice on (device);   // (the events and the stream must be of one device)
  if (!on.ok) return hipErrorInvalidDevice;
  std::unique_lock<std::mutex> use (g_staging.mu, std::try_to_lock);
  // small reads, the first ones, and reads while another thread holds the buffers: one plain copy
  if (bytes * grow < kLeast || !use.owns_lock () || !g_staging.wanted (bytes * grow) || !g_staging.open (device))
  {
    hipError_t e = hipStreamSynchronize (stream);
    if (e != hipSuccess || !widen) return e != hipSuccess ? e : hipMemcpy (out, src, (size_t) bytes, hipMemcpyDeviceToHost);
    std::vector<float> tmp ((size_t) n);
    e = hipMemcpy (tmp.data (), src, (size_t) bytes, hipMemcpyDeviceToHost);
    place ((char *) out, (const char *) tmp.data (), bytes, true);
    return e;
  }
  const int64_t eighth = ((bytes + kThreads - 1) / kThreads + 4095) & ~(int64_t) 4095;
  const int64_t chunk = std::max (kLeastChunk, std::min (kChunk, eighth));
  const int64_t chunks = (bytes + chunk - 1) / chunk;
  const int nthr = (int) std::min<int64_t> ((int64_t) g_staging.pool.threads.size () + 1, chunks);
  std::atomic<int> err { hipSuccess };
  // thread t takes chunks t, t + nthr, ...: it queues the copy of its next chunk into one of its two
  // buffers, then waits for the one before and puts it in place
  const std::function<void (int)> work = [&] (int t) {
    auto fail = [&] (hipError_t e) {
      if (e != hipSuccess) err = e;
      return e != hipSuccess;
    };
    if (t > 0 && fail (hipSetDevice (device))) return;
    auto queue = [&] (int64_t c, int slot) {
      const int64_t at = c * chunk, len = std::min (chunk, bytes - at);
      hipError_t e = hipMemcpyAsync (g_staging.buf + slot * kChunk, (const char *) src + at, (size_t) len,
                                     hipMemcpyDeviceToHost, stream);
      return e != hipSuccess ? e : hipEventRecord (g_staging.ev[slot], stream);
    };
    int k = 0;
    bool queued = !fail (queue (t, 2 * t));
    for (int64_t c = t; c < chunks && queued; c += nthr, k ^= 1)
    {
      const int slot = 2 * t + k;
      // (the other buffer's chunk was put in place in the round before)
      queued = c + nthr < chunks && !fail (queue (c + nthr, 2 * t + (k ^ 1)));
      if (fail (hipEventSynchronize (g_staging.ev[slot]))) break;
      const int64_t at = c * chunk, len = std::min (chunk, bytes - at);
      place ((char *) out + at * grow, g_staging.buf + slot * kChunk, len, widen);
    }
  };
  g_staging.pool.run (nthr, work);
  // after an error no copy into the buffers may still be in flight when they are used again
  if (err != hipSuccess) (void) hipStreamSynchronize (stream);
  return (hipError_t) err.load ();
}

}  // namespace yee
