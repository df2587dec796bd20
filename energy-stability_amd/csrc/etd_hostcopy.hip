// etd_hostcopy.hip -- fields between the host's pageable memory (FP64) and
// the device (FP64 or FP32).
//
// A copy to or from pageable memory goes through the runtime's pinned buffer
// on one thread: 17 GB/s for the 60 MB of an FP64 field at n = 196, and for
// FP32 storage a second pass on that thread converts, into pages that are
// fresh each time.  Here a field passes through three pinned slots: the
// calling thread keeps the copies going, and it and up to HC_THREADS - 1
// others convert (or copy) pieces of the chunks that have arrived.
// A piece goes to whoever is free and nobody waits for a thread that has not
// begun: after a caller's OpenMP region its threads hold every CPU for a
// while, a new thread then starts 3 to 4 ms late, and the calling thread does
// the work alone.  A helper that lost its CPU in the middle of a piece is
// waited for.
// Measured, median of one field read (set) in ms, the runtime's pageable copy
// (and, for FP32, a conversion through the heap) against this: FP64 n = 148 1.46
// (0.69) -> 0.68 (0.67), 196 3.5 (2.05) -> 1.41 (1.46), 260 8.0 (4.7) -> 3.1
// (3.2); FP32 148 1.30 (1.14) -> 0.38 (0.39), 196 3.5 (2.9) -> 0.75 (0.79), 260
// 21.8 (16.7) -> 1.60 (1.72); n = 36 FP32 21 to 90 -> 20 us.  After an OpenMP
// region: FP64 196 3.55 (2.0) -> 3.57 (1.6), 260 8.1 (4.7) -> 6.0 (3.55, but one
// copy in ten 6.5 to 10), FP32 196 7.7 (2.85) -> 1.33 (1.84), 260 29.6 (17) -> 2.7
// (3.6).  Chunks: a copy costs about 13 us
// besides its bytes, so 512 KiB pieces reach 21 GB/s, 4 MiB 43 GB/s; more
// than 4 threads add nothing.
#include <hip/hip_runtime.h>
#include <emmintrin.h>
#include <pthread.h>
#include <signal.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <new>
#include <utility>

#include "etd_internal.h"

#define HC_THREADS 4
#define HC_CHUNK ((size_t)4 << 20)   // most device bytes per slot
#define HC_SHARE ((size_t)8 << 20)   // host bytes that pay for one more thread (from two on)
#define HC_SLOTS 3
#define HC_PIECES 8                  // of a chunk, for the threads
#define HC_MIN ((size_t)64 << 10)    // least device bytes per slot
// FP64 fields up to this: the runtime's own path (n = 68, read 147 us there,
// 142 here, set 100 and 128; n = 84 read 273 and 222, set 148 and 190; n = 100
// set 236 and 258, n = 132 set 506 and 490)
#define HC_DIRECT_GET ((size_t)3 << 20)
#define HC_DIRECT_PUT ((size_t)8 << 20)
// FP32 fields up to this: one copy through one slot, no events (read, two
// chunks against one slot: n = 36 39 and 20 us, n = 52 49 and 35, n = 68 71 and
// 66, n = 84 108 and 125; a temporary on the heap, as before the slots, 21 to
// 90, 43, 104, 195)
#define HC_ONE ((size_t)2 << 20)
// and set, up to this: one call from the stack (through a slot n = 8 15.7, n = 12
// 15.9 us, so 13.1 and 13.5; copying from pinned memory is quicker from 32 KB on)
#define HC_SMALL ((size_t)8 << 10)

// host FP64 values from device ones, past the cache for long runs
static void widen(double *dst, const double *src, size_t cnt) { memcpy(dst, src, sizeof(double) * cnt); }
static void widen(double *dst, const float *src, size_t cnt) {
  size_t i = 0;
  if (cnt >= 32768 && ((uintptr_t)dst & 7) == 0) {
    if ((uintptr_t)dst & 15) {
      dst[0] = src[0];
      i = 1;
    }
    for (; i + 4 <= cnt; i += 4) {
      const __m128 v = _mm_loadu_ps(src + i);
      _mm_stream_pd(dst + i, _mm_cvtps_pd(v));
      _mm_stream_pd(dst + i + 2, _mm_cvtps_pd(_mm_movehl_ps(v, v)));
    }
    _mm_sfence();
  }
  for (; i < cnt; i++) dst[i] = src[i];
}
static void narrow(double *dst, const double *src, size_t cnt) { memcpy(dst, src, sizeof(double) * cnt); }
static void narrow(float *dst, const double *src, size_t cnt) {
  for (size_t i = 0; i < cnt; i++) dst[i] = (float)src[i];
}

template <typename T>
struct hc_job {
  etd_ctx *c;
  T *dev;
  double *host;
  size_t cnt, per;  // elements in all, per chunk
  size_t nch;       // chunks
  int put;
  // the host side: pieces of the chunks below ready go to whoever takes the
  // next one; done counts the finished ones of each slot
  size_t pc;   // elements per piece, HC_PIECES of them per chunk
  std::atomic<size_t> ready, next, done[HC_SLOTS];
  std::atomic<int> refs;  // who still looks at this record

  void *pin;        // HC_SLOTS chunks

  T *slot(size_t k) const { return (T *)pin + (k % HC_SLOTS) * per; }
  size_t len(size_t k) const { return (k + 1) * per <= cnt ? per : cnt - k * per; }
  // elements [a, b) of chunk k between its slot and the host
  void part(size_t k, size_t a, size_t b) const {
    if (put) narrow(slot(k) + a, host + k * per + a, b - a);
    else widen(host + k * per + a, slot(k) + a, b - a);
  }
  hipError_t start(size_t k) const {
    const size_t b = sizeof(T) * len(k);
    hipError_t e = put ? hipMemcpyAsync(dev + k * per, slot(k), b, hipMemcpyHostToDevice, c->stream)
                       : hipMemcpyAsync(slot(k), dev + k * per, b, hipMemcpyDeviceToHost, c->stream);
    return e != hipSuccess ? e : hipEventRecord(c->io_ev[k % HC_SLOTS], c->stream);
  }
  hipError_t wait(size_t k) const { return hipEventSynchronize(c->io_ev[k % HC_SLOTS]); }
};

template <typename T>
static bool hc_take(hc_job<T> *j) {
  size_t i = j->next.load(std::memory_order_relaxed);
  do {
    if (i >= j->ready.load(std::memory_order_acquire) * HC_PIECES) return false;
  } while (!j->next.compare_exchange_weak(i, i + 1, std::memory_order_relaxed));
  const size_t k = i / HC_PIECES, n = j->len(k), a = i % HC_PIECES * j->pc, b = a + j->pc < n ? a + j->pc : n;
  if (b > a) j->part(k, a, b);
  j->done[k % HC_SLOTS].fetch_add(1, std::memory_order_release);
  return true;
}
// the helper threads of all calls, HC_LIVE at most (four copies at a time get
// all three of theirs, later ones do with fewer).  A place is taken by one call (HC_CLAIMED), its
// thread made and finished; then the next call that takes it, or the last
// context to close, joins the thread: the library may be unloaded after that.
#define HC_LIVE 12
#define HC_MADE 1
#define HC_FINISHED 2
#define HC_CLAIMED 4
static struct hc_place {
  pthread_t th;
  std::atomic<int> st;
  void *job;
} hc_at[HC_LIVE];

template <typename T>
static void hc_drop(hc_job<T> *j) {
  if (j->refs.fetch_sub(1, std::memory_order_acq_rel) == 1) delete j;
}
// a worker makes no HIP call (a thread's first one costs a few hundred
// microseconds); one that comes after the last piece finds nothing to take
template <typename T>
static void *hc_thread(void *p) {
  hc_place *const at = (hc_place *)p;
  hc_job<T> *j = (hc_job<T> *)at->job;
  while (j->next.load(std::memory_order_relaxed) < j->nch * HC_PIECES)
    if (!hc_take(j)) _mm_pause();
  hc_drop(j);
  at->st.fetch_or(HC_FINISHED, std::memory_order_release);
  return nullptr;
}
template <typename T>
static bool hc_worker(hc_job<T> *j) {
  for (hc_place &at : hc_at) {
    int st = at.st.load(std::memory_order_acquire);
    if ((st != 0 && st != (HC_MADE | HC_FINISHED)) ||
        !at.st.compare_exchange_strong(st, HC_CLAIMED, std::memory_order_acquire))
      continue;
    if (st) (void)pthread_join(at.th, nullptr);
    at.job = j;
    j->refs.fetch_add(1, std::memory_order_relaxed);
    const bool ok = !pthread_create(&at.th, nullptr, hc_thread<T>, &at);
    if (!ok) j->refs.fetch_sub(1, std::memory_order_relaxed);
    at.st.fetch_xor(ok ? HC_CLAIMED | HC_MADE : HC_CLAIMED, std::memory_order_release);
    return ok;
  }
  return false;
}

// the calling thread: copies and events, and pieces while it waits for them
template <typename T>
static hipError_t hc_run(hc_job<T> *j) {
  hipError_t e = hipSuccess;
  auto finished = [&](size_t k) {
    while (j->done[k % HC_SLOTS].load(std::memory_order_acquire) < (k / HC_SLOTS + 1) * HC_PIECES)
      if (!hc_take(j)) _mm_pause();
  };
  if (j->put) {
    for (size_t k = 0; k <= j->nch; k++) {
      if (k < j->nch) {
        if (k >= HC_SLOTS && (e = j->wait(k - HC_SLOTS)) != hipSuccess) return e;
        j->ready.store(k + 1, std::memory_order_release);
      }
      if (k == 0) continue;
      finished(k - 1);
      if ((e = j->start(k - 1)) != hipSuccess) return e;
    }
    return e;
  }
  for (size_t k = 0; k < j->nch && k < HC_SLOTS; k++)
    if ((e = j->start(k)) != hipSuccess) return e;
  for (size_t k = 0; k < j->nch; k++) {
    if ((e = j->wait(k)) != hipSuccess) return e;
    j->ready.store(k + 1, std::memory_order_release);
    if (k == 0 || k - 1 + HC_SLOTS >= j->nch) continue;
    finished(k - 1);
    if ((e = j->start(k - 1 + HC_SLOTS)) != hipSuccess) return e;
  }
  if (j->nch) finished(j->nch - 1);
  return e;
}

// Pinned memory for a call's slots.  It is taken for the call and given back
// after it (a copy is over when it returns), so contexts share it: allocating
// it per context cost an ensemble of 20 a millisecond each.  At most
// HC_POOL buffers wait between calls, one for each copy that has all its
// helpers (HC_LIVE / 3), 12 MiB each at most; the last context to close frees
// them.
#define HC_POOL 4
static std::mutex pool_mu;
static struct {
  void *p;
  size_t bytes;
} pool_buf[HC_POOL];
static int pool_n, pool_users;

static void *pool_take(size_t need, size_t *bytes) {
  {
    std::lock_guard<std::mutex> l(pool_mu);
    for (int i = 0; i < pool_n; i++)
      if (pool_buf[i].bytes >= need) {
        void *p = pool_buf[i].p;
        *bytes = pool_buf[i].bytes;
        pool_buf[i] = pool_buf[--pool_n];
        return p;
      }
  }
  void *p = nullptr;
  if (hipHostMalloc(&p, need, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  *bytes = need;
  return p;
}
static void pool_give(void *p, size_t bytes) {
  if (!p) return;
  {
    std::lock_guard<std::mutex> l(pool_mu);
    if (pool_users > 0) {
      if (pool_n < HC_POOL) {
        pool_buf[pool_n++] = {p, bytes};
        return;
      }
      for (int i = 0; i < pool_n; i++)  // full: the larger one stays
        if (pool_buf[i].bytes < bytes) {
          std::swap(pool_buf[i].p, p);
          std::swap(pool_buf[i].bytes, bytes);
        }
    }
  }
  (void)hipHostFree(p);
}
void host_copy_open(void) {
  std::lock_guard<std::mutex> l(pool_mu);
  pool_users++;
}
void host_copy_close(etd_ctx *c) {
  for (int i = 0; i < c->io_nev; i++) (void)hipEventDestroy(c->io_ev[i]);
  std::lock_guard<std::mutex> l(pool_mu);
  if (--pool_users == 0) {
    for (hc_place &at : hc_at)
      if (at.st.load(std::memory_order_acquire) & HC_MADE) {
        (void)pthread_join(at.th, nullptr);
        at.st.store(0, std::memory_order_relaxed);
      }
    while (pool_n) (void)hipHostFree(pool_buf[--pool_n].p);
  }
}

// the slots' events; 0 when they cannot be had.  An event belongs to the
// device that is current when it is made, and the calling thread may have
// another one than the context's.
static int hc_events(etd_ctx *c) {
  if (c->io_nev == HC_SLOTS) return 1;
  int cur = c->device;
  hipError_t e = hipGetDevice(&cur);
  if (e == hipSuccess && cur != c->device) e = hipSetDevice(c->device);
  for (; e == hipSuccess && c->io_nev < HC_SLOTS; c->io_nev += e == hipSuccess)
    e = hipEventCreateWithFlags(&c->io_ev[c->io_nev], hipEventDisableTiming);
  if (cur != c->device) (void)hipSetDevice(cur);
  if (e != hipSuccess) (void)hipGetLastError();
  return e == hipSuccess;
}

// one copy: FP64 directly, FP32 through one slot, or the heap where pinned
// memory cannot be had
static hipError_t hc_one(etd_ctx *c, double *dev, double *host, size_t cnt, int put) {
  hipError_t e = put ? hipMemcpyAsync(dev, host, sizeof(double) * cnt, hipMemcpyHostToDevice, c->stream)
                     : hipMemcpyAsync(host, dev, sizeof(double) * cnt, hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  return e;
}
static hipError_t hc_one(etd_ctx *c, float *dev, double *host, size_t cnt, int put) {
  if (put && sizeof(float) * cnt <= HC_SMALL) {
    float t[HC_SMALL / sizeof(float)];
    narrow(t, host, cnt);
    return hipMemcpyWithStream(dev, t, sizeof(float) * cnt, hipMemcpyHostToDevice, c->stream);
  }
  size_t pinned = 0;
  float *pin = (float *)pool_take(sizeof(float) * cnt, &pinned), *t = pin;
  if (!t && !(t = (float *)malloc(sizeof(float) * cnt))) return hipErrorOutOfMemory;
  hipError_t e = hipSuccess;
  if (put) {
    narrow(t, host, cnt);
    e = hipMemcpyAsync(dev, t, sizeof(float) * cnt, hipMemcpyHostToDevice, c->stream);
  } else {
    e = hipMemcpyAsync(t, dev, sizeof(float) * cnt, hipMemcpyDeviceToHost, c->stream);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  if (e == hipSuccess && !put) widen(host, t, cnt);
  if (pin) pool_give(pin, pinned);
  else free(t);
  return e;
}

// whether the runtime can copy to and from p itself: pinned memory.  One such
// FP64 copy runs at the rate of the bus (n = 196 1.06 ms, through the slots
// 1.4; n = 260 2.46 and 3.1).
static bool hc_pinned(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

template <typename T>
hipError_t host_copy(etd_ctx *c, T *dev, double *host, size_t cnt, int put) {
  const size_t bytes = sizeof(T) * cnt;
  if (bytes <= (sizeof(T) == 4 ? HC_ONE : put ? HC_DIRECT_PUT : HC_DIRECT_GET) || (sizeof(T) == 8 && hc_pinned(host)))
    return hc_one(c, dev, host, cnt, put);
  // a quarter of the field per chunk, at most HC_CHUNK, in whole 4 KiB; half
  // of it up to 4 MiB (quarters that short took 430 us from the device at
  // 1 MiB, halves 70 us)
  size_t per = (bytes / (bytes <= HC_CHUNK ? 2 : 4) + 4095) / 4096 * 4096;
  per = per < HC_MIN ? HC_MIN : per > HC_CHUNK ? HC_CHUNK : per;
  const size_t nch = (bytes + per - 1) / per;
  size_t pinned = 0;
  void *pin = hc_events(c) ? pool_take((nch < HC_SLOTS ? nch : HC_SLOTS) * per, &pinned) : nullptr;
  if (!pin) return hc_one(c, dev, host, cnt, put);
  hc_job<T> *const j = new (std::nothrow) hc_job<T>;
  if (!j) {
    pool_give(pin, pinned);
    return hc_one(c, dev, host, cnt, put);
  }
  j->pin = pin;
  j->c = c;
  j->dev = dev;
  j->host = host;
  j->cnt = cnt;
  j->per = per / sizeof(T);
  j->nch = nch;
  j->put = put;
  j->pc = (j->per / HC_PIECES + 8) & ~(size_t)7;  // whole cache lines of the host buffer
  j->ready = 0;
  j->next = 0;
  for (int t = 0; t < HC_SLOTS; t++) j->done[t] = 0;
  j->refs = 1;
  int want = (int)(sizeof(double) * cnt / HC_SHARE) - 1;  // the calling thread is one
  want = want > HC_THREADS - 1 ? HC_THREADS - 1 : want;
  if (want > 0) {
    // the process's signals stay with its own threads: a helper inherits a mask that blocks them all
    sigset_t all, old;
    sigfillset(&all);
    const int masked = !pthread_sigmask(SIG_SETMASK, &all, &old);
    while (want > 0 && masked && hc_worker(j)) want--;  // fewer threads, or none, do as well
    if (masked) (void)pthread_sigmask(SIG_SETMASK, &old, nullptr);
  }
  hipError_t e = hc_run(j);
  // no piece is given out any more (after an error some are left); those that
  // were are done before the buffers are anyone else's
  size_t taken = j->next.exchange(nch * HC_PIECES), got;
  do {
    got = 0;
    for (int t = 0; t < HC_SLOTS; t++) got += j->done[t].load(std::memory_order_acquire);
  } while (got < taken);
  hc_drop(j);
  // the slots are free, and what was put is on the device, after this
  const hipError_t es = hipStreamSynchronize(c->stream);
  pool_give(pin, pinned);
  return e != hipSuccess ? e : es;
}
template hipError_t host_copy<double>(etd_ctx *, double *, double *, size_t, int);
template hipError_t host_copy<float>(etd_ctx *, float *, double *, size_t, int);
