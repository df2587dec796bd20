// The field copies (csrc/etd_hostcopy.hip) on the CPU: the source itself with
// the few HIP calls that it makes replaced by a model of the runtime.  Device
// memory is host memory; copies and events run only when something waits for
// them, in stream order, so a slot that is read or reused too early shows.
// An event must be of the device of the stream that it is recorded on.
#include <stdio.h>
#include <string.h>

#include <deque>
#include <map>
#include <random>
#include <string>
#include <thread>
#include <vector>

#include <signal.h>

// the thread calls of the copies are looked at on the way
static int model_create(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
#include <pthread.h>
static int model_join(pthread_t, void **);
#define pthread_create model_create
#define pthread_join model_join
#include "etd_hostcopy.hip"
#undef pthread_create
#undef pthread_join

static int cur_dev;
struct op {
  void *to;
  const void *from;
  size_t bytes;
  hipEvent_t ev;
};
static std::deque<op> queue;          // of the one stream
static const int stream_dev = 1;
static std::map<hipEvent_t, int> event_dev;
static int copies, mallocs;
static const void *copied_host;       // the host side of the last copy

static void run_until(hipEvent_t ev) {
  while (!queue.empty()) {
    const op o = queue.front();
    queue.pop_front();
    if (o.bytes) memcpy(o.to, o.from, o.bytes);
    if (ev && o.ev == ev) return;
  }
}
hipError_t hipGetDevice(int *d) {
  *d = cur_dev;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  cur_dev = d;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind kind, hipStream_t) {
  queue.push_back({to, from, bytes, nullptr});
  copies++;
  copied_host = kind == hipMemcpyHostToDevice ? from : to;
  return hipSuccess;
}
hipError_t hipMemcpyWithStream(void *to, const void *from, size_t bytes, hipMemcpyKind, hipStream_t) {
  run_until(nullptr);
  memcpy(to, from, bytes);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = (hipEvent_t) new int;
  event_dev[*e] = cur_dev;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  event_dev.erase(e);
  delete (int *)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  if (event_dev.at(e) != stream_dev) return hipErrorInvalidHandle;
  queue.push_back({nullptr, nullptr, 0, e});
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  run_until(e);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  run_until(nullptr);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
  mallocs++;
  *p = malloc(bytes);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
  free(p);
  return hipSuccess;
}
static const char *known, *known_end;  // host memory that the runtime has pinned
static int unknown_is_error;           // what a query of other memory gives: an error, or a type of its own
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  const bool k = (const char *)p >= known && (const char *)p < known_end;
  if (!k && unknown_is_error) return hipErrorInvalidValue;
  a->type = k ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }

// helper threads: made, joined, and those that a signal could run on
static std::atomic<int> made, joined, unblocked;
struct entry {
  void *(*f)(void *);
  void *arg;
};
static void *enter(void *p) {
  const entry e = *(entry *)p;
  delete (entry *)p;
  sigset_t now;
  pthread_sigmask(SIG_SETMASK, nullptr, &now);
  if (!sigismember(&now, SIGINT) || !sigismember(&now, SIGALRM) || !sigismember(&now, SIGUSR1)) unblocked++;
  return e.f(e.arg);
}
static int model_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
  made++;
  return pthread_create(t, a, enter, new entry{f, arg});
}
static int model_join(pthread_t t, void **r) {
  joined++;
  return pthread_join(t, r);
}

#define CHECK(x)                                       \
  do {                                                 \
    if (!(x)) {                                        \
      printf("line %d: %s\n", __LINE__, #x);           \
      exit(1);                                         \
    }                                                  \
  } while (0)

struct context {
  etd_ctx c = {};
  explicit context(int dev = stream_dev) {
    c.device = stream_dev;
    cur_dev = dev;
    host_copy_open();
  }
  ~context() { host_copy_close(&c); }
};

template <typename T>
static void trip(context &x, size_t cnt, size_t offset) {
  std::mt19937_64 r(cnt + offset);
  std::vector<char> a(8 * cnt + 64), b(8 * cnt + 64);
  std::vector<T> dev(cnt);
  double *from = (double *)(a.data() + offset), *to = (double *)(b.data() + offset);
  for (size_t i = 0; i < cnt; i++) {
    const double v = (double)(int64_t)r() * 0x1p-40;
    memcpy(from + i, &v, 8);
  }
  CHECK(host_copy<T>(&x.c, dev.data(), from, cnt, 1) == hipSuccess && queue.empty());
  CHECK(host_copy<T>(&x.c, dev.data(), to, cnt, 0) == hipSuccess && queue.empty());
  for (size_t i = 0; i < cnt; i++) {
    double u, v;
    memcpy(&u, from + i, 8);
    memcpy(&v, to + i, 8);
    CHECK((double)(T)u == v);
  }
}
// fields of n^3: one copy, two chunks, four chunks and more, none to three helper threads, a short last chunk
static void trips() {
  context x;
  for (size_t n : {1, 8, 12, 13, 68, 84, 104, 132, 148, 164, 197}) {
    trip<double>(x, n * n * n, 0);
    trip<float>(x, n * n * n, 8);
  }
  trip<float>(x, 84 * 84 * 84, 0);
}
// the calling thread's device is another than the context's
static void device() {
  context x(0);
  trip<double>(x, 148 * 148 * 148, 0);
  trip<float>(x, 148 * 148 * 148, 0);
  CHECK(cur_dev == 0);
}
// a buffer that is pinned already is copied to and from as it is; other memory goes through the slots, as ever
static void pinned() {
  context x;
  const size_t cnt = 148 * 148 * 148;
  std::vector<double> host(cnt, 1.5), dev(cnt);
  for (int put = 0; put < 2; put++)
    for (unknown_is_error = 0; unknown_is_error < 2; unknown_is_error++) {
      known = (const char *)host.data(), known_end = known + 8 * cnt;
      copies = mallocs = 0;
      CHECK(host_copy<double>(&x.c, dev.data(), host.data(), cnt, put) == hipSuccess && queue.empty());
      CHECK(copies == 1 && copied_host == host.data() && mallocs == 0);
      known = known_end = nullptr;
      CHECK(host_copy<double>(&x.c, dev.data(), host.data(), cnt, put) == hipSuccess && queue.empty());
      CHECK(copies > 2);
    }
}
// the process's signals stay with its own threads
static void signals() {
  context x;
  sigset_t before, after;
  pthread_sigmask(SIG_SETMASK, nullptr, &before);
  trip<double>(x, 164 * 164 * 164, 0);
  trip<float>(x, 164 * 164 * 164, 0);
  pthread_sigmask(SIG_SETMASK, nullptr, &after);
  CHECK(made > 0 && sigismember(&after, SIGINT) == sigismember(&before, SIGINT));
}
// no helper is left, not even in its last instructions, when the last context
// has closed: the library may be unloaded then.  Several threads copy at once.
static void threads() {
  context x;
  std::vector<std::thread> th;
  for (int t = 0; t < 4; t++)
    th.emplace_back([t] {
      for (int k = 0; k < 3; k++) {
        std::vector<float> buf(148 * 148 * 148);
        hc_job<float> *j = new hc_job<float>;
        j->c = nullptr, j->dev = nullptr, j->host = nullptr, j->put = 0;
        j->cnt = buf.size(), j->per = buf.size(), j->nch = 1, j->pc = buf.size() / HC_PIECES, j->pin = buf.data();
        std::vector<double> out(buf.size());
        j->host = out.data();
        j->ready = 1, j->next = 0, j->refs = 1;
        for (auto &d : j->done) d = 0;
        for (int w = 0; w < 3; w++) hc_worker(j);
        while (hc_take(j)) {}
        while (j->done[0] < HC_PIECES) _mm_pause();
        hc_drop(j);
      }
    });
  for (auto &t : th) t.join();
}

int main(int, char **argv) {
  const std::map<std::string, void (*)()> what = {{"trips", trips}, {"device", device}, {"pinned", pinned},
                                                     {"signals", signals}, {"threads", threads}};
  what.at(argv[1])();
  CHECK(event_dev.empty());
  CHECK(argv[1] != std::string("threads") || (made > 3 && joined == made));
  CHECK(argv[1] != std::string("signals") || unblocked == 0);
  puts("ok");
  return 0;
}
