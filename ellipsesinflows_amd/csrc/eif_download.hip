// Device arrays into the caller's (pageable) memory, through pinned staging
// that a device's contexts share.  A device-to-host copy into pageable memory
// goes through the runtime's bounce buffer with one host thread copying
// between the chunks, so the link idles while that thread copies and first
// touches the pages.  The fields into fresh numpy arrays, before and now:
// 128x128 (0.4 MB) 0.19 -> 0.05 ms, 512x1024 (12.6 MB) 2.2 -> 1.2 ms,
// 2048x4096 (201.6 MB) 20 -> 7.3 ms, of which the copies themselves take 6.4.
#include "eif_internal.hpp"
#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace eif {

// Each worker owns two slots of a chunk: one is filled by the device while
// the host copies the other out.  Downloads up to DL_SMALL take one slot and
// no thread.  Above, a worker for each DL_STRIP, up to DL_WORKERS: 201.6 MB
// take 16.2 ms with one, 7.3 with three and 7.1 with six (the link).
constexpr size_t DL_CHUNK = 1u << 20;
constexpr size_t DL_SMALL = 2 * DL_CHUNK;
constexpr size_t DL_STRIP = 4u << 20;
constexpr unsigned DL_WORKERS = 3;

// A device's sets of slots, each used by one download at a time.  Downloads of
// one thread do not overlap and share the first set; the others serve threads
// that download at the same time, also from one context, and a download that
// finds none free copies directly.  Made when first needed and given back with
// the device's last context.  With a set for each context the first downloads
// took 0.34 ms at 128x128 and 2.0 at 512x1024 (0.05 and 0.9 now), and every
// context held up to 6 MiB.
constexpr int DL_SETS = 4;
constexpr int DL_DEVICES = 64;

struct Staging {
  bool busy = false;
  unsigned workers = 0;  // of 2 slots each
  char *buf = nullptr;
  hipEvent_t ev[2 * DL_WORKERS] = {};
};

static std::mutex g_staging_mu;
static struct {
  int contexts = 0;
  Staging sets[DL_SETS];
} g_staging[DL_DEVICES];

// the calling thread on a device, its own again at the end
struct DeviceScope {
  int was = -1;
  hipError_t err;
  explicit DeviceScope(int device) {
    err = hipGetDevice(&was);
    if (err == hipSuccess && was != device)
      err = hipSetDevice(device);
    else
      was = -1;
  }
  ~DeviceScope() {
    if (was >= 0) (void)hipSetDevice(was);
  }
};

static void staging_drop(Staging *s) {
  if (s->buf) (void)hipHostFree(s->buf);
  s->buf = nullptr;
  for (auto &e : s->ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  s->workers = 0;
}

void staging_join(Ctx *c) {
  if (c->device < 0 || c->device >= DL_DEVICES) return;
  std::lock_guard<std::mutex> lk(g_staging_mu);
  g_staging[c->device].contexts++;
  c->staging = true;
}

void staging_leave(Ctx *c) {
  if (!c->staging) return;
  std::lock_guard<std::mutex> lk(g_staging_mu);
  c->staging = false;
  if (--g_staging[c->device].contexts > 0) return;
  for (auto &s : g_staging[c->device].sets) staging_drop(&s);
}

// a set for this many workers, held while this lives; null: none wanted (0) or
// none to be had
struct StagingUse {
  Staging *s = nullptr;
  StagingUse(Ctx *c, unsigned workers) {
    if (!c->staging || workers == 0) return;
    std::lock_guard<std::mutex> lk(g_staging_mu);
    for (auto &t : g_staging[c->device].sets)
      if (!t.busy) {
        if (t.workers >= workers || grow(&t, workers)) s = &t;
        break;
      }
    if (s) s->busy = true;
  }
  ~StagingUse() {
    if (!s) return;
    std::lock_guard<std::mutex> lk(g_staging_mu);
    s->busy = false;
  }
  StagingUse(const StagingUse &) = delete;

 private:
  static bool grow(Staging *t, unsigned workers) {
    staging_drop(t);
    hipError_t e = hipHostMalloc((void **)&t->buf, 2 * (size_t)workers * DL_CHUNK, 0);
    for (unsigned k = 0; e == hipSuccess && k < 2 * workers; k++)
      e = hipEventCreateWithFlags(&t->ev[k], hipEventDisableTiming);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      staging_drop(t);
      return false;
    }
    t->workers = workers;
    return true;
  }
};

// memory that the runtime knows (pinned, managed, device) is copied to directly
static bool known_to_runtime(const void *p) {
  hipPointerAttribute_t at;
  const hipError_t e = hipPointerGetAttributes(&at, p);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return at.type != hipMemoryTypeUnregistered;
}

// bytes [lo, hi) of the parts laid end to end, in chunks through slots k0 and k0 + 1
static hipError_t strip(Ctx *c, Staging *s, const Download *parts, int n, size_t lo, size_t hi,
                        unsigned k0) {
  hipError_t e = hipSuccess;
  struct {
    char *dst;
    size_t bytes;
  } job[2];
  unsigned queued = 0, taken = 0;  // chunks
  auto take = [&]() {
    const unsigned k = taken++ & 1;
    const hipError_t w = hipEventSynchronize(s->ev[k0 + k]);
    if (w == hipSuccess) memcpy(job[k].dst, s->buf + (k0 + k) * DL_CHUNK, job[k].bytes);
    return w;
  };
  size_t base = 0;
  for (int p = 0; p < n; p++) {
    const size_t end = base + parts[p].bytes;
    while (lo < std::min(hi, end)) {
      const unsigned k = queued & 1;
      if (queued - taken == 2 && (e = take()) != hipSuccess) return e;
      const size_t b = std::min(DL_CHUNK, std::min(hi, end) - lo);
      job[k].dst = (char *)parts[p].host + (lo - base);
      job[k].bytes = b;
      e = hipMemcpyAsync(s->buf + (k0 + k) * DL_CHUNK, (const char *)parts[p].dev + (lo - base), b,
                         hipMemcpyDeviceToHost, c->stream);
      if (e == hipSuccess) e = hipEventRecord(s->ev[k0 + k], c->stream);
      if (e != hipSuccess) return e;
      queued++;
      lo += b;
    }
    base = end;
  }
  while (taken < queued)
    if ((e = take()) != hipSuccess) return e;
  return hipSuccess;
}

// The parts with a host address, after the work queued on the context's
// stream; returns when they have arrived.
int download(Ctx *c, const Download *all, int n_all) {
  Download parts[DOWNLOAD_PARTS];
  int n = 0;
  size_t total = 0;
  bool direct = false;
  for (int k = 0; k < n_all; k++) {
    if (!all[k].host || !all[k].bytes) continue;
    direct = direct || known_to_runtime(all[k].host);
    total += all[k].bytes;
    parts[n++] = all[k];
  }
  const unsigned cpus = std::max(1u, std::thread::hardware_concurrency());
  const unsigned workers =
      (unsigned)std::min<size_t>(std::min(DL_WORKERS, cpus), std::max<size_t>(1, total / DL_STRIP));
  const DeviceScope on(c->device);
  EIF_HIP(on.err);
  const StagingUse use(c, direct ? 0 : workers);
  if (!use.s) {
    for (int k = 0; k < n; k++)
      EIF_HIP(hipMemcpyAsync(parts[k].host, parts[k].dev, parts[k].bytes, hipMemcpyDeviceToHost,
                             c->stream));
    EIF_HIP(hipStreamSynchronize(c->stream));
    return EIF_OK;
  }
  if (total <= DL_SMALL) {
    hipError_t e = hipSuccess;
    size_t off = 0;
    for (int k = 0; k < n && e == hipSuccess; k++) {
      e = hipMemcpyAsync(use.s->buf + off, parts[k].dev, parts[k].bytes, hipMemcpyDeviceToHost,
                         c->stream);
      off += parts[k].bytes;
    }
    const hipError_t w = hipStreamSynchronize(c->stream);  // no copy outlives the set's use
    EIF_HIP(e);
    EIF_HIP(w);
    off = 0;
    for (int k = 0; k < n; k++) {
      memcpy(parts[k].host, use.s->buf + off, parts[k].bytes);
      off += parts[k].bytes;
    }
    return EIF_OK;
  }
  // strips of whole 4 KiB; the calling thread takes the first, and those for
  // which no thread could be started
  const size_t step = (total / workers + 4095) / 4096 * 4096;
  hipError_t err[DL_WORKERS] = {};
  auto work = [&](unsigned w) {
    const DeviceScope mine(c->device);
    err[w] = mine.err;
    if (mine.err == hipSuccess)
      err[w] = strip(c, use.s, parts, n, w * step,
                     w + 1 == workers ? total : std::min(total, (w + 1) * step), 2 * w);
  };
  std::thread th[DL_WORKERS];
  unsigned started = 1;
  try {
    for (; started < workers; started++) th[started] = std::thread(work, started);
  } catch (const std::exception &) {
  }
  work(0);
  for (unsigned w = started; w < workers; w++) work(w);
  for (unsigned w = 1; w < started; w++) th[w].join();
  hipError_t e = hipSuccess;
  for (unsigned w = 0; w < workers; w++)
    if (e == hipSuccess) e = err[w];
  // a strip that failed may have left copies into its slots behind
  if (e != hipSuccess) (void)hipStreamSynchronize(c->stream);
  EIF_HIP(e);
  EIF_HIP(hipStreamSynchronize(c->stream));
  return EIF_OK;
}

int download(Ctx *c, void *host, const void *dev, size_t bytes) {
  if (!host) EIF_HIP(hipErrorInvalidValue);
  const Download d = {host, dev, bytes};
  return download(c, &d, 1);
}

}  // namespace eif
