// yk_runtime.hip -- device context of the library: one HIP stream (default
// priority), error reporting, allocation, padded copies, stream timing.
#include <hip/hip_runtime.h>
#include <pthread.h>
#include <sched.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>
#include <sys/stat.h>
#include <atomic>

#include "yk.h"
#include "yk_dev.h"

static __thread char g_err[512];
static hipStream_t g_stream = nullptr;
static int g_ready = 0;
static pthread_mutex_t g_init_mu = PTHREAD_MUTEX_INITIALIZER;
static pthread_mutex_t g_lib_mu = PTHREAD_RECURSIVE_MUTEX_INITIALIZER_NP;

void yk_lock(void) { pthread_mutex_lock(&g_lib_mu); }
void yk_unlock(void) { pthread_mutex_unlock(&g_lib_mu); }
static hipEvent_t g_t0 = nullptr, g_t1 = nullptr;

int yk_set_error(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int yk_hip_fail(hipError_t e, const char *what) {
  // the error is reported here; HIP's copy of it is consumed so that a later
  // hipGetLastError check does not report it again from an unrelated call
  (void)hipGetLastError();
  return yk_set_error(e == hipErrorOutOfMemory ? YK_ENOMEM : YK_EHIP, "%s: %s", what,
                      hipGetErrorString(e));
}

extern "C" const char *yk_last_error(void) { return g_err; }

extern "C" int yk_set_error_c(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

hipStream_t yk_stream(void) { return g_stream; }

// Work-item tickets of the persistent scans: per-XCD counters, zeroed in
// stream order before each launch that uses them.  A static device array,
// so that taking them allocates nothing (its address is resolved once, at
// initialisation).
static __device__ __align__(256) int yk_tick_store[64];
static int *g_tick = nullptr;

__global__ void yk_tick_zero_kernel(int *t) { t[threadIdx.x] = 0; }

int yk_item_tickets(int **out) {
  hipLaunchKernelGGL(yk_tick_zero_kernel, dim3(1), dim3(64), 0, g_stream, g_tick);
  YK_HIP(hipGetLastError());
  *out = g_tick;
  return YK_OK;
}

extern "C" int yk_init(void) {
  if (g_ready) return YK_OK;
  pthread_mutex_lock(&g_init_mu);
  int rc = YK_OK;
  if (!g_ready) {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n < 1) {
      rc = yk_set_error(YK_ENODEV, "no GPU visible to HIP (%s)",
                        e == hipSuccess ? "0 devices" : hipGetErrorString(e));
    } else if ((e = hipSetDevice(0)) != hipSuccess) {
      rc = yk_hip_fail(e, "hipSetDevice");
    } else if ((e = hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking)) != hipSuccess) {
      rc = yk_hip_fail(e, "hipStreamCreate");
    } else if ((e = hipEventCreate(&g_t0)) != hipSuccess ||
               (e = hipEventCreate(&g_t1)) != hipSuccess) {
      rc = yk_hip_fail(e, "hipEventCreate");
    } else if ((e = hipGetSymbolAddress((void **)&g_tick, HIP_SYMBOL(yk_tick_store))) !=
               hipSuccess) {
      rc = yk_hip_fail(e, "hipGetSymbolAddress(item tickets)");
    } else {
      rc = yk_prof_setup();
      if (rc == YK_OK) g_ready = 1;
    }
  }
  pthread_mutex_unlock(&g_init_mu);
  return rc;
}

extern "C" int yk_ld(int d) { return (d + 15) & ~15; }

extern "C" int yk_malloc(void **p, size_t bytes) {
  YK_TRY(yk_init());
  *p = nullptr;
  if (bytes == 0) bytes = 256;
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) return yk_hip_fail(e, "hipMalloc");
  return YK_OK;
}

extern "C" int yk_free(void *p) {
  if (!p) return YK_OK;
  hipError_t e = hipFree(p);
  if (e != hipSuccess) return yk_hip_fail(e, "hipFree");
  return YK_OK;
}

extern "C" int yk_memcpy_h2d(void *dst, const void *src, size_t bytes) {
  YK_TRY(yk_init());
  if (!bytes) return YK_OK;
  YK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_stream));
  YK_HIP(hipStreamSynchronize(g_stream));
  return YK_OK;
}

extern "C" int yk_host_alloc(void **p, size_t bytes) {
  YK_TRY(yk_init());
  *p = nullptr;
  // coherent and mapped: kernels may also write it directly
  if (hipHostMalloc(p, bytes ? bytes : 1, hipHostMallocCoherent | hipHostMallocMapped) !=
      hipSuccess) {
    (void)hipGetLastError();
    return yk_set_error(YK_ENOMEM, "hipHostMalloc(%zu) failed", bytes);
  }
  return YK_OK;
}

extern "C" int yk_host_free(void *p) {
  if (p) YK_HIP(hipHostFree(p));
  return YK_OK;
}

// largest readback through the pinned landing buffer of yk_read_small (one
// memcpy of it costs less than the second wait of a pageable copy)
#define YK_READ_SMALL ((size_t)256 << 10)
// smallest copies through the staging threads: down 4 MB (17 GB/s plain, 22
// staged; 32 MB 17 and 38), up 16 MB (37 and 43; plain is ahead below)
#define YK_STAGE_MIN_DOWN ((size_t)4 << 20)
#define YK_STAGE_MIN_UP ((size_t)16 << 20)
static int yk_copy_staged_up(char *dev, const char *host, size_t bytes);
static int yk_copy_staged_down(char *host, const char *dev, size_t bytes);

// Memory at p that HIP knows (pinned or mapped host memory, or a device's): the
// DMA reaches it by itself, and a detour through the pinned buffers only costs
// a host copy (to pinned memory, plain and staged: 4 MB 0.082 and 0.154 ms, 32
// MB 0.60 and 0.80; 256 KB through the landing buffer 0.019 instead of 0.013).
static bool yk_known_to_hip(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();  // consumed: ordinary host memory
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

extern "C" int yk_memcpy_d2h(void *dst, const void *src, size_t bytes) {
  YK_TRY(yk_init());
  if (!bytes) return YK_OK;
  if (bytes <= 256 || (bytes <= YK_READ_SMALL && !yk_known_to_hip(dst)))
    return yk_read_small(dst, src, bytes);
  if (bytes >= YK_STAGE_MIN_DOWN && !yk_known_to_hip(dst))
    return yk_copy_staged_down((char *)dst, (const char *)src, bytes);
  YK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_stream));
  YK_HIP(hipStreamSynchronize(g_stream));
  return YK_OK;
}

// A few device values (flags, counters, a small call's results) read back
// with one wait: the copy lands in a pinned buffer behind the queued work.  A
// copy into pageable memory instead waits for the stream, then goes through a
// bounce buffer with a wait of its own.
int yk_read_small(void *dst, const void *src, size_t bytes) {
  static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
  static void *buf = nullptr;
  if (bytes > YK_READ_SMALL)
    return yk_set_error(YK_EINVAL, "yk_read_small: %zu bytes > %zu", bytes, YK_READ_SMALL);
  pthread_mutex_lock(&mu);
  hipError_t e = hipSuccess;
  if (!buf) e = hipHostMalloc(&buf, YK_READ_SMALL, hipHostMallocDefault);
  if (e == hipSuccess) e = hipMemcpyAsync(buf, src, bytes, hipMemcpyDeviceToHost, g_stream);
  if (e == hipSuccess) e = hipStreamSynchronize(g_stream);
  if (e == hipSuccess) memcpy(dst, buf, bytes);
  pthread_mutex_unlock(&mu);
  return e == hipSuccess ? YK_OK : yk_hip_fail(e, "small readback");
}

extern "C" int yk_memcpy_d2d(void *dst, const void *src, size_t bytes) {
  YK_TRY(yk_init());
  if (!bytes) return YK_OK;
  YK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, g_stream));
  return YK_OK;
}

// plain 16-byte-per-lane copy: the reference point for HBM traffic counters
__global__ void yk_copy16_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

extern "C" int yk_copy_kernel(void *dst, const void *src, size_t bytes) {
  YK_TRY(yk_init());
  if (bytes % 16) return yk_set_error(YK_EINVAL, "yk_copy_kernel: size %zu not a multiple of 16", bytes);
  if (!bytes) return YK_OK;
  hipLaunchKernelGGL(yk_copy16_kernel, dim3(4096), dim3(256), 0, g_stream, (const uint4 *)src,
                     (uint4 *)dst, bytes / 16);
  YK_HIP(hipGetLastError());
  return YK_OK;
}

__global__ void yk_fill_u32_kernel(uint32_t *p, uint32_t v, size_t n) {
  size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

// Byte fill done by a kernel (never a memset node), multiple of 4 bytes.
extern "C" int yk_memset(void *dst, int value, size_t bytes) {
  YK_TRY(yk_init());
  if (!bytes) return YK_OK;
  if (bytes % 4) return yk_set_error(YK_EINVAL, "yk_memset: size %zu not a multiple of 4", bytes);
  uint32_t b = (uint32_t)(value & 0xff);
  uint32_t v = b | (b << 8) | (b << 16) | (b << 24);
  size_t n = bytes / 4;
  int blocks = (int)((n + 255) / 256);
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(yk_fill_u32_kernel, dim3(blocks), dim3(256), 0, g_stream,
                     (uint32_t *)dst, v, n);
  YK_HIP(hipGetLastError());
  return YK_OK;
}

extern "C" int yk_sync(void) {
  YK_TRY(yk_init());
  YK_HIP(hipStreamSynchronize(g_stream));
  return YK_OK;
}

// Copies of YK_STAGE_MIN_* bytes and more from and to pageable host memory go
// through pinned buffers, the host copies of up to YK_STAGE_THREADS threads
// overlapping the DMAs.  (A plain copy to pageable memory goes in 1 MB pieces,
// 20 us on the bus and ~70 us between them.  256 MB: 17 GB/s plain, 51 with four
// threads, 42 with eight.)  The pinned buffers (64 MB in all) are allocated at
// the first such copy and kept until the process ends; a mutex keeps one staged
// copy at a time.
#define YK_STAGE_THREADS 4
#define YK_STAGE_SLICE ((size_t)2 << 20)  // one thread per so many bytes
#define YK_STAGE_BYTES ((size_t)8 << 20)
#define YK_STAGE_BUFS (2 * YK_STAGE_THREADS)
static pthread_mutex_t g_stage_mu = PTHREAD_MUTEX_INITIALIZER;
static void *g_stage_buf[YK_STAGE_BUFS];
static hipEvent_t g_stage_ev[YK_STAGE_BUFS];
static hipStream_t g_stage_st[YK_STAGE_THREADS];  // up
static int g_stage_ready = 0;

static int yk_stage_setup(bool up) {
  for (int t = 0; up && t < YK_STAGE_THREADS; t++)
    if (!g_stage_st[t]) YK_HIP(hipStreamCreateWithFlags(&g_stage_st[t], hipStreamNonBlocking));
  if (g_stage_ready) return YK_OK;
  for (int b = 0; b < YK_STAGE_BUFS; b++) {
    YK_HIP(hipHostMalloc(&g_stage_buf[b], YK_STAGE_BYTES, hipHostMallocDefault));
    YK_HIP(hipEventCreateWithFlags(&g_stage_ev[b], hipEventDisableTiming));
  }
  g_stage_ready = 1;
  return YK_OK;
}

// job(t) on `ways` threads, the caller's among them; where one cannot start,
// the caller does its job too
static void yk_stage_threads(void *(*fn)(void *), char *jobs, size_t job_bytes, int ways) {
  pthread_t th[YK_STAGE_THREADS];
  bool started[YK_STAGE_THREADS] = {false};
  for (int t = 1; t < ways; t++)
    started[t] = pthread_create(&th[t], nullptr, fn, jobs + t * job_bytes) == 0;
  fn(jobs);
  for (int t = 1; t < ways; t++) {
    if (started[t])
      pthread_join(th[t], nullptr);
    else
      fn(jobs + t * job_bytes);
  }
}

static int yk_stage_ways(size_t bytes) {
  const size_t w = bytes / YK_STAGE_SLICE;
  return w < 1 ? 1 : w > YK_STAGE_THREADS ? YK_STAGE_THREADS : (int)w;
}

// Up: each thread pushes a contiguous slice through two buffers on a stream of
// its own (default priority; 512 MB 9.9 ms, on one stream 10.7).
struct YkStageUp {
  char *dev;
  const char *host;
  size_t bytes;
  int t;
  hipError_t err;
};

static void *yk_stage_up_worker(void *arg) {
  YkStageUp *j = (YkStageUp *)arg;
  hipStream_t st = g_stage_st[j->t];
  // two pieces of a slice or more, so that the buffers overlap
  size_t piece = (j->bytes / 2 + 4095) & ~(size_t)4095;
  if (piece > YK_STAGE_BYTES) piece = YK_STAGE_BYTES;
  bool pend[2] = {false, false};
  size_t off = 0;
  for (int b = 0; off < j->bytes && j->err == hipSuccess; b ^= 1) {
    const size_t n = j->bytes - off < piece ? j->bytes - off : piece;
    const int slot = 2 * j->t + b;
    hipError_t e = pend[b] ? hipEventSynchronize(g_stage_ev[slot]) : hipSuccess;
    if (e == hipSuccess) {
      memcpy(g_stage_buf[slot], j->host + off, n);
      e = hipMemcpyAsync(j->dev + off, g_stage_buf[slot], n, hipMemcpyHostToDevice, st);
    }
    if (e == hipSuccess) e = hipEventRecord(g_stage_ev[slot], st);
    j->err = e;
    pend[b] = true;
    off += n;
  }
  const hipError_t e = hipStreamSynchronize(st);
  if (j->err == hipSuccess) j->err = e;
  return nullptr;
}

static int yk_copy_staged_up(char *dev, const char *host, size_t bytes) {
  YK_HIP(hipStreamSynchronize(g_stream));  // earlier work on the device memory
  pthread_mutex_lock(&g_stage_mu);
  int rc = yk_stage_setup(true);
  if (rc == YK_OK) {
    const size_t per = (bytes / yk_stage_ways(bytes) + 4095) & ~(size_t)4095;
    YkStageUp job[YK_STAGE_THREADS];
    int nt = 0;
    for (size_t o = 0; nt < YK_STAGE_THREADS && o < bytes; o += per, nt++)
      job[nt] = {dev + o, host + o, bytes - o < per ? bytes - o : per, nt, hipSuccess};
    yk_stage_threads(yk_stage_up_worker, (char *)job, sizeof job[0], nt);
    for (int t = 0; t < nt && rc == YK_OK; t++)
      if (job[t].err != hipSuccess) rc = yk_hip_fail(job[t].err, "staged copy");
  }
  pthread_mutex_unlock(&g_stage_mu);
  return rc;
}

// Down: pieces come one after the other on the library's stream, and the
// threads share each piece's host copy.  (After copies on several streams the
// allocations of a later call take longer: two k-means training calls in a row,
// 16 sub-spaces of 94,555 points, d = 24, k = 93, 3.1 against 2.6 ms a call.  A
// piece costs ~9 us besides its bytes, hence few and large ones.  8 MB 0.25 ms,
// 48 MB 1.09, 512 MB 10.5; a slice for each thread on the one stream 0.32, 1.33
// and 10.7, on four streams 0.25, 1.30 and 10.1.)
struct YkStageDown {
  const char *dev;
  char *host;
  size_t bytes, piece;
  long npiece;
  int ways;
  std::atomic<long> next;                // (piece, part) to copy, in order
  std::atomic<long> at[YK_STAGE_BUFS];   // the piece that a buffer holds or waits for
  std::atomic<int> left[YK_STAGE_BUFS];  // its parts not yet copied
  std::atomic<int> err;
};

static void yk_stage_down_queue(YkStageDown *j, long c) {
  const int slot = (int)(c % YK_STAGE_BUFS);
  const size_t off = (size_t)c * j->piece;
  const size_t n = j->bytes - off < j->piece ? j->bytes - off : j->piece;
  hipError_t e =
      hipMemcpyAsync(g_stage_buf[slot], j->dev + off, n, hipMemcpyDeviceToHost, g_stream);
  if (e == hipSuccess) e = hipEventRecord(g_stage_ev[slot], g_stream);
  if (e != hipSuccess) {
    j->err.store(e);
    return;
  }
  j->left[slot].store(j->ways, std::memory_order_relaxed);
  j->at[slot].store(c, std::memory_order_release);
}

static void *yk_stage_down_worker(void *arg) {
  YkStageDown *j = *(YkStageDown **)arg;
  for (;;) {
    const long u = j->next.fetch_add(1), c = u / j->ways;
    if (c >= j->npiece) break;
    const int slot = (int)(c % YK_STAGE_BUFS);
    // (queued by whoever ends the buffer's last piece, all of whose parts were
    // taken before this one)
    while (j->at[slot].load(std::memory_order_acquire) != c) {
      if (j->err.load()) return nullptr;
      sched_yield();
    }
    const hipError_t e = hipEventSynchronize(g_stage_ev[slot]);
    if (e != hipSuccess) {
      j->err.store(e);
      return nullptr;
    }
    const size_t off = (size_t)c * j->piece;
    const size_t n = j->bytes - off < j->piece ? j->bytes - off : j->piece;
    const size_t per = (n / j->ways + 64) & ~(size_t)63, o = per * (u % j->ways);
    if (o < n)
      memcpy(j->host + off + o, (const char *)g_stage_buf[slot] + o, n - o < per ? n - o : per);
    if (j->left[slot].fetch_sub(1) == 1 && c + YK_STAGE_BUFS < j->npiece)
      yk_stage_down_queue(j, c + YK_STAGE_BUFS);
  }
  return nullptr;
}

static int yk_copy_staged_down(char *host, const char *dev, size_t bytes) {
  pthread_mutex_lock(&g_stage_mu);
  int rc = yk_stage_setup(false);
  if (rc == YK_OK) {
    YkStageDown j;
    j.dev = dev;
    j.host = host;
    j.bytes = bytes;
    // quarters: an eighth at a time 8 MB take 0.29 ms, from 32 MB on the same
    j.piece = (bytes / 4 + 4095) & ~(size_t)4095;
    if (j.piece > YK_STAGE_BYTES) j.piece = YK_STAGE_BYTES;
    j.npiece = (long)((bytes + j.piece - 1) / j.piece);
    j.ways = yk_stage_ways(bytes);
    j.next.store(0);
    j.err.store(0);
    for (auto &a : j.at) a.store(-1);
    for (long c = 0; c < j.npiece && c < YK_STAGE_BUFS && !j.err.load(); c++)
      yk_stage_down_queue(&j, c);
    YkStageDown *job[YK_STAGE_THREADS] = {&j, &j, &j, &j};
    yk_stage_threads(yk_stage_down_worker, (char *)job, sizeof job[0], j.ways);
    if (j.err.load()) {
      (void)hipStreamSynchronize(g_stream);  // nothing is left in flight
      rc = yk_hip_fail((hipError_t)j.err.load(), "staged copy");
    }
  }
  pthread_mutex_unlock(&g_stage_mu);
  return rc;
}

// Rows of d floats, dense on the host, and of ld on the device: the dense
// bytes cross the bus in one copy per YK_DENSE_BYTES, a kernel spreads or
// collects the rows.  (A 2-D copy of pageable memory goes row by row: 19.0 ms
// for a search of 9 queries in 2,055 vectors, d = 157, now 0.157 ms; the
// kernel itself is bound by HBM.)  The dense buffer is kept between calls.
#define YK_DENSE_BYTES ((size_t)64 << 20)
static pthread_mutex_t g_dense_mu = PTHREAD_MUTEX_INITIALIZER;
static float *g_dense = nullptr;
static size_t g_dense_bytes = 0;

__global__ __launch_bounds__(256) void yk_spread_rows_kernel(const float *__restrict__ src, long n,
                                                             int d, int ld4,
                                                             float4 *__restrict__ dst) {
  const long t = blockIdx.x * 256L + threadIdx.x;
  if (t >= n * ld4) return;
  const long row = t / ld4;
  const int c = (int)(t - row * ld4) * 4;
  const float *p = src + row * d + c;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);  // pad columns zero
  if (c < d) v.x = p[0];
  if (c + 1 < d) v.y = p[1];
  if (c + 2 < d) v.z = p[2];
  if (c + 3 < d) v.w = p[3];
  dst[t] = v;
}

__global__ __launch_bounds__(256) void yk_collect_rows_kernel(const float *__restrict__ src, long n,
                                                              int d, int ld,
                                                              float *__restrict__ dst) {
  const long t = blockIdx.x * 256L + threadIdx.x;
  if (t >= n * d) return;
  const long row = t / d;
  dst[t] = src[row * ld + (t - row * d)];
}

// under g_dense_mu
static int yk_dense_buffer(size_t bytes, float **out) {
  if (bytes > g_dense_bytes) {
    if (g_dense) YK_HIP(hipFree(g_dense));
    g_dense = nullptr;
    g_dense_bytes = 0;
    YK_HIP(hipMalloc((void **)&g_dense, bytes));
    g_dense_bytes = bytes;
  }
  *out = g_dense;
  return YK_OK;
}

// the rows by one 2-D copy: to pinned memory (256 KB 0.012 ms, in two steps
// 0.029; 32 MB 0.55 and 0.67), and where no dense buffer is to be had
static int yk_copy_2d(float *dev, float *host, long n, int d, bool up) {
  const size_t dev_row = sizeof(float) * (size_t)yk_ld(d), row = sizeof(float) * (size_t)d;
  if (up) {
    YK_TRY(yk_memset(dev, 0, dev_row * (size_t)n));
    YK_HIP(hipMemcpy2DAsync(dev, dev_row, host, row, row, n, hipMemcpyHostToDevice, g_stream));
  } else {
    YK_HIP(hipMemcpy2DAsync(host, row, dev, dev_row, row, n, hipMemcpyDeviceToHost, g_stream));
  }
  YK_HIP(hipStreamSynchronize(g_stream));
  return YK_OK;
}

static int yk_dense_copy(float *dev, float *host, long n, int d, bool up) {
  const int ld = yk_ld(d);
  const bool known = yk_known_to_hip(host);
  if (known && !up) return yk_copy_2d(dev, host, n, d, false);
  const size_t row = sizeof(float) * (size_t)d;
  long step = (long)(YK_DENSE_BYTES / row);  // rows per copy
  if (step < 1) step = 1;
  if (step > n) step = n;
  float *buf;
  if (yk_dense_buffer(row * (size_t)step, &buf) != YK_OK) return yk_copy_2d(dev, host, n, d, up);
  for (long i = 0; i < n; i += step) {
    const long m = n - i < step ? n - i : step;
    const size_t bytes = row * (size_t)m;
    if (!up) {
      const long t = m * d;
      hipLaunchKernelGGL(yk_collect_rows_kernel, dim3((unsigned)((t + 255) / 256)), dim3(256), 0,
                         g_stream, dev + i * ld, m, d, ld, buf);
      YK_HIP(hipGetLastError());
      YK_TRY(yk_memcpy_d2h(host + i * d, buf, bytes));
      continue;
    }
    if (bytes >= YK_STAGE_MIN_UP && !known)
      YK_TRY(yk_copy_staged_up((char *)buf, (const char *)(host + i * d), bytes));
    else
      YK_HIP(hipMemcpyAsync(buf, host + i * d, bytes, hipMemcpyHostToDevice, g_stream));
    const long t = m * (ld / 4);
    hipLaunchKernelGGL(yk_spread_rows_kernel, dim3((unsigned)((t + 255) / 256)), dim3(256), 0,
                       g_stream, buf, m, d, ld / 4, (float4 *)(dev + i * ld));
    YK_HIP(hipGetLastError());
  }
  // the buffer is free for the next caller, the data complete
  YK_HIP(hipStreamSynchronize(g_stream));
  return YK_OK;
}

// host n x d (dense) -> device n x ld (pad columns zeroed)
extern "C" int yk_upload_vectors(float *dst, const float *src, long n, int d) {
  YK_TRY(yk_init());
  if (n <= 0) return YK_OK;
  const size_t bytes = sizeof(float) * (size_t)n * d;
  if (yk_ld(d) != d) {
    pthread_mutex_lock(&g_dense_mu);
    const int rc = yk_dense_copy(dst, (float *)src, n, d, true);
    pthread_mutex_unlock(&g_dense_mu);
    return rc;
  }
  if (bytes >= YK_STAGE_MIN_UP && !yk_known_to_hip(src))
    return yk_copy_staged_up((char *)dst, (const char *)src, bytes);
  YK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_stream));
  YK_HIP(hipStreamSynchronize(g_stream));
  return YK_OK;
}

extern "C" int yk_copy_cols(float *dst, int ldd, const float *src, int lds, long n, int ncols) {
  YK_TRY(yk_init());
  if (n <= 0 || ncols <= 0) return YK_OK;
  if (ncols > ldd || ncols > lds) return yk_set_error(YK_EINVAL, "yk_copy_cols: ncols > stride");
  YK_HIP(hipMemcpy2DAsync(dst, sizeof(float) * ldd, src, sizeof(float) * lds,
                          sizeof(float) * ncols, n, hipMemcpyDeviceToDevice, g_stream));
  return YK_OK;
}

extern "C" int yk_download_vectors(float *dst, const float *src, long n, int d) {
  YK_TRY(yk_init());
  if (n <= 0) return YK_OK;
  if (yk_ld(d) == d) return yk_memcpy_d2h(dst, src, sizeof(float) * (size_t)n * d);
  pthread_mutex_lock(&g_dense_mu);
  const int rc = yk_dense_copy((float *)src, dst, n, d, false);
  pthread_mutex_unlock(&g_dense_mu);
  return rc;
}

extern "C" int yk_timer_start(void) {
  YK_TRY(yk_init());
  YK_HIP(hipEventRecord(g_t0, g_stream));
  return YK_OK;
}

extern "C" int yk_timer_stop(float *ms) {
  YK_HIP(hipEventRecord(g_t1, g_stream));
  YK_HIP(hipEventSynchronize(g_t1));
  YK_HIP(hipEventElapsedTime(ms, g_t0, g_t1));
  return YK_OK;
}

extern "C" int yk_device_info(char *buf, int len) {
  YK_TRY(yk_init());
  hipDeviceProp_t p;
  YK_HIP(hipGetDeviceProperties(&p, 0));
  snprintf(buf, len, "%s gcn=%s cus=%d lds/block=%zu clock_khz=%d mem=%zuMiB", p.name,
           p.gcnArchName, p.multiProcessorCount, (size_t)p.sharedMemPerBlock, p.clockRate,
           (size_t)(p.totalGlobalMem >> 20));
  return YK_OK;
}

// ---------------------------------------------------------------------------
// per-kernel event timing (used by the benchmark to time the dominant kernel
// on the stream it runs on)

#define YK_PROF_SLOTS 16
#define YK_PROF_EV 4096
static int g_prof_on = 0;
static hipEvent_t g_pev[YK_PROF_EV][2];
static int g_pev_n = 0;
static int g_pev_slot[YK_PROF_EV];
static double g_prof_ms[YK_PROF_SLOTS];
static long g_prof_cnt[YK_PROF_SLOTS];

int yk_prof_setup(void) {
  for (int i = 0; i < YK_PROF_EV; i++) {
    hipError_t e = hipEventCreate(&g_pev[i][0]);
    if (e == hipSuccess) e = hipEventCreate(&g_pev[i][1]);
    if (e != hipSuccess) return yk_hip_fail(e, "hipEventCreate(prof)");
  }
  return YK_OK;
}

static void yk_prof_flush(void) {
  for (int i = 0; i < g_pev_n; i++) {
    float ms = 0;
    // a pair whose events failed is left out of the sums, and its error is
    // consumed here (HIP keeps the last error for the next hipGetLastError,
    // which would otherwise report it from an unrelated launch)
    if (hipEventSynchronize(g_pev[i][1]) == hipSuccess &&
        hipEventElapsedTime(&ms, g_pev[i][0], g_pev[i][1]) == hipSuccess) {
      g_prof_ms[g_pev_slot[i]] += ms;
      g_prof_cnt[g_pev_slot[i]]++;
    } else {
      (void)hipGetLastError();
    }
  }
  g_pev_n = 0;
}

int yk_prof_begin(int slot) {
  if (!g_prof_on) return -1;
  // no timing inside a stream capture: the records would become nodes of
  // the captured graph, never completed as ordinary events
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(g_stream, &cs) != hipSuccess) {
    (void)hipGetLastError();  // consumed: the launch goes ahead untimed
    return -1;
  }
  if (cs != hipStreamCaptureStatusNone) return -1;
  if (g_pev_n == YK_PROF_EV) yk_prof_flush();
  const int i = g_pev_n;
  if (hipEventRecord(g_pev[i][0], g_stream) != hipSuccess) {
    (void)hipGetLastError();  // consumed: the launch goes ahead untimed
    return -1;
  }
  g_pev_slot[i] = slot;
  g_pev_n++;
  return i;
}

void yk_prof_end(int tok) {
  if (tok < 0) return;
  // a failed record leaves the pair unfinished: yk_prof_flush skips it
  if (hipEventRecord(g_pev[tok][1], g_stream) != hipSuccess) (void)hipGetLastError();
}

extern "C" int yk_prof_enable(int on) {
  YK_TRY(yk_init());
  g_prof_on = on;
  return YK_OK;
}

extern "C" int yk_prof_reset(void) {
  YK_TRY(yk_init());
  YK_HIP(hipStreamSynchronize(g_stream));
  g_pev_n = 0;
  memset(g_prof_ms, 0, sizeof(g_prof_ms));
  memset(g_prof_cnt, 0, sizeof(g_prof_cnt));
  return YK_OK;
}

extern "C" int yk_prof_get(int which, double *total_ms, long *count) {
  if (which < 0 || which >= YK_PROF_SLOTS) return yk_set_error(YK_EINVAL, "prof slot");
  YK_HIP(hipStreamSynchronize(g_stream));
  yk_prof_flush();
  *total_ms = g_prof_ms[which];
  *count = g_prof_cnt[which];
  return YK_OK;
}

// ---------------------------------------------------------------------------
// persistent-grid sizing

#define YK_OCC_CACHE 256
static const void *g_occ_fn[YK_OCC_CACHE];
static int g_occ_block[YK_OCC_CACHE], g_occ_val[YK_OCC_CACHE], g_occ_n = 0;  // val: per CU
static int g_cu_count = 0;
static pthread_mutex_t g_occ_mu = PTHREAD_MUTEX_INITIALIZER;

int yk_resident_wgs(const void *fn, int block, int most) {
  pthread_mutex_lock(&g_occ_mu);
  int per_cu = 0;
  for (int i = 0; i < g_occ_n; i++)
    if (g_occ_fn[i] == fn && g_occ_block[i] == block) per_cu = g_occ_val[i];
  if (!per_cu) {
    if (!g_cu_count) {
      hipDeviceProp_t p;
      if (hipGetDeviceProperties(&p, 0) == hipSuccess) {
        g_cu_count = p.multiProcessorCount;
      } else {
        (void)hipGetLastError();  // consumed: the grid is sized for 256 CUs instead
        g_cu_count = 256;
      }
    }
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, block, 0) != hipSuccess) {
      (void)hipGetLastError();  // consumed: one workgroup per CU is assumed instead
      per_cu = 1;
    }
    if (per_cu < 1) per_cu = 1;
    if (g_occ_n < YK_OCC_CACHE) {
      g_occ_fn[g_occ_n] = fn;
      g_occ_block[g_occ_n] = block;
      g_occ_val[g_occ_n++] = per_cu;
    }
  }
  const int res = (most > 0 && per_cu > most ? most : per_cu) * g_cu_count;
  pthread_mutex_unlock(&g_occ_mu);
  return res < 8 ? 8 : res & ~7;
}

// ---------------------------------------------------------------------------
// autotuning cache: "key value" lines in a text file
// ($YAEL_MI355X_TUNE_CACHE, default ~/.cache/yael_mi355x_tune.txt), read
// once per process into memory; later lines of a key win.  Every choice it
// holds is a launch plan whose results are the same bits whichever plan
// runs (a schedule, never an arithmetic), so a stale or foreign file can
// only cost time.

#define YK_TUNE_MAX 512
static char g_tune_key[YK_TUNE_MAX][128];
static int g_tune_val[YK_TUNE_MAX];
static int g_tune_n = 0, g_tune_loaded = 0;
static pthread_mutex_t g_tune_mu = PTHREAD_MUTEX_INITIALIZER;

static const char *yk_tune_path(char *buf, size_t len) {
  const char *e = getenv("YAEL_MI355X_TUNE_CACHE");
  if (e && *e) return e;
  const char *home = getenv("HOME");
  snprintf(buf, len, "%s/.cache/yael_mi355x_tune.txt", home ? home : "/tmp");
  return buf;
}

static void yk_tune_set_locked(const char *key, int val) {
  for (int i = 0; i < g_tune_n; i++)
    if (!strcmp(g_tune_key[i], key)) {
      g_tune_val[i] = val;
      return;
    }
  if (g_tune_n == YK_TUNE_MAX) return;
  snprintf(g_tune_key[g_tune_n], sizeof g_tune_key[0], "%s", key);
  g_tune_val[g_tune_n++] = val;
}

static void yk_tune_load_locked(void) {
  if (g_tune_loaded) return;
  g_tune_loaded = 1;
  char pbuf[512];
  FILE *f = fopen(yk_tune_path(pbuf, sizeof pbuf), "r");
  if (!f) return;
  char k[128];
  int v;
  while (fscanf(f, "%127s %d", k, &v) == 2) yk_tune_set_locked(k, v);
  fclose(f);
}

extern "C" int yk_tune_get(const char *key, int *val) {
  pthread_mutex_lock(&g_tune_mu);
  yk_tune_load_locked();
  int found = 0;
  for (int i = 0; i < g_tune_n && !found; i++)
    if (!strcmp(g_tune_key[i], key)) {
      *val = g_tune_val[i];
      found = 1;
    }
  pthread_mutex_unlock(&g_tune_mu);
  return found;
}

extern "C" void yk_tune_put(const char *key, int val) {
  pthread_mutex_lock(&g_tune_mu);
  yk_tune_load_locked();
  yk_tune_set_locked(key, val);
  char pbuf[512];
  const char *path = yk_tune_path(pbuf, sizeof pbuf);
  char dir[512];
  snprintf(dir, sizeof dir, "%s", path);
  char *slash = strrchr(dir, '/');
  if (slash && slash != dir) {
    *slash = 0;
    mkdir(dir, 0755);  // one level (~/.cache); best effort
  }
  FILE *f = fopen(path, "a");
  if (f) {
    fprintf(f, "%s %d\n", key, val);
    fclose(f);
  }
  pthread_mutex_unlock(&g_tune_mu);
}

// 0 when YAEL_MI355X_TUNE=0: every search then runs its default plan
extern "C" int yk_tune_enabled(void) {
  const char *e = getenv("YAEL_MI355X_TUNE");
  return !(e && e[0] == '0');
}

// Milliseconds of run() on the library stream, between two events.
int yk_time_ms(int (*run)(void *), void *arg, float *ms) {
  YK_TRY(yk_init());
  hipEvent_t e0, e1;
  YK_HIP(hipEventCreate(&e0));
  hipError_t e = hipEventCreate(&e1);
  if (e != hipSuccess) {
    (void)hipEventDestroy(e0);
    return yk_hip_fail(e, "hipEventCreate");
  }
  int rc = YK_OK;
  if ((e = hipEventRecord(e0, g_stream)) != hipSuccess) rc = yk_hip_fail(e, "hipEventRecord");
  if (rc == YK_OK) rc = run(arg);
  if (rc == YK_OK && (e = hipEventRecord(e1, g_stream)) != hipSuccess)
    rc = yk_hip_fail(e, "hipEventRecord");
  if (rc == YK_OK && (e = hipEventSynchronize(e1)) != hipSuccess)
    rc = yk_hip_fail(e, "hipEventSynchronize");
  if (rc == YK_OK && (e = hipEventElapsedTime(ms, e0, e1)) != hipSuccess)
    rc = yk_hip_fail(e, "hipEventElapsedTime");
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}
