/* The server's order of work, without a GPU: this program defines the HIP calls the library makes, so
 * every copy and launch only counts as queued on its stream, and as done once the host has waited for it
 * (a stream or event synchronized, an event found complete).  A job that has ended must have nothing
 * queued: its memory goes back to the pool then, for any job on any stream.
 *
 * Jobs of all four element types, in both of the server's modes.  Exit status 0 and "ok" when it holds.
 */
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "muscle_hip.h"

#define STREAMS 64
#define EVENTS 1024
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static long queued[STREAMS], done[STREAMS];         /* by stream; stream 0 is the default one */
static struct { long stream, at; } events[EVENTS];  /* what an event waits for */
static long nstreams = 1, nevents = 1, ops;

static void enqueue(hipStream_t s) {
  pthread_mutex_lock(&mu);
  queued[(long)s]++;
  ops++;
  pthread_mutex_unlock(&mu);
}
static void finish(long s, long at) {
  pthread_mutex_lock(&mu);
  if (at > done[s]) done[s] = at;
  pthread_mutex_unlock(&mu);
}
static long unfinished(void) {
  long n = 0;
  pthread_mutex_lock(&mu);
  for (long s = 0; s < nstreams; ++s) n += queued[s] - done[s];
  pthread_mutex_unlock(&mu);
  return n;
}

/* what a kernel's launch syntax calls before hipLaunchKernel */
static __thread struct { dim3 grid, block; size_t lds; hipStream_t stream; } config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  config.grid = g, config.block = b, config.lds = lds, config.stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = config.grid, *b = config.block, *lds = config.lds, *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t lds, hipStream_t s) {
  (void)f, (void)g, (void)b, (void)a, (void)lds;
  enqueue(s);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* x, size_t n, hipMemcpyKind k, hipStream_t s) {
  (void)k;
  memcpy(d, x, n);
  enqueue(s);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* x, size_t n, hipMemcpyKind k) {
  (void)k;
  memcpy(d, x, n);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned flags) {
  (void)flags;
  *s = (hipStream_t)nstreams++;
  return nstreams <= STREAMS ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  finish((long)s, queued[(long)s]);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
  for (long s = 0; s < nstreams; ++s) finish(s, queued[s]);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
  (void)flags;
  *e = (hipEvent_t)nevents++;
  return nevents <= EVENTS ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  events[(long)e].stream = (long)s;
  events[(long)e].at = queued[(long)s];
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  finish(events[(long)e].stream, events[(long)e].at);
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { return hipEventSynchronize(e); }
hipError_t hipMalloc(void** p, size_t n) { return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) { (void)flags; return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) { (void)a, (void)d; *v = 256; return hipSuccess; }

static int fails;
static void expect(int ok, const char* what, long a, long b) {
  if (!ok) ++fails, printf("FAIL: %s (%ld, %ld): %s\n", what, a, b, muscle_hip_last_error());
}

int main(void) {
  /* chains ((x y) z), with extents from one tile to several, and a modes-of-two outer product */
  static const int64_t sizes[4][5] = {{1, 5, 7, 6, 9}, {1, 40, 300, 70, 33}, {1, 128, 64, 256, 8}, {1, 512, 2, 512, 16}};
  static double leaf[512 * 512 * 2];
  int jobs = 0;
  for (int mode = 0; mode < 2; ++mode) {
    muscle_hip_server_t srv = NULL;
    expect(muscle_hip_server_create((int64_t)64 << 20, 4, mode, &srv) == MUSCLE_HIP_OK, "create", mode, 0);
    if (!srv) return 1;
    for (int it = 0; it < 16; ++it) {
      const int dtype = it % 4;
      const int64_t* e = sizes[it / 4];
      const int32_t lx[2] = {1, 2}, ly[2] = {2, 3}, lz[2] = {3, 4};
      const int64_t ex[2] = {e[1], e[2]}, ey[2] = {e[2], e[3]}, ez[2] = {e[3], e[4]};
      const int64_t sx[2] = {1, e[1]}, sy[2] = {1, e[2]}, sz[2] = {1, e[3]};
      const muscle_hip_tensor_t leaves[3] = {
          {dtype, 2, leaf, lx, ex, sx}, {dtype, 2, leaf, ly, ey, sy}, {dtype, 2, leaf, lz, ez, sz}};
      const int32_t lhs[2] = {0, 3}, rhs[2] = {1, 2}, off[3] = {0, 2, 4}, modes[4] = {1, 3, 1, 4};
      const muscle_hip_job_t job = {3, 2, leaves, lhs, rhs, off, modes, 5, e};
      int64_t id = -1;
      muscle_hip_job_result_t r;
      expect(muscle_hip_server_submit(srv, &job, &id) == MUSCLE_HIP_OK, "submit", mode, it);
      expect(muscle_hip_server_wait(srv, id, 60.0, &r) == MUSCLE_HIP_OK && r.status == MUSCLE_HIP_OK, "wait", mode, it);
      expect(unfinished() == 0, "work still queued for a job that has ended (mode, job)", mode, it);
      expect(muscle_hip_server_release(srv, id) == MUSCLE_HIP_OK, "release", mode, it);
      hipDeviceSynchronize(); /* each job counts for itself */
      ++jobs;
    }
    expect(muscle_hip_server_destroy(srv) == MUSCLE_HIP_OK, "destroy", mode, 0);
  }
  expect(ops > 4 * jobs, "copies and launches seen", ops, jobs);
  printf("%s: %d jobs, %ld copies and launches\n", fails ? "FAILED" : "ok", jobs, ops);
  return fails != 0;
}
