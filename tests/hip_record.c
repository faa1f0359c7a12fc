/* A HIP runtime on the CPU that records what the library asks of it, for
 * tests of the library's host side (tests/test_host_runtime.py): loaded with
 * RTLD_GLOBAL before librkx.so, its symbols take the place of the runtime's.
 *
 * Work on a stream waits in a queue until something waits for that stream;
 * hipStreamQuery runs the oldest entry.  Streams do not wait for each other
 * (the library's are non-blocking).  Device memory is host memory; copies move
 * their bytes at once, so only their order is modelled.  A kernel launch does
 * nothing but count as one attempted step in the solves' pinned block, as
 * the step control reports to a solve's host_view: launch k makes attempt k
 * and runs the control of attempt k - 1. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

enum { kMaxOps = 1 << 16, kMaxBlocks = 4096, kMaxPinned = 256, kMaxGraphs = 64 };

typedef struct {
  hipStream_t stream;
  int graph;              /* 1 + the executable graph the launch belongs to */
  int launch;
  char *dst;              /* what a copy or a clear writes */
  size_t bytes;
} op_t;

typedef struct {
  char *p;
  size_t bytes;
} block_t;

typedef struct {          /* the library's host_view, in front of its pinned blocks */
  double t, h;
  int acc, rej, cur, done;
} view_t;

static op_t ops[kMaxOps];
static int nops;
static block_t blocks[kMaxBlocks];
static int nblocks;
static block_t pinned[kMaxPinned];
static int npinned;
static size_t live, limit;
static int graph_launches[kMaxGraphs], ngraphs, capturing = -1;
static view_t *view;
static unsigned last_grid;
static int attempts, done_after;

static struct {
  int graph_destroyed_early;      /* executable graphs destroyed with launches queued */
  int unordered_writes;           /* writes to memory that another stream has still to write */
  int graph_replays;
  int allocations;                /* of device memory */
  int waits;                      /* for a stream */
  int pageable_copies;            /* between device memory and memory that is not pinned */
  unsigned pinned_flags;          /* of the pinned block made last */
} rec;

static void run_op(int i)
{
  const op_t o = ops[i];
  memmove(ops + i, ops + i + 1, (size_t) (--nops - i) * sizeof(op_t));
  if (!o.launch || !view || view->done)
    return;
  view->acc = attempts++;
  if (view->acc >= done_after)
    view->done = 1;
}
static void drain(hipStream_t s, int all)
{
  for (int i = 0; i < nops;)
    if (all || ops[i].stream == s)
      run_op(i);
    else
      ++i;
}
static hipError_t queue(hipStream_t s, int launch, int graph, void *dst, size_t bytes)
{
  char *d = (char *) dst;
  if (nops == kMaxOps)
    drain(s, 0);
  for (int i = 0; dst && i < nops; ++i)
    if (ops[i].stream != s && ops[i].dst && ops[i].dst < d + bytes && d < ops[i].dst + ops[i].bytes)
      ++rec.unordered_writes;
  ops[nops++] = (op_t){s, graph, launch, d, bytes};
  return hipSuccess;
}

/* for the tests */
int rec_graph_destroyed_early(void) { return rec.graph_destroyed_early; }
int rec_unordered_writes(void) { return rec.unordered_writes; }
int rec_graph_replays(void) { return rec.graph_replays; }
int rec_allocations(void) { return rec.allocations; }
int rec_waits(void) { return rec.waits; }
int rec_pageable_copies(void) { return rec.pageable_copies; }
unsigned rec_pinned_flags(void) { return rec.pinned_flags; }
unsigned rec_last_grid(void) { return last_grid; }   /* workgroups of the last launch */
size_t rec_live_bytes(void) { return live; }
void rec_limit(size_t bytes) { limit = bytes; }
/* the next solve ends after this many attempts */
void rec_next_solve(int n)
{
  attempts = 0;
  done_after = n;
}
static size_t last_copy_block, last_copy_bytes;
/* bytes of the block that the last copy of `bytes` to the device went into */
void rec_watch_copy(size_t bytes)
{
  last_copy_bytes = bytes;
  last_copy_block = 0;
}
size_t rec_copy_block(void) { return last_copy_block; }

/* the runtime */
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d)
{
  (void) a, (void) d;
  *v = 256;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { (void) e; return "recorded"; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l)
{
  (void) f, (void) b, (void) l;
  *n = 1;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
  (void) p;
  memset(a, 0, sizeof(*a));
  return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t bytes)
{
  if (nblocks == kMaxBlocks || (limit && live + bytes > limit))
    return hipErrorOutOfMemory;
  *p = calloc(1, bytes);
  blocks[nblocks++] = (block_t){(char *) *p, bytes};
  live += bytes;
  ++rec.allocations;
  return hipSuccess;
}
hipError_t hipFree(void *p)
{
  drain(NULL, 1);
  for (int i = 0; i < nblocks; ++i)
    if (blocks[i].p == p) {
      live -= blocks[i].bytes;
      blocks[i] = blocks[--nblocks];
      free(p);
      return hipSuccess;
    }
  return hipErrorInvalidValue;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
  *p = calloc(1, bytes);
  rec.pinned_flags = flags;
  if (flags)                        /* a batch's snapshots ask for none */
    view = (view_t *) *p;
  if (npinned < kMaxPinned)
    pinned[npinned++] = (block_t){(char *) *p, bytes};
  return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
  if ((char *) view == (char *) p)
    view = NULL;
  for (int i = 0; i < npinned; ++i)
    if (pinned[i].p == p)
      pinned[i--] = pinned[--npinned];
  free(p);
  return hipSuccess;
}

static int within(const block_t *b, int n, const void *p)
{
  for (int i = 0; i < n; ++i)
    if (b[i].p <= (const char *) p && (const char *) p < b[i].p + b[i].bytes)
      return 1;
  return 0;
}
static int pageable(const void *p)
{
  return !within(blocks, nblocks, p) && !within(pinned, npinned, p);
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
  (void) k;
  memmove(d, s, n);
  if (pageable(d) || pageable(s))
    ++rec.pageable_copies;
  for (int i = 0; n == last_copy_bytes && i < nblocks; ++i)
    if (blocks[i].p <= (char *) d && (char *) d < blocks[i].p + blocks[i].bytes)
      last_copy_block = blocks[i].bytes;
  return queue(st, 0, 0, d, n);
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
  hipMemcpyAsync(d, s, n, k, NULL);
  drain(NULL, 0);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
  memset(d, v, n);
  return queue(st, 0, 0, d, n);
}
/* on device memory the call may return before the clear has run */
hipError_t hipMemset(void *d, int v, size_t n) { return hipMemsetAsync(d, v, n, NULL); }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f)
{
  (void) f;
  *s = (hipStream_t) calloc(1, 64);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
  ++rec.waits;
  drain(s, 0);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { drain(NULL, 1); return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s)
{
  for (int i = 0; i < nops; ++i)
    if (ops[i].stream == s) {
      run_op(i);
      return hipErrorNotReady;
    }
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f)
{
  (void) f;
  *e = (hipEvent_t) calloc(1, sizeof(hipStream_t));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { *(hipStream_t *) e = s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { drain(*(hipStream_t *) e, 0); return hipSuccess; }

static struct {
  dim3 g, b;
  size_t l;
  hipStream_t s;
} config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s)
{
  config.g = g;
  config.b = b;
  config.l = l;
  config.s = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s)
{
  *g = config.g;
  *b = config.b;
  *l = config.l;
  *s = config.s;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t l, hipStream_t s)
{
  (void) f, (void) b, (void) a, (void) l;
  last_grid = g.x;
  if (capturing >= 0) {
    ++graph_launches[capturing];
    return hipSuccess;
  }
  return queue(s, 1, 0, NULL, 0);
}

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m)
{
  (void) s, (void) m;
  capturing = ngraphs++ % kMaxGraphs;
  graph_launches[capturing] = 0;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
  (void) s;
  *g = (hipGraph_t) (size_t) (capturing + 1);
  capturing = -1;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *n, char *log,
                               size_t size)
{
  (void) n, (void) log, (void) size;
  *e = (hipGraphExec_t) g;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s)
{
  const int id = (int) (size_t) e;
  ++rec.graph_replays;
  for (int k = 0; k < graph_launches[id - 1]; ++k)
    queue(s, 1, id, NULL, 0);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e)
{
  for (int i = 0; i < nops; ++i)
    if (ops[i].graph == (int) (size_t) e) {
      ++rec.graph_destroyed_early;
      break;
    }
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { (void) g; return hipSuccess; }
