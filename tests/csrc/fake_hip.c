// A HIP runtime without a device, for tests of the library's host code on the
// CPU: device memory is host memory, kernels are not run, allocations, copies
// and synchronizations fail on request, and the pointers that some kernels must
// be given are checked at their launch.
//
// Built as libamdhip64.so.7 and found through LD_LIBRARY_PATH by a child process.
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;
typedef struct { int pending; } stream_t;

enum { kOk = 0, kOutOfMemory = 2, kUnknown = 999 };

// ---- what the test sets and reads
int fake_malloc_at = -1, fake_malloc_times = 0;  // the next mallocs but `at` fail, `times` of them
int fake_copy_at = -1;                           // the asynchronous copy that fails
int fake_stream_fails = 0;                       // streams cannot be created
int fake_sync_fails = 0;                         // stream synchronizations fail
unsigned fake_flags = 0;                         // status flags after the next reset
int fake_flags_times = 0;
int fake_nwords = 0;                             // list lengths the neighbor kernel leaves
unsigned long long fake_total = 0;               // words that long lists need
unsigned long long fake_tape_need = 0;           // words a tape lacks, once
int fake_mallocs = 0, fake_violations = 0, fake_long_lists = 0, fake_streams = 0, fake_syncs = 0;
char fake_note[256];

static struct { void* p; size_t bytes; } g_mem[4096];
static int g_nmem = 0;
static stream_t* g_streams[256];

int fake_live(void) { return g_nmem; }
long long fake_live_bytes(void) {
  long long b = 0;
  for (int i = 0; i < g_nmem; ++i) b += (long long)g_mem[i].bytes;
  return b;
}
int fake_pending_streams(void) {
  int n = 0;
  for (int i = 0; i < 256; ++i) n += g_streams[i] && g_streams[i]->pending;
  return n;
}
int fake_all_streams(void) {
  int n = 0;
  for (int i = 0; i < 256; ++i) n += g_streams[i] != NULL;
  return n;
}

static void violation(const char* what) {
  ++fake_violations;
  snprintf(fake_note, sizeof(fake_note), "%s", what);
}

// ---- memory
int hipMalloc(void** p, size_t bytes) {
  ++fake_mallocs;
  *p = NULL;
  if (fake_malloc_at > 0) {
    --fake_malloc_at;
  } else if (fake_malloc_at == 0 && fake_malloc_times > 0) {
    if (--fake_malloc_times == 0) fake_malloc_at = -1;
    return kOutOfMemory;
  }
  *p = calloc(bytes ? bytes : 1, 1);
  if (!*p || g_nmem == 4096) abort();
  g_mem[g_nmem].p = *p;
  g_mem[g_nmem++].bytes = bytes;
  return kOk;
}
int hipFree(void* p) {
  if (!p) return kOk;
  for (int i = 0; i < g_nmem; ++i)
    if (g_mem[i].p == p) {
      g_mem[i] = g_mem[--g_nmem];
      free(p);
      return kOk;
    }
  violation("hipFree of memory that is not allocated");
  return kUnknown;
}
int hipMemGetAddressRange(void** base, size_t* bytes, void* p) {
  for (int i = 0; i < g_nmem; ++i)
    if (p >= g_mem[i].p && (char*)p < (char*)g_mem[i].p + g_mem[i].bytes) {
      *base = g_mem[i].p;
      *bytes = g_mem[i].bytes;
      return kOk;
    }
  return kUnknown;
}
// Every allocation and stream is gone (the host memory stays, so that a use of it
// shows as a violation and not as a crash).
int hipDeviceReset(void) {
  g_nmem = 0;
  memset(g_streams, 0, sizeof(g_streams));
  return kOk;
}
int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  (void)flags;
  *p = calloc(bytes ? bytes : 1, 1);
  return kOk;
}
int hipHostFree(void* p) {
  free(p);
  return kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
  (void)kind;
  if (n && (!d || !s)) {
    violation("hipMemcpy of null");
    return kUnknown;
  }
  if (n) memcpy(d, s, n);
  return kOk;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, stream_t* st) {
  if (fake_copy_at == 0) {
    fake_copy_at = -1;
    return kUnknown;
  }
  if (fake_copy_at > 0) --fake_copy_at;
  if (st) st->pending = 1;
  return hipMemcpy(d, s, n, kind);
}
int hipMemsetAsync(void* d, int v, size_t n, stream_t* st) {
  if (st) st->pending = 1;
  if (!d) violation("hipMemsetAsync of null");
  else memset(d, v, n);
  return kOk;
}
int hipGetSymbolAddress(void** p, const void* sym) {
  static void* scratch = NULL;
  (void)sym;
  if (!scratch) scratch = calloc(64u << 20, 1);
  *p = scratch;
  return kOk;
}

// ---- devices, streams, events, graphs
int hipGetDeviceCount(int* n) { *n = 1; return kOk; }
int hipSetDevice(int d) { (void)d; return kOk; }
int hipGetDevice(int* d) { *d = 0; return kOk; }
int hipGetLastError(void) { return kOk; }
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "error"; }
int hipStreamCreateWithFlags(stream_t** s, unsigned flags) {
  (void)flags;
  if (fake_stream_fails) return kUnknown;  // (*s is not promised to be written)
  *s = calloc(1, sizeof(stream_t));
  ++fake_streams;
  for (int i = 0; i < 256; ++i)
    if (!g_streams[i]) {
      g_streams[i] = *s;
      return kOk;
    }
  abort();
}
int hipStreamDestroy(stream_t* s) {
  for (int i = 0; i < 256; ++i)
    if (g_streams[i] == s) {
      g_streams[i] = NULL;
      free(s);
      return kOk;
    }
  violation("hipStreamDestroy of no stream");
  return kUnknown;
}
static int known(stream_t* s) {
  for (int i = 0; i < 256; ++i)
    if (g_streams[i] == s) return 1;
  return s == NULL;
}
int hipStreamSynchronize(stream_t* s) {
  ++fake_syncs;
  if (!known(s)) {
    violation("hipStreamSynchronize of no stream");
    return kUnknown;
  }
  if (fake_sync_fails) return kUnknown;
  if (s) s->pending = 0;
  return kOk;
}
int hipDeviceSynchronize(void) {
  for (int i = 0; i < 256; ++i)
    if (g_streams[i]) g_streams[i]->pending = 0;
  return kOk;
}
int hipStreamWaitEvent(stream_t* s, void* e, unsigned f) { (void)s; (void)e; (void)f; return kOk; }
int hipStreamBeginCapture(stream_t* s, int mode) { (void)s; (void)mode; return kOk; }
int hipStreamEndCapture(stream_t* s, void** g) { (void)s; *g = malloc(1); return kOk; }
int hipGraphInstantiate(void** x, void* g, void* a, void* b, size_t n) {
  (void)g; (void)a; (void)b; (void)n;
  *x = malloc(1);
  return kOk;
}
int hipGraphLaunch(void* x, stream_t* s) { (void)x; if (s) s->pending = 1; return kOk; }
int hipGraphDestroy(void* g) { free(g); return kOk; }
int hipGraphExecDestroy(void* x) { free(x); return kOk; }
int hipEventCreate(void** e) { *e = malloc(1); return kOk; }
int hipEventCreateWithFlags(void** e, unsigned f) { (void)f; *e = malloc(1); return kOk; }
int hipEventDestroy(void* e) { free(e); return kOk; }
int hipEventRecord(void* e, stream_t* s) { (void)e; (void)s; return kOk; }
int hipEventSynchronize(void* e) { (void)e; return kOk; }
int hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 1.0f; return kOk; }

// ---- kernels
static struct { const void* host; char name[128]; } g_kernels[512];
static int g_nkernels = 0;
static _Thread_local struct { dim3_t grid, block; size_t lds; stream_t* stream; } g_call;

void** __hipRegisterFatBinary(const void* data) {
  static void* handle;
  (void)data;
  return &handle;
}
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** h, const void* host, char* dev, const char* name, unsigned limit,
                           void* tid, void* bid, void* bdim, void* gdim, int* wsize) {
  (void)h; (void)dev; (void)limit; (void)tid; (void)bid; (void)bdim; (void)gdim; (void)wsize;
  if (g_nkernels == 512) abort();
  g_kernels[g_nkernels].host = host;
  snprintf(g_kernels[g_nkernels++].name, 128, "%s", name);
}
void __hipRegisterVar(void** h, void* var, char* host, char* dev, int ext, size_t size, int c,
                      int g) {
  (void)h; (void)var; (void)host; (void)dev; (void)ext; (void)size; (void)c; (void)g;
}
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, stream_t* stream) {
  g_call.grid = grid;
  g_call.block = block;
  g_call.lds = lds;
  g_call.stream = stream;
  return kOk;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* lds, stream_t** stream) {
  *grid = g_call.grid;
  *block = g_call.block;
  *lds = g_call.lds;
  *stream = g_call.stream;
  return kOk;
}

static void* ptr(void** args, int i) { return *(void**)args[i]; }
static long long i64(void** args, int i) { return *(long long*)args[i]; }
static void need(void** args, int i, const char* what) {
  if (!ptr(args, i)) violation(what);
}
static void need_list(void** args, int i, const char* what) {
  if (!ptr(args, i) && i64(args, i + 1) > 0) violation(what);
}

int hipLaunchKernel(const void* host, dim3_t grid, dim3_t block, void** args, size_t lds,
                    stream_t* stream) {
  (void)grid; (void)block; (void)lds;
  const char* name = "";
  for (int i = 0; i < g_nkernels; ++i)
    if (g_kernels[i].host == host) name = g_kernels[i].name;
  if (stream) stream->pending = 1;
  if (strstr(name, "k_reset_flags")) {
    *(unsigned*)ptr(args, 0) = fake_flags_times > 0 ? fake_flags : 0u;
    *(int*)ptr(args, 1) = 1;  // substeps started
    if (fake_flags_times > 0) --fake_flags_times;
  } else if (strstr(name, "7k_table")) {
    need(args, 15, "k_table without a cell table");
  } else if (strstr(name, "11k_neighbors")) {
    const int n = *(int*)args[0];
    for (int i = 0; i < n; ++i) ((int*)ptr(args, 7))[i] = fake_nwords;
    need_list(args, 9, "k_neighbors without a list buffer");
  } else if (strstr(name, "k_store_rows")) {
    need_list(args, 5, "k_store_rows without a list buffer");
  } else if (strstr(name, "k_dense_lists")) {
    need_list(args, 6, "k_dense_lists without a list buffer");
  } else if (strstr(name, "k_long_lists")) {
    ++fake_long_lists;
    need_list(args, 5, "k_long_lists without a list buffer");
    ((int*)ptr(args, 3))[0] = 1;  // some lists are stored before one does not fit
    *(unsigned long long*)ptr(args, 7) = fake_total;
  } else if (strstr(name, "k_tape_copy")) {
    need(args, 7, "k_tape_copy without a list buffer");
    need(args, 9, "k_tape_copy without a tape");
    need_list(args, 15, "k_tape_copy without a tape's list buffer");
    if (fake_tape_need) *(unsigned long long*)ptr(args, 17) = fake_tape_need;
    fake_tape_need = 0;
  } else if (strstr(name, "k_adj_seed")) {
    need(args, 1, "k_adj_seed without a tape");
  } else if (strstr(name, "k_soa_to_f4")) {
    need(args, 2, "k_soa_to_f4 without an adjoint buffer");
  } else if (strstr(name, "k_f4_to_soa")) {
    need(args, 1, "k_f4_to_soa without an adjoint buffer");
    need(args, 2, "k_f4_to_soa without a staging buffer");
  } else if (strstr(name, "k_zero_f64")) {
    need(args, 1, "k_zero_f64 without an adjoint buffer");
  }
  return kOk;
}
