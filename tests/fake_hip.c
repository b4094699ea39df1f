/* A HIP runtime that launches nothing: it notes the calls that order streams, and holds them to the rules a real one has (an event is
 * recorded on a stream of its own device).  A stream handle's device is its bits 12 and up; the null stream is the current device's. */
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

static char notes[1 << 16];
static size_t used;
static int current, next_event;
static int event_device[256];
static char launches[1 << 16];   /* a line per launch: kernel, stream, grid, and for kernels of the softmax queues their address */
static size_t launched;
static unsigned char segments[512];   /* the first bytes of the last convolution kernel's argument: its segments */
static struct { const void* f; const char* name; } kernels[512];
static int n_kernels;

static void note(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  if (used < sizeof(notes) - 256) used += vsnprintf(notes + used, 256, fmt, ap);
  va_end(ap);
}
static int device_of(const void* s) { return s ? (int)((size_t)s >> 12) : current; }

const char* fake_notes(void) { return notes; }
const char* fake_launches(void) { return launches; }
const void* fake_segments(void) { return segments; }
void fake_reset(int device) { used = 0; notes[0] = 0; launched = 0; launches[0] = 0; current = device; }
int fake_current(void) { return current; }

int hipGetDevice(int* d) { *d = current; return 0; }
int hipSetDevice(int d) { current = d; return 0; }
int hipStreamGetDevice(void* s, int* d) { *d = device_of(s); return 0; }
int hipEventCreateWithFlags(void** e, unsigned flags) {
  (void)flags;
  event_device[++next_event] = current;
  *e = (void*)(size_t)next_event;
  return 0;
}
int hipEventRecord(void* e, void* s) {
  note("record %lx ", (unsigned long)(size_t)s);
  return event_device[(size_t)e] == device_of(s) ? 0 : 400;   /* hipErrorInvalidHandle */
}
int hipStreamWaitEvent(void* s, void* e, unsigned flags) {
  (void)e; (void)flags;
  note("wait %lx ", (unsigned long)(size_t)s);
  return 0;
}
typedef struct { unsigned x, y, z; } dim3_t;
static struct { dim3_t grid, block; size_t lds; void* stream; } config;
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void* s) {
  config.grid = grid; config.block = block; config.lds = lds; config.stream = s;
  return 0;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* lds, void** s) {
  *grid = config.grid; *block = config.block; *lds = config.lds; *s = config.stream;
  return 0;
}
void __hipRegisterFunction(void** modules, const void* f, char* device_function, const char* name, unsigned limit, void* tid, void* bid, void* block, void* grid, int* size) {
  (void)modules; (void)device_function; (void)limit; (void)tid; (void)bid; (void)block; (void)grid; (void)size;
  if (n_kernels < 512) { kernels[n_kernels].f = f; kernels[n_kernels++].name = name; }
}
int hipLaunchKernel(const void* f, dim3_t grid, dim3_t block, void** args, size_t lds, void* s) {
  const char* name = "?";
  const void* queue = 0;
  (void)block; (void)lds;
  for (int i = 0; i < n_kernels; ++i)
    if (kernels[i].f == f) name = kernels[i].name;
  if (strstr(name, "stream_queue_clear_kernel")) queue = *(void**)args[0];
  if (strstr(name, "softmax_stream_kernel")) queue = *(void**)args[1];
  if (strstr(name, "conv_norm_kernel") || strstr(name, "conv_norm_bwd_kernel")) memcpy(segments, args[0], sizeof(segments));
  note("launch %lx:%d ", (unsigned long)(size_t)s, current);
  if (launched < sizeof(launches) - 256)
    launched += snprintf(launches + launched, 256, "%s %lx %u %lx\n", name, (unsigned long)(size_t)s, grid.x, (unsigned long)(size_t)queue);
  return 0;
}
int hipFuncSetAttribute(const void* f, int attr, int value) { (void)f; (void)attr; (void)value; return 0; }
int fake_cus = 256, fake_capturing, fake_no_host_memory;
unsigned long long fake_host_words[8];   /* the first pinned memory that is asked for */
int hipDeviceGetAttribute(int* v, int attr, int d) { (void)attr; (void)d; *v = fake_cus; return 0; }
int hipStreamIsCapturing(void* s, int* status) { (void)s; *status = fake_capturing; return 0; }
int hipThreadExchangeStreamCaptureMode(int* mode) { (void)mode; return 0; }
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  (void)flags;
  if (fake_no_host_memory || n > sizeof(fake_host_words)) return 2;   /* hipErrorOutOfMemory */
  *p = fake_host_words;
  return 0;
}
int hipGetDevicePropertiesR0600(void* p, int d) { (void)p; (void)d; return 1; }
int hipGetSymbolAddress(void** p, const void* symbol) { (void)symbol; *p = (void*)4096; return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { return e ? "an error" : "none"; }
