// A stand-in for the HIP runtime that records what the library enqueues instead of running it, so that the host
// code's launches, streams and events can be checked without a GPU.  Built with the runtime's SONAME and symbol
// version and opened before libslotscan.so (test_host_streams.py).
//
// One log line per operation: "<thread> launch <kernel> <stream> <grid x> <grid y>", "<thread> record <event>
// <stream>", "<thread> wait <stream> <event>".  <thread> is what stub_thread() set.
#include <pthread.h>
#include <stdio.h>
#include <string.h>
#include <time.h>

typedef struct { unsigned x, y, z; } Dim3;
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static pthread_cond_t cv = PTHREAD_COND_INITIALIZER;
static char text[1 << 20];
static size_t len;
static __thread int self;
static struct { const void* fn; const char* name; } kern[1024];
static int nkern;
static long handle = 0x1000;
static int records[16], hold_thread = -1, hold_other = -1;
static int launches, fail_launch = -1;
static void* capturing[64];
static unsigned long long capture_id[64];
static int ncapturing;

static void put(const char* s) {                         // mu is held
    const size_t n = strlen(s);
    if (len + n < sizeof text) { memcpy(text + len, s, n); len += n; text[len] = 0; }
}
void stub_thread(int id) { self = id; }
const char* stub_log(void) { return text; }
void stub_reset(void) {
    pthread_mutex_lock(&mu);
    len = 0; text[0] = 0; launches = 0; fail_launch = -1; hold_thread = hold_other = -1;
    memset(records, 0, sizeof records);
    pthread_mutex_unlock(&mu);
}
// thread a's next wait is held until thread b has recorded an event (or half a second has passed)
void stub_hold(int a, int b) { hold_thread = a; hold_other = b; }
// launch number n (from 0) reports an error
void stub_fail_launch(int n) { fail_launch = n; }
// the stream belongs to a capture from now on (id 0: no longer)
void stub_capture(void* stream, unsigned long long id) {
    pthread_mutex_lock(&mu);
    capturing[ncapturing] = stream;
    capture_id[ncapturing++] = id;
    pthread_mutex_unlock(&mu);
}

void** __hipRegisterFatBinary(const void* d) { (void)d; static void* h; return &h; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* fn, char* df, const char* name, unsigned lim, void* a, void* b, Dim3* c,
                           Dim3* d, int* w) {
    (void)m; (void)df; (void)lim; (void)a; (void)b; (void)c; (void)d; (void)w;
    if (nkern < 1024) { kern[nkern].fn = fn; kern[nkern++].name = name; }
}
void __hipRegisterVar(void** m, void* v, char* h, char* n, int e, size_t s, int c, int g) {
    (void)m; (void)v; (void)h; (void)n; (void)e; (void)s; (void)c; (void)g;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* s, void** st) { (void)g; (void)b; (void)s; (void)st; return 0; }

static int launch(const void* fn, Dim3 g, void* st) {
    const char* name = "?";
    for (int i = 0; i < nkern; i++) if (kern[i].fn == fn) name = kern[i].name;
    char line[1024];
    pthread_mutex_lock(&mu);
    snprintf(line, sizeof line, "%d launch %s %p %u %u\n", self, name, st, g.x, g.y);
    put(line);
    launches++;
    pthread_mutex_unlock(&mu);
    return 0;
}
int hipExtLaunchKernel(const void* fn, Dim3 g, Dim3 b, void** args, size_t shm, void* st, void* e0, void* e1, int flags) {
    (void)b; (void)args; (void)shm; (void)e0; (void)e1; (void)flags;
    return launch(fn, g, st);
}
int hipLaunchKernel(const void* fn, Dim3 g, Dim3 b, void** args, size_t shm, void* st) {
    (void)b; (void)args; (void)shm;
    return launch(fn, g, st);
}
int hipGetLastError(void) { return fail_launch >= 0 && launches == fail_launch + 1 ? 1 : 0; }
const char* hipGetErrorString(int e) { return e ? "stub error" : "no error"; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { (void)a; (void)d; *v = 0; return 0; }
int hipGetSymbolAddress(void** p, const void* s) { (void)s; *p = (void*)0x100000; return 0; }

static void* fresh(void) {
    pthread_mutex_lock(&mu);
    handle += 0x10;
    void* h = (void*)handle;
    pthread_mutex_unlock(&mu);
    return h;
}
int hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; *s = fresh(); return 0; }
int hipStreamDestroy(void* s) { (void)s; return 0; }
int hipEventCreateWithFlags(void** e, unsigned f) { (void)f; *e = fresh(); return 0; }
int hipEventCreate(void** e) { *e = fresh(); return 0; }
int hipEventSynchronize(void* e) { (void)e; return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 0.f; return 0; }
int hipStreamGetCaptureInfo(void* s, int* status, unsigned long long* id) {
    pthread_mutex_lock(&mu);
    *status = 0;
    *id = 0;
    for (int i = 0; i < ncapturing; i++)
        if (capturing[i] == s) { *id = capture_id[i]; *status = capture_id[i] ? 1 : 0; }
    pthread_mutex_unlock(&mu);
    return 0;
}
int hipEventRecord(void* e, void* st) {
    char line[128];
    pthread_mutex_lock(&mu);
    snprintf(line, sizeof line, "%d record %p %p\n", self, e, st);
    put(line);
    records[self & 15]++;
    pthread_cond_broadcast(&cv);
    pthread_mutex_unlock(&mu);
    return 0;
}
int hipStreamWaitEvent(void* st, void* e, unsigned f) {
    (void)f;
    char line[128];
    pthread_mutex_lock(&mu);
    if (hold_thread == self) {
        hold_thread = -1;
        struct timespec t;
        clock_gettime(CLOCK_REALTIME, &t);
        t.tv_nsec += 500000000;
        if (t.tv_nsec >= 1000000000) { t.tv_nsec -= 1000000000; t.tv_sec++; }
        while (!records[hold_other & 15] && !pthread_cond_timedwait(&cv, &mu, &t)) {}
    }
    snprintf(line, sizeof line, "%d wait %p %p\n", self, st, e);
    put(line);
    pthread_mutex_unlock(&mu);
    return 0;
}
