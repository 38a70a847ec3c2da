// hip_stub.cpp -- a HIP runtime without a GPU, for tests of the library's host side: four
// devices whose memory is host memory, launches that do nothing, and a record of which device
// was current at every call that depends on it.  Built as a library of the runtime's soname and
// loaded ahead of libycn.so, whose undefined symbols it covers.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
struct Handle {   // a stream or an event
    int dev;
};
struct Dim3 {
    uint32_t x, y, z;
};
struct LaunchConfig {
    Dim3 grid, block;
    size_t shared;
    void *stream;
};
constexpr int kOk = 0, kInvalidDevice = 101, kDevices = 4;
thread_local int current = 0;
thread_local LaunchConfig pending;

std::map<const void *, std::string> &kernels() {
    static std::map<const void *, std::string> k;
    return k;
}
std::string record;            // one line per call: call, current device, detail
std::string watched;           // launches of kernels whose name holds this leave their arguments
int watchedArgs = 0;

void note(const char *call, const std::string &detail) {
    record += std::string(call) + " " + std::to_string(current) + " " + detail + "\n";
}
int give(void **p, size_t n) {
    *p = std::calloc(1, n ? n : 1);
    return *p ? kOk : 2;
}
void *make(const char *call) {
    note(call, "-");
    return new Handle{current};
}
}  // namespace

extern "C" {

const char *stub_record() { return record.c_str(); }
void stub_clear() { record.clear(); }
void stub_watch(const char *name, int args) {
    watched = name;
    watchedArgs = args;
}

int hipGetDeviceCount(int *n) { *n = kDevices; return kOk; }
int hipGetDevice(int *d) { *d = current; return kOk; }
int hipSetDevice(int d) {
    if (d < 0 || d >= kDevices) return kInvalidDevice;
    current = d;
    return kOk;
}
int hipDeviceSynchronize() { return kOk; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 256; return kOk; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 2; return kOk; }
const char *hipGetErrorString(int) { return "stub error"; }
int hipGetLastError() { return kOk; }

int hipMalloc(void **p, size_t n) { note("hipMalloc", "-"); return give(p, n); }
int hipHostMalloc(void **p, size_t n, unsigned) { note("hipHostMalloc", "-"); return give(p, n); }
int hipFree(void *p) { std::free(p); return kOk; }
int hipHostFree(void *p) { std::free(p); return kOk; }
int hipMemcpy(void *d, const void *s, size_t n, int) { std::memcpy(d, s, n); return kOk; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { std::memcpy(d, s, n); return kOk; }
int hipMemset(void *d, int v, size_t n) { std::memset(d, v, n); return kOk; }
int hipMemsetAsync(void *d, int v, size_t n, void *) { std::memset(d, v, n); return kOk; }
int hipGetSymbolAddress(void **p, const void *) {   // the largest device array: the noise scratch
    static char *scratch[kDevices] = {};
    if (!scratch[current]) scratch[current] = (char *)std::calloc(1, 16 << 20);
    *p = scratch[current];
    return kOk;
}

int hipStreamCreateWithFlags(void **s, unsigned) { *s = make("hipStreamCreateWithFlags"); return kOk; }
int hipStreamDestroy(void *s) { delete (Handle *)s; return kOk; }
int hipStreamSynchronize(void *) { return kOk; }
int hipStreamQuery(void *) { return kOk; }
int hipStreamWaitEvent(void *, void *, unsigned) { return kOk; }
int hipStreamBeginCapture(void *, int) { return kOk; }
int hipStreamEndCapture(void *, void **g) { *g = new Handle{current}; return kOk; }
int hipGraphInstantiate(void **e, void *, void **, char *, size_t) { *e = make("hipGraphInstantiate"); return kOk; }
int hipGraphLaunch(void *, void *) { return kOk; }
int hipGraphDestroy(void *g) { delete (Handle *)g; return kOk; }
int hipGraphExecDestroy(void *e) { delete (Handle *)e; return kOk; }

int hipEventCreate(void **e) { *e = make("hipEventCreate"); return kOk; }
int hipEventCreateWithFlags(void **e, unsigned) { *e = make("hipEventCreateWithFlags"); return kOk; }
int hipEventDestroy(void *e) { delete (Handle *)e; return kOk; }
int hipEventRecord(void *, void *) { return kOk; }
int hipEventQuery(void *) { return kOk; }
int hipEventSynchronize(void *) { return kOk; }
int hipEventElapsedTime(float *ms, void *, void *) { *ms = 1.f; return kOk; }

void **__hipRegisterFatBinary(const void *) { static void *m; return &m; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    kernels()[host] = name;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void *s) { pending = {g, b, sh, s}; return kOk; }
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *sh, void **s) {
    *g = pending.grid;
    *b = pending.block;
    *sh = pending.shared;
    *s = pending.stream;
    return kOk;
}
int hipLaunchKernel(const void *f, Dim3, Dim3, void **args, size_t, void *) {
    std::string detail = kernels()[f];
    if (!watched.empty() && detail.find(watched) != std::string::npos)
        for (int i = 1; i < watchedArgs; ++i) {   // (argument 0 is a structure)
            uint64_t v;
            std::memcpy(&v, args[i], sizeof v);
            detail += " " + std::to_string(v);
        }
    note("hipLaunchKernel", detail);
    return kOk;
}

}  // extern "C"
