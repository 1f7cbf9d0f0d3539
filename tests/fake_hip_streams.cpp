// The stream, event and copy calls of the HIP runtime that stage.cpp makes, as a model of their order: no device, every copy a
// memcpy at the moment it is enqueued.  A stream has a clock -- for every stream, how many of its operations are certain to be done
// before the next operation of this one starts -- an event keeps the clock of its last record, a wait takes it over, and what
// the host has waited for precedes everything enqueued later.
#include <hip/hip_runtime_api.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
typedef std::map<uintptr_t, uint64_t> Clock;
std::mutex mu;
std::map<uintptr_t, Clock> streams;
std::map<uintptr_t, Clock> events;
Clock host;
uintptr_t next_handle = 0x1000;
std::string log_text;
char error_text[512];

uintptr_t key(const void* p) { return reinterpret_cast<uintptr_t>(p); }
void merge(Clock& into, const Clock& from) {
    for (auto& [s, n] : from)
        if (into[s] < n) into[s] = n;
}
uint64_t operation(uintptr_t s) {
    merge(streams[s], host);
    return ++streams[s][s];
}
std::string text(const Clock& c) {
    std::string out;
    for (auto& [s, n] : c) out += " " + std::to_string(s) + ":" + std::to_string(n);
    return out;
}
}  // namespace

namespace moe {
void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(error_text, sizeof error_text, fmt, ap);
    va_end(ap);
}
}  // namespace moe

extern "C" {
const char* moe_last_error(void) { return error_text; }

// a kernel on `stream`; returns its number there
uint64_t fake_kernel(void* stream) {
    std::lock_guard<std::mutex> lk(mu);
    return operation(key(stream));
}
// "stream:operations" pairs that precede the next operation of `stream`
const char* fake_clock(void* stream) {
    static std::string out;
    std::lock_guard<std::mutex> lk(mu);
    merge(streams[key(stream)], host);
    out = text(streams[key(stream)]);
    return out.c_str();
}
// a line per copy so far: destination, bytes, stream, its number there, clock
const char* fake_copies(void) {
    static std::string out;
    std::lock_guard<std::mutex> lk(mu);
    out = log_text;
    return out.c_str();
}

const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    std::lock_guard<std::mutex> lk(mu);
    *s = reinterpret_cast<hipStream_t>(next_handle++);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    std::lock_guard<std::mutex> lk(mu);
    merge(host, streams[key(s)]);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    std::lock_guard<std::mutex> lk(mu);
    *e = reinterpret_cast<hipEvent_t>(next_handle++);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::mutex> lk(mu);
    merge(streams[key(s)], host);
    events[key(e)] = streams[key(s)];
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::mutex> lk(mu);
    merge(host, events[key(e)]);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    std::lock_guard<std::mutex> lk(mu);
    merge(streams[key(s)], events[key(e)]);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
    std::lock_guard<std::mutex> lk(mu);
    memcpy(dst, src, n);
    const uint64_t number = operation(key(s));
    log_text += std::to_string(key(dst)) + " " + std::to_string(n) + " " + std::to_string(key(s)) + " " + std::to_string(number) + " |" +
                text(streams[key(s)]) + "\n";
    return hipSuccess;
}
}  // extern "C"
