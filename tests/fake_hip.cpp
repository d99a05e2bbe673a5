// Stand-in for the HIP runtime, for tests of the host code without a device.
// Loaded before libtangerine_gpu.so, its functions take the runtime's place:
// device memory is host memory within a limit, copies are done at once, kernels are
// recorded and not run.  A test reads what was launched and allocated, and makes an
// allocation or a launch fail.

#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {

struct Call
{
	dim3 grid, block;
	size_t lds;
	hipStream_t stream;
};

std::recursive_mutex mutex;
std::map<const void*, std::string> kernels;
std::map<const void*, size_t> allocations;
std::map<const void*, void*> variables;
std::string launches, failing;
size_t limit = size_t(1) << 38, used = 0, peak = 0, mallocs = 0;
long pending = 0;  // asynchronous calls since the last wait
thread_local Call call;
hipError_t last = hipSuccess;

using Lock = std::lock_guard<std::recursive_mutex>;

hipError_t fails(hipError_t e) { return last = e; }

hipError_t waited()
{
	Lock lock(mutex);
	pending = 0;
	return hipSuccess;
}

hipError_t issued()
{
	Lock lock(mutex);
	++pending;
	return hipSuccess;
}

template <class T>
hipError_t handle(T* out)
{
	*out = reinterpret_cast<T>(std::malloc(1));
	return hipSuccess;
}

}  // namespace

extern "C" {

// ---- for the tests
void fake_limit(size_t bytes) { limit = bytes; }
size_t fake_used() { return used; }
size_t fake_peak() { const size_t p = peak; peak = used; return p; }
size_t fake_mallocs() { return mallocs; }
long fake_pending() { return pending; }
void fake_fail(const char* kernel) { failing = kernel; }
// Launches since the last call: a line each, kernel, workgroups, threads, LDS bytes.
const char* fake_launches()
{
	static std::string out;
	out.swap(launches);
	launches.clear();
	return out.c_str();
}

// ---- modules and launches
void** __hipRegisterFatBinary(const void*) { return new void*(nullptr); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
	kernels[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) { variables[var] = std::calloc(1, size); }
hipError_t hipGetSymbolAddress(void** p, const void* var) { *p = variables[var]; return *p ? hipSuccess : fails(hipErrorInvalidSymbol); }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
	call = Call{ grid, block, lds, stream };
	return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
	*grid = call.grid;
	*block = call.block;
	*lds = call.lds;
	*stream = call.stream;
	return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t lds, hipStream_t)
{
	Lock lock(mutex);
	const std::string name = kernels.count(f) ? kernels[f] : "?";
	if (grid.x == 0 || block.x == 0 || block.x > 1024 || lds > 160 * 1024) return fails(hipErrorInvalidConfiguration);
	if (!failing.empty() && name.find(failing) != std::string::npos) return fails(hipErrorLaunchFailure);
	launches += name + " " + std::to_string(grid.x) + " " + std::to_string(block.x) + " " + std::to_string(lds) + "\n";
	return issued();
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }

// ---- memory
hipError_t hipMalloc(void** p, size_t n)
{
	Lock lock(mutex);
	++mallocs;
	*p = used + n <= limit ? std::malloc(n) : nullptr;
	if (!*p) return fails(hipErrorOutOfMemory);
	allocations[*p] = n;
	used += n;
	peak = used > peak ? used : peak;
	return hipSuccess;
}
hipError_t hipFree(void* p)
{
	Lock lock(mutex);
	pending = 0;
	used -= allocations[p];
	allocations.erase(p);
	std::free(p);
	return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return waited(); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return issued(); }
hipError_t hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return issued(); }

// ---- devices, streams, events, graphs
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipDeviceSynchronize() { return waited(); }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t* p, int)
{
	std::memset(p, 0, sizeof(*p));
	std::strcpy(p->gcnArchName, "gfx950");
	p->multiProcessorCount = 256;
	p->warpSize = 64;
	return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipStreamCreate(hipStream_t* s) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return waited(); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) { return handle(x); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return issued(); }
hipError_t hipGraphDestroy(hipGraph_t g) { std::free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { std::free(x); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return waited(); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }

}  // extern "C"
