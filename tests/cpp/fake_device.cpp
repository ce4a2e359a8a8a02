// The HIP runtime calls of the library's host code, answered in host memory,
// for tests of that code where there is no GPU: preloaded before the real
// runtime (LD_PRELOAD). Kernels do nothing. Asynchronous copies and events
// wait in one queue until a synchronization or a query reaches them, and every
// copy is checked against the allocations it touches. The fake_* functions
// are the test's side of it.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>

namespace {

struct Op {
	void *dst;
	const void *src;
	size_t n;
	hipEvent_t ev; // a record when set
};
std::recursive_mutex mu;
std::deque<Op> q;
std::map<uintptr_t, size_t> mem;   // device and pinned allocations
std::map<uintptr_t, bool> pinned;  // of them the pinned ones
std::map<hipEvent_t, int> records; // an event's records still queued
size_t used, limit = (size_t)-1, copied_max;
long out_of_range, launches, fail_at = -1;
thread_local hipError_t last = hipSuccess;
struct Conf {
	dim3 g, b;
	size_t lds;
	hipStream_t st;
};
thread_local Conf conf;

typedef std::lock_guard<std::recursive_mutex> Lock;

hipError_t ret(hipError_t e)
{
	if (e != hipSuccess) last = e;
	return e;
}

// whether n bytes at p lie inside the allocation that p is in (memory of no allocation is the caller's)
bool inside(const void *p, size_t n, bool *ours)
{
	auto it = mem.upper_bound((uintptr_t)p);
	*ours = false;
	if (it == mem.begin()) return true;
	--it;
	if ((uintptr_t)p >= it->first + it->second) return true;
	*ours = true;
	return (uintptr_t)p + n <= it->first + it->second;
}

void run_one()
{
	const Op o = q.front();
	q.pop_front();
	if (o.ev) records[o.ev]--;
	else memcpy(o.dst, o.src, o.n);
}
void drain()
{
	while (!q.empty()) run_one();
}

hipError_t add(void **p, size_t n, bool host)
{
	Lock l(mu);
	if (!host && (used + n < used || used + n > limit)) return ret(hipErrorOutOfMemory);
	*p = calloc(1, n ? n : 1);
	mem[(uintptr_t)*p] = n;
	pinned[(uintptr_t)*p] = host;
	if (!host) used += n;
	return hipSuccess;
}
hipError_t drop(void *p)
{
	Lock l(mu);
	drain();
	auto it = mem.find((uintptr_t)p);
	if (it == mem.end()) return ret(hipErrorInvalidValue);
	if (!pinned[it->first]) used -= it->second;
	mem.erase(it);
	free(p);
	return hipSuccess;
}
uintptr_t handles = 16;

} // namespace

extern "C" {

long fake_pending() { Lock l(mu); return (long)q.size(); }
long fake_out_of_range() { return out_of_range; }
long fake_launches() { return launches; }
void fake_fail_launch(long n) { fail_at = launches + n; } // the n-th launch from here on fails
size_t fake_used() { return used; }
void fake_limit(size_t n) { limit = n; }
size_t fake_largest() // largest device allocation
{
	Lock l(mu);
	size_t m = 0;
	for (auto &x : mem)
		if (!pinned[x.first] && x.second > m) m = x.second;
	return m;
}

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
	memset(p, 0, sizeof *p);
	strcpy(p->gcnArchName, "gfx950");
	return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : e == hipErrorNotReady ? "not ready" : "error"; }
hipError_t hipGetLastError()
{
	const hipError_t e = last;
	last = hipSuccess;
	return e;
}
hipError_t hipMalloc(void **p, size_t n) { return add(p, n, false); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return add(p, n, true); }
hipError_t hipFree(void *p) { return drop(p); }
hipError_t hipHostFree(void *p) { return drop(p); }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
	static char room[1 << 20];
	return *p = room, hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) { return *s = (hipStream_t)(handles += 16), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; } // (one queue: always behind it)
hipError_t hipStreamSynchronize(hipStream_t)
{
	Lock l(mu);
	drain();
	return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)(handles += 16), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
	Lock l(mu);
	records[e]++;
	q.push_back(Op{ nullptr, nullptr, 0, e });
	return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
	Lock l(mu);
	while (records[e] > 0) run_one();
	return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e)
{
	Lock l(mu);
	if (records[e] == 0) return hipSuccess;
	run_one();
	return ret(hipErrorNotReady);
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t)
{
	Lock l(mu);
	bool od, os;
	const bool ok = inside(dst, n, &od) & inside(src, n, &os);
	if (!ok) {
		out_of_range++;
		return hipSuccess;
	}
	if (!od) drain(); // pageable memory: the runtime's own staging, done on return
	if (od && os) q.push_back(Op{ dst, src, n, nullptr });
	else memcpy(dst, src, n);
	return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind k)
{
	const hipError_t e = hipMemcpyAsync(dst, src, n, k, nullptr);
	Lock l(mu);
	drain();
	return e;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t)
{
	Lock l(mu);
	bool ours;
	if (!inside(p, n, &ours)) return out_of_range++, hipSuccess;
	drain();
	memset(p, v, n);
	return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st) { return conf = Conf{ g, b, lds, st }, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *st)
{
	return *g = conf.g, *b = conf.b, *lds = conf.lds, *st = conf.st, hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3 g, dim3 b, void **, size_t lds, hipStream_t)
{
	Lock l(mu);
	if (++launches == fail_at) return ret(hipErrorLaunchFailure);
	if (!g.x || !g.y || !g.z || (unsigned long)g.x * b.x > 0xffffffffu || g.y > 65535 || g.z > 65535 || b.x * b.y * b.z > 1024 || lds > 160 * 1024)
		return ret(hipErrorInvalidConfiguration);
	return hipSuccess;
}

} // extern "C"
