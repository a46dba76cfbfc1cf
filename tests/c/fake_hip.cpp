/*
 * The HIP runtime calls and kernel launchers that pt_host.cpp uses, on host
 * memory, for CPU tests of its host paths (tests/test_host_paths.py builds
 * this file and pt_host.cpp, pt_terms.cpp into one library).
 *
 * Device memory is address space that is only backed where it is touched, up
 * to a limit that a test sets.  Every operation runs when it is called, i.e.
 * in the order in which a stream would run it.  A tile launch walks its
 * positions as the kernel does and leaves 1 + ijk in the energy of each item
 * (0 times that for all tiles of an ijk but the first).
 */
#include <hip/hip_runtime.h>

#include <sys/mman.h>

#include <math.h>
#include <string.h>

#include <chrono>
#include <condition_variable>
#include <map>
#include <mutex>
#include <set>

#include "pt_engine.h"

namespace {

std::mutex mu;
std::map<void *, size_t> live;       /* device allocations */
size_t used = 0, limit = (size_t)1 << 40, peak = 0;
std::set<hipStream_t> streams;
long next_handle = 1;
long created = 0, bad = 0;           /* streams made; uses of a dead one */
long packs[2] = {0, 0};              /* pack jobs: plain, transposed */
long filters = 0, tiles = 0;
bool energy_nan = false, tiles_fail = false;

/* filters in flight of a test with two threads: the first waits for the
 * second one, or 0.3 s */
std::condition_variable cv;
int meet = 0, met = 0;

hipError_t
use(hipStream_t s)
{
	std::lock_guard<std::mutex> lk(mu);
	if (s && !streams.count(s)) {
		++bad;
		return hipErrorInvalidHandle;
	}
	return hipSuccess;
}

int64_t
item_of(const pt_launch &p, int64_t it)
{
	it += p.pos0;
	if (p.kgrp <= 1)
		return p.item0 + it;
	const int64_t nt = p.n_tiles, G = p.kgrp, m = p.n_seq / nt;
	const int64_t grp = it / (G * nt), r = it - grp * G * nt;
	const int64_t gsz = G < m - grp * G ? G : m - grp * G;
	const int64_t pos = p.item0 / nt + grp * G + r % gsz;
	return (p.perm ? (int64_t)p.perm[pos] : pos) * nt + r / gsz;
}

} /* namespace */

extern "C" {

/* ---- controls of the tests */
void
fake_limit(size_t bytes)
{
	std::lock_guard<std::mutex> lk(mu);
	limit = bytes;
	peak = used;
}

/* 0 bytes in use, 1 their peak since fake_limit, 2 streams created, 3 uses
 * of a dead stream, 4 and 5 pack jobs (plain, transposed), 6 filters, 7 tile
 * launches */
long
fake_count(int what)
{
	std::lock_guard<std::mutex> lk(mu);
	const long v[] = {(long)used, (long)peak, created, bad, packs[0],
	    packs[1], filters, tiles};
	return v[what];
}

void
fake_nan(int on)
{
	energy_nan = on != 0;
}

void
fake_fail_tiles(int on)
{
	tiles_fail = on != 0;
}

void
fake_meet(int n)
{
	std::lock_guard<std::mutex> lk(mu);
	meet = n;
	met = 0;
}

/* what hipDeviceReset does to the streams of a process */
void
fake_reset_streams(void)
{
	std::lock_guard<std::mutex> lk(mu);
	streams.clear();
}

size_t
fake_arena(void)
{
	return PT_NOALLOC_ARENA;
}

void *
fake_region(size_t bytes)
{
	void *p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE |
	    MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
	return p == MAP_FAILED ? nullptr : p;
}

void
fake_region_free(void *p, size_t bytes)
{
	(void)munmap(p, bytes);
}

/* ---- HIP runtime */
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e)
{
	return e == hipErrorOutOfMemory ? "out of memory" : "error";
}

hipError_t
hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
	*v = 256;
	return hipSuccess;
}

hipError_t
hipMalloc(void **p, size_t n)
{
	std::lock_guard<std::mutex> lk(mu);
	if (n > limit - used || !(*p = fake_region(n)))
		return hipErrorOutOfMemory;
	live[*p] = n;
	used += n;
	peak = used > peak ? used : peak;
	return hipSuccess;
}

hipError_t
hipFree(void *p)
{
	std::lock_guard<std::mutex> lk(mu);
	auto it = live.find(p);
	if (it != live.end()) {
		used -= it->second;
		fake_region_free(p, it->second);
		live.erase(it);
	}
	return hipSuccess;
}

hipError_t
hipHostMalloc(void **p, size_t n, unsigned)
{
	*p = malloc(n);
	return *p ? hipSuccess : hipErrorOutOfMemory;
}

hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }

hipError_t
hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
	memcpy(d, s, n);
	return hipSuccess;
}

hipError_t
hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
	const hipError_t e = use(st);
	if (e == hipSuccess)
		memcpy(d, s, n);
	return e;
}

hipError_t
hipMemset(void *d, int v, size_t n)
{
	memset(d, v, n);
	return hipSuccess;
}

hipError_t
hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
	memset(d, v, n);
	return use(st);
}

hipError_t
hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
	std::lock_guard<std::mutex> lk(mu);
	*s = (hipStream_t)(next_handle++ * 16);
	streams.insert(*s);
	++created;
	return hipSuccess;
}

hipError_t
hipStreamDestroy(hipStream_t s)
{
	const hipError_t e = use(s);
	std::lock_guard<std::mutex> lk(mu);
	streams.erase(s);
	return e;
}

hipError_t hipStreamSynchronize(hipStream_t s) { return use(s); }

/* asking whether a handle is a stream is no use of it */
hipError_t
hipStreamQuery(hipStream_t s)
{
	std::lock_guard<std::mutex> lk(mu);
	return !s || streams.count(s) ? hipSuccess : hipErrorInvalidHandle;
}

hipError_t
hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode)
{
	return use(s);
}

hipError_t
hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
	*g = (hipGraph_t)16;
	return use(s);
}

hipError_t
hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *,
    size_t)
{
	*x = (hipGraphExec_t)16;
	return hipSuccess;
}

hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { return use(s); }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

hipError_t
hipEventCreate(hipEvent_t *e)
{
	*e = (hipEvent_t)16;
	return hipSuccess;
}

hipError_t
hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
	return hipEventCreate(e);
}

hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t s) { return use(s); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

hipError_t
hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
	*ms = 1.0f;
	return hipSuccess;
}

/* ---- kernel launchers */
int
pt_launch_tiles(int form, const struct pt_launch *p, int n, void *stream)
{
	(void)form;
	const hipError_t e = use((hipStream_t)stream);
	if (e != hipSuccess || tiles_fail)
		return e ? (int)e : (int)hipErrorUnknown;
	for (int q = 0; q < n; ++q)
		for (int64_t t = 0; t < p[q].n_chunk; ++t) {
			const int64_t it = item_of(p[q], t);
			p[q].partial[it] = it % p[q].n_tiles ? 0.0 :
			    1.0 + (double)(it / p[q].n_tiles);
		}
	std::lock_guard<std::mutex> lk(mu);
	++tiles;
	return 0;
}

int
pt_launch_filter(const int32_t *perm, int64_t n, int32_t lo, int32_t hi,
    int32_t *out, void *stream)
{
	const hipError_t e = use((hipStream_t)stream);
	for (int64_t t = 0; t < n && e == hipSuccess; ++t)
		if (perm[t] >= lo && perm[t] < hi)
			*out++ = perm[t];
	std::unique_lock<std::mutex> lk(mu);
	++filters;
	if (met < meet) {
		++met;
		cv.notify_all();
		cv.wait_for(lk, std::chrono::milliseconds(300), [] {
			return met >= meet;
		});
	}
	return (int)e;
}

int
pt_launch_reduce(const double *const *x, const int64_t *n, int cnt,
    double *out, void *stream)
{
	for (int q = 0; q < cnt; ++q) {
		out[q] = energy_nan ? NAN : 0.0;
		for (int64_t t = 0; t < n[q]; ++t)
			out[q] += x[q][t];
	}
	return (int)use((hipStream_t)stream);
}

int
pt_launch_reduce_batch(const struct pt_launch *segs, const int64_t *begin,
    int nseg, double *out, void *stream)
{
	for (int s = 0; s < nseg; ++s) {
		out[s] = 0;
		for (int64_t t = 0; t < begin[s + 1] - begin[s]; ++t)
			out[s] += segs[s].partial[t];
	}
	return (int)use((hipStream_t)stream);
}

int
pt_launch_segsum(const double *x, int64_t nseg, int64_t seglen, double *out,
    void *stream)
{
	for (int64_t s = 0; s < nseg; ++s) {
		out[s] = 0;
		for (int64_t t = 0; t < seglen; ++t)
			out[s] += x[s * seglen + t];
	}
	return (int)use((hipStream_t)stream);
}

int
pt_launch_pack(const struct pt_pack_job *jobs, int n, int form, void *stream)
{
	(void)form;
	std::unique_lock<std::mutex> lk(mu);
	for (int q = 0; q < n; ++q)
		++packs[jobs[q].tr != 0];
	lk.unlock();
	return (int)use((hipStream_t)stream);
}

int
pt_launch_split(const double *, uint32_t *, int64_t, int, double, void *stream)
{
	return (int)use((hipStream_t)stream);
}

int
pt_launch_absmax(const double *, int64_t, double *, void *stream)
{
	return (int)use((hipStream_t)stream);
}

int
pt_launch_copy(const double *, double *, int64_t, void *stream)
{
	return (int)use((hipStream_t)stream);
}

int
pt_launch_synth(const void *, int, void *, int64_t, int, void *stream)
{
	return (int)use((hipStream_t)stream);
}

} /* extern "C" */
