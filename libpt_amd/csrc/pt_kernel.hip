/*
 * CDNA4 (gfx950) kernels around the tile kernel (pt_tiles.h): energy
 * reductions, operand packing and splitting, family maxima, the synthetic
 * generator and a plain copy.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "pt_engine.h"
#include "synth.h"

namespace {

__device__ __forceinline__ void
kahan(double &s, double &cmp, double x)
{
	double y = x - cmp;
	double t = s + y;
	cmp = (t - s) - y;
	s = t;
}

/* fixed-order compensated sum of x[0..n) by one workgroup of 1024 */
__device__ __forceinline__ void
reduce_block(const double *x, int64_t n, double *out)
{
	__shared__ double sh[1024];
	double s = 0.0, c = 0.0;
	for (int64_t t = threadIdx.x; t < n; t += 1024)
		kahan(s, c, x[t]);
	sh[threadIdx.x] = s - c;
	__syncthreads();
	for (int w = 512; w >= 1; w >>= 1) {
		if ((int)threadIdx.x < w)
			sh[threadIdx.x] += sh[threadIdx.x + w];
		__syncthreads();
	}
	if (threadIdx.x == 0)
		out[0] = sh[0];
}

/* up to four sums, one workgroup each: fixed-order compensated */
struct reduce_args {
	const double *x[4];
	int64_t n[4];
};

__global__ __launch_bounds__(1024) void
k_reduce(reduce_args a, double *out)
{
	reduce_block(a.x[blockIdx.x], a.n[blockIdx.x], out + blockIdx.x);
}

/* one workgroup per segment: out[s] = the k_reduce sum of its partials */
__global__ __launch_bounds__(1024) void
k_reduce_batch(const pt_launch *segs, const int64_t *begin, double *out)
{
	const int s = blockIdx.x;
	reduce_block(segs[s].partial, begin[s + 1] - begin[s], out + s);
}

/* out[s] = sum of segment s (in order) */
__global__ void
k_segsum(const double *x, int64_t nseg, int64_t seglen, double *out)
{
	int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= nseg)
		return;
	double acc = 0.0, c = 0.0;
	for (int64_t t = 0; t < seglen; ++t)
		kahan(acc, c, x[s * seglen + t]);
	out[s] = acc - c;
}

__device__ __forceinline__ void
split2(double x, int fp16, uint16_t &hb, uint16_t &lb)
{
	if (fp16) {
		_Float16 h = (_Float16)x;
		_Float16 l = (_Float16)(x - (double)h);
		hb = __builtin_bit_cast(uint16_t, h);
		lb = __builtin_bit_cast(uint16_t, l);
	} else {
		__bf16 h = (__bf16)(float)x;
		__bf16 l = (__bf16)(float)(x - (double)(float)h);
		hb = __builtin_bit_cast(uint16_t, h);
		lb = __builtin_bit_cast(uint16_t, l);
	}
}

/*
 * Operand packing (pt_slab_bytes): one launch for all operands of a plan;
 * one workgroup makes the fragments of one (slab, row block, kappa chunk) of
 * a job for PACK_COLS columns.  It reads the plane along its contiguous index
 * (columns, or rows with tr), PACK_BATCH loads at a time, lays the fragments
 * out in LDS and writes them as whole 1 KB runs (64 bytes for each of the
 * fr rows that the fragments of a plane below 16 rows hold); rows and kappa
 * beyond the extents, and tri pairs with column >= row, are zero.  Bound by HBM (each
 * element read once and written once) or, in small plans, by the launch and
 * one load latency per batch.
 */
constexpr int PACK_COLS = 32, PACK_BATCH = 8, PACK_JOBS = 28;

struct pack_args {
	pt_pack_job job[PACK_JOBS];
	int n;
};

__device__ __forceinline__ int64_t
pack_groups(const pt_pack_job &j)
{
	return ((j.tri ? (j.rows + 15) / 16 * 16 : j.cols) + PACK_COLS - 1) /
	    PACK_COLS;
}

template <int F>
__global__ __launch_bounds__(256) void
k_pack(pack_args args)
{
	constexpr bool SPLIT = F == PT_FORM_BF16X3 || F == PT_FORM_F16X3;
	constexpr int KC = F == PT_FORM_FP64 ? 8 : 16;
	typedef typename std::conditional<F == PT_FORM_FP32, float, double>::type
	    T;
	/* fragment stride: 8-byte pieces of consecutive columns fall on
	 * consecutive pairs of banks */
	constexpr int FS = PT_FRAG + 8;
	__shared__ __attribute__((aligned(16))) char lds[PACK_COLS * FS];
	int q = 0;
	while (q + 1 < args.n && (int64_t)blockIdx.x >= args.job[q + 1].at)
		++q;
	const pt_pack_job &J = args.job[q];
	const int64_t K = J.K, rows = J.rows, cols = J.cols;
	const bool tri = J.tri, tr = J.tr;
	const int64_t nch = (K + KC - 1) / KC, nrb = (rows + 15) / 16;
	const int64_t ncg = pack_groups(J);
	const uint32_t bid = (uint32_t)(blockIdx.x - J.at);
	const uint32_t cg = bid % (uint32_t)ncg, b1 = bid / (uint32_t)ncg;
	const uint32_t ch = b1 % (uint32_t)nch, b2 = b1 / (uint32_t)nch;
	const uint32_t rb = b2 % (uint32_t)nrb, r = b2 / (uint32_t)nrb;
	const int64_t c0 = (int64_t)cg * PACK_COLS;
	const int64_t bcols = tri ? 16 * ((int64_t)rb + 1) : cols;
	if (c0 >= bcols)
		return;
	const int64_t pl = tri ? rows * (rows - 1) / 2 : rows * cols;
	const T *sp = (const T *)J.src + ((int64_t)r * K + (int64_t)ch * KC) * pl;
	const int tid = threadIdx.x;
	/* element n = tid + 256 it of the group: column (or, tr, row) fastest */
	auto place = [&](int n, int &row, int &col, int &kk) {
		row = tr ? n % 16 : n / PACK_COLS % 16;
		col = tr ? n / 16 % PACK_COLS : n % PACK_COLS;
		kk = n / (16 * PACK_COLS);
	};
	static_assert(16 * KC * PACK_COLS % (256 * PACK_BATCH) == 0, "batches");
	for (int n0 = tid; n0 < 16 * KC * PACK_COLS; n0 += 256 * PACK_BATCH) {
		T x[PACK_BATCH];
#pragma unroll
		for (int b = 0; b < PACK_BATCH; ++b) {
			int row, col, kk;
			place(n0 + 256 * b, row, col, kk);
			const int64_t u = 16 * (int64_t)rb + row, w = c0 + col;
			x[b] = 0;
			if ((int64_t)ch * KC + kk < K && u < rows &&
			    (tri ? w < u : w < cols))
				x[b] = sp[kk * pl + (tri ? u * (u - 1) / 2 + w : tr ?
				    w * rows + u : u * cols + w)];
		}
#pragma unroll
		for (int b = 0; b < PACK_BATCH; ++b) {
			int row, col, kk;
			place(n0 + 256 * b, row, col, kk);
			constexpr int KQ = KC / 4;
			const int e = kk % KQ;
			char *d = lds + col * FS + 16 * (16 * (kk / KQ) + row);
			if constexpr (SPLIT) {
				uint16_t hb, lb;
				split2(x[b] * J.scale, F == PT_FORM_F16X3, hb, lb);
				*(uint16_t *)(d + 2 * e) = hb;
				*(uint16_t *)(d + 8 + 2 * e) = lb;
			} else {
				*(T *)(d + e * sizeof(T)) = x[b];
			}
		}
	}
	__syncthreads();
	const int64_t f0 = tri ? nch * (r * 8 * nrb * (nrb + 1) +
	    8 * (int64_t)rb * (rb + 1)) + ch * bcols + c0 :
	    ((r * nrb + rb) * nch + ch) * cols + c0;
	const int frs = 31 - __clz(J.fr), fb = 64 << frs;
	for (int n = tid; n < (4 * PACK_COLS) << frs; n += 256) {
		const int col = n >> (frs + 2), l = n & ((4 << frs) - 1);
		if (c0 + col >= bcols)
			break;
		const int row = l & (J.fr - 1);
		const uint64_t *s8 = (const uint64_t *)(lds + col * FS +
		    16 * (16 * (l >> frs) + row));
		uint64_t *d8 = (uint64_t *)(J.dst + (f0 + col) * fb + 16 * l);
		d8[0] = s8[0];
		d8[1] = s8[1];
	}
}

/* the entries of perm in [lo, hi), in order, by one workgroup: 16 waves
 * take consecutive runs of 64 entries and add the counts of the waves
 * before them */
__global__ __launch_bounds__(1024) void
k_filter(const int32_t *perm, int64_t n, int32_t lo, int32_t hi, int32_t *out)
{
	__shared__ int cnt[2][16];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	int64_t base = 0;
	for (int64_t t0 = 0, b = 0; t0 < n; t0 += 1024, b ^= 1) {
		const int64_t t = t0 + threadIdx.x;
		const int32_t x = t < n ? perm[t] : -1;
		const bool in = t < n && x >= lo && x < hi;
		const uint64_t m = __ballot(in);
		if (lane == 0)
			cnt[b][wave] = __popcll(m);
		/* the other buffer's readers have passed this barrier's
		 * predecessor when it is written again */
		__syncthreads();
		int64_t at = base;
		for (int w = 0; w < 16; ++w) {
			if (w < wave)
				at += cnt[b][w];
			base += cnt[b][w];
		}
		if (in)
			out[at + __popcll(m & ((1ull << lane) - 1))] = x;
	}
}

/* hi + lo split of (x * scale) into bf16 or fp16 pairs */
__global__ void
k_split(const double *src, uint32_t *dst, int64_t n, int fp16, double scale)
{
	for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
	    t += (int64_t)gridDim.x * blockDim.x) {
		uint16_t hb, lb;
		split2(src[t] * scale, fp16, hb, lb);
		dst[t] = (uint32_t)hb | ((uint32_t)lb << 16);
	}
}

/* max |x| as the bit pattern of a non-negative double (order-free) */
__global__ void
k_absmax(const double *src, int64_t n, unsigned long long *out)
{
	__shared__ double sh[256];
	double m = 0.0;
	for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
	    t += (int64_t)gridDim.x * blockDim.x)
		m = fmax(m, fabs(src[t]));
	sh[threadIdx.x] = m;
	__syncthreads();
	for (int w = 128; w >= 1; w >>= 1) {
		if ((int)threadIdx.x < w)
			sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + w]);
		__syncthreads();
	}
	if (threadIdx.x == 0)
		atomicMax(out, (unsigned long long)__double_as_longlong(sh[0]));
}

/* plain copy (traffic counter calibration) */
__global__ void
k_copy(const double *src, double *dst, int64_t n)
{
	for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
	    t += (int64_t)gridDim.x * blockDim.x)
		dst[t] = src[t];
}

__global__ void
k_synth(pt_synth_spec spec, int tensor, void *dst, int64_t n, int fp32)
{
	for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
	    t += (int64_t)gridDim.x * blockDim.x) {
		double x = pt_synth_elem(&spec, tensor, t);
		if (fp32)
			((float *)dst)[t] = (float)x;
		else
			((double *)dst)[t] = x;
	}
}

} /* namespace */

extern "C" int
pt_launch_tiles(int form, const struct pt_launch *p, int n, void *stream)
{
	switch (form) {
	case PT_FORM_FP64: return pt_launch_tiles_fp64(p, n, stream);
	case PT_FORM_FP32: return pt_launch_tiles_fp32(p, n, stream);
	case PT_FORM_BF16X3: return pt_launch_tiles_bf16x3(p, n, stream);
	case PT_FORM_F16X3: return pt_launch_tiles_f16x3(p, n, stream);
	}
	return (int)hipErrorInvalidValue;
}

extern "C" int
pt_launch_reduce_batch(const struct pt_launch *segs, const int64_t *begin,
    int nseg, double *out, void *stream)
{
	if (nseg <= 0)
		return 0;
	k_reduce_batch<<<nseg, 1024, 0, (hipStream_t)stream>>>(segs, begin, out);
	return (int)hipGetLastError();
}

extern "C" int
pt_launch_reduce(const double *const *x, const int64_t *n, int cnt,
    double *out, void *stream)
{
	if (cnt <= 0)
		return 0;
	if (cnt > 4)
		return (int)hipErrorInvalidValue;
	reduce_args a = {};
	for (int q = 0; q < cnt; ++q) {
		a.x[q] = x[q];
		a.n[q] = n[q];
	}
	k_reduce<<<cnt, 1024, 0, (hipStream_t)stream>>>(a, out);
	return (int)hipGetLastError();
}

extern "C" int
pt_launch_segsum(const double *x, int64_t nseg, int64_t seglen, double *out,
    void *stream)
{
	if (nseg <= 0)
		return 0;
	k_segsum<<<(unsigned)((nseg + 255) / 256), 256, 0, (hipStream_t)stream>>>(
	    x, nseg, seglen, out);
	return (int)hipGetLastError();
}

extern "C" int
pt_launch_split(const double *src, uint32_t *dst, int64_t n, int fp16,
    double scale, void *stream)
{
	if (n <= 0)
		return 0;
	int64_t nb = (n + 255) / 256;
	k_split<<<(unsigned)(nb < 65536 ? nb : 65536), 256, 0,
	    (hipStream_t)stream>>>(src, dst, n, fp16, scale);
	return (int)hipGetLastError();
}

extern "C" int
pt_launch_pack(const struct pt_pack_job *jobs, int n, int form, void *stream)
{
	const hipStream_t st = (hipStream_t)stream;
	const int el = form == PT_FORM_FP32 ? 4 : 8;
	/* a launch takes up to PACK_JOBS jobs and fewer than 2^32 threads; a job
	 * of more goes in runs of whole slabs */
	constexpr int64_t MOST = ((int64_t)1 << 24) - 1;
	pack_args a;
	a.n = 0;
	int64_t blocks = 0;
	auto go = [&]() {
		if (a.n == 0)
			return 0;
		const dim3 grid((unsigned)blocks);
		if (form == PT_FORM_FP64)
			k_pack<PT_FORM_FP64><<<grid, 256, 0, st>>>(a);
		else if (form == PT_FORM_FP32)
			k_pack<PT_FORM_FP32><<<grid, 256, 0, st>>>(a);
		else if (form == PT_FORM_BF16X3)
			k_pack<PT_FORM_BF16X3><<<grid, 256, 0, st>>>(a);
		else
			k_pack<PT_FORM_F16X3><<<grid, 256, 0, st>>>(a);
		a.n = 0;
		blocks = 0;
		return (int)hipGetLastError();
	};
	for (int q = 0; q < n; ++q) {
		const pt_pack_job &j = jobs[q];
		const int64_t nrb = (j.rows + 15) / 16;
		const int64_t ncg = ((j.tri ? 16 * nrb : j.cols) + PACK_COLS - 1) /
		    PACK_COLS;
		const int64_t per = pt_chunks(form, j.K) * nrb * ncg;
		if (j.R <= 0 || per <= 0)
			continue;
		if (per > MOST)
			return (int)hipErrorInvalidValue;
		const int64_t pl = j.tri ? j.rows * (j.rows - 1) / 2 :
		    j.rows * j.cols;
		const int64_t slab = pt_slab_bytes(form, j.K, j.rows, j.cols, j.tri);
		for (int64_t r = 0; r < j.R;) {
			if (a.n == PACK_JOBS || MOST - blocks < per) {
				const int rc = go();
				if (rc != 0)
					return rc;
			}
			const int64_t m = (MOST - blocks) / per < j.R - r ?
			    (MOST - blocks) / per : j.R - r;
			pt_pack_job &o = a.job[a.n++];
			o = j;
			o.src = j.src + r * j.K * pl * el;
			o.dst = j.dst + r * slab;
			o.at = blocks;
			o.fr = pt_frag_rows(j.rows);
			blocks += per * m;
			r += m;
		}
	}
	return go();
}

extern "C" int
pt_launch_filter(const int32_t *perm, int64_t n, int32_t lo, int32_t hi,
    int32_t *out, void *stream)
{
	if (n <= 0)
		return 0;
	k_filter<<<1, 1024, 0, (hipStream_t)stream>>>(perm, n, lo, hi, out);
	return (int)hipGetLastError();
}

extern "C" int
pt_launch_absmax(const double *src, int64_t n, double *out, void *stream)
{
	if (n <= 0)
		return 0;
	int64_t nb = (n + 255) / 256;
	k_absmax<<<(unsigned)(nb < 4096 ? nb : 4096), 256, 0,
	    (hipStream_t)stream>>>(src, n, (unsigned long long *)out);
	return (int)hipGetLastError();
}

extern "C" int
pt_launch_copy(const double *src, double *dst, int64_t n, void *stream)
{
	if (n <= 0)
		return 0;
	k_copy<<<16384, 256, 0, (hipStream_t)stream>>>(src, dst, n);
	return (int)hipGetLastError();
}

extern "C" int
pt_launch_synth(const void *spec, int tensor, void *dst, int64_t n, int fp32,
    void *stream)
{
	if (n <= 0)
		return 0;
	int64_t nb = (n + 255) / 256;
	k_synth<<<(unsigned)(nb < 65536 ? nb : 65536), 256, 0,
	    (hipStream_t)stream>>>(*(const pt_synth_spec *)spec, tensor, dst, n,
	    fp32);
	return (int)hipGetLastError();
}
