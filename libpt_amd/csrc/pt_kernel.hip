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

/* one workgroup, fixed-order compensated sum of x[0..n) */
__global__ __launch_bounds__(1024) void
k_reduce(const double *x, int64_t n, double *out)
{
	reduce_block(x, n, out);
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
 * Operand packing (pt_slab_frags): one workgroup makes the fragments of one
 * (slab, row block, kappa chunk) for PACK_COLS columns.  It reads the
 * plane along its contiguous index (columns, or rows with TR), lays the
 * fragments out in LDS and writes them as whole 1 KB runs; rows and kappa
 * beyond the extents, and tri pairs with column >= row, are zero.  Bound
 * by HBM (each element read once and written once).
 */
constexpr int PACK_COLS = 32;

template <int F>
__global__ __launch_bounds__(256) void
k_pack(const void *src, char *dst, int64_t K, int64_t rows, int64_t cols,
    int tri, int tr, double scale, int64_t nch, int64_t nrb, int64_t ncg)
{
	constexpr bool SPLIT = F == PT_FORM_BF16X3 || F == PT_FORM_F16X3;
	constexpr int KC = F == PT_FORM_FP64 ? 8 : 16;
	typedef typename std::conditional<F == PT_FORM_FP32, float, double>::type
	    T;
	/* fragment stride: 8-byte pieces of consecutive columns fall on
	 * consecutive pairs of banks */
	constexpr int FS = PT_FRAG + 8;
	__shared__ __attribute__((aligned(16))) char lds[PACK_COLS * FS];
	const int64_t bid = blockIdx.x;
	const int64_t cg = bid % ncg, ch = bid / ncg % nch;
	const int64_t rb = bid / (ncg * nch) % nrb, r = bid / (ncg * nch * nrb);
	const int64_t c0 = cg * PACK_COLS, bcols = tri ? 16 * (rb + 1) : cols;
	if (c0 >= bcols)
		return;
	const int64_t pl = tri ? rows * (rows - 1) / 2 : rows * cols;
	const T *sp = (const T *)src + (r * K + ch * KC) * pl;
	for (int n = threadIdx.x; n < 16 * KC * PACK_COLS; n += 256) {
		int row, kk, col;
		if (tr) {
			row = n % 16;
			col = n / 16 % PACK_COLS;
			kk = n / (16 * PACK_COLS);
		} else {
			col = n % PACK_COLS;
			row = n / PACK_COLS % 16;
			kk = n / (16 * PACK_COLS);
		}
		const int64_t u = 16 * rb + row, w = c0 + col;
		T x = 0;
		if (ch * KC + kk < K && u < rows && (tri ? w < u : w < cols))
			x = sp[kk * pl + (tri ? u * (u - 1) / 2 + w : tr ?
			    w * rows + u : u * cols + w)];
		constexpr int KQ = KC / 4;
		const int e = kk % KQ;
		char *d = lds + col * FS + 16 * (16 * (kk / KQ) + row);
		if constexpr (SPLIT) {
			uint16_t hb, lb;
			split2(x * scale, F == PT_FORM_F16X3, hb, lb);
			*(uint16_t *)(d + 2 * e) = hb;
			*(uint16_t *)(d + 8 + 2 * e) = lb;
		} else {
			*(T *)(d + e * sizeof(T)) = x;
		}
	}
	__syncthreads();
	const int64_t f0 = tri ? nch * (r * 8 * nrb * (nrb + 1) +
	    8 * rb * (rb + 1)) + ch * bcols + c0 :
	    ((r * nrb + rb) * nch + ch) * cols + c0;
	for (int n = threadIdx.x; n < 64 * PACK_COLS; n += 256) {
		const int col = n / 64, l = n % 64;
		if (c0 + col >= bcols)
			break;
		const uint64_t *s8 = (const uint64_t *)(lds + col * FS + 16 * l);
		uint64_t *d8 = (uint64_t *)(dst + (f0 + col) * PT_FRAG + 16 * l);
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
		double x = src[t] * scale;
		uint16_t hb, lb;
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
pt_launch_tiles(int form, const struct pt_launch *p, void *stream)
{
	if (p->n_chunk <= 0)
		return 0;
	switch (form) {
	case PT_FORM_FP64: return pt_launch_tiles_fp64(p, stream);
	case PT_FORM_FP32: return pt_launch_tiles_fp32(p, stream);
	case PT_FORM_BF16X3: return pt_launch_tiles_bf16x3(p, stream);
	case PT_FORM_F16X3: return pt_launch_tiles_f16x3(p, stream);
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
pt_launch_reduce(const double *x, int64_t n, double *out, void *stream)
{
	k_reduce<<<1, 1024, 0, (hipStream_t)stream>>>(x, n, out);
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
pt_launch_pack(const void *src, void *dst, int64_t R, int64_t K, int64_t rows,
    int64_t cols, int tri, int tr, int form, double scale, void *stream)
{
	const int64_t nch = pt_chunks(form, K), nrb = (rows + 15) / 16;
	const int64_t ncg = ((tri ? 16 * nrb : cols) + PACK_COLS - 1) / PACK_COLS;
	if (R <= 0 || nch <= 0 || nrb <= 0 || ncg <= 0)
		return 0;
	/* at most 2^30 workgroups per launch, in whole slabs */
	const int64_t per = nch * nrb * ncg;
	const int64_t step = per < ((int64_t)1 << 30) ? ((int64_t)1 << 30) / per : 1;
	const int64_t pl = tri ? rows * (rows - 1) / 2 : rows * cols;
	const int64_t slab = pt_slab_frags(form, K, rows, cols, tri) * PT_FRAG;
	const int el = form == PT_FORM_FP32 ? 4 : 8;
	for (int64_t r = 0; r < R; r += step) {
		const dim3 grid((unsigned)(per * (step < R - r ? step : R - r)));
		const void *sp = (const char *)src + r * K * pl * el;
		char *dp = (char *)dst + r * slab;
		const hipStream_t st = (hipStream_t)stream;
#define PACK(F) k_pack<F><<<grid, 256, 0, st>>>(sp, dp, K, rows, cols, tri, \
    tr, scale, nch, nrb, ncg)
		if (form == PT_FORM_FP64)
			PACK(PT_FORM_FP64);
		else if (form == PT_FORM_FP32)
			PACK(PT_FORM_FP32);
		else if (form == PT_FORM_BF16X3)
			PACK(PT_FORM_BF16X3);
		else
			PACK(PT_FORM_F16X3);
#undef PACK
		const int rc = (int)hipGetLastError();
		if (rc != 0)
			return rc;
	}
	return 0;
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
