/*
 * CDNA4 (gfx950) tile kernel of the perturbative-triples engine, one
 * translation unit per arithmetic form (pt_tiles_*.hip).
 *
 * k_tiles: one workgroup = one ijk item x one (A, B, C) tile of 32 a x 32 b
 * x TC c.  W of the tile stays in MFMA accumulators and never goes to
 * memory:
 *
 *   phase 1 -- accumulator layout [a][b]@c (16 x 16 blocks, one c each);
 *       wave w of NW owns the whole a, b range at c = C0 + NW x + w:
 *       terms whose single index is a  (A = S rows a,  B = Q[.][b][c])
 *       terms whose single index is b  (A = Q[.][a][c], B = S rows b)
 *   transpose through LDS to layout [a][c]@b; wave w owns b = B0 + NW y + w
 *   phase 2 -- terms whose single index is c
 *       (A = Q[.][a][b], B = S rows c)
 *   epilogue -- for every (a, b, c) of the reference's triangle:
 *       disconnected term Z, denominator Dn, energy W (W - Z) / Dn
 *       ((fT): (W_L - Z_L) W_R / Dn), compensated FP64 sum per lane,
 *       one deterministic reduction per workgroup into partial[item];
 *       the Z and Dn operands are staged in LDS, those of (a, c) held
 *       in registers per lane.
 *
 * Operands go from the packed copies straight into the registers of the
 * wave that multiplies them.  A packed Q slab is a sequence of fragments of
 * 1 KB, 16 rows (u) x PT_KC kappa in the lane order of the MFMA operand, so
 * a fragment is one coalesced 16-byte load per lane, and since each wave
 * owns its own w (c in phase 1, b in phase 2) and the full range of the
 * other two indices, every Q fragment of a tile is loaded by exactly one
 * wave and used by both 16-row blocks of S: there is nothing in Q to share
 * through LDS.  FP64 and FP32 load S the same way and have no barrier in the
 * step loop (the two waves of a SIMD drift apart and fill each other's
 * waits); the split forms stage S in LDS panels, a barrier per eight steps.
 * Each fragment register is reloaded for the next step soon after its MFMAs.
 *   Against the kernel that staged all operands in LDS (two slots, a barrier
 * per step, one wave per 16 a x 16 b x TC c), with the launch order and the
 * later changes noted below: MFMA pipe 84 % busy instead of 67 % at rpt v=477
 * in FP64, where the card's clock then falls from 2.2 to about 2 GHz (a share of
 * the triples: 292 -> 245 ms); rpt o=20 v=120 331 -> 211 ms with 11 ms of
 * copies, FP32 upt 24/200/20/204 292 -> 184 ms, split BF16 rpt v=477 258 ->
 * 163 ms, a batch of 8 systems of v 40 to 160 198 -> 120 ms.  Bound by the
 * MFMA pipe and power in FP64 and FP32, by L2 and HBM bandwidth in the split
 * forms: at full MFMA rate a CU's four SIMDs would take 64 bytes of Q per
 * clock (16 KB per wave and 1024 MFMA cycles), all that its L1 can give; L2
 * delivers 30 to 32 bytes per clock and CU (16 to 17 TB/s), which is the .44
 * that the pipe is busy.
 *
 * Forms: FP64 (v_mfma_f64_16x16x4_f64), FP32 (v_mfma_f32_16x16x4_f32),
 * split BF16 / FP16 (hi+lo pairs, hi*hi + lo*hi + hi*lo packed into the
 * k slots of v_mfma_f32_16x16x32_{bf16,f16}, FP32 accumulation, FP64
 * epilogue).
 *
 * MFMA lane layouts (checked on gfx950): A[m][k] lane m + 16*(k/KL),
 * B[k][n] lane n + 16*(k/KL) (KL = 1 for x4, 8 consecutive k for x32);
 * D[m][n] lane n + 16*(m/4) reg m%4 for f32 results, but
 * lane n + 16*(m%4) reg m/4 for v_mfma_f64_16x16x4_f64.
 */
#ifndef LIBPT_AMD_PT_TILES_H
#define LIBPT_AMD_PT_TILES_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "pt_engine.h"

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

namespace {

template <int F> struct Form;

template <> struct Form<PT_FORM_FP64> {
	typedef double G;   /* S element in HBM */
	typedef double AE;  /* accumulator element */
	typedef v4d ACC;
	typedef double ER;  /* epilogue real */
	static constexpr int KC = 8;    /* kappa per fragment */
	static constexpr bool ROW_F64 = true, SPLIT = false, PAN = false;
	static constexpr int LAG = 1;   /* groups between use and reload */
};

template <> struct Form<PT_FORM_FP32> {
	typedef float G;
	typedef float AE;
	typedef v4f ACC;
	typedef float ER;
	static constexpr int KC = 16;
	static constexpr bool ROW_F64 = false, SPLIT = false, PAN = false;
	static constexpr int LAG = 1;   /* groups between use and reload */
};

template <> struct Form<PT_FORM_BF16X3> {
	typedef uint32_t G;  /* hi in bits 0-15, lo in bits 16-31 */
	typedef float AE;
	typedef v4f ACC;
	typedef double ER;
	static constexpr int KC = 16;
	static constexpr bool ROW_F64 = false, SPLIT = true;
	static constexpr bool PAN = true;   /* S staged in LDS panels */
	static constexpr int LAG = 2;
};

template <> struct Form<PT_FORM_F16X3> : Form<PT_FORM_BF16X3> {};

/* ---------------------------------------------------------------- MFMA */

__device__ __forceinline__ v4d
mma(double a, double b, v4d c)
{
	return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ v4f
mma(float a, float b, v4f c)
{
	return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

/* one K=32 bf16 / f16 MFMA (v_mfma_f32_16x16x32_{bf16,f16}, full rate on
 * gfx950) on operands of four 32-bit words (eight 16-bit values) per lane.
 * A and B fill their eight slots of each lane group with the same
 * (kappa, hi/lo) pattern, so each slot contributes one product of the
 * same kappa whatever the instruction's k order within the lane group. */
template <int F>
__device__ __forceinline__ v4f
mma32(v4u a, v4u b, v4f c)
{
	if constexpr (F == PT_FORM_BF16X3)
		return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
		    __builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0,
		    0, 0);
	else
		return __builtin_amdgcn_mfma_f32_16x16x32_f16(
		    __builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0,
		    0);
}

/* ---------------------------------------------------------- S operand */

/* the S fragment of a step as its MFMAs take it.  FP64, FP32: the loaded
 * words.  Split: Q fragments hold, per lane, hi k0 k1, hi k2 k3, lo k0 k1,
 * lo k2 k3 and go to the MFMA as they are; S comes as (hi, hi) for
 * hi*hi + lo*hi and (lo, 0) for hi*lo. */
template <int F>
struct SFrag {
	v4u w;
	__device__ __forceinline__ void set(v4u e, uint32_t sgn)
	{
		if constexpr (F == PT_FORM_FP64) {
			w = v4u{e[0], e[1] ^ sgn, e[2], e[3] ^ sgn};
		} else if constexpr (F == PT_FORM_FP32) {
			w = v4u{e[0] ^ sgn, e[1] ^ sgn, e[2] ^ sgn, e[3] ^ sgn};
		} else {
			/* API words hi | lo << 16 of kappa 0 .. 3 -> hi 01, hi 23,
			 * lo 01, lo 23 */
			const uint32_t s2 = sgn | (sgn >> 16);
			w = v4u{__builtin_amdgcn_perm(e[1], e[0], 0x05040100u) ^ s2,
			    __builtin_amdgcn_perm(e[3], e[2], 0x05040100u) ^ s2,
			    __builtin_amdgcn_perm(e[1], e[0], 0x07060302u) ^ s2,
			    __builtin_amdgcn_perm(e[3], e[2], 0x07060302u) ^ s2};
		}
	}
};

/* an accumulator block as one register tuple: without it the compiler splits
 * the blocks at control flow into their elements (because they start as
 * constants or are put together from LDS reads) and copies them there */
template <class ACC>
__device__ __forceinline__ void
pin(ACC &x)
{
	__asm__ volatile("" : "+v"(x));
}

/* NMF MFMAs add one Q fragment times one S fragment; part p of them.  QA:
 * Q is the A operand (rows of D), else B. */
template <int F> constexpr int NMF = F == PT_FORM_FP32 ? 4 : 2;

template <int F, bool QA>
__device__ __forceinline__ typename Form<F>::ACC
mma_part(int p, v4u q, const SFrag<F> &s, typename Form<F>::ACC c)
{
	if constexpr (F == PT_FORM_FP64) {
		const v2d x = __builtin_bit_cast(v2d, q), y = __builtin_bit_cast(v2d,
		    s.w);
		return QA ? mma(x[p], y[p], c) : mma(y[p], x[p], c);
	} else if constexpr (F == PT_FORM_FP32) {
		const v4f x = __builtin_bit_cast(v4f, q), y = __builtin_bit_cast(v4f,
		    s.w);
		return QA ? mma(x[p], y[p], c) : mma(y[p], x[p], c);
	} else {
		const v4u y = p ? v4u{s.w[2], s.w[3], 0u, 0u} :
		    v4u{s.w[0], s.w[1], s.w[0], s.w[1]};
		return QA ? mma32<F>(q, y, c) : mma32<F>(y, q, c);
	}
}

/* ---------------------------------------------------------- epilogue */

__device__ __forceinline__ void
kahan(double &s, double &cmp, double x)
{
	double y = x - cmp;
	double t = s + y;
	cmp = (t - s) - y;
	s = t;
}

/*
 * Energy terms of one lane's NB elements (a, b0 + BS y, c), y = 0 .. NB-1,
 * in y order, even y added to (esum, ecmp)[0], odd ones to [1]: the
 * disconnected term Z, the denominator Dn = d_ia + d_jb + d_kc and
 * W (W - Z) / Dn, or for two W sets (W_L - Z) W_R / Dn
 * (src/pt.c:700,927).  Everything comes from registers
 * and LDS; every element's values are made whether or not the triangle keeps
 * it, and only the sum is masked.  W values: ew[64 y] (one set; the right
 * set with two) and ew[64 (y + NB)] (the left set).  ac: the (a, c) values
 * of i_oovv and t2, [G jk, Z jk, G ik, Z ik (, G ji, Z ji)] (mixed spin: GB,
 * ZB; same spin also ji).  sbc: the same for (b, c), sbc[(32 n + BS y) TC]
 * (sbc points at this lane's b0 and c).  sav, sbv, scv: the values that
 * depend on a, b, c only, n = u i, f i, u j, f j, (same spin: u k, f k,)
 * d1 i (a), d1 j (b), d1 k (c), at sav[32 n], sbv[32 n + BS y], scv[TC n];
 * mixed spin c: u2 k, f2 k, d2 k.  sba: the (b, a) values; mixed spin: GA, ZA
 * for ji at sba[(32 n + BS y) 32]; same spin: G, Z (n & 1) for jk, ik, ji
 * (n / 2) at sba[8 NB (n / 2) + 8 y + 4 (n & 1)].
 *   Bound by latency: an element is about 20 LDS reads and 30 dependent FP64
 * operations, with one or two waves per SIMD.  Elements go in pairs, whose
 * chains interleave, and nothing in the loop comes from global memory.  Against
 * one element at a time with the same-spin (b, a) values read from global
 * memory (us or ms, same-spin / mixed-spin items): split BF16 rpt v=96 272 /
 * 1025 -> 251 / 1010 us, v=256 4.53 / 10.1 -> 4.27 / 9.95 ms; FP32 upt v=200 a
 * share 189 -> 183 ms, rpt_mp v=101 call 142 -> 136 ms; FP64 rpt v=100 1.03 /
 * 5.53 -> 0.99 / 5.52 ms, v=120 call 208 -> 206 ms.
 */
template <int F, int KIND, int NSET, int NB, int BS, int TC>
__device__ __forceinline__ void
epi_block(const pt_launch &p, int a, int c, int b0,
    const typename Form<F>::AE *ew, const typename Form<F>::ER *ac,
    const typename Form<F>::ER *sav, const typename Form<F>::ER *sbv,
    const typename Form<F>::ER *scv, const typename Form<F>::ER *sbc,
    const typename Form<F>::ER *sba, double (&esum)[2], double (&ecmp)[2])
{
	typedef typename Form<F>::ER ER;
	const ER s0 = (ER)p.inv_scale[0], s1 = (ER)p.inv_scale[1];
	/* W (W - Z) or the two-set form of element h, over Dn, into the sum */
	auto add = [&](int y, int h, bool in, ER z, ER dn) {
		ER t;
		if constexpr (NSET == 1) {
			ER w = (ER)ew[64 * (y + h)];
			if (Form<F>::SPLIT)
				w *= s0;
			t = w * (w - z) / dn;
		} else {
			ER wl = (ER)ew[64 * (y + h + NB)], wr = (ER)ew[64 * (y + h)];
			if (Form<F>::SPLIT) {
				wl *= s0;
				wr *= s1;
			}
			t = (wl - z) * wr / dn;
		}
		double s = esum[h], e = ecmp[h];
		kahan(s, e, (double)t);
		esum[h] = in ? s : esum[h];
		ecmp[h] = in ? e : ecmp[h];
	};
	const ER uia = sav[0], fia = sav[32], uja = sav[64], fja = sav[96];
	if constexpr (KIND == PT_AAA) {
		/* src/pt.c:162-175, for (u, G) = (t1 or l1, i_oovv) and
		 * (f, Z) = (f_ov or f2_ov, t2 or l2) */
		const ER uka = sav[128], fka = sav[160], dia = sav[192];
		const ER uic = scv[0], fic = scv[TC], ujc = scv[2 * TC];
		const ER fjc = scv[3 * TC], ukc = scv[4 * TC], fkc = scv[5 * TC];
		const ER dkc = scv[6 * TC];
#pragma unroll 1
		for (int y = 0; y < NB; y += 2) {
			ER zu[2], zf[2], dn[2];
#pragma unroll
			for (int h = 0; h < 2; ++h) {
				const ER *bc = sbc + BS * (y + h) * TC;
				zu[h] = uia * bc[0] - uja * bc[64 * TC] - uka * bc[128 * TC];
				zf[h] = fia * bc[32 * TC] - fja * bc[96 * TC] -
				    fka * bc[160 * TC];
			}
#pragma unroll
			for (int h = 0; h < 2; ++h) {
				const ER *bv = sbv + BS * (y + h);
				zu[h] = zu[h] - bv[0] * ac[0] + bv[64] * ac[2] +
				    bv[128] * ac[4];
				zf[h] = zf[h] - bv[32] * ac[1] + bv[96] * ac[3] +
				    bv[160] * ac[5];
				dn[h] = dia + bv[192] + dkc;
			}
#pragma unroll
			for (int h = 0; h < 2; ++h) {
				const ER *ba = sba + 8 * (y + h);
				zu[h] = zu[h] - uic * ba[0] + ujc * ba[8 * NB] +
				    ukc * ba[16 * NB];
				zf[h] = zf[h] - fic * ba[4] + fjc * ba[8 * NB + 4] +
				    fkc * ba[16 * NB + 4];
			}
#pragma unroll
			for (int h = 0; h < 2; ++h) {
				const int b = b0 + BS * (y + h);
				add(y, h, a > b && b > c, zu[h] + zf[h], dn[h]);
			}
		}
	} else {
		/* src/pt.c:177-185 and :433-442 */
		const ER dia = sav[128];
		const ER u2c = scv[0], f2c = scv[TC], dkc = scv[2 * TC];
#pragma unroll 1
		for (int y = 0; y < NB; y += 2) {
			ER z[2], dn[2];
#pragma unroll
			for (int h = 0; h < 2; ++h) {
				const int bb = BS * (y + h);
				const ER uib = sbv[bb], fib = sbv[32 + bb];
				const ER ujb = sbv[64 + bb], fjb = sbv[96 + bb];
				const ER gjkbc = sbc[bb * TC], zjkbc = sbc[(32 + bb) * TC];
				const ER gikbc = sbc[(64 + bb) * TC];
				const ER zikbc = sbc[(96 + bb) * TC];
				const ER gjiba = sba[bb * 32], zjiba = sba[(32 + bb) * 32];
				z[h] = (uia * gjkbc + fia * zjkbc)
				    - (uib * ac[0] + fib * ac[1])
				    - (uja * gikbc + fja * zikbc)
				    + (ujb * ac[2] + fjb * ac[3])
				    + (u2c * gjiba + f2c * zjiba);
				dn[h] = dia + sbv[128 + bb] + dkc;
			}
#pragma unroll
			for (int h = 0; h < 2; ++h)
				add(y, h, a > b0 + BS * (y + h), z[h], dn[h]);
		}
	}
}

/* values the whole wave shares: readfirstlane tells the compiler so, which
 * keeps them (and everything derived from them) in scalar registers */
__device__ __forceinline__ int
uni(int x)
{
	return __builtin_amdgcn_readfirstlane(x);
}

__device__ __forceinline__ int64_t
uni64(int64_t x)
{
	const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
	const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
	return (int64_t)(((uint64_t)hi << 32) | lo);
}

/* buffer descriptors: loads at offsets at or beyond the descriptor's byte
 * count return zero, which handles tile edges, invalid pairs and the kappa
 * tail without branches */
__device__ __forceinline__ __amdgpu_buffer_rsrc_t
brsrc(const void *base, int64_t bytes)
{
	const int nrec = bytes <= 0 ? 0 : bytes > 0x7fffffff ? 0x7fffffff :
	    (int)bytes;
	return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, nrec,
	    0x00020000);
}

#define PT_OOR 0x80000000u  /* an offset every descriptor rejects */

/* buffer store / load of one accumulator value at lane offset vofs plus a
 * constant offset sofs: the constant goes to a scalar register, so a run of
 * them costs no vector registers for addresses */
template <class AE>
__device__ __forceinline__ void
bstore_ae(__amdgpu_buffer_rsrc_t r, uint32_t vofs, int sofs, AE v)
{
	if constexpr (sizeof(AE) == 8)
		__builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r,
		    (int)vofs, sofs, 0);
	else
		__builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t,
		    v), r, (int)vofs, sofs, 0);
}

template <class AE>
__device__ __forceinline__ AE
bload_ae(__amdgpu_buffer_rsrc_t r, uint32_t vofs, int sofs)
{
	if constexpr (sizeof(AE) == 8)
		return __builtin_bit_cast(AE,
		    __builtin_amdgcn_raw_buffer_load_b64(r, (int)vofs, sofs, 0));
	else
		return __builtin_bit_cast(AE,
		    __builtin_amdgcn_raw_buffer_load_b32(r, (int)vofs, sofs, 0));
}



/* ------------------------------------------------------ terms of an item */

/* one term of the item's tile, in LDS, made once per item by one thread
 * each; every field is read as a wave-uniform value */
struct TermP {
	uint64_t q[2];    /* chunk 0 of the two u blocks at the tile's first w */
	uint64_t s;       /* S element (row 0, kappa 0) */
	uint32_t dq[2];   /* bytes from one chunk to the next */
	uint32_t xa, xb;  /* bytes from w to w + 1 and, over 16 w, w + 16 */
	uint32_t sst;     /* bytes between S rows */
	uint32_t sbytes;  /* bytes of the S rows from s */
	int32_t nch;      /* kappa chunks */
	uint32_t sgn;     /* sign bit to flip in S */
	uint32_t lst;     /* Q bytes from a lane's u to u + 1, and << 16 from one
	                     quarter of a row to the next */
	int32_t lim;      /* u of the tile that have data (above 32: all) */
};

/* the term's addresses for the tile (A0, B0, C0).  A packed slab is
 * [row block of 16][chunk][column][fragment of 64 fr bytes]: rows u and
 * columns w, or (tr) rows w and columns u; tri: columns 0 .. 16 (block + 1) -
 * 1 only. */
template <int F>
__device__ __forceinline__ void
make_term(const pt_launch &p, const pt_term &t, int i, int j, int k, int A0,
    int B0, int C0, TermP &o)
{
	constexpr int ES = (int)sizeof(typename Form<F>::G);
	const int na = p.na, nc = p.nc;
	const int u0 = t.role == PT_ROLE_A ? B0 : A0;
	const int w0 = t.role == PT_ROLE_C ? B0 : C0;
	const int fb = 64 * t.fr;
	const char *qb = (const char *)p.buf[t.q_buf] + t.q_off[0] * i +
	    t.q_off[1] * j + t.q_off[2] * k;
	for (int e = 0; e < 2; ++e) {
		const int64_t ub = u0 / 16 + e;
		int64_t off, cols;
		if (t.tri) {
			off = t.nch * 8 * ub * (ub + 1) + w0;
			cols = 16 * (ub + 1);
		} else if (t.tr) {
			off = (int64_t)(w0 / 16) * t.nch * t.cols + 16 * ub;
			cols = t.cols;
		} else {
			off = ub * t.nch * t.cols + w0;
			cols = t.cols;
		}
		o.q[e] = (uint64_t)qb + fb * (uint64_t)off;
		o.dq[e] = (uint32_t)(fb * cols);
	}
	o.xa = t.tr ? 16 : fb;
	o.xb = t.tr ? (uint32_t)((int64_t)t.nch * t.cols * fb) : 16 * fb;
	o.s = (uint64_t)p.buf[t.s_buf] + ES * (uint64_t)(t.s_off[0] * i +
	    t.s_off[1] * j + t.s_off[2] * k);
	o.sst = (uint32_t)(t.s_st * ES);
	const int64_t sb = (t.role == PT_ROLE_C ? nc : na) * t.s_st * ES;
	o.sbytes = (uint32_t)(sb > 0x7fffffff ? 0x7fffffff : sb);
	o.nch = t.nch;
	o.sgn = t.sign < 0 ? 0x80000000u : 0u;
	/* lane (u, quarter): row u of the fragment, or (tr) column u */
	o.lst = (t.tr ? fb : 16) | (uint32_t)(16 * t.fr) << 16;
	o.lim = t.tr ? na - u0 : t.fr < 16 ? t.fr : 32;
}

/*
 * The terms [t0, t1) of one role, over all their kappa chunks, added to the
 * accumulators.  The wave owns w = w0 + NW x + wave, x = 0 .. NX-1, of the
 * tile; per chunk it holds the fragments (x, u block e) and the NSB S
 * blocks; B::id(x, e, s) is the accumulator block of a fragment and an S
 * block.  mask: the blocks that hold an element of the triangle inside the
 * extents; they are computed in groups (half of x, e, s), and a group
 * without any is skipped, so that the tiles cut by the diagonal or by the
 * end of an index pay for 16 x 16 blocks and not for whole tiles.  The
 * fragments that serve a block of the mask are a range of x for each e;
 * those outside it may not exist, so the nearest one of the range is read
 * in their place (their blocks are never used).
 *
 * Step n = (term, chunk).  A step's MFMAs go in four groups (half of x, e);
 * a group's fragments are loaded for the next step LAG groups after their
 * MFMAs, so 4 - LAG groups of loads are in flight per wave; the loads after
 * the last step are all out of range and return zero.
 *   How far ahead decides how the workgroups of an XCD share its L2.  With a
 * whole step to arrive even loads that miss L2 are hidden, and workgroups
 * that read the same slabs drift apart until each fetches them for itself;
 * with less, the first one waits for HBM, the ones behind it hit and catch
 * up, and they run together.  The split forms, bound by L2 and HBM, take
 * LAG = 2: rpt v=477 split-BF16 209 -> 165 to 177 ms for 0 -> 2 (3: 216 ms, its
 * hits wait too); rft v=300 F16X3 92 ms for either (3: 116 ms).  FP64 and
 * FP32 take 1, from 0: within 1 % everywhere (2: v=120 FP64 211 -> 216 ms).
 *
 * S is the same for all waves, and its rows are scattered 64-byte pieces in
 * the API layout: loaded by each wave for itself, a 16-row block costs the
 * vector cache as much as four Q fragments.  FP64 and FP32, whose steps take
 * 2048 and 4096 MFMA cycles, do that.  In the split forms (1024 cycles) S
 * was a third of the cache accesses and a sixth of the L2 requests, so there
 * the waves stage it together in LDS (PAN), in panels of PC
 * steps: while a panel is used, each wave loads its NI fragments of the next
 * one into registers; they go to the other of two buffers at the panel's
 * end, behind the only barrier of the loop.  A fragment is [row][quarter ^
 * (row / 4)] in 16-byte pieces: the four lanes of a row load 64 contiguous
 * bytes, and the 16 lanes of a read phase (rows at one quarter) fall on
 * distinct banks.  rft v=300 F16X3 101 -> 92 ms, rpt v=477 split-BF16 210 ->
 * 206 ms (128 mixed-spin ijk of it 235 -> 259 TFLOP/s); in FP64 it gave
 * nothing at v=477 and cost 2 to 4 % at v=64 to 160, where the barriers
 * couple the waves.
 *
 * One loop serves full and cut tiles: with loop variants chosen by control
 * flow the accumulators, more than half of the registers, meet at joins
 * after every variant, and the register allocator then spills dozens of
 * blocks there and inside the loops.
 */
constexpr int PC = 8;               /* steps per S panel */
constexpr int PANEL = PC * 2 * 1024; /* bytes, for two S blocks */

/* a barrier that waits for this wave's LDS accesses only (the compiler's
 * waits for every global load in flight too) */
__device__ __forceinline__ void
lds_barrier()
{
	__asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
	__builtin_amdgcn_s_barrier();
	__asm__ volatile("" ::: "memory");
}

/* the x next to x in lo .. hi; of an empty range (lo > hi = -1) its lo: the
 * scalar offset of a load is made from it, and must not be negative */
constexpr int
near_x(int x, int lo, int hi)
{
	return (x > hi ? hi : x) < lo ? lo : x > hi ? hi : x;
}

static_assert(near_x(0, 3, -1) == 3 && near_x(3, 3, -1) == 3, "empty range");
static_assert(near_x(0, 1, 2) == 1 && near_x(3, 1, 2) == 2 &&
    near_x(2, 1, 3) == 2, "nearest");

/* orders LDS accesses of the lanes of a wave (which runs them in program
 * order: no instruction, but the compiler keeps to it) */
__device__ __forceinline__ void
wave_sync()
{
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
}

/* panels: two panel buffers; par: the one to fill first, updated (the
 * previous call's last panel may still be read from the other) */
template <int F, int NW, int NX, int NSB, int ROLE, class B, int NACC>
__device__ __forceinline__ void
run_terms(typename Form<F>::ACC (&acc)[NACC], const TermP *tp, int t0, int t1,
    int s0, int sext, int wave, int ln, int lg, uint32_t mask, char *panels,
    int &par)
{
	static_assert(Form<F>::KC * sizeof(typename Form<F>::G) == 64,
	    "a chunk of S is 64 bytes per row");
	constexpr bool QA = ROLE != PT_ROLE_A;
	constexpr int XB = 16 / NW;      /* x per 16 w */
	/* panel fragments (step, S block) are dealt to the waves in order */
	constexpr bool PAN = Form<F>::PAN;
	constexpr int LAG = Form<F>::LAG;
	constexpr int NI = PAN ? PC * NSB / NW : NSB, ND = NW / NSB;
	static_assert(PC * NSB % NW == 0 && NW % NSB == 0, "panel split");
	if (t0 >= t1)
		return;
	uint64_t q0, q1;
	uint32_t dq0, dq1, xa, xb, sgn;
	int left;
	bool more = true;
	uint32_t vo[2];
	/* the x of each e that may be read (xhi < 0: none), the groups */
	constexpr int NH = NX / 2;
	int xlo[2], xhi[2];
	uint32_t grp = 0;
#pragma unroll
	for (int e = 0; e < 2; ++e) {
		xlo[e] = NX - 1;
		xhi[e] = -1;
#pragma unroll
		for (int x = 0; x < NX; ++x)
#pragma unroll
			for (int s = 0; s < NSB; ++s)
				if (mask >> B::id(x, e, s) & 1) {
					xlo[e] = x < xlo[e] ? x : xlo[e];
					xhi[e] = x;
					grp |= 1u << ((x / NH * 2 + e) * NSB + s);
				}
		xlo[e] = uni(xlo[e]);
		xhi[e] = uni(xhi[e]);
	}
	grp = (uint32_t)uni((int)grp);
	/* scalars and lane offsets of term t */
	auto term = [&](int t) {
		const TermP &T = tp[t];
		q0 = (uint64_t)uni64((int64_t)T.q[0]);
		q1 = (uint64_t)uni64((int64_t)T.q[1]);
		dq0 = (uint32_t)uni((int)T.dq[0]);
		dq1 = (uint32_t)uni((int)T.dq[1]);
		xa = (uint32_t)uni((int)T.xa);
		xb = (uint32_t)uni((int)T.xb);
		sgn = (uint32_t)uni((int)T.sgn);
		left = uni(T.nch);
		const uint32_t lst = (uint32_t)uni((int)T.lst);
		const int lim = uni(T.lim);
		q0 += (uint64_t)xa * (uint32_t)wave;
		q1 += (uint64_t)xa * (uint32_t)wave;
#pragma unroll
		for (int e = 0; e < 2; ++e)
			vo[e] = xhi[e] < 0 || 16 * e + ln >= lim ? PT_OOR :
			    __umul24(lst & 0xffff, ln) + __umul24(lst >> 16, lg);
	};
	/* lanes without data take an offset that every descriptor rejects; the
	 * scalar offset is never relied on for a range check */
	auto load_q = [&](int x, int e) {
		x = near_x(x, xlo[e], xhi[e]);
		const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
		    (void *)(e ? q1 : q0), (short)0, 0x7fffffff, 0x00020000);
		return __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(r,
		    (int)vo[e], (int)((uint32_t)(x % XB) * NW * xa +
		    (uint32_t)(x / XB) * xb), 0));
	};
	/* S loads.  PAN: panel staging, this wave's S block, and its next step
	 * as (term st, chunk sc).  Else both blocks of the next step. */
	const int lane = 16 * lg + ln, se = PAN ? wave % NSB : 0;
	const int srow = s0 + 16 * se + (PAN ? lane >> 2 : ln);
	const uint32_t sq = 16u * (PAN ? (lane & 3) ^ (lane >> 4) : lg);
	int st = t0, sc = PAN ? wave / NSB : 0, snch, sbytes;
	uint64_t sp;
	uint32_t so[PAN ? 1 : NSB];
	auto sterm = [&]() {
		const TermP &T = tp[st];
		sp = (uint64_t)uni64((int64_t)T.s);
		sbytes = uni((int)T.sbytes);
		snch = uni(T.nch);
		const uint32_t sst = (uint32_t)uni((int)T.sst);
#pragma unroll
		for (int e = 0; e < (PAN ? 1 : NSB); ++e)
			so[e] = srow + 16 * e < sext ?
			    (uint32_t)(srow + 16 * e) * sst + sq : PT_OOR;
	};
	v4u sr[NI];
	auto stage_load = [&]() {
#pragma unroll
		for (int i = 0; i < NI; ++i) {
			if (PAN || i == 0)
				while (sc >= snch && st < t1) {
					sc -= snch;
					if (++st < t1) {
						sterm();
					} else {
#pragma unroll
						for (int e = 0; e < (PAN ? 1 : NSB); ++e)
							so[e] = PT_OOR;
					}
				}
			const int at = 64 * sc;   /* KC elements of S per chunk */
			const __amdgpu_buffer_rsrc_t r =
			    __builtin_amdgcn_make_buffer_rsrc((void *)(sp + at),
			    (short)0, sbytes > at ? sbytes - at : 0, 0x00020000);
			sr[i] = __builtin_bit_cast(v4u,
			    __builtin_amdgcn_raw_buffer_load_b128(r,
			    (int)so[PAN ? 0 : i], 0, 0));
			if (PAN)
				sc += ND;
		}
		if (!PAN)
			++sc;
	};
	auto stage_write = [&]() {
		char *d = panels + par * PANEL + 1024 * wave + 16 * lane;
#pragma unroll
		for (int i = 0; i < NI; ++i)
			*(v4u *)(d + 1024 * NW * i) = sr[i];
	};
	const uint32_t rofs = 16u * (4 * ln + (lg ^ (ln >> 2)));

	term(t0);
	sterm();
	int t = t0, n = 0;
	stage_load();
	v4u q[2 * NX];
	/* the fragments of group g = (half of x, e) */
	auto load_g = [&](int g) {
#pragma unroll
		for (int x = (g >> 1) * NH; x < ((g >> 1) + 1) * NH; ++x)
			q[2 * x + (g & 1)] = load_q(x, g & 1);
	};
#pragma unroll
	for (int g = 0; g < 4 - LAG; ++g)
		load_g(g);
	if constexpr (PAN) {
		stage_write();
		lds_barrier();
		stage_load();
	}
	do {
		SFrag<F> s[NSB];
#pragma unroll
		for (int e = 0; e < NSB; ++e)
			s[e].set(PAN ? *(const v4u *)(panels + par * PANEL + rofs +
			    1024 * (NSB * n + e)) : sr[e], sgn);
		if constexpr (!PAN)
			stage_load();
#pragma unroll
		for (int g = 0; g < 4; ++g) {
			const int h = g >> 1, e = g & 1;
#pragma unroll
			for (int b = 0; b < NSB; ++b)
				if (grp >> (g * NSB + b) & 1) {
#pragma unroll
					for (int m = 0; m < NMF<F>; ++m)
#pragma unroll
					for (int x = h * NH; x < (h + 1) * NH; ++x) {
						const int a = B::id(x, e, b);
						acc[a] = mma_part<F, QA>(m, q[2 * x + e], s[b],
						    acc[a]);
					}
				}
			if (g == LAG) {
				/* on to the next step */
				if (--left > 0) {
					q0 += dq0;
					q1 += dq1;
				} else if (++t < t1) {
					term(t);
				} else {
					more = false;
					vo[0] = vo[1] = PT_OOR;
				}
			}
			load_g((g + 4 - LAG) & 3);
			__builtin_amdgcn_sched_barrier(0);
		}
		if (PAN && ++n == PC) {
			n = 0;
			par ^= 1;
			if (more) {
				stage_write();
				lds_barrier();
				stage_load();
			}
		}
	} while (more);
	if (n != 0)
		par ^= 1;
}

/* -------------------------------------------------------------- kernel */

/*
 * Workgroup geometry, per wave count NW (pt_tcw, pt_cw in pt_engine.h give
 * the same numbers to the host).  Tile 32 a x 32 b x TC c; CW = TC / NW c
 * per wave in phase 1, BW = 32 / NW b per wave in phase 2, NACC 16 x 16
 * blocks per wave in either.
 *   NW = 4: TC = 32 for FP32 and the split forms (32 FP32 blocks of 4
 *           registers), 16 for FP64 (16 blocks of 8 registers): 128
 *           accumulator registers, two workgroups per CU (two waves per
 *           SIMD).
 *   NW = 8: TC = 32, one workgroup per CU.
 */
template <int F, int NSET, int NW>
struct Geo {
	static constexpr int TC = NW == 8 || F != PT_FORM_FP64 ? 32 : 16;
	static constexpr int CW = TC / NW, BW = 32 / NW, NCB = TC / 16;
	static constexpr int NACC = 4 * CW;
	static constexpr int THREADS = 64 * NW;
	static constexpr int WG_PER_CU = NW == 8 ? 1 : 2;
	/* accumulator block of phase 1 (c of the wave, a block, b block) and
	 * of phase 2 (b of the wave, a block, c block).  In either, bit 1 is
	 * the a block, so the transpose of an a block stays in its blocks. */
	static constexpr int blk1(int x, int ab, int bb)
	{
		return (2 * x + ab) * 2 + bb;
	}
	static constexpr int blk2(int y, int ab, int cb)
	{
		return NCB == 2 ? (2 * y + ab) * 2 + cb :
		    (2 * (y >> 1) + ab) * 2 + (y & 1);
	}
};

/* accumulator block of (x, u block, S block) for each role */
template <class GM> struct RoleA {
	static constexpr int id(int x, int e, int s) { return GM::blk1(x, s, e); }
};

template <class GM> struct RoleB {
	static constexpr int id(int x, int e, int s) { return GM::blk1(x, e, s); }
};

template <class GM> struct RoleC {
	static constexpr int id(int y, int e, int s) { return GM::blk2(y, e, s); }
};

/*
 * LDS of one item: the term table, the waves' sums, and one area used in
 * turn for the S panels, the transpose's two buffers (of TRC (a block,
 * register) columns each) and the epilogue's W columns and staged operands.
 */
template <int F, int KIND, int NSET, int NW>
struct Lds {
	typedef Geo<F, NSET, NW> GM;
	static constexpr bool same = KIND == PT_AAA;
	static constexpr int TC = GM::TC, AES = (int)sizeof(typename Form<F>::AE);
	static constexpr int ERS = (int)sizeof(typename Form<F>::ER);
	static constexpr int NTERM = NSET * (same ? PT_TERMS_SAME :
	    PT_TERMS_MIXED);
	static constexpr int TRW = TC + 1, TRC = 2;
	static constexpr int TRB = TRC * 4 * 32 * TRW;  /* values per buffer */
	static constexpr int NPB = same ? 6 : 4;        /* (b, c) blocks */
	static constexpr int NBC = NPB * 32 * TC, NBV = (NPB + 1) * 32;
	static constexpr int NCV = (same ? NPB + 1 : 3) * TC;  /* c vectors */
	static constexpr int NCOL = 24 * GM::BW;  /* a wave's (b, a) values */
	static constexpr int NBA = same ? NW * NCOL : 2 * 32 * 32;
	static constexpr int EBYTES = NW * NSET * GM::BW * 64 * AES;
	static constexpr int B1 = 2 * TRB * AES;
	static constexpr int B2 = EBYTES + (NBC + 2 * NBV + NCV + NBA) * ERS;
	static constexpr int RED = NTERM * (int)sizeof(TermP);
	static constexpr int MEM = (RED + 8 * NW + 15) / 16 * 16;
	static constexpr int BYTES = MEM + (B1 > B2 ? B1 : B2);
	static_assert(B1 >= 2 * PANEL, "the S panels");
	static_assert(BYTES * GM::WG_PER_CU <= 160 * 1024 - 256,
	    "LDS of the workgroups of a CU");
	static_assert(NBC % GM::THREADS == 0 && NTERM <= GM::THREADS &&
	    (same || NBA % GM::THREADS == 0),
	    "staging by whole passes of the workgroup");
};

/*
 * One work item (ijk, tile) of a spin case: everything between reading the
 * item and writing its energy to partial[it].  KIND is the spin case,
 * PT_AAA or PT_AAB.  With two W sets the sets are formed one after the
 * other; wsv is the item's save area for W of set 0 (4 NACC values per lane
 * per wave); lds: Lds::BYTES.  keep false: the energy is not written (and
 * wsv is null: what goes to the save area is dropped).
 */
template <int F, int KIND, int NSET, int NW>
__device__ __forceinline__ void
tile_item(const pt_launch &p, int64_t it, typename Form<F>::AE *wsv,
    char *lds, bool keep = true)
{
	typedef Form<F> FM;
	typedef Geo<F, NSET, NW> GM;
	typedef typename FM::AE AE;
	typedef typename FM::ACC ACC;
	typedef typename FM::ER ER;
	constexpr int TC = GM::TC, CW = GM::CW, BW = GM::BW, NCB = GM::NCB;
	constexpr int NACC = GM::NACC, NT = GM::THREADS;
	constexpr bool same = KIND == PT_AAA;

	typedef Lds<F, KIND, NSET, NW> LD;
	constexpr int TRW = LD::TRW, TRC = LD::TRC, TRB = LD::TRB;
	constexpr int NPB = LD::NPB, NBC = LD::NBC, NBV = LD::NBV, NBA = LD::NBA;
	constexpr int NCV = LD::NCV, NCOL = LD::NCOL;
	constexpr int EBYTES = LD::EBYTES, NTERM = LD::NTERM;
	TermP *const tp = (TermP *)lds;
	double *const red = (double *)(lds + LD::RED);
	char *const smem = lds + LD::MEM;

	const int tid = threadIdx.x % NT, lane = tid & 63;
	const int wave = uni(tid >> 6);
	const int ln = lane & 15, lg = lane >> 4;

	const int64_t ijk_id = it / p.n_tiles;
	const int tile = (int)(it - ijk_id * p.n_tiles);
	const int i = p.ijk[3 * ijk_id], j = p.ijk[3 * ijk_id + 1];
	const int k = p.ijk[3 * ijk_id + 2];
	const int A0 = p.tiles[3 * tile] * 32, B0 = p.tiles[3 * tile + 1] * 32;
	const int C0 = p.tiles[3 * tile + 2] * TC;
	const int na = p.na, nc = p.nc;

	if (tid < NTERM)
		make_term<F>(p, p.terms[tid], i, j, k, A0, B0, C0, tp[tid]);

	/* accumulator blocks that hold an element of the triangle, a bit each:
	 * a > b, and b > c for the same-spin case */
	uint32_t m1 = 0, m2 = 0;
#pragma unroll
	for (int ab = 0; ab < 2; ++ab) {
		const int a0 = A0 + 16 * ab, a1 = (a0 + 16 < na ? a0 + 16 : na) - 1;
#pragma unroll
		for (int x = 0; x < CW; ++x)
#pragma unroll
			for (int bb = 0; bb < 2; ++bb) {
				const int b0 = B0 + 16 * bb, c = C0 + NW * x + wave;
				const int b1 = (b0 + 16 < na ? b0 + 16 : na) - 1;
				if (a0 < na && b0 < na && c < nc && a1 > b0 &&
				    (!same || b1 > c))
					m1 |= 1u << GM::blk1(x, ab, bb);
			}
#pragma unroll
		for (int y = 0; y < BW; ++y)
#pragma unroll
			for (int cb = 0; cb < NCB; ++cb) {
				const int b = B0 + NW * y + wave, c0 = C0 + 16 * cb;
				if (a0 < na && b < na && c0 < nc && a1 > b &&
				    (!same || b > c0))
					m2 |= 1u << GM::blk2(y, ab, cb);
			}
	}
	m1 = (uint32_t)uni((int)m1);
	m2 = (uint32_t)uni((int)m2);
	ACC acc[NACC];
#pragma unroll
	for (int x = 0; x < NACC; ++x)
		acc[x] = ACC{0, 0, 0, 0};
#pragma unroll
	for (int x = 0; x < NACC; ++x)
		pin(acc[x]);
	/* save area of W set 0: value (r, x) of (wave, lane) at element
	 * ((r NACC + x) NW + wave) 64 + lane */
	constexpr int WST = NW * 64 * (int)sizeof(AE);
	const __amdgpu_buffer_rsrc_t wr = brsrc(wsv, NSET == 2 && wsv ?
	    (int64_t)4 * NACC * WST : 0);
	const uint32_t wvo = (uint32_t)((wave * 64 + lane) * sizeof(AE));

	/* terms of one W set: role a, role b, role c; set 1 follows set 0 */
	const int nset_terms = uni(p.nterm1 + p.nterm2);
	const int nta = uni(p.nterm_a), nt1 = uni(p.nterm1);
	__syncthreads();

	/* [a][b]@c -> [a][c]@b: per (a block, register) a 32 b x TC c matrix
	 * for each of the four lane groups, TRC of them per barrier */
	auto transpose = [&]() {
		AE *X = (AE *)smem;
#pragma unroll
		for (int g = 0; g < 8 / TRC; ++g) {
			AE *Y = X + (g & 1) * TRB + lg * 32 * TRW;
#pragma unroll
			for (int h = 0; h < TRC; ++h) {
				const int ab = (g * TRC + h) >> 2, r = (g * TRC + h) & 3;
#pragma unroll
				for (int x = 0; x < CW; ++x)
#pragma unroll
					for (int bb = 0; bb < 2; ++bb)
						Y[h * 4 * 32 * TRW + (16 * bb + ln) * TRW +
						    NW * x + wave] = acc[GM::blk1(x, ab, bb)][r];
			}
			__syncthreads();
#pragma unroll
			for (int h = 0; h < TRC; ++h) {
				const int ab = (g * TRC + h) >> 2, r = (g * TRC + h) & 3;
#pragma unroll
				for (int y = 0; y < BW; ++y)
#pragma unroll
					for (int cb = 0; cb < NCB; ++cb)
						acc[GM::blk2(y, ab, cb)][r] =
						    Y[h * 4 * 32 * TRW + (NW * y + wave) * TRW +
						    16 * cb + ln];
			}
		}
		__syncthreads();
#pragma unroll
		for (int x = 0; x < NACC; ++x)
			pin(acc[x]);
	};

	int par = 0;   /* S panel buffer */
#pragma unroll 1
	for (int s = 0; s < NSET; ++s) {
		const int ts = s * nset_terms;
		/* a wave without any block has no terms to walk (with panels it
		 * stages its part all the same) */
		const bool w1 = m1 || FM::PAN, w2 = m2 || FM::PAN;
		run_terms<F, NW, CW, 2, PT_ROLE_A, RoleA<GM>>(acc, tp, ts,
		    ts + (w1 ? nta : 0), A0, na, wave, ln, lg, m1, smem, par);
		run_terms<F, NW, CW, 2, PT_ROLE_B, RoleB<GM>>(acc, tp, ts + nta,
		    ts + (w1 ? nt1 : nta), B0, na, wave, ln, lg, m1, smem, par);
		if (FM::PAN)
			lds_barrier();   /* the last panel's reads */
		transpose();
		run_terms<F, NW, BW, NCB, PT_ROLE_C, RoleC<GM>>(acc, tp, ts + nt1,
		    ts + (w2 ? nset_terms : nt1), C0, nc, wave, ln, lg, m2, smem,
		    par);
		if (NSET == 2 && s == 0) {
			/* W of set 0 to the save area, lane-contiguous per (r, x,
			 * wave); the accumulators restart for set 1 */
#pragma unroll
			for (int r = 0; r < 4; ++r)
#pragma unroll
				for (int x = 0; x < NACC; ++x) {
					bstore_ae<AE>(wr, wvo, (r * NACC + x) * WST,
					    acc[x][r]);
					acc[x][r] = 0;
				}
#pragma unroll
			for (int x = 0; x < NACC; ++x)
				pin(acc[x]);
		}
	}

	/* epilogue: layout [a][c]@b; the lane holds c = C0 + 16 cb + ln.  Each
	 * (register, a block, c block) column of BW b goes through the lane's
	 * own LDS slots, so that the element loop runs with a runtime index. */
	double esum[2] = {0.0, 0.0}, ecmp[2] = {0.0, 0.0};
	AE *E = (AE *)smem + wave * (NSET * BW * 64) + lane;
	/* the tile's epilogue operands, staged in LDS behind the W values: the
	 * (b, c) blocks of i_oovv and t2, [G jk, Z jk, G ik, Z ik (, G ji, Z
	 * ji)][32 b][TC c] (mixed spin: the GB, ZB blocks; same spin: GA, ZA with
	 * ji), the vectors [u i, f i, u j, f j, (u k, f k,) d1][32] of a (d1 i)
	 * and b (d1 j), those of c (same spin: the same, d1 k; mixed: u2 k, f2 k,
	 * d2 k), and the (b, a) blocks: for the mixed spin case those of the
	 * same-spin arrays for ji, [GA, ZA][32 b][32 a]; the six of the same-spin
	 * case do not fit, so each wave keeps the values of one (a block,
	 * register) at a time, [jk, ik, ji][BW b][G, Z][4 a], loaded one ahead.
	 * Rows and columns beyond the arrays repeat the last one; the epilogue
	 * masks those elements. */
	if (FM::PAN)
		lds_barrier();   /* the last panel's reads */
	ER *const stg = (ER *)(smem + EBYTES);
	ER *const sva = stg + NBC + NBV, *const svc = sva + NBV;
	ER *const sab = svc + NCV;
	const ER *sbc = stg + wave * TC + ln;
	const ER *sbv = stg + NBC + wave;
	/* block n: (G, Z)[n & 1] of pair n / 2 = jk, ik (, ji); mixed spin: rows
	 * (jk + b) vb, same spin: jk + b v, v = vb */
	const ER *G = (const ER *)(same ? p.epi.GA : p.epi.GB);
	const ER *Z = (const ER *)(same ? p.epi.ZA : p.epi.ZB);
	const int64_t po = same ? p.oa : p.ob;
	const int64_t pr = same ? p.va * p.va : p.va * p.vb;
	const int64_t pjk = ((int64_t)j * po + k) * pr;
	const int64_t pik = ((int64_t)i * po + k) * pr;
	const int64_t pji = ((int64_t)j * p.oa + i) * pr;
	{
#pragma unroll
		for (int q = 0; q < NBC / NT; ++q) {
			const int n = tid + q * NT;
			const int arr = n / (32 * TC), bl = (n / TC) % 32, cl = n % TC;
			const int b = B0 + bl < na ? B0 + bl : na - 1;
			const int c = C0 + cl < nc ? C0 + cl : nc - 1;
			const int64_t pb = arr < 2 ? pjk : arr < 4 ? pik : pji;
			stg[n] = ((arr & 1) ? Z : G)[pb + (int64_t)b * p.vb + c];
		}
		/* vector n: (u, f)[n & 1] at occupied index (i, j, k)[n / 2], the
		 * last one d1 */
		const ER *u1 = (const ER *)p.epi.u1, *u2 = (const ER *)p.epi.u2;
		const ER *f1 = (const ER *)p.epi.f1, *f2 = (const ER *)p.epi.f2;
		const ER *d1 = (const ER *)p.epi.d1, *d2 = (const ER *)p.epi.d2;
		for (int n = tid; n < 2 * NBV + NCV; n += NT) {
			const bool of_c = n >= 2 * NBV, of_a = !of_c && n >= NBV;
			const int m = of_c ? n - 2 * NBV : of_a ? n - NBV : n;
			const int arr = of_c ? m / TC : m / 32;
			const int l = of_c ? C0 + m % TC : (of_a ? A0 : B0) + m % 32;
			const int top = (of_c ? nc - 1 : na - 1), x = l < top ? l : top;
			const int64_t d1r = of_c ? k : of_a ? i : j;
			const int64_t r1 = arr < 2 ? i : arr < 4 ? j : k;
			const ER *src = (arr & 1) ? f1 + r1 * p.va : u1 + r1 * p.va;
			if (arr == NPB)
				src = d1 + d1r * p.va;
			if (!same && of_c)
				src = (arr == 0 ? u2 : arr == 1 ? f2 : d2) + (int64_t)k * p.vb;
			stg[NBC + n] = src[x];
		}
	}
	if constexpr (!same) {
		const ER *GA = (const ER *)p.epi.GA, *ZA = (const ER *)p.epi.ZA;
		const int64_t ji = ((int64_t)j * p.oa + i) * p.va;
#pragma unroll
		for (int q = 0; q < NBA / NT; ++q) {
			const int n = tid + q * NT;
			const int arr = n / 1024, bl = (n / 32) % 32, al = n % 32;
			const int b = B0 + bl < na ? B0 + bl : na - 1;
			const int a = A0 + al < na ? A0 + al : na - 1;
			sab[n] = (arr ? ZA : GA)[(ji + b) * p.va + a];
		}
	}
	/* row of a lane group in (a block, register) */
	auto row_a = [&](int ab, int r, int g) {
		return 16 * ab + (FM::ROW_F64 ? g + 4 * r : 4 * g + r);
	};
	/* same spin: the wave's (b, a) values of (a block, register) */
	constexpr int NCV1 = same ? (NCOL + 63) / 64 : 1;
	ER cv[NCV1];
	ER *const scol = sab + wave * NCOL;
	const ER *cp[NCV1];   /* at a = 0 */
#pragma unroll
	for (int q = 0; q < NCV1; ++q) {
		const int m = lane + 64 * q, y = m / 8 % BW;
		const int b = B0 + NW * y + wave;
		const int64_t rb = (int64_t)(b < na ? b : na - 1) * p.vb;
		const int64_t r0 = rb + pjk, r1 = rb + pik, r2 = rb + pji;
		const int64_t e = m < 8 * BW ? r0 : m < 16 * BW ? r1 : r2;
		cp[q] = ((m & 4) ? Z : G) + e;
		cv[q] = 0;
	}
	/* (a, c) values of a column, [G, Z] for jk, ik (, ji) */
	ER ac[NPB];
	auto load_ac = [&](int ab, int r, int cb)
	    __attribute__((always_inline)) {
		const int a = A0 + row_a(ab, r, lg), c = C0 + 16 * cb + ln;
		const int64_t e = (int64_t)(a < na ? a : na - 1) * p.vb +
		    (c < nc ? c : nc - 1);
#pragma unroll
		for (int q = 0; q < NPB; ++q)
			ac[q] = ((q & 1) ? Z : G)[(q < 2 ? pjk : q < 4 ? pik : pji) + e];
	};
	__syncthreads();
#pragma unroll
	for (int n = -1; n < 8; ++n) {
		const int ab = n >> 2, r = n & 3;
		if constexpr (same) {
			/* other lanes of the wave read these, and read the last ones */
			if (n >= 0) {
				wave_sync();
#pragma unroll
				for (int q = 0; q < NCV1; ++q)
					if (lane + 64 * q < NCOL)
						scol[lane + 64 * q] = cv[q];
				wave_sync();
			}
			if (n < 7) {
				const int a = A0 + row_a((n + 1) >> 2, (n + 1) & 3, lane & 3);
#pragma unroll
				for (int q = 0; q < NCV1; ++q)
					cv[q] = cp[q][a < na ? a : na - 1];
			}
		}
		if (n < 0)
			continue;
#pragma unroll
		for (int cb = 0; cb < NCB; ++cb) {
			uint32_t col = 0;
#pragma unroll
			for (int y = 0; y < BW; ++y)
				col |= 1u << GM::blk2(y, ab, cb);
			if (!(m2 & col))
				continue;
			load_ac(ab, r, cb);
#pragma unroll
			for (int y = 0; y < BW; ++y) {
				const int x = GM::blk2(y, ab, cb);
				E[y * 64] = acc[x][r];
				if (NSET == 2)
					E[(BW + y) * 64] = bload_ae<AE>(wr, wvo,
					    (r * NACC + x) * WST);
			}
			const int al = row_a(ab, r, lg);
			const int a = A0 + al, c = C0 + 16 * cb + ln;
			if (a < na && c < nc)
				epi_block<F, KIND, NSET, BW, NW, TC>(p, a, c, B0 + wave, E,
				    ac, sva + al, sbv, svc + 16 * cb + ln, sbc + 16 * cb,
				    same ? scol + lg : sab + wave * 32 + al, esum, ecmp);
		}
	}

	/* deterministic workgroup reduction */
	double e = (esum[0] - ecmp[0]) + (esum[1] - ecmp[1]);
#pragma unroll
	for (int off = 32; off >= 1; off >>= 1)
		e += __shfl_xor(e, off);
	if (lane == 0)
		red[wave] = e;
	__syncthreads();
	if (tid == 0) {
		double t = (red[0] + red[1]) + (red[2] + red[3]);
		if constexpr (NW == 8)
			t += (red[4] + red[5]) + (red[6] + red[7]);
		if (keep)
			p.partial[it] = t;
	}
}
/* save area `slot` of wsave (two W sets; pt_wsave_bytes each) */
template <int F, int NW>
__device__ __forceinline__ typename Form<F>::AE *
wsave_of(void *wsave, int64_t slot)
{
	constexpr int64_t bytes = (int64_t)NW * Geo<F, 2, NW>::NACC * 4 * 64 *
	    sizeof(typename Form<F>::AE);
	return (typename Form<F>::AE *)((char *)wsave + slot * bytes);
}

/*
 * One launch segment: n_chunk positions of a run of one spin case's items
 * (item = ijk * n_tiles + tile).  XCD-aware order: workgroup n runs on XCD n % 8,
 * and each XCD gets a contiguous run of the launch's positions, so the
 * workgroups running together on one XCD share operand slices in its L2.
 * With kgrp > 1 the positions take the ijk in groups of kgrp, tile-major
 * within a group, in the order of the perm list (null: the work list's),
 * which puts ijk that share slabs next to each other (pt_ijk_order): the 64
 * workgroups that an XCD runs together are on a tile or two, for ijk that
 * share their slabs.  Each item still writes its own energy at its place in
 * the work list, so the energies do not depend on kgrp or perm.  One
 * workgroup per item, handed out by the dispatcher in order; with two W
 * sets position n of the segment keeps W of set 0 in save area wslot0 + n.
 */
__device__ __forceinline__ int64_t
item_of(const pt_launch &p, int64_t it)
{
	it += p.pos0;
	if (p.kgrp <= 1)
		return p.item0 + it;
	const int64_t nt = p.n_tiles, G = p.kgrp, m = p.n_seq / nt;
	const int64_t grp = it / (G * nt), r = it - grp * G * nt;
	const int64_t gsz = G < m - grp * G ? G : m - grp * G;
	const int64_t tile = r / gsz, g = r - tile * gsz;
	const int64_t pos = p.item0 / nt + grp * G + g;
	return (p.perm ? (int64_t)p.perm[pos] : pos) * nt + tile;
}

template <int F, int KIND, int NSET, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 1 : 2) void
k_tiles(pt_launch p)
{
	__shared__ __attribute__((aligned(16))) char
	    lds[Lds<F, KIND, NSET, NW>::BYTES];
	const int64_t per = (p.n_chunk + 7) / 8;
	const int64_t it = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
	if (it >= p.n_chunk)
		return;
	tile_item<F, KIND, NSET, NW>(p, item_of(p, it), NSET == 2 ?
	    wsave_of<F, NW>(p.wsave, p.wslot0 + it) : nullptr, lds);
}

/*
 * Two items, next to each other in launch order, per workgroup: four waves
 * each, the whole CU.  Every item of a launch has the same terms and panels,
 * so both halves meet the same barriers, and the two items of a CU walk their
 * slabs in step; mostly they have the same tile and share slabs, and what one
 * half fetched the other finds in L1 or L2 instead of fetching it again.
 * That pays where the split forms wait for HBM, i.e. where the slabs that
 * the workgroups of an XCD use together outgrow its L2; below, two workgroups
 * that drift apart fill each other's barriers and epilogues.  The change is
 * gradual (48 ijk of rpt o=10 in split BF16, one item per workgroup -> pairs,
 * same-spin and mixed-spin ms): v=300 8.03 -> 8.01 and 18.6 -> 19.0, v=352
 * 12.7 -> 12.3 and 28.9 -> 28.6, v=400 23.1 -> 22.1 and 50.8 -> 50.3, v=477
 * 46.6 -> 41.2 and 94.8 -> 93.6, v=600 134 -> 101 and 238 -> 230; two W sets
 * (rft F16X3, other sets of ijk) v=256 9.1 -> 9.5 and 20.6 -> 21.3, v=350 30.3
 * -> 30.1 and 76.6 -> 76.5, v=384 42.5 -> 34.7 and 77.9 -> 77.6, v=400 52.0 ->
 * 43.9 and 102 -> 101, v=440 82.2 -> 62.2 and 143 -> 142, v=477 110 -> 82.6 and
 * 188 -> 184, v=600 216 -> 182 and 459 -> 449; rft BF16X3 v=420 72.8 -> 56.3 and
 * 135 -> 132, uft BF16X3 450/440 72.7 -> 66.5 and 58.8 -> 54.9).  Launches of
 * one to eight ijk
 * share fewer slabs: from 8 % slower to 20 % faster at v=384 to 600, without
 * a trend.  At v=48 to 200 pairs cost up to 25 %, and FP64 and FP32 lose by
 * them (FP64 2 to 20 % at v=64 to 200 and 4 % at v=477, FP32 up to 16 %).
 */
constexpr int PAIR_NA = 384;

template <int F, int KIND, int NSET>
__global__ __launch_bounds__(512, 1) void
k_tiles_pair(pt_launch p)
{
	typedef Lds<F, KIND, NSET, 4> LD;
	__shared__ __attribute__((aligned(16))) char lds[2 * LD::BYTES];
	const int half = uni((int)threadIdx.x / 256);
	const int64_t per = (p.n_chunk + 15) / 16 * 2;
	const int64_t lo = (blockIdx.x & 7) * per;
	const int64_t hi = lo + per < p.n_chunk ? lo + per : p.n_chunk;
	const int64_t i0 = lo + 2 * (int64_t)(blockIdx.x >> 3);
	if (i0 >= hi)
		return;
	/* an odd end: the second half does the first one's item and drops it */
	const bool keep = i0 + half < hi;
	const int64_t it = keep ? i0 + half : i0;
	tile_item<F, KIND, NSET, 4>(p, item_of(p, it), NSET == 2 && keep ?
	    wsave_of<F, 4>(p.wsave, p.wslot0 + it) : nullptr,
	    lds + half * LD::BYTES, keep);
}

/* the segments of one launch, of either spin case: workgroups first[s] ..
 * first[s + 1] - 1 (first a multiple of 8, so that workgroup n of a segment
 * is on XCD n % 8) */
struct seg_args {
	pt_launch seg[PT_MAX_SEGS];
	int32_t first[PT_MAX_SEGS];
	int32_t n;
};

template <int F, int NSET, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 1 : 2) void
k_tiles_segs(seg_args a)
{
	constexpr int B0 = Lds<F, PT_AAA, NSET, NW>::BYTES;
	constexpr int B1 = Lds<F, PT_AAB, NSET, NW>::BYTES;
	__shared__ __attribute__((aligned(16))) char lds[B0 > B1 ? B0 : B1];
	int s = 0;
	while (s + 1 < a.n && (int)blockIdx.x >= a.first[s + 1])
		++s;
	const pt_launch &p = a.seg[s];
	const int n = (int)blockIdx.x - a.first[s];
	const int64_t per = (p.n_chunk + 7) / 8;
	const int64_t it = (n & 7) * per + (n >> 3);
	if (it >= p.n_chunk)
		return;
	const int64_t item = item_of(p, it);
	typename Form<F>::AE *w = NSET == 2 ?
	    wsave_of<F, NW>(p.wsave, p.wslot0 + it) : nullptr;
	if (p.kind == PT_AAA)
		tile_item<F, PT_AAA, NSET, NW>(p, item, w, lds);
	else
		tile_item<F, PT_AAB, NSET, NW>(p, item, w, lds);
}

/*
 * The same items from a persistent grid: workgroup w serves XCD w % 8 and
 * takes that XCD's run of launch positions, [x per, x per + per), one at a
 * time from the XCD's counter, in order.  The counter is fetched by one
 * thread between two barriers that every wave meets outside any divergent
 * branch (the previous item's partial-energy store is behind the first),
 * the value is read back as a wave-uniform scalar, and the loop ends for
 * the whole workgroup when it passes the run's end, which the host bounds;
 * no workgroup waits on another.  With two W sets each workgroup keeps W of
 * set 0 in its own save area (slot w).
 */
template <int F, int KIND, int NSET, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 1 : 2) void
k_tiles_p(pt_launch p)
{
	__shared__ __attribute__((aligned(16))) char
	    lds[Lds<F, KIND, NSET, NW>::BYTES];
	__shared__ int s_next;
	const int64_t per = (p.n_chunk + 7) / 8;
	const int x = blockIdx.x & 7;
	const int64_t lo = x * per;
	const int64_t cnt = p.n_chunk - lo < per ? p.n_chunk - lo : per;
	for (;;) {
		__syncthreads();
		if (threadIdx.x == 0)
			s_next = (int)atomicAdd(p.ctr + x, 1u);
		__syncthreads();
		const int64_t r = __builtin_amdgcn_readfirstlane(s_next);
		if (r >= cnt)
			break;
		tile_item<F, KIND, NSET, NW>(p, item_of(p, lo + r), NSET == 2 ?
		    wsave_of<F, NW>(p.wsave, blockIdx.x) : nullptr, lds);
	}
}

/* the 8 item counters of a persistent launch, zeroed on its stream by a
 * kernel (a graph may record it) */
__global__ void
k_zero_ctr(uint32_t *c)
{
	if (threadIdx.x < 8)
		c[threadIdx.x] = 0u;
}

template <int F, int NSET, int NW>
int
launch_geo(const pt_launch *p, int n, hipStream_t s)
{
	typedef Geo<F, NSET, NW> GM;
	if (n < 1 || n > PT_MAX_SEGS)
		return (int)hipErrorInvalidValue;
	for (int q = 0; q < n; ++q)
		if (p[q].tcw != GM::TC || p[q].nw != NW || p[q].nset != NSET ||
		    (n > 1 && p[q].ctr))
			return (int)hipErrorInvalidValue;
	dim3 block(GM::THREADS);
	if (p->ctr) {
		/* persistent grid: one save area per workgroup */
		if (p->pgrid <= 0 || p->pgrid % 8 || p->n_chunk > INT32_MAX / 2 ||
		    (NSET == 2 && (!p->wsave || p->pgrid > p->nwsave)))
			return (int)hipErrorInvalidValue;
		k_zero_ctr<<<1, 64, 0, s>>>(p->ctr);
		dim3 grid((unsigned)p->pgrid);
		if (p->kind == PT_AAA)
			k_tiles_p<F, PT_AAA, NSET, NW><<<grid, block, 0, s>>>(*p);
		else
			k_tiles_p<F, PT_AAB, NSET, NW><<<grid, block, 0, s>>>(*p);
		return (int)hipGetLastError();
	}
	seg_args a;
	a.n = n;
	int64_t wgs = 0;
	for (int q = 0; q < n; ++q) {
		/* one save area per item */
		if (NSET == 2 && (!p[q].wsave || p[q].wslot0 < 0 ||
		    p[q].wslot0 + p[q].n_chunk > p[q].nwsave))
			return (int)hipErrorInvalidValue;
		a.seg[q] = p[q];
		a.first[q] = (int32_t)wgs;
		wgs += 8 * ((p[q].n_chunk + 7) / 8);
		if (wgs > INT32_MAX / 2)
			return (int)hipErrorInvalidValue;
	}
	const dim3 grid((unsigned)wgs);
	if constexpr (Form<F>::PAN && NW == 4)
		if (n == 1 && p->na >= PAIR_NA) {
			const dim3 pairs((unsigned)(8 * ((p->n_chunk + 15) / 16)));
			if (p->kind == PT_AAA)
				k_tiles_pair<F, PT_AAA, NSET><<<pairs, 512, 0, s>>>(*p);
			else
				k_tiles_pair<F, PT_AAB, NSET><<<pairs, 512, 0, s>>>(*p);
			return (int)hipGetLastError();
		}
	if (n > 1)
		k_tiles_segs<F, NSET, NW><<<grid, block, 0, s>>>(a);
	else if (p->kind == PT_AAA)
		k_tiles<F, PT_AAA, NSET, NW><<<grid, block, 0, s>>>(*p);
	else
		k_tiles<F, PT_AAB, NSET, NW><<<grid, block, 0, s>>>(*p);
	return (int)hipGetLastError();
}

template <int F>
int
launch_form(const pt_launch *p, int n, hipStream_t s)
{
	if (p->nw == 8)
		return p->nset == 1 ? launch_geo<F, 1, 8>(p, n, s) :
		    launch_geo<F, 2, 8>(p, n, s);
	return p->nset == 1 ? launch_geo<F, 1, 4>(p, n, s) :
	    launch_geo<F, 2, 4>(p, n, s);
}

} /* namespace */

#endif
