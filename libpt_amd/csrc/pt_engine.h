/*
 * Internal interface between the host engine and the device kernels of
 * libpt_amd (not part of the public C API).
 *
 * A spin case of one system is a list of *terms*.  Each term adds
 *     sign * sum_kappa S[s][kappa] * Q[kappa][u][w]
 * to the connected triples W[a][b][c] of one ijk item, where the single
 * index s and the pair (u, w) are the output indices a, b, c in some role
 * (role = which of a/b/c the S operand carries; (u, w) are the other two in
 * a, b, c order).  S and Q are strided slices of the input tensors whose
 * base offsets are linear in the occupied indices (i, j, k).
 *
 * The terms of every spin case of libpt (src/pt.c:236-290, :361-432,
 * :588-696, :773-915) are written in this form by pt_terms.cpp.
 */
#ifndef LIBPT_AMD_PT_ENGINE_H
#define LIBPT_AMD_PT_ENGINE_H

#include <stddef.h>
#include <stdint.h>

enum pt_form {
	PT_FORM_FP64 = 0,   /* FP64 operands, v_mfma_f64_16x16x4_f64 */
	PT_FORM_FP32 = 1,   /* FP32 operands, v_mfma_f32_16x16x4_f32 (_mp) */
	PT_FORM_BF16X3 = 2, /* hi+lo BF16 pairs, 3 products per kappa packed
	                       into v_mfma_f32_16x16x32_bf16 */
	PT_FORM_F16X3 = 3,  /* hi+lo FP16 pairs (scaled), the same with
	                       v_mfma_f32_16x16x32_f16 */
	PT_NFORM = 4
};

enum pt_kind { PT_AAA = 0, PT_AAB = 1 };
enum pt_role { PT_ROLE_A = 0, PT_ROLE_B = 1, PT_ROLE_C = 2 };

#define PT_MAX_TERMS 40
#define PT_MAX_BUFS 26
#define PT_MAX_SEGS 4    /* spin cases (segments) of one tile launch */

/* kappa per fragment of the packed Q operands: a fragment is 1 KB, 16 rows
 * of 64 bytes (8 FP64, 16 FP32, or 16 split values: per 4 kappa hi 0-3 and
 * lo 0-3), in the lane order of the MFMA operand: lane 16 g + row holds
 * the row's g-th quarter.  The fragments of a plane of 1, 2, 4 or 8 rows
 * (rounded up) hold only these: quarter g of a row at 16 (rows g + row).  A
 * spin of two orbitals would else pad eightfold. */
#define PT_FRAG 1024
static inline int
pt_frag_rows(int64_t rows)
{
	return rows > 8 ? 16 : rows > 4 ? 8 : rows > 2 ? 4 : rows > 1 ? 2 : 1;
}

static inline int
pt_kc(int form)
{
	return form == 0 ? 8 : 16;
}

/* kappa chunks of a slab of K kappa (zero padded) */
static inline int64_t
pt_chunks(int form, int64_t K)
{
	return (K + pt_kc(form) - 1) / pt_kc(form);
}

/* bytes of a packed slab [row block of 16][chunk][column] of fragments: rows
 * and columns of the plane; tri: the pairs row > column of a square plane,
 * block b holding its columns 0 .. 16 (b + 1) - 1 */
static inline int64_t
pt_slab_bytes(int form, int64_t K, int64_t rows, int64_t cols, int tri)
{
	const int64_t nb = (rows + 15) / 16;
	return pt_chunks(form, K) * (tri ? 8 * nb * (nb + 1) : nb * cols) *
	    (PT_FRAG / 16 * pt_frag_rows(rows));
}

/* Workgroup geometry (the kernel's Geo): NW = 4 waves, tile 32 a x 32 b x
 * TC c with TC = 16 for FP64 and 32 for FP32 and the split forms (128
 * accumulator registers per lane either way), two workgroups per CU; or
 * NW = 8 waves, tile 32 a x 32 b x 32 c, one workgroup per CU.  (fT) forms
 * its two W sets one after the other in the same registers, so the
 * geometry does not depend on the W-set count. */
#define PT_TA 32
#define PT_TB 32

/* default wave count of a form: 4 (two workgroups per CU) measured ahead
 * of 8 at o=45, v=477 in every form; the tuner's record for a size, or
 * LIBPT_AMD_WAVES=4 or 8, overrides it for new plans */
static inline int
pt_nw_default(int form)
{
	(void)form;
	return 4;
}

static inline int
pt_tcw(int form, int nset, int nw)
{
	(void)nset;
	return nw == 8 || form != 0 ? 32 : 16;
}

static inline int
pt_cw(int form, int nset, int nw)
{
	return nw == 8 ? 16 : pt_tcw(form, nset, nw);
}

/*
 * S operands are read in the API layout (kappa contiguous; the split forms
 * from hi | lo << 16 copies), Q operands from packed copies (PT_FRAG).  The
 * pair (u, w) is the two indices that S does not carry, in a, b, c order;
 * the packed rows are u and the columns w, or (tr) rows w and columns u.
 */
struct pt_term {
	int64_t s_off[3];  /* S base offset (elements) = s_off . (i, j, k) */
	int64_t q_off[3];  /* Q slab offset (bytes of the packed copy) */
	int64_t s_st;      /* stride of the single index s (kappa stride 1) */
	int64_t cols;      /* columns of the packed plane */
	int32_t s_buf, q_buf;
	int32_t role, set, sign, K;
	int32_t nch;       /* kappa chunks */
	int32_t tri;       /* packed triangle u > w (pt_slab_bytes) */
	int32_t tr;
	int32_t fr;        /* rows of a fragment (pt_frag_rows) */
};

/* terms of one W set of a spin case */
#define PT_TERMS_SAME 18
#define PT_TERMS_MIXED 16

/* epilogue inputs (element type: double, or float for PT_FORM_FP32) */
struct pt_epi {
	const void *d1, *d2;  /* d_ov of the pair spin / odd spin */
	const void *u1, *u2;  /* t1 (T) or l1 (fT) */
	const void *f1, *f2;  /* f_ov (T) or f2_ov (fT) */
	const void *GA, *GB;  /* i_oovv same-spin / mixed blocks */
	const void *ZA, *ZB;  /* t2 (T) or l2 (fT) same-spin / mixed blocks */
};

struct pt_launch {
	const void *buf[PT_MAX_BUFS];
	const struct pt_term *terms; /* device array: per W set, role a, role b,
	                                role c */
	int32_t nterm1, nterm2;      /* per W set: roles a and b, role c */
	int32_t kind, nset;
	int64_t oa, va, ob, vb;      /* aaa: ob = oa, vb = va */
	int32_t na, nc;              /* extents of a (= b) and c */
	int32_t tcw;                 /* c tile width (pt_tcw) */
	int32_t nterm_a;             /* per W set: terms with role a */
	const int32_t *ijk;          /* [n_ijk][3] */
	const int32_t *tiles;        /* [n_tiles][3]: blocks (A, B, C), A >= B */
	int32_t n_tiles, nw;         /* tiles per ijk, waves per workgroup */
	int64_t item0, n_seq;        /* a run of items: n_seq of them, from item0
	                                (whole ijk); its positions are ordered
	                                by kgrp and perm */
	int64_t pos0, n_chunk;       /* the launch's: positions [pos0, pos0 +
	                                n_chunk) of the run */
	double *partial;             /* energy of each item */
	double inv_scale[2];         /* per W set: 1 / (operand scale product) */
	void *wsave;                 /* two W sets: W of set 0 of each item
	                                of the launch (pt_wsave_bytes each,
	                                position pos0 + n at slot wslot0 +
	                                n), else unused */
	int32_t nwsave, wslot0;      /* save areas in wsave */
	int32_t kgrp;                /* > 1: the run's ijk are taken in groups
	                                of kgrp, each group's items
	                                tile-major; 1: items in order */
	const int32_t *perm;         /* kgrp > 1: the run's ijk in order (null:
	                                item0 / n_tiles and on) */
	uint32_t *ctr;               /* non-null: a persistent grid of pgrid
	                                workgroups takes the items from these
	                                8 counters (one per XCD, zeroed by the
	                                launch), with one save area per
	                                workgroup (nwsave >= pgrid); null: one
	                                workgroup per item */
	int32_t pgrid;
	struct pt_epi epi;
};

#ifdef __cplusplus
extern "C" {
#endif
/* bytes of one item's saved W set: NW waves x CW blocks x 4 values x 64
 * lanes */
static inline int64_t
pt_wsave_bytes(int form, int nset, int nw)
{
	return (int64_t)nw * pt_cw(form, nset, nw) * 4 * 64 *
	    (form == 0 ? 8 : 4);
}

/* items per launch with two W sets: each item of a launch has its own save
 * area, so this bounds the areas to 4 GB (32768 items of 128 KB) */
static inline int64_t
pt_ft_chunk(int form, int nw)
{
	return ((int64_t)4 << 30) / pt_wsave_bytes(form, 2, nw);
}

/* kernel launchers (pt_tiles_*.hip, pt_kernel.hip); return hipError_t as int */
/* n <= PT_MAX_SEGS segments (n_chunk > 0) of one geometry and W-set count in
 * one launch, in order; a persistent grid takes one */
int pt_launch_tiles(int form, const struct pt_launch *p, int n,
    void *stream);
int pt_launch_tiles_fp64(const struct pt_launch *p, int n, void *stream);
int pt_launch_tiles_fp32(const struct pt_launch *p, int n, void *stream);
int pt_launch_tiles_bf16x3(const struct pt_launch *p, int n, void *stream);
int pt_launch_tiles_f16x3(const struct pt_launch *p, int n, void *stream);
/* out[s] = fixed-order sum of segment s's partials (as pt_launch_reduce) */
int pt_launch_reduce_batch(const struct pt_launch *segs,
    const int64_t *begin, int nseg, double *out, void *stream);
/* out[q] = fixed-order sum of x[q][0..n[q]) for q < cnt <= 4 */
int pt_launch_reduce(const double *const *x, const int64_t *n, int cnt,
    double *out, void *stream);
int pt_launch_segsum(const double *x, int64_t nseg, int64_t seglen,
    double *out, void *stream);
int pt_launch_split(const double *src, uint32_t *dst, int64_t n, int fp16,
    double scale, void *stream);
/* [R slabs][K][plane] -> packed slabs (pt_slab_bytes) of the plane's rows
 * and columns; the source plane is [rows][cols], [cols][rows] (tr), or the
 * packed pairs row > column (tri); the split forms store hi and lo of
 * x * scale.  at, fr: set by the launch. */
struct pt_pack_job {
	const char *src;
	char *dst;
	int64_t R, K, rows, cols;
	double scale;
	int64_t at;
	int32_t tri, tr, fr;
};
int pt_launch_pack(const struct pt_pack_job *jobs, int n, int form,
    void *stream);
/* out = the entries of perm[0..n) in [lo, hi), in order (one workgroup) */
int pt_launch_filter(const int32_t *perm, int64_t n, int32_t lo, int32_t hi,
    int32_t *out, void *stream);
int pt_launch_absmax(const double *src, int64_t n, double *out, void *stream);
int pt_launch_copy(const double *src, double *dst, int64_t n, void *stream);
int pt_launch_synth(const void *spec, int tensor, void *dst, int64_t n,
    int fp32, void *stream);

/* bytes of the allocation-free call's static array.  LIBPT_AMD_NOALLOC_SCRATCH
 * of them decide which calls are taken; the packed rows' padding (to 16, or to
 * a power of two below) brings those to at most 496 MiB, for 13 and 17
 * virtual orbitals.  The rest is room for the transposed copies (with them
 * the largest call takes 887 MiB) and for (fT) save areas: a launch holds as
 * many items as there are areas, and the copies are left out where fewer than
 * PT_NOALLOC_AREAS, eight rounds of workgroups, would remain (uft 5/17/198/17
 * FP64, whose copies leave 1100: 2.58 s with them, 2.26 s without) */
#define PT_NOALLOC_ARENA ((size_t)1 << 30)
#define PT_NOALLOC_AREAS 4096

/* host engine (pt_host.cpp) for pt_noalloc.hip: the device every call
 * runs on (made current; -1 on error), the calling thread's error text
 * (NULL clears it), and one call whose device buffers all come from
 * [scratch, scratch + cap) */
int pt_device_init(void);
void pt_set_error(const char *msg);
double pt_noalloc_energy(int call, int form, size_t oa, size_t va,
    size_t ob, size_t vb, const void *const *dev_arrays, void *scratch,
    size_t cap, void *stream);
#ifdef __cplusplus
}
#endif

#endif /* LIBPT_AMD_PT_ENGINE_H */
