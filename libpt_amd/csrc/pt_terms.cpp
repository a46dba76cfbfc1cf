/*
 * Term tables: every contraction of the connected triples W of libpt's
 * spin cases, written as (role, sign, S slice, Q slice) for the tile
 * kernel.  Index maps restate src/pt.c:40-160 (GEMM wrappers) combined with
 * the permutation passes of src/pt.c:236-290 (same spin) and
 * src/pt.c:361-432 (mixed spin); the (fT) builds of src/pt.c:588-696 and
 * :773-915 reuse the same tables on other operand buffers.
 *
 * Occupied slots: 0 = i, 1 = j, 2 = k.  Operand buffer slots (per W set s,
 * base 13*s): TA TB TC OA OB OC in the API layout (S operands), VA VB VC,
 * TA TB TC and TA transposed packed (Q operands); the same-spin case uses
 * the A slots.
 */
#include <string.h>

#include "pt_engine.h"
#include "pt_terms.h"

namespace {

enum { I = 0, J = 1, K = 2 };
enum { A = PT_ROLE_A, B = PT_ROLE_B, C = PT_ROLE_C };

struct TermBuilder {
	pt_term t;
	int form;
	TermBuilder(int form_, int role, int set, int sign, int64_t kext)
	{
		memset(&t, 0, sizeof(t));
		form = form_;
		t.role = role;
		t.set = set;
		t.sign = sign;
		t.K = (int32_t)kext;
		t.nch = (int32_t)pt_chunks(form, kext);
	}
	/* S[s][kappa] = buf[sbuf] + sum occ*coef + s*s_st + kappa */
	TermBuilder &S(int buf, int o1, int64_t c1, int o2, int64_t c2,
	    int64_t st)
	{
		t.s_buf = buf;
		t.s_off[o1] += c1;
		t.s_off[o2] += c2;
		t.s_st = st;
		return *this;
	}
	/* Q: slab o1 of buf, packed with the rows u of extent nu and the
	 * columns w of extent nw, or (tr) with rows w and columns u */
	TermBuilder &Q(int buf, int o1, int64_t nu, int64_t nw, bool tr = false)
	{
		t.q_buf = buf;
		t.tr = tr;
		t.cols = tr ? nu : nw;
		t.fr = pt_frag_rows(tr ? nw : nu);
		t.q_off[o1] = pt_slab_bytes(form, t.K, tr ? nw : nu, t.cols, 0);
		return *this;
	}
	/* Q: slab o1 of buf, the packed pairs u > w of extent n */
	TermBuilder &Qtri(int buf, int o1, int64_t n)
	{
		t.q_buf = buf;
		t.tri = 1;
		t.fr = pt_frag_rows(n);
		t.q_off[o1] = pt_slab_bytes(form, t.K, n, n, 1);
		return *this;
	}
	pt_term done() { return t; }
};

} /* namespace */

void
pt_terms_same(pt_term_list &out, int form, int set, int64_t o, int64_t v,
    bool copies)
{
	const int b0 = PT_SET_BUFS * set;
	const int bT = b0 + 0, bO = b0 + 3, bV = b0 + 6, bTq = b0 + 9;
	/* T with its plane transposed: a copy, or the plain one read so */
	const int bTt = copies ? b0 + 12 : bTq;
	const int64_t vv = v * v;

	/* ovvv: Y_pqr(x; y,z) = sum_d T[p,q,x,d] V[r,d,(y,z)],
	 * (p,q,r) = (i,j,k) +, (i,k,j) -, (k,j,i) -  (src/pt.c:236-261) */
	const int pqr[3][3] = {{I, J, K}, {I, K, J}, {K, J, I}};
	const int sg1[3] = {+1, -1, -1};
	for (int n = 0; n < 3; ++n) {
		const int p = pqr[n][0], q = pqr[n][1], r = pqr[n][2];
		const int s = sg1[n];
		/* +Y(c; a,b) */
		out.push_back(TermBuilder(form, C, set, +s, v)
		    .S(bT, p, o * vv, q, vv, v).Qtri(bV, r, v).done());
		/* -Y(b; a,c) */
		out.push_back(TermBuilder(form, B, set, -s, v)
		    .S(bT, p, o * vv, q, vv, v).Qtri(bV, r, v).done());
		/* +Y(a; b,c) */
		out.push_back(TermBuilder(form, A, set, +s, v)
		    .S(bT, p, o * vv, q, vv, v).Qtri(bV, r, v).done());
	}
	/* oovo: X_(p;q,r)(x,y,z) = sum_l T[p,l,x,y] O[q,r,z,l],
	 * (p;q,r) = (i;j,k) +, (j;i,k) -, (k;j,i) -  (src/pt.c:263-290) */
	const int pqr2[3][3] = {{I, J, K}, {J, I, K}, {K, J, I}};
	for (int n = 0; n < 3; ++n) {
		const int p = pqr2[n][0], q = pqr2[n][1], r = pqr2[n][2];
		const int s = sg1[n];
		/* +X(b,c,a): S = O[q,r][a][l], Q = T[p][l][b][c] */
		out.push_back(TermBuilder(form, A, set, +s, o)
		    .S(bO, q, o * v * o, r, v * o, o).Q(bTq, p, v, v).done());
		/* -X(a,c,b): S = O[q,r][b][l], Q = T[p][l][a][c] */
		out.push_back(TermBuilder(form, B, set, -s, o)
		    .S(bO, q, o * v * o, r, v * o, o).Q(bTq, p, v, v).done());
		/* -X(b,a,c): S = O[q,r][c][l], Q = T[p][l][b][a] */
		out.push_back(TermBuilder(form, C, set, -s, o)
		    .S(bO, q, o * v * o, r, v * o, o)
		    .Q(bTt, p, v, v, !copies).done());
	}
}

void
pt_terms_mixed(pt_term_list &out, int form, int set, int64_t oa, int64_t va,
    int64_t ob, int64_t vb, bool copies)
{
	const int b0 = PT_SET_BUFS * set;
	const int TA = b0 + 0, TB = b0 + 1, TC = b0 + 2;
	const int OA = b0 + 3, OB = b0 + 4, OC = b0 + 5;
	const int VA = b0 + 6, VB = b0 + 7, VC = b0 + 8;
	const int TAq = b0 + 9, TBq = b0 + 10, TCq = b0 + 11;

	/* src/pt.c:361-367: -sum_d TA[i,j,a,d] VC[k,d,c,b] + (a<->b); the
	 * plane (c, b) of VC packed transposed, or read so */
	out.push_back(TermBuilder(form, A, set, -1, va)
	    .S(TA, I, oa * va * va, J, va * va, va)
	    .Q(VC, K, va, vb, !copies).done());
	out.push_back(TermBuilder(form, B, set, +1, va)
	    .S(TA, I, oa * va * va, J, va * va, va)
	    .Q(VC, K, va, vb, !copies).done());
	/* :369-375: -sum_d TB[i,k,a,d] VB[j,d,b,c] + (a<->b) */
	out.push_back(TermBuilder(form, A, set, -1, vb)
	    .S(TB, I, ob * va * vb, K, va * vb, vb).Q(VB, J, va, vb).done());
	out.push_back(TermBuilder(form, B, set, +1, vb)
	    .S(TB, I, ob * va * vb, K, va * vb, vb).Q(VB, J, va, vb).done());
	/* :377-383: +sum_d TB[j,k,a,d] VB[i,d,b,c] - (a<->b) */
	out.push_back(TermBuilder(form, A, set, +1, vb)
	    .S(TB, J, ob * va * vb, K, va * vb, vb).Q(VB, I, va, vb).done());
	out.push_back(TermBuilder(form, B, set, -1, vb)
	    .S(TB, J, ob * va * vb, K, va * vb, vb).Q(VB, I, va, vb).done());
	/* :385-392: -sum_d TC[k,j,c,d] VA[i,d,(a,b)] + sum_d TC[k,i,c,d] VA[j,..] */
	out.push_back(TermBuilder(form, C, set, -1, va)
	    .S(TC, K, oa * vb * va, J, vb * va, va).Qtri(VA, I, va).done());
	out.push_back(TermBuilder(form, C, set, +1, va)
	    .S(TC, K, oa * vb * va, I, vb * va, va).Qtri(VA, J, va).done());
	/* :394-406: -sum_l TA[i,l,a,b] OC[k,j,c,l] + sum_l TA[j,l,a,b] OC[k,i,c,l] */
	out.push_back(TermBuilder(form, C, set, -1, oa)
	    .S(OC, K, oa * vb * oa, J, vb * oa, oa).Q(TAq, I, va, va).done());
	out.push_back(TermBuilder(form, C, set, +1, oa)
	    .S(OC, K, oa * vb * oa, I, vb * oa, oa).Q(TAq, J, va, va).done());
	/* :408-414: -sum_l TB[i,l,a,c] OB[j,k,b,l] + sum_l TB[i,l,b,c] OB[j,k,a,l] */
	out.push_back(TermBuilder(form, B, set, -1, ob)
	    .S(OB, J, ob * va * ob, K, va * ob, ob).Q(TBq, I, va, vb).done());
	out.push_back(TermBuilder(form, A, set, +1, ob)
	    .S(OB, J, ob * va * ob, K, va * ob, ob).Q(TBq, I, va, vb).done());
	/* :416-422: -sum_l TB[j,l,b,c] OB[i,k,a,l] + sum_l TB[j,l,a,c] OB[i,k,b,l] */
	out.push_back(TermBuilder(form, A, set, -1, ob)
	    .S(OB, I, ob * va * ob, K, va * ob, ob).Q(TBq, J, va, vb).done());
	out.push_back(TermBuilder(form, B, set, +1, ob)
	    .S(OB, I, ob * va * ob, K, va * ob, ob).Q(TBq, J, va, vb).done());
	/* :424-432: -sum_l TC[k,l,c,a] OA[j,i,b,l] + sum_l TC[k,l,c,b] OA[j,i,a,l];
	 * the plane (c, a) of TC packed transposed, or read so */
	out.push_back(TermBuilder(form, B, set, -1, oa)
	    .S(OA, J, oa * va * oa, I, va * oa, oa)
	    .Q(TCq, K, va, vb, !copies).done());
	out.push_back(TermBuilder(form, A, set, +1, oa)
	    .S(OA, J, oa * va * oa, I, va * oa, oa)
	    .Q(TCq, K, va, vb, !copies).done());
}

int
pt_terms_order(pt_term_list &terms, int *n_role_a)
{
	/* W set 0, then W set 1; within a set role a, role b, role c, each
	 * group in table order.  Both sets have the same structure, so the
	 * counts of set 0 hold for every set. */
	int nset = 1;
	for (const pt_term &t : terms)
		nset = t.set + 1 > nset ? t.set + 1 : nset;
	pt_term_list out;
	int na = 0, n1 = 0;
	for (int s = 0; s < nset; ++s)
		for (int role = PT_ROLE_A; role <= PT_ROLE_C; ++role)
			for (const pt_term &t : terms)
				if (t.set == s && t.role == role) {
					out.push_back(t);
					if (s == 0 && role == PT_ROLE_A)
						++na;
					if (s == 0 && role != PT_ROLE_C)
						++n1;
				}
	terms = out;
	if (n_role_a)
		*n_role_a = na;
	return n1;
}
