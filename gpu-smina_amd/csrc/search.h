/*
 * The docking search on one wavefront: model::eval_deriv, BFGS with its line
 * searches, mutation, Metropolis and the output container, for one chain
 * (or one item) per wave64.
 *
 * Work layout inside a wave:
 *   conf and change vectors: element k in lane k (k < 64);
 *   atoms: atom i in lane i mod 64, coordinates and forces in LDS;
 *   frames: one per lane (set_conf top-down, derivative bottom-up, level-serial
 *     as the tree requires; FP32 walks each frame's path in one lane);
 *   intramolecular pairs: pair-parallel, a scalar per pair left in LDS; lane i
 *     then walks atom i's neighbour list (packed codes in LDS) in evaluation
 *     order, so every atom's force accumulates in exactly smina's order with
 *     no atomics;
 *   receptor maps: one corner-packed cell gather per heavy atom.
 * The model itself (types, frames, neighbour lists) is staged in LDS once
 * per workgroup; the hot loops read global memory only for the receptor map
 * cells and the pair tables.  Control (BFGS, line search, Metropolis, RNG)
 * is wave-uniform: every lane computes the same scalars.
 *
 * With T = double the search is "ordered": every sum runs in smina's CPU
 * order (energies serially over atoms and pairs in list order, dot products
 * serially over the change vector), reproducing the CPU restatement bit for
 * bit.  With T = float, energies use a fixed butterfly reduction.
 */
#ifndef SGPU_SEARCH_H
#define SGPU_SEARCH_H

#include "wave.h"
#include "rng.h"
#include "atom_types.h"
#include "spline.h"
#include "gridterm.h"
#include "../../include/sgpu.h"

namespace sgpu
{

// pairs per lane and batch of the intramolecular pair loop
constexpr int PAIR_BATCH = 4;
// receptor atoms per batch of the direct term
constexpr int REC_BATCH = 4;
// LDS of a workgroup: the staged model (int blob, real blob) then each
// wave's working state
struct WavePlan
{
	int nmax;   // movable atoms
	int fmax;   // frames
	int cmax;   // conf
	int gmax;   // change
	int pmax;   // pairs
	int hmax;   // Hessian entries (change size squared)
	int imax;   // model int blob
	int tmax;   // model real blob
	int amax;   // all atoms (movable + fixed)
	int pair_lds; // FP64: the pairs' force factors are held in LDS (eval_deriv's PS)
	int bytes;  // LDS bytes per workgroup
};

// reals per atom of the coordinate and force arrays: FP32 pads to 16 bytes
// so that a lane's random read of an atom is one ds_read_b128
template<typename T>
constexpr int atom_stride()
{
	return sizeof(T) == 4 ? 4 : 3;
}
constexpr int FRAME_REALS = 12; // origin and rotation matrix of a frame
constexpr int QUAT_REALS = 4;

template<typename T>
struct WaveMem
{
	T* fr;     // [frames][12]: origin, rotation matrix
	T* fq;     // [frames][4]
	T* fax;    // [frames][4]: world axis
	T* pf;     // per pair slot: FP32 the force over the distance vector, FP64 (dor, curl factor)
	T* tq;     // FP32: the torque prefix sums, in the pairs' place after the atoms have read them
	T* coords;
	T* forces;
	T* ff;     // ordered search: frames' forces and torques
	T* ft;
	T* gbuf;
	T* xstage;
};

// The search's own vectors in the search precision S: the staged conf and
// direction of a line-search trial, the Hessian and the BFGS update's
// scratch.  With S = T the conf stage and the scratch share the evaluation's
// buffers (xstage, gbuf).
template<typename S>
struct SearchMem
{
	S* xstage;
	S* pstage;
	S* hess;
	S* smhy;
};

// Per-wave LDS: the evaluation's region in T, then the search's in S
template<typename T>
__host__ __device__ inline int pair_lds_elems(const WavePlan& p)
{
	// slot 0 belongs to the padding of the neighbour lists
	if (Real<T>::ordered)
		return p.pair_lds ? 2 * (p.pmax + 1) : 0;
	return 4 + ((p.pmax > 4 * p.nmax ? p.pmax : 4 * p.nmax) + 3) / 4 * 4;
}
template<typename T>
__host__ __device__ inline int eval_lds_elems(const WavePlan& p)
{
	return p.fmax * (FRAME_REALS + 2 * QUAT_REALS + (Real<T>::ordered ? 6 : 0)) + pair_lds_elems<T>(p) +
			atom_stride<T>() * (p.amax + p.nmax) + p.gmax + p.cmax;
}
template<typename T, typename S>
__host__ __device__ inline int search_lds_elems(const WavePlan& p)
{
	return p.gmax + p.hmax + (sizeof(S) != sizeof(T) ? p.cmax + p.gmax : 0);
}
template<typename T, typename S>
__host__ __device__ inline int wave_lds_bytes(const WavePlan& p)
{
	const int eb = (eval_lds_elems<T>(p) * int(sizeof(T)) + 15) / 16 * 16;
	return eb + (search_lds_elems<T, S>(p) * int(sizeof(S)) + 15) / 16 * 16;
}
// model region in bytes, rounded to 16
template<typename T>
__host__ __device__ inline int model_lds_bytes(const WavePlan& p)
{
	return (p.imax + 3) / 4 * 16 + (p.tmax * int(sizeof(T)) + 15) / 16 * 16;
}
template<typename T, typename S = T>
__host__ __device__ inline int block_lds_bytes(const WavePlan& p, int waves)
{
	return model_lds_bytes<T>(p) + waves * wave_lds_bytes<T, S>(p);
}

// one wave's LDS (16-byte aligned) as its evaluation and search buffers;
// the arrays read 16 bytes at a time come first
template<typename T, typename S>
__device__ inline void carve(unsigned char* base, const WavePlan& p, WaveMem<T>& w, SearchMem<S>& sm)
{
	T* q = reinterpret_cast<T*>(base);
	w.fr = q;
	q += FRAME_REALS * p.fmax;
	w.fq = q;
	q += QUAT_REALS * p.fmax;
	w.fax = q;
	q += QUAT_REALS * p.fmax;
	w.pf = q;
	w.tq = q + 4;
	q += pair_lds_elems<T>(p);
	w.coords = q; // movable atoms, then the fixed atoms (copied once)
	q += atom_stride<T>() * p.amax;
	w.forces = q;
	q += atom_stride<T>() * p.nmax;
	w.ff = q;
	w.ft = q + 3 * p.fmax;
	if (Real<T>::ordered)
		q += 6 * p.fmax;
	w.gbuf = q;
	q += p.gmax;
	w.xstage = q;
	S* r = reinterpret_cast<S*>(base + (eval_lds_elems<T>(p) * int(sizeof(T)) + 15) / 16 * 16);
	sm.pstage = r;
	r += p.gmax;
	sm.hess = r;
	r += p.hmax;
	if constexpr (sizeof(S) == sizeof(T))
	{
		sm.xstage = reinterpret_cast<S*>(w.xstage);
		sm.smhy = reinterpret_cast<S*>(w.gbuf);
	}
	else
	{
		sm.xstage = r;
		r += p.cmax;
		sm.smhy = r;
	}
}

// 16-byte LDS accesses
struct alignas(16) F4
{
	float a, b, c, d;
};
struct alignas(16) D2
{
	double a, b;
};
struct alignas(16) I4
{
	int a, b, c, d;
};
// three reals of a record of 4 (FP32: one 16-byte access)
__device__ inline V3<float> ld_rec(const float* p)
{
	const F4 v = *reinterpret_cast<const F4*>(p);
	return {v.a, v.b, v.c};
}
__device__ inline V3<double> ld_rec(const double* p) { return ld3(p); }
__device__ inline Q4<float> ld_quat(const float* p)
{
	const F4 v = *reinterpret_cast<const F4*>(p);
	return {v.a, v.b, v.c, v.d};
}
__device__ inline Q4<double> ld_quat(const double* p)
{
	const D2 u = *reinterpret_cast<const D2*>(p), v = *reinterpret_cast<const D2*>(p + 2);
	return {u.a, u.b, v.a, v.b};
}
__device__ inline void st_quat(float* p, Q4<float> q) { *reinterpret_cast<F4*>(p) = F4{q.a, q.b, q.c, q.d}; }
__device__ inline void st_quat(double* p, Q4<double> q)
{
	*reinterpret_cast<D2*>(p) = D2{q.a, q.b};
	*reinterpret_cast<D2*>(p + 2) = D2{q.c, q.d};
}
// an atom's entry of the coordinate or force array
__device__ inline V3<float> ld_atom(const float* p, int i) { return ld_rec(p + 4 * i); }
__device__ inline V3<double> ld_atom(const double* p, int i) { return ld3(p + 3 * i); }
__device__ inline void st_atom(float* p, int i, V3<float> v) { *reinterpret_cast<F4*>(p + 4 * i) = F4{v.x, v.y, v.z, 0.0f}; }
__device__ inline void st_atom(double* p, int i, V3<double> v) { st3(p + 3 * i, v); }
// FP32: an atom's force with its receptor energy in the fourth word
__device__ inline void st_force(float* p, int i, V3<float> v, float e) { *reinterpret_cast<F4*>(p + 4 * i) = F4{v.x, v.y, v.z, e}; }
// a frame's origin and rotation matrix
__device__ inline void ld_frame(const float* p, V3<float>& o, float* R)
{
	const F4 u = *reinterpret_cast<const F4*>(p), v = *reinterpret_cast<const F4*>(p + 4),
			 w = *reinterpret_cast<const F4*>(p + 8);
	o = {u.a, u.b, u.c};
	R[0] = u.d, R[1] = v.a, R[2] = v.b, R[3] = v.c, R[4] = v.d, R[5] = w.a, R[6] = w.b, R[7] = w.c, R[8] = w.d;
}
__device__ inline void ld_frame(const double* p, V3<double>& o, double* R)
{
	D2 v[6];
	for (int k = 0; k < 6; k++)
		v[k] = *reinterpret_cast<const D2*>(p + 2 * k);
	o = {v[0].a, v[0].b, v[1].a};
	R[0] = v[1].b, R[1] = v[2].a, R[2] = v[2].b, R[3] = v[3].a, R[4] = v[3].b, R[5] = v[4].a, R[6] = v[4].b,
	R[7] = v[5].a, R[8] = v[5].b;
}
template<typename T>
__device__ inline void st_frame(T* p, V3<T> o, const T* R)
{
	st3(p, o);
	for (int k = 0; k < 9; k++)
		p[3 + k] = R[k];
}
template<typename T>
__device__ inline V3<T> frame_origin(const WaveMem<T>& W, int f) { return ld3(W.fr + FRAME_REALS * f); }

// receptor back ends: precomputed maps (smina's cache) or the receptor
// atoms themselves (non_cache)
enum Backend
{
	BK_MAPS = 0,
	BK_DIRECT = 1
};

// the evaluation back end
template<typename T>
struct EvalCtx
{
	TablePtrs<T> tab;
	int backend;       // 0: receptor maps (cache), 1: direct receptor (non_cache)
	GridPtrs<T> grid;
	ReceptorPtrs<T> rec;
	T slope;
	T v[3];
	int* error;        // set to 1 on an exact atom overlap (non_cache)
	// the user grid (--user_grid), one corner-packed map: added by the
	// direct back end at each heavy atom with its slope, and by the final
	// rescoring (the maps carry it from their build)
	GridPtrs<T> ug;
	int has_ug;
};

// the context's hot scalars in registers of their own
template<typename T>
__device__ __forceinline__ GridPtrs<T> own_grid(GridPtrs<T> g)
{
	g.cells = own(g.cells);
	g.ncells = own(g.ncells);
	g.slope = own(g.slope);
	for (int d = 0; d < 3; d++)
	{
		g.dim[d] = own(g.dim[d]);
		g.init[d] = own(g.init[d]);
		g.factor[d] = own(g.factor[d]);
		g.factor_inv[d] = own(g.factor_inv[d]);
		g.dim_fl_minus_1[d] = own(g.dim_fl_minus_1[d]);
	}
	return g;
}
template<typename T, int BK>
__device__ __forceinline__ EvalCtx<T> own_context(EvalCtx<T> ec)
{
	ec.tab.smooth = own(ec.tab.smooth);
	ec.tab.n = own(ec.tab.n);
	ec.tab.factor_t = own(ec.tab.factor_t);
	ec.tab.cutoff_t = own(ec.tab.cutoff_t);
	for (int d = 0; d < 3; d++)
		ec.v[d] = own(ec.v[d]);
	if constexpr (BK == BK_MAPS)
		ec.grid = own_grid(ec.grid);
	else
	{
		ec.slope = own(ec.slope);
		ec.rec.cell_start = own(ec.rec.cell_start);
		ec.rec.cell_recs = own(ec.rec.cell_recs);
		for (int d = 0; d < 3; d++)
		{
			ec.rec.cell_off[d] = own(ec.rec.cell_off[d]);
			ec.rec.cell_dim[d] = own(ec.rec.cell_dim[d]);
			ec.rec.begin[d] = own(ec.rec.begin[d]);
			ec.rec.end[d] = own(ec.rec.end[d]);
			ec.rec.enabled[d] = own(ec.rec.enabled[d]);
		}
	}
	return ec;
}

// the model a wave works on: counts, and the packed records of the blobs
// (layout.h) in LDS
template<typename T>
struct MV
{
	ModelHdr h;
	const int2* am;    // per movable atom
	const int* type;   // all atoms
	const int* code;   // neighbour codes
	const int* prec;   // pair records
	const int2* fm;    // per frame
	const int* fpath;  // root-to-frame paths, frame indices as bytes, MAX_PATH / 4 words per frame
	const int* child;  // per frame: first entry of clist and the number of children
	const int* clist;
	const int* heavy;
	const int* tree;   // TR_FIELDS per tree
	const int* cmap;   // per conf element
	const int* gmap;   // per change element
	const T* xyz0;     // [all atoms][3]
	const T* local;    // [movable][4]
	const T* forig;    // [frames][4]
	const T* faxis;    // [frames][4]
	const T* charge;   // partial charges, movable then fixed atoms

	__device__ __forceinline__ int tr(int t, int field) const { return tree[TR_FIELDS * t + field]; }
};

// FP32 neighbour codes as staged in LDS: the partner's and the slot's byte
// offsets in the coordinate and pair arrays, so that an address is one add
__device__ __forceinline__ int staged_code(int c) { return code_partner(c) * 16 | int(unsigned(code_slot(c)) << 18); }
__device__ __forceinline__ V3<float> code_atom(const WaveMem<float>& W, int c)
{
	return ld_rec(reinterpret_cast<const float*>(reinterpret_cast<const char*>(W.coords) + (c & 0xffff)));
}
__device__ __forceinline__ float code_force(const WaveMem<float>& W, int c)
{
	return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(W.pf) + (unsigned(c) >> 16));
}

// copy model m into the workgroup's LDS (every thread of the block takes
// part; the caller synchronises the block afterwards) and view it there.
// The movable atoms' records come first in the int blob and take their
// type's map slot on the way.
template<typename T>
__device__ inline MV<T> stage_model(const BatchPtrs<T>& B, int m, unsigned char* lds, const WavePlan& plan,
		const int* slot_of)
{
	const ModelHdr h = B.hdr[m];
	int* li = reinterpret_cast<int*>(lds);
	T* lt = reinterpret_cast<T*>(lds + (plan.imax + 3) / 4 * 16);
	const int tid = int(threadIdx.x), nt = int(blockDim.x);
	const int* gi = B.iblob + h.iblob_off;
	for (int k = tid; k < h.natoms; k += nt)
	{
		const int w = gi[2 * k];
		li[2 * k] = slot_of && atom_heavy(w) ? atom_with_slot(w, slot_of[atom_type_of(w)]) : w;
		li[2 * k + 1] = gi[2 * k + 1];
	}
	for (int k = 2 * h.natoms + tid; k < h.iblob_len; k += nt)
	{
		const int w = gi[k];
		li[k] = !Real<T>::ordered && unsigned(k - h.o_code) < unsigned(h.ncodes) ? staged_code(w) : w;
	}
	for (int k = tid; k < h.tblob_len; k += nt)
		lt[k] = B.tblob[h.tblob_off + k];
	MV<T> v;
	v.h = h;
	v.h.natoms = own(uniform(h.natoms));
	v.h.ninflex = own(uniform(h.ninflex));
	v.h.nframes = own(uniform(h.nframes));
	v.h.ntrees = own(uniform(h.ntrees));
	v.h.npairs = own(uniform(h.npairs));
	v.h.nother = own(uniform(h.nother));
	v.h.conf_size = own(uniform(h.conf_size));
	v.h.change_size = own(uniform(h.change_size));
	v.h.heavy = own(uniform(h.heavy));
	v.h.nlevels = own(uniform(h.nlevels));
	v.h.path_ok = own(uniform(h.path_ok));
	v.h.one_ligand = own(uniform(h.one_ligand));
	v.am = reinterpret_cast<const int2*>(li);
	v.type = li + own(uniform(h.o_type));
	v.code = li + own(uniform(h.o_code));
	v.prec = li + own(uniform(h.o_prec));
	v.fm = reinterpret_cast<const int2*>(li + own(uniform(h.o_fm)));
	v.fpath = li + own(uniform(h.o_fpath));
	v.child = li + own(uniform(h.o_child));
	v.clist = li + own(uniform(h.o_clist));
	v.heavy = li + own(uniform(h.o_heavy));
	v.tree = li + own(uniform(h.o_tree));
	v.cmap = li + own(uniform(h.o_cmap));
	v.gmap = li + own(uniform(h.o_gmap));
	v.xyz0 = lt + own(uniform(h.o_xyz0));
	v.local = lt + own(uniform(h.o_local));
	v.forig = lt + own(uniform(h.o_forig));
	v.faxis = lt + own(uniform(h.o_faxis));
	v.charge = lt + own(uniform(h.o_charge));
	return v;
}

// ------------------------------------------------------------------ set_conf
// model::set (src/lib/model.cpp:837-841): frames level by level
// (rigid_body::set_conf, first_segment::set_conf, segment::set_conf,
// src/lib/tree.h:111-195), then every atom x = origin + R * local.  One lane
// per frame (at most 64).
template<typename T>
__device__ __forceinline__ void set_conf(const MV<T>& m, WaveMem<T>& W, T x_lane)
{
	const int lane = lane_id();
	if (lane < m.h.conf_size)
		W.xstage[lane] = x_lane;
	lsync();
	const int F = m.h.nframes;
	const int f = lane;
	if (!Real<T>::ordered && m.h.path_ok)
	{
		// Ancestor walk.  A segment's rotation q(R_p l, theta) * q_p equals
		// q_p * q(l, theta), l its axis in the input coordinates (every frame
		// starts unrotated), so each frame's own factor is made once by its
		// lane and the walk composes the path's factors and rotates its
		// relative origins.
		int fx = 0;
		if (f < F)
		{
			fx = m.fm[f].x;
			const int ci = frame_conf(fx);
			Q4<T> lq;
			if (frame_kind(fx) == SGPU_FRAME_RIGID_ROOT)
				lq = {W.xstage[ci + 3], W.xstage[ci + 4], W.xstage[ci + 5], W.xstage[ci + 6]};
			else
				lq = axis_angle_q(ld_rec(m.faxis + 4 * f), W.xstage[ci]);
			st_quat(W.fq + QUAT_REALS * f, lq);
		}
		lsync();
		if (f < F)
		{
			const int d = frame_depth(fx) + 1;
			const int* path = m.fpath + f * (MAX_PATH / 4);
			int word = path[0];
			const int r = word & 255;
			const int rx = m.fm[r].x;
			const int rci = frame_conf(rx);
			V3<T> o = frame_kind(rx) == SGPU_FRAME_RIGID_ROOT
					? v3(W.xstage[rci], W.xstage[rci + 1], W.xstage[rci + 2])
					: ld_rec(m.forig + 4 * r);
			Q4<T> q = ld_quat(W.fq + QUAT_REALS * r);
			Q4<T> qp = {T(1), T(0), T(0), T(0)};
			for (int k = 1; k < d; k++)
			{
				if ((k & 3) == 0)
					word = path[k >> 2];
				const int c = (word >> (8 * (k & 3))) & 255;
				const Q4<T> qc = ld_quat(W.fq + QUAT_REALS * c);
				o = o + q_rotate(q, ld_rec(m.forig + 4 * c));
				qp = q;
				q = qmul(q, qc);
			}
			T R[9];
			q_to_mat(q, R);
			st_frame(W.fr + FRAME_REALS * f, o, R);
			// the world axis: the frame's own axis under its parent's rotation
			// (a first segment's parent rotation is the identity)
			if (frame_kind(fx) != SGPU_FRAME_RIGID_ROOT)
				st3(W.fax + QUAT_REALS * f, q_rotate(qp, ld_rec(m.faxis + 4 * f)));
		}
		lsync();
	}
	else
	{
		// Level by level in smina's order; the half angle's cosine and sine
		// depend on the conf alone, so every frame makes them once before the
		// levels.
		int fx = 0, parent = 0;
		T ch = 1, sh = 0;
		if (f < F)
		{
			const int2 fm = m.fm[f];
			fx = fm.x;
			parent = frame_parent(fm.y);
			if (frame_kind(fx) != SGPU_FRAME_RIGID_ROOT)
			{
				const Q4<T> h = axis_angle_q(v3(T(1), T(0), T(0)), W.xstage[frame_conf(fx)]);
				ch = h.a;
				sh = h.b;
			}
		}
		for (int L = 0; L < m.h.nlevels; L++)
		{
			if (f < F && frame_depth(fx) == L)
			{
				const int kind = frame_kind(fx);
				const int ci = frame_conf(fx);
				Q4<T> q;
				V3<T> o;
				if (kind == SGPU_FRAME_RIGID_ROOT)
				{
					o = v3(W.xstage[ci], W.xstage[ci + 1], W.xstage[ci + 2]);
					q = {W.xstage[ci + 3], W.xstage[ci + 4], W.xstage[ci + 5], W.xstage[ci + 6]};
				}
				else if (kind == SGPU_FRAME_FIRST_SEGMENT)
				{
					o = ld_rec(m.forig + 4 * f);
					const V3<T> ax = ld_rec(m.faxis + 4 * f);
					q = {ch, sh * ax.x, sh * ax.y, sh * ax.z};
					st3(W.fax + QUAT_REALS * f, ax);
				}
				else
				{
					T pR[9];
					V3<T> po;
					ld_frame(W.fr + FRAME_REALS * parent, po, pR);
					const Q4<T> pq = ld_quat(W.fq + QUAT_REALS * parent);
					o = po + mat_vec(pR, ld_rec(m.forig + 4 * f));
					const V3<T> ax = mat_vec(pR, ld_rec(m.faxis + 4 * f));
					st3(W.fax + QUAT_REALS * f, ax);
					q = qmul(Q4<T>{ch, sh * ax.x, sh * ax.y, sh * ax.z}, pq);
					q_normalize_approx(q);
				}
				T R[9];
				q_to_mat(q, R);
				st_frame(W.fr + FRAME_REALS * f, o, R);
				st_quat(W.fq + QUAT_REALS * f, q);
			}
			lsync();
		}
	}
	for (int i = lane; i < m.h.natoms; i += WAVE)
	{
		T R[9];
		V3<T> o;
		ld_frame(W.fr + FRAME_REALS * atom_frame(m.am[i].x), o, R);
		st_atom(W.coords, i, o + mat_vec(R, ld_rec(m.local + 4 * i)));
	}
	lsync();
}

// what a wave's LDS holds throughout a kernel: the hydrogens' forces (FP64),
// the fixed atoms (flexible-residue atoms that do not move) after the movable ones in the
// coordinate array, and the pair slot of the lists' padding, no force
template<typename T, bool PS>
__device__ inline void init_wave(const MV<T>& m, WaveMem<T>& W)
{
	if constexpr (Real<T>::ordered) // the hydrogens' forces, which stay 0
		for (int i = lane_id(); i < m.h.natoms; i += WAVE)
			st_atom(W.forces, i, v3(T(0), T(0), T(0)));
	if (PS && lane_id() == 0)
	{
		W.pf[0] = 0;
		if constexpr (Real<T>::ordered)
			W.pf[1] = -1;
	}
	for (int k = lane_id(); k < m.h.ninflex; k += WAVE)
		st_atom(W.coords, m.h.natoms + k, ld3(m.xyz0 + 3 * (m.h.natoms + k)));
	lsync();
}

// precalculate_splines::eval_deriv, one component, no slow terms
// (src/lib/precalculate.h:418-450) with Spline::eval_deriv
// (src/lib/splines.h:103-121): the spline at r = sqrt(r2), its derivative
// over r, in FP64 (the FP32 search rounds the results)
template<typename T>
__device__ inline void spline_deriv(const TablePtrs<T>& tab, int tri, T r2, T& e, T& dor)
{
	const double r = __builtin_sqrt(double(r2));
	double val, der;
	spline_eval(tab.spl, tab.spl_cut, tab.fraction, tab.nseg, tri, r, val, der);
	e = T(val);
	dor = T(der / r);
}

// precalculate_linear_element::eval_deriv, one component
// (src/lib/precalculate.h:111-151), or the spline's
template<typename T>
__device__ inline void table_deriv(const TablePtrs<T>& tab, int tri, T r2, T& e, T& dor)
{
	if (tab.kind == 1)
	{
		spline_deriv(tab, tri, r2, e, dor);
		return;
	}
	const T r2f = tab.factor_t * r2;
	const int i1 = int(r2f);
	const T rem = r2f - T(i1);
	const T* p = tab.smooth + (size_t(tri) * tab.n + i1) * 2;
	const T e1 = p[0], d1 = p[1], e2 = p[2], d2 = p[3];
	e = e1 + rem * (e2 - e1);
	dor = d1 + rem * (d2 - d1);
}

// the four-component knots of a pair with charges qa, qb in table order
// (the atom of the smaller type first): result_components::eval
// (src/lib/result_components.h:73-79) of each knot's value and derivative,
// c0 + |qa| c1 + |qb| c2 + qa qb c3 summed in that order.  p: the pair's
// (e, dor) row at knot i1 in smooth, q: its row in qsmooth.
template<typename T>
__device__ inline void charged_knots(const T* p, const T* q, T qa, T qb, T& e1, T& d1, T& e2, T& d2)
{
	const T aa = Real<T>::abs(qa), ab = Real<T>::abs(qb), qq = qa * qb;
	e1 = p[0] + aa * q[0] + ab * q[2] + qq * q[4];
	d1 = p[1] + aa * q[1] + ab * q[3] + qq * q[5];
	e2 = p[2] + aa * q[6] + ab * q[8] + qq * q[10];
	d2 = p[3] + aa * q[7] + ab * q[9] + qq * q[11];
}

// precalculate_linear::eval_deriv (src/lib/precalculate.h:245-293) of
// atoms of types t1, t2 and charges q1, q2 with four-component tables: the
// element of (min type, max type) with the atoms in that order
template<typename T>
__device__ inline void table_deriv_charged(const TablePtrs<T>& tab, int t1, int t2, T q1, T q2, T r2, T& e, T& dor)
{
	const T r2f = tab.factor_t * r2;
	const int i1 = int(r2f);
	const T rem = r2f - T(i1);
	const size_t k = size_t(tri_index_permissive(t1, t2)) * tab.n + i1;
	const bool in_order = t1 <= t2;
	T e1, d1, e2, d2;
	charged_knots(tab.smooth + 2 * k, tab.qsmooth + 6 * k, in_order ? q1 : q2, in_order ? q2 : q1, e1, d1, e2, d2);
	e = e1 + rem * (e2 - e1);
	dor = d1 + rem * (d2 - d1);
}

// non_cache::eval_deriv of one atom (src/lib/non_cache.cpp:109-191): box
// clamp with penalty, then the receptor atoms of the clamped point's cell.
// q1: the atom's partial charge (read with four-component tables only).
template<typename T>
__device__ inline T direct_term(const EvalCtx<T>& ec, int t1, T q1, V3<T> ac, V3<T>& out)
{
	const ReceptorPtrs<T>& r = ec.rec;
	T a[3] = {ac.x, ac.y, ac.z};
	T adj[3] = {ac.x, ac.y, ac.z};
	T oobd[3] = {0, 0, 0};
	T oob = 0;
	for (int j = 0; j < 3; j++)
		if (r.enabled[j])
		{
			if (a[j] < T(r.begin[j]))
			{
				adj[j] = T(r.begin[j]);
				oobd[j] = -1;
				oob += Real<T>::abs(a[j] - T(r.begin[j]));
			}
			else if (a[j] > T(r.end[j]))
			{
				adj[j] = T(r.end[j]);
				oobd[j] = 1;
				oob += Real<T>::abs(a[j] - T(r.end[j]));
			}
		}
	oob *= ec.slope;
	for (int j = 0; j < 3; j++)
		oobd[j] *= ec.slope;
	int ix[3];
	for (int j = 0; j < 3; j++)
	{
		ix[j] = int(__builtin_floor(double(adj[j]) / 3.0)) - r.cell_off[j];
		ix[j] = ix[j] < 0 ? 0 : (ix[j] >= r.cell_dim[j] ? r.cell_dim[j] - 1 : ix[j]);
	}
	const int cell = ix[0] + r.cell_dim[0] * (ix[1] + r.cell_dim[1] * ix[2]);
	T this_e = 0;
	V3<T> deriv = v3(T(0), T(0), T(0));
	const V3<T> adjv = v3(adj[0], adj[1], adj[2]);
	// The list in batches of REC_BATCH, accumulated in list order: the next
	// batch's records are loaded ahead and a batch's table rows are in flight
	// together (an entry out of range reads row 0 and is skipped).  The loop
	// is bound by the latency of these dependent loads, not by their bytes:
	// one entry at a time (index, position, type, row, each waited for) took
	// 330 ms against 121 ms for the FP32 refinement of the 1,024-ligand
	// screen's saved poses, and 230 ms against 160 ms for the FP64 refinement
	// of 256 parsed poses with splines.
	const int k0 = r.cell_start[cell], k1 = r.cell_start[cell + 1];
	RecAtom<T> next[REC_BATCH];
#pragma unroll
	for (int u = 0; u < REC_BATCH; u++)
		next[u] = r.cell_recs[k0 + u < k1 ? k0 + u : 0];
	for (int k = k0; k < k1; k += REC_BATCH)
	{
		V3<T> rba[REC_BATCH];
		T r2[REC_BATCH], pe[REC_BATCH], pd[REC_BATCH];
		int type[REC_BATCH], idx[REC_BATCH];
		bool ok[REC_BATCH];
#pragma unroll
		for (int u = 0; u < REC_BATCH; u++)
		{
			rba[u] = adjv - v3(next[u].x, next[u].y, next[u].z);
			r2[u] = norm_sqr(rba[u]);
			ok[u] = k + u < k1 && r2[u] < ec.tab.cutoff_t;
			type[u] = rec_type(next[u]);
			idx[u] = rec_index(next[u]);
		}
#pragma unroll
		for (int u = 0; u < REC_BATCH; u++)
			next[u] = r.cell_recs[k + REC_BATCH + u < k1 ? k + REC_BATCH + u : 0];
		if (ec.tab.kind == 1)
		{
			SplineRow row[REC_BATCH];
#pragma unroll
			for (int u = 0; u < REC_BATCH; u++)
				row[u] = spline_row(ec.tab.spl, ec.tab.spl_cut, ec.tab.fraction, ec.tab.nseg,
						tri_index_permissive(t1, type[u]), __builtin_sqrt(double(ok[u] ? r2[u] : T(0))));
#pragma unroll
			for (int u = 0; u < REC_BATCH; u++)
			{
				double val, der;
				spline_value(row[u], val, der);
				pe[u] = T(val);
				pd[u] = T(der / row[u].r);
			}
		}
		else if (ec.tab.ncomp == 4)
		{
#pragma unroll
			for (int u = 0; u < REC_BATCH; u++)
				table_deriv_charged(ec.tab, t1, type[u], q1, r.charge[ok[u] ? idx[u] : 0], ok[u] ? r2[u] : T(0), pe[u],
						pd[u]);
		}
		else
		{
			T e1[REC_BATCH], d1[REC_BATCH], e2[REC_BATCH], d2[REC_BATCH], rem[REC_BATCH];
#pragma unroll
			for (int u = 0; u < REC_BATCH; u++)
			{
				const T r2f = ec.tab.factor_t * r2[u];
				const int i1 = ok[u] ? int(r2f) : 0;
				rem[u] = r2f - T(i1);
				const T* p = ec.tab.smooth + (ok[u] ? size_t(tri_index_permissive(t1, type[u])) * ec.tab.n + i1 : 0) * 2;
				e1[u] = p[0];
				d1[u] = p[1];
				e2[u] = p[2];
				d2[u] = p[3];
			}
#pragma unroll
			for (int u = 0; u < REC_BATCH; u++)
			{
				pe[u] = e1[u] + rem[u] * (e2[u] - e1[u]);
				pd[u] = d1[u] + rem[u] * (d2[u] - d1[u]);
			}
		}
#pragma unroll
		for (int u = 0; u < REC_BATCH; u++)
			if (ok[u])
			{
				if (r2[u] < Real<T>::eps())
					atomicOr(ec.error, 1); // bit 0: exact overlap (other bits belong to the caller)
				this_e += pe[u];
				deriv.x += pd[u] * rba[u].x;
				deriv.y += pd[u] * rba[u].y;
				deriv.z += pd[u] * rba[u].z;
			}
	}
	// the user grid at the atom's own position, with the back end's slope
	V3<T> ug_deriv = v3(T(0), T(0), T(0));
	if (ec.has_ug)
		this_e += grid_finish(ec.ug, grid_fetch(ec.ug, 0, ac), T(1000), ec.slope, ug_deriv);
	deriv.x += ug_deriv.x;
	deriv.y += ug_deriv.y;
	deriv.z += ug_deriv.z;
	curl(this_e, deriv, ec.v[1]);
	out = v3(deriv.x + oobd[0], deriv.y + oobd[1], deriv.z + oobd[2]);
	return this_e + oob;
}

// The pairs of atom i, each evaluated from this end, forces added to f in
// evaluation order; the pair's first atom leaves its energy in pbuf.  For
// FP64 models whose pairs don't fit LDS.
template<typename T, bool SPL>
__device__ __forceinline__ void atom_pairs(const MV<T>& m, const EvalCtx<T>& ec, const WaveMem<T>& W, T* pbuf, int i,
		V3<T> xi, int k0, int k1, V3<T>& f)
{
	const T cutoff_sqr = ec.tab.cutoff_t;
	for (int k = k0; k < k1; k += PAIR_BATCH)
	{
		int cd[PAIR_BATCH];
		bool isb[PAIR_BATCH];
		T rx[PAIR_BATCH], ry[PAIR_BATCH], rz[PAIR_BATCH], r2[PAIR_BATCH], rem[PAIR_BATCH];
		T e1[PAIR_BATCH], d1[PAIR_BATCH], e2[PAIR_BATCH], d2[PAIR_BATCH];
#pragma unroll
		for (int u = 0; u < PAIR_BATCH; u++)
		{
			const int code = m.code[k + u];
			const int slot = code_slot(code);
			const int pr = m.prec[slot > 0 ? slot - 1 : 0];
			const int j = code_partner(code);
			const bool is_b = slot > 0 && prec_b(pr) == i;
			cd[u] = slot;
			isb[u] = is_b;
			const V3<T> xj = ld_atom(W.coords, j);
			// r = x_b - x_a
			rx[u] = is_b ? xi.x - xj.x : xj.x - xi.x;
			ry[u] = is_b ? xi.y - xj.y : xj.y - xi.y;
			rz[u] = is_b ? xi.z - xj.z : xj.z - xi.z;
			r2[u] = sqr(rx[u]) + sqr(ry[u]) + sqr(rz[u]);
			// precalculate_linear_element::eval_deriv (src/lib/precalculate.h:111-151)
			if (SPL && ec.tab.kind == 1)
			{
				// the spline's value and derivative over r, carried
				// through the interpolation below unchanged (rem 0)
				if (r2[u] < cutoff_sqr)
					spline_deriv(ec.tab, prec_tri(pr), r2[u], e1[u], d1[u]);
				else
					e1[u] = d1[u] = 0;
				rem[u] = 0;
				e2[u] = e1[u];
				d2[u] = d1[u];
				continue;
			}
			const T r2f = ec.tab.factor_t * r2[u];
			const int i1 = r2[u] < cutoff_sqr ? int(r2f) : 0;
			rem[u] = r2f - T(i1);
			const size_t kn = size_t(prec_tri(pr)) * ec.tab.n + i1;
			const T* tp = ec.tab.smooth + kn * 2;
			if (SPL && ec.tab.ncomp == 4)
			{
				// four components: the pair's charges in table order
				const int ia = is_b ? j : i, ib = is_b ? i : j;
				const bool in_order = m.type[ia] <= m.type[ib];
				const T qa = m.charge[in_order ? ia : ib], qb = m.charge[in_order ? ib : ia];
				charged_knots(tp, ec.tab.qsmooth + kn * 6, qa, qb, e1[u], d1[u], e2[u], d2[u]);
				continue;
			}
			e1[u] = tp[0];
			d1[u] = tp[1];
			e2[u] = tp[2];
			d2[u] = tp[3];
		}
#pragma unroll
		for (int u = 0; u < PAIR_BATCH; u++)
		{
			if (cd[u] == 0)
				break; // the list's padding
			const int pair = cd[u] - 1;
			const bool is_b = isb[u];
			T pe = 0;
			if (r2[u] < cutoff_sqr)
			{
				pe = e1[u] + rem[u] * (e2[u] - e1[u]);
				const T dor = d1[u] + rem[u] * (d2[u] - d1[u]);
				V3<T> fr = v3(dor * rx[u], dor * ry[u], dor * rz[u]);
				curl(pe, fr, pair < m.h.nother ? ec.v[2] : ec.v[0]);
				f = is_b ? f + fr : f - fr;
			}
			if (!is_b)
				pbuf[pair] = pe;
		}
	}
}

// a frame's share of the gradient: a root's force and torque, a segment's
// torque about its axis
template<typename T>
__device__ __forceinline__ void store_frame_gradient(const MV<T>& m, WaveMem<T>& W, int fx, int f, V3<T> force,
		V3<T> torque)
{
	const int gi = frame_change(fx);
	if (frame_kind(fx) == SGPU_FRAME_RIGID_ROOT)
	{
		st3(W.gbuf + gi, force);
		st3(W.gbuf + gi + 3, torque);
	}
	else
		W.gbuf[gi] = dot(torque, ld3(W.fax + QUAT_REALS * f));
}

// ------------------------------------------------------------------ eval_deriv
// acc plus the 16 lanes of each row of v in lane order, row by row: every
// lane of a row ends with its row's sum.  One fused multiply-add by 1 per
// element (the exact sum, rounded once), its operand broadcast within the
// row by the instruction.  The whole wave must be active.
__device__ __forceinline__ double row_ordered_add(double acc, double v)
{
#define SGPU_ROW_ADD(k) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #k " row_mask:0xf bank_mask:0xf\n\t"
	asm("s_nop 1\n\t" SGPU_ROW_ADD(0) SGPU_ROW_ADD(1) SGPU_ROW_ADD(2) SGPU_ROW_ADD(3) SGPU_ROW_ADD(4) SGPU_ROW_ADD(5)
					SGPU_ROW_ADD(6) SGPU_ROW_ADD(7) SGPU_ROW_ADD(8) SGPU_ROW_ADD(9) SGPU_ROW_ADD(10) SGPU_ROW_ADD(11)
							SGPU_ROW_ADD(12) SGPU_ROW_ADD(13) SGPU_ROW_ADD(14) SGPU_ROW_ADD(15)
			: "+&v"(acc) // (not v's register: every instruction reads v)
			: "v"(v), "v"(1.0));
#undef SGPU_ROW_ADD
	return acc;
}

// The sum of v over lanes 0..cnt-1 in lane order, added to acc (uniform);
// the lanes from cnt on hold 0, which changes no sum.  The whole wave must be
// active.  Bound by the chain of dependent additions: 64 take 505 clocks,
// against 1,380 with each element read into scalar registers.
__device__ __forceinline__ double ordered_add(double acc, double v, int cnt)
{
	for (int l = 0; l < cnt; l += 16)
		acc = readlane(row_ordered_add(acc, v), l);
	return acc;
}
__device__ __forceinline__ float ordered_add(float acc, float v, int cnt)
{
	for (int l = 0; l < cnt; l++)
		acc += readlane(v, l);
	return acc;
}

// The ordered search's energies of pairs [begin, end) from the wave's global
// scratch, in list order (other pairs, then each ligand's)
template<typename T>
__device__ __forceinline__ T ordered_pair_sum(const T* pbuf, int begin, int end)
{
	T acc = 0;
	for (int p = begin; p < end; p += WAVE)
		acc = ordered_add(acc, p + lane_id() < end ? pbuf[p + lane_id()] : T(0), end - p < WAVE ? end - p : WAVE);
	return acc;
}

// force x (xi - xj) with the product rounded before it is added (the pair's
// own force, as both of its atoms add it)
__device__ __forceinline__ V3<float> rounded_scale(float k, V3<float> d)
{
	V3<float> f = v3(k * d.x, k * d.y, k * d.z);
	asm("" : "+v"(f.x), "+v"(f.y), "+v"(f.z)); // not fused into the sum
	return f;
}

// a number of passes known at compile time
template<int N>
struct BatchSize
{
	static constexpr int value = N;
};

// model::eval_deriv (src/lib/model.cpp:969-983).  x: conf element in this
// lane; returns e (uniform) and the gradient element in g_lane.  BK: the
// receptor back end (BK_MAPS or BK_DIRECT), fixed per kernel.  SPL: the
// pair loops can read the spline and four-component tables (off in the search
// kernel of smina's own search, which keeps its registers without them).
//
// Intramolecular pairs are evaluated once each, pair-parallel (pair t * 64 +
// lane), and leave a scalar per pair in LDS; each atom then walks its
// neighbour list in evaluation order and adds factor x (x_i - x_j), which is
// the pair's force on it from either end with the same rounding.  One float a
// pair (instead of the force's three) halves a large ligand's LDS.  FP64
// keeps two doubles, the table's derivative and the curl factor: smina rounds
// their product with the distance in two steps.
// PS false (FP64 models whose pairs don't fit LDS): each atom evaluates every
// pair of its list itself; pbuf is then, and for several ligands, the wave's
// pair-energy scratch in global memory.
template<typename T, int BK, bool SPL = true, bool PS = true, bool TAIL = true>
__device__ __forceinline__ T eval_deriv(const MV<T>& m, const EvalCtx<T>& ec, WaveMem<T>& W, T* pbuf, T x_lane,
		T& g_lane)
{
	constexpr bool ORD = Real<T>::ordered;
	static_assert(PS || ORD, "the FP32 search holds its pairs in LDS");
	const int lane = lane_id();
	set_conf(m, W, x_lane);
	const int N = m.h.natoms;
	const int P = m.h.npairs;
	const T cutoff_sqr = ec.tab.cutoff_t;
	const T factor = ec.tab.factor_t;
	T e_part = 0;           // FP32: this lane's energies
	T e_other = 0, e_lig = 0; // FP64: the other pairs' sum and the ligand's
	// The lanes take the atoms, or of a model with more than 64 atoms but at
	// most 64 heavy ones the heavy atoms, so that they pass once over the
	// atoms, not twice: hydrogens have no receptor term, and no pairs unless
	// the caller's model lists some (then every atom takes a lane: ALL_LANES
	// is past any count)
	const bool by_heavy = N > WAVE && m.h.heavy <= WAVE;
	const int M = by_heavy ? m.h.heavy : N;
	// FP64: the first 64 atoms' map cells are fetched now and consumed after
	// the pairs, which hide the fetch (chains with a CU to themselves)
	GridSample<T> gs0;
	if constexpr (ORD && BK == BK_MAPS)
	{
		const int i = by_heavy ? m.heavy[lane < M ? lane : 0] : lane < N ? lane : 0;
		gs0 = grid_fetch(ec.grid, atom_slot(m.am[i].x), ld_atom(W.coords, i));
	}
	if constexpr (PS)
	{
		// the curl caps of the two pair kinds; a cap below epsilon zeroes the
		// term, as v < epsilon does in curl
		const T v_lig = ec.v[0] < Real<T>::eps() ? T(0) : ec.v[0];
		const T v_oth = ec.v[2] < Real<T>::eps() ? T(0) : ec.v[2];
		const int last_knot = ec.tab.n - 2;
		const int row_bytes = 8 * ec.tab.n;
		const int nother = m.h.nother;
		auto batch = [&](auto size, int t0) __attribute__((always_inline)) {
			constexpr int NB = decltype(size)::value;
			// phases across the batch: records, coordinates, table rows, then
			// the arithmetic, so each phase's loads are in flight together
			int rc[NB];
#pragma unroll
			for (int u = 0; u < NB; u++)
			{
				const int p = (t0 + u) * WAVE + lane;
				rc[u] = m.prec[p < P ? p : 0];
			}
			T rx[NB], ry[NB], rz[NB], r2[NB], rem[NB];
			T e1[NB], d1[NB], e2[NB], d2[NB];
#pragma unroll
			for (int u = 0; u < NB; u++)
			{
				const V3<T> xa = ld_atom(W.coords, prec_a(rc[u])), xb = ld_atom(W.coords, prec_b(rc[u]));
				rx[u] = xb.x - xa.x;
				ry[u] = xb.y - xa.y;
				rz[u] = xb.z - xa.z;
			}
#pragma unroll
			for (int u = 0; u < NB; u++)
			{
				r2[u] = sqr(rx[u]) + sqr(ry[u]) + sqr(rz[u]);
				// precalculate_linear_element::eval_deriv (src/lib/precalculate.h:111-151);
				// the knot is clamped so that the row read stays in the table.
				// With the spline tables, the spline's value and derivative
				// over r pass through the interpolation below unchanged.
				if (SPL && ec.tab.kind == 1)
				{
					if (r2[u] < cutoff_sqr)
						spline_deriv(ec.tab, prec_tri(rc[u]), r2[u], e1[u], d1[u]);
					else
						e1[u] = d1[u] = T(0);
					rem[u] = T(0);
					e2[u] = e1[u];
					d2[u] = d1[u];
					continue;
				}
				const T r2f = factor * r2[u];
				const int i1 = ORD ? (r2[u] < cutoff_sqr ? int(r2f) : 0) : min(int(r2f), last_knot);
				rem[u] = r2f - T(i1);
				// (FP32: a 32-bit byte offset from the scalar base)
				const T* tp;
				if constexpr (ORD)
					tp = ec.tab.smooth + (size_t(prec_tri(rc[u])) * ec.tab.n + i1) * 2;
				else
					tp = reinterpret_cast<const T*>(reinterpret_cast<const char*>(ec.tab.smooth) +
							(__umul24(unsigned(prec_tri(rc[u])), unsigned(row_bytes)) + 8u * unsigned(i1)));
				if (SPL && ec.tab.ncomp == 4)
				{
					// four components: the pair's charges in table order
					const int ia = prec_a(rc[u]), ib = prec_b(rc[u]);
					const bool in_order = m.type[ia] <= m.type[ib];
					const T qa = m.charge[in_order ? ia : ib], qb = m.charge[in_order ? ib : ia];
					charged_knots(tp, ec.tab.qsmooth + 3 * (tp - ec.tab.smooth), qa, qb, e1[u], d1[u], e2[u], d2[u]);
					continue;
				}
				e1[u] = tp[0];
				d1[u] = tp[1];
				e2[u] = tp[2];
				d2[u] = tp[3];
			}
#pragma unroll
			for (int u = 0; u < NB; u++)
			{
				const int base = (t0 + u) * WAVE;
				const int p = base + lane;
				const bool ok = p < P && r2[u] < cutoff_sqr;
				T pe = e1[u] + rem[u] * (e2[u] - e1[u]);
				const T dor = d1[u] + rem[u] * (d2[u] - d1[u]);
				const T v = p < nother ? v_oth : v_lig;
				if constexpr (!ORD)
				{
					// curl (src/lib/curl.h:28-43) without branches
					const T k = pe > 0 ? Real<T>::fdiv(v, v + pe) : T(1);
					const T fk = ok ? dor * (k * k) : T(0);
					e_part += ok ? pe * k : T(0);
					if (p < P)
						W.pf[p + 1] = fk;
				}
				else
				{
					T t2 = 1;
					if (ok && pe > 0)
					{
						const T k = v == T(0) ? T(0) : Real<T>::fdiv(v, v + pe);
						pe *= k;
						t2 = sqr(k);
					}
					if (!ok)
					{
						pe = 0;
						t2 = -1; // no force
					}
					if (p < P)
						*reinterpret_cast<D2*>(W.pf + 2 * (p + 1)) = D2{dor, t2};
					if (!m.h.one_ligand)
					{
						if (p < P)
							pbuf[p] = pe;
					}
					else if (base < P)
					{
						const int cnt = P - base < WAVE ? P - base : WAVE;
						if (base + WAVE <= nother)
							e_other = ordered_add(e_other, pe, WAVE);
						else if (base >= nother)
							e_lig = ordered_add(e_lig, pe, cnt);
						else
						{
							e_other = ordered_add(e_other, p < nother ? pe : T(0), WAVE);
							e_lig = ordered_add(e_lig, p < nother ? T(0) : pe, cnt);
						}
					}
				}
			}
		};
		// TAIL: the last one or two passes take a batch of their own size, so
		// that no pass runs empty (1,024 ligands in FP32: 800 -> 775 ms, in
		// mixed precision 412 -> 399 ms of 256).  The FP32 evaluation of
		// speculative chains, one wave on a SIMD, runs full batches: the
		// extra code cost it more than the empty passes (128 chains of a
		// 38-heavy-atom ligand: 228 against 225 ms).
		if constexpr (TAIL)
		{
			const int passes = (P + WAVE - 1) / WAVE;
			int t0 = 0;
			for (; passes - t0 > 2; t0 += PAIR_BATCH)
				batch(BatchSize<PAIR_BATCH>{}, t0);
			if (passes - t0 == 2)
				batch(BatchSize<2>{}, t0);
			else if (passes - t0 == 1)
				batch(BatchSize<1>{}, t0);
		}
		else
			for (int t0 = 0; t0 * WAVE < P; t0 += PAIR_BATCH)
				batch(BatchSize<PAIR_BATCH>{}, t0);
		lsync();
	}
	// per movable atom: receptor term, then its pair forces in list order
	T e = 0; // FP64: the atoms' sum
	for (int base = 0; base < M; base += WAVE)
	{
		T ea = 0;
		if (base + lane < M)
		{
			const int i = by_heavy ? m.heavy[base + lane] : base + lane;
			const int2 am = m.am[i];
			const int aw = am.x;
			const bool heavy = atom_heavy(aw);
			const V3<T> xi = ld_atom(W.coords, i);
			const int k0 = atom_nbr_begin(am.y), k1 = atom_nbr_end(am.y);
			V3<T> d = v3(T(0), T(0), T(0));
			if constexpr (!ORD)
			{
				// the map gather is issued first and consumed last, so its
				// latency overlaps the list walk
				GridSample<T> gs;
				if constexpr (BK == BK_MAPS)
					gs = grid_fetch(ec.grid, atom_slot(aw), xi);
				V3<T> fp = v3(T(0), T(0), T(0));
				for (int k = k0; k < k1; k += NBR_BATCH)
				{
					const I4 cd = *reinterpret_cast<const I4*>(m.code + k);
					const V3<T> xj[NBR_BATCH] = {code_atom(W, cd.a), code_atom(W, cd.b), code_atom(W, cd.c),
							code_atom(W, cd.d)};
					const T fk[NBR_BATCH] = {code_force(W, cd.a), code_force(W, cd.b), code_force(W, cd.c),
							code_force(W, cd.d)};
#pragma unroll
					for (int u = 0; u < NBR_BATCH; u++)
						fp = fp + rounded_scale(fk[u], xi - xj[u]);
				}
				if (heavy)
				{
					if constexpr (BK == BK_MAPS)
					{
						ea = grid_finish(ec.grid, gs, ec.v[1], d);
						if (SPL && ec.grid.qcells && m.charge[i] != T(0))
							grid_charge_term(ec.grid, atom_slot(aw), xi, ec.v[1], m.charge[i], ea, d);
					}
					else
						ea = direct_term(ec, atom_type_of(aw), m.charge[i], xi, d);
				}
				st_force(W.forces, i, d + fp, ea);
			}
			else
			{
				if (heavy)
				{
					if constexpr (BK == BK_MAPS)
					{
						if (base > 0)
							gs0 = grid_fetch(ec.grid, atom_slot(aw), xi);
						ea = grid_finish(ec.grid, gs0, ec.v[1], d);
						if (SPL && ec.grid.qcells && m.charge[i] != T(0))
							grid_charge_term(ec.grid, atom_slot(aw), xi, ec.v[1], m.charge[i], ea, d);
					}
					else
						ea = direct_term(ec, atom_type_of(aw), m.charge[i], xi, d);
				}
				if constexpr (PS)
					for (int k = k0; k < k1; k += NBR_BATCH)
					{
						const I4 cd = *reinterpret_cast<const I4*>(m.code + k);
						const int c[NBR_BATCH] = {cd.a, cd.b, cd.c, cd.d};
						V3<T> r[NBR_BATCH];
						D2 s[NBR_BATCH];
#pragma unroll
						for (int u = 0; u < NBR_BATCH; u++)
						{
							r[u] = xi - ld_atom(W.coords, code_partner(c[u]));
							s[u] = *reinterpret_cast<const D2*>(W.pf + 2 * code_slot(c[u]));
						}
#pragma unroll
						for (int u = 0; u < NBR_BATCH; u++)
							if (!(s[u].b < 0))
							{
								d.x += s[u].a * r[u].x * s[u].b;
								d.y += s[u].a * r[u].y * s[u].b;
								d.z += s[u].a * r[u].z * s[u].b;
							}
					}
				else
					atom_pairs<T, SPL>(m, ec, W, pbuf, i, xi, k0, k1, d);
				st_atom(W.forces, i, d);
			}
		}
		if constexpr (ORD)
			e = ordered_add(e, ea, M - base < WAVE ? M - base : WAVE);
	}
	lsync();
	const int F = m.h.nframes;
	const int f = lane;
	if constexpr (!ORD)
	{
		// Inclusive prefix sums over the atoms of the force (in place) and of
		// (x - o0) x force (o0: frame 0's origin; into the pair buffer, free
		// now): every frame's subtree is a contiguous atom range, so the
		// derivative reads its sums as two differences
		const V3<T> o0 = frame_origin(W, 0);
		V3<T> carry_f = v3(T(0), T(0), T(0)), carry_t = carry_f;
		for (int base = 0; base < N; base += WAVE)
		{
			const int i = base + lane;
			V3<T> force = v3(T(0), T(0), T(0)), tq = force;
			if (i < N && (!by_heavy || atom_heavy(m.am[i].x)))
			{
				const F4 fe = *reinterpret_cast<const F4*>(W.forces + 4 * i);
				e_part += fe.d;
				force = v3(fe.a, fe.b, fe.c);
				tq = cross(ld_atom(W.coords, i) - o0, force);
			}
			const V3<T> sf = v3(wave_inclusive_scan(force.x), wave_inclusive_scan(force.y),
							  wave_inclusive_scan(force.z)) + carry_f;
			const V3<T> st = v3(wave_inclusive_scan(tq.x), wave_inclusive_scan(tq.y), wave_inclusive_scan(tq.z)) +
					carry_t;
			if (i < N)
			{
				st_atom(W.forces, i, sf);
				st_atom(W.tq, i, st);
			}
			carry_f = v3(readlane(sf.x, WAVE - 1), readlane(sf.y, WAVE - 1), readlane(sf.z, WAVE - 1));
			carry_t = v3(readlane(st.x, WAVE - 1), readlane(st.y, WAVE - 1), readlane(st.z, WAVE - 1));
		}
		lsync();
		e = wave_sum(e_part);
		// derivative, direct: each frame's force and torque over its
		// subtree's atoms (a contiguous range) from the prefix sums, equal to
		// smina's bottom-up accumulation (src/lib/tree.h:88-97, :214-289) up
		// to rounding: torque about the frame's origin o is
		// sum (x - o0) x f - (o - o0) x sum f
		if (f < F)
		{
			const int2 fm = m.fm[f];
			const int b = frame_begin(fm.y), en = frame_send(fm.y);
			V3<T> fs = ld_atom(W.forces, en - 1), ts = ld_atom(W.tq, en - 1);
			if (b > 0)
			{
				fs = fs - ld_atom(W.forces, b - 1);
				ts = ts - ld_atom(W.tq, b - 1);
			}
			const V3<T> to = ts - cross(frame_origin(W, f) - frame_origin(W, 0), fs);
			store_frame_gradient(m, W, fm.x, f, fs, to);
		}
		lsync();
	}
	else
	{
		if (m.h.one_ligand && PS)
		{
			e += e_other;
			e += e_lig;
		}
		else
		{
			gsync(); // the pair energies went through global memory
			e += ordered_pair_sum(pbuf, 0, m.h.nother);
			for (int t = 0; t < m.h.ntrees; t++)
				if (m.tr(t, TR_LIG))
					e += ordered_pair_sum(pbuf, m.tr(t, TR_PB), m.tr(t, TR_PE));
		}
		// derivative: per-frame sums, then the tree bottom-up; a lane keeps
		// its frame's sums until its level
		int2 fm{0, 0};
		int child = 0;
		V3<T> o = v3(T(0), T(0), T(0)), fo = o, to = o;
		if (f < F)
		{
			fm = m.fm[f];
			child = m.child[f];
			o = frame_origin(W, f);
			const int b = frame_begin(fm.y), en = frame_end(fm.y);
#pragma unroll 4
			for (int i = b; i < en; i++)
			{
				const V3<T> fi = ld_atom(W.forces, i);
				fo = fo + fi;
				to = to + cross(ld_atom(W.coords, i) - o, fi);
			}
		}
		for (int L = m.h.nlevels - 1; L >= 0; L--)
		{
			if (f < F && frame_depth(fm.x) == L)
			{
				const int cs = child_start(child), cc = child_count(child);
				for (int k = 0; k < cc; k++)
				{
					const int c = m.clist[cs + k];
					const V3<T> cf = ld3(W.ff + 3 * c);
					fo = fo + cf;
					const V3<T> r = frame_origin(W, c) - o;
					to = to + (cross(r, cf) + ld3(W.ft + 3 * c));
				}
				st3(W.ff + 3 * f, fo);
				st3(W.ft + 3 * f, to);
				store_frame_gradient(m, W, fm.x, f, fo, to);
			}
			lsync();
		}
	}
	g_lane = lane < m.h.change_size ? W.gbuf[lane] : T(0);
	lsync();
	return e;
}

} // namespace sgpu

#endif
