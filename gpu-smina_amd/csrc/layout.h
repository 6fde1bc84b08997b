/*
 * Device-memory layout of the docking search (HBM, gfx950).
 *
 * A batch of models is packed per model into one contiguous int blob and
 * one contiguous real blob (the reference's FlatModel / DevModels,
 * src/gpu/gpu_flatten_data.h:16-46, src/gpu/gpu_dev_structs.h:137).  A
 * workgroup copies its model's two blobs into LDS with coalesced loads once,
 * then every wave of the workgroup (one Monte Carlo chain each, all of the
 * same ligand) reads the model from LDS only.  ModelHdr holds the counts
 * and each array's offset inside the blobs.
 *
 * int blob:  movable atoms' records (two words: frame, type, heavy flag and
 *            map slot; the range of the neighbour list), atom types (movable
 *            then fixed), neighbour codes, pair records, frame records, paths
 *            and children, heavy atoms, trees, conf / change maps;
 * real blob: initial coordinates (movable then fixed, 3 reals each), local
 *            coordinates, frame origins and axes (4 reals each; segment:
 *            relative to the parent), partial charges (movable then fixed).
 * Packed records keep the addresses a wave holds few: with an array for each
 * field the search kernels held some 100 uniform values and moved 130 to 300
 * of them through vector lanes.
 *
 * A neighbour code is one word: the partner atom (bits 0-15) and the pair's
 * slot, its index plus one (16-31).  Each atom's list is padded to a multiple
 * of 4 codes with entries of slot 0 (the atom itself, no force), so that a
 * lane reads 4 codes at once and needs no check for the end of its list.  A
 * pair record is one word: atoms a (0-7) and b (8-15), the table index
 * (16-24).
 *
 * Receptor maps are stored per ligand type as corner-packed cells: for each
 * grid cell (x fastest), its 8 corner values in the order f000 f100 f010
 * f110 f001 f101 f011 f111, so one trilinear gather is one 32-byte (FP32)
 * or 64-byte (FP64) load.
 */
#ifndef SGPU_LAYOUT_H
#define SGPU_LAYOUT_H

#include <hip/hip_runtime.h>

namespace sgpu
{

constexpr int WAVE = 64;
constexpr int LDS_LIMIT = 160 * 1024; // a workgroup's LDS
// A model's limits: those of the calls' interface, within what the packed
// records below hold.
constexpr int MAX_ATOMS = 255;    // movable + fixed atoms (bytes of the pair and frame records)
constexpr int MAX_PAIRS = 8191;
constexpr int MAX_FRAMES = 64;    // a lane each; bytes of the atom records and of the paths
constexpr int MAX_CHANGE = 64;    // a lane per element
constexpr int MAX_CONF = 64;
constexpr int MAX_TREES = 16;
constexpr int MAX_POSES = 64;     // saved minima of a chain: a lane each
constexpr int MAX_PATH = 32;      // frames on a root-to-frame path (ancestor walk of set_conf)
constexpr int MAX_CHAINS_PER_GROUP = 8; // waves of one Monte Carlo workgroup

// conf element kinds: position component, quaternion component a..d, torsion
enum ConfKind
{
	CK_POSITION = 0,
	CK_QUAT0 = 1, // CK_QUAT0 + component
	CK_TORSION = 5
};
// change element kinds: position, orientation component x..z, torsion
enum ChangeKind
{
	GK_POSITION = 0,
	GK_ORIENT0 = 1, // GK_ORIENT0 + component
	GK_TORSION = 4
};

constexpr int NBR_BATCH = 4; // codes a neighbour list is padded to
// The packed fields that a larger limit would overflow: bytes for atoms and
// frames, 16 bits for a range of neighbour codes (two per pair and a list's
// padding), and in the FP32 form of a code (search.h) 16 bits each for the
// byte offsets of an atom's 16 bytes and of a pair's 4.
static_assert(MAX_ATOMS <= 255 && MAX_FRAMES <= 255 && MAX_CONF <= 255 && MAX_CHANGE <= 255, "bytes of the records");
static_assert(2 * MAX_PAIRS + (NBR_BATCH - 1) * MAX_ATOMS <= 0xffff, "a neighbour range in an atom's record");
static_assert(16 * MAX_ATOMS <= 0xffff && 4 * (MAX_PAIRS + 1) <= 0xffff, "byte offsets of a staged neighbour code");
__host__ __device__ inline int make_code(int partner, int slot) { return int(unsigned(partner) | (unsigned(slot) << 16)); }
__host__ __device__ inline int code_partner(int c) { return c & 0xffff; }
__host__ __device__ inline int code_slot(int c) { return int(unsigned(c) >> 16); }

// pair record: atoms a and b, table index
__host__ __device__ inline int make_prec(int a, int b, int tri) { return a | (b << 8) | (tri << 16); }
__host__ __device__ inline int prec_a(int w) { return w & 255; }
__host__ __device__ inline int prec_b(int w) { return (w >> 8) & 255; }
__host__ __device__ inline int prec_tri(int w) { return w >> 16; }

// movable atom's record: word 0 frame (0-7), type (8-15), map slot (16-23),
// heavy (24); word 1 first neighbour code (0-15) and the one past the last
// (16-31)
__host__ __device__ inline int make_atom(int frame, int type, bool heavy) { return frame | (type << 8) | (int(heavy) << 24); }
__host__ __device__ inline int atom_frame(int w) { return w & 255; }
__host__ __device__ inline int atom_type_of(int w) { return (w >> 8) & 255; }
__host__ __device__ inline int atom_slot(int w) { return (w >> 16) & 255; }
__host__ __device__ inline bool atom_heavy(int w) { return (w >> 24) & 1; }
__host__ __device__ inline int atom_with_slot(int w, int slot) { return (w & ~(255 << 16)) | ((slot & 255) << 16); }
__host__ __device__ inline int atom_nbr_begin(int w) { return w & 0xffff; }
__host__ __device__ inline int atom_nbr_end(int w) { return int(unsigned(w) >> 16); }

// frame's record: word 0 kind (0-7), conf index (8-15), change index
// (16-23), depth in its tree (24-31); word 1 atom range begin (0-7), end of
// the subtree's atoms (8-15), end (16-23), parent (24-31, 255: none)
__host__ __device__ inline int make_frame0(int kind, int conf, int change, int depth)
{
	return kind | (conf << 8) | (change << 16) | (depth << 24);
}
__host__ __device__ inline int make_frame1(int begin, int send, int end, int parent)
{
	return int(unsigned(begin) | (unsigned(send) << 8) | (unsigned(end) << 16) | (unsigned(parent) << 24));
}
__host__ __device__ inline int frame_kind(int w) { return w & 255; }
__host__ __device__ inline int frame_conf(int w) { return (w >> 8) & 255; }
__host__ __device__ inline int frame_change(int w) { return (w >> 16) & 255; }
__host__ __device__ inline int frame_depth(int w) { return int(unsigned(w) >> 24); }
__host__ __device__ inline int frame_begin(int w) { return w & 255; }
__host__ __device__ inline int frame_send(int w) { return (w >> 8) & 255; }
__host__ __device__ inline int frame_end(int w) { return (w >> 16) & 255; }
__host__ __device__ inline int frame_parent(int w) { return int(unsigned(w) >> 24); }
// a frame's children: first entry of the children list and their number
__host__ __device__ inline int make_child(int start, int count) { return start | (count << 8); }
__host__ __device__ inline int child_start(int w) { return w & 255; }
__host__ __device__ inline int child_count(int w) { return w >> 8; }

// per tree: root frame, conf and change index of the root, ligand flag,
// torsions, atom range, ligand-internal pair range
enum TreeField
{
	TR_ROOT = 0,
	TR_CONF,
	TR_CHANGE,
	TR_LIG,
	TR_NTORS,
	TR_AB,
	TR_AE,
	TR_PB,
	TR_PE,
	TR_FIELDS
};

// conf / change map entry: the element's kind, and the other space's index
// (orientation: its first)
__host__ __device__ inline int make_map(int kind, int index) { return kind | (index << 8); }
__host__ __device__ inline int map_kind(int w) { return w & 255; }
__host__ __device__ inline int map_index(int w) { return w >> 8; }

struct ModelHdr
{
	int natoms, ninflex, nframes, ntrees, nligands, npairs, nother;
	int conf_size, change_size, heavy, nlevels, num_tors; // (heavy: heavy_atoms, ALL_LANES)
	int path_ok; // every root-to-frame path has at most MAX_PATH frames
	int ncodes;
	int one_ligand; // one ligand whose pairs are all those after the other pairs
	int iblob_off, iblob_len; // in the batch int blob
	int tblob_off, tblob_len; // in the batch real blob
	// offsets inside the int blob (the movable atoms' records at 0)
	int o_type, o_code, o_prec, o_fm, o_fpath, o_child, o_clist, o_heavy, o_tree, o_cmap, o_gmap;
	// offsets inside the real blob
	int o_xyz0, o_local, o_forig, o_faxis, o_charge;
};

// ModelHdr::heavy: the movable heavy atoms, and whether every atom takes a lane
// of the evaluation whatever their number (a pair holds a hydrogen, or there
// is no heavy atom).  One value for both: the search kernels have no scalar
// register to spare, and a second one cost a single chain up to 6%.
constexpr int ALL_LANES = 1 << 16;
__host__ __device__ inline int heavy_atoms(const ModelHdr& h) { return h.heavy & (ALL_LANES - 1); }

template<typename T>
struct BatchPtrs
{
	const ModelHdr* hdr;
	const int* iblob;
	const T* tblob;
};

// scoring tables on the device: smooth as (e, dor) pairs per point; fast
// values kept in FP64 for the grid build and the final rescoring.  With
// charge-dependent terms (ncomp 4) smooth and fast hold the first (type
// only) component and qsmooth / qfast the other three (|q_a|, |q_b| and
// q_a q_b dependent) of the pair (min type, max type).
template<typename T>
struct TablePtrs
{
	const T* smooth; // [378][n][2]
	const double* fast; // [378][n]
	int ncomp;           // 1 or 4
	const T* qsmooth;    // [378][n][3][2] (ncomp 4)
	const double* qfast; // [378][n][3] (ncomp 4)
	int n;
	T factor_t;          // points per A^2 and the squared cutoff in the evaluation's precision
	T cutoff_t;
	// precalculate_splines (kind 1; FP64 direct evaluation only)
	int kind;            // 0: linear tables, 1: splines
	const double* spl;   // [378][nseg][5]: x, a, b, c, d
	const double* spl_cut; // [378]: 0 for a zero spline
	double fraction;     // segment length
	int nseg;
};

// one receptor map set (cache back end)
template<typename T>
struct GridPtrs
{
	const T* cells;      // [type slot][cells][8]
	const T* qcells;     // charge maps, same slots (ncomp 4), else null
	const int* slot_of;  // [27] -> map slot or -1
	int dim[3];          // points per axis
	int ncells;          // (dim0-1)(dim1-1)(dim2-1)
	T init[3];
	T factor[3];
	T factor_inv[3];
	T dim_fl_minus_1[3];
	T slope;
};

// one entry of a cell's list of receptor atoms, in one 16-byte (FP32) or
// 32-byte (FP64) record: position, type (5 bits) and receptor index (the
// rest), so that a lane reads an atom with one aligned load and the entries
// of a list follow each other
template<typename T> struct RecMeta;
template<> struct RecMeta<float> { using type = unsigned; };
template<> struct RecMeta<double> { using type = unsigned long long; };
template<typename T>
struct alignas(4 * sizeof(T)) RecAtom
{
	T x, y, z;
	typename RecMeta<T>::type meta;
};
template<typename T>
__host__ __device__ inline RecAtom<T> make_rec_atom(T x, T y, T z, int type, int index)
{
	return {x, y, z, typename RecMeta<T>::type(unsigned(type) | (unsigned(index) << 5))};
}
template<typename T>
__host__ __device__ inline int rec_type(const RecAtom<T>& a) { return int(unsigned(a.meta) & 31u); }
template<typename T>
__host__ __device__ inline int rec_index(const RecAtom<T>& a) { return int(unsigned(a.meta) >> 5); }

// receptor for the direct (non_cache) back end: atoms and 3 A cells over
// the box holding, in receptor order, the atoms within the cutoff of the
// cell's brick
template<typename T>
struct ReceptorPtrs
{
	const T* xyz;        // [natoms*3] all atoms (H included)
	const int* type;
	const T* charge;     // [natoms] partial charges
	int natoms;
	const int* cell_start; // [ncells+1]
	const RecAtom<T>* cell_recs;
	int cell_off[3];
	int cell_dim[3];
	double begin[3];
	double end[3];
	int enabled[3];
};

} // namespace sgpu

#endif
