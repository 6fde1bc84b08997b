/*
 * Receptor map build on the device (the reference's build_grids_kernel,
 * src/gpu/gpu_device.cu:133-186, restating cache::populate,
 * src/lib/cache.cpp:116-210).
 *
 * 1. cell lists: for each 3 A cell, in receptor order, the heavy receptor
 *    atoms within the cutoff of both the box and the cell's brick.  The
 *    brick of a cell is [floor, ceil] (x 3 A) of the first probe coordinate
 *    falling into it, per dimension: that is the brick smina's szv_grid_cache
 *    builds (src/lib/szv_grid.h:100-130), degenerate where a probe lies on a
 *    3 A boundary.  Count pass, scan, ordered fill (one workgroup per cell,
 *    prefix sums keep receptor order).
 * 2. points: the workgroups of a cell stage its list in LDS as records;
 *    each wave sums tiles of 4 x 4 x 4 of the cell's points over the list
 *    (FP64, in list order) for every needed ligand type.  The linear tables
 *    are first repacked to one row per receptor type and knot holding all
 *    the ligand types' values, so that an atom in range costs one contiguous
 *    read.
 *    With a user grid (--user_grid), each point adds its value as
 *    cache::populate does (src/lib/cache.cpp:204-205).  With
 *    charge-dependent terms the point also sums the charge map
 *    (src/lib/cache.cpp:172-187): the map gets type-only plus |q_rec|
 *    components, the charge map the |q_lig| plus q_rec q_lig components
 *    that the evaluation scales by the ligand atom's charge.
 * 3. pack: point maps -> corner-packed cells (8 corner values per cell).
 */
#include <hip/hip_runtime.h>
#include "launch.h"
#include "atom_types.h"
#include "spline.h"
#include "gridterm.h"

namespace sgpu
{

constexpr int CELL_THREADS = 256;
constexpr int MAX_GRID_TYPES = 16;

__device__ inline double clamp_to(double lo, double hi, double x)
{
	if (x <= lo)
		return lo;
	else if (x >= hi)
		return hi;
	return x;
}
// brick_distance_sqr (src/lib/brick.h:26-40)
__device__ inline double brick_dist2(const double* lo, const double* hi, const double* v)
{
	const double c0 = clamp_to(lo[0], hi[0], v[0]);
	const double c1 = clamp_to(lo[1], hi[1], v[1]);
	const double c2 = clamp_to(lo[2], hi[2], v[2]);
	return (c0 - v[0]) * (c0 - v[0]) + (c1 - v[1]) * (c1 - v[1]) + (c2 - v[2]) * (c2 - v[2]);
}

__device__ inline bool cell_has(const GridBuildArgs& a, int cell, int atom)
{
	const int t = a.rec_type[atom];
	if (t >= NUM_ATOM_TYPES || is_hydrogen_type(t))
		return false;
	const double* v = a.rec_xyz + 3 * atom;
	if (!(brick_dist2(a.box_lo, a.box_hi, v) < a.cutoff_sqr))
		return false;
	const int cx = cell % a.cell_dim[0];
	const int cy = (cell / a.cell_dim[0]) % a.cell_dim[1];
	const int cz = cell / (a.cell_dim[0] * a.cell_dim[1]);
	const double lo[3] = {a.cell_lo[cx], a.cell_lo[a.cell_dim[0] + cy], a.cell_lo[a.cell_dim[0] + a.cell_dim[1] + cz]};
	const double hi[3] = {a.cell_hi[cx], a.cell_hi[a.cell_dim[0] + cy], a.cell_hi[a.cell_dim[0] + a.cell_dim[1] + cz]};
	return brick_dist2(lo, hi, v) < a.cutoff_sqr;
}

// block-wide exclusive prefix sum of one flag per thread
__device__ inline int block_scan(int flag, int& total)
{
	__shared__ int warp_sums[CELL_THREADS / 64];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	const unsigned long long mask = __ballot(flag);
	const int before = __popcll(mask & ((1ull << lane) - 1ull));
	if (lane == 0)
		warp_sums[w] = __popcll(mask);
	__syncthreads();
	int off = 0;
	total = 0;
	for (int k = 0; k < CELL_THREADS / 64; k++)
	{
		if (k < w)
			off += warp_sums[k];
		total += warp_sums[k];
	}
	__syncthreads();
	return off + before;
}

__global__ __launch_bounds__(CELL_THREADS) void cell_count_kernel(GridBuildArgs a)
{
	const int cell = blockIdx.x;
	int count = 0;
	for (int base = 0; base < a.rec_n; base += CELL_THREADS)
	{
		const int i = base + int(threadIdx.x);
		const int f = (i < a.rec_n && cell_has(a, cell, i)) ? 1 : 0;
		int total;
		block_scan(f, total);
		count += total;
	}
	if (threadIdx.x == 0)
		a.cell_start[cell + 1] = count;
}

// prefix sums of the counts in place (start[0] = 0), one workgroup: a run of
// cells per thread, then the runs' sums across the workgroup (1,728 cells: 6 us
// against 156 us by one thread)
__global__ __launch_bounds__(CELL_THREADS) void cell_scan_kernel(int* start, int ncells)
{
	__shared__ int run_sum[CELL_THREADS];
	const int t = int(threadIdx.x);
	const int run = (ncells + CELL_THREADS - 1) / CELL_THREADS;
	const int lo = t * run, hi = lo + run < ncells ? lo + run : ncells;
	int sum = 0;
	for (int c = lo; c < hi; c++)
		sum += start[c + 1];
	run_sum[t] = sum;
	__syncthreads();
	for (int off = 1; off < CELL_THREADS; off *= 2)
	{
		const int v = t >= off ? run_sum[t - off] : 0;
		__syncthreads();
		run_sum[t] += v;
		__syncthreads();
	}
	int acc = run_sum[t] - sum;
	for (int c = lo; c < hi; c++)
	{
		acc += start[c + 1];
		start[c + 1] = acc;
	}
	if (t == 0)
		start[0] = 0;
}

__global__ __launch_bounds__(CELL_THREADS) void cell_fill_kernel(GridBuildArgs a)
{
	const int cell = blockIdx.x;
	int out = a.cell_start[cell];
	for (int base = 0; base < a.rec_n; base += CELL_THREADS)
	{
		const int i = base + int(threadIdx.x);
		const int f = (i < a.rec_n && cell_has(a, cell, i)) ? 1 : 0;
		int total;
		const int pos = block_scan(f, total);
		if (f)
			a.cell_atoms[out + pos] = i;
		out += total;
	}
}

__global__ __launch_bounds__(256) void cell_records_kernel(const double* xyz, const int* type, const int* cell_atoms,
		int total, RecAtom<float>* rec32, RecAtom<double>* rec64)
{
	const int k = int(blockIdx.x * blockDim.x + threadIdx.x);
	if (k >= total)
		return;
	const int i = cell_atoms[k];
	const double x = xyz[3 * size_t(i)], y = xyz[3 * size_t(i) + 1], z = xyz[3 * size_t(i) + 2];
	rec64[k] = make_rec_atom<double>(x, y, z, type[i], i);
	rec32[k] = make_rec_atom<float>(float(x), float(y), float(z), type[i], i);
}

// the linear tables by receptor type and knot: rows[t1][knot][nt], the
// needed ligand types' values next to each other (nt a multiple of 2: 16-byte
// reads), zeros past them
__global__ __launch_bounds__(256) void type_rows_kernel(const double* fast, int table_n, const int* types, int ntypes,
		int nt, double* rows)
{
	const size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (k >= size_t(NUM_ATOM_TYPES) * table_n * nt)
		return;
	const int j = int(k % nt);
	const size_t r = k / nt;
	const int knot = int(r % table_n), t1 = int(r / table_n);
	rows[k] = j < ntypes ? fast[size_t(tri_index_permissive(t1, types[j])) * table_n + knot] : 0.0;
}

constexpr int POINT_WAVES = 4;
constexpr int POINT_LIST = 512; // records in LDS at once
constexpr int MAX_SPLIT = 256;  // workgroups of a cell
enum PointTables
{
	POINTS_LINEAR = 0,
	POINTS_CHARGED = 1,
	POINTS_SPLINE = 2
};

// One cell's points, its tiles split over gridDim.y workgroups.  Bound by the
// table rows' gathers: a tile's 64 points walk the same list (broadcast reads
// from LDS) and skip an atom none of them reaches.  A thread per x-fastest
// point (nine lists a wave, an index, a position and a type load per entry, a
// gather per ligand type) took 1,676 us for the 531,441 points and 8 types of
// a 30 A box, this 307 us (345 with all of a cell's tiles in one workgroup;
// four entries' rows in flight at once: no faster).  With one workgroup a cell, a
// box of few cells or of many points a cell left most of the device idle: a
// whole build of a 12 A box at 0.1 A took 4.7 ms (linear) and 40 ms (spline),
// of a 22.5 A box at 0.375 A with splines 1.77 ms; split, 1.1, 2.6 and 1.27 ms.
template<int NT, int KIND>
__global__ __launch_bounds__(64 * POINT_WAVES) void grid_points_kernel(GridBuildArgs a, const double* rows,
		double* points, double* qpoints)
{
	__shared__ double lx[POINT_LIST], ly[POINT_LIST], lz[POINT_LIST];
	__shared__ int lt[POINT_LIST];
	__shared__ double lq[KIND == POINTS_CHARGED ? POINT_LIST : 1];
	const int cell = int(blockIdx.x);
	const int c[3] = {cell % a.cell_dim[0], (cell / a.cell_dim[0]) % a.cell_dim[1],
			cell / (a.cell_dim[0] * a.cell_dim[1])};
	// the cell's points along each axis
	int first[3], count[3], tiles[3];
	const int* pf = a.cell_point;
	for (int d = 0; d < 3; d++)
	{
		first[d] = pf[c[d]];
		count[d] = pf[c[d] + 1] - first[d];
		tiles[d] = (count[d] + 3) / 4;
		pf += a.cell_dim[d] + 1;
	}
	const int ntiles = tiles[0] * tiles[1] * tiles[2];
	const int k0 = a.cell_start[cell], k1 = a.cell_start[cell + 1];
	const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
	const size_t npts = size_t(a.dim[0]) * a.dim[1] * a.dim[2];
	int staged = -1; // the list's part in LDS
	for (int t0 = int(blockIdx.y) * POINT_WAVES; t0 < ntiles; t0 += int(gridDim.y) * POINT_WAVES)
	{
		const int tile = t0 + wave;
		const int px = 4 * (tile % tiles[0]) + (lane & 3);
		const int py = 4 * ((tile / tiles[0]) % tiles[1]) + ((lane >> 2) & 3);
		const int pz = 4 * (tile / (tiles[0] * tiles[1])) + (lane >> 4);
		const bool mine = tile < ntiles && px < count[0] && py < count[1] && pz < count[2];
		const int x = first[0] + px, y = first[1] + py, z = first[2] + pz;
		// grid::index_to_argument
		const double probe[3] = {a.init[0] + a.factor_inv[0] * x, a.init[1] + a.factor_inv[1] * y,
				a.init[2] + a.factor_inv[2] * z};
		double aff[NT], caff[KIND == POINTS_CHARGED ? NT : 1];
		for (int j = 0; j < NT; j++)
			aff[j] = 0;
		for (double& q : caff)
			q = 0;
		for (int part = 0; k0 + part * POINT_LIST < k1; part++)
		{
			const int base = k0 + part * POINT_LIST;
			const int len = k1 - base < POINT_LIST ? k1 - base : POINT_LIST;
			if (staged != part)
			{
				__syncthreads(); // the part before it is done with
				for (int k = int(threadIdx.x); k < len; k += 64 * POINT_WAVES)
				{
					const int i = a.cell_atoms[base + k];
					lx[k] = a.rec_xyz[3 * size_t(i)];
					ly[k] = a.rec_xyz[3 * size_t(i) + 1];
					lz[k] = a.rec_xyz[3 * size_t(i) + 2];
					lt[k] = a.rec_type[i];
					if constexpr (KIND == POINTS_CHARGED)
						lq[k] = a.rec_q[i];
				}
				__syncthreads();
				staged = part;
			}
			for (int k = 0; k < len; k++)
			{
				const double d0 = lx[k] - probe[0], d1 = ly[k] - probe[1], d2 = lz[k] - probe[2];
				const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
				if (!(mine && r2 <= a.cutoff_sqr))
					continue;
				const int t1 = lt[k];
				if constexpr (KIND == POINTS_SPLINE)
				{
					// precalculate_splines::eval_fast: the spline's value
					const double r = __builtin_sqrt(r2);
					for (int j = 0; j < NT; j++)
						if (j < a.ntypes)
						{
							double val, der;
							spline_eval(a.spl, a.spl_cut, a.fraction, a.nseg, tri_index_permissive(t1, a.types[j]), r,
									val, der);
							aff[j] += val;
						}
				}
				else if constexpr (KIND == POINTS_CHARGED)
				{
					// precalculate_linear::eval_fast_data of (receptor type,
					// ligand type): the components swapped when t1 > t2
					const size_t idx = size_t(a.factor * r2);
					const double q = lq[k];
					const double aq = q < 0 ? -q : q;
					for (int j = 0; j < NT; j++)
						if (j < a.ntypes)
						{
							const int tt = a.types[j];
							const size_t e = size_t(tri_index_permissive(t1, tt)) * a.table_n + idx;
							const double* qf = a.qfast + 3 * e;
							const bool in_order = t1 <= tt;
							const double c1 = in_order ? qf[0] : qf[1], c2 = in_order ? qf[1] : qf[0];
							aff[j] += a.fast[e] + c1 * aq;
							caff[j] += c2 + qf[2] * q;
						}
				}
				else
				{
					const double* row = rows + (size_t(t1) * a.table_n + size_t(a.factor * r2)) * NT;
					double v[NT];
					for (int j = 0; j < NT; j++)
						v[j] = row[j];
					for (int j = 0; j < NT; j++)
						aff[j] += v[j];
				}
			}
		}
		if (mine)
		{
			// the user grid at (x, y, z) as a location in A: the reference's own
			// expression, kept as it is
			const double uge =
					a.has_ug ? grid_value(a.ug, v3(double(x), double(y), double(z)), 1000.0, a.ug_slope) : 0.0;
			const size_t p = size_t(x) + size_t(a.dim[0]) * (size_t(y) + size_t(a.dim[1]) * z);
			for (int j = 0; j < NT; j++)
				if (j < a.ntypes)
				{
					points[size_t(j) * npts + p] = a.has_ug ? aff[j] + uge : aff[j];
					if constexpr (KIND == POINTS_CHARGED)
						qpoints[size_t(j) * npts + p] = caff[j];
				}
		}
	}
}

template<typename T>
__global__ __launch_bounds__(256) void grid_pack_kernel(const double* points, int ntypes, int d0, int d1, int d2, T* cells)
{
	const size_t nc = size_t(d0 - 1) * (d1 - 1) * (d2 - 1);
	const size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (k >= nc * ntypes)
		return;
	const int s = int(k / nc);
	const size_t c = k % nc;
	const int x = int(c % (d0 - 1));
	const int y = int((c / (d0 - 1)) % (d1 - 1));
	const int z = int(c / (size_t(d0 - 1) * (d1 - 1)));
	const double* m = points + size_t(s) * d0 * d1 * d2;
	auto at = [&](int i, int j, int l) { return m[size_t(i) + size_t(d0) * (size_t(j) + size_t(d1) * l)]; };
	T* out = cells + k * 8;
	out[0] = T(at(x, y, z));
	out[1] = T(at(x + 1, y, z));
	out[2] = T(at(x, y + 1, z));
	out[3] = T(at(x + 1, y + 1, z));
	out[4] = T(at(x, y, z + 1));
	out[5] = T(at(x + 1, y, z + 1));
	out[6] = T(at(x, y + 1, z + 1));
	out[7] = T(at(x + 1, y + 1, z + 1));
}

hipError_t launch_cell_count(const GridBuildArgs& a, hipStream_t st)
{
	const int ncells = a.cell_dim[0] * a.cell_dim[1] * a.cell_dim[2];
	hipLaunchKernelGGL(cell_count_kernel, dim3(ncells), dim3(CELL_THREADS), 0, st, a);
	hipError_t e = hipGetLastError();
	if (e != hipSuccess)
		return e;
	hipLaunchKernelGGL(cell_scan_kernel, dim3(1), dim3(CELL_THREADS), 0, st, a.cell_start, ncells);
	return hipGetLastError();
}

hipError_t launch_cell_fill(const GridBuildArgs& a, hipStream_t st)
{
	const int ncells = a.cell_dim[0] * a.cell_dim[1] * a.cell_dim[2];
	hipLaunchKernelGGL(cell_fill_kernel, dim3(ncells), dim3(CELL_THREADS), 0, st, a);
	return hipGetLastError();
}

hipError_t launch_cell_records(const double* xyz, const int* type, const int* cell_atoms, int total,
		RecAtom<float>* rec32, RecAtom<double>* rec64, hipStream_t st)
{
	if (total < 1)
		return hipSuccess;
	hipLaunchKernelGGL(cell_records_kernel, dim3(unsigned((total + 255) / 256)), dim3(256), 0, st, xyz, type,
			cell_atoms, total, rec32, rec64);
	return hipGetLastError();
}

// reals of a row of the repacked tables for ntypes types (0: not used)
static int row_reals(const GridBuildArgs& a)
{
	return a.kind != 0 || a.ncomp == 4 ? 0 : a.ntypes <= 4 ? 4 : a.ntypes <= 8 ? 8 : 16;
}
size_t grid_row_bytes(const GridBuildArgs& a)
{
	return size_t(NUM_ATOM_TYPES) * a.table_n * row_reals(a) * sizeof(double);
}

hipError_t launch_grid_points(const GridBuildArgs& a, double* rows, double* points, double* qpoints, hipStream_t st)
{
	if (a.ntypes > MAX_GRID_TYPES || (a.ncomp == 4 && (!qpoints || !a.qfast || !a.rec_q || a.kind != 0)))
		return hipErrorInvalidValue;
	const int nt = row_reals(a);
	if (nt > 0)
	{
		const size_t n = size_t(NUM_ATOM_TYPES) * a.table_n * nt;
		hipLaunchKernelGGL(type_rows_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, a.fast, a.table_n, a.types,
				a.ntypes, nt, rows);
		const hipError_t e = hipGetLastError();
		if (e != hipSuccess)
			return e;
	}
	auto fn = a.kind == 1    ? grid_points_kernel<MAX_GRID_TYPES, POINTS_SPLINE>
	          : a.ncomp == 4 ? grid_points_kernel<MAX_GRID_TYPES, POINTS_CHARGED>
	          : nt == 4      ? grid_points_kernel<4, POINTS_LINEAR>
	          : nt == 8      ? grid_points_kernel<8, POINTS_LINEAR>
	                         : grid_points_kernel<16, POINTS_LINEAR>;
	const int ncells = a.cell_dim[0] * a.cell_dim[1] * a.cell_dim[2];
	// a tile per wave, so that a few cells of many points fill the device, too
	const int split = (a.cell_tiles + POINT_WAVES - 1) / POINT_WAVES;
	hipLaunchKernelGGL(fn, dim3(unsigned(ncells), unsigned(split < MAX_SPLIT ? split : MAX_SPLIT)), dim3(64 * POINT_WAVES),
			0, st, a, rows, points, qpoints);
	return hipGetLastError();
}

template<typename T>
hipError_t launch_grid_pack(const double* points, int ntypes, const int* dim, T* cells, hipStream_t st)
{
	const size_t nc = size_t(dim[0] - 1) * (dim[1] - 1) * (dim[2] - 1) * ntypes;
	hipLaunchKernelGGL(grid_pack_kernel<T>, dim3(unsigned((nc + 255) / 256)), dim3(256), 0, st, points, ntypes, dim[0],
			dim[1], dim[2], cells);
	return hipGetLastError();
}
template hipError_t launch_grid_pack<float>(const double*, int, const int*, float*, hipStream_t);
template hipError_t launch_grid_pack<double>(const double*, int, const int*, double*, hipStream_t);

} // namespace sgpu
