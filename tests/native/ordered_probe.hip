/*
 * A probe of the ordered FP64 sums (search.h): row_ordered_add with an
 * accumulator of its own and with the elements themselves as the accumulator,
 * and ordered_add over the first cnt lanes.  One wave.
 */
#include "../../gpu-smina_amd/csrc/search.h"

namespace
{

__global__ __launch_bounds__(64) void rows(const double* acc, const double* v, double* own, double* same)
{
	const int lane = sgpu::lane_id();
	const double x = v[lane];
	own[lane] = sgpu::row_ordered_add(acc[lane], x);
	same[lane] = sgpu::row_ordered_add(x, x);
}

__global__ __launch_bounds__(64) void sums(const double* acc, const double* v, int cnt, double* out, float* outf)
{
	const int lane = sgpu::lane_id();
	const double x = lane < cnt ? v[lane] : 0.0;
	const double e = sgpu::ordered_add(acc[0], x, cnt);
	const float ef = sgpu::ordered_add(float(acc[0]), float(x), cnt);
	if (lane == 0)
	{
		out[0] = e;
		outf[0] = ef;
	}
}

} // namespace

// acc[64], v[64]; own[64], same[64]; out[64] and outf[64]: the sums over the
// first 1..64 lanes.  Host arrays.  Returns the first HIP error.
extern "C" int ordered_probe(const double* acc, const double* v, double* own, double* same, double* out, float* outf)
{
	double* d = nullptr;
	hipError_t e = hipMalloc(reinterpret_cast<void**>(&d), 6 * 64 * sizeof(double));
	if (e != hipSuccess)
		return int(e);
	float* df = reinterpret_cast<float*>(d + 5 * 64);
	e = hipMemcpy(d, acc, 64 * sizeof(double), hipMemcpyHostToDevice);
	if (e == hipSuccess)
		e = hipMemcpy(d + 64, v, 64 * sizeof(double), hipMemcpyHostToDevice);
	if (e == hipSuccess)
	{
		hipLaunchKernelGGL(rows, dim3(1), dim3(64), 0, nullptr, d, d + 64, d + 128, d + 192);
		for (int cnt = 1; cnt <= 64; cnt++)
			hipLaunchKernelGGL(sums, dim3(1), dim3(64), 0, nullptr, d, d + 64, cnt, d + 256 + cnt - 1, df + cnt - 1);
		e = hipGetLastError();
	}
	if (e == hipSuccess)
		e = hipMemcpy(own, d + 128, 64 * sizeof(double), hipMemcpyDeviceToHost);
	if (e == hipSuccess)
		e = hipMemcpy(same, d + 192, 64 * sizeof(double), hipMemcpyDeviceToHost);
	if (e == hipSuccess)
		e = hipMemcpy(out, d + 256, 64 * sizeof(double), hipMemcpyDeviceToHost);
	if (e == hipSuccess)
		e = hipMemcpy(outf, df, 64 * sizeof(float), hipMemcpyDeviceToHost);
	const hipError_t f = hipFree(d);
	return int(e != hipSuccess ? e : f);
}
