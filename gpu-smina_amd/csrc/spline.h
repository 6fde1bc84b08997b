/*
 * Spline::eval_deriv (src/lib/splines.h:103-121) over the spline tables of
 * precalculate_splines (src/lib/precalculate.h:313-455): per type pair, nseg
 * cubic segments of `fraction` A, coefficients (x, a, b, c, d) in FP64.  A
 * pair whose terms vanish has cutoff 0 and evaluates to zero.
 */
#ifndef SGPU_SPLINE_H
#define SGPU_SPLINE_H

#include "pmath.h"

namespace sgpu
{

// a pair's coefficients at the distance r, read before they are used
// (in: r is inside the pair's cutoff; else any row, and the value is 0)
struct SplineRow
{
	double s[5];
	double r;
	bool in;
};
SGPU_HD SplineRow spline_row(const double* spl, const double* cut, double fraction, int nseg, int tri, double r)
{
	SplineRow w;
	w.r = r;
	w.in = r < cut[tri];
	unsigned index = w.in ? unsigned(r / fraction) : 0u;
	index = index < unsigned(nseg) ? index : unsigned(nseg - 1);
	const double* s = spl + (size_t(tri) * nseg + index) * 5;
	for (int k = 0; k < 5; k++)
		w.s[k] = s[k];
	return w;
}
SGPU_HD void spline_value(const SplineRow& w, double& val, double& der)
{
	const double* s = w.s;
	const double lx = w.r - s[0];
	val = w.in ? ((s[1] * lx + s[2]) * lx + s[3]) * lx + s[4] : 0;
	der = w.in ? (3 * s[1] * lx + 2 * s[2]) * lx + s[3] : 0;
}

SGPU_HD void spline_eval(const double* spl, const double* cut, double fraction, int nseg, int tri, double r,
		double& val, double& der)
{
	spline_value(spline_row(spl, cut, fraction, nseg, tri, r), val, der);
}

} // namespace sgpu

#endif
