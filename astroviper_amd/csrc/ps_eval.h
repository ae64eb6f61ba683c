// ps_eval.h -- the prolate-spheroidal function on the device.
#pragma once

#include "avgrid_internal.h"

namespace av {

// Schwab's rational approximation (M=6, alpha=1) as in
// core/imaging/imaging_utils/gcf_prolate_spheroidal.py:102-158: the two
// coefficient tables are the published ones and must be identical.
static __constant__ double c_ps_p[2][5] = {
    {8.203343e-2, -3.644705e-1, 6.278660e-1, -5.335581e-1, 2.312756e-1},
    {4.028559e-3, -3.697768e-2, 1.021332e-1, -1.201436e-1, 6.412774e-2}};
static __constant__ double c_ps_q[2][3] = {{1.0000000e0, 8.212018e-1, 2.078043e-1},
                                    {1.0000000e0, 9.599102e-1, 2.918724e-1}};

__device__ inline void ps_eval(double uin, double &grdsf, double &kern) {
  double u = fabs(uin);
  int part = 0;
  double uend = 0.0;  // |u| > 1 (or NaN) keeps the zero defaults
  if (u >= 0.0 && u < 0.75) {
    part = 0;
    uend = 0.75;
  }
  if (u >= 0.75 && u <= 1.0) {
    part = 1;
    uend = 1.0;
  }
  double d = u * u - uend * uend;
  double d2 = d * d, d3 = d2 * d, d4 = d2 * d2;
  double top = c_ps_p[part][0];
  top += c_ps_p[part][1] * d;
  top += c_ps_p[part][2] * d2;
  top += c_ps_p[part][3] * d3;
  top += c_ps_p[part][4] * d4;
  double bot = c_ps_q[part][0];
  bot += c_ps_q[part][1] * d;
  bot += c_ps_q[part][2] * d2;
  double g = 0.0;
  if (bot > 0.0) g = top / bot;
  if (u > 1.0) g = 0.0;
  grdsf = g;
  kern = (1.0 - u * u) * g;
}

}  // namespace av
