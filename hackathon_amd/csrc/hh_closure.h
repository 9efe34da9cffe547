// Dirichlet closure of the compact right-hand sides: the stencil weights times
// the known boundary values next to a point (2D_Program/main_functions/
// rhs.c:126-148, 3D_Program/main_functions/rhs.c:55-62,167-174).
#pragma once
#include "hh_common.h"

namespace hh {

// Point (i, j) of an Nx x Ny grid, cq = its row's weights (bm, am, b, a, bp,
// ap), u on the extended grid: the sum over its neighbours on the boundary,
// subtracted from v one by one in the reference's order.
HH_DEV double2 dirichlet2d(double2 v, int Nx, int Ny, int i, int j, const double2 *cq, const double2 *u) {
    const int X = Nx + 2;
    for (int dj = -1; dj <= 1; dj++)
        for (int di = -1; di <= 1; di++) {
            const int ii = i + di, jj = j + dj;
            if (ii >= 0 && ii < Nx && jj >= 0 && jj < Ny) continue;
            const double2 w = dj == 1 ? (di == 0 ? cq[5] : cq[4]) : dj == 0 ? (di == 0 ? cq[3] : cq[2]) : (di == 0 ? cq[1] : cq[0]);
            v = csub<double>(v, cmul<double>(w, u[(ii + 1) + (long)(jj + 1) * X]));
        }
    return v;
}

// Layer l of Nz layers, g = the point's position in an extended layer, X and
// XY = row and layer length of the extended grid, coef = the operator's table
// (a..d, ap..dp, am..dm per layer): fourth and sixth order, z faces.
HH_DEV double2 dirichlet3d(double2 v, long X, long XY, int Nz, int l, long g, const double2 *coef, const double2 *u) {
    for (int side = 0; side < 2; side++) {
        if (l != (side == 0 ? 0 : Nz - 1)) continue;
        const double2 *q = u + g + (side == 0 ? 0 : (Nz + 1) * XY);
        const double2 *cq = coef + 12L * l + (side == 0 ? 8 : 4);
        const double2 corner = cadd<double>(cadd<double>(cadd<double>(q[-1 - X], q[1 - X]), q[-1 + X]), q[1 + X]);
        const double2 xn = cadd<double>(q[-1], q[1]), yn = cadd<double>(q[-X], q[X]);
        double2 w = cadd<double>(cmul<double>(cq[0], corner), cmul<double>(cq[1], xn));
        w = cadd<double>(cadd<double>(w, cmul<double>(cq[2], yn)), cmul<double>(cq[3], q[0]));
        v = csub<double>(v, w);
    }
    return v;
}

}  // namespace hh
