// FD coefficient tables by stencil radius RO = order / 2, for the kernels that are instantiated for several orders.
//
// Coefficients (_FD_COEF_LEAST_SQUARE, FP32 as the reference spells them):
//   order 16: first staggered c1..c8 kernels/fd_coef.h:479-486, central second e0..e8 :535-543
//   order 12: first staggered c1..c6 of stg_d1<12> (kernels/fd_coefficients.h:16-60); no central set (density
//             gradient only)
//   order 8 : as common.h
#pragma once

#include "common.h"

namespace tti {

template <int RO>
struct FD;
template <>
struct FD<4>
{
    static constexpr float c[5] = { 0.0f, C1, C2, C3, C4 };
    static constexpr float e[5] = { E0, E1, E2, E3, E4 };
};
template <>
struct FD<6>
{
    static constexpr float c[7] = { 0.0f, 1.2403120e+0f, -1.1141390e-1f, 2.5759060e-2f, -6.4207590e-3f,
                                    1.3095870e-3f, -1.5512770e-4f };
    static constexpr float e[7] = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
};
template <>
struct FD<8>
{
    static constexpr float c[9] = { 0.0f, 1.254298E+00f, -1.234902E-01f, 3.470321E-02f, -1.201822E-02f,
                                    4.188332E-03f, -1.310232E-03f, 3.233353E-04f, -4.675068E-05f };
    static constexpr float e[9] = { -0.3162230E+1f, 0.1875943E+1f, -0.3859840E+0f, 0.1228261E+0f, -0.4233006E-1f,
                                    0.1379639E-1f, -0.3846673E-2f, 0.8026637E-3f, -0.9257725E-4f };
};

} // namespace tti
