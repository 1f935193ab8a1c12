// Stencil planes of the 3D operators and the order of their terms.
#pragma once

namespace cdr {
namespace k3 {

// stencil planes, 1-based (src/3d/ftn/BMG_stencils_f90.h:46-48)
enum { kp = 1, kpw, kps, kb, kpsw, kpnw, kbw, kbnw, kbn, kbne, kbe, kbse, kbs, kbsw };

// The 26 neighbour terms of the 27-point operator in the reference's order
// (src/3d/ftn/BMG3_SymStd_residual.f90:71-97): X(si, sj, sk, plane, oi, oj, ok) = coefficient
// at (i,j,k) + s times q at (i,j,k) + o.  The 7-point operator is the sub-list below
// (src/3d/ftn/BMG3_SymStd_residual.f90:106-112).
#define NB27_LIST(X)                                                                              \
    X(0, 0, 0, kpw, -1, 0, 0) X(0, 1, 0, kpnw, -1, 1, 0) X(0, 1, 0, kps, 0, 1, 0)                 \
    X(1, 1, 0, kpsw, 1, 1, 0) X(1, 0, 0, kpw, 1, 0, 0) X(1, 0, 0, kpnw, 1, -1, 0)                 \
    X(0, 0, 0, kps, 0, -1, 0) X(0, 0, 0, kpsw, -1, -1, 0) X(0, 0, 0, kb, 0, 0, -1)                \
    X(0, 0, 0, kbw, -1, 0, -1) X(0, 1, 0, kbnw, -1, 1, -1) X(0, 1, 0, kbn, 0, 1, -1)              \
    X(1, 1, 0, kbne, 1, 1, -1) X(1, 0, 0, kbe, 1, 0, -1) X(1, 0, 0, kbse, 1, -1, -1)              \
    X(0, 0, 0, kbs, 0, -1, -1) X(0, 0, 0, kbsw, -1, -1, -1) X(0, 0, 1, kb, 0, 0, 1)               \
    X(0, 0, 1, kbe, -1, 0, 1) X(0, 1, 1, kbse, -1, 1, 1) X(0, 1, 1, kbs, 0, 1, 1)                 \
    X(1, 1, 1, kbsw, 1, 1, 1) X(1, 0, 1, kbw, 1, 0, 1) X(1, 0, 1, kbnw, 1, -1, 1)                 \
    X(0, 0, 1, kbn, 0, -1, 1) X(0, 0, 1, kbne, -1, -1, 1)
#define NB7_LIST(X)                                                                               \
    X(0, 0, 0, kpw, -1, 0, 0) X(0, 1, 0, kps, 0, 1, 0) X(1, 0, 0, kpw, 1, 0, 0)                   \
    X(0, 0, 0, kps, 0, -1, 0) X(0, 0, 0, kb, 0, 0, -1) X(0, 0, 1, kb, 0, 0, 1)

}  // namespace k3
}  // namespace cdr
