// Null-space local-solve kernels for stencils of 43 nodes with 21 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS(43, 21)
