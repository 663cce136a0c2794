// Null-space local-solve kernels for stencils of 21 nodes with 10 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS(21, 10)
