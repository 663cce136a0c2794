// Null-space local-solve kernels for stencils of 31 nodes with 15 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS(31, 15)
