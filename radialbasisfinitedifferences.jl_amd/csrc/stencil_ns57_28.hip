// Null-space local-solve kernels for stencils of 57 nodes with 28 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS(57, 28)
