// Null-space local-solve kernels for stencils of 20 nodes with 10 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS(20, 10)
