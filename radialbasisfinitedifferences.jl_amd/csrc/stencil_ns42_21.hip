// Null-space local-solve kernels for stencils of 42 nodes with 21 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS(42, 21)
