// Null-space local-solve kernels for stencils of up to 42 nodes with 10 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS_UPTO(42, 10)
