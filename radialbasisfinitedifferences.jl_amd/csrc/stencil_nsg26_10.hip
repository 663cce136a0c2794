// Null-space local-solve kernels for stencils of up to 26 nodes with 10 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS_UPTO(26, 10)
