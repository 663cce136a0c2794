// Null-space local-solve kernels for stencils of up to 31 nodes with 15 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS_UPTO(31, 15)
