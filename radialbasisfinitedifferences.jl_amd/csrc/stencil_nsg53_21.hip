// Null-space local-solve kernels for stencils of up to 53 nodes with 21 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS_UPTO(53, 21)
