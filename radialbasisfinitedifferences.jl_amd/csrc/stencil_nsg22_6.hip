// Null-space local-solve kernels for stencils of up to 22 nodes with 6 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS_UPTO(22, 6)
