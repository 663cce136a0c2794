// Null-space local-solve kernels for stencils of up to 47 nodes with 15 monomials.
#include "stencil_ns.hpp"

RBFFD_DEFINE_NS_UPTO(47, 15)
