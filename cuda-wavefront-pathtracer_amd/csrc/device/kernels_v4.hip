// device/kernels_v4.hip - the kernels of the BVH4 layout for the triangle test CWP_TRI (instantiated here
// only; compiled once per test).
#include "device/kernels.h"

namespace cwp {
namespace dev {
template void pickTri<4, CWP_TRI>(int, int, Kernels&);
}  // namespace dev
}  // namespace cwp
