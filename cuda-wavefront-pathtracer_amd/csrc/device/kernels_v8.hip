// device/kernels_v8.hip - the kernels of the compressed BVH8 layout for the triangle test CWP_TRI (instantiated here
// only; compiled once per test).
#include "device/kernels.h"

namespace cwp {
namespace dev {
template void pickTri<8, CWP_TRI>(int, int, Kernels&);
}  // namespace dev
}  // namespace cwp
