// The 16-wave scan kernels of float16 activations (scan16_kernel.hpp).
#include "scan16_kernel.hpp"

namespace m3 {

template int launch_scan16<_Float16>(const m3_scan_args&, const ScanGeom&, const float*, bool,
                                 hipStream_t);

}  // namespace m3
