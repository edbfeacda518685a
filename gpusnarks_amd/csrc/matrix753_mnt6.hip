// Matrix passes of the 753-bit field MNT6-753 Fr.
#include "matrix753_kernels.h"

namespace gsn {

GSN_MAT753_LAUNCHES(FMnt6)

}  // namespace gsn
