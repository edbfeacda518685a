// Matrix passes of the 753-bit field MNT4-753 Fr.
#include "matrix753_kernels.h"

namespace gsn {

GSN_MAT753_LAUNCHES(FMnt4)

}  // namespace gsn
