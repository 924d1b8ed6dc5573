// fast_r5.hip -- the register-FFT passes of the transform lengths with a
// factor 5 (mixed-radix in-register FFTs, reg_fft.hpp): the y and z
// passes for the lengths of at most 28 registers per component, the strided 3-D
// y passes for the longer ones.
#include "fast_launch.hpp"

namespace mmx {

MMX_R5_SHORT(MMX_INST_Z)
MMX_R5_SHORT(MMX_INST_FILM)
MMX_R5_SHORT(MMX_INST_Y)
MMX_R5_LONG(MMX_INST_Y)

} // namespace mmx
