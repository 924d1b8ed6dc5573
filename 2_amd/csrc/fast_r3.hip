// fast_r3.hip -- the register-FFT passes of the transform lengths with a
// factor 3 (mixed-radix in-register FFTs, reg_fft.hpp): the y and z
// passes for the lengths of at most 28 registers per component, the strided 3-D
// y passes for the longer ones.
#include "fast_launch.hpp"

namespace mmx {

MMX_R3_SHORT(MMX_INST_Z)
MMX_R3_SHORT(MMX_INST_FILM)
MMX_R3_SHORT(MMX_INST_Y)
MMX_R3_LONG(MMX_INST_Y)

} // namespace mmx
