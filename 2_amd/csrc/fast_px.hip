// fast_px.hip -- the x-pass launchers (xf, and xi with uniform parameters) of
// the lengths that have a register-FFT x pass (fast_launch.hpp), in a file of
// its own so that it compiles in parallel with the other instantiations.
#include "fast_launch.hpp"

namespace mmx {

MMX_XF_LENGTHS(MMX_INST_XF)
#define MMX_INST_XI_PLAIN(L) MMX_INST_XI(L, XI_UNIFORM)
MMX_X_LENGTHS(MMX_INST_XI_PLAIN)
#undef MMX_INST_XI_PLAIN

} // namespace mmx
