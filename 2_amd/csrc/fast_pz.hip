// fast_pz.hip -- the z-pass launchers, and those of a film's y, of the
// power-of-two lengths (fast_launch.hpp), in a file of its own so that it
// compiles in parallel with the other instantiations.
#include "fast_launch.hpp"

namespace mmx {

MMX_POW2_LENGTHS(MMX_INST_Z)
MMX_POW2_FILM(MMX_INST_FILM)

} // namespace mmx
