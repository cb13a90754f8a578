// The sizes shared by the renderer and the service's reservations, for tests.
#include "../../drawlab_amd/csrc/render_sizes.h"

extern "C" {
uint32_t guide_train_blocks(uint32_t rows) { return dl_sizes::guide_train_blocks(rows); }
}
