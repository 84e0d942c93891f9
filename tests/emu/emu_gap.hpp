// A poisoned gap between members of a structure (test infrastructure).
#pragma once

#include <sanitizer/asan_interface.h>

namespace emu {
struct Gap {
    alignas(8) char room[4096];
    Gap() { __asan_poison_memory_region(room, sizeof room); }
};
}  // namespace emu

#define EMU_CAT2(a, b) a##b
#define EMU_CAT(a, b) EMU_CAT2(a, b)
#define EMU_GAP EMU_CAT(gap_, __COUNTER__)
