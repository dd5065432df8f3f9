// Host check of mom5_amd/csrc/planes.h (tests/test_planes.py).
#include "planes.h"

static_assert(plane_at(0, 1 << 28) == 0, "the first plane");
static_assert(plane_at(15, 1 << 20) == 15u << 20, "inside 32 bits");
static_assert(plane_at(15, 1 << 28) == (size_t)15 << 28, "past 31 bits");
static_assert(plane_at(15, (1 << 29) - 1) == 15 * ((size_t)(1 << 29) - 1), "past 32 bits");

static_assert(level_fits(1), "the smallest");
static_assert(level_fits((1LL << 29) - 1), "the largest");
static_assert(!level_fits(1LL << 29), "one more");

int main() { return 0; }
