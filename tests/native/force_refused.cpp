// A count-mode force whose workspace the device refuses has not been made: the
// next one takes the number that it would have had, and so its result.  This
// program's own hipMalloc stands in front of the runtime's and refuses on demand.
#include "lgca.h"

#include <dlfcn.h>

#include <cstdio>
#include <vector>

static bool refuse = false;

extern "C" __attribute__((visibility("default"))) int hipMalloc(void** p, unsigned long n)
{
    static int (*real)(void**, unsigned long) = (int (*)(void**, unsigned long))dlsym(RTLD_NEXT, "hipMalloc");
    return refuse ? 2 /* hipErrorOutOfMemory */ : real(p, n);
}

static lgca_lattice* lattice()
{
    lgca_lattice* h = nullptr;
    if (lgca_create(&h, LGCA_FHP_II, 320, 200, 1, 0) != LGCA_OK || lgca_set_seed(h, 9) != LGCA_OK ||
        lgca_init_random(h, 0.3) != LGCA_OK || lgca_apply_body_force_count(h, LGCA_FORCE_X, 5, nullptr) != LGCA_OK) {
        std::printf("FAILED: no lattice\n");
        return nullptr;
    }
    return h;
}

int main()
{
    lgca_lattice *a = lattice(), *b = lattice();
    if (!a || !b) return 1;
    refuse = true;
    const lgca_status st = lgca_apply_body_force_count(a, LGCA_FORCE_X, 700, nullptr);
    refuse = false;
    if (st != LGCA_ERR_OUT_OF_MEMORY) {
        std::printf("FAILED: status %d where memory is refused\n", (int)st);
        return 1;
    }
    int64_t na = -1, nb = -2;
    if (lgca_apply_body_force_count(a, LGCA_FORCE_X, 700, &na) != LGCA_OK ||
        lgca_apply_body_force_count(b, LGCA_FORCE_X, 700, &nb) != LGCA_OK)
        return 1;
    std::vector<uint8_t> sa(320 * 200), sb(320 * 200);
    if (lgca_get_state_u8(a, sa.data()) != LGCA_OK || lgca_get_state_u8(b, sb.data()) != LGCA_OK) return 1;
    if (na != nb || sa != sb) {
        std::printf("FAILED: the refused call counted (%lld and %lld reverted)\n", (long long)na, (long long)nb);
        return 1;
    }
    lgca_destroy(a);
    lgca_destroy(b);
    std::printf("REFUSED CALL PASSED\n");
    return 0;
}
