// The rollback's host code, as libdflash_hip.so has it, on the CPU: its three launches are the functions below, which the dynamic
// linker finds before the library's own.  They print what they are asked for and refuse the one that the command line names.
//   rollback_check <launch to refuse, counted from 0, or -1> <rows of a window> <channels of a window, 0: no qkv> <Dk> [<Dk> ...]
// One tape cache per Dk; its window and state are 0x100000 and 0x300000 before the verify step, 0x500000 and 0x700000 after it, plus
// 0x1000000 per cache.  Prints a line per launch, the status, and "armed window state" of every cache.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../include/dflash_cache.h"

static int g_launch = 0, g_refuse = -1;
static int launch(const char* what, int n) {
    const bool refused = g_launch++ == g_refuse;
    std::printf("%s %d%s\n", what, n, refused ? " refused" : "");
    return refused ? DFLASH_UNSUPPORTED : DFLASH_OK;
}

namespace dflash {
struct ConvWindows;
__attribute__((visibility("default"))) int rebuild_conv_batched(void*, int n, const void* const*, const void* const*, void* const*, int, int,
                                                                int, int, int, int, const int32_t*) {
    return launch("windows", n);
}
__attribute__((visibility("default"))) int tape_replay_windows(void*, int n, const void* const*, int, const void* const*, const void* const*, int,
                                                               int, const void* const*, void* const*, int, int, int, int, int, int, int, int,
                                                               const ConvWindows&) {
    return launch("replay+windows", n);
}
}  // namespace dflash

extern "C" int dflash_tape_replay_batched(void*, int n, const void* const*, int, const void* const*, const void* const*, int, int, const void* const*,
                                          void* const*, int, int, const int32_t*, int, int, int, int, int, int, int) {
    return launch("replay", n);
}

int main(int argc, char** argv) {
    if (argc < 5) return 2;
    g_refuse = std::atoi(argv[1]);
    const int keep = std::atoi(argv[2]), C = std::atoi(argv[3]);
    std::vector<dflash_cache_t*> caches;
    for (int i = 4; i < argc; ++i) {
        const uintptr_t base = (uintptr_t)(i - 4) * 0x1000000;
        auto at = [&](uintptr_t x) { return reinterpret_cast<void*>(base + x); };
        dflash_cache_t* c = dflash_cache_create(DFLASH_CACHE_TAPE, keep + 1);
        dflash_cache_set_slot(c, 0, at(0x100000));
        dflash_cache_set_slot(c, 1, at(0x300000));
        dflash_cache_arm_rollback(c, 0);
        dflash_cache_set_slot(c, 0, at(0x500000));
        dflash_cache_set_slot(c, 1, at(0x700000));
        if (dflash_cache_record_tape(c, at(0x900000), DFLASH_F32, at(0xa00000), at(0xb00000), DFLASH_BF16, 3, C ? at(0xc00000) : nullptr, 2,
                                     DFLASH_F32, 1, 7, 1, 1, std::atoi(argv[i]), 1, C))
            return 3;
        caches.push_back(c);
    }
    const int rc = dflash_restore_target_cache_after_acceptance(caches.data(), (int)caches.size(), nullptr, 3, 2, 7, nullptr);
    std::printf("status %d\n", rc);
    for (size_t i = 0; i < caches.size(); ++i) {
        auto rel = [&](int slot) { return (unsigned long)((uintptr_t)dflash_cache_get_slot(caches[i], slot) - i * 0x1000000); };
        std::printf("%d %lx %lx\n", dflash_cache_is_armed(caches[i]), rel(0), rel(1));
        dflash_cache_destroy(caches[i]);
    }
    return 0;
}
