// Checks of the planner (petar_amd/csrc/pth_plan.h) that its C entry point
// does not reach; no GPU.  Usage: plan_check <check>; prints what is wrong,
// exit code 1 if anything is.
//   reuse  one Plan object taken through host-made, device-made and plain
//          plans: the host holds items exactly where it made them
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/petar_hip.h"
#include "../../petar_amd/csrc/pth_plan.h"

using namespace pth;

static int bad = 0;
#define CHECK(cond, ...)                 \
    do {                                 \
        if (!(cond)) {                   \
            std::printf(__VA_ARGS__);    \
            std::printf(" (%s)\n", #cond); \
            bad = 1;                     \
        }                                \
    } while (0)

static void reuse()
{
    struct Step {
        int mode, max_ipl, chunk_j;
        bool on_device;
        int n_walk;
    };
    const Step steps[] = {{PTH_EXEC_FUSED, 4, 0, true, 200}, {PTH_EXEC_FUSED, 2, 0, true, 200},
                          {PTH_EXEC_FUSED, 3, 128, true, 200}, {PTH_EXEC_PLAIN, 2, 0, true, 200},
                          {PTH_EXEC_FUSED, 2, 0, false, 50}, {PTH_EXEC_FUSED, 1, 512, true, 200},
                          {PTH_EXEC_FUSED, 4, 512, false, 0}, {PTH_EXEC_FUSED, 2, 0, true, 0}};
    Plan P;
    for (const Step &s : steps) {
        const std::vector<int> ni(s.n_walk, 300), ne(s.n_walk, 5000), ns(s.n_walk, 900);
        const bool ok = make_plan(s.n_walk, ni.data(), ne.data(), ns.data(), s.mode, s.chunk_j, s.max_ipl, P, 1,
                                  false, 0, s.on_device);
        const bool fused = s.mode == PTH_EXEC_FUSED, dev = fused && s.on_device && s.max_ipl <= 2;
        CHECK(ok, "mode %d max_ipl %d", s.mode, s.max_ipl);
        CHECK(P.on_device == dev, "mode %d max_ipl %d: on_device %d", s.mode, s.max_ipl, P.on_device);
        CHECK((P.n_slots > 0) == (fused && s.n_walk > 0), "mode %d max_ipl %d: n_slots %d", s.mode, s.max_ipl, P.n_slots);
        CHECK(P.items.size() == (size_t)(dev ? 0 : P.n_slots), "mode %d max_ipl %d: %zu items on the host, %d slots",
              s.mode, s.max_ipl, P.items.size(), P.n_slots);
        CHECK(P.ritems.size() == (size_t)(dev ? 0 : P.n_ritems), "mode %d max_ipl %d: %zu reduction items, %d",
              s.mode, s.max_ipl, P.ritems.size(), P.n_ritems);
    }
}

int main(int argc, char **argv)
{
    if (argc == 2 && !std::strcmp(argv[1], "reuse")) reuse();
    else {
        std::printf("usage: plan_check reuse\n");
        return 2;
    }
    if (!bad) std::printf("ok\n");
    return bad;
}
