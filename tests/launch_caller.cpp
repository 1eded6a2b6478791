// The GEMM launchers on operands that lack the form they read: each says so and launches nothing, so this
// program needs no GPU.  Prints one line per launcher and exits 0 where all of them refuse.
#include <cstdio>

#include "jxmoe_kernels.h"

namespace {
int bad = 0;
void expect_refused(const char* what, bool launched) {
    std::printf("%s: %s\n", what, launched ? "launched" : "refused");
    bad += launched;
}
}  // namespace

int main() {
    const int types[] = {jx::T_Q4_0, jx::T_Q8_0, jx::T_Q4_K, jx::T_Q5_K, jx::T_Q5_0, jx::T_Q6_K};
    uint8_t byte = 0;
    for (int type : types) {
        jx::QMat m;
        m.type = type;
        m.rows = m.cols = 256;
        m.nrt = 8;
        const jx::ActQ8 none;
        const jx::ActH no_forms;
        jx::Groups grp;
        char what[64];
        std::snprintf(what, sizeof what, "type %d gate/up", type);
        expect_refused(what, jx::launch_mfma_gateup(m, m, none, no_forms, grp, 1, none, no_forms, nullptr, nullptr));
        std::snprintf(what, sizeof what, "type %d down", type);
        expect_refused(what, jx::launch_mfma_down_block(m, none, no_forms, grp, 1, nullptr, nullptr));
        std::snprintf(what, sizeof what, "type %d fp16 down", type);
        expect_refused(what, jx::launch_mfma_down(m, no_forms, grp, 1, nullptr, nullptr));
        m.g6 = m.bt = &byte;  // codes and a table, but not the activations' forms
        std::snprintf(what, sizeof what, "type %d gate/up codes", type);
        expect_refused(what, jx::launch_mfma_gateup(m, m, none, no_forms, grp, 1, none, no_forms, nullptr, nullptr));
    }
    return bad ? 1 : 0;
}
