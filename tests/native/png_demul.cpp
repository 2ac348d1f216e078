// The demultiplied channels of PNG output (png_demul.h): the table's construction and the
// expression that the rows' kernel evaluates, for every alpha and channel value and for the
// factors that stand for a table row, under UndefinedBehaviorSanitizer with its check of
// conversions from floating point.
//
// Built and run by tests/test_host_sanitizers.py; prints "ok <table rows>" and exits 0, or
// names the first value that is not the rule's and exits 1.
#include "../../resvg_amd/csrc/png_demul.h"
#include <cstdio>

using namespace rvk_png;

int main() {
    Demul t{};
    if (!make_demul(t)) {
        std::printf("no factors\n");
        return 1;
    }
    int rows = 0;
    for (uint32_t a = 0; a < 256; a++) {
        const float r = t.r[a];
        rows += by_table(r);
        for (uint32_t c = 0; c < 256; c++) {
            uint32_t v = straight_channel(c, r);  // as the kernel: before the table's value replaces it
            if (by_table(r)) v = t.special[table_row(r)][c];
            if (v == demul_rule(c, a)) continue;
            std::printf("alpha %u channel %u: %u\n", a, c, v);
            return 1;
        }
    }
    std::printf("ok %d\n", rows);
    return 0;
}
