// The dispatch rules of z2h_rules.h for one query per line of stdin; prints 0 or 1 per query.
#include "../../zonos2.cpp_amd/csrc/z2h_rules.h"
#include <cstdio>
#include <cstring>

int main() {
    char what[32];
    long long a, b, c, d, e;
    while (std::scanf("%31s %lld %lld %lld %lld %lld", what, &a, &b, &c, &d, &e) == 6) {
        if (!std::strcmp(what, "tall")) std::printf("%d\n", (int) z2r::f16_tall_tiles(a, b, (int) c, (int) d));
        else if (!std::strcmp(what, "few")) std::printf("%d\n", (int) z2r::f16_few_rows(a, (int) b, (int) c));
        else if (!std::strcmp(what, "rdown")) std::printf("%d\n", (int) z2r::router_down_reuse((int) a, (int) b, c != 0));
        else if (!std::strcmp(what, "qexp")) std::printf("%d\n", (int) z2r::quant_gemm_experts(a != 0, b, (int) c, d, e));
        else return 1;
    }
    return 0;
}
