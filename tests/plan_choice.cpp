// The plan of a plain GEMM on 256 CUs, for every "M N K" on the standard input: macro tile, parts.
#include <cstdio>

#include "fo_plan.h"

int main() {
    int M, N, K;
    while (std::scanf("%d %d %d", &M, &N, &K) == 3) {
        const fo::Plan p = fo::make_plan(128, 128, M, N, K, true, true, true, fo::Macro{0, 0}, 256);
        std::printf("%d %d %d\n", p.macro.m, p.macro.n, p.splits);
    }
    return 0;
}
