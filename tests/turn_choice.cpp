// Panels of K between the places at which the XCDs begin, in 256x128 tiles (and in 128x128 ones) on 256 CUs, for every "M N K" on the standard input.
#include <cstdio>

#include "fo_plan.h"

int main() {
    int M, N, K;
    while (std::scanf("%d %d %d", &M, &N, &K) == 3)
        std::printf("%d %d\n", fo::turn_panels(fo::Macro{256, 128}, M, N, K, 256), fo::turn_panels(fo::Macro{128, 128}, M, N, K, 256));
    return 0;
}
