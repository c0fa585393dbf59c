// ratio_of() of the library against the division, for every pair of sizes a parameter record can hold. Built and run by
// tests/test_quotients_cpu.py.
#include <stdio.h>

#include "rmx_common.h"

int main() {
    long wrong = 0;
    for (int b = 1; b <= 0x3fff; b++) {
        const float fb = (float)b, recip = 1.0f / fb;
        for (int a = 1; a <= 0x3fff; a++) wrong += ratio_of((float)a, fb, recip) != (float)a / fb;
    }
    printf("%ld\n", wrong);
    return wrong != 0;
}
