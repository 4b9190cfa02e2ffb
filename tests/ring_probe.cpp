// Test helper: the cells that wrapped_run names, in order.
#include "boids_internal.h"

extern "C" int run_cells(int x0, int x1, int G, int* out)
{
    int n = 0;
    for (int part = 0; part < 2; ++part) {
        int a, z;
        boids::wrapped_run(x0, x1, G, part, &a, &z);
        for (int c = a; c <= z && n < 4 * G; ++c) out[n++] = c;
    }
    return n;
}
