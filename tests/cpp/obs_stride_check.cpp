// The checkpoint spacings of observed solves (obs_stride_max, obs_first_stride in
// va_kernels.hpp) followed through a forward on the host: for every cap, slot count,
// previous and new step count, the checkpoints fit the slots and every segment the
// row buffer of stride_max rows.  Prints "checked <n> bad <m>".
#include <stdio.h>
#include <stdlib.h>

#include "va_kernels.hpp"

int main(int argc, char **argv)
{
    const int top = argc > 1 ? atoi(argv[1]) : 80;
    long checked = 0, bad = 0;
    for (int cap = 1; cap <= top; ++cap)
        for (int slots = 2; slots <= 34; slots += 2) {
            const int smax = va::obs_stride_max(cap, slots);
            for (int prev = 0; prev <= cap; ++prev)
                for (int steps = 0; steps <= cap; ++steps) {
                    // k_obs_fwd: a checkpoint at every stride-th step below the cap
                    int stride = va::obs_first_stride(prev, slots, smax), nck = 0;
                    bool ok = stride >= 1 && (stride & (stride - 1)) == 0;
                    for (int count = 0; count < steps; ++count)
                        if ((count & (stride - 1)) == 0) {
                            if (nck >= slots) {
                                stride *= 2;
                                nck = slots / 2;
                            }
                            ok = ok && nck < slots && nck == count / stride;
                            ++nck;
                        }
                    // the reverse: segments of stride rows, the last one shorter
                    const int nseg = (steps + stride - 1) / stride;
                    ok = ok && stride <= smax && nseg <= nck;
                    // one level: every segment in stride_max rows
                    for (int j = 0; j < nseg; ++j) {
                        const int n0 = j * stride;
                        const int len = steps - n0 < stride ? steps - n0 : stride;
                        ok = ok && len >= 1 && len <= smax;
                    }
                    // a solve with the same steps again never fills the slots
                    if (steps == prev && prev < cap)
                        ok = ok && stride == va::obs_first_stride(prev, slots, smax);
                    ++checked;
                    bad += !ok;
                    if (!ok && bad < 5)
                        printf("cap %d slots %d smax %d prev %d steps %d stride %d\n", cap, slots,
                               smax, prev, steps, stride);
                }
        }
    printf("checked %ld bad %ld\n", checked, bad);
    return 0;
}
