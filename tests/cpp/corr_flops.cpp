// Prints, for steps per period n = 1..600: n, log2 of the correlation's transform length (0: direct
// sum) and the engine's flop counts per element of 1000 FID points, general and autocorrelation.
#include "fake_hip.h"

#include "../../blochlib_amd/csrc/blfid_host.cpp"

int main() {
    for (int n = 1; n <= 600; n++)
        std::printf("%d %d %.17g %.17g\n", n, corr_fft_ln(n), corr_flops_per_elem(n, 1000),
                    corr_flops_per_elem(n, 1000, true));
    return 0;
}
