// kb_weights.cpp -- the device's float Kaiser-Bessel weights (gadgetron_amd/csrc/gt_kb.h)
// on the host, for the gridding kernels' error against double sums over them.
#include "gt_kb.h"

// Positions p[n] on a grid of nos cells: first cell and KW weights of each window.
extern "C" void kb_weights(const float* p, int n, float nos, float W, float os_factor, int KW, int* first, float* w) {
    const float radius = W / 2.0f, one_over_W = 1.0f / W, beta = gt::kb_beta(W, os_factor);
    for (int i = 0; i < n; i++) {
        first[i] = int(std::ceil(p[i] - radius));
        const int last = int(std::floor(p[i] + radius));
        for (int k = 0; k < KW; k++) {
            const int cell = first[i] + k;
            const float u = std::fabs(float(cell) - p[i]);
            w[i * KW + k] = cell <= last && !(u > radius) ? gt::kb1(u, nos, one_over_W, beta) : 0.0f;
        }
    }
}
