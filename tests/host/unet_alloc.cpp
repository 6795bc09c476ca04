// A training step whose n-th allocation fails, for every n, on a network that has trained on
// a smaller grid: the step reports it, and either grid trains afterwards with every buffer in
// place (as many as on a network that never failed).
#include <cstdio>

#include "shk_projection.h"

void fail_allocation(long n);
void fill_memory(double v);
long allocations();
long live_allocations();

int train(shk_unet *net, int nx, int ny, int nz) {
    static float x[4];
    double loss;
    return shk_unet_train_step(net, nx, ny, nz, x, x, x, x, x, x, 0.8, 0.0f, &loss);
}

int main() {
    fill_memory(1.0);  // sums of kernels: positive
    int bad = 0;
    long whole = 0, tried = 0;
    for (long k = 0; k < 2 || k / 2 <= tried; ++k) {
        const long n = k / 2;   // 0: none fails
        const bool again = k & 1;   // the same grid afterwards, or the smaller one
        shk_unet *net = nullptr;
        fail_allocation(0);
        if (shk_unet_create(1, 0, &net) || train(net, 16, 16, 16)) return 2;
        fail_allocation(n);
        const int rc = train(net, 64, 48, 32);
        if (n == 0) tried = allocations();
        fail_allocation(0);
        if (rc != (n ? SHK_OUT_OF_MEMORY : SHK_OK)) ++bad, std::printf("allocation %ld: status %d\n", n, rc);
        if (again ? train(net, 64, 48, 32) : train(net, 16, 16, 16))
            ++bad, std::printf("allocation %ld: the next step fails\n", n);
        if (k == 0) whole = live_allocations();
        if (live_allocations() != whole)
            ++bad, std::printf("allocation %ld, %s grid next: %ld buffers of %ld\n", n, again ? "the same" : "the smaller", live_allocations(), whole);
        shk_unet_destroy(net);
        if (live_allocations()) ++bad, std::printf("allocation %ld: %ld left\n", n, live_allocations());
    }
    std::printf("%ld allocations, %d wrong\n", tried, bad);
    return bad != 0 || tried < 10;
}
