// The learned preconditioner's buffers, their n-th allocation failing for every n: the next
// solve has them all (as many as where nothing failed).
#include <cstdio>

#include "ctx_internal.h"

void fail_allocation(long n);
long allocations();
long live_allocations();

namespace shk {
// nothing to solve: the solve ends after its set-up
int true_residual(shk_ctx *, const double *, double *, double out[4], const double *, float *) {
    out[0] = out[1] = out[2] = out[3] = 0.0;
    return SHK_OK;
}
void fill_true_residual(shk_result *, const double *) {}
}

int main(int, char **argv) {
    shk_unet *net = nullptr;
    if (shk_unet_create(1, 0, &net) || shk_unet_save(net, argv[1])) return 2;
    shk_unet_destroy(net);
    int bad = 0;
    long whole = 0, tried = 0;
    for (long n = 0; n == 0 || n <= tried; ++n) {
        shk_ctx *c = new shk_ctx();
        c->dims = {32, 32, 32};
        c->dims.bx = 8;
        c->nbx = c->nby = c->nbz = 4;
        c->n_active = 64;
        c->unknowns = 64 * 512;
        c->prm.precond = 2;
        c->prm.unet_weights = argv[1];
        (void)c->x64.ensure(64 * 512);
        shk_result res{};
        fail_allocation(n);
        const int rc = shk::unet_solve(c, &res);
        if (n == 0) tried = allocations();
        fail_allocation(0);
        if (rc != (n ? SHK_OUT_OF_MEMORY : SHK_OK)) ++bad, std::printf("allocation %ld: status %d\n", n, rc);
        if (shk::unet_solve(c, &res)) ++bad, std::printf("allocation %ld: the next solve fails\n", n);
        if (n == 0) whole = live_allocations();
        if (live_allocations() != whole)
            ++bad, std::printf("allocation %ld: %ld buffers of %ld\n", n, live_allocations(), whole);
        shk::unet_destroy(c->unet);
        c->x64.release();
        delete c;
        if (live_allocations()) ++bad, std::printf("allocation %ld: %ld left\n", n, live_allocations());
    }
    std::printf("%ld allocations, %d wrong\n", tried, bad);
    return bad != 0 || tried < 10;
}
