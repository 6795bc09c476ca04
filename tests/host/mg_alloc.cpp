// The multigrid tables of a new brick set, their n-th allocation failing for every n: the
// next projection builds them whole (as many buffers as where nothing failed).
#include <cstdio>

#include "ctx_internal.h"

void fail_allocation(long n);
long allocations();
long live_allocations();

namespace shk {
int mg_setup(shk_ctx *c);
}

void bricks(shk_ctx &c, int keep) {
    const int n = c.nbx * c.nby * c.nbz;
    c.h_slot.assign(n, -1);
    c.h_coord.clear();
    for (int b = 0; b < n; ++b)
        if (b % keep == 0) {
            c.h_slot[b] = (int)c.h_coord.size();
            c.h_coord.push_back(make_int4(b % c.nbx, b / c.nbx % c.nby, b / (c.nbx * c.nby), 0));
        }
    c.n_active = (int)c.h_coord.size();
}

int main() {
    int bad = 0;
    long whole = 0, tried = 0;
    for (long n = 0; n == 0 || n <= tried; ++n) {
        fail_allocation(0);
        shk_ctx *c = new shk_ctx();
        c->dims = {70, 61, 52};
        c->dims.bx = 8;
        c->nbx = 9;
        c->nby = 8;
        c->nbz = 7;
        bricks(*c, 3);
        if (shk::mg_setup(c)) return 2;
        bricks(*c, 1);
        fail_allocation(n);
        const int rc = shk::mg_setup(c);
        if (n == 0) tried = allocations();
        fail_allocation(0);
        if (rc != (n ? SHK_OUT_OF_MEMORY : SHK_OK)) ++bad, std::printf("allocation %ld: status %d\n", n, rc);
        if (shk::mg_setup(c)) ++bad, std::printf("allocation %ld: the next setup fails\n", n);
        if (n == 0) whole = live_allocations();
        if (live_allocations() != whole)
            ++bad, std::printf("allocation %ld: %ld buffers of %ld\n", n, live_allocations(), whole);
        shk::mg_destroy(c->mg);
        delete c;
        if (live_allocations()) ++bad, std::printf("allocation %ld: %ld left\n", n, live_allocations());
    }
    std::printf("%ld allocations, %d wrong\n", tried, bad);
    return bad != 0 || tried < 10;
}
