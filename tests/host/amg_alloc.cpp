// The aggregation hierarchy of a CSR matrix, its n-th allocation failing for every n: the next
// solve builds it whole (as many buffers as where nothing failed).
#include <cstdio>
#include <vector>

#include "ctx_internal.h"

void fail_allocation(long n);
long allocations();
long live_allocations();

int main() {
    // 1D Laplacian, one Dirichlet end
    const int64_t rows = 3000;
    std::vector<int64_t> ptr{0}, col;
    std::vector<double> val;
    for (int64_t i = 0; i < rows; ++i) {
        if (i) col.push_back(i - 1), val.push_back(-1.0);
        col.push_back(i), val.push_back(i ? 2.0 : 3.0);
        if (i + 1 < rows) col.push_back(i + 1), val.push_back(-1.0);
        ptr.push_back((int64_t)col.size());
    }
    int bad = 0;
    long whole = 0, tried = 0;
    for (long n = 0; n == 0 || n <= tried; ++n) {
        shk_ctx *c = new shk_ctx();
        fail_allocation(n);
        const int rc = shk::amg_setup(c, rows, ptr.data(), col.data(), val.data());
        if (n == 0) tried = allocations();
        fail_allocation(0);
        if (rc != (n ? SHK_OUT_OF_MEMORY : SHK_OK)) ++bad, std::printf("allocation %ld: status %d\n", n, rc);
        if (shk::amg_setup(c, rows, ptr.data(), col.data(), val.data()))
            ++bad, std::printf("allocation %ld: the next setup fails\n", n);
        if (n == 0) whole = live_allocations();
        if (live_allocations() != whole)
            ++bad, std::printf("allocation %ld: %ld buffers of %ld\n", n, live_allocations(), whole);
        shk::amg_destroy(c->amg);
        delete c;
        if (live_allocations()) ++bad, std::printf("allocation %ld: %ld left\n", n, live_allocations());
    }
    std::printf("%ld allocations, %d wrong\n", tried, bad);
    return bad != 0 || tried < 10;
}
