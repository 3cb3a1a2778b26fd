// Prints the tile kernels' plans (cubework_amd/csrc/gemm_plan.hip) of the products on stdin, host only: one
// "layout M N K steps lda ldb aligned_a aligned_b" a line, as "cfg rows full slices rest" (rest: the tiles that are sliced).
#include <cstdio>

#include "../../cubework_amd/csrc/gemm_plan.h"

int main() {
    long long layout, M, N, K, steps, lda, ldb, al_a, al_b;
    while (scanf("%lld %lld %lld %lld %lld %lld %lld %lld %lld", &layout, &M, &N, &K, &steps, &lda, &ldb, &al_a, &al_b) == 9) {
        const cw::TilePlan p = cw::tile_plan((int)layout, M, N, K, (int)steps, lda, ldb, al_a != 0, al_b != 0, 0, -1);
        printf("%d %d %d %d %lld\n", p.cfg, p.rows, p.full, p.slices, (long long)p.tiles - p.full);
    }
    return 0;
}
