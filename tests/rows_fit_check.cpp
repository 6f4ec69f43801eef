// Runs csrc/rows_fit.h on the host against a memory of `limit` rows.
// Usage: rows_fit_check <want> <have> <most> <limit>; prints the rows granted and then
// each size asked for.
#include <cstdio>
#include <cstdlib>

#include "rows_fit.h"

int main(int argc, char **argv) {
    if (argc != 5) return 2;
    const long long want = atoll(argv[1]), have = atoll(argv[2]), most = atoll(argv[3]), limit = atoll(argv[4]);
    long long asked[64];
    int n = 0;
    const long long got = gaje::rows_fit(want, have, most, [&](int64_t rows) {
        if (n < 64) asked[n++] = rows;
        return rows <= limit;
    });
    printf("%lld", got);
    for (int i = 0; i < n; ++i) printf(" %lld", asked[i]);
    printf("\n");
}
