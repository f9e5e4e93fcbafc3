// Reads "nnz wmax wsmall" lines and prints small, packed and sum32 of each.
#include <cstdio>

#include "widths.h"

int main() {
    long long nnz;
    unsigned long long wmax;
    int wsmall;
    while (scanf("%lld %llu %d", &nnz, &wmax, &wsmall) == 3) {
        const pggc::ContractWidths r = pggc::contract_widths(nnz, wmax, wsmall != 0);
        printf("%d %d %d\n", r.small, r.packed, r.sum32);
    }
    return 0;
}
