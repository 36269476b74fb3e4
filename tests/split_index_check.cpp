// Host-side check of trmoe::split_index (where a K split's partial lies): reads
// "split rows cols row col" lines from stdin and prints one index per line.
// Built by tests/test_split_index.py.
#include "trmoe_map.h"

#include <stdio.h>

int main() {
    int split, rows, cols, row, col;
    while (scanf("%d %d %d %d %d", &split, &rows, &cols, &row, &col) == 5)
        printf("%lld\n", (long long)trmoe::split_index(split, rows, cols, row, col));
    return 0;
}
