// Prints trd_pick's instance and workgroups for each "m cus cols" on stdin.
#include <cstdio>

#include "trd_shape.h"

int main() {
    int m, cus, cols;
    while (std::scanf("%d %d %d", &m, &cus, &cols) == 3) {
        const dzhip::TrdPick p = dzhip::trd_pick(m, cus, cols);
        std::printf("%d %d %d\n", p.nq, p.cw, p.groups);
    }
}
