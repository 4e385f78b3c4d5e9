// Host-side check of the waves' weight copies of a K row (Q4Piece, q4_common.h): for
// every N % 8 == 0 up to 1032 and every wave of every 256-column tile, each lane's 16- and
// 4-byte copy lies inside the row's 18 N bytes, and every byte of the wave's own
// columns is copied to its place.  Prints "ok" and exits 0, or the failing case and 1.
#include <cstdio>
#include <vector>

#include "q4_common.h"

int main() {
    constexpr int COLS = 64, TILE = 256;
    for (int N = 8; N <= 1032; N += 8) {
        const long row = 18L * N;
        for (int n = 0; n < (N + TILE - 1) / TILE * TILE; n += COLS) {
            const mcq4::Q4Piece p(n, COLS, N);
            std::vector<long> from(1024 + 4 * 64, -1);          // source byte of every slot byte
            for (int lane = 0; lane < 64; ++lane) {
                const long a = (long)p.start + p.off16(lane), b = (long)p.start + p.off4(lane);
                if (a < 0 || a + 16 > row || a % 16 || b < 0 || b + 4 > row || b % 4) {
                    printf("N=%d column %d lane %d: bytes %ld, %ld of a row of %ld\n", N, n, lane, a, b, row);
                    return 1;
                }
                for (int i = 0; i < 16; ++i) from[16 * lane + i] = a + i;
                for (int i = 0; i < 4; ++i) from[1024 + 4 * lane + i] = b + i;
            }
            for (long i = 0; i < 18L * COLS && n + i / 18 < N; ++i)
                if (from[i] != 18L * n + i) {
                    printf("N=%d column %d: slot byte %ld holds row byte %ld\n", N, n, i, from[i]);
                    return 1;
                }
        }
    }
    printf("ok\n");
    return 0;
}
