// Host build of pocket-engine_amd/csrc/pkv_index.h: the kernels' index
// arithmetic against the bounds of the buffers it indexes. Prints what is out
// of bounds and returns 1, else "ok".
#include "../pocket-engine_amd/csrc/pkv_index.h"

#include <climits>
#include <cstdio>
#include <cstring>

static int bad = 0;
#define CHECK(cond, ...)                                     \
    do {                                                     \
        if (!(cond) && bad++ < 20) printf(__VA_ARGS__), puts(""); \
    } while (0)

// Ranges tile [0, W) and every later one is empty, for the settings that
// pkv_attn_decode_config takes (1 .. 64 workgroups per CU, 1 .. 2^20 keys at
// least) on 256 CUs, twice as many workgroups over an E4M3 cache and up to 4
// ranges to a workgroup.
static void ranges() {
    const int wgs[] = {1, 3, 64}, mins[] = {1, 32, 1000, 1 << 20}, mult[] = {1, 2, 4, 8};
    const int keys[] = {1, 31, 32, 33, 4097, 300000, 1 << 20, (1 << 20) + 1, 1 << 28, INT_MAX - (1 << 18)};
    for (int wg : wgs)
        for (int lo : mins)
            for (int m : mult)
                for (int W : keys) {
                    const int n = 256 * wg * m, most = (W + n - 1) / n, R = lo > most ? lo : most;
                    int at = 0;
                    for (int b = 0; b < n; b++) {
                        const int s = pkv::range_start(b, R, W), e = pkv::range_end(s, R, W);
                        CHECK(s == at && e >= s && e <= W && e - s <= R, "range %d of %d, R %d, W %d: [%d, %d) after %d",
                              b, n, R, W, s, e, at);
                        at = e;
                    }
                    CHECK(at == W, "%d ranges, R %d: keys %d of %d", n, R, at, W);
                }
}

int main() {
    ranges();
    puts(bad ? "failed" : "ok");
    return bad != 0;
}
