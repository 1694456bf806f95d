// Host build of pocket-engine_amd/csrc/pkv_index.h: the kernels' index
// arithmetic against the bounds of the buffers it indexes. Prints what is out
// of bounds and returns 1, else "ok".
#include "../pocket-engine_amd/csrc/pkv_index.h"

#include <climits>
#include <cstdio>
#include <vector>

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

// Every head of every token read from its place in the row and stored once,
// none of a token without a slot (-1, or past the pool) in the cache, nothing
// out of the rows, the query output or the cache; waves past the last token do
// nothing. As prep_kernel<P> walks it, 32 lanes of 8 values per half-wave.
static void prep_rows(int Hq, int Hkv, int T, int P) {
    const pkv::PrepPairs pr(Hq, Hkv);
    const int nu = pr.units(), groups = pr.groups(P), heads = 2 * Hq + 2 * Hkv, slots = T;
    const unsigned grid = pkv::prep_grid(T, groups);
    std::vector<int> q(T * Hq), kv[2] = {std::vector<int>(slots * Hkv), std::vector<int>(slots * Hkv)};
    auto slot_of = [&](int t) { return t % 7 == 0 ? -1 : t % 7 == 3 ? slots : T - 1 - t; };
    for (long i = 0; i < 4l * grid; i++) {
        const int t = (int)(i / groups), u0 = (int)(i % groups) * P;
        if (t >= T) continue;
        const bool has_slot = slot_of(t) >= 0 && slot_of(t) < slots;
        for (int hv = 0; hv < 2; hv++)
            for (int k = 0; k < P; k++) {
                const int load = u0 + k < nu - 1 ? u0 + k : nu - 1, src = pr.source(load, hv);
                CHECK(load >= 0 && src >= 0 && src < heads, "%d / %d heads, unit %d half %d: row head %d", Hq, Hkv, load,
                      hv, src);
            }
        for (int k = 0; k < P && u0 + k < nu; k++) {
            const int u = u0 + k;
            if (!pr.is_q(u) && !has_slot) break;
            for (int hv = 0; hv < 2; hv++) {
                const int h = pr.head(u, hv), src = pr.source(u, hv);
                if (!pr.has(u, hv)) continue;
                const int n = pr.is_q(u) ? Hq : Hkv;
                CHECK(h >= 0 && h < n, "%d / %d heads, unit %d half %d: head %d of %d", Hq, Hkv, u, hv, h, n);
                CHECK(src == (pr.is_q(u) ? 2 * h : 2 * Hq + (pr.is_v(u) ? Hkv : 0) + h), "unit %d: source %d", u, src);
                if (pr.is_q(u)) q[t * Hq + h]++;
                else kv[pr.is_v(u)][slot_of(t) * Hkv + h]++;
            }
        }
    }
    for (int n : q) CHECK(n == 1, "%d / %d heads, T %d, P %d: a q head stored %d times", Hq, Hkv, T, P, n);
    for (auto& c : kv)
        for (int s = 0; s < slots; s++)
            for (int h = 0; h < Hkv; h++) {
                const int t = T - 1 - s, want = slot_of(t) == s;
                CHECK(c[s * Hkv + h] == want, "%d / %d heads, T %d, P %d: slot %d head %d stored %d times", Hq, Hkv, T, P,
                      s, h, c[s * Hkv + h]);
            }
}
static void prep() {
    for (int Hq = 2; Hq <= 64; Hq += 2)
        for (int Hkv = 0; Hkv <= 16; Hkv++)
            for (int T : {1, 2, 3, 37})
                for (int P : {1, 4}) prep_rows(Hq, Hkv, T, P);
    // the last wave of the largest launches: token T - 1's last pairs, no wrap
    for (int Hq : {2, 16, 64})
        for (int P : {1, 4}) {
            const pkv::PrepPairs pr(Hq, 8);
            const int T = 1 << 24, groups = pr.groups(P);
            const long waves = 4l * pkv::prep_grid(T, groups), last = (long)T * groups - 1;
            CHECK(last < waves && waves <= last + 4 && last / groups == T - 1 && P * (last % groups) < pr.units(),
                  "grid of %d tokens, %d heads", T, Hq);
        }
}

int main() {
    ranges();
    prep();
    puts(bad ? "failed" : "ok");
    return bad != 0;
}
