// The batched path's workspace (qw6_moe.h) on the CPU: layers of different shapes
// in turn, allocations that fail, and the buffers' places. Prints "ok" or the line that failed.
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <vector>

#include "qw6_moe.h"

using namespace qw6;

#define CHECK(c)                                                 \
    do {                                                         \
        if (!(c)) {                                              \
            printf("line %d: %s\n", __LINE__, #c);               \
            exit(1);                                             \
        }                                                        \
    } while (0)

struct Span {
    uintptr_t a;
    size_t n;
};

// What the kernels of a hidden x inter call of T tokens write or read of the workspace.
static std::vector<Span> used(const PrefillWs& w, uint32_t T, uint32_t hidden, uint32_t inter) {
    const bool three = T < kPrefill3PartBelow;
    const size_t K = 8, E = T * K + T, t = T, parts = three ? 3 : 2;
    return {{(uintptr_t)w.pidx, t * K * 4}, {(uintptr_t)w.pw, t * K * 4},
            {(uintptr_t)w.ent_tok, E * 4}, {(uintptr_t)w.ent_w, E * 4}, {(uintptr_t)w.ent_pos, t * K * 4},
            {(uintptr_t)w.tiles, (size_t)prefill_tiles_max(T, 8, 256, three) * 16}, {(uintptr_t)w.n_tiles, 8},
            {(uintptr_t)w.logits, t * 256 * 4}, {(uintptr_t)w.xn, t * hidden * 4},
            {(uintptr_t)w.xp, t * hidden * 2 * parts}, {(uintptr_t)w.xs, t * (hidden / 32) * 8},
            {(uintptr_t)w.xinv, t * 4}, {(uintptr_t)w.mp, E * inter * 2 * parts},
            {(uintptr_t)w.ms, E * (inter / 32) * 8}, {(uintptr_t)w.minv, E * (inter / 64) * 4},
            {(uintptr_t)w.ybuf, E * hidden * 4}};
}

int main() {
    constexpr uintptr_t kBase = (uintptr_t)1 << 40;   // addresses only: nothing is read or written
    const uint32_t dims[] = {256, 512, 1024, 2048};
    for (uint32_t max_T : {1u, 17u, 63u, 64u, 65u, 2048u, kPrefillMaxBatch}) {
        PrefillWsOwner o = {};
        uint32_t n = 0;
        uintptr_t at = 0;
        size_t size = 0;
        bool fails = false;
        auto alloc = [&](size_t bytes, void** p) {
            if (fails) return -1;
            at = kBase * ++n;
            size = bytes;
            *p = (void*)at;
            return 0;
        };
        srand(7);
        for (int i = 0; i < 400; i++) {
            const uint32_t h = dims[rand() % 4], m = dims[rand() % 4];
            fails = rand() % 2;
            const PrefillWsOwner before = o;
            const int rc = grow_prefill_ws(o, max_T, h, m, alloc);
            const bool held = before.hidden >= h && before.inter >= m;
            CHECK(rc == (fails && !held ? -1 : 0));
            if (rc) {   // nothing changed
                CHECK(o.hidden == before.hidden && o.inter == before.inter && o.ws.ybuf == before.ws.ybuf &&
                      o.ws.xp == before.ws.xp && o.ws.mp == before.ws.mp && o.ws.minv == before.ws.minv);
                continue;
            }
            CHECK(o.hidden >= h && o.inter >= m && o.hidden >= before.hidden && o.inter >= before.inter);
            if (held) CHECK(o.ws.ybuf == before.ws.ybuf && o.ws.pidx == before.ws.pidx);
            std::vector<uint32_t> ts = {1, 16, 17, 33, 63, 64, 65, 100, max_T};
            for (uint32_t T : ts) {
                if (T > max_T) continue;
                std::vector<Span> s = used(o.ws, T, h, m);
                std::sort(s.begin(), s.end(), [](const Span& a, const Span& b) { return a.a < b.a; });
                CHECK(s.front().a >= at && s.back().a + s.back().n <= at + size);
                for (size_t k = 0; k < s.size(); k++) {
                    CHECK(s[k].a % 256 == 0);
                    if (k) CHECK(s[k - 1].a + s[k - 1].n <= s[k].a);
                }
            }
        }
        CHECK(o.hidden == 2048 && o.inter == 2048 && n <= 7);
    }
    printf("ok\n");
    return 0;
}
