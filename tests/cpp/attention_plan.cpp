// Sweeps of the attention's chunk rule and workspace size (csrc/attention_plan.hpp).
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "attention_plan.hpp"

using namespace anelm;

static void need(bool ok, const char* what, long a, long b, long c = 0, long d = 0) {
    if (ok) return;
    std::printf("%s: %ld %ld %ld %ld\n", what, a, b, c, d);
    std::exit(1);
}

int main() {
    // One ring: its chunks cover it; with pairs for at most half the CUs every
    // ring past one workgroup's rows is split, and with few of them a short
    // ring is spread over at least 64 workgroups, whatever the capacity is.
    for (int P = 1; P <= kMaxPairs; P++) {
        int most = 1;
        for (int len = 1; len <= 9000; len++) {
            const int c = ring_chunk(P, len), n = ring_chunks(P, len);
            need(c == 64 || c == 128 || c == 256 || c == 512, "chunk", P, len, c);
            need(len <= kWholeRows ? n == 1 : (long)n * c >= len && (long)(n - 1) * c < len, "cover", P, len, n);
            need(len <= kWholeRows || P > 128 || n >= 2, "one workgroup on a long ring", P, len);
            need(len < 500 || P < 8 || P * n >= 64, "short ring on few workgroups", P, len, n);
            most = std::max(most, n);
            need(max_chunks(P, len) == most, "max_chunks", P, len, most, max_chunks(P, len));
        }
    }
    // Every call with at most the batch and the capacity that a workspace was
    // sized for fits in it, at each side of each of the rules' lines.
    const int caps[] = {1, 64, 65, 128, 129, 200, 256, 257, 384, 512, 513, 640, 1000, 1024, 1025, 1563, 2048, 3968, 3969,
                        4096, 6000, 8192, 16256, 16257, 27500, 32768, 65536, 131072, 262144};
    const long batches[] = {1, 2, 3, 4, 5, 8, 13, 16, 17, 31, 32, 48, 64, 65, 100, 128, 129, 256, 300, 1000};
    for (int nkv : {1, 2, 3, 4, 8, 10, 32, 128})
        for (int D : {64, 256})
            for (long batch : batches)
                for (int cap : caps) {
                    const int nh = 2 * nkv;
                    const size_t S = ws_bytes_for(batch, nh, nkv, D, cap);
                    std::vector<long> bs;
                    for (long b = 1; b <= batch && b <= 80; b++) bs.push_back(b);
                    for (long b : batches)
                        if (b <= batch) bs.push_back(b);
                    for (long b : bs)
                        for (int k : caps) {
                            if (k > cap) break;
                            const int n = max_chunks((int)std::min(b * nkv, (long)kMaxPairs), k);
                            if (n == 1) continue;
                            need(partial_bytes(b, nh, n, D) <= ctr_offset(S) && (size_t)(b * nkv) <= ctr_slots(S),
                                 "workspace", b, k, nkv, n);
                        }
                }
    std::puts("ok");
    return 0;
}
