// How a decode attention launch splits rings into chunks, and the workspace
// that takes: plain arithmetic, the same on the host and in the kernel.
#pragma once

#include <cstddef>
#include <initializer_list>

#ifdef __HIPCC__
#define ANELM_HD __host__ __device__
#else
#define ANELM_HD
#endif

namespace anelm {

constexpr int kMinChunk = 64, kMaxChunk = 512;   // ring positions per workgroup of a split launch
constexpr int kWholeRows = 128;                  // rings up to this long are never split
// Chunks of 64, 128 and 256 are for launches of up to so many rows (see ring_chunk)
constexpr int kRows64 = 16384, kRows128 = 75000, kRows256 = 220000;
constexpr int kMaxPairs = kRows256 / kMaxChunk + 1;   // from here on every ring takes kMaxChunk

// Positions per workgroup for a ring of len rows in a launch of `pairs`
// (sequence, kv head) pairs, at most kMaxPairs.  A split ring costs its last
// workgroup three more memory round trips (partials stored, counted, read
// back: 2 us), and merging them takes longer the more there are; a CU pulls a
// ring in at no more than about 45 GB/s, whatever its waves, so few workgroups
// are slow too.  The rows are the launch's if all its rings are as long as
// this one: 64 loses to 128 from the second workgroup per CU on, 128 to 256
// and 256 to 512 from the third or fourth, whose merges and set-up outweigh
// the shorter chunks; past 16 chunks of 64 the merge takes as long as a chunk.
// Rings that fit one chunk are not split where two parts each are more than a
// workgroup per CU (512 rows: where the rings alone are).  The ring's own
// length decides, not the capacity: a short ring in a long capacity is spread
// as well as in its own.
// us per launch with chunks of 64 / 128 / 256 / 512 (8 waves, 8 kv heads,
// groups of 4, fused q/k norm, capacity 4096; this rule's in brackets):
//     1 sequence  x  500 rows: [ 8.5]/  9.8 / 13.7 / 19.0
//     1 sequence  x 4096 rows:  18.6 /[15.3]/ 16.0 / 21.5
//     5 sequences x 1024 rows:  16.8 /[14.4]/ 15.6 / 22.0
//     6 sequences x 4096 rows:  50.6 / 40.2 /[37.2]/ 38.7
//     8 sequences x  256 rows: [ 9.7]/ 10.7 / 12.3 / 12.3
//     8 sequences x  500 rows:  12.7 /[11.8]/ 15.1 / 19.9
//     8 sequences x 1024 rows:  21.9 /[17.1]/ 17.0 / 23.3   (ragged [13.5] / 14.8)
//    16 sequences x  256 rows:  15.5 /[11.6]/ 12.8 / 12.9
//    16 sequences x 2048 rows:  66.4 / 54.7 / 50.4 /[48.0]
//    24 sequences x  256 rows:  22.2 / 15.1 /[13.7]/ 13.7
//    32 sequences x  500 rows:  41.8 / 31.3 / 26.7 /[25.0]
//    48 sequences x 1024 rows: 103.5 / 80.7 / 71.4 /[68.5]
ANELM_HD inline int ring_chunk(int pairs, int len) {
    if (len <= 256 && pairs > 128) return pairs < 256 ? 256 : 512;
    if (len <= 512 && pairs >= 256) return 512;
    const int rows = pairs * len;
    if (rows > kRows256) return 512;
    if (rows > kRows128) return 256;
    return rows > kRows64 || len > 16 * kMinChunk ? 128 : 64;
}

// Chunks of a ring of len rows: one workgroup does it alone up to kWholeRows.
ANELM_HD inline int ring_chunks(int pairs, int len) {
    const int c = ring_chunk(pairs, len);
    return len <= kWholeRows ? 1 : (len + c - 1) / c;
}

// The most chunks that any ring of at most `bound` rows has: at the longest
// ring of one chunk size.
inline int max_chunks(int pairs, int bound) {
    int most = 1;
    for (int last : {bound, 256, 512, 16 * kMinChunk, kRows64 / pairs, kRows128 / pairs, kRows256 / pairs}) {
        const int n = last <= bound ? ring_chunks(pairs, last) : 1;
        most = n > most ? n : most;
    }
    return most;
}

// Split launches: the partials from the workspace's start, and one counter
// per (sequence, kv head) in a region whose place depends on the workspace's
// size alone: its last 64th, from a 256-byte boundary.  Every call given the
// same workspace and size therefore finds each counter at the same address,
// left at zero by the calls before, whatever its batch, chunking or ring
// lengths, and no call's partials reach into the region (checked per call).
inline size_t partial_bytes(long batch, int nh, int nsplit, int D) {
    return ((size_t)batch * nh * nsplit * (D + 2) * sizeof(float) + 255) & ~(size_t)255;
}
inline size_t ctr_offset(size_t ws_bytes) { return (ws_bytes - ws_bytes / 64) & ~(size_t)255; }
inline size_t ctr_slots(size_t ws_bytes) { return (ws_bytes - ctr_offset(ws_bytes)) / sizeof(unsigned); }

// The chunk that the workspace is sized for: the largest that gives
// kSizedBlocks workgroups, or else 64.  Every launch fits in what it gives,
// for the same batch or, with the maximum over the batches, a smaller one:
// chunks of 64 throughout are the most that any ring has, and chunks of 512
// the fewest; where the size is for chunks between, it holds kSizedBlocks of
// them, and no launch with chunks below 512 has more than its rows (kRows64,
// kRows128, kRows256) come to, and one per pair (under kMaxPairs of them).
constexpr long kSizedBlocks = 2048;
static_assert(kSizedBlocks >= kRows256 / 256 + kMaxPairs && kRows256 / 256 >= kRows128 / 128 &&
                  kRows256 / 256 >= kRows64 / 64,
              "every launch's partials fit the workspace");
inline int ws_chunk(long pairs, int bound) {
    for (int c = kMaxChunk; c > kMinChunk; c >>= 1) {
        if (pairs * ((bound + c - 1) / c) >= kSizedBlocks) return c;
    }
    return kMinChunk;
}

// A size that serves every call with at most `batch` sequences and a ring
// bound of at most `cap`.  The chunk follows the batch (ws_chunk), so a
// smaller batch can need more partials than the largest one: the maximum is
// taken over the batches up to `batch`.  Past the batch at which the chunk
// reaches its maximum the partials only grow with the batch, so the loop
// stops there and `batch` itself is counted last.
inline size_t ws_bytes_for(long batch, int nh, int nkv, int D, int cap) {
    size_t P = 0;
    auto count = [&](long b) {
        const int chunk = ws_chunk(b * nkv, cap);
        const long nsplit = (cap + chunk - 1) / chunk;
        if (nsplit > 1) {
            const size_t pb = partial_bytes(b, nh, (int)nsplit, D);
            P = pb > P ? pb : P;
        }
    };
    for (long b = 1; b < batch && ws_chunk(b * nkv, cap) < kMaxChunk; b++) count(b);
    count(batch);
    if (P == 0) return 0;
    const size_t pairs = (size_t)batch * nkv;
    size_t S = (((P + 256) * 64 / 63 + 256) + 255) & ~(size_t)255;
    if (S < 256 * pairs) S = 256 * pairs;
    while (ctr_offset(S) < P || ctr_slots(S) < pairs) S += 256;
    return S;
}

}  // namespace anelm
