// The order in which the query tiles of causal attention go out where each has a workgroup of its own (sdpa.hip).
#pragma once

namespace axhip {
struct CausalTile {
    unsigned head, tile;
};
constexpr unsigned CAUSAL_GROUP = 32;       // heads

// Workgroup `block` of heads * nq.  A tile visits more keys the later it is, so the long ones go first and the short ones even out the ends; but heads whose
// tiles are spread over the whole launch share nothing of K and V in L2 (256 heads of [2048, 128] 1470 -> 1560 us).  So the `last` heads go longest
// first over all of them, and those before in groups of 32, longest first within a group: workgroups go to the 8 XCDs in turn, so that a head of a group of a
// multiple of eight stays on one XCD, and inside an XCD to its four shader engines in turn, so that each of these gets its share of every length only where
// four neighbours have the same (groups of 8: 512 heads of [1024, 96], whose tiles have four lengths, 620 -> 790 us).
__host__ __device__ inline CausalTile causal_tile(unsigned block, unsigned heads, unsigned nq, unsigned last) {
    const unsigned first = heads - last;                     // a multiple of 32
    if (block < first * nq) {
        const unsigned group = block / (CAUSAL_GROUP * nq), r = block - group * CAUSAL_GROUP * nq;
        return {group * CAUSAL_GROUP + r % CAUSAL_GROUP, nq - 1 - r / CAUSAL_GROUP};
    }
    block -= first * nq;
    const unsigned longer = block / last;
    return {first + block - longer * last, nq - 1 - longer};
}

// Heads that go longest first over all: tiles for twice the workgroups that the chip holds at once (for half of them: 88 of [1780, 128] 430 -> 540 us, once: 60 of [3367, 32]
// 304 -> 367, one and a half times: 61 of [4096, 32] 428 -> 457).
inline unsigned causal_last(long long heads, long long nq, long long resident) {
    const long long spread = 2 * resident / nq + 1;
    return (unsigned)(heads > spread ? heads - (heads - spread) / CAUSAL_GROUP * CAUSAL_GROUP : heads);
}
}  // namespace axhip
