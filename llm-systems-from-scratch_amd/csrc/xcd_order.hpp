// Order of a launch's workgroups over the eight XCDs (plain arithmetic, host and device).
#pragma once

namespace mi355 {

#if defined(__HIP__)
#define MI355_ORDER __host__ __device__ __forceinline__
#else
#define MI355_ORDER inline
#endif

// Logical id of workgroup `bid`, of which the first n have work.  Workgroup ids are dealt round-robin to the 8 XCDs, each with
// an L2 of its own; the XCDs take whole chunks in turn, so that the workgroups of a chunk, which read the same rows, are resident
// on one XCD at about the same time.  What is left after the whole rounds of eight chunks is cut into eight runs of the same
// length (give or take one): an XCD that got a whole chunk of them would work on it while others have none.
MI355_ORDER int xcd_even_id(int bid, int n, int chunk) {
    const int round = 8 * chunk, whole = n / round * round, xcd = bid % 8;
    if (bid < whole) {
        const int k = bid / 8, turn = k / chunk;
        return (turn * 8 + xcd) * chunk + (k - turn * chunk);
    }
    const int left = n - whole, more = left % 8;
    return whole + xcd * (left / 8) + (xcd < more ? xcd : more) + (bid - whole) / 8;
}

// Units of heads, each unit of every head a workgroup: `group` query heads read the rows of one kv head, of which there are n_groups.  An XCD takes every
// eighth kv head, chunk_heads query heads (whole kv heads) at a time, unit by unit.  The last n_groups % 8 kv heads come in front of all, on all XCDs.
// round > 0: an XCD's compute units, where all workgroups are resident at once.  They get workgroups in rounds then, and every other round goes the other way,
// so that units of falling cost meet.
struct HeadUnit {
    int unit, head;                               // unit -1: no work
};
MI355_ORDER int xcd_units_front(int n_units, int group, int n_groups) { return n_groups % 8 * group * n_units; }
MI355_ORDER int xcd_units_grid(int n_units, int group, int n_groups) {
    return (xcd_units_front(n_units, group, n_groups) + 7) / 8 * 8 + n_groups / 8 * 8 * group * n_units;
}
// Whether that grid can be launched: its threads are counted in 32 bits.
MI355_ORDER bool xcd_units_fit(long long n_units, long long group, long long n_groups, int threads) { return (n_units * group * n_groups + 7) * threads < 1LL << 32; }
// Whether shares of split keys, each a whole grid of them, the ids running on from one to the next, are spread evenly over the XCDs: not where workgroups without
// work fill up a share's grid, as then the few with work begin on the same XCDs in every share.
MI355_ORDER bool xcd_units_spread(int n_groups, int n_split) { return n_split <= 1 || n_groups % 8 == 0; }
MI355_ORDER int turned(int i, int n, int width) {
    const int start = width > 0 ? i / width * width : 0;
    return width > 0 && (i / width & 1) && start + width <= n ? 2 * start + width - 1 - i : i;
}
MI355_ORDER HeadUnit xcd_unit(int bid, int n_units, int group, int n_groups, int chunk_heads, int round) {
    const int front = xcd_units_front(n_units, group, n_groups), front8 = (front + 7) / 8 * 8;
    if (bid < front8) {
        if (bid >= front) return {-1, 0};
        const int heads = n_groups % 8 * group, i = turned(bid, front, 8 * round), unit = i / heads;
        return {unit, n_groups / 8 * 8 * group + i - unit * heads};
    }
    const int xcd = (bid - front8) & 7, heads = n_groups / 8 * group, i = turned((bid - front8) >> 3, n_units * heads, round);
    const int h0 = i / (n_units * chunk_heads) * chunk_heads, in_chunk = i - h0 * n_units, here = chunk_heads < heads - h0 ? chunk_heads : heads - h0;
    const int unit = in_chunk / here, hx = h0 + in_chunk - unit * here, g = hx / group;        // the XCD's query head and kv head
    return {unit, (8 * g + xcd) * group + hx - g * group};
}

#undef MI355_ORDER

}  // namespace mi355
