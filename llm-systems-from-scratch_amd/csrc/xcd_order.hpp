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

#undef MI355_ORDER

}  // namespace mi355
