// Where the waves of gemm_split.hip read B: plain arithmetic, so that a host program can walk it too.
//
// A half round is rows 32 r + 16 k .. + 15.  Lane l reads columns TN (l % 32) .. of rows 8 (l / 32) + e, e = 0 .. 7, through a descriptor
// that begins at the tile's first column of the half round's first row and ends with B.  The range check sees the vector offset
// only.  The last round of the matrix can hold rows past K: a row is part of the vector offset there.  In every other round row e
// of a lane is a row of B with another one behind it: the row rides in the scalar offset, which costs no registers.  Lanes whose columns
// lie past N read the tile's first one; the second column of a lane may be the next row's first.
#pragma once

namespace nncv_hip {

struct SplitBRows {
  long long first;  // element that the descriptor begins at
  unsigned bytes;   // its size; none for rounds below the first and halves past K
};

constexpr SplitBRows split_b_rows(int r, int k, int n0, int N, int K) {
  const long long first = (32ll * r + 16 * k) * N + n0, left = ((long long)K * N - first) * 4;
  return {first, r < 0 || 32 * r + 16 * k >= K ? 0u : left > 0xffffffffll ? 0xffffffffu : (unsigned)left};
}

constexpr unsigned split_b_lane(int lane, int TN, int n0, int N) {
  const int col = TN * (lane & 31);
  return (8u * (unsigned)(lane >> 5) * (unsigned)N + (unsigned)(n0 + col < N ? col : 0)) * 4u;
}

// offset of row e, in the vector offset (`last`: the first round that a wave walks) or the scalar one
constexpr unsigned split_b_vector(unsigned lane_at, int e, int N, bool last) { return last ? lane_at + (unsigned)e * ((unsigned)N * 4u) : lane_at; }
constexpr unsigned split_b_scalar(int e, int N, bool last) { return last ? 0u : (unsigned)e * ((unsigned)N * 4u); }

}  // namespace nncv_hip
