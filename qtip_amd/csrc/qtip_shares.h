// Attention of one token over ranges of the cached keys whose shares the next matvec puts together: how the ranges lie, from
// the position in device memory alone, so that a recorded graph needs no other form as its context grows.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qtip_shares {

constexpr int kMaxRanges = 4;
// Ranges in use, of `ranges` that there is room for.  A range repeats the transform in front of the attention, and a second one
// costs the reader a round trip more (0.5 to 1 us); more than 40 heads and their ranges fill the chip, and two ranges gain
// nothing there.  us a token, one range / one for every 160 keys, 330, 400, 500, 700 and 900 keys: 8 layers of 4096, 32 heads
// 459/462 463/462 465/462 477/462 486/464; 4 layers of 8192, 64 heads on 8, 559/563 562/566 563/567 570/566 578/567 (at 900 keys two
// ranges: 588/586, on another card); at 8 to 300 keys the same.  Behind a narrower o the line comes early: 6 layers of 2048, 390, 500 and
// 600 keys, 32 heads of 64 255/259 256/262 263.5/263.1, 16 of 128 260/262 262/264 270/265.
// Past 1000 keys, four ranges against a launch that puts together as many as were best there (eight of 32 heads and fewer; of 64 one up to
// 2559 keys, then four), 1024, 2000 and 4000 keys: 4 layers of 4096, 32 heads 276/262 283/268 303/288, separate projections 273/262
// 281/267 302/287; 4 layers of 2048, 16 heads on 4, 203/190 204/194 217/205; 2 layers of 8192, 64 heads on 8, 297/298 310/306 325/323,
// 64 on 64 (separate) 331/328 344/338 359/356.
__host__ __device__ constexpr int active(int nkeys, int ranges, int heads) {
  const int a = nkeys < (heads > 40 ? 640 : 380) ? 1 : nkeys / 160;
  return a < ranges ? a : ranges;
}
__host__ __device__ constexpr int keys_of(int nkeys, int active) {
  return active == 1 ? nkeys : (active == 2 ? (nkeys + 1) / 2 : (active == 3 ? (nkeys + 2) / 3 : (nkeys + 3) / 4));
}
// a range's share: D unnormalised outputs, the largest score, the sum of exponentials; 16-byte aligned
__host__ __device__ constexpr int floats(int head_dim) { return head_dim + 4; }

struct ShareArgs {
  const float* shares;  // [heads][ranges][floats(head_dim)]
  const long* pos;      // the token's position
  int ranges, log_dim, max_len;
};

}  // namespace qtip_shares
