// Which matrices a matvec cuts into half units of row blocks (HALF at matvec_kernel), compiled for the host alone too.
#pragma once

namespace qtip {

// m / 32 = whole * full_range + left row blocks, full_range = compute units / S workgroups to each of S ranges of k, wl_per wave-loads
// to a range.  The left-over blocks, when they fill at most half a round of the full grid, are each cut into the two row halves.  The half
// units follow the whole ones in the same two-stage load pipeline, so the whole units must end on an even item.
//
// Behind whole units at 2 bits only: 10240x8192 11.1 -> 9.8 us, 12288x4096 7.15 -> 6.6 us; at 3 and 4 bits the doubled stream costs what
// the halved decode saves (12288x4096 at 3 bits 7.8 / 8.0).
// Matrices that do not fill one round: half the decode per workgroup on twice the workgroups against two readings of the stream.  At 2 bits always (4096x4096 4.8 -> 4.55 us, 4096x11008 7.9 -> 6.5).  At 3 and 4 bits from so many wave-loads
// a wave on that the saved decode outweighs a launch of more workgroups, later where the halves take more than half of the chip.
// us from cold memory, whole / halves, by wave-loads a wave (one range unless given):
//   4 bits, up to half of the chip: 2048 rows, 1 4.44/4.64, 2 5.04/5.15, 2.5 5.78/5.85, 3 6.35/6.12, 4 6.82/6.67, 7 9.55/9.12; 512 rows,
//           1 4.17/4.27, 2 4.90/4.83, 3 6.12/5.77, 4 6.61/6.20, 7 9.15/8.20
//           more of it: 4096 rows, 1 4.53/4.75, 2 5.18/5.47, 3 6.43/6.43, 3.5 6.64/6.74, 4 7.45/7.30, 5.4 8.94/8.70, 7 10.87/10.06;
//           2048 rows in two ranges, 2 5.18/5.46, 3.5 6.58/6.76, 5 8.42/8.25, 7 10.81/10.13
//   3 bits, up to half of the chip: 2048 rows, 1 4.29/4.31, 2 5.02/5.06, 2.25 5.72/5.57, 3 6.39/6.08, 4 7.43/6.65, 7 10.32/9.45
//           more of it: 4096 rows, 2.25 5.87/6.02, 2.7 6.16/6.20, 3 6.62/6.53, 4 7.53/7.16, 5.4 9.06/8.97, 7 11.09/11.38; 2048 rows in
//           two ranges, 2.7 6.18/6.19, 3.5 6.90/6.65, 5 8.80/8.78, 7 10.99/11.33; 1024 rows in four, 6 9.74/9.76
constexpr bool half_units(int bits, int left, int whole, int full_range, int S, int wl_per, int cus) {
  constexpr int waves = 16;
  if (left <= 0 || 2 * left > full_range) return false;
  if (whole > 0) return bits == 2 && (((wl_per + waves - 1) / waves) & 1) == 0;
  const bool most = 4 * left * S > cus;
  if (bits == 3) return most ? wl_per >= 3 * waves && wl_per < 6 * waves : wl_per > 2 * waves;
  return bits == 2 || wl_per >= (most ? 4 : 3) * waves;
}

// log2 of how many workgroups apart the halves of a block are (0: side by side).  Eight, in S ranges 8 / S, put them on one XCD, which the
// workgroups go round: the second reading of the block's stream hits in L2.  Behind whole units a pair that starts together is 1 % slower.
// At 2 bits so are streams up to about 5 MB (left * S * wl_per KB), which two XCDs read as fast as one: us, one XCD / side by side, 512x1024
// 3.69/3.56, 2048x1024 3.90/3.71, 4096x1024 3.97/3.87, 1024x4096 in two ranges 4.14/4.00, 1024x8192 5.49/5.42; above it 2048x11008
// 6.54/6.65, 4096x11008 6.99/7.28, 2048x14336 7.55/8.12.  At 3 and 4 bits one XCD from the lines above on: 3 bits 512x4608 5.34/5.51,
// 4096x11008 8.93/10.23; 4 bits 2048x6144 6.02/6.08, 4096x11008 8.82/10.28 (512x6144 5.79/5.67, against 6.06 in whole units).
constexpr int half_apart(int bits, int left, int whole, int S, int wl_per, int cus) {
  if (whole > 0 || (bits == 2 && left * S * wl_per < 20 * cus)) return 0;
  return S == 1 ? 3 : (S == 2 ? 2 : (S == 4 ? 1 : 0));
}

}  // namespace qtip
