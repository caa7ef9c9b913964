// LDS layout of the small-output GEMM kernel (gemm_fp8_small): host and device
// arithmetic only, so that it can be checked on the CPU.
#pragma once

// Tile of TM = 64 * MJ rows by TN = 64 * NI columns; each of the 4 waves owns
// a 32 * MJ by 32 * NI quadrant.  K goes through S slots of 128 bytes (the
// ring's slot layout), each an LDS array of its own.  When K is done the tile's
// bf16 result is staged in the slots: rows 0 .. kStageRows-1 in slot 0, the
// others (the last 32 of 128 x 256, whose 64 KB exceed a 48 KB slot) in slot 1.
template <int MJ, int NI, int S>
struct SmallTile {
  static constexpr int TM = 64 * MJ, TN = 64 * NI;
  static constexpr int kSlotBytes = (TM + TN) * 128;
  static constexpr int kLoadsA = TM / 32, kLoadsB = TN / 32;  // per wave and slot
  static constexpr int kLoads = kLoadsA + kLoadsB;
  static constexpr int kRowBytes = 2 * TN;
  // Whole blocks of 32 rows, which one wave writes: its rows share a slot.
  static constexpr int kFit = kSlotBytes / kRowBytes / 32 * 32;
  static constexpr int kStageRows = kFit < TM ? kFit : TM;
  static constexpr int stage_slot(int r) { return r < kStageRows ? 0 : 1; }
  static constexpr int stage_offset(int r) {  // bytes, within the row's slot
    return (r - stage_slot(r) * kStageRows) * kRowBytes;
  }
  static_assert(stage_slot(TM - 1) < S && stage_offset(TM - 1) + kRowBytes <= kSlotBytes &&
                    stage_offset(kStageRows - 1) + kRowBytes <= kSlotBytes,
                "every staged row lies within its slot");
};
