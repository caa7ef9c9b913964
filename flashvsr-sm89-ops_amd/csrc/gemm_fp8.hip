// FP8 (OCP e4m3fn) GEMM on CDNA4 matrix cores, contract M:
//   C[m,n] = epilogue( sum_k A[m,k] * B[n,k] )      A [M,K], B [N,K], K-contiguous
// which is torch._scaled_mm(x8, W8.t(), ...) of FP8Linear._mm
// (flashvsr_sm89_ops/fp8_linear.py:28-30).
//
// One workgroup = 4 wavefronts (one per SIMD) computes a 256 x 256 tile; each
// wave owns a 128 x 128 quadrant = 4 x 4 v_mfma_f32_32x32x64_f8f6f4 tiles with
// fp32 accumulators (256 per lane).  The weight operand is fed as the MFMA "A"
// side and the activation as the "B" side, so each lane's accumulators hold 4
// consecutive output columns of one output row.
//
// Main loop of large outputs (K a multiple of 256, at least 512): a persistent
// kernel, one workgroup per CU, streaming K through two 64 KB LDS pair slots
// (128 bytes of K for the 256 A rows and 256 B rows) filled by buffer_load ...
// lds straight from memory, one load per MFMA; the last K steps of a tile
// already load the next tile's first pairs (details at gemm_fp8_ring; 192- and
// 128-row tiles too).  Outputs that large tiles would spread over too few CUs
// (and every K that is a multiple of 128 only) take tiles of 64 x 64 to 128 x
// 256 (gemm_fp8_small); plan_gemm picks the tile.  Other K (a multiple of 16)
// use a register-staged loop with K step 128.  Every kernel but the last sums
// K in the same order, so the tile does not change a result's bits.
//
// Epilogue: y = acc * (sa[m] * sb[n]) + bias[n], rounded to bf16, leaves
// through a per-wave LDS staging area as 16-byte row chunks:
//   FVSR_EPI_BIAS      C = y
//   FVSR_EPI_ROWMAX    C = y, plus max(C) over each row's 128-column slab
//   FVSR_EPI_GATE_ADD  C = bf16(res + bf16(gate[n] * y))
// Workgroups are renumbered so each XCD (workgroup ids are dispatched round
// robin over the 8 XCDs) walks a contiguous, M-grouped range of tiles.
#include <utility>

#include "common.h"
#include "small_tile.h"

// Buffer loads straight into LDS (buffer_load_dwordx4 ... lds): the 16 bytes
// at base + voffset + soffset of every lane land at M0 + 16 * lane.
typedef int i32x4_t __attribute__((ext_vector_type(4)));
__device__ void fvsr_buffer_load_lds(i32x4_t rsrc, __attribute__((address_space(3))) void* lds,
                                     int size, int voffset, int soffset, int offset, int aux)
    __asm("llvm.amdgcn.raw.buffer.load.lds");
// Raw buffer store of 16 bytes at base + voffset + soffset; a store whose
// voffset lies past the descriptor's byte count is dropped by the hardware.
__device__ void fvsr_buffer_store_b128(u32x4_t data, i32x4_t rsrc, int voffset, int soffset,
                                       int aux) __asm("llvm.amdgcn.raw.buffer.store.v4i32");

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
#define LDS_AS __attribute__((address_space(3)))

constexpr int BM = 256, BN = 256;
constexpr int kThreads = 256;
constexpr int kGroupM = 8;

struct EpiArgs {
  const float* sa;
  const float* sb;
  const uint16_t* bias;
  uint16_t* c;
  int64_t ldc;
  float* amax_part;
  int64_t nparts;
  const uint16_t* res;
  const uint16_t* gate;
  int sa_row, sb_col;
  int vec_params;  // sb (per column) 16-byte aligned and bias 8-byte aligned
  int res_vec;     // gate-add: N, ldc multiples of 8 and res / c / gate 16-byte aligned
  int direct;      // c 16-byte aligned, ldc % 8 == 0, (M + 256) * ldc * 2 below 2^32
};

FVSR_DEV void map_tile(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  const int q = total / 8, r = total % 8;
  const int xcd = bid % 8, loc = bid / 8;
  const int logical = xcd < r ? xcd * (q + 1) + loc : r * (q + 1) + (xcd - r) * q + loc;
  const int per_group = kGroupM * tiles_n;
  const int group = logical / per_group;
  const int first_m = group * kGroupM;
  const int gsize = min(tiles_m - first_m, kGroupM);
  const int in_group = logical % per_group;
  if (tiles_n <= 8) {
    // Narrow N (the 1536-wide projections: 6 column tiles): the column tiles
    // of one row panel run side by side, so the panel (K = 8960 for ffn2) is
    // fetched once per round (ffn2 232 -> 228 us, o 56.5 -> 55.6 us).
    tm = first_m + in_group / tiles_n;
    tn = in_group % tiles_n;
  } else {
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
  }
}

FVSR_DEV void zero_acc(v16f (&acc)[4][4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
}

template <int MJ>
FVSR_DEV void mfma_block(v16f (&acc)[4][MJ], const v8i (&fa)[MJ], const v8i (&fb)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[i], fa[j], acc[i][j], 0, 0,
                                                                   0, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Epilogue through a bf16 [256][256] LDS tile held in four 64-row pieces.
// ---------------------------------------------------------------------------
struct CTile {
  uint16_t LDS_AS* part[4];  // rows 64*i .. 64*i+63
  __device__ __forceinline__ uint16_t LDS_AS* row(int r) const { return part[r >> 6] + (r & 63) * BN; }
};

// Second half of the block-wide epilogue: the TM x TN bf16 tile staged in LDS
// (row_of(r) points at row r; its 4-column unit u sits at u ^ (r % (TN / 4)))
// leaves as 16-byte chunks, TN / 8 threads per row, with the row-max and
// gate-add epilogues applied on the way.
template <int EPI, int TM, int TN, class RowOf>
FVSR_DEV void epi_rows(const RowOf& row_of, int64_t m0, int64_t n0, int64_t M, int64_t N,
                       const EpiArgs& ep) {
  static_assert(EPI != FVSR_EPI_ROWMAX || TN % 128 == 0, "row maxima are per 128 columns");
  constexpr int kChunks = TN / 8, kMask = TN / 4 - 1;
  const int cpos = threadIdx.x % kChunks;
  const int64_t slab0 = n0 / 128;
  for (int rr = threadIdx.x / kChunks; rr < TM; rr += kThreads / kChunks) {
    const int64_t m = m0 + rr;
    const int nl = cpos * 8;
    const int64_t n = n0 + nl;
    const uint16_t LDS_AS* crow = row_of(rr);
    const u32x2_t lo = *(const u32x2_t LDS_AS*)(crow + (((nl >> 2) ^ (rr & kMask)) * 4));
    const u32x2_t hi = *(const u32x2_t LDS_AS*)(crow + ((((nl >> 2) + 1) ^ (rr & kMask)) * 4));
    u32x4_t v = {lo[0], lo[1], hi[0], hi[1]};
    float vmax = -__builtin_huge_valf();
    if (EPI == FVSR_EPI_ROWMAX) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if (n + 2 * w < N) vmax = fmaxf(vmax, bf_lo(v[w]));
        if (n + 2 * w + 1 < N) vmax = fmaxf(vmax, bf_hi(v[w]));
      }
    }
    if (m < M && n < N) {
      uint16_t* cp = ep.c + m * ep.ldc + n;
      if (EPI == FVSR_EPI_GATE_ADD) {
        const uint16_t* rp = ep.res + m * ep.ldc + n;
        if (n + 7 < N && ((((uintptr_t)cp) | (uintptr_t)rp | (uintptr_t)(ep.gate + n)) & 15) == 0) {
          const u32x4_t rv = *(const u32x4_t*)rp;
          const u32x4_t gv = *(const u32x4_t*)(ep.gate + n);
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const float t0 = round_bf16(bf_lo(gv[w]) * bf_lo(v[w]));
            const float t1 = round_bf16(bf_hi(gv[w]) * bf_hi(v[w]));
            v[w] = pack_bf16x2(bf_lo(rv[w]) + t0, bf_hi(rv[w]) + t1);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            if (n + e >= N) break;
            const float y = (e & 1) ? bf_hi(v[e >> 1]) : bf_lo(v[e >> 1]);
            const float t = round_bf16(bf2f(ep.gate[n + e]) * y);
            const float o = round_bf16(bf2f(rp[e]) + t);
            const uint32_t ob = pack_bf16x2(o, 0.0f) & 0xffffu;
            v[e >> 1] = (e & 1) ? ((v[e >> 1] & 0xffffu) | (ob << 16))
                                : ((v[e >> 1] & 0xffff0000u) | ob);
          }
        }
      }
      if (n + 7 < N && (((uintptr_t)cp) & 15) == 0) {
        *(u32x4_t*)cp = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (n + e < N) cp[e] = (uint16_t)((e & 1) ? (v[e >> 1] >> 16) : (v[e >> 1] & 0xffffu));
      }
    }
    if (EPI == FVSR_EPI_ROWMAX) {
      // 16 threads cover one 128-column slab of this row.
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, o, 64));
      const int64_t slab = slab0 + (cpos >> 4);
      if ((cpos & 15) == 0 && m < M && n < N && slab < ep.nparts)
        ep.amax_part[m * ep.nparts + slab] = vmax;
    }
  }
}

template <int EPI>
FVSR_DEV void epilogue(const v16f (&acc)[4][4], const CTile& ct, int64_t m0, int64_t n0,
                       int64_t M, int64_t N, const EpiArgs& ep, int wm, int wn, int lane) {
  // Phase 1: acc[i][j][g*4+r] is row ml = wm*128 + j*32 + (lane&31), column
  // nl = wn*128 + i*32 + g*8 + (lane>>5)*4 + r.  8-byte units are XOR-swizzled
  // with the row so 32 lanes writing 32 rows do not share banks.
  float sam[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t mg = m0 + wm * 128 + j * 32 + (lane & 31);
    sam[j] = ep.sa[ep.sa_row ? (mg < M ? mg : M - 1) : 0];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int nl = wn * 128 + i * 32 + g * 8 + (lane >> 5) * 4;
      float sbv[4], bv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t ng = n0 + nl + r < N ? n0 + nl + r : N - 1;
        sbv[r] = ep.sb[ep.sb_col ? ng : 0];
        bv[r] = ep.bias ? bf2f(ep.bias[ng]) : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int ml = wm * 128 + j * 32 + (lane & 31);
        float y[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = acc[i][j][g * 4 + r] * (sam[j] * sbv[r]) + bv[r];
        const int unit = (nl >> 2) ^ (ml & 63);
        *(u32x2_t LDS_AS*)(ct.row(ml) + unit * 4) =
            u32x2_t{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
      }
    }
  }
  __syncthreads();

  epi_rows<EPI, BM, BN>([&](int r) { return ct.row(r); }, m0, n0, M, N, ep);
}

// ---------------------------------------------------------------------------
// Main loop, K % 256 == 0 and K >= 512: persistent direct-to-LDS ring.
// ---------------------------------------------------------------------------
// Tile shapes of the ring kernel: 256 output columns (B rows) by TM = 64 * MJ
// output rows (A rows); each of the 4 waves owns TM / 2 rows (MJ blocks of
// 32) by 128 columns (4 blocks).  MJ = 4 (256 x 256) has the least LDS traffic
// per MFMA; MJ = 3 and 2 are for outputs whose rounds they fill better (C1:
// 4224 x 1536 is 102 tiles of 256 rows but 198 of 128, 22 -> 15.5 us; 7000 x
// 1536 is 168 tiles of 256 rows but 222 of 192: K = 1536 20.9 -> 18.9 us,
// K = 8960 87.7 -> 74.5 us).
template <int MJ>
struct Tile {
  static constexpr int TM = 64 * MJ;
  static constexpr int kPairBytes = (TM + BN) * 128;  // 64 KB (MJ 4) or 48 KB (MJ 2)
  static constexpr int kLoadsA = TM / 32;              // A loads per wave per pair
};

// The ring holds K in pairs of 64-byte steps: a pair slot keeps 128 bytes of
// every A row and B row, so each load covers whole 128-byte lines.
// 16-byte chunk c of row r sits at chunk position c ^ (r & 7) ^ ((r >> 3) & 1):
// any 8 consecutive rows read at one logical chunk hit 8 distinct 16-byte
// bank groups, and any 16 consecutive rows 16 distinct (row parity, chunk)
// pairs, so ds_read_b128 is conflict-free whether the LDS serves 8 or 16
// lanes per cycle.
FVSR_DEV int swz128(int r, int c) { return c ^ (r & 7) ^ ((r >> 3) & 1); }

// Per-lane byte offsets of the 16-byte pieces this lane streams for one pair:
// load t of an operand covers 8 of the wave's rows (A: TM / 4 rows per wave,
// B: 64), lane l taking row 8*t + l/8 (clamped to the matrix) and the chunk
// that lands at position l % 8.  Offsets fit 32 bits (checked on the host),
// so each load is a uniform base plus a per-lane 32-bit offset.
template <int MJ>
struct DmaOffs {
  uint32_t a[Tile<MJ>::kLoadsA], b[8];
  uint32_t ta, tb;  // L2 prefetch (long K): row starts of this lane's A row and B row
};

template <int MJ>
FVSR_DEV void dma_offsets(DmaOffs<MJ>& o, int64_t m0, int64_t n0, int64_t M, int64_t N,
                          int64_t lda, int64_t ldb, int wave, int lane) {
  const int rl = lane >> 3;
  const int c = lane & 7;
#pragma unroll
  for (int t = 0; t < Tile<MJ>::kLoadsA; ++t) {
    const int r = wave * (Tile<MJ>::TM / 4) + t * 8 + rl;
    const int64_t ga = m0 + r < M ? m0 + r : M - 1;
    o.a[t] = (uint32_t)(ga * lda + swz128(r, c) * 16);  // the swizzle is an involution in c
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int r = wave * 64 + t * 8 + rl;
    const int64_t gb = n0 + r < N ? n0 + r : N - 1;
    o.b[t] = (uint32_t)(gb * ldb + swz128(r, c) * 16);
  }
  {
    const int64_t ra = m0 + wave * (Tile<MJ>::TM / 4) + lane % (Tile<MJ>::TM / 4);
    const int64_t rb = n0 + wave * 64 + lane;
    o.ta = (uint32_t)((ra < M ? ra : M - 1) * lda);
    o.tb = (uint32_t)((rb < N ? rb : N - 1) * ldb);
  }
}

// Raw buffer descriptor over `base` (stride 0, range `bytes`; no range limit
// below 4 GB by default).
FVSR_DEV i32x4_t make_rsrc(const void* base, uint32_t bytes = 0xffffffffu) {
  const uint64_t p = (uint64_t)base;
  return i32x4_t{(int)(uint32_t)p, (int)(uint32_t)(p >> 32), (int)bytes, 0x00020000};
}

// Stream one pair (A and B bytes [k0, k0+128) of the tile's rows) into a pair
// slot.  The per-lane offsets stay in VGPRs and k0 rides in the scalar offset.
template <int MJ>
FVSR_DEV void issue_pair(uint8_t LDS_AS* slot, i32x4_t ra, i32x4_t rb, int k0,
                         const DmaOffs<MJ>& o, int wave) {
  constexpr int LA = Tile<MJ>::kLoadsA;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    if (t < LA)
      fvsr_buffer_load_lds(ra, (void LDS_AS*)(slot + (wave * LA + t) * 1024), 16,
                           __builtin_bit_cast(int, o.a[t]), k0, 0, 0);
    fvsr_buffer_load_lds(rb, (void LDS_AS*)(slot + Tile<MJ>::TM * 128 + (wave * 8 + t) * 1024),
                         16, __builtin_bit_cast(int, o.b[t]), k0, 0, 0);
  }
}

// MFMA fragment of one 64-byte step (half `hs` of a pair) of row r: lane
// half h takes logical chunks 4hs + 2h and 4hs + 2h + 1.
FVSR_DEV v8i read_frag(const uint8_t LDS_AS* base, int r, int c0) {
  const u32x4_t lo = *(const u32x4_t LDS_AS*)(base + r * 128 + (swz128(r, c0) << 4));
  const u32x4_t hi = *(const u32x4_t LDS_AS*)(base + r * 128 + (swz128(r, c0 + 1) << 4));
  return v8i{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3],
             (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
}

// All fragments of one step (the wave's A rows, then its B rows).
template <int MJ>
FVSR_DEV void read_step(const uint8_t LDS_AS* slot, int hs, int wm, int wn, int lane,
                        v8i (&fa)[MJ], v8i (&fb)[4]) {
  const int c0 = 4 * hs + 2 * (lane >> 5);
  const int ra = wm * (32 * MJ) + (lane & 31), rb = wn * 128 + (lane & 31);
#pragma unroll
  for (int j = 0; j < MJ; ++j) fa[j] = read_frag(slot, ra + 32 * j, c0);
#pragma unroll
  for (int i = 0; i < 4; ++i) fb[i] = read_frag(slot + Tile<MJ>::TM * 128, rb + 32 * i, c0);
}

// Scheduling-group masks of __builtin_amdgcn_sched_group_barrier.
constexpr int kSgMfma = 0x008, kSgVmemRead = 0x020, kSgDsRead = 0x100;

// s_waitcnt immediate (gfx9 encoding): vmcnt in bits 3:0 and 15:14, expcnt
// 6:4 (left open), lgkmcnt 11:8 (15 = left open).
constexpr int waitcnt_imm(int vm, int lgkm) {
  return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8);
}
constexpr int kWaitVm0 = waitcnt_imm(0, 15);

struct RingCtx {
  i32x4_t ra, rb;
  int wave, wm, wn, lane;
  int kmax;               // K offset of the last pair
  uint8_t LDS_AS* touch;  // 512 bytes of LDS that nothing reads
};

// Long K (ffn2, K = 8960): the operand panels are used by few tiles, so most
// pair loads miss L2, and the two LDS pair slots put them only one pair ahead
// of the MFMAs.  Each pair step also fetches, into a dummy LDS word, the
// first 4 bytes of this lane's A row and B row two pairs further on: the
// 128-byte lines land in L2 ahead of the pair's own loads.  Exactly two such
// loads follow every pair's loads, so a pair is waited for with vmcnt(2).
// (ffn2 218 -> 208 us; at K = 1536 the panels stay in L2 and the extra loads
// cost 5-8%, so they are only issued for K >= 4096.)
constexpr int kTouchAhead = 2;
template <int MJ>
FVSR_DEV void touch_pairs(const RingCtx& c, const DmaOffs<MJ>& o, int k0) {
  const int kt = min(k0 + kTouchAhead * 128, c.kmax);
  fvsr_buffer_load_lds(c.ra, (void LDS_AS*)c.touch, 4, __builtin_bit_cast(int, o.ta), kt, 0, 0);
  fvsr_buffer_load_lds(c.rb, (void LDS_AS*)(c.touch + 256), 4, __builtin_bit_cast(int, o.tb), kt,
                       0, 0);
}

// One 64-byte K step s of a tile (fragments of s in fa/fb):
//   PAIR (s odd): wait until this wave's loads of the next pair (steps s+1,
//     s+2) have landed and its reads of step s are done, then barrier: the
//     pair is in LDS for every wave and the pair slot holding steps s-1, s
//     is free; stream the pair of steps s+3, s+4 into it (`ds`, K offset k0,
//     per-lane offsets `o`: the next tile's when past the end) -- two steps
//     ahead of the reads that need it;
//   read step s+1's fragments (pair slot `rd`, half RH) into na/nb;
//   run the 4 * MJ MFMAs of step s (ZERO: start the accumulators from 0).
// The loads are spread evenly over the MFMAs (a burst of them stalls the
// wave's instruction stream) and the reads go with the first half of the
// MFMAs, leaving the second half of the step for them to land.
// Scheduling of one step: MFMA q is preceded by its share of the NL loads
// (PAIR steps) and, in the first half of the step, followed by its share of
// the ND fragment reads.
template <bool PAIR, int NM, int NL, int ND, int Q>
FVSR_DEV void sched_slot() {
  if (PAIR) __builtin_amdgcn_sched_group_barrier(kSgVmemRead, NL * (Q + 1) / NM - NL * Q / NM, 0);
  __builtin_amdgcn_sched_group_barrier(kSgMfma, 1, 0);
  if (2 * Q < NM)
    __builtin_amdgcn_sched_group_barrier(kSgDsRead, ND * (Q + 1) / (NM / 2) - ND * Q / (NM / 2),
                                         0);
}

template <bool PAIR, int NM, int NL, int ND, int... Q>
FVSR_DEV void sched_step(std::integer_sequence<int, Q...>) {
  (sched_slot<PAIR, NM, NL, ND, Q>(), ...);
}

template <int MJ, bool PAIR, int RH, bool ZERO, bool TOUCH>
FVSR_DEV void ring_step(const RingCtx& c, const DmaOffs<MJ>& o, int k0, const uint8_t LDS_AS* rd,
                        uint8_t LDS_AS* ds, v16f (&acc)[4][MJ], const v8i (&fa)[MJ],
                        const v8i (&fb)[4], v8i (&na)[MJ], v8i (&nb)[4]) {
  __builtin_amdgcn_sched_barrier(0);  // nothing (MFMAs included) moves across a step boundary
  if (PAIR) {
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(TOUCH ? 2 : 0, 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");  // no LDS access may move across the barrier
    __builtin_amdgcn_sched_barrier(0);
    issue_pair(ds, c.ra, c.rb, k0, o, c.wave);
    if (TOUCH) touch_pairs<MJ>(c, o, k0);
  }
  read_step<MJ>(rd, RH, c.wm, c.wn, c.lane, na, nb);
  if (ZERO) {
    const v16f z = {};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[i], fa[j], z, 0, 0, 0, 0,
                                                                     0, 0);
  } else {
    mfma_block<MJ>(acc, fa, fb);
  }
  sched_step<PAIR, 4 * MJ, Tile<MJ>::kLoadsA + 8, 2 * (MJ + 4)>(
      std::make_integer_sequence<int, 4 * MJ>{});
}

// Per-wave epilogue area: 32 rows x 64 columns of bf16 staging (4 KB, one
// eighth of the wave's 128 x 128 quadrant per pass; 8-byte units XOR-swizzled
// with the row so that 16 lanes writing 16 rows cover all banks), then the
// quadrant's epilogue parameters as fp32: sa of its 128 rows, sb and bias of
// its 128 columns (1.5 KB).
constexpr int kEpiStageBytes = 32 * 128;
constexpr int kEpiWaveBytes = kEpiStageBytes + 3 * 128 * 4;
FVSR_DEV int epi_off(int row, int unit) { return row * 128 + ((unit ^ (row & 15)) << 3); }

// This lane's share of the wave's parameters (rows / columns q*64 + lane of
// the wave's `wrows` rows and 128 columns; rows past them are loaded but not
// used), loaded into registers ahead of time and parked in LDS by
// put_epi_params.
struct EpiParamRegs {
  float sa[2], sb[2];
  uint32_t bias[2];
};

FVSR_DEV void fetch_epi_params(EpiParamRegs& r, const EpiArgs& e, int64_t m0, int64_t n0,
                               int64_t M, int64_t N, int wm, int wn, int wrows, int lane) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int64_t m = m0 + wm * wrows + q * 64 + lane, n = n0 + wn * 128 + q * 64 + lane;
    const int64_t mc = m < M ? m : M - 1, nc = n < N ? n : N - 1;
    r.sa[q] = e.sa[e.sa_row ? mc : 0];
    r.sb[q] = e.sb[e.sb_col ? nc : 0];
    r.bias[q] = e.bias ? (uint32_t)e.bias[nc] << 16 : 0u;
  }
}

FVSR_DEV void put_epi_params(const EpiParamRegs& r, uint8_t LDS_AS* prm, int lane) {
  float LDS_AS* sa_l = (float LDS_AS*)prm;
  float LDS_AS* sb_l = sa_l + 128;
  uint32_t LDS_AS* bi_l = (uint32_t LDS_AS*)(sb_l + 128);
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    sa_l[q * 64 + lane] = r.sa[q];
    sb_l[q * 64 + lane] = r.sb[q];
    bi_l[q * 64 + lane] = r.bias[q];
  }
}

// Phase 1 of pass (ip, j): y = acc * (sa * sb) + bias for column blocks
// 2ip, 2ip+1 and row block j, as bf16 into the staging area.
FVSR_DEV void epi_stage(const v16f (&acc)[4][4], uint16_t LDS_AS* stg,
                        const uint8_t LDS_AS* prm, int lane, int ip, int j) {
  const float LDS_AS* sa_l = (const float LDS_AS*)prm;
  const float LDS_AS* sb_l = sa_l + 128;
  const float LDS_AS* bi_l = sb_l + 128;
  const int h = lane >> 5;
  const int row = lane & 31;
  const float sam = sa_l[j * 32 + row];
#pragma unroll
  for (int ii = 0; ii < 2; ++ii)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int cl = (2 * ip + ii) * 32 + g * 8 + h * 4;
      const f32x4_t sb = *(const f32x4_t LDS_AS*)(sb_l + cl);
      const f32x4_t bw = *(const f32x4_t LDS_AS*)(bi_l + cl);
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = acc[2 * ip + ii][j][g * 4 + r] * (sam * sb[r]) + bw[r];
      *(u32x2_t LDS_AS*)((uint8_t LDS_AS*)stg + epi_off(row, ii * 8 + g * 2 + h)) =
          u32x2_t{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    }
}

// Phase 2 of pass (ip, j): 32 rows of 64 columns leave as 16-byte chunks (8
// lanes per row), with the gate-add / row-max epilogues applied on the way.
template <int EPI>
FVSR_DEV void epi_store(const uint16_t LDS_AS* stg, int64_t mw, int64_t nw, int64_t M, int64_t N,
                        const EpiArgs& e, int lane, int ip, int j, float (&vmax)[4]) {
  const int c8 = lane & 7;
  const int64_t n = nw + ip * 64 + c8 * 8;
  // Gate-add with vector rows: the pass's four residual rows and its gate
  // columns are loaded before any store (the stores may alias them when c ==
  // res, which would otherwise order each load after the previous store).
  u32x4_t rv[4], gv = {0u, 0u, 0u, 0u};
  if (EPI == FVSR_EPI_GATE_ADD && e.res_vec) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int64_t m = mw + j * 32 + s * 8 + (lane >> 3);
      const bool ok = m < M && n < N;
      rv[s] = *(const u32x4_t*)(e.res + (ok ? m : 0) * e.ldc + (ok ? n : 0));
    }
    gv = *(const u32x4_t*)(e.gate + (n < N ? n : 0));
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int row = s * 8 + (lane >> 3);
    const int64_t m = mw + j * 32 + row;
    const u32x2_t lo = *(const u32x2_t LDS_AS*)((const uint8_t LDS_AS*)stg + epi_off(row, 2 * c8));
    const u32x2_t hi =
        *(const u32x2_t LDS_AS*)((const uint8_t LDS_AS*)stg + epi_off(row, 2 * c8 + 1));
    u32x4_t v = {lo[0], lo[1], hi[0], hi[1]};
    if (EPI == FVSR_EPI_ROWMAX) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if (n + 2 * w < N) vmax[s] = fmaxf(vmax[s], bf_lo(v[w]));
        if (n + 2 * w + 1 < N) vmax[s] = fmaxf(vmax[s], bf_hi(v[w]));
      }
    }
    if (m < M && n < N) {
      uint16_t* cp = e.c + m * e.ldc + n;
      if (EPI == FVSR_EPI_GATE_ADD) {
        const uint16_t* rp = e.res + m * e.ldc + n;
        if (e.res_vec) {
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const float t0 = round_bf16(bf_lo(gv[w]) * bf_lo(v[w]));
            const float t1 = round_bf16(bf_hi(gv[w]) * bf_hi(v[w]));
            v[w] = pack_bf16x2(bf_lo(rv[s][w]) + t0, bf_hi(rv[s][w]) + t1);
          }
        } else {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            if (n + q >= N) break;
            const float y = (q & 1) ? bf_hi(v[q >> 1]) : bf_lo(v[q >> 1]);
            const float t = round_bf16(bf2f(e.gate[n + q]) * y);
            const float o = round_bf16(bf2f(rp[q]) + t);
            const uint32_t ob = pack_bf16x2(o, 0.0f) & 0xffffu;
            v[q >> 1] = (q & 1) ? ((v[q >> 1] & 0xffffu) | (ob << 16))
                                : ((v[q >> 1] & 0xffff0000u) | ob);
          }
        }
      }
      if (n + 7 < N && (((uintptr_t)cp) & 15) == 0) {
        *(u32x4_t*)cp = v;
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (n + q < N) cp[q] = (uint16_t)((q & 1) ? (v[q >> 1] >> 16) : (v[q >> 1] & 0xffffu));
      }
    }
  }
}

// Epilogue of tiles whose 256 columns all lie inside the output (bias and
// row-max epilogues).  The same eight 32 x 64 passes (column half ip, row
// block j) through the wave's staging area as epi_stage / epi_store, arranged
// so that nothing waits on LDS per value: the column scales and biases of one
// 64-column half are read into registers once (64 VGPRs), and the passes are
// software-pipelined -- pass p's staged rows are read back as 16-byte row
// chunks, pass p + 1 is converted and written over them, then pass p's chunks
// are stored (8 lanes = one 128-byte row segment).  A wave's LDS accesses
// execute in order, so the rewrite cannot overtake the reads.  Stores go
// through a buffer descriptor spanning the M output rows: stores of rows past
// M are dropped by its range check.
struct FastParams {
  f32x4_t sb[2][4], bias[2][4];
};

FVSR_DEV void fast_params(FastParams& fp, const uint8_t LDS_AS* prm, int ip, int h) {
  const float LDS_AS* sb_l = (const float LDS_AS*)prm + 128;
  const float LDS_AS* bi_l = sb_l + 128;
#pragma unroll
  for (int ii = 0; ii < 2; ++ii)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int cl = (2 * ip + ii) * 32 + g * 8 + h * 4;
      fp.sb[ii][g] = *(const f32x4_t LDS_AS*)(sb_l + cl);
      fp.bias[ii][g] = *(const f32x4_t LDS_AS*)(bi_l + cl);
    }
}

// max(m, a, b) in one instruction, a NaN passed over as fmaxf does.
FVSR_DEV float max3(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}

// Convert pass (ip, j) and write it to the staging area.  ROWMAX: vm follows
// the largest value of the lane's row (before its rounding to bf16, which is
// monotone): half an instruction per value here, where taking it from the
// stored bf16 chunks unpacked and compared each (+27 us on 108 at 8448 x 8960
// x 1536; now +1, and +4 on 206 at 16896).
template <int EPI, int MJ>
FVSR_DEV void fast_stage(const v16f (&acc)[4][MJ], const FastParams& fp, float sam,
                         uint16_t LDS_AS* stg, int ip, int j, int row, int h, float& vm) {
#pragma unroll
  for (int ii = 0; ii < 2; ++ii)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        y[r] = acc[2 * ip + ii][j][g * 4 + r] * (sam * fp.sb[ii][g][r]) + fp.bias[ii][g][r];
      if (EPI == FVSR_EPI_ROWMAX) vm = max3(max3(vm, y[0], y[1]), y[2], y[3]);
      *(u32x2_t LDS_AS*)((uint8_t LDS_AS*)stg + epi_off(row, ii * 8 + g * 2 + h)) =
          u32x2_t{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    }
}

// Read the staged pass back: row s * 8 + lane / 8, 16-byte chunk lane % 8.
FVSR_DEV void fast_read(const uint16_t LDS_AS* stg, u32x4_t (&v)[4], int lane) {
  const int c8 = lane & 7;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int r8 = s * 8 + (lane >> 3);
    const u32x2_t lo = *(const u32x2_t LDS_AS*)((const uint8_t LDS_AS*)stg + epi_off(r8, 2 * c8));
    const u32x2_t hi =
        *(const u32x2_t LDS_AS*)((const uint8_t LDS_AS*)stg + epi_off(r8, 2 * c8 + 1));
    v[s] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
  }
}

// Byte offsets into the output are unsigned 32-bit (the host admits outputs
// below 4 GiB); the sum is formed in uint32_t and handed to the intrinsic's
// int operand bit for bit.  The stores are non-temporal (cache policy `nt`):
// every workgroup writes its 128 KB output tile at about the same moment, and
// allocating those lines in L2 evicted the operand panels the next tiles read
// (qkv 111 -> 107 us, ffn0 217 -> 207 us, C1 15.5 -> 14.1 us; bit-identical).
constexpr int kStoreNT = 2;  // aux bits of the raw buffer store: nt
FVSR_DEV void fast_store(const u32x4_t (&v)[4], i32x4_t rc, uint32_t voff, int64_t ldc, int ip,
                         int j) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const uint32_t off = voff + (uint32_t)((j * 32 + s * 8) * ldc * 2 + ip * 128);
    fvsr_buffer_store_b128(v[s], rc, __builtin_bit_cast(int, off), 0, kStoreNT);
  }
}

template <int EPI, int MJ>
FVSR_DEV void epi_fast(const v16f (&acc)[4][MJ], uint16_t LDS_AS* stg, const uint8_t LDS_AS* prm,
                       int64_t mw, int64_t nw, int64_t M, const EpiArgs& e, i32x4_t rc,
                       int lane) {
  const float LDS_AS* sa_l = (const float LDS_AS*)prm;
  const int h = lane >> 5, row = lane & 31;
  float sam[MJ];
#pragma unroll
  for (int j = 0; j < MJ; ++j) sam[j] = sa_l[j * 32 + row];
  // Store offset of row lane / 8, chunk lane % 8; each pass adds its row
  // block, row group and column half (all in the offset the range check
  // covers).
  const uint32_t voff = (uint32_t)(((mw + (lane >> 3)) * e.ldc + nw + (lane & 7) * 8) * 2);
  float vm[MJ];
#pragma unroll
  for (int j = 0; j < MJ; ++j) vm[j] = -__builtin_huge_valf();
  FastParams fp;
  fast_params(fp, prm, 0, h);
  fast_stage<EPI, MJ>(acc, fp, sam[0], stg, 0, 0, row, h, vm[0]);
  // Passes p = ip * MJ + j.
#pragma unroll
  for (int p = 0; p < 2 * MJ; ++p) {
    const int ip = p / MJ, j = p % MJ;
    u32x4_t v[4];
    fast_read(stg, v, lane);
    if (p == MJ - 1) fast_params(fp, prm, 1, h);
    if (p + 1 < 2 * MJ)
      fast_stage<EPI, MJ>(acc, fp, sam[(p + 1) % MJ], stg, (p + 1) / MJ, (p + 1) % MJ, row, h,
                          vm[(p + 1) % MJ]);
    fast_store(v, rc, voff, e.ldc, ip, j);
  }
  if (EPI == FVSR_EPI_ROWMAX) {
    // The row's other values of the slab are in lane ^ 32.
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(vm[j]),
                                                       __float_as_uint(vm[j]), false, false);
      const float v = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      const int64_t m = mw + j * 32 + row;
      if (h == 0 && m < M) e.amax_part[m * e.nparts + nw / 128] = round_bf16(v);
    }
  }
}

FVSR_DEV void tile_origin(int t, int tiles_m, int tiles_n, int tile_rows, int64_t& m0,
                          int64_t& n0) {
  int tm, tn;
  map_tile(t, tiles_m, tiles_n, tm, tn);
  m0 = (int64_t)tm * tile_rows;
  n0 = (int64_t)tn * BN;
}

// Persistent kernel (K a multiple of 256, at least 512).  Workgroup b takes
// tiles b, b + G, b + 2G, ... (G = grid size, a multiple of 8, so its tiles
// stay within its XCD's M-grouped range).  The K steps of consecutive tiles
// form one stream through the two pair slots: the last two pair loads of a
// tile already fetch the next tile's pairs 0 and 1 (pair q lives in slot
// q % 2, and K/128 is even) and its last step reads the next tile's step-0
// fragments, so the epilogue overlaps the next tile's first loads.  The
// epilogue stages through a spare 32 KB that no load targets (8 KB per
// wave).  After a workgroup's last tile the same stream re-fetches that
// tile's first pairs (harmless) and the workgroup drains its loads before it
// exits.
template <int EPI, bool DIRECT, int MJ, bool TOUCH = false>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void gemm_fp8_ring(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B,
                   int64_t ldb, int64_t M, int64_t N, int64_t K, EpiArgs ep) {
  static_assert(MJ == 4 || DIRECT, "128- and 192-row tiles take the fast epilogue only");
  constexpr int TM = Tile<MJ>::TM;
  __shared__ __attribute__((aligned(1024))) uint8_t pair0[Tile<MJ>::kPairBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t pair1[Tile<MJ>::kPairBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t spare[4 * kEpiWaveBytes];
  __shared__ __attribute__((aligned(256))) uint8_t touch_lds[TOUCH ? 512 : 4];
  uint8_t LDS_AS* p0 = (uint8_t LDS_AS*)pair0;
  uint8_t LDS_AS* p1 = (uint8_t LDS_AS*)pair1;

  const int tiles_m = (int)((M + TM - 1) / TM), tiles_n = (int)((N + BN - 1) / BN);
  const int tiles = tiles_m * tiles_n;
  int t = blockIdx.x;
  if (t >= tiles) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  uint8_t LDS_AS* epa = (uint8_t LDS_AS*)spare + wave * kEpiWaveBytes;
  uint16_t LDS_AS* stg = (uint16_t LDS_AS*)epa;
  uint8_t LDS_AS* prm = epa + kEpiStageBytes;
  const int KT = (int)(K / 64);

  RingCtx c{make_rsrc(A), make_rsrc(B), wave, wm, wn, lane, (int)K - 128,
            (uint8_t LDS_AS*)touch_lds};
  int64_t m0, n0;
  tile_origin(t, tiles_m, tiles_n, TM, m0, n0);
  DmaOffs<MJ> cur;
  dma_offsets<MJ>(cur, m0, n0, M, N, lda, ldb, wave, lane);
  issue_pair<MJ>(p0, c.ra, c.rb, 0, cur, wave);
  issue_pair<MJ>(p1, c.ra, c.rb, 128, cur, wave);
  if (TOUCH) touch_pairs<MJ>(c, cur, 128);
  // The first pair (the older half of the loads in flight) has landed.
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(Tile<MJ>::kLoadsA + 8 + (TOUCH ? 2 : 0), 15));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  v16f acc[4][MJ];
  v8i fa[MJ], fb[4], na[MJ], nb[4];
  read_step<MJ>(p0, 0, wm, wn, lane, fa, fb);

  for (;;) {
    // First trip: steps 0-3 (accumulators start from 0 at step 0).
    ring_step<MJ, false, 1, true, TOUCH>(c, cur, 0, p0, p0, acc, fa, fb, na, nb);
    ring_step<MJ, true, 0, false, TOUCH>(c, cur, 2 * 128, p1, p0, acc, na, nb, fa, fb);
    ring_step<MJ, false, 1, false, TOUCH>(c, cur, 0, p1, p1, acc, fa, fb, na, nb);
    ring_step<MJ, true, 0, false, TOUCH>(c, cur, 3 * 128, p0, p1, acc, na, nb, fa, fb);
    // Steady state: steps kt .. kt+3 load pairs kt/2 + 2 and kt/2 + 3.
    for (int kt = 4; kt < KT - 4; kt += 4) {
      ring_step<MJ, false, 1, false, TOUCH>(c, cur, 0, p0, p0, acc, fa, fb, na, nb);
      ring_step<MJ, true, 0, false, TOUCH>(c, cur, (kt + 4) * 64, p1, p0, acc, na, nb, fa, fb);
      ring_step<MJ, false, 1, false, TOUCH>(c, cur, 0, p1, p1, acc, fa, fb, na, nb);
      ring_step<MJ, true, 0, false, TOUCH>(c, cur, (kt + 6) * 64, p0, p1, acc, na, nb, fa, fb);
    }
    // Last trip: steps KT-4 .. KT-1; their loads are the next tile's pairs 0
    // and 1 and the last reads are the next tile's step 0.
    const int tn = t + (int)gridDim.x;
    int64_t m1 = m0, n1 = n0;
    if (tn < tiles) tile_origin(tn, tiles_m, tiles_n, TM, m1, n1);
    DmaOffs<MJ> nxt;
    dma_offsets<MJ>(nxt, m1, n1, M, N, lda, ldb, wave, lane);
    // This tile's epilogue parameters load under the last trip's MFMAs.
    EpiParamRegs epr;
    fetch_epi_params(epr, ep, m0, n0, M, N, wm, wn, TM / 2, lane);
    ring_step<MJ, false, 1, false, TOUCH>(c, nxt, 0, p0, p0, acc, fa, fb, na, nb);
    ring_step<MJ, true, 0, false, TOUCH>(c, nxt, 0, p1, p0, acc, na, nb, fa, fb);
    ring_step<MJ, false, 1, false, TOUCH>(c, nxt, 0, p1, p1, acc, fa, fb, na, nb);
    ring_step<MJ, true, 0, false, TOUCH>(c, nxt, 128, p0, p1, acc, na, nb, fa, fb);

    // Epilogue (fa/fb now hold the next tile's step-0 fragments): passes of
    // 32 rows x 64 columns through the wave's own staging area.
    const int el = lane_here();
    const int64_t mw = m0 + wm * (TM / 2), nw = n0 + wn * 128;
    put_epi_params(epr, prm, el);
    if constexpr (DIRECT) {
      epi_fast<EPI, MJ>(acc, stg, prm, mw, nw, M, ep,
                        make_rsrc(ep.c, (uint32_t)(M * ep.ldc * 2)), el);
    } else {
      float vmax[4][4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s) vmax[j][s] = -__builtin_huge_valf();
#pragma unroll
      for (int ip = 0; ip < 2; ++ip)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          epi_stage(acc, stg, prm, el, ip, j);
          epi_store<EPI>(stg, mw, nw, M, N, ep, el, ip, j, vmax[j]);
        }
      if (EPI == FVSR_EPI_ROWMAX) {
        // 8 lanes per row cover 64 columns per pass; both ip passes = the slab.
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            float v = vmax[j][s];
#pragma unroll
            for (int o = 4; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
            const int64_t m = mw + j * 32 + s * 8 + (el >> 3);
            if ((el & 7) == 0 && m < M && nw < N) ep.amax_part[m * ep.nparts + nw / 128] = v;
          }
      }
    }
    // Stores and the next tile's loads drain before the ring moves on.
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    t = tn;
    if (t >= tiles) break;
    m0 = m1;
    n0 = n1;
    cur = nxt;
  }
}

// ---------------------------------------------------------------------------
// Small outputs, K % 128 == 0: one tile per workgroup, S-slot LDS pipeline.
// ---------------------------------------------------------------------------
// What bounds it: the LDS.  A step's time follows its LDS bytes (fragment
// reads, each operand row twice, plus the loads' writes) at 128 bytes per
// clock: 64 x 64 48 KB, 64 x 128 72 KB, 128 x 128 96 KB, 128 x 256 144 KB
// against measured 380, 620, 810 and 1240 clocks of a 128-byte K step; its
// MFMAs take 128, 256, 512 and 1024.  Three or four slots cover the memory
// latency (with two, 128 x 128 takes 47 us where four take 29, K = 8960).
// Measured (graph-replayed, 256 x 256 or 128 x 256 ring -> here, us, N = 1536):
// M = 512, K = 1536 14.0 -> 5.5; M = 2079 15.3 -> 11.3; K = 8960: M = 512 57.5
// -> 16.2, M = 1152 59.1 -> 24.4, M = 3072 58.5 -> 45.5.
// Scheduling of one step: MFMA q is preceded by its share of the NL loads and,
// in the first half of the step, followed by its share of the ND fragment reads.
template <bool LOADS, int NM, int NL, int ND, int Q>
FVSR_DEV void small_slot() {
  constexpr int NH = NM / 2;
  if (LOADS) __builtin_amdgcn_sched_group_barrier(kSgVmemRead, NL * (Q + 1) / NM - NL * Q / NM, 0);
  __builtin_amdgcn_sched_group_barrier(kSgMfma, 1, 0);
  if (Q < NH)
    __builtin_amdgcn_sched_group_barrier(kSgDsRead, ND * (Q + 1) / NH - ND * Q / NH, 0);
}
template <bool LOADS, int NM, int NL, int ND, int... Q>
FVSR_DEV void small_sched(std::integer_sequence<int, Q...>) {
  (small_slot<LOADS, NM, NL, ND, Q>(), ...);
}

template <int MJ, int NI, int S>
struct SmallCtx {
  i32x4_t ra, rb;
  uint32_t oa[SmallTile<MJ, NI, S>::kLoadsA], ob[SmallTile<MJ, NI, S>::kLoadsB];
  int wave, wm, wn, lane, KT;
};

template <int MJ, int NI, int S>
FVSR_DEV void small_issue(uint8_t LDS_AS* slot, const SmallCtx<MJ, NI, S>& c, int kt) {
  using T = SmallTile<MJ, NI, S>;
#pragma unroll
  for (int t = 0; t < T::kLoadsA; ++t)
    fvsr_buffer_load_lds(c.ra, (void LDS_AS*)(slot + (c.wave * T::kLoadsA + t) * 1024), 16,
                         __builtin_bit_cast(int, c.oa[t]), kt * 128, 0, 0);
#pragma unroll
  for (int t = 0; t < T::kLoadsB; ++t)
    fvsr_buffer_load_lds(c.rb, (void LDS_AS*)(slot + T::TM * 128 + (c.wave * T::kLoadsB + t) * 1024),
                         16, __builtin_bit_cast(int, c.ob[t]), kt * 128, 0, 0);
}

// MFMA fragments of one slot: both 64-byte halves of the wave's rows.
template <int MJ, int NI>
struct SmallFrags {
  v8i a[2][MJ], b[2][NI];
};

template <int MJ, int NI, int S>
FVSR_DEV void small_read(const uint8_t LDS_AS* slot, const SmallCtx<MJ, NI, S>& c,
                         SmallFrags<MJ, NI>& f) {
  const int ra = c.wm * (32 * MJ) + (c.lane & 31), rb = c.wn * (32 * NI) + (c.lane & 31);
#pragma unroll
  for (int hs = 0; hs < 2; ++hs) {
    const int c0 = 4 * hs + 2 * (c.lane >> 5);
#pragma unroll
    for (int j = 0; j < MJ; ++j) f.a[hs][j] = read_frag(slot, ra + 32 * j, c0);
#pragma unroll
    for (int i = 0; i < NI; ++i)
      f.b[hs][i] = read_frag(slot + SmallTile<MJ, NI, S>::TM * 128, rb + 32 * i, c0);
  }
}

// Step kt (128 bytes of K, whose fragments were read into `f` one step ago):
// wait until this wave's loads of slot kt + 1 have landed and its reads of
// slot kt are done, barrier (the same holds for every wave: slot kt + 1 is
// whole and slot kt is free), stream step kt + S into slot kt (`cur`), read
// slot kt + 1's fragments into `g` and run the step's MFMAs.  STEADY: step
// kt + S exists, so the loads need no branch and are spread over the MFMAs.
template <int MJ, int NI, int S, bool STEADY>
FVSR_DEV void small_step(uint8_t LDS_AS* cur, const uint8_t LDS_AS* nxt,
                         const SmallCtx<MJ, NI, S>& c, int kt, v16f (&acc)[NI][MJ],
                         const SmallFrags<MJ, NI>& f, SmallFrags<MJ, NI>& g) {
  using T = SmallTile<MJ, NI, S>;
  __builtin_amdgcn_sched_barrier(0);
  if (STEADY || kt + S <= c.KT)
    __builtin_amdgcn_s_waitcnt(waitcnt_imm((S - 2) * T::kLoads, 0));
  else
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  if (STEADY || kt + S < c.KT) small_issue<MJ, NI, S>(cur, c, kt + S);
  small_read<MJ, NI, S>(nxt, c, g);
#pragma unroll
  for (int hs = 0; hs < 2; ++hs)
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.b[hs][i], f.a[hs][j],
                                                                     acc[i][j], 0, 0, 0, 0, 0, 0);
  small_sched<STEADY, 2 * MJ * NI, T::kLoads, 4 * (MJ + NI)>(
      std::make_integer_sequence<int, 2 * MJ * NI>{});
}

template <int EPI, int MJ, int NI, int S, int WPC>
__global__ __launch_bounds__(kThreads, WPC) void gemm_fp8_small(
    const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
    int64_t M, int64_t N, int64_t K, EpiArgs ep) {
  using T = SmallTile<MJ, NI, S>;
  static_assert(S == 3 || S == 4, "");
  __shared__ __attribute__((aligned(1024))) uint8_t slot0[T::kSlotBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t slot1[T::kSlotBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t slot2[T::kSlotBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t slot3[S > 3 ? T::kSlotBytes : 16];
  __shared__ __attribute__((aligned(16))) float prm[T::TM + 2 * T::TN];  // sa, sb, bias
  uint8_t LDS_AS* sl[4] = {(uint8_t LDS_AS*)slot0, (uint8_t LDS_AS*)slot1, (uint8_t LDS_AS*)slot2,
                           (uint8_t LDS_AS*)slot3};
  const int tiles_m = (int)((M + T::TM - 1) / T::TM), tiles_n = (int)((N + T::TN - 1) / T::TN);
  int tm, tn;
  map_tile(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * T::TM, n0 = (int64_t)tn * T::TN;
  SmallCtx<MJ, NI, S> c;
  c.ra = make_rsrc(A);
  c.rb = make_rsrc(B);
  c.lane = threadIdx.x & 63;
  c.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  c.wm = c.wave & 1;
  c.wn = c.wave >> 1;
  c.KT = (int)(K / 128);
  const int rl = c.lane >> 3, cl = c.lane & 7;
#pragma unroll
  for (int t = 0; t < T::kLoadsA; ++t) {
    const int r = c.wave * (T::TM / 4) + t * 8 + rl;
    c.oa[t] = (uint32_t)((m0 + r < M ? m0 + r : M - 1) * lda + swz128(r, cl) * 16);
  }
#pragma unroll
  for (int t = 0; t < T::kLoadsB; ++t) {
    const int r = c.wave * (T::TN / 4) + t * 8 + rl;
    c.ob[t] = (uint32_t)((n0 + r < N ? n0 + r : N - 1) * ldb + swz128(r, cl) * 16);
  }
  // The tile's epilogue parameters are fetched ahead of the operands (one row
  // and one column per thread) and parked in LDS after the K loop.
  static_assert(T::TM <= kThreads && T::TN <= kThreads, "one parameter per thread");
  const int64_t pm = m0 + threadIdx.x < M ? m0 + threadIdx.x : M - 1;
  const int64_t pn = n0 + threadIdx.x < N ? n0 + threadIdx.x : N - 1;
  const float psa = ep.sa[ep.sa_row ? pm : 0], psb = ep.sb[ep.sb_col ? pn : 0];
  const uint16_t pbias = ep.bias ? ep.bias[pn] : (uint16_t)0;
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < c.KT) small_issue<MJ, NI, S>(sl[s], c, s);
  v16f acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  if (c.KT >= S)
    __builtin_amdgcn_s_waitcnt(waitcnt_imm((S - 1) * T::kLoads, 15));
  else
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  SmallFrags<MJ, NI> f[2];
  small_read<MJ, NI, S>(sl[0], c, f[0]);
  constexpr int U = S % 2 ? 2 * S : S;  // steps per trip: slots and fragment sets both repeat
  int kt = 0;
  for (; kt + U + S <= c.KT; kt += U) {
#pragma unroll
    for (int s = 0; s < U; ++s)
      small_step<MJ, NI, S, true>(sl[s % S], sl[(s + 1) % S], c, kt + s, acc, f[s % 2],
                                  f[(s + 1) % 2]);
  }
  for (; kt < c.KT; kt += U) {
#pragma unroll
    for (int s = 0; s < U; ++s)
      if (kt + s < c.KT)
        small_step<MJ, NI, S, false>(sl[s % S], sl[(s + 1) % S], c, kt + s, acc, f[s % 2],
                                     f[(s + 1) % 2]);
  }

  if (threadIdx.x < T::TM) prm[threadIdx.x] = psa;
  if (threadIdx.x < T::TN) {
    prm[T::TM + threadIdx.x] = psb;
    prm[T::TM + T::TN + threadIdx.x] = bf2f(pbias);
  }
  __syncthreads();  // ... and every wave is done with the slots: the tile is staged in them
  const auto row_of = [&](int r) {
    if constexpr (T::kStageRows == T::TM)
      return (uint16_t LDS_AS*)(sl[0] + T::stage_offset(r));
    else
      return (uint16_t LDS_AS*)((T::stage_slot(r) ? sl[1] : sl[0]) + T::stage_offset(r));
  };
  const float LDS_AS* pl = (const float LDS_AS*)prm;
  const int h = c.lane >> 5;
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int ml = c.wm * (32 * MJ) + j * 32 + (c.lane & 31);
    const float sam = pl[ml];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int nl = c.wn * (32 * NI) + i * 32 + g * 8 + h * 4;
        const f32x4_t sb = *(const f32x4_t LDS_AS*)(pl + T::TM + nl);
        const f32x4_t bv = *(const f32x4_t LDS_AS*)(pl + T::TM + T::TN + nl);
        float y[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = acc[i][j][g * 4 + r] * (sam * sb[r]) + bv[r];
        *(u32x2_t LDS_AS*)(row_of(ml) + (((nl >> 2) ^ (ml & (T::TN / 4 - 1))) * 4)) =
            u32x2_t{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
      }
  }
  __syncthreads();
  epi_rows<EPI, T::TM, T::TN>(row_of, m0, n0, M, N, ep);
}

// ---------------------------------------------------------------------------
// Main loop, any K % 16 == 0: register-staged, K step 128, LDS double buffer.
// ---------------------------------------------------------------------------
constexpr int BKG = 128;
constexpr int kStageG = (BM + BN) * BKG;  // 64 KB
constexpr int kChunksG = (BM * BKG / 16) / kThreads;  // 8

FVSR_DEV int swz_g(int row, int chunk) { return row * BKG + ((chunk ^ (row & 7)) << 4); }

FVSR_DEV void load_stage_g(const uint8_t* __restrict__ g, int64_t ld, int64_t row0, int64_t rows,
                           int64_t k0, int64_t K, u32x4_t (&r)[kChunksG]) {
#pragma unroll
  for (int i = 0; i < kChunksG; ++i) {
    const int id = threadIdx.x + kThreads * i;
    const int row = id >> 3, chunk = id & 7;
    int64_t gr = row0 + row;
    gr = gr < rows ? gr : rows - 1;
    const int64_t k = k0 + chunk * 16;
    r[i] = k < K ? *(const u32x4_t*)(g + gr * ld + k) : u32x4_t{0u, 0u, 0u, 0u};
  }
}

FVSR_DEV void store_stage_g(uint8_t LDS_AS* lds, const u32x4_t (&r)[kChunksG]) {
#pragma unroll
  for (int i = 0; i < kChunksG; ++i) {
    const int id = threadIdx.x + kThreads * i;
    *(u32x4_t LDS_AS*)(lds + swz_g(id >> 3, id & 7)) = r[i];
  }
}

FVSR_DEV v8i read_frag_g(const uint8_t LDS_AS* lds, int rb, int s, int lane) {
  const int row = rb + (lane & 31);
  const int c0 = s * 4 + (lane >> 5) * 2;
  const u32x4_t lo = *(const u32x4_t LDS_AS*)(lds + swz_g(row, c0));
  const u32x4_t hi = *(const u32x4_t LDS_AS*)(lds + swz_g(row, c0 + 1));
  return v8i{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3],
             (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
}

template <int EPI>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void gemm_fp8_generic(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B,
                      int64_t ldb, int64_t M, int64_t N, int64_t K, EpiArgs ep) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * kStageG];
  uint8_t LDS_AS* lds = (uint8_t LDS_AS*)smem;
  const int tiles_m = (int)((M + BM - 1) / BM), tiles_n = (int)((N + BN - 1) / BN);
  int tm, tn;
  map_tile(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;

  v16f acc[4][4];
  zero_acc(acc);
  u32x4_t ra[kChunksG], rb[kChunksG];
  const int KT = (int)((K + BKG - 1) / BKG);
  load_stage_g(A, lda, m0, M, 0, K, ra);
  load_stage_g(B, ldb, n0, N, 0, K, rb);
  store_stage_g(lds, ra);
  store_stage_g(lds + BM * BKG, rb);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    uint8_t LDS_AS* cur = lds + (kt & 1) * kStageG;
    uint8_t LDS_AS* nxt = lds + ((kt + 1) & 1) * kStageG;
    const bool more = kt + 1 < KT;
    if (more) {
      load_stage_g(A, lda, m0, M, (int64_t)(kt + 1) * BKG, K, ra);
      load_stage_g(B, ldb, n0, N, (int64_t)(kt + 1) * BKG, K, rb);
    }
#pragma unroll
    for (int s = 0; s < BKG / 64; ++s) {
      v8i fa[4], fb[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) fa[j] = read_frag_g(cur, wm * 128 + j * 32, s, lane);
#pragma unroll
      for (int i = 0; i < 4; ++i) fb[i] = read_frag_g(cur + BM * BKG, wn * 128 + i * 32, s, lane);
      mfma_block(acc, fa, fb);
    }
    if (more) {
      store_stage_g(nxt, ra);
      store_stage_g(nxt + BM * BKG, rb);
    }
    __syncthreads();
  }
  const CTile ct{{(uint16_t LDS_AS*)lds, (uint16_t LDS_AS*)(lds + 32768),
                  (uint16_t LDS_AS*)(lds + 65536), (uint16_t LDS_AS*)(lds + 98304)}};
  epilogue<EPI>(acc, ct, m0, n0, M, N, ep, wm, wn, lane);
}

// Kernels by tile: the register-staged fallback, the small-tile pipeline and
// the persistent ring (kRing: general epilogue; kRing128 / 192 / 256: fast
// epilogue).
enum class Path { kGeneric, k64x64, k64x128, k128x128, k128x256, kRing, kRing128, kRing192,
                  kRing256 };
constexpr int64_t kTouchMinK = 4096;  // L2 prefetch of the pair loads from this K on

struct GemmArgs {
  const uint8_t* a;
  int64_t lda;
  const uint8_t* b;
  int64_t ldb, M, N, K;
  EpiArgs ep;
};

template <class Kernel>
int start(Kernel kernel, unsigned grid, hipStream_t st, const GemmArgs& g) {
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, st, g.a, g.lda, g.b, g.ldb, g.M, g.N,
                     g.K, g.ep);
  return fvsr_launch_status();
}

template <int EPI>
int launch(Path path, unsigned grid, hipStream_t st, const GemmArgs& g) {
  switch (path) {
    case Path::kGeneric:
      return start(gemm_fp8_generic<EPI>, grid, st, g);
    case Path::kRing:
      return start(gemm_fp8_ring<EPI, false, 4>, grid, st, g);
    case Path::k64x64:  // row maxima need 128-column tiles
      if constexpr (EPI == FVSR_EPI_ROWMAX) break;
      else return start(gemm_fp8_small<EPI, 1, 1, 4, 2>, grid, st, g);
    case Path::k64x128:
      return start(gemm_fp8_small<EPI, 1, 2, 3, 2>, grid, st, g);
    case Path::k128x128:
      return start(gemm_fp8_small<EPI, 2, 2, 4, 1>, grid, st, g);
    case Path::k128x256:
      return start(gemm_fp8_small<EPI, 2, 4, 3, 1>, grid, st, g);
    default:
      break;
  }
  if constexpr (EPI != FVSR_EPI_GATE_ADD) {  // gate-add keeps the general epilogue
    if (path == Path::kRing128) return start(gemm_fp8_ring<EPI, true, 2>, grid, st, g);
    if (path == Path::kRing192) return start(gemm_fp8_ring<EPI, true, 3>, grid, st, g);
    if (path == Path::kRing256)
      return g.K >= kTouchMinK ? start(gemm_fp8_ring<EPI, true, 4, true>, grid, st, g)
                               : start(gemm_fp8_ring<EPI, true, 4>, grid, st, g);
  }
  return FVSR_EUNSUPPORTED;  // a plan that this epilogue has no kernel for
}

// Workgroups of the persistent kernel: one per CU, rounded down to a multiple
// of the 8 XCDs.
int64_t persistent_slots() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < 8)
    cus = 256;
  return (cus / 8) * 8;
}

struct Plan {
  Path path;
  unsigned grid;
};

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The kernel whose tiles finish first, by what its launch is measured to take:
//   start + rounds * (epilogue + K / 128 * step),  rounds = ceil(tiles / CUs),
// in ns (64-row tiles: times 1 + rounds / 800, they read the most operand bytes:
// 56 rounds, 12996 x 8960 x 1536 with gate-add, 331 us against the ring's 307).
// A CU works its tiles off one after the other (or two of the small ones side by
// side at half speed each).  `step` is the K loop's: LDS traffic at 128 bytes per
// clock (fragment reads plus the loads' writes) up to 128 x 128, MFMAs (64 clocks
// each) at 256 x 256; deep_step the same at long K, where the 256-row kernel
// prefetches into L2.  The epilogue's part is what short K turns on: the general
// epilogue of kRing takes 12 us a tile for the bias and 32 for the gate-add
// where kRing256's takes 11, and two 64 x 128 tiles to a CU hide most of theirs
// under the other's K loop.
//
// The figures are a fit to 2895 measured calls, each by every kernel that could
// take it (69 sets of K 128-8960, N 1280-8960 and epilogue, with whole and
// partial column tiles, aligned and unaligned rows; M from 100 to 16896),
// adjusted where the fit chose wrongly and checked on 2964 others: the choice is
// on average 0.5% slower than the fastest, 3.5% at the 95th percentile, 20% at
// most.  Priced by rounds * step alone it was 5.3%, 31% and 60%, and in places
// slower than 256 x 256 everywhere had been (us, now / so / 256 x 256): K =
// 1536, N = 1400: M = 12300 42.1 / 52.3 / 47.2; N = 4600: M = 4224 47.9 / 52.3 /
// 47.9; K = 4096, N = 1280 with row maxima: M = 5014 30.8 / 34.5 / 31.6 (128-row
// ring); gate-add, K = 1536, N = 1400: M = 7000 30.6 / 42.0 / 42.8.
Plan plan_gemm(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int epilogue,
               bool direct) {
  struct Option {
    Path path;
    int rows, cols, start;
    int epilogue[3];  // bias, row maxima, gate-add
    int unaligned;    // more per tile where the output's rows are not 16-byte chunks
    int step, deep_step;  // deep: K >= kTouchMinK
  };
  static constexpr Option kOptions[] = {
      {Path::kRing256, 256, 256, -3220, {10640, 11180, 0}, 0, 845, 1050},
      {Path::kRing, 256, 256, -3650, {12400, 22780, 32160}, 5360, 865, 995},
      {Path::kRing192, 192, 256, -1280, {7800, 8100, 0}, 0, 730, 770},
      {Path::kRing128, 128, 256, -600, {6280, 6600, 0}, 0, 550, 740},
      {Path::k128x256, 128, 256, -2460, {12020, 15440, 18740}, 2760, 600, 540},
      {Path::k128x128, 128, 128, 30, {6220, 7600, 9080}, 1680, 350, 390},
      {Path::k64x128, 64, 128, 2860, {1360, 1640, 2320}, 780, 225, 245},
      {Path::k64x64, 64, 64, 3100, {1000, 1500, 1640}, 680, 140, 150},
  };
  static_assert(FVSR_EPI_BIAS == 0 && FVSR_EPI_ROWMAX == 1 && FVSR_EPI_GATE_ADD == 2, "");
  // Every row offset of either operand within 32 bits; the ring takes K in
  // pairs of 128 bytes, at least two of them.
  const bool small = K % 128 == 0 && K > 0 && K < 0x7fffffffLL &&
                     (M - 1) * lda + K <= 0xffffffffLL && (N - 1) * ldb + K <= 0xffffffffLL;
  const bool ring = small && K % 256 == 0 && K >= 512;
  // The fast epilogue needs whole column tiles.
  const bool fast = ring && epilogue != FVSR_EPI_GATE_ADD && direct && N % BN == 0;
  const int64_t slots = persistent_slots();
  Plan best{Path::kGeneric, (unsigned)(cdiv(M, BM) * cdiv(N, BN))};
  int64_t best_cost = INT64_MAX;
  for (const Option& o : kOptions) {
    bool ok = small, persistent = true;
    switch (o.path) {
      case Path::kRing: ok = ring && !fast; break;
      case Path::kRing128: case Path::kRing192: case Path::kRing256: ok = fast; break;
      case Path::k64x64: ok = small && epilogue != FVSR_EPI_ROWMAX; [[fallthrough]];
      default: persistent = false;
    }
    if (!ok) continue;
    const int64_t tiles = cdiv(M, o.rows) * cdiv(N, o.cols);
    if (tiles > 0x7fffffff) continue;
    const int64_t rounds = cdiv(tiles, slots);
    const int64_t tile = o.epilogue[epilogue] + (direct ? 0 : o.unaligned) +
                         K / 128 * (K >= kTouchMinK ? o.deep_step : o.step);
    const int64_t cost = o.start + rounds * (tile + (o.rows == 64 ? tile * rounds / 800 : 0));
    if (cost >= best_cost) continue;
    best_cost = cost;
    // Persistent kernels: the fewest workgroups (a multiple of the 8 XCDs)
    // that still finish in the same number of rounds as one per CU, so no CU
    // holds a round more than another (ffn0 2310 tiles: 232 workgroups of 10
    // tiles and fewer instead of 256 of 9 or 10; qkv 240, o and ffn2 200): the
    // critical path is unchanged and the idle CUs' power goes to the others'
    // clock (ffn0 216 -> 210 us, o 40.8 -> 39.7 us).
    best = {o.path, (unsigned)(persistent && tiles > slots ? 8 * cdiv(tiles, 8 * rounds) : tiles)};
  }
  return best;
}

}  // namespace

extern "C" int64_t fvsr_gemm_amax_parts(int64_t N) { return (N + 127) / 128; }

extern "C" const char* fvsr_gemm_tile(int64_t M, int64_t N, int64_t K, int epilogue, int rows16) {
  if (M <= 0 || N <= 0 || K <= 0 || epilogue < FVSR_EPI_BIAS || epilogue > FVSR_EPI_GATE_ADD)
    return "";
  switch (plan_gemm(M, N, K, K, K, epilogue, rows16 != 0).path) {
    case Path::k64x64: return "64x64";
    case Path::k64x128: return "64x128";
    case Path::k128x128: return "128x128";
    case Path::k128x256: return "128x256";
    case Path::kRing: return "ring";
    case Path::kRing128: return "ring128";
    case Path::kRing192: return "ring192";
    case Path::kRing256: return K >= kTouchMinK ? "ring256 prefetching" : "ring256";
    default: return "generic";
  }
}

extern "C" int fvsr_fp8_gemm(const void* a, int64_t lda, const float* sa, int sa_mode,
                             const void* b, int64_t ldb, const float* sb, int sb_mode,
                             const void* bias, void* c, int64_t ldc, int64_t M, int64_t N,
                             int64_t K, int epilogue, float* amax_part, const void* res,
                             const void* gate, void* stream) {
  if (M < 0 || N < 0 || K < 0) return FVSR_EINVAL;
  if (epilogue != FVSR_EPI_BIAS && epilogue != FVSR_EPI_ROWMAX && epilogue != FVSR_EPI_GATE_ADD)
    return FVSR_EINVAL;
  if (M == 0 || N == 0) return FVSR_OK;
  if (!a || !b || !sa || !sb || !c) return FVSR_EINVAL;
  if (K % 16 || lda < K || ldb < K || lda % 16 || ldb % 16 || ldc < N) return FVSR_EUNSUPPORTED;
  if (((uintptr_t)a & 15) || ((uintptr_t)b & 15)) return FVSR_EUNSUPPORTED;
  if (epilogue == FVSR_EPI_ROWMAX && !amax_part) return FVSR_EINVAL;
  if (epilogue == FVSR_EPI_GATE_ADD && (!res || !gate)) return FVSR_EINVAL;
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  if (tiles > 0x7fffffff) return FVSR_EUNSUPPORTED;
  const int sb_col = sb_mode == FVSR_SCALE_ROW;
  const int vec_params = (!sb_col || ((uintptr_t)sb & 15) == 0) && ((uintptr_t)bias & 7) == 0;
  const int res_vec = epilogue == FVSR_EPI_GATE_ADD && N % 8 == 0 && ldc % 8 == 0 &&
                      ((((uintptr_t)res) | (uintptr_t)c | (uintptr_t)gate) & 15) == 0;
  const int direct = ((uintptr_t)c & 15) == 0 && ldc % 8 == 0 && (M + BM) * ldc * 2 <= 0xffffffffLL;
  EpiArgs ep{sa, sb, (const uint16_t*)bias, (uint16_t*)c, ldc, amax_part,
             fvsr_gemm_amax_parts(N), (const uint16_t*)res, (const uint16_t*)gate,
             sa_mode == FVSR_SCALE_ROW, sb_col, vec_params, res_vec, direct};
  hipStream_t st = (hipStream_t)stream;
  const GemmArgs g{(const uint8_t*)a, lda, (const uint8_t*)b, ldb, M, N, K, ep};
  const Plan plan = plan_gemm(M, N, K, lda, ldb, epilogue, direct != 0);
  switch (epilogue) {
    case FVSR_EPI_BIAS:
      return launch<FVSR_EPI_BIAS>(plan.path, plan.grid, st, g);
    case FVSR_EPI_ROWMAX:
      return launch<FVSR_EPI_ROWMAX>(plan.path, plan.grid, st, g);
    default:
      return launch<FVSR_EPI_GATE_ADD>(plan.path, plan.grid, st, g);
  }
}
