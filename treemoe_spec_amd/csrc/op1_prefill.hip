// op1 expert GEMMs for many rows per expert (prefill / batched trees) on gfx950.
//
// When an expert receives tens to thousands of rows the weight-streaming
// kernels (which re-read an expert's weights once per 64-row tile) are the
// wrong shape.  These kernels tile both operands:
//
//   workgroup = NW waves (2 row halves x NW / 2 column groups) = BM sorted rows
//   x BN weight rows; each wave owns BM/2 x 32 NJ outputs = (BM/64) x NJ
//   v_mfma_f32_32x32x16 tiles (on gfx950 the 32x32 form sustains ~2.2
//   PFLOP/s, the 16x16x32 form ~1.3).
//   Operands go from global memory straight into LDS (16-byte buffer loads
//   with the LDS flag: lane i of a load lands at byte 16 i of its 1 KB block,
//   no registers involved), several steps deep.  LDS rows hold one K step of
//   64 (128 bytes: a whole cache line per row and load) with the 16-byte chunks
//   XOR-swizzled (swz), which the loads arrange by choosing each lane's source
//   chunk; 16 consecutive rows read at one logical chunk then hit 16 distinct
//   4-bank groups.
//
// Three tile configurations:
//   Tile256  256 rows x 256 weight rows on 4 waves, one per SIMD, hand-
//            pipelined (PipeLoop): many rows per expert and enough jobs (use_tile256);
//   Tile128  128 x 256 on 8 waves, three 48 KB stages;
//   TileDec  64 x 128 on 4 waves, three 24 KB stages, so two workgroups share
//            a CU: gate/up when the tile list leaves at most 16 rows per entry,
//            down where the other tile has too few jobs for the chip.
// A tile whose M-tile holds fewer than BM real rows runs the MFMAs of the
// 64-row parts that hold them only.
//
// Gate/up: B = BN / 2 rows of w1 and the same rows of w3, so each wave holds
// the gate and up sums of the same outputs and applies SwiGLU in registers; h
// is written row-major [sorted row, I] through an LDS-staged, coalesced store.
// Down: B = BN rows of w2 over one K segment; the gate weight multiplies the
// fp32 sums before the store of the partial y[segment].
//
// M-tiles are BM consecutive rows of one expert in the compact expert-major
// order (expert_offsets).  Launch order: workgroups are dealt to the 8 XCDs
// in turn, and each XCD owns one eighth of the column jobs for every M-tile,
// walked expert by expert, M fastest, when the experts average two M-tiles
// or more, else in super-blocks of 8 M-tiles x 4 columns (expert_job; the
// self-routed decode gate/up always takes the super-blocks, job_of).
#pragma clang fp contract(off)

#include <algorithm>
#include <cmath>

#include "op1_bucket.h"
#include "tm_common.h"

namespace {

constexpr uint32_t kOOR = 0x80000000u;   // out-of-range buffer offset: loads 0

// Tile configuration: BM sorted rows per M-tile, K steps of BK, NS stages,
// BN weight rows per workgroup, NTH threads (NTH / 64 waves as 2 row halves x
// NTH / 128 column groups; a wave owns BM/2 x 32 NJ outputs).
template <int BM, int BK, int NS, int BN = 256, int NTH = 512>
struct Tile {
  static constexpr int PBM = BM;
  static constexpr int PBK = BK;
  static constexpr int NSTAGE = NS;
  static constexpr int PBN = BN;                  // weight rows per workgroup
  static constexpr int NT = NTH;                  // threads per workgroup
  static constexpr int NW = NTH / 64;             // waves
  static constexpr int NJ = BN / (16 * NW);       // 32-column accumulator tiles per wave
  static constexpr int PROW = PBK * 2;            // LDS row, bytes (PROW / 16 swizzled chunks)
  static constexpr int CPR = PROW / 16;           // 16-byte chunks per row
  static constexpr int RPB = 256 / PROW;          // rows per 256 B (one pass over the 64 banks)
  static constexpr int RPK = 1024 / PROW;         // rows per 1 KB load block
  static constexpr int ABYTES = PBM * PROW;       // A tile of one step
  static constexpr int BBYTES = PBN * PROW;       // B tile of one step
  static constexpr int STAGE = ABYTES + BBYTES;   // one stage in LDS
  static constexpr int ALD = ABYTES / (NT * 16);  // 16-byte loads per thread per step: A
  static constexpr int BLD = BBYTES / (NT * 16);  //                                   B
  static constexpr int LDS_PER_STEP = ALD + BLD;
  static constexpr int MT = PBM / 64;             // 32-row accumulator tiles per wave
  // one wave per SIMD; A and B tiles in a ring of NS buffers (k_loop_pipe)
  static constexpr bool PIPE = NJ == 4;
  static constexpr int BUF = PIPE ? ABYTES : STAGE;  // one LDS buffer
  // h staging: rows of PBN / 2 columns, padded by 16 bytes; rows per stage:
  // the whole tile in one stage when it fits
  static constexpr int HSTRIDE = PBN + 16;
  static constexpr int HROWS = PBM * HSTRIDE <= BUF ? PBM : PBM / 4;
  static_assert(ALD >= 1 && BLD >= 1 && BLD % 2 == 0 && CPR >= 4, "tile shape");
  static_assert((NJ == 2 || NJ == 4) && (NW == 4 || NW == 8), "wave layout");
  static_assert(NS == (PIPE ? 5 : 3), "buffer rotation");
  static_assert(HROWS * HSTRIDE <= BUF && (PBM + HROWS - 1) / HROWS <= NS, "h staging");
  static_assert(NS * BUF <= 160 * 1024, "LDS");
  static_assert(!PIPE || (PBK == 64 && ABYTES == BBYTES), "k_loop_pipe's buffers");
};
using Tile128 = Tile<128, 64, 3>;
// Many rows per expert: 256 x 256 on four waves of 128 x 128 outputs.
using Tile256 = Tile<256, 64, 5, 256, 256>;
// Few rows per expert: 64-row M-tiles against 128 weight rows with 4 waves,
// 72 KB of LDS, so two workgroups share a CU.  Same per-output K order as
// Tile128, so the same bits.
using TileDec = Tile<64, 64, 3, 128, 256>;

typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pbuf(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           0x00020000);
}

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// 32x32x16 MFMA with the weights as the first operand: x holds 32 sorted rows
// and w 32 weight rows (lane l: row l % 32, k 8 (l / 32) .. +7), and lane l gets
// C[row l % 32][column 8 (v / 4) + 4 (l / 32) + v % 4] in accumulator value v,
// so its values 4 q .. 4 q + 3 are four consecutive output columns of one row
// (acc_col): the epilogues pack and store them as one vector.  (DT:
// TM_DTYPE_BF16 or TM_DTYPE_F16 operands, same lane layout.)
template <int DT>
__device__ __forceinline__ f32x16_t pmfma(u32x4_t x, u32x4_t w, f32x16_t c) {
  if constexpr (DT == TM_DTYPE_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, w),
                                                  __builtin_bit_cast(f16x8_t, x), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, w),
                                                   __builtin_bit_cast(bf16x8_t, x), c, 0, 0, 0);
}

// First of the four output columns that accumulator values 4 q .. 4 q + 3 hold.
__device__ __forceinline__ int acc_col(int q, int lane) { return 8 * q + 4 * (lane >> 5); }

// Two fp32 values to the 16-bit type, round to nearest even, packed in order
// (bf16: v_cvt_pk_bf16_f32).  fp16 converts one value at a time, as Half16 does:
// the product that ends a value then fuses with its conversion (v_fma_mixlo_f16,
// v_fma_mixhi_f16) and is rounded once, where a conversion of the pair rounds
// the fp32 product again.
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
template <int DT>
__device__ __forceinline__ uint32_t pack16(float lo, float hi) {
  if constexpr (DT == TM_DTYPE_F16) {
    return (uint32_t)tm_f32_to_f16(lo) | ((uint32_t)tm_f32_to_f16(hi) << 16);
  } else {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  }
}

// Byte offset in a swizzled tile of logical chunk c (16 B) of row r: chunk c
// is stored at c ^ ((r / RPB) % CPR), so 16 consecutive rows read at one
// logical chunk cover 16 distinct 4-bank groups.
template <class C>
__device__ __forceinline__ int swz(int r, int c) {
  return r * C::PROW + ((c ^ ((r / C::RPB) & (C::CPR - 1))) << 4);
}

constexpr int kCUs = 256;
constexpr int kXcds = 8;  // workgroup i runs on XCD i % 8
constexpr int SBM = 8;    // super-block: M-tile slots (consecutive: mostly one expert) ..
constexpr int SBN = 4;    // .. x column jobs, M fastest

// Job of launch index L over the layer's real M-tiles (n_mt of them) in the
// super-block order (the self-routed decode gate/up, whose waves compute it
// in registers, and expert_job when most experts take one M-tile): M-tile
// and column job, or false for a launch index past the real jobs (those are
// the launch's last indices, so the real jobs all start in the first round).
// XCD x = L % 8 owns the column jobs [x * cpx, (x + 1) * cpx) for every
// M-tile, so each weight block is read through one XCD's L2 only, and walks
// them in strips of SBN columns, each strip in groups of SBM M-tiles, M
// fastest (the last strip and group may be narrower): the ~32 workgroups
// resident on the XCD share each A tile across SBN columns and each weight
// block across the M-tiles of one expert.
__device__ __forceinline__ bool job_of(int L, int n_mt, int ncol, int* mt, int* col) {
  const int x = L % kXcds, l = L / kXcds;
  const int cpx = (ncol + kXcds - 1) / kXcds;
  if (l >= n_mt * cpx) return false;
  const int s = l / (n_mt * SBN);                // column strip
  const int ws = min(SBN, cpx - s * SBN);         // its width
  const int j = l - s * n_mt * SBN;
  const int g = j / (SBM * ws);                  // M-tile group within the strip
  const int mg = min(SBM, n_mt - g * SBM);       // its size
  const int jj = j - g * SBM * ws;
  *mt = g * SBM + jj % mg;
  *col = x * cpx + s * SBN + jj / mg;
  return *col < ncol;
}

// One workgroup's job: rows p0 .. p0 + rows of expert e against column job
// col; single: the expert's only M-tile.
struct Job {
  int e, p0, rows, col;
  bool single;
};

// Job of launch index L for the prefill GEMMs, or false for a launch index
// past the real jobs (those are the launch's last indices).  Lane e of every
// wave holds expert e's row count (no LDS, no barrier); wave scans of
// ceil(rows_e / BM) and ceil(rows_e / 64) give the M-tiles and the 64-row tiles
// before each expert, so the owner of M-tile m is found with a ballot instead
// of a loop of dependent loads over the experts.  When the active experts
// average two M-tiles or more, XCD x = L % 8 walks its column jobs
// [x * cpx, (x + 1) * cpx) of every M-tile one expert at a time, the
// expert's M-tiles fastest, then its columns: the ~32 workgroups resident on
// an XCD then run the jobs of one expert or of a few adjacent ones, so all
// the M-tiles that read a weight block run together and share it in that
// L2, and each A tile is shared by the expert's nearby columns.  With fewer
// M-tiles it takes the super-block order (job_of), whose resident jobs read
// several experts' weights at once.  (Same box, bit-identical, expert order
// against super-blocks: config 5 1787 against 1801 us, T = 2048 uniform 1719
// against 1771, T = 4096 3111 against 3202, T = 1536 1374 against 1411; but
// T = 128 535 against 501, T = 256 542 against 513, T = 512 720 against 705,
// where most experts take one M-tile.)
// An expert whose first entry in the 64-row tile list is masked (expert -1,
// as Routing.exclude_experts leaves it) has no jobs, like the weight-streaming
// kernels skip its tiles.
template <class C>
__device__ __forceinline__ bool expert_job(int L, const int32_t* __restrict__ offsets,
                                           const int32_t* __restrict__ tiles, int max_tiles,
                                           int E, int mt_max, int ncol, Job* job) {
  const int x = L % kXcds, l = L / kXcds;
  const int cpx = (ncol + kXcds - 1) / kXcds;
  const int lane = threadIdx.x & 63;
  int off = 0, cnt = 0;
  if (lane < E) {
    off = offsets[lane];
    cnt = offsets[lane + 1] - off;
  }
  const int n = (cnt + C::PBM - 1) / C::PBM;
  const int n64 = (cnt + TM_GEMM_TILE_M - 1) / TM_GEMM_TILE_M;
  int incl = n, incl64 = n64;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(incl, o), t64 = __shfl_up(incl64, o);
    if (lane >= o) {
      incl += t;
      incl64 += t64;
    }
  }
  const int first = incl - n;  // M-tiles of the experts before this lane's
  const int total = __shfl(incl, 63);
  const int active = __popcll(__ballot(n > 0));
  int m = -1, c = 0;
  if (total < 2 * active) {
    // Mostly one M-tile per expert: the super-block order, whose jobs
    // resident together read different experts' weights.
    int jm = -1, jc = 0;
    const bool ok = job_of(L, min(total, mt_max), ncol, &jm, &jc);
    m = ok ? jm : -1;
    c = jc;
  } else {
    // the expert (lane) whose column range of this XCD holds l
    const bool mine = n > 0 && l >= first * cpx && l < incl * cpx;
    const unsigned long long owner = __ballot(mine);
    if (owner != 0ull) {
      const int src = __ffsll((long long)owner) - 1;
      const int j = l - first * cpx;
      m = __shfl(first + (n > 0 ? j % n : 0), src);
      c = __shfl(x * cpx + (n > 0 ? j / n : 0), src);
    }
  }
  m = __builtin_amdgcn_readfirstlane(m);
  job->col = __builtin_amdgcn_readfirstlane(c);
  if (m < 0 || m >= mt_max || job->col >= ncol) return false;
  const unsigned long long own = __ballot(m >= first && m < incl);
  if (own == 0ull) return false;
  const int e = __ffsll((long long)own) - 1;
  const int tile64 = __builtin_amdgcn_readlane(incl64 - n64, e);
  if (tile64 >= max_tiles || tiles[4 * tile64] != e) return false;
  const int m0 = (m - __builtin_amdgcn_readlane(first, e)) * C::PBM;
  job->e = e;
  job->p0 = __builtin_amdgcn_readlane(off, e) + m0;
  job->rows = min(C::PBM, __builtin_amdgcn_readlane(cnt, e) - m0);
  job->single = __builtin_amdgcn_readlane(n, e) == 1;
  return true;
}

// Launch size: 8 XCDs x (M-tile bound) x the columns of one XCD's range.
int64_t launch_jobs(int64_t mt_max, int64_t ncol) {
  return kXcds * mt_max * ((ncol + kXcds - 1) / kXcds);
}

// Upper bound of the M-tiles over E experts holding `slots` rows.
template <class C>
int64_t mtile_bound(int64_t slots, int64_t E) {
  return (slots + C::PBM - 1) / C::PBM + E;
}

// Global -> LDS: load i of a thread moves one 16-byte chunk.  Load i of wave
// w fills the 1 KB block 8 i + w of its tile (RPK rows); lane l writes byte
// 16 l of the block, i.e. row RPK (8 i + w) + l / CPR at stored chunk
// l % CPR, so it fetches the logical chunk that the swizzle stores there.
template <class C>
struct DmaLoad {
  const void* pa;         // A
  const void *pb0, *pb1;  // B: the first and the second half of its loads
  uint32_t na, nb;        // bytes behind pa, and behind each of pb0 and pb1
  uint32_t aoff[C::ALD];  // byte offset of the chunk at k = 0, or kOOR
  uint32_t boff[C::BLD];
};

// Row of load i for this thread, and the logical chunk it fetches.
template <class C>
__device__ __forceinline__ int dma_row(int i) {
  return C::RPK * (C::NW * i + (threadIdx.x >> 6)) + ((threadIdx.x & 63) / C::CPR);
}
template <class C>
__device__ __forceinline__ int dma_chunk(int row) {
  return (threadIdx.x & (C::CPR - 1)) ^ ((row / C::RPB) & (C::CPR - 1));
}

// One 16-byte buffer load per lane into LDS at `lds` + 16 lane (lds
// wave-uniform), from byte voffset (per lane) + soffset (wave-uniform).  A
// plain function: the host compilation pass rejects the builtin inside some
// instantiations of the templates below.
__device__ __forceinline__ void lds_load16(__amdgpu_buffer_rsrc_t r, uint8_t* lds,
                                           uint32_t voffset, uint32_t soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, voffset, soffset, 0, 0);
}
// The same with the non-temporal cache policy (weights streamed through).
__device__ __forceinline__ void lds_load16_nt(__amdgpu_buffer_rsrc_t r, uint8_t* lds,
                                              uint32_t voffset, uint32_t soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, voffset, soffset, 0, 2);
}

// Load i of step `kstep` (K bytes PROW kstep ..) of the A tile into `at` or of
// the B tile into `bt`.  The K position is the load's scalar offset, so a step costs no
// vector arithmetic; past the end of K the buffer has no bytes, so the load
// is out of range and stores zeros without memory traffic.  Every step issues
// all LDS_PER_STEP loads, so the wait counts below stay exact.
template <class C>
__device__ __forceinline__ void dma_a(const DmaLoad<C>& d, uint8_t* at, int i, int kstep, int nk) {
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // LDS base: wave-uniform
  lds_load16(pbuf(d.pa, kstep < nk ? d.na : 0u), at + (C::NW * i + w) * 1024, d.aoff[i],
             (uint32_t)kstep * (uint32_t)C::PROW);
}
template <class C, bool NTB>
__device__ __forceinline__ void dma_b(const DmaLoad<C>& d, uint8_t* bt, int i, int kstep, int nk) {
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const __amdgpu_buffer_rsrc_t r = pbuf(i < C::BLD / 2 ? d.pb0 : d.pb1, kstep < nk ? d.nb : 0u);
  uint8_t* const lds = bt + (C::NW * i + w) * 1024;
  if constexpr (NTB)
    lds_load16_nt(r, lds, d.boff[i], (uint32_t)kstep * (uint32_t)C::PROW);
  else
    lds_load16(r, lds, d.boff[i], (uint32_t)kstep * (uint32_t)C::PROW);
}
template <class C, bool NTB>
__device__ __forceinline__ void dma_step(const DmaLoad<C>& d, uint8_t* st, int kstep, int nk) {
#pragma unroll
  for (int i = 0; i < C::ALD; ++i) dma_a<C>(d, st, i, kstep, nk);
#pragma unroll
  for (int i = 0; i < C::BLD; ++i) dma_b<C, NTB>(d, st + C::ABYTES, i, kstep, nk);
}

// Wait until at most n of this thread's vector-memory operations are
// outstanding (s_waitcnt vmcnt(n); the other counters are left alone).
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Fragment of 32 rows starting at `row`, k-step s (16 columns): lane l reads
// row l % 32, logical chunk 2 s + l / 32.
template <class C>
__device__ __forceinline__ u32x4_t frag(const uint8_t* tile, int row, int s, int lane) {
  return *reinterpret_cast<const u32x4_t*>(tile + swz<C>(row + (lane & 31), 2 * s + (lane >> 5)));
}

// acc[i][j] += A[32 M wm + 32 i, :] B[brow[j], :]^T over one staged step.  M
// (<= MT) is the accumulator tiles per wave along the rows: M = MT covers the
// whole M-tile, a smaller M its first 64 M rows (a tile with at most 64 M real
// rows, whose other rows are zeros).
template <class C, int M, int DT>
__device__ __forceinline__ void compute_step(const uint8_t* st, const int (&brow)[C::NJ],
                                             f32x16_t (&acc)[M][C::NJ]) {
  const int lane = threadIdx.x & 63;
  const int wm = (threadIdx.x >> 6) & 1;
  constexpr int S = C::PBK / 16;
  // The fragments of k-step s + 1 are read between the MFMAs of k-step s (one
  // MFMA, then one LDS read, while reads remain), so each MFMA waits only for
  // reads issued a k-step earlier.
  u32x4_t a[2][M], b[2][2];
#pragma unroll
  for (int i = 0; i < M; ++i) a[0][i] = frag<C>(st, 32 * M * wm + 32 * i, 0, lane);
#pragma unroll
  for (int j = 0; j < 2; ++j) b[0][j] = frag<C>(st + C::ABYTES, brow[j], 0, lane);
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int cur = s & 1, nxt = cur ^ 1;
    __builtin_amdgcn_sched_barrier(0);
    if (s + 1 < S) {
#pragma unroll
      for (int i = 0; i < M; ++i) a[nxt][i] = frag<C>(st, 32 * M * wm + 32 * i, s + 1, lane);
#pragma unroll
      for (int j = 0; j < 2; ++j) b[nxt][j] = frag<C>(st + C::ABYTES, brow[j], s + 1, lane);
    }
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = pmfma<DT>(a[cur][i], b[cur][j], acc[i][j]);
    if (s + 1 < S) {
#pragma unroll
      for (int k = 0; k < M + 2 && k < 2 * M; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
      }
      if constexpr (2 * M > M + 2)
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * M - (M + 2), 0);
    }
  }
  // keep the next step's wait, barrier and loads after these MFMAs
  __builtin_amdgcn_sched_barrier(0);
}

// The LDS buffers: distinct arrays used in a fixed rotation, so the compiler
// can tell the one being read from the ones being loaded (s3 and s4 are used by
// Tile256 only).
struct Stages {
  uint8_t* s0;
  uint8_t* s1;
  uint8_t* s2;
  uint8_t* s3;
  uint8_t* s4;
};
#define TM_STAGES(C)                                                                   \
  __shared__ __attribute__((aligned(16))) uint8_t s0[C::BUF];                          \
  __shared__ __attribute__((aligned(16))) uint8_t s1[C::BUF];                          \
  __shared__ __attribute__((aligned(16))) uint8_t s2[C::BUF];                          \
  __shared__ __attribute__((aligned(16))) uint8_t s3[C::NSTAGE > 3 ? C::BUF : 16];     \
  __shared__ __attribute__((aligned(16))) uint8_t s4[C::NSTAGE > 4 ? C::BUF : 16];     \
  const Stages sb{s0, s1, s2, s3, s4}

// A workgroup barrier (after this wave's LDS operations) that the compiler
// schedules nothing across.
__device__ __forceinline__ void step_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  tm_lds_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

// Byte offset of the fragment chunk of k-step s (see frag) within the 32 LDS
// rows it starts at: the swizzle repeats every 32 rows, so fragments 32 rows
// apart are a constant apart.
template <class C>
__device__ __forceinline__ int frag_off(int lane, int s) {
  static_assert((32 / C::RPB) % C::CPR == 0, "swizzle period");
  return swz<C>(lane & 31, 2 * s + (lane >> 5));
}

// K loop of the 256-row tile: four waves, one per SIMD, each owning 128 x 128
// outputs (M x 4 accumulator tiles, 16 M registers each, in AGPRs).  With one
// wave per SIMD nothing else hides a wait, so the loop is pipelined by hand:
// while the MFMAs of one 16-deep k-step run, the fragments of the next one
// are read into a second register set (the reads in the first groups of
// MFMAs, so that the last one has arrived when they end) and operand loads go
// out between the groups.
// A step is four k-steps with one barrier B(k) before the last.  The five
// buffers hold single operand tiles in the order B0 A0 B1 A1 ..: step k reads
// buffers 2k and 2k + 1 (mod 5), step k + 1 the next two, and the fifth is
// being loaded.
//   s = 0, 1: MFMAs (k, s), reads (k, s + 1), B loads of step k + 2
//   s = 2:    MFMAs (k, 2), reads (k, 3)
//   B(k):     this wave's loads of step k + 1 done (vmcnt), its reads of step
//             k done (lgkmcnt), all waves
//   s = 3:    MFMAs (k, 3), reads (k + 1, 0), A loads of step k + 2
// After B(k) every wave's loads of step k + 1 have landed, and both buffers of
// step k are free: that of its B tile takes the A tile of step k + 2, that of its
// A tile the B tile of step k + 3.  So the weights, most of which come from HBM,
// have more than a step and a half to arrive and the rows, which other
// workgroups of the XCD share, most of one.  A wave reads 256 fragment rows
// per 128 x 128 outputs where two waves of 128 x 64 read 384: a third less LDS
// traffic.
// What bounds it: operands and the clock.  Under this loop the clock falls from 2.4
// to 1.8-1.95 GHz (GRBM_GUI_ACTIVE over the dispatches' time, T = 2048 skewed), the
// matrix cores are busy 53-58 % of its cycles and the waves wait 55-62 % of theirs,
// so the operand bytes moved (hence one wave per SIMD with large tiles and whole
// 128-byte lines per load) count as much as the stalls.  H = 4096, I = 14336,
// E = 8, same box, against the 8-wave loop of two 4-wave halves half a step apart
// with K steps of 32 (down: 128-row tiles, steps of 64) that it replaces, gate/up
// with SwiGLU by a reciprocal (its division adds 1.5 %, T = 6011 2258 -> 2293 us on
// a slower box): T = 6011 gate/up 2560 -> 2200 us, down 1437 -> 1188; T = 2048
// skewed 995 -> 858 and 573 -> 481; T = 517, on 128-row tiles before, 430 -> 355 and
// 262 -> 166.  The same loop with K steps of 32 in four stages took 2410 and 1340 us
// at T = 6011.
template <class C, int M, int DT, bool NTB>
struct PipeLoop {
  static constexpr int NJ = C::NJ, AL = C::ALD, BL = C::BLD;
  static constexpr int RG = M > 1 ? M - 1 : 1;         // MFMA groups (of NJ) that carry reads
  static constexpr int RPG = (M + NJ + RG - 1) / RG;   // reads per such group
  static constexpr int APG = (AL + M - 1) / M;         // A loads per group of s = 3
  static constexpr int BPG = (BL / 2 + M - 1) / M;     // B loads per group of s = 0, 1

  uint8_t* buf[5];
  int fo[4];                // frag_off of the four k-steps
  int arow, brow[C::NJ];    // LDS byte offsets of the wave's first row fragment, its columns
  u32x4_t a[2][M], b[2][C::NJ];

  // fragment q of k-step s: the NJ weight fragments, then the M row fragments
  __device__ __forceinline__ void read(int set, const uint8_t* at, const uint8_t* bt, int s,
                                       int q) {
    if (q < NJ)
      b[set][q] = *reinterpret_cast<const u32x4_t*>(bt + brow[q] + fo[s]);
    else
      a[set][q - NJ] =
          *reinterpret_cast<const u32x4_t*>(at + arow + (q - NJ) * 32 * C::PROW + fo[s]);
  }

  // Step k, whose tiles are in buffers U = 2k and U + 1 (mod 5).
  template <int U>
  __device__ __forceinline__ void step(const DmaLoad<C>& d, int k, int nk,
                                       f32x16_t (&acc)[M][C::NJ]) {
    uint8_t* const bt = buf[U % 5];
    uint8_t* const at = buf[(U + 1) % 5];
    uint8_t* const bn = buf[(U + 2) % 5];
    uint8_t* const an = buf[(U + 3) % 5];
    uint8_t* const bnn = buf[(U + 4) % 5];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int g = 0; g < M; ++g) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = g * RPG; q < (g + 1) * RPG && q < M + NJ; ++q) {
          if (s < 3)
            read((s + 1) & 1, at, bt, s + 1, q);
          else
            read(0, an, bn, 0, q);
        }
        if (s < 2) {
#pragma unroll
          for (int i = g * BPG; i < (g + 1) * BPG && i < BL / 2; ++i)
            dma_b<C, NTB>(d, bnn, s * (BL / 2) + i, k + 2, nk);
        } else if (s == 3) {
#pragma unroll
          for (int i = g * APG; i < (g + 1) * APG && i < AL; ++i) dma_a<C>(d, bt, i, k + 2, nk);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[g][j] = pmfma<DT>(a[s & 1][g], b[s & 1][j], acc[g][j]);
      }
      if (s == 2) {
        wait_vm<BL>();
        step_barrier();
      }
    }
  }

  __device__ __forceinline__ void run(const Stages& sb, const DmaLoad<C>& d, int nk,
                                      const int (&first_row)[C::NJ], f32x16_t (&acc)[M][C::NJ]) {
    const int lane = threadIdx.x & 63;
    const int wm = (threadIdx.x >> 6) & 1;
    buf[0] = sb.s0;
    buf[1] = sb.s1;
    buf[2] = sb.s2;
    buf[3] = sb.s3;
    buf[4] = sb.s4;
    arow = 32 * M * wm * C::PROW;
#pragma unroll
    for (int j = 0; j < NJ; ++j) brow[j] = first_row[j] * C::PROW;
#pragma unroll
    for (int s = 0; s < 4; ++s) fo[s] = frag_off<C>(lane, s);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int i = 0; i < BL; ++i) dma_b<C, NTB>(d, buf[2 * u], i, u, nk);
#pragma unroll
      for (int i = 0; i < AL; ++i) dma_a<C>(d, buf[2 * u + 1], i, u, nk);
    }
    wait_vm<AL + BL>();
    step_barrier();
#pragma unroll
    for (int q = 0; q < NJ + M; ++q) read(0, buf[1], buf[0], 0, q);
    int k = 0;
    for (; k + 5 <= nk; k += 5) {
      step<0>(d, k, nk, acc);
      step<2>(d, k + 1, nk, acc);
      step<4>(d, k + 2, nk, acc);
      step<6>(d, k + 3, nk, acc);
      step<8>(d, k + 4, nk, acc);
    }
    // the last nk % 5 steps in straight-line code: a branch inside the rotation
    // would make the compiler wait for every load at each merge
    if (k < nk) {
      step<0>(d, k, nk, acc);
      if (k + 1 < nk) {
        step<2>(d, k + 1, nk, acc);
        if (k + 2 < nk) {
          step<4>(d, k + 2, nk, acc);
          if (k + 3 < nk) step<6>(d, k + 3, nk, acc);
        }
      }
    }
    // the last loads (zeros past the end) must land before the buffers are reused
    wait_vm<0>();
    __syncthreads();
  }
};

// The K loop shared by both GEMMs over nk steps.  At the top of step k, steps
// k .. k+NS-2 are in flight; the thread waits for its loads of step k, the
// barrier makes every thread's loads visible and frees the stage of step k-1,
// step k+NS-1 goes into that stage, then step k's MFMAs run.  The barrier
// waits for this wave's LDS reads only (tm_lds_barrier), not for its
// outstanding loads: the loads of the next steps stay in flight.
template <class C, int M, int DT, bool NTB>
__device__ __forceinline__ void k_loop(const Stages& sb, const DmaLoad<C>& d, int nk,
                                       const int (&brow)[C::NJ], f32x16_t (&acc)[M][C::NJ]) {
  if constexpr (C::PIPE) {
    PipeLoop<C, M, DT, NTB> loop;
    loop.run(sb, d, nk, brow, acc);
  } else {
    constexpr int NS = C::NSTAGE;
    uint8_t* const st[3] = {sb.s0, sb.s1, sb.s2};
#pragma unroll
    for (int u = 0; u < NS - 1; ++u) dma_step<C, NTB>(d, st[u], u, nk);
    for (int k = 0; k < nk; k += NS) {
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        wait_vm<(NS - 2) * C::LDS_PER_STEP>();
        tm_lds_barrier();
        dma_step<C, NTB>(d, st[(u + NS - 1) % NS], k + u + NS - 1, nk);
        if (u == 0 || k + u < nk) compute_step<C, M, DT>(st[u], brow, acc);
      }
    }
    // the last loads (zeros past the end) must land before the stages are reused
    wait_vm<0>();
    __syncthreads();
  }
}

// ------------------------------------------------------------- gate/up --
// h[p, n] = bf16( silu(x[tok(p)] . w1[e, n]) * (x[tok(p)] . w3[e, n]) ) for the
// rows p of one M-tile and the 128 columns n of one column block.
template <class C>
__device__ __forceinline__ uint8_t* h_stage(const Stages& sb, int m) {
  const int s = m / C::HROWS;
  uint8_t* base = s == 0 ? sb.s0 : s == 1 ? sb.s1 : s == 2 ? sb.s2 : sb.s3;
  return base + (m % C::HROWS) * C::HSTRIDE;
}

// silu(a) b in fp32, silu(a) = a / (1 + e^-a), as the weight-streaming gate/up
// computes it.  __expf rounds a log2(e) before the base-2 exponential, so its
// relative error grows with |a|, about |a| 2^-24: 5e-6 where e^-a overflows, far
// below the 2^-9 (bf16) or 2^-12 (fp16) of the rounding of h.  The division is
// the IEEE one: the reciprocal instruction flushes a subnormal result, which
// made silu(a) 0 for a between -88.7 and -87.3, where it is a normal number
// (same box, one layer: T = 517 587 -> 593 us, T = 2048 1413 -> 1427, T = 6011
// 3535 -> 3570).
__device__ __forceinline__ float swiglu(float a, float b) {
  return (a / (1.0f + __expf(-a))) * b;
}

// The MFMAs and the epilogue of one gate/up tile with M accumulator tiles
// per wave (see compute_step): SwiGLU in registers, the bf16 tile staged in
// LDS, then a coalesced store of its `rows` rows.
template <class C, int M, int DT, bool NTB>
__device__ __forceinline__ void gemm1_tile(const Stages& sb, const DmaLoad<C>& d, int nk,
                                           int rows, int p0, int n0, int I,
                                           uint16_t* __restrict__ h) {
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int wm = wave & 1, wn = wave >> 1;
  constexpr int NJ = C::NJ, NH = NJ / 2;
  f32x16_t acc[M][NJ];
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  // accumulator column blocks: the first NH hold w1 rows, the others the same w3 rows
  int brow[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    brow[j] = (j / NH) * (C::PBN / 2) + 32 * NH * wn + 32 * (j % NH);
  k_loop<C, M, DT, NTB>(sb, d, nk, brow, acc);
#pragma unroll
  for (int i = 0; i < M; ++i) {
    uint8_t* const hr = h_stage<C>(sb, 32 * M * wm + 32 * i + (lane & 31));
#pragma unroll
    for (int j = 0; j < NH; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float hv[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) hv[v] = swiglu(acc[i][j][4 * q + v], acc[i][NH + j][4 * q + v]);
        const u32x2_t p = {pack16<DT>(hv[0], hv[1]), pack16<DT>(hv[2], hv[3])};
        *reinterpret_cast<u32x2_t*>(hr + (32 * NH * wn + 32 * j + acc_col(q, lane)) * 2) = p;
      }
  }
  __syncthreads();
  constexpr int PPR = C::PBN / 16;  // 16-byte pieces of an h row (PBN / 2 columns)
#pragma unroll
  for (int j = 0; j < 64 * M * PPR / C::NT; ++j) {
    const int piece = tid + C::NT * j;  // 64 M rows x PPR pieces
    const int r = piece / PPR, c16 = piece % PPR;
    if (r < rows) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(h_stage<C>(sb, r) + c16 * 16);
      *reinterpret_cast<u32x4_t*>(h + (size_t)(p0 + r) * I + n0 + c16 * 8) = v;
    }
  }
}

// gemm1_tile with the fewest accumulator tiles M <= MM per wave whose 64 M
// rows (two waves of 32 M) cover `rows`.  Each output keeps the same K order
// whatever M is, so the bits do not depend on it.
template <class C, int MM, int DT, bool NTB>
__device__ __forceinline__ void gemm1_rows(const Stages& sb, const DmaLoad<C>& d, int nk,
                                           int rows, int p0, int n0, int I,
                                           uint16_t* __restrict__ h) {
  if constexpr (MM > 1) {
    if (rows <= 64 * (MM - 1)) {
      gemm1_rows<C, MM - 1, DT, NTB>(sb, d, nk, rows, p0, n0, I, h);
      return;
    }
  }
  gemm1_tile<C, MM, DT, NTB>(sb, d, nk, rows, p0, n0, I, h);
}

// One gate/up job: M-tile (expert e, sorted rows p0 .. p0 + rows) against
// column block cb; d.ra and d.aoff (the A rows) are set by the caller.
template <class C, int DT>
__device__ __forceinline__ void gemm1_job(const Stages& sb, DmaLoad<C>& d,
                                          const uint16_t* __restrict__ w1,
                                          const uint16_t* __restrict__ w3,
                                          uint16_t* __restrict__ h, int e, int p0, int rows,
                                          bool single, int cb, int H, int I) {
  const int n0 = cb * (C::PBN / 2);  // first h column of the block
  const size_t ebase = (size_t)e * I * H;
  d.pb0 = w1 + ebase;
  d.pb1 = w3 + ebase;
  d.nb = (uint32_t)((size_t)I * H * 2);
#pragma unroll
  for (int i = 0; i < C::BLD; ++i) {
    const int r = dma_row<C>(i);  // first half of the loads: w1 rows; second: the same w3 rows
    d.boff[i] = (uint32_t)(n0 + (r & (C::PBN / 2 - 1))) * (uint32_t)H * 2u +
                (uint32_t)dma_chunk<C>(r) * 16u;
  }
  // A tile with fewer than BM real rows (an expert's last) runs the MFMAs of
  // its first ceil(rows / 64) 64-row quarters only; its A rows past `rows`
  // are loaded as zeros without memory traffic.  An expert that takes one
  // M-tile has its weights read by this job alone: they stream through with
  // the non-temporal policy (a load-only probe streams 7.1 TB/s with it, 6.2
  // without).  With several M-tiles the other jobs of the expert find them in
  // L2, so those loads stay cached.
  if (single)
    gemm1_rows<C, C::MT, DT, true>(sb, d, H / C::PBK, rows, p0, n0, I, h);
  else gemm1_rows<C, C::MT, DT, false>(sb, d, H / C::PBK, rows, p0, n0, I, h);
}

template <class C, int DT>
__global__ void __launch_bounds__(C::NT)
tm_prefill_gemm1_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w1,
                        const uint16_t* __restrict__ w3, uint16_t* __restrict__ h,
                        const int32_t* __restrict__ sorted_slots,
                        const int32_t* __restrict__ offsets, const int32_t* __restrict__ tiles,
                        int max_tiles, int E, int H, int I, int mt_max, uint32_t x_bytes) {
  TM_STAGES(C);
  Job jb;
  if (!expert_job<C>((int)blockIdx.x, offsets, tiles, max_tiles, E, mt_max, I / (C::PBN / 2),
                     &jb))
    return;
  DmaLoad<C> d;
  d.pa = x;
  d.na = x_bytes;
#pragma unroll
  for (int i = 0; i < C::ALD; ++i) {
    const int r = dma_row<C>(i);
    d.aoff[i] = r < jb.rows ? (uint32_t)(sorted_slots[jb.p0 + r] >> 1) * (uint32_t)H * 2u +
                                  (uint32_t)dma_chunk<C>(r) * 16u
                            : kOOR;
  }
  gemm1_job<C, DT>(sb, d, w1, w3, h, jb.e, jb.p0, jb.rows, jb.single, jb.col, H, I);
}

// ------------------------------------------------ gate/up, self-routed --
// At few tokens the budget routing and bucketing run inside the gate/up
// launch instead of in a launch of their own.  Launch index 0 runs the
// routing phases of the routing kernel (tmb::bucket_phases, same code and
// floating-point order) and writes every routing output (topk_ids,
// gates_flat, the layouts, demand) for the down GEMM, the combine and the
// Routing handle; indices 1 .. 7 exit, so GEMM job j = index - 8 keeps XCD
// j % 8 (job_of).  Every wave of a GEMM workgroup derives its job from the
// router gates by itself, one token per lane, with cross-lane operations only
// (rr_job): no LDS and no barrier, one round of global loads (the gates), and
// the same operations in the same order as the phases, so the same experts,
// counts and rows.  Measured on MI355X against the routing launch, same box,
// whole layer: config 2 440 against 445 us, config 3 (B = 4) 247 against
// 252.5 us, the TP-2 and TP-4 shares 5 us faster each.  Tried first: every
// GEMM workgroup running the LDS phases themselves (their barriers cost it
// as much as the routing launch saved), and a per-wave view with one
// reduction chain per expert in turn (~9 us per job instead of ~5).
constexpr int kRrMaxTokens = 64;       // one token per lane
constexpr int kRrMaxExperts = 16;      // gates of a token held in registers
constexpr int kRvMaxBlocks = 256;      // reference padded blocks (the writer's LDS)
constexpr int kRvLeaders = 8;          // launch indices before the GEMM jobs
using RvShared = tmb::BucketSharedT<kRrMaxTokens, kRrMaxTokens * kRrMaxExperts, kRvMaxBlocks>;

// Position of the j-th set bit (j from 0) of m, which has more than j.
__device__ __forceinline__ int nth_set_bit(unsigned long long m, int j) {
  int pos = 0;
#pragma unroll
  for (int w = 32; w >= 1; w >>= 1) {
    const unsigned long long low = m & ((1ull << w) - 1ull);
    const int c = __popcll(low);
    if (j >= c) {
      j -= c;
      pos += w;
      m >>= w;
    }
  }
  return pos;
}

// The job of GEMM launch index l (M-tile of BM rows of one expert x column
// block, job_of over the layer's real M-tiles) from the router gates, in one
// wave: lane t holds token t's gates, EM >= E registers of them.  The expert
// of each routed slot, each expert's count and compact offset, and the
// M-tiles follow tmb::bucket_phases step by step:
//   demand[e] = 0 + accept[t] gates[t, e] in lane t (0 past T), then the xor
//   halving tree; crit[e] likewise with fmaxf (critical-path objective only);
//   keep = ranks in the order (crit desc,) demand desc, e asc;
//   masked top-2 per token, offered in expert order;
//   the slots of expert e in slot order are the tokens whose top-2 holds e
//   (the two picks differ), so each expert's rows are the set bits of one
//   64-bit ballot, in token order, and its count that ballot's popcount.
// The EM halving trees run interleaved and everything after them on wave-
// uniform (scalar) values: a wave spends about a microsecond here beyond the
// gates' load.  Returns false when l has no job.  `mask` is the expert's
// token ballot and m0 the rank of the M-tile's first row among its rows.
template <class C, int EM>
__device__ __forceinline__ bool rr_job(const tmb::BucketArgs& a, int l, int ncol, int mt_max,
                                       int* e_out, int* p0_out, int* rows_out, int* m0_out,
                                       bool* single_out, int* cb_out,
                                       unsigned long long* mask_out) {
  const int lane = threadIdx.x & 63;
  const int T = a.T, E = a.E;
  const bool tok = lane < T;
  // the accept probability is read with the gates (one memory round trip:
  // loaded after the gates had arrived it cost a second one, ~2 us per job)
  const float a_ld = a.accept[tok ? lane : 0];
  float g[EM];
  if ((E & 3) == 0 && (reinterpret_cast<uintptr_t>(a.gates) & 15) == 0) {
#pragma unroll
    for (int q = 0; q < EM / 4; ++q) {
      const bool ok = tok && 4 * q < E;
      const float4 v = *reinterpret_cast<const float4*>(a.gates + (ok ? lane * E + 4 * q : 0));
      g[4 * q] = ok ? v.x : 0.0f;
      g[4 * q + 1] = ok ? v.y : 0.0f;
      g[4 * q + 2] = ok ? v.z : 0.0f;
      g[4 * q + 3] = ok ? v.w : 0.0f;
    }
  } else {
#pragma unroll
    for (int e = 0; e < EM; ++e) {
      const bool ok = tok && e < E;
      const float v = a.gates[ok ? lane * E + e : 0];
      g[e] = ok ? v : 0.0f;
    }
  }
  // with a budget of every expert, all are kept whatever the demand
  unsigned long long keep = (1ull << E) - 1ull;
  if (a.budget < E) {
    float demand[EM];
    keep = tmb::keep_set<EM>(a, g, a_ld, tok, lane, demand);
  }
  // masked top-2 of this lane's token
  tmb::Top2 r{-1, -1, 0.0f, 0.0f};
#pragma unroll
  for (int e = 0; e < EM; ++e)
    if (e < E) r.offer(((keep >> e) & 1ull) ? g[e] : 0.0f, e);
  const int i1 = tok ? r.i1 : -1;
  const int i2 = tok ? r.i2 : -1;
  // per-expert counts, compact offsets and M-tiles on scalars
  int cnt[EM], off_e[EM], ps[EM];
  int run_off = 0, run_mt = 0;
#pragma unroll
  for (int e = 0; e < EM; ++e) {
    cnt[e] = __popcll(__ballot(i1 == e || i2 == e));
    off_e[e] = run_off;
    ps[e] = run_mt;
    run_off += cnt[e];
    run_mt += (cnt[e] + C::PBM - 1) / C::PBM;
  }
  const int n_mt = min(run_mt, mt_max);
  int mt, cb;
  if (!job_of(l, n_mt, ncol, &mt, &cb)) return false;
  int e = -1;
#pragma unroll
  for (int k = 0; k < EM; ++k)
    if (e < 0 && mt < ps[k] + (cnt[k] + C::PBM - 1) / C::PBM) e = k;
  if (e < 0) return false;
  int cnt_e = 0, off_sel = 0, ps_sel = 0;
#pragma unroll
  for (int k = 0; k < EM; ++k)
    if (k == e) {
      cnt_e = cnt[k];
      off_sel = off_e[k];
      ps_sel = ps[k];
    }
  const int m0 = (mt - ps_sel) * C::PBM;
  *e_out = e;
  *m0_out = m0;
  *p0_out = off_sel + m0;
  *rows_out = min(C::PBM, cnt_e - m0);
  *single_out = (cnt_e + C::PBM - 1) / C::PBM == 1;
  *cb_out = cb;
  *mask_out = __ballot(i1 == e || i2 == e);
  return true;
}

template <class C, int DT, int EM>
__global__ void __launch_bounds__(C::NT)
tm_prefill_gemm1_routed_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w1,
                               const uint16_t* __restrict__ w3, uint16_t* __restrict__ h,
                               tmb::BucketArgs ra, int H, int I, int mt_max, uint32_t x_bytes) {
  TM_STAGES(C);
  static_assert(sizeof(RvShared) <= C::BUF, "the routing writer uses the first stage");
  const int L = (int)blockIdx.x;
  if (L < kRvLeaders) {
    if (L == 0) tmb::bucket_phases<C::NT, RvShared>(ra, *reinterpret_cast<RvShared*>(s0));
    return;
  }
  int e, p0, rows, m0, cb;
  bool single;
  unsigned long long mask;
  if (!rr_job<C, EM>(ra, L - kRvLeaders, I / (C::PBN / 2), mt_max, &e, &p0, &rows, &m0,
                     &single, &cb, &mask))
    return;
  DmaLoad<C> d;
  d.pa = x;
  d.na = x_bytes;
#pragma unroll
  for (int i = 0; i < C::ALD; ++i) {
    const int r = dma_row<C>(i);
    d.aoff[i] = r < rows ? (uint32_t)nth_set_bit(mask, m0 + r) * (uint32_t)H * 2u +
                               (uint32_t)dma_chunk<C>(r) * 16u
                         : kOOR;
  }
  gemm1_job<C, DT>(sb, d, w1, w3, h, e, p0, rows, single, cb, H, I);
}

// ---------------------------------------------------------------- down --
// y[s, p, n] = gates_flat[slot(p)] * sum_{k in segment s} h[p, k] w2[e, n, k]
// for the rows p of one M-tile and BN output columns n.  The fp32 partials
// go straight from the accumulators, 16 bytes per lane and store; a lane's
// rows (one per accumulator row block) have their gates loaded before the K
// loop.
template <class C, int M, int DT, bool NTB>
__device__ __forceinline__ void gemm2_tile(const Stages& sb, const DmaLoad<C>& d, int nk,
                                           int rows, int p0, int H,
                                           const float* __restrict__ gates_flat,
                                           const int32_t* __restrict__ sorted_slots,
                                           float* __restrict__ ys) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = wave & 1, wn = wave >> 1;
  constexpr int NJ = C::NJ;
  float gate[M];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    const int m = 32 * M * wm + 32 * i + (lane & 31);
    gate[i] = gates_flat[sorted_slots[p0 + min(m, rows - 1)]];
  }
  f32x16_t acc[M][NJ];
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  int brow[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) brow[j] = 32 * NJ * wn + 32 * j;
  k_loop<C, M, DT, NTB>(sb, d, nk, brow, acc);
#pragma unroll
  for (int i = 0; i < M; ++i) {
    const int m = 32 * M * wm + 32 * i + (lane & 31);
    if (m < rows) {
      float* const yr = ys + (size_t)(p0 + m) * H + 32 * NJ * wn;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4_t o;
#pragma unroll
          for (int v = 0; v < 4; ++v) o[v] = acc[i][j][4 * q + v] * gate[i];
          *reinterpret_cast<f32x4_t*>(yr + 32 * j + acc_col(q, lane)) = o;
        }
    }
  }
}

// gemm2_tile with the fewest accumulator tiles that cover `rows`, as gemm1_rows.
template <class C, int MM, int DT, bool NTB>
__device__ __forceinline__ void gemm2_rows(const Stages& sb, const DmaLoad<C>& d, int nk,
                                           int rows, int p0, int H,
                                           const float* __restrict__ gates_flat,
                                           const int32_t* __restrict__ sorted_slots,
                                           float* __restrict__ ys) {
  if constexpr (MM > 1) {
    if (rows <= 64 * (MM - 1)) {
      gemm2_rows<C, MM - 1, DT, NTB>(sb, d, nk, rows, p0, H, gates_flat, sorted_slots, ys);
      return;
    }
  }
  gemm2_tile<C, MM, DT, NTB>(sb, d, nk, rows, p0, H, gates_flat, sorted_slots, ys);
}

template <class C, int DT>
__global__ void __launch_bounds__(C::NT)
tm_prefill_gemm2_kernel(const uint16_t* __restrict__ h, const uint16_t* __restrict__ w2,
                        float* __restrict__ y, const float* __restrict__ gates_flat,
                        const int32_t* __restrict__ sorted_slots,
                        const int32_t* __restrict__ offsets, const int32_t* __restrict__ tiles,
                        int max_tiles, int E, int R, int H, int I, int klen, int nsplit,
                        int mt_max, uint32_t h_bytes) {
  TM_STAGES(C);
  const int ncb = H / C::PBN;
  Job jb;  // col = (segment, column block), segment-major
  if (!expert_job<C>((int)blockIdx.x, offsets, tiles, max_tiles, E, mt_max, ncb * nsplit, &jb))
    return;
  // Each XCD owns a contiguous range of these jobs, so segment-major puts
  // one K segment on each XCD (2 segments over 8 XCDs: 4 each) and an XCD
  // reads the h rows of its segment only, instead of all of h.
  const int seg = jb.col / ncb;
  const int cb = jb.col - seg * ncb;
  const int n0 = cb * C::PBN;
  const uint32_t k0 = (uint32_t)seg * (uint32_t)klen * 2u;  // segment start, bytes

  DmaLoad<C> d;
  d.pa = h;
  d.na = h_bytes;
  d.pb0 = d.pb1 = w2 + (size_t)jb.e * H * I;
  d.nb = (uint32_t)((size_t)H * I * 2);
#pragma unroll
  for (int i = 0; i < C::ALD; ++i) {
    const int r = dma_row<C>(i);
    d.aoff[i] = r < jb.rows ? (uint32_t)(jb.p0 + r) * (uint32_t)I * 2u + k0 +
                                  (uint32_t)dma_chunk<C>(r) * 16u
                            : kOOR;
  }
#pragma unroll
  for (int i = 0; i < C::BLD; ++i) {
    const int r = dma_row<C>(i);
    d.boff[i] = (uint32_t)(n0 + r) * (uint32_t)I * 2u + k0 + (uint32_t)dma_chunk<C>(r) * 16u;
  }
  float* ys = y + (size_t)seg * R * H + n0;
  const int nk = klen / C::PBK;
  if (jb.single)
    gemm2_rows<C, C::MT, DT, true>(sb, d, nk, jb.rows, jb.p0, H, gates_flat,
                                            sorted_slots, ys);
  else
    gemm2_rows<C, C::MT, DT, false>(sb, d, nk, jb.rows, jb.p0, H, gates_flat, sorted_slots, ys);
}

bool aligned16(const void* p) { return ((uintptr_t)p % 16) == 0; }

// M-tiles of BM rows that `active` experts averaging `rows` rows take, their loads
// taken as spread evenly over +-20 % of the average.
double expected_mtiles(double active, double rows, int BM) {
  const double lo = 0.8 * rows, hi = 1.2 * rows;
  int64_t k = (int64_t)(lo / BM) + 1;
  double n = (double)k;
  for (; (double)(k * BM) < hi; ++k) n += (hi - (double)(k * BM)) / (hi - lo);
  return active * n;
}

// Tile256 for a GEMM of `ncol` column jobs (256 weight rows each) whose jobs run
// over K: where the experts average 112 rows or more, and its jobs, half as many
// as Tile128's, still come out ahead in rounds over the CUs.  An XCD runs its
// cpx columns of every M-tile on its 32 CUs (a last round counts in full once it
// is likely to have a sixth of the CUs' jobs); a Tile256 round takes 1.3 + 150 / K
// Tile128 rounds (the prologue and epilogue weigh more at a short K).  From 112
// rows on an expert often has more rows than a 128-row tile holds, and its
// weights pass through LDS twice.  Tile128 against Tile256, same box, us:
//   H = 4096, I = 14336, E = 8   T = 448 gate/up 343 / 366, down 253 / 168;
//     T = 517 418 / 370, 241 / 163; T = 2048 1028 / 890, 538 / 484
//   H = 4096, I = 1792, E = 8    T = 700 70 / 80, 43 / 48; T = 1200 114 / 89, 66 / 51
//   H = 1024, I = 3584, E = 8    T = 700 41 / 40, 25 / 33; T = 1200 55 / 64, 39 / 35
//   H = 512, I = 2048, E = 8     T = 700 18 / 27, 17 / 24; T = 3000 51 / 48, 33 / 28
// Over 348 layers of H = 256 .. 4096, E = 2 .. 64, T = 112 .. 6000, the tile it picks
// is 2 % behind the better of the two in the mean, the 256-row tile everywhere
// 12 %.
bool use_tile256(int64_t T, int64_t E, int64_t max_tiles, int64_t ncol, int64_t K) {
  if (2 * T < 112 * E) return false;
  // the routed experts, from the tile list's bound: a + (2T - a) / 64 tiles
  int64_t active = 1;
  while (active < E && active + (2 * T - active) / TM_GEMM_TILE_M < max_tiles) ++active;
  const double rows = 2.0 * (double)T / (double)active;
  const double cpx = (double)((ncol + kXcds - 1) / kXcds);
  const auto rounds = [&](int BM) {
    const double r = expected_mtiles((double)active, rows, BM) * cpx / (kCUs / kXcds);
    return std::floor(r) + std::min(1.0, 6.0 * (r - std::floor(r)));
  };
  return (1.3 + 150.0 / (double)K) * rounds(256) <= rounds(128);
}

// Rows of the gate/up tile.  TileDec when the tile list leaves at most 16 rows per
// entry (2T <= 16 max_tiles: few rows per active expert, e.g. 64 tree tokens over
// 8 experts): half the weight rows per workgroup and two workgroups per CU
// stream the weights faster there (config 2 gate/up 302 -> 289 us same-box).
int gate_up_rows(int64_t max_tiles, int64_t T, int64_t H, int64_t I, int64_t E) {
  if (use_tile256(T, E, max_tiles, I / (Tile256::PBN / 2), H)) return 256;
  return 2 * T <= 16 * max_tiles ? 64 : 128;
}

// Rows of the down tile.  TileDec (twice the column jobs, two workgroups per CU)
// where the 128-row tile's jobs leave CUs without one and few experts exceed its
// 64 rows.  Down + combine on Tile128 against TileDec, four K segments, E = 8,
// I = 3584: H = 1024 (at most 144 jobs) T = 16 18.2 against 14.6 us, T = 64 18.9 /
// 15.1, T = 64 budget 4 19.8 / 14.1, T = 200 23.3 / 18.6; where the jobs fill the
// CUs, H = 4096, I = 14336, T = 64 budget 4 79.7 / 84.0.
int down_rows(int64_t max_tiles, int64_t split, int64_t T, int64_t H, int64_t I, int64_t E) {
  const int64_t ncol = H / Tile128::PBN * split;
  if (use_tile256(T, E, max_tiles, ncol, I / split)) return 256;
  const int64_t mt128 = std::min<int64_t>(max_tiles, mtile_bound<Tile128>(2 * T, E));
  return 2 * T <= 64 * E && mt128 * ncol < kCUs ? 64 : 128;
}

// The gate/up launch with tile C: jobs for the M-tile bound (the tile list's
// length, capped by what 2T rows in E experts can take).
template <class C, int DT>
int launch_gemm1(const void* x, const void* w1, const void* w3, void* h,
                 const int32_t* sorted_slots, const int32_t* expert_offsets,
                 const int32_t* tiles, int64_t max_tiles, int64_t T, int64_t H, int64_t I,
                 int64_t E, hipStream_t stream) {
  const int64_t mt_max = std::min<int64_t>(max_tiles, mtile_bound<C>(2 * T, E));
  const int64_t jobs = launch_jobs(mt_max, I / (C::PBN / 2));
  if (jobs > INT32_MAX) return TM_ERR_SHAPE;
  hipLaunchKernelGGL((tm_prefill_gemm1_kernel<C, DT>), dim3((unsigned)jobs), dim3(C::NT), 0, stream,
                     (const uint16_t*)x, (const uint16_t*)w1, (const uint16_t*)w3,
                     (uint16_t*)h, sorted_slots, expert_offsets, tiles, (int)max_tiles,
                     (int)E, (int)H, (int)I, (int)mt_max, (uint32_t)(T * H * 2));
  return TM_OK;
}

// The self-routed gate/up launch with tile C.
template <class C, int DT>
int launch_gemm1_routed(const void* x, const void* w1, const void* w3, void* h,
                        const tmb::BucketArgs& ra, int64_t T, int64_t H, int64_t I,
                        hipStream_t stream) {
  const int64_t mt_max = std::min<int64_t>(ra.max_tiles, mtile_bound<C>(2 * T, ra.E));
  const int64_t jobs = launch_jobs(mt_max, I / (C::PBN / 2)) + kRvLeaders;
  if (jobs > INT32_MAX) return TM_ERR_SHAPE;
  if (ra.E <= 8)
    hipLaunchKernelGGL((tm_prefill_gemm1_routed_kernel<C, DT, 8>), dim3((unsigned)jobs),
                       dim3(C::NT), 0, stream, (const uint16_t*)x, (const uint16_t*)w1,
                       (const uint16_t*)w3, (uint16_t*)h, ra, (int)H, (int)I, (int)mt_max,
                       (uint32_t)(T * H * 2));
  else
    hipLaunchKernelGGL((tm_prefill_gemm1_routed_kernel<C, DT, kRrMaxExperts>),
                       dim3((unsigned)jobs), dim3(C::NT), 0, stream, (const uint16_t*)x,
                       (const uint16_t*)w1, (const uint16_t*)w3, (uint16_t*)h, ra, (int)H,
                       (int)I, (int)mt_max, (uint32_t)(T * H * 2));
  return TM_OK;
}

}  // namespace

extern "C" int tm_op1_prefill_gemm1(const void* x, const void* w1, const void* w3, void* h,
                                    const int32_t* sorted_slots, const int32_t* expert_offsets,
                                    const int32_t* tiles, int64_t max_tiles, int64_t T,
                                    int64_t H, int64_t I, int64_t E, int dtype, void* stream) {
  if (T < 1 || T > TM_MAX_TOKENS || E < 2 || E > TM_MAX_EXPERTS || max_tiles < 1)
    return TM_ERR_SHAPE;
  if (dtype != TM_DTYPE_BF16 && dtype != TM_DTYPE_F16) return TM_ERR_ARG;
  if (H < Tile128::PBK || (H % Tile128::PBK) != 0 || I < Tile128::PBN / 2 ||
      (I % (Tile128::PBN / 2)) != 0)
    return TM_ERR_SHAPE;
  if (I * H * 2 >= (int64_t)kOOR || T * H * 2 >= (int64_t)kOOR || 2 * T * I * 2 >= (int64_t)kOOR)
    return TM_ERR_SHAPE;
  if (!aligned16(x) || !aligned16(w1) || !aligned16(w3) || !aligned16(h)) return TM_ERR_ALIGN;
  const int tile = gate_up_rows(max_tiles, T, H, I, E);
  const hipStream_t st = (hipStream_t)stream;
  const bool f16 = dtype == TM_DTYPE_F16;
  int rc;
  if (tile == 256) {
    rc = f16 ? launch_gemm1<Tile256, TM_DTYPE_F16>(x, w1, w3, h, sorted_slots, expert_offsets,
                                                   tiles, max_tiles, T, H, I, E, st)
             : launch_gemm1<Tile256, TM_DTYPE_BF16>(x, w1, w3, h, sorted_slots, expert_offsets,
                                                    tiles, max_tiles, T, H, I, E, st);
  } else if (tile == 64) {
    rc = f16 ? launch_gemm1<TileDec, TM_DTYPE_F16>(x, w1, w3, h, sorted_slots, expert_offsets,
                                                   tiles, max_tiles, T, H, I, E, st)
             : launch_gemm1<TileDec, TM_DTYPE_BF16>(x, w1, w3, h, sorted_slots, expert_offsets,
                                                    tiles, max_tiles, T, H, I, E, st);
  } else {
    rc = f16 ? launch_gemm1<Tile128, TM_DTYPE_F16>(x, w1, w3, h, sorted_slots, expert_offsets,
                                                   tiles, max_tiles, T, H, I, E, st)
             : launch_gemm1<Tile128, TM_DTYPE_BF16>(x, w1, w3, h, sorted_slots, expert_offsets,
                                                    tiles, max_tiles, T, H, I, E, st);
  }
  if (rc) return rc;
  TM_HIP_CHECK_LAUNCH();
  return TM_OK;
}

extern "C" int tm_op1_prefill_tiles(int64_t max_tiles, int64_t split, int64_t T, int64_t H,
                                    int64_t I, int64_t E, int64_t* gate_up, int64_t* down) {
  if (T < 1 || T > TM_MAX_TOKENS || E < 2 || E > TM_MAX_EXPERTS || max_tiles < 1 || split < 1 ||
      H < 1 || I < split)
    return TM_ERR_SHAPE;
  if (gate_up == nullptr || down == nullptr) return TM_ERR_ARG;
  *gate_up = gate_up_rows(max_tiles, T, H, I, E);
  *down = down_rows(max_tiles, split, T, H, I, E);
  return TM_OK;
}

extern "C" int tm_op1_prefill_gemm1_routed(
    const void* x, const void* w1, const void* w3, void* h, const float* gates,
    const float* accept, int64_t T, int64_t H, int64_t I, int64_t E, int64_t budget, float tau,
    int objective, int64_t block_m, int64_t max_blocks, int64_t max_tiles, int64_t* topk_ids,
    float* gates_flat, int64_t* padded_slots, int64_t* block_expert_ids, int64_t* slot_to_row,
    float* demand, int32_t* expert_offsets, int32_t* sorted_slots, int32_t* slot_pos,
    int32_t* tiles, int dtype, void* stream) {
  if (T < 1 || T > kRrMaxTokens || E < 2 || E > kRrMaxExperts) return TM_ERR_SHAPE;
  if (budget < 2 || budget > E) return TM_ERR_ARG;
  if (objective != TM_OBJECTIVE_MASS && objective != TM_OBJECTIVE_CRITICAL_PATH) return TM_ERR_ARG;
  if (block_m != 16 && block_m != 32) return TM_ERR_ARG;
  if (max_blocks < 1 || max_blocks > kRvMaxBlocks || max_tiles < 1) return TM_ERR_SHAPE;
  if (dtype != TM_DTYPE_BF16 && dtype != TM_DTYPE_F16) return TM_ERR_ARG;
  if (H < Tile128::PBK || (H % Tile128::PBK) != 0 || I < Tile128::PBN / 2 ||
      (I % (Tile128::PBN / 2)) != 0)
    return TM_ERR_SHAPE;
  if (I * H * 2 >= (int64_t)kOOR || T * H * 2 >= (int64_t)kOOR || 2 * T * I * 2 >= (int64_t)kOOR)
    return TM_ERR_SHAPE;
  if (!aligned16(x) || !aligned16(w1) || !aligned16(w3) || !aligned16(h)) return TM_ERR_ALIGN;
  tmb::BucketArgs ra;
  ra.gates = gates;
  ra.accept = accept;
  ra.T = (int)T;
  ra.E = (int)E;
  ra.budget = (int)budget;
  ra.objective = objective;
  ra.BM = (int)block_m;
  ra.max_blocks = (int)max_blocks;
  ra.max_tiles = (int)max_tiles;
  ra.tau = tau;
  ra.topk_ids = topk_ids;
  ra.gates_flat = gates_flat;
  ra.padded_slots = padded_slots;
  ra.block_expert_ids = block_expert_ids;
  ra.slot_to_row = slot_to_row;
  ra.demand_out = demand;
  ra.expert_offsets = expert_offsets;
  ra.sorted_slots = sorted_slots;
  ra.slot_pos = slot_pos;
  ra.tiles = tiles;
  // the tile rule of tm_op1_prefill_gemm1 without the 256-row tile (T <= 64: at
  // most 64 rows per expert)
  const bool dec = 2 * T <= 16 * max_tiles;
  const hipStream_t st = (hipStream_t)stream;
  const bool f16 = dtype == TM_DTYPE_F16;
  int rc;
  if (dec) {
    rc = f16 ? launch_gemm1_routed<TileDec, TM_DTYPE_F16>(x, w1, w3, h, ra, T, H, I, st)
             : launch_gemm1_routed<TileDec, TM_DTYPE_BF16>(x, w1, w3, h, ra, T, H, I, st);
  } else {
    rc = f16 ? launch_gemm1_routed<Tile128, TM_DTYPE_F16>(x, w1, w3, h, ra, T, H, I, st)
             : launch_gemm1_routed<Tile128, TM_DTYPE_BF16>(x, w1, w3, h, ra, T, H, I, st);
  }
  if (rc) return rc;
  TM_HIP_CHECK_LAUNCH();
  return TM_OK;
}

namespace {

// The down launch with tile C.
template <class C>
int launch_gemm2(const void* h, const void* w2, float* y, const float* gates_flat,
                 const int32_t* sorted_slots, const int32_t* expert_offsets,
                 const int32_t* tiles, int64_t max_tiles, int64_t split, int64_t T, int64_t H,
                 int64_t I, int64_t E, int dtype, hipStream_t stream) {
  const int64_t klen = I / split;
  const int64_t mt_max = std::min<int64_t>(max_tiles, mtile_bound<C>(2 * T, E));
  const int64_t jobs = launch_jobs(mt_max, (H / C::PBN) * split);
  if (jobs > INT32_MAX) return TM_ERR_SHAPE;
  hipLaunchKernelGGL((dtype == TM_DTYPE_F16 ? tm_prefill_gemm2_kernel<C, TM_DTYPE_F16>
                                            : tm_prefill_gemm2_kernel<C, TM_DTYPE_BF16>),
                     dim3((unsigned)jobs), dim3(C::NT), 0, stream, (const uint16_t*)h,
                     (const uint16_t*)w2, y, gates_flat, sorted_slots, expert_offsets, tiles,
                     (int)max_tiles, (int)E, (int)(2 * T), (int)H, (int)I, (int)klen,
                     (int)split, (int)mt_max, (uint32_t)(2 * T * I * 2));
  return TM_OK;
}

}  // namespace

extern "C" int tm_op1_prefill_gemm2(const void* h, const void* w2, float* y,
                                    const float* gates_flat, const int32_t* sorted_slots,
                                    const int32_t* expert_offsets, const int32_t* tiles,
                                    int64_t max_tiles, int64_t split, int64_t T, int64_t H,
                                    int64_t I, int64_t E, int dtype, void* stream) {
  using C = Tile128;
  if (T < 1 || T > TM_MAX_TOKENS || E < 2 || E > TM_MAX_EXPERTS || max_tiles < 1)
    return TM_ERR_SHAPE;
  if (dtype != TM_DTYPE_BF16 && dtype != TM_DTYPE_F16) return TM_ERR_ARG;
  if (split < 1 || (I % split) != 0) return TM_ERR_SHAPE;
  const int64_t klen = I / split;
  if (klen < C::PBK || (klen % C::PBK) != 0 || H < C::PBN || (H % C::PBN) != 0) return TM_ERR_SHAPE;
  if (H * I * 2 >= (int64_t)kOOR || 2 * T * I * 2 >= (int64_t)kOOR) return TM_ERR_SHAPE;
  if (!aligned16(h) || !aligned16(w2) || !aligned16(y)) return TM_ERR_ALIGN;
  const int tile = down_rows(max_tiles, split, T, H, I, E);
  const hipStream_t st = (hipStream_t)stream;
  const int rc =
      tile == 256  ? launch_gemm2<Tile256>(h, w2, y, gates_flat, sorted_slots, expert_offsets,
                                           tiles, max_tiles, split, T, H, I, E, dtype, st)
      : tile == 64 ? launch_gemm2<TileDec>(h, w2, y, gates_flat, sorted_slots, expert_offsets,
                                           tiles, max_tiles, split, T, H, I, E, dtype, st)
                   : launch_gemm2<Tile128>(h, w2, y, gates_flat, sorted_slots, expert_offsets,
                                           tiles, max_tiles, split, T, H, I, E, dtype, st);
  if (rc) return rc;
  TM_HIP_CHECK_LAUNCH();
  return TM_OK;
}
