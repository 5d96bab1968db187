// C[M,N] = A[M,K] * B[N,K]^T (+ bias[N]) for gfx950 -- the nn.Linear "TN"
// GEMM of every decoder projection. Same contract as DecodeKernels'
// dk::launch_gemm_tn (csrc/gemm_wmma.cuh:191-219): fp32 accumulation, bias
// added in fp32, one rounding to the model dtype; K, lda, ldb multiples of 8;
// A and B 16-byte aligned; any M, N and ldc.
//
// Two kernels, both on v_mfma_f32_16x16x32_{bf16,f16}:
//
// * skinny (M <= 64, decode): the op streams the weight matrix once, so it is
//   bound by HBM bandwidth -- and, per CU, by how many cache lines its loads
//   touch: an MFMA fragment load of 16 rows touches 16 lines. Weight fragments
//   therefore go straight to registers (each weight byte is used once), while
//   activation tiles are loaded once per workgroup with contiguous 16-byte
//   loads into LDS and shared by the waves that own different output columns.
//   Up to 14 waves per workgroup, split between N (16 columns each) and K; the
//   grid is planned at one workgroup per CU, with wide column tiles to cut the
//   activation re-reads and, given a workspace, the K reduction split over
//   workgroups (fp32 partial tiles summed in order by a second kernel). Buffer
//   loads with descriptor bounds make rows past M/N and columns past K read as
//   zero, and DEPTH-deep register rings of weights and activations keep loads
//   in flight across the per-step barrier.
// * LDS-DMA (M > 64, batched decode and prefill): A and B tiles go from HBM
//   straight into LDS (buffer_load ... lds), bank-conflict-free XOR-swizzled,
//   through a multi-stage ring; eleven tile shapes from 256x256 down to 64x64. A
//   time model picks the tile and the K split of a call (kTileModel), so that
//   batches of a few hundred rows still fill all 256 CUs. The output tile
//   leaves through the freed ring, read back row by row for 16-byte stores. At
//   M <= 64 its 64-row tiles (64 or 128 columns, K split) replace the skinny
//   kernel where the model has them faster (decode_plan).
#include <algorithm>
#include <type_traits>

#include "../../include/decodekernels_amd.h"
#include "dk_device.h"
#include "dk_host.h"

namespace dk {
namespace gemm {

// ---------------------------------------------------------------------------
// Skinny kernel
// ---------------------------------------------------------------------------
// Word 3 of a gfx9-family buffer resource for raw (untyped) loads.
constexpr int kRsrcWord3 = 0x00020000;
// Byte offset that is outside every buffer resource used here: loads there
// return zero without touching memory.
constexpr int kOutOfRange = 0x7fffffff;
// The same for offsets to which a K offset may be added, vector or scalar (both below 2^31; unsigned).
constexpr unsigned kNowhere = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0,
                                           static_cast<int>(bytes < kOutOfRange ? bytes : kOutOfRange), kRsrcWord3);
}

// ---------------------------------------------------------------------------
// Skinny kernel (M <= 64) with LDS-shared activations
// ---------------------------------------------------------------------------
// Workgroup = WN x WK waves: wave (wn, wk) owns output columns n0 + 16 wn ...
// and K chunks c = j * WK + wk (BK = 64 columns each). The activation tile
// of a chunk (16 MT rows x 64) is loaded once per K-group with contiguous
// 16-byte loads (8 lanes cover a 128-byte row segment), written to LDS and
// read by the WN waves of that group, so each activation byte crosses the
// L1 once per workgroup instead of once per wave. Weight fragments go
// straight from HBM to registers; weights and activations both run through
// DEPTH-deep register rings. All waves step through the chunks together (one
// barrier per step); the WK partial tiles are summed through LDS at the end.
constexpr int kLdsBK = 64;
#ifndef DK_SKINNY_ROT
#define DK_SKINNY_ROT 5  // unsplit K walk of workgroup x starts at chunk (x * DK_SKINNY_ROT) mod chunks
#endif
constexpr int kLdsARow = kLdsBK + 8;  // padded LDS row (elements)

template <int MT, int WN>
struct ARegs {
  static constexpr int kVecs = 16 * MT * kLdsBK / 8;                             // 16-byte vectors per tile
  static constexpr int kPerLane = (kVecs + WN * kWave - 1) / (WN * kWave);     // per lane of the K-group
  static constexpr bool kPartial = kVecs % (WN * kWave) != 0;                  // some lanes idle
  u32x4 v[kPerLane];
};

template <typename E, int MT, int WN, int WK, int DEPTH>
__global__ __launch_bounds__(WN * WK * kWave) void gemm_skinny_lds_kernel(const uint16_t* __restrict__ A,
                                                                          const uint16_t* __restrict__ B,
                                                                          const uint16_t* __restrict__ bias,
                                                                          uint16_t* __restrict__ C, int M, int N,
                                                                          int K, int lda, int ldb, int ldc,
                                                                          float* __restrict__ part, int k_split) {
  constexpr int NT = WN * WK * kWave;
  constexpr int KS = kLdsBK / 32;  // k-steps per chunk
  // Split-K (part != nullptr): workgroup row blockIdx.y covers K columns
  // [kb, ke) (k_split a multiple of kLdsBK) and writes its fp32 partial tile to
  // part[blockIdx.y][M][N], without the bias; a second kernel sums the splits.
  const int kb = part != nullptr ? static_cast<int>(blockIdx.y) * k_split : 0;
  const int ke = part != nullptr ? min(K, kb + k_split) : K;
  using AR = ARegs<MT, WN>;
  // The activation tiles and, after the K loop's last barrier, the partial
  // output tiles share one LDS allocation.
  constexpr size_t kBytesA = sizeof(uint16_t) * WK * 2 * 16 * MT * kLdsARow;
  constexpr size_t kBytesRed = sizeof(f32x4) * WK * WN * MT * kWave;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kBytesA > kBytesRed ? kBytesA : kBytesRed];
  auto lds_a = reinterpret_cast<uint16_t(*)[2][16 * MT * kLdsARow]>(smem);
  auto red = reinterpret_cast<f32x4(*)[WN][MT][kWave]>(smem);

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wn = wave % WN;
  const int wk = wave / WN;
  const int gl = wn * kWave + lane;  // lane index inside the K-group
  const int l16 = lane % 16;
  const int lg = lane / 16;
  const int n0 = blockIdx.x * (16 * WN);
  const int ncol0 = n0 + 16 * wn;

  const __amdgpu_buffer_rsrc_t rb =
      rsrc(B + static_cast<int64_t>(ncol0) * ldb, static_cast<int64_t>(max(0, min(16, N - ncol0))) * ldb * 2);
  const __amdgpu_buffer_rsrc_t ra = rsrc(A, static_cast<int64_t>(M) * lda * 2);
  const __amdgpu_buffer_rsrc_t r_none = rsrc(A, 0);
  const int boff = l16 * ldb * 2 + 16 * lg;

  const int n_chunks = (ke - kb + kLdsBK - 1) / kLdsBK;
  const int steps = (n_chunks + WK - 1) / WK;  // chunk steps of the whole workgroup
  // Unsplit, every workgroup walks the whole K range in lockstep with the
  // others: at a given moment they read the same column offset of rows a
  // fixed stride apart, which at some base addresses lands on few HBM
  // channels (measured: qkv M=1 18.3 us at 11 of 12 weight placements, 14.9 at
  // the twelfth). Starting workgroup x's walk at chunk x * DK_SKINNY_ROT mod
  // n_chunks spreads the concurrent reads: 14.3-14.6 us at every placement,
  // gate_up M=16 54.5 -> 44.0 us. Split workgroups already start at different
  // K offsets (rotating them measured 1-5% slower). Chunk c of the walk reads
  // K chunk (c + rot) mod n_chunks; the partial sums are deterministic.
  const int rot = DK_SKINNY_ROT > 0 && part == nullptr && n_chunks > 0
                      ? static_cast<int>((blockIdx.x * static_cast<unsigned>(DK_SKINNY_ROT)) % n_chunks)
                      : 0;
  auto chunk = [&](int c) { return c + rot >= n_chunks ? c + rot - n_chunks : c + rot; };

  // Activation tile of chunk c: vector v of the group covers row v / 8, columns 8 (v % 8) ...
  auto load_a = [&](int step, AR& r) {
    const int c = step * WK + wk;
    const bool live = step < steps && c < n_chunks;
    const __amdgpu_buffer_rsrc_t rr = live ? ra : r_none;
    const int cc = chunk(c);
#pragma unroll
    for (int j = 0; j < AR::kPerLane; ++j) {
      const int v = gl + j * WN * kWave;
      const int row = v / 8;
      const int k = kb + cc * kLdsBK + 8 * (v % 8);
      const bool in = k < ke && (!AR::kPartial || v < AR::kVecs);
      r.v[j] = __builtin_amdgcn_raw_buffer_load_b128(rr, in ? row * lda * 2 + 2 * k : kOutOfRange, 0, 0);
    }
  };
  auto store_a = [&](int buf, const AR& r) {
#pragma unroll
    for (int j = 0; j < AR::kPerLane; ++j) {
      const int v = gl + j * WN * kWave;
      if (!AR::kPartial || v < AR::kVecs) *reinterpret_cast<u32x4*>(&lds_a[wk][buf][(v / 8) * kLdsARow + 8 * (v % 8)]) = r.v[j];
    }
  };
  // Weight fragments of chunk step `step` for this wave: KS k-steps.
  auto load_b = [&](int step, u32x4 (&bf)[KS]) {
    const int c = step * WK + wk;
    const bool live = step < steps && c < n_chunks;
    const __amdgpu_buffer_rsrc_t rr = live ? rb : r_none;
    const int cc = chunk(c);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int k = kb + cc * kLdsBK + 32 * s + 8 * lg;
      bf[s] = __builtin_amdgcn_raw_buffer_load_b128(rr, k < ke ? boff + 2 * (kb + cc * kLdsBK + 32 * s) : kOutOfRange, 0,
                                                    0);
    }
  };

  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Step j's weight fragments and activation vectors live in ring slot
  // j % DEPTH; both are issued DEPTH steps ahead. Loads complete in issue
  // order, so the wait for step j + 1's activations (stored to LDS during
  // step j) covers only loads issued up to step j + 1 - DEPTH: DEPTH - 1
  // steps of both operands stay in flight across each barrier.
  u32x4 bring[DEPTH][KS];
  AR aring[DEPTH];
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    load_a(d, aring[d]);
    load_b(d, bring[d]);
  }
  store_a(0, aring[0]);
  load_a(DEPTH, aring[0]);
  __syncthreads();

  for (int base = 0; base < steps; base += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int step = base + d;
      const int d1 = (d + 1) % DEPTH;
      if (step < steps) {
        const uint16_t* at = lds_a[wk][step & 1];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            const u32x4 af = *reinterpret_cast<const u32x4*>(&at[(16 * i + l16) * kLdsARow + 32 * s + 8 * lg]);
            acc[i] = E::mfma_16x16x32(af, bring[d][s], acc[i]);
          }
        }
      }
      load_b(step + DEPTH, bring[d]);
      if (step + 1 < steps) store_a((step + 1) & 1, aring[d1]);
      load_a(step + 1 + DEPTH, aring[d1]);
      __syncthreads();
    }
  }

#pragma unroll
  for (int i = 0; i < MT; ++i) red[wk][wn][i][lane] = acc[i];
  __syncthreads();

  // acc[i] of wave (wn, *) lane l, reg r: C[16 i + 4 (l/16) + r][n0 + 16 wn + l % 16].
  for (int e = threadIdx.x; e < MT * 16 * 16 * WN; e += NT) {
    const int cn = e % (16 * WN);
    const int m = e / (16 * WN);
    const int n = n0 + cn;
    if (m >= M || n >= N) continue;
    const int i = m / 16;
    const int src_lane = 16 * ((m % 16) / 4) + (cn % 16);
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < WK; ++w) v += red[w][cn / 16][i][src_lane][m % 4];
    if (part != nullptr) {
      part[(static_cast<int64_t>(blockIdx.y) * M + m) * N + n] = v;
      continue;
    }
    if (bias != nullptr) v += E::to_float(bias[n]);
    C[static_cast<int64_t>(m) * ldc + n] = E::from_float(v);
  }
}

// Sums the split-K partial tiles (of either kernel) in split order, adds the
// bias in fp32 and rounds once: C[m][n] = round(sum_s part[s][m][n] + bias[n]).
// One thread per 4 consecutive columns of a row; 16-byte loads when N % 4 == 0
// (every partial row then starts 16-byte aligned). With S > 0 (= splits) the
// S partial loads and the bias load are issued together before the in-order
// sum: loaded one split at a time, each waited for in turn, the reduce took
// S round trips. S = 0 is the general runtime-count loop.
template <typename E, int S>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ part, int splits, int M,
                                                                 int N, const uint16_t* __restrict__ bias,
                                                                 uint16_t* __restrict__ C, int ldc, int vec_store) {
  const int n4 = (N + 3) / 4;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= static_cast<int64_t>(M) * n4) return;
  const int m = static_cast<int>(idx / n4);
  const int n = static_cast<int>(idx % n4) * 4;
  const int64_t plane = static_cast<int64_t>(M) * N;
  const float* p = part + static_cast<int64_t>(m) * N + n;
  auto load_bias = [&](float (&b)[4]) {  // columns past N are not stored: clamped addresses
    if (bias != nullptr) {
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = E::to_float(bias[min(n + r, N - 1)]);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = 0.0f;
    }
  };
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  float b[4];
  if (S > 0 && N % 4 == 0) {
    f32x4 x[S > 0 ? S : 1];
#pragma unroll
    for (int sp = 0; sp < S; ++sp) x[sp] = *reinterpret_cast<const f32x4*>(p + sp * plane);
    load_bias(b);
#pragma unroll
    for (int sp = 0; sp < S; ++sp)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] += x[sp][r];
  } else if (N % 4 == 0) {
    for (int sp = 0; sp < splits; ++sp) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(p + sp * plane);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] += x[r];
    }
    load_bias(b);
  } else {
    for (int sp = 0; sp < splits; ++sp) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) v[r] += p[sp * plane + r];
    }
    load_bias(b);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] += b[r];
  uint16_t* c = C + static_cast<int64_t>(m) * ldc + n;
  if (vec_store && n + 3 < N) {
    *reinterpret_cast<u32x2*>(c) = u32x2{pack2<E>(v[0], v[1]), pack2<E>(v[2], v[3])};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) c[r] = E::from_float(v[r]);
  }
}

template <typename E>
void launch_splitk_reduce(const float* part, int splits, int M, int N, const uint16_t* bias, uint16_t* C, int ldc,
                          hipStream_t s) {
  const int64_t threads = static_cast<int64_t>(M) * ((N + 3) / 4);
  const dim3 grid(static_cast<unsigned>((threads + 255) / 256));
  const int vec = (ldc % 4 == 0 && aligned_to(C, 8)) ? 1 : 0;
#define DK_REDUCE_CASE(S_)                                                                                 \
  case S_:                                                                                                 \
    hipLaunchKernelGGL((gemm_splitk_reduce_kernel<E, S_>), grid, dim3(256), 0, s, part, splits, M, N, bias, C, \
                       ldc, vec);                                                                          \
    return;
  switch (splits) {
    DK_REDUCE_CASE(2)
    DK_REDUCE_CASE(3)
    DK_REDUCE_CASE(4)
    DK_REDUCE_CASE(5)
    DK_REDUCE_CASE(6)
    DK_REDUCE_CASE(7)
    DK_REDUCE_CASE(8)
    default:
      hipLaunchKernelGGL((gemm_splitk_reduce_kernel<E, 0>), grid, dim3(256), 0, s, part, splits, M, N, bias, C, ldc,
                         vec);
  }
#undef DK_REDUCE_CASE
}

// ---------------------------------------------------------------------------
// LDS-DMA kernel (M > 64)
// ---------------------------------------------------------------------------
// BM x BN output tile per workgroup of WM x WN waves. K advances in 64-column
// slices; a slice of A (BM rows) and of B (BN rows) goes from HBM straight into
// LDS with buffer_load ... lds (16 bytes per lane, one 1 KB instruction per 8
// rows, no registers), through a STAGES-deep ring: slice t + STAGES - 1 is in
// flight while slice t is multiplied. A slice row is 128 bytes = 8 chunks of 16
// bytes, and chunk c of row r is stored at position c ^ (r & 7). gfx950's LDS
// has 64 banks of 4 bytes and serves a ds_read_b128 in four cycles of 16 lanes:
// the lanes that share bit 5 and the parity of bits 2..4 of the lane id
// (measured with SQ_LDS_BANK_CONFLICT on pairs of active lanes). A fragment
// read (lane l: row l % 16, chunk 2 (l / 32) + (l / 16) % 2 + 4 h) puts 8 rows
// with chunk c and 8 rows with chunk c ^ 1 in each such group, and the XOR
// sends those 16 reads to 16 distinct 16-byte bank groups; unswizzled or
// 16-byte-padded rows conflict 2-way. The load lanes fetch the permuted chunks,
// so global reads stay whole 128-byte row segments.
//
// Tiles are numbered so that each XCD (workgroups go to the 8 XCDs round
// robin) takes a contiguous run of them, walked in groups of kGroupM tile rows:
// the ~32 workgroups resident on one XCD share A rows and B rows in its L2.
constexpr int kDmaBK = 64;
constexpr int kXcds = 8;
#ifndef DK_GEMM_GROUP_M
#define DK_GEMM_GROUP_M 4  // tile rows per group of the XCD-contiguous tile order
#endif
constexpr int kGroupM = DK_GEMM_GROUP_M;

__device__ __forceinline__ int swz(int r) { return r & 7; }

template <int BM, int BN>
__device__ __forceinline__ void dma_tile_of(int id, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  int pid = id;
  if (total % kXcds == 0) pid = (id % kXcds) * (total / kXcds) + id / kXcds;
  const int per_group = kGroupM * tiles_n;
  const int first_m = (pid / per_group) * kGroupM;
  const int gm = min(tiles_m - first_m, kGroupM);
  tm = first_m + (pid % per_group) % gm;
  tn = (pid % per_group) / gm;
}

// The order in which a workgroup takes the K slices of [kb, kb + 64 ktiles):
// from slice `rot` on, round to slice rot - 1 (rot = 0: in order).
struct KWalk {
  int kb, end, ktiles, rot;
  // rot_inv: 0, or 2^32 / ktiles rounded up, for column tile tn to start at slice
  // tn mod ktiles (exact for tn ktiles < 2^32; an integer division in every
  // workgroup showed in the shortest calls).
  __device__ __forceinline__ KWalk(int kb_, int ktiles_, int tn, unsigned rot_inv)
      : kb(kb_),
        end(kb_ + ktiles_ * kDmaBK),
        ktiles(ktiles_),
        rot(rot_inv != 0 ? max(0, tn - static_cast<int>(__umulhi(tn, rot_inv)) * ktiles_) : 0) {}
  // First column of the walk's slice t; past the range for t >= ktiles.
  __device__ __forceinline__ int at(int t) const {
    const int r = t + rot;
    return kb + (t < ktiles && r >= ktiles ? r - ktiles : r) * kDmaBK;
  }
  // First column of the slice after the one at column k0 (before the walk's end).
  __device__ __forceinline__ int after(int k0) const { return k0 + kDmaBK == end ? kb : k0 + kDmaBK; }
};

// Bytes of a wave's output tile staged in LDS: 16 TM rows of 16 TN 16-bit
// columns, padded by 16 bytes a row.
template <int TM, int TN>
constexpr int stage_bytes() {
  return 16 * TM * (32 * TN + 16);
}

// Writes a wave's 16 TM x 16 TN output tile at (m0, n0): acc[i][j] lane l, reg
// r = C[m0 + 16 i + l % 16][n0 + 16 j + 4 (l / 16) + r]. With part != nullptr
// the fp32 sums go to part[blockIdx.y][M][N] without the bias; else bias and
// rounding, through LDS. Called by every wave of the workgroup, with no loads
// into LDS in flight; `lds` holds stage_bytes() for each wave.
template <typename E, int TM, int TN>
__device__ __forceinline__ void store_tile(const f32x4 (&acc)[TM][TN], u32x4* lds, int lane, int wave, int m0, int n0,
                                           const uint16_t* __restrict__ bias, uint16_t* __restrict__ C, int M, int N,
                                           int ldc, int vec_store, float* __restrict__ part) {
  constexpr int kPitch = 32 * TN + 16;  // bytes per staged output row
  const int l16 = lane % 16;
  const int lg = lane / 16;
  if (part != nullptr) {  // fp32 partial tile, no bias
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + 16 * j + 4 * lg;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = m0 + 16 * i + l16;
        if (m >= M) continue;
        float* prow = part + (static_cast<int64_t>(blockIdx.y) * M + m) * N;
        if (N % 4 == 0 && n + 3 < N) {
          *reinterpret_cast<f32x4*>(prow + n) = acc[i][j];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < N) prow[n + r] = acc[i][j][r];
        }
      }
    }
    return;
  }

  // Every bias value this lane adds, loaded before any store, with clamped
  // addresses and no branch per element so that the loads issue together.
  // (Loaded one at a time under a bounds branch, each was waited for behind
  // the stores before it: up to 6 us at M = N = 4096.) Columns past N are
  // never stored, so their clamped values do not matter.
  float bj[TN][4];
  if (bias != nullptr) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + 16 * j + 4 * lg;
#pragma unroll
      for (int r = 0; r < 4; ++r) bj[j][r] = E::to_float(bias[min(n + r, N - 1)]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) bj[j][r] = 0.0f;
  }

  // The output goes through LDS: each wave writes its tile into its own part
  // of the allocation in the MFMA layout (8 bytes per lane), then
  // reads it back row by row, 16 bytes per lane, so a store writes whole row
  // segments instead of 32-byte pieces of 16 rows. Rows are padded by 16 bytes.
  constexpr int kNc = 2 * TN;  // 16-byte chunks per tile row
  char* stg = reinterpret_cast<char*>(lds) + wave * stage_bytes<TM, TN>();
  __syncthreads();  // every wave is done with the ring
#pragma unroll
  for (int j = 0; j < TN; ++j) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = 16 * i + l16;
      const int c = 2 * j + lg / 2;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = acc[i][j][r] + bj[j][r];
      *reinterpret_cast<u32x2*>(stg + row * kPitch + c * 16 + (lg % 2) * 8) =
          u32x2{pack2<E>(v[0], v[1]), pack2<E>(v[2], v[3])};
    }
  }
  __syncthreads();  // the tile's rows come from the other lanes of the wave
  if (vec_store <= 0 || (N % 8 != 0 && n0 + 16 * TN > N)) {
    // Rows that allow only 4- or 2-byte stores, and the last columns of an N that
    // is no multiple of a lane's 8: consecutive lanes take consecutive columns, so
    // that a store still writes whole row segments. (As pieces of each lane's own
    // 16 bytes, a store touched 64 pieces of 4 to 8 rows, up to 40% of a call: M,
    // N, K = 1108, 11013, 368 40.0 -> 24.9 us, 3976, 22398, 336 228 -> 132, in 256
    // x 256 tiles; 128 x 128 tiles 1.2 times faster on average, 64 x 64 1.05. In a
    // grid of 2 x 4 waves a row's segment is half as long as in 4 x 2, which had
    // cost another 5%.)
    const auto narrow = [&](auto width) {
      constexpr int kW = decltype(width)::value;  // columns per store
      constexpr int kPerRow = 16 * TN / kW;
#pragma unroll 4
      for (int it = 0; it < 16 * TM * kPerRow / kWave; ++it) {
        const int idx = it * kWave + lane;
        const int row = idx / kPerRow;
        const int c = idx % kPerRow * kW;
        const char* from = stg + row * kPitch + 2 * c;
        const int m = m0 + row;
        const int n = n0 + c;
        if (m >= M || n >= N) continue;
        uint16_t* to = C + static_cast<int64_t>(m) * ldc + n;
        if (kW == 2 && n + 1 < N)
          *reinterpret_cast<uint32_t*>(to) = *reinterpret_cast<const uint32_t*>(from);
        else
          *to = *reinterpret_cast<const uint16_t*>(from);
      }
    };
    if (vec_store >= 0) narrow(std::integral_constant<int, 2>{});
    else narrow(std::integral_constant<int, 1>{});
    return;
  }
  constexpr int kChunks = 16 * TM * kNc;  // 16-byte chunks of a wave's tile
  static_assert(kChunks % kWave == 0, "whole passes");
#pragma unroll
  for (int it = 0; it < kChunks / kWave; ++it) {
    const int idx = it * kWave + lane;
    const int row = idx / kNc;
    const int c = idx % kNc;
    const u32x4 val = *reinterpret_cast<const u32x4*>(stg + row * kPitch + c * 16);
    const int m = m0 + row;
    const int n = n0 + 8 * c;
    if (m >= M || n >= N) continue;
    uint16_t* to = C + static_cast<int64_t>(m) * ldc + n;
    if (vec_store == 2) {
      *reinterpret_cast<u32x4*>(to) = val;
    } else {
      *reinterpret_cast<u32x2*>(to) = u32x2{val[0], val[1]};
      *reinterpret_cast<u32x2*>(to + 4) = u32x2{val[2], val[3]};
    }
  }
}

// The ring body: every wave waits for slice t, meets the others at a barrier,
// starts slice t + STAGES - 1 and multiplies.
template <typename E, int BM, int BN, int WM, int WN, int STAGES>
__device__ __forceinline__ void ring_tile(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                          const uint16_t* __restrict__ bias, uint16_t* __restrict__ C, int M, int N,
                                          int K, int lda, int ldb, int ldc, int vec_store, float* __restrict__ part,
                                          int k_split, unsigned rot_inv) {
  constexpr int NW = WM * WN;
  constexpr int TM = BM / WM / 16;  // 16-row fragments per wave
  constexpr int TN = BN / WN / 16;
  constexpr int LA = BM / 8 / NW;   // 1 KB DMA loads per wave per slice
  // B's 8-row load groups need not divide among the waves (128 x 160: 20 groups
  // for 8 waves). A wave past the last group issues a load that moves nothing,
  // aimed at a spare 1 KB, so that every wave has the same count in flight.
  constexpr int kGroupsB = BN / 8;
  constexpr int LB = (kGroupsB + NW - 1) / NW;
  constexpr bool kTailB = kGroupsB % NW != 0;
  constexpr int kSlice = (BM + BN) * 8;  // u32x4 per slice
  static_assert(BM % (8 * NW) == 0 && BN % 8 == 0 && TM >= 1 && TN >= 1 && BN % (16 * WN) == 0, "tile shape");
  static_assert(STAGES >= 2 && (STAGES - 2) * (LA + LB) < 64, "vmcnt range");
  constexpr int kStageWave = stage_bytes<TM, TN>();
  constexpr int kRingU4 = STAGES * kSlice + (kTailB ? 64 : 0);
  constexpr int kLdsU4 = kRingU4 > NW * kStageWave / 16 ? kRingU4 : NW * kStageWave / 16;
  static_assert(kLdsU4 * 16 <= 160 * 1024, "LDS of one workgroup (gfx950: 160 KB)");
  __shared__ u32x4 lds[kLdsU4];

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave % WM;
  const int wn = wave / WM;
  const int l16 = lane % 16;
  const int lg = lane / 16;

  // Split-K (part != nullptr): workgroup row blockIdx.y covers K columns
  // [kb, ke) (k_split a multiple of kDmaBK) and writes its fp32 partial tile to
  // part[blockIdx.y][M][N], without the bias; gemm_splitk_reduce_kernel sums them.
  const int kb = part != nullptr ? static_cast<int>(blockIdx.y) * k_split : 0;
  const int ke = part != nullptr ? min(K, kb + k_split) : K;
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = (N + BN - 1) / BN;
  int tm, tn;
  dma_tile_of<BM, BN>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM;
  const int n0 = tn * BN;
  const int rows_a = min(BM, M - m0);
  const int rows_b = min(BN, N - n0);
  // Rows past M (N) lie past num_records and read as zero.
  const __amdgpu_buffer_rsrc_t ra =
      rsrc(A + static_cast<int64_t>(m0) * lda, (static_cast<int64_t>(rows_a - 1) * lda + K) * 2);
  const __amdgpu_buffer_rsrc_t rb =
      rsrc(B + static_cast<int64_t>(n0) * ldb, (static_cast<int64_t>(rows_b - 1) * ldb + K) * 2);

  // DMA lane roles: load j of this wave fills tile rows 8 g .. 8 g + 7 (g = wave + j NW);
  // lane l writes position l % 8 of row 8 g + l / 8, i.e. chunk (l % 8) ^ swz(row) = (l % 8) ^ (l / 8).
  const int kc = 8 * ((lane % 8) ^ (lane / 8));  // first column of this lane's 16 bytes in a slice
  unsigned offa[LA], offb[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int r = 8 * (wave + j * NW) + lane / 8;
    offa[j] = r < rows_a ? static_cast<unsigned>(r * lda * 2 + 2 * kc) : kNowhere;
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    const int r = 8 * (wave + j * NW) + lane / 8;
    offb[j] = r < rows_b && r < BN ? static_cast<unsigned>(r * ldb * 2 + 2 * kc) : kNowhere;
  }
  const int ktiles = (ke - kb + kDmaBK - 1) / kDmaBK;
  const int full = (ke - kb) / kDmaBK;  // slices that lie wholly inside the K range
  const KWalk walk(kb, ktiles, tn, rot_inv);
  // The slice at column k0 into ring buffer `buf`. Checked: also for slices that
  // end past the K range, or start there (those lanes are out of range and move
  // no data), so that each wave keeps the same count in flight from slice to
  // slice. Whole slices need one addition per load (rows past M or N stay out
  // of range: kNowhere + 2 k0 is still above every resource's extent), and `k0`
  // steps with the walk (a compare and a select per slice). With the K offset
  // as the loads' scalar offset instead, as in the ping-pong body, the larger
  // tiles were 1-6% slower (us): 128 x 128 at M, N, K = 192, 16384, 3072 36.4
  // against 34.3 and at 768, 3584, 3584 36.5 against 34.9. The uneven 128 x 160
  // tile keeps the scalar offset: at 1003, 4608, 3584 38.2 against 41.0 with warm
  // weights, though 43.4 against 42.5 with cold ones.
  constexpr bool kScalarK = kTailB;
  auto issue = [&](bool checked, int k0, int buf) {
    const bool scalar = kScalarK && !checked;
    u32x4* base = lds + buf * kSlice;
    const unsigned out = checked && k0 + kc >= ke ? kNowhere : 0;  // or-ed in: a choice per load became a branch
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      const int off = static_cast<int>(scalar ? offa[j] : (offa[j] + 2 * k0) | out);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          ra, (__attribute__((address_space(3))) void*)(base + (wave + j * NW) * 64), 16, off, scalar ? 2 * k0 : 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      u32x4* to = base + BM * 8 + (wave + j * NW) * 64;
      if (kTailB && j == LB - 1 && wave + j * NW >= kGroupsB) to = lds + STAGES * kSlice;  // (offb is out of range)
      const int off = static_cast<int>(scalar ? offb[j] : (offb[j] + 2 * k0) | out);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)to, 16, off,
                                               scalar ? 2 * k0 : 0, 0, 0);
    }
  };

  // Fragment read offsets (u32x4) inside a slice, for the two 32-column halves.
  int ia[TM][2], ib[TN][2];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = wm * (BM / WM) + 16 * i + l16;
    ia[i][0] = r * 8 + (lg ^ swz(r));
    ia[i][1] = r * 8 + ((4 + lg) ^ swz(r));
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int r = wn * (BN / WN) + 16 * j + l16;
    ib[j][0] = BM * 8 + r * 8 + (lg ^ swz(r));
    ib[j][1] = BM * 8 + r * 8 + ((4 + lg) ^ swz(r));
  }

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) issue(true, walk.at(s), s);

  // vmcnt(n) with expcnt / lgkmcnt left at their maxima (gfx9 encoding).
  constexpr int kWaitN = (STAGES - 2) * (LA + LB);
  constexpr int kWaitImm = (kWaitN & 15) | ((kWaitN >> 4) << 14) | (7 << 4) | (15 << 8);

  // The next slice, in ring buffer u; the loads of the slice STAGES - 1 later start at column k0.
  auto step = [&](bool checked, int k0, int u) {
    // This wave's loads of the slice have landed; the barrier extends that to
    // every wave and ensures all reads of the buffer refilled next are done.
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitImm);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    issue(checked, k0, (u + STAGES - 1) % STAGES);
    const u32x4* sl = lds + u * kSlice;
    // Small tiles read both halves' fragments before the first MFMA, one LDS
    // round trip a slice instead of two: o_proj at M = 250 (64 x 64) 16.4 -> 15.6
    // us, qkv at M = 512 (128 x 128) 32.9 -> 30.8. Larger ones have no registers
    // for it.
    constexpr int kHalves = TM + TN <= 7 ? 2 : 1;
    u32x4 af[kHalves][TM], bf[kHalves][TN];
    auto read = [&](int h) {
#pragma unroll
      for (int i = 0; i < TM; ++i) af[h % kHalves][i] = sl[ia[i][h]];
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[h % kHalves][j] = sl[ib[j][h]];
    };
    if (kHalves == 2) {
      read(0);
      read(1);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (kHalves == 1) read(h);
      // A wave that has its fragments issues its MFMAs ahead of the other
      // wave on the SIMD, which meanwhile reads its own: the two drift
      // out of phase instead of reading and multiplying in lockstep
      // (measured 1-4% at M = 1024 / 4096).
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = E::mfma_16x16x32(bf[h % kHalves][j], af[h % kHalves][i], acc[i][j]);
      __builtin_amdgcn_s_setprio(0);
    }
  };
  int t0 = 0;
  int k0 = walk.at(STAGES - 1);
  for (; t0 + 2 * STAGES - 2 < full; t0 += STAGES) {
#pragma unroll
    for (int u = 0; u < STAGES; ++u) {
      step(false, k0, u);
      k0 = walk.after(k0);
    }
  }
  for (; t0 < ktiles; t0 += STAGES) {
#pragma unroll
    for (int u = 0; u < STAGES; ++u)
      if (t0 + u < ktiles) step(true, walk.at(t0 + u + STAGES - 1), u);
  }

  // The loads issued past the last slice move no data, but none may still be
  // in flight into this workgroup's LDS when it exits.
  __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));

  store_tile<E, TM, TN>(acc, lds, lane, wave, m0 + wm * (BM / WM), n0 + wn * (BN / WN), bias, C, M, N, ldc, vec_store, part);
}

// ---------------------------------------------------------------------------
// Ping-pong body (256-row and 256-column tiles)
// ---------------------------------------------------------------------------
// The ring body reads a slice's fragments and multiplies them in turn, every
// wave at once: per 256 x 256 slice the LDS reads and the MFMAs each take
// about 2000 cycles, and 4000 passed. Here the two waves of a SIMD alternate:
// while one multiplies (16 MFMAs, raised priority) the other reads its next
// fragments and starts its share of the loads, with a barrier at every swap.
// Waves 4-7 run one barrier behind waves 0-3.
//
// A slice's A and B are kept as two halves each: half i holds, for every wave
// row (column) of the grid, its i-th 1/2 of the rows (columns), so a wave's
// tile is four quadrants A_i x B_j and a slice four phases:
//   read A0, x B0 | read B1, A0 x B1 | read A1, A1 x B1 | read the next B0, A1 x B0.
// A half is refilled for slice t + 2 in the phase after the one that read it
// last (B0, A0, B1, A1 in turn, one half per phase), so each load has seven
// phases to land and the wait before each barrier leaves the newest six halves
// in flight. Both hazards are closed by the barriers: a wave waits for its own
// reads (lgkmcnt(0)) and for its own loads of the half read next (vmcnt)
// before the first barrier of a phase, and the wave one barrier behind has
// passed that wait before the other enters its next phase.
//
// What bounds it is the phase's memory part, so it holds nothing but the
// reads, the loads and their LDS addresses: a whole slice's K offset is the
// loads' scalar offset (with it in the vector offset, and compared with the K
// range per lane, the 256 x 256 tile took 674 us on gate_up at M = 4096, with
// the ring body 741; now 643, hipBLASLt 641, same run). M = N = 4096: K = 4096
// 112.5 -> 93.2 us, K = 14336 383 -> 346 us. Waiting for the reads only when
// they are used, without the raised priority, with the loads in two phases
// instead of four, or starting each XCD at another K offset were all within 1%.

// A barrier that neither LDS reads nor loads into LDS are moved across.
__device__ __forceinline__ void pp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Waits for this wave's fragment reads and until at most VM of its loads into
// LDS are in flight, then for the other waves.
template <int VM>
__device__ __forceinline__ void pp_wait_barrier() {
  static_assert(VM < 64, "vmcnt range");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4));
  pp_barrier();
}

template <typename E, int BM, int BN, int WM, int WN>
__device__ __forceinline__ void ping_pong_tile(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                               const uint16_t* __restrict__ bias, uint16_t* __restrict__ C, int M,
                                               int N, int K, int lda, int ldb, int ldc, int vec_store,
                                               float* __restrict__ part, int k_split, unsigned rot_inv) {
  constexpr int NW = WM * WN;
  static_assert(NW == 8, "two waves per SIMD, one of each half of the workgroup");
  constexpr int QR = BM / 2 / WM;  // rows of A (of B) of one half that a wave multiplies
  constexpr int QC = BN / 2 / WN;
  constexpr int QM = QR / 16;      // 16-row fragments of a half per wave
  constexpr int QN = QC / 16;
  static_assert(QR % 16 == 0 && QC % 16 == 0 && QM >= 1 && QN >= 1, "tile shape");
  constexpr int kGroupsA = BM / 16;  // 8-row load groups of a half
  constexpr int kGroupsB = BN / 16;
  constexpr int LA = (kGroupsA + NW - 1) / NW;
  constexpr int LB = (kGroupsB + NW - 1) / NW;
  constexpr bool kTail = kGroupsA % NW != 0 || kGroupsB % NW != 0;
  constexpr int kHalfA = BM / 2 * 8;  // u32x4 of a half
  constexpr int kHalfB = BN / 2 * 8;
  constexpr int kSlice = 2 * (kHalfA + kHalfB);
  constexpr int kStage = NW * stage_bytes<2 * QM, 2 * QN>() / 16;
  constexpr int kRing = 2 * kSlice + (kTail ? 64 : 0);
  constexpr int kLdsU4 = kRing > kStage ? kRing : kStage;
  static_assert(kLdsU4 * 16 <= 160 * 1024, "LDS of one workgroup (gfx950: 160 KB)");
  __shared__ u32x4 lds[kLdsU4];

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / WN;
  const int wn = wave % WN;
  const int l16 = lane % 16;
  const int lg = lane / 16;

  const int kb = part != nullptr ? static_cast<int>(blockIdx.y) * k_split : 0;
  const int ke = part != nullptr ? min(K, kb + k_split) : K;
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = (N + BN - 1) / BN;
  int tm, tn;
  dma_tile_of<BM, BN>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM;
  const int n0 = tn * BN;
  const int rows_a = min(BM, M - m0);
  const int rows_b = min(BN, N - n0);
  const __amdgpu_buffer_rsrc_t ra =
      rsrc(A + static_cast<int64_t>(m0) * lda, (static_cast<int64_t>(rows_a - 1) * lda + K) * 2);
  const __amdgpu_buffer_rsrc_t rb =
      rsrc(B + static_cast<int64_t>(n0) * ldb, (static_cast<int64_t>(rows_b - 1) * ldb + K) * 2);

  const int kc = 8 * ((lane % 8) ^ (lane / 8));  // first column of this lane's 16 bytes in a slice (the swizzle)
  unsigned offa[2][LA], offb[2][LB];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      const int rr = 8 * (wave + j * NW) + lane / 8;
      const int r = rr / QR * (2 * QR) + i * QR + rr % QR;
      offa[i][j] = rr < 8 * kGroupsA && r < rows_a ? static_cast<unsigned>(r * lda * 2 + 2 * kc) : kNowhere;
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int rr = 8 * (wave + j * NW) + lane / 8;
      const int r = rr / QC * (2 * QC) + i * QC + rr % QC;
      offb[i][j] = rr < 8 * kGroupsB && r < rows_b ? static_cast<unsigned>(r * ldb * 2 + 2 * kc) : kNowhere;
    }
  }
  const int ktiles = (ke - kb + kDmaBK - 1) / kDmaBK;
  const int full = (ke - kb) / kDmaBK;
  const KWalk walk(kb, ktiles, tn, rot_inv);
  // The loads of half `i` of the slice at column k0 into buffer `buf`. Checked:
  // also for slices that end past the K range (or start there: nothing is moved).
  auto issue_a = [&](bool checked, int k0, int buf, int i) {
    u32x4* base = lds + buf * kSlice + i * kHalfA;
    const bool in = k0 + kc < ke;
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      const int off = static_cast<int>(checked ? (in ? offa[i][j] + 2 * k0 : kNowhere) : offa[i][j]);
      u32x4* to = wave + j * NW < kGroupsA ? base + (wave + j * NW) * 64 : lds + 2 * kSlice;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)to, 16, off,
                                               checked ? 0 : 2 * k0, 0, 0);
    }
  };
  auto issue_b = [&](bool checked, int k0, int buf, int i) {
    u32x4* base = lds + buf * kSlice + 2 * kHalfA + i * kHalfB;
    const bool in = k0 + kc < ke;
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int off = static_cast<int>(checked ? (in ? offb[i][j] + 2 * k0 : kNowhere) : offb[i][j]);
      u32x4* to = wave + j * NW < kGroupsB ? base + (wave + j * NW) * 64 : lds + 2 * kSlice;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)to, 16, off,
                                               checked ? 0 : 2 * k0, 0, 0);
    }
  };

  const int fa = (wm * QR + l16) * 8 + (lg ^ (l16 & 7));
  const int fb = (wn * QC + l16) * 8 + (lg ^ (l16 & 7));
  auto read_a = [&](int buf, int i, u32x4 (&f)[QM][2]) {
    const u32x4* base = lds + buf * kSlice + i * kHalfA;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < QM; ++q) f[q][h] = base[(fa ^ (4 * h)) + 128 * q];
  };
  auto read_b = [&](int buf, int i, u32x4 (&f)[QN][2]) {
    const u32x4* base = lds + buf * kSlice + 2 * kHalfA + i * kHalfB;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < QN; ++q) f[q][h] = base[(fb ^ (4 * h)) + 128 * q];
  };

  f32x4 acc[2 * QM][2 * QN];
#pragma unroll
  for (int i = 0; i < 2 * QM; ++i)
#pragma unroll
    for (int j = 0; j < 2 * QN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 af[QM][2], b1[QN][2], bx[QN][2], by[QN][2];

  auto multiply = [&](int i, int j, const u32x4 (&b)[QN][2]) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < QM; ++q)
#pragma unroll
        for (int r = 0; r < QN; ++r)
          acc[i * QM + q][j * QN + r] = E::mfma_16x16x32(b[r][h], af[q][h], acc[i * QM + q][j * QN + r]);
    __builtin_amdgcn_s_setprio(0);
  };

  // Six of a slice's eight half loads stay in flight (see above).
  auto mem_done = [&]() { pp_wait_barrier<3 * (LA + LB)>(); };
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    issue_b(true, walk.at(s), s, 0);
    issue_a(true, walk.at(s), s, 0);
    issue_b(true, walk.at(s), s, 1);
    issue_a(true, walk.at(s), s, 1);
  }
  mem_done();  // halves B0 and A0 of slice 0 are in LDS
  read_b(0, 0, bx);
  mem_done();
  if (wave >= NW / 2) pp_barrier();

  // One K slice from buffer `buf`, which the slice at column k0 refills; b0
  // holds its B0 fragments, those of the next slice go to bn.
  auto slice = [&](bool checked, int k0, int buf, const u32x4 (&b0)[QN][2], u32x4 (&bn)[QN][2]) {
    read_a(buf, 0, af);
    issue_b(checked, k0, buf, 0);
    mem_done();
    multiply(0, 0, b0);
    pp_barrier();
    read_b(buf, 1, b1);
    issue_a(checked, k0, buf, 0);
    mem_done();
    multiply(0, 1, b1);
    pp_barrier();
    read_a(buf, 1, af);
    issue_b(checked, k0, buf, 1);
    mem_done();
    multiply(1, 1, b1);
    pp_barrier();
    read_b(buf ^ 1, 0, bn);
    issue_a(checked, k0, buf, 1);
    mem_done();
    multiply(1, 0, b0);
    pp_barrier();
  };
  int t = 0;
  int k0 = walk.at(2);
  for (; t + 3 < full; t += 2) {
    slice(false, k0, 0, bx, by);
    k0 = walk.after(k0);
    slice(false, k0, 1, by, bx);
    k0 = walk.after(k0);
  }
  for (; t < ktiles; t += 2) {
    slice(true, walk.at(t + 2), 0, bx, by);
    if (t + 1 < ktiles) slice(true, walk.at(t + 3), 1, by, bx);
  }
  if (wave < NW / 2) pp_barrier();

  // The loads issued past the last slice move no data, but none may still be
  // in flight into this workgroup's LDS when it is used again.
  __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
  store_tile<E, 2 * QM, 2 * QN>(acc, lds, lane, wave, m0 + wm * 2 * QR, n0 + wn * 2 * QC, bias, C, M, N, ldc, vec_store,
                                part);
}

// 2-stage tiles (256 x 256, 256 x 192, 192 x 256, 256 x 128, 128 x 256) run the
// ping-pong body, the others the ring.
// Two waves per SIMD as the register target, also where the LDS allows one: with
// the whole register file the compiler keeps the sums of the 4-wave tiles in
// accumulation registers and moves them back and forth each slice (64 x 64: 36
// ns a slice, 5.6 -> 6.1 us at N = K = 896).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wpass-failed"
template <typename E, int BM, int BN, int WM, int WN, int STAGES>
__global__ __launch_bounds__(WM * WN * kWave, 2) void gemm_dma_kernel(const uint16_t* __restrict__ A,
                                                                   const uint16_t* __restrict__ B,
                                                                   const uint16_t* __restrict__ bias,
                                                                   uint16_t* __restrict__ C, int M, int N, int K,
                                                                   int lda, int ldb, int ldc, int vec_store,
                                                                   float* __restrict__ part, int k_split, unsigned rot_inv) {
  if constexpr (STAGES == 2)
    ping_pong_tile<E, BM, BN, WM, WN>(A, B, bias, C, M, N, K, lda, ldb, ldc, vec_store, part, k_split, rot_inv);
  else
    ring_tile<E, BM, BN, WM, WN, STAGES>(A, B, bias, C, M, N, K, lda, ldb, ldc, vec_store, part, k_split, rot_inv);
}
#pragma clang diagnostic pop

// With part != nullptr the K splits write fp32 partial tiles; `reduce` then
// launches gemm_splitk_reduce_kernel, otherwise the caller consumes them.
template <typename E, int BM, int BN, int WM, int WN, int STAGES>
hipError_t launch_dma(const uint16_t* A, const uint16_t* B, const uint16_t* bias, uint16_t* C, int M, int N, int K,
                      int lda, int ldb, int ldc, hipStream_t s, float* part, int splits, int k_split, bool reduce, int rot_step) {
  const int64_t tiles = ceil_div64(M, BM) * ceil_div64(N, BN);
  const unsigned rot_inv = rot_step != 0 ? static_cast<unsigned>(ceil_div64(int64_t{1} << 32, K / kDmaBK)) : 0;
  // Output stores of 16 bytes (2), or 8 (1), 4 (0) or 2 (-1) where C's rows allow only that.
  const int vec = (ldc % 8 == 0 && aligned_to(C, 16))  ? 2
                  : (ldc % 4 == 0 && aligned_to(C, 8)) ? 1
                  : (ldc % 2 == 0 && aligned_to(C, 4)) ? 0
                                                       : -1;
  hipLaunchKernelGGL((gemm_dma_kernel<E, BM, BN, WM, WN, STAGES>),
                     dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(part != nullptr ? splits : 1)),
                     dim3(WM * WN * kWave), 0, s, A, B, bias, C, M, N, K, lda, ldb, ldc, vec, part,
                     part != nullptr ? k_split : K, rot_inv);
  if (part == nullptr || !reduce) return hipGetLastError();
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  launch_splitk_reduce<E>(part, splits, M, N, bias, C, ldc, s);
  return hipGetLastError();
}

using DmaLauncher = hipError_t (*)(const uint16_t*, const uint16_t*, const uint16_t*, uint16_t*, int, int, int, int,
                                   int, int, hipStream_t, float*, int, int, bool, int);

// Launchers of kTiles' tile shapes, in the same order. The waves of the 256 x
// 256 tile form a 2 x 4 grid (0-2% faster than 4 x 2).
template <typename E>
const DmaLauncher* tile_launchers() {
  static const DmaLauncher fns[] = {
      launch_dma<E, 256, 256, 2, 4, 2>, launch_dma<E, 256, 192, 4, 2, 2>, launch_dma<E, 192, 256, 2, 4, 2>,
      launch_dma<E, 256, 128, 4, 2, 2>, launch_dma<E, 128, 256, 2, 4, 2>, launch_dma<E, 128, 128, 4, 2, 3>,
      launch_dma<E, 128, 160, 4, 2, 4>, launch_dma<E, 128, 64, 2, 2, 4>,  launch_dma<E, 64, 64, 2, 2, 4>,
      launch_dma<E, 64, 128, 2, 2, 4>,  launch_dma<E, 192, 192, 4, 2, 3>,
  };
  return fns;
}

#ifndef DK_SKINNY_DEPTH
#define DK_SKINNY_DEPTH 2  // k-steps of weights and activations in flight per wave
#endif
#ifndef DK_SKINNY_MIN_WGS
#define DK_SKINNY_MIN_WGS 192  // wide plan (N > 32768): fewest workgroups the N split may leave, M > 16
#endif
#ifndef DK_SKINNY_MIN_WGS_M16
#define DK_SKINNY_MIN_WGS_M16 384  // the same for M <= 16
#endif

// Launch shape of the skinny kernel: MT 16-row activation tiles, WN x WK
// waves per workgroup (WN along N, 16 columns each; WK along K), and, with a
// workspace, the K reduction split over `splits` workgroup rows of k_split
// columns each.
struct SkinnyPlan {
  int mt, wn, wk, splits, k_split;
};

// Plan of grids with more than one workgroup per CU (N > 32768): as many waves
// along N as keep >= 384 (M <= 16) or >= 192 workgroups, the rest along K.
inline SkinnyPlan skinny_plan_wide(int M, int N, int K) {
  SkinnyPlan p{};
  p.mt = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
  const int min_wgs = p.mt == 1 ? DK_SKINNY_MIN_WGS_M16 : DK_SKINNY_MIN_WGS;
  p.wn = (M > 32 && N >= 24576) ? 8 : (N >= 64 * min_wgs ? 4 : (N >= 32 * min_wgs ? 2 : 1));
  p.wk = 8 / p.wn;
  p.splits = 1;
  p.k_split = K;
  return p;
}

// Workgroup shapes (WN, WK) of the plans below, narrowest first.
constexpr int kSkinnyShapes[][2] = {{1, 8}, {2, 4}, {4, 2}, {6, 2}, {7, 2}, {8, 1}};
constexpr int kSkinnyShapeCount = static_cast<int>(sizeof(kSkinnyShapes) / sizeof(kSkinnyShapes[0]));
constexpr int kSkinnyCus = 256;

// The widest unsplit grid that fits one workgroup per CU (the narrowest shape
// with <= 256 column tiles); wn = 0 when none does.
inline SkinnyPlan skinny_plan_unsplit(int M, int N, int K) {
  SkinnyPlan p{};
  p.mt = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
  p.splits = 1;
  p.k_split = K;
  for (const auto& sh : kSkinnyShapes) {
    if (ceil_div64(N, 16 * sh[0]) <= kSkinnyCus) {
      p.wn = sh[0];
      p.wk = sh[1];
      return p;
    }
  }
  return p;
}

// Every workgroup re-reads the activation rows of its K range (M x k_split
// elements) for its 16 WN x k_split weights, so wide column tiles cut that
// traffic; splitting K over workgroup rows then keeps the grid at the CU
// count, at the price of an fp32 partial tile per split and a second kernel
// that sums them. The plan, fitted to interleaved cold timings of every
// candidate shape at M = 1 ... 64 on the Llama-3-8B projections (bf16,
// MI355X):
//  1. the widest unsplit grid of at most one workgroup per CU, if it fills
//     >= 3/4 of the CUs and each workgroup re-reads <= 256 KiB of activations;
//  2. else, with a workspace, the grids of 2 ... 8 K splits (>= 512 columns
//     each, <= 256 workgroups) within 10% of the fullest one: the fewest
//     splits whose workgroups re-read at most max(128 KiB, half their weight
//     bytes) of activations, or failing that the fewest activation bytes;
//  3. else the unsplit grid of 1, or for N > 32768 (no grid of one workgroup
//     per CU) the wide plan.
// A 257th workgroup puts two on one CU and doubles that CU's time. Where 64-row
// tiles are faster, they run instead (decode_plan).
inline SkinnyPlan skinny_plan(int M, int N, int K, bool split_ok) {
  constexpr int64_t kKiB = 1024;
  SkinnyPlan u = skinny_plan_unsplit(M, N, K);
  if (u.wn > 0 && static_cast<int64_t>(M) * K * 2 <= 256 * kKiB &&
      4 * ceil_div64(N, 16 * u.wn) >= 3 * kSkinnyCus)
    return u;
  if (split_ok && K > 0) {
    struct Cand {
      int wn, wk, splits, k_split;
      int64_t wgs;
    };
    Cand cand[kSkinnyShapeCount * 7];
    int nc = 0;
    int64_t max_wgs = 0;
    for (const auto& sh : kSkinnyShapes) {
      const int64_t tiles = ceil_div64(N, 16 * sh[0]);
      for (int s = 2; s <= 8; ++s) {
        if (K / s < 512) break;
        const int per = (K + s - 1) / s;
        const int ks = (per + kLdsBK - 1) / kLdsBK * kLdsBK;
        if ((K + ks - 1) / ks != s) continue;  // every split non-empty
        if (tiles * s > kSkinnyCus) break;
        cand[nc++] = Cand{sh[0], sh[1], s, ks, tiles * s};
        max_wgs = std::max(max_wgs, tiles * s);
      }
    }
    const Cand* best = nullptr;
    bool best_ok = false;
    for (int i = 0; i < nc; ++i) {
      const Cand& c = cand[i];
      if (10 * c.wgs < 9 * max_wgs) continue;  // within 10% of the fullest grid
      const int64_t act = static_cast<int64_t>(M) * c.k_split * 2;
      const int64_t wts = int64_t{16} * c.wn * c.k_split * 2;
      const bool ok = act <= std::max<int64_t>(128 * kKiB, wts / 2);
      if (best == nullptr || (ok && !best_ok)) {
        best = &c;
        best_ok = ok;
        continue;
      }
      if (ok != best_ok) continue;
      const int64_t best_act = static_cast<int64_t>(M) * best->k_split;
      const bool better = ok ? (c.splits < best->splits)
                             : (static_cast<int64_t>(M) * c.k_split < best_act ||
                                (static_cast<int64_t>(M) * c.k_split == best_act && c.splits < best->splits));
      if (better) best = &c;
    }
    if (best != nullptr) {
      SkinnyPlan p = u;
      p.wn = best->wn;
      p.wk = best->wk;
      p.splits = best->splits;
      p.k_split = best->k_split;
      return p;
    }
  }
  return u.wn > 0 ? u : skinny_plan_wide(M, N, K);
}

// What a call runs: tile `shape` of kTiles, or (shape < 0) the skinny kernel
// with wn x wk waves; K split over workgroup rows of k_split columns.
struct Plan {
  int shape, wn, wk, splits, k_split, rot_step;
};

// Largest split-K workspace a tiled plan asks for (bytes); larger splits are not considered.
constexpr int64_t kMaxWorkspace = int64_t{64} << 20;

inline int64_t plan_workspace_bytes(const Plan& p, int M, int N) {
  return p.splits > 1 ? static_cast<int64_t>(p.splits) * M * N * static_cast<int64_t>(sizeof(float)) : 0;
}

// K-walk rotation (see gemm_skinny_lds_kernel): column tile j starts its walk
// j slices in. With one tile row every weight byte is read by one workgroup,
// and spreading the walks spreads the reads over the HBM channels where rows
// are a few KB apart: gate_up (N 28672, K 4096) at M = 64 / 128 / 250 52.4 / 57.8 /
// 69.5 -> 42.2 / 50.0 / 62.5 us, N = 128256 at M = 16 219 -> 176. By K, over ten
// tiles and eight widths: 0.91-0.93 of the time in order at 2048, 4096, 6144,
// 8192 and 16384, 0.97-0.99 at 1536, 2560, 3072, 3584, 9216, 1.00 up to 1024
// (N 9728, K 1024 at M = 65 9.4 -> 10.0). With more tile rows, whose workgroups
// share weight rows, and below 128 workgroups it measured 0-4% slower.
inline int rotation(int64_t tiles_m, int64_t tiles_n, int splits, int K) {
  return splits == 1 && tiles_m == 1 && tiles_n >= 128 && K >= 1536 && K % kDmaBK == 0 ? 1 : 0;
}

// Time model that picks what a call runs, in us. A grid of W workgroups, each
// of n slices of 64 columns, takes
//   ceil(W / 256) x (n x slice + tile)
// with `ragged` for `slice` where K % 64 != 0 (rows then start off 128-byte lines, and
// a slice's row segments lie in two), and a K split adds
//   split + splits x M x N x 8 B / partials
// (the fp32 partials written and read back; times `odd` where N % 4 != 0, whose
// partial rows are stored and read in 4-byte pieces). Candidates: every tile
// shape with 1, 2, 3, 4, 6 and 8 splits (at least 512 columns each, at most 256
// tiles and 768 workgroups, partials within kMaxWorkspace). Constants are fitted
// for the best picks, not the best times (so `slice` and `tile` are no
// measurements), to calls with weights and activations cold in every cache,
// the state that a layer's weights are in. Fitted to three sets of operands in
// turn, which the last-level cache holds up to 85 MB each, a model misjudges
// HBM-bound calls: down of Llama-3-8B (N 4096, K 14336) at M = 64 / 256 took 30.7 /
// 51.2 us with such picks (64 x 64 in 4 splits, 128 x 128 in 4), 29.6 / 48.7 with
// these.
struct TimeModel {
  double split, partials, odd;
};
struct TileShape {
  int bm, bn;
  double slice_us, ragged_us, tile_us;
};

inline double split_us(const TimeModel& m, int splits, int M, int N) {
  if (splits == 1) return 0.0;
  return m.split + splits * (static_cast<double>(M) * N) * 8.0 / m.partials * (N % 4 != 0 ? m.odd : 1.0);
}

// Takes the fastest of `best` (at best_t, if >= 0) and the candidates of tile shape `i` with costs `sh`.
inline void try_tile(const TimeModel& m, const TileShape& sh, int i, int M, int N, int K, bool split_ok, Plan& best,
                     double& best_t) {
  const int64_t tiles_m = ceil_div64(M, sh.bm);
  const int64_t tiles = tiles_m * ceil_div64(N, sh.bn);
  for (const int s : {1, 2, 3, 4, 6, 8}) {
    int ks = K;
    if (s > 1) {
      if (!split_ok || tiles > kSkinnyCus || tiles * s > 3 * kSkinnyCus || K / s < 512 ||
          static_cast<int64_t>(s) * M * N * static_cast<int64_t>(sizeof(float)) > kMaxWorkspace)
        break;
      ks = ((K + s - 1) / s + kDmaBK - 1) / kDmaBK * kDmaBK;
      if ((K + ks - 1) / ks != s) continue;  // every split non-empty
    }
    const double n = static_cast<double>((ks + kDmaBK - 1) / kDmaBK);
    const double slice = K % kDmaBK == 0 ? sh.slice_us : sh.ragged_us;
    const double t = static_cast<double>(ceil_div64(tiles * s, kSkinnyCus)) * (n * slice + sh.tile_us) +
                     split_us(m, s, M, N);
    if (best_t < 0 || t < best_t) {
      best = Plan{i, 0, 0, s, ks, rotation(tiles_m, ceil_div64(N, sh.bn), s, K)};
      best_t = t;
    }
  }
}

// M > 64. Fitted to 2252 (M, N, K): the projections of Llama-3-8B, Qwen2.5-7B,
// Qwen2.5-0.5B and Phi-3 at M = 65 ... 4096 and 1300 drawn ones, every candidate
// timed. The pick is 0.8% slower than the fastest candidate on average (1% on
// sizes left out of a fit, 17% at most for a projection). Against a plan of nine
// tiles in the ring body alone, fitted to three projections, 0.927 of the time
// (geometric mean), more than 5% slower at 22 sizes (10% at most); against a
// model fitted to warm calls whose splits that plan capped, 0.956, more than 5%
// slower at 32 (16%).
constexpr TimeModel kTileModel{2.7, 6.28e6, 3.53};
constexpr TileShape kTiles[] = {
    {256, 256, 1.18, 1.52, 9.44},   {256, 192, 0.962, 1.26, 10.7},  {192, 256, 0.971, 1.26, 9.13},
    {256, 128, 0.716, 1.21, 6.41},  {128, 256, 0.883, 1.24, 7.19},  {128, 128, 0.509, 0.847, 4.19},
    {128, 160, 0.638, 0.909, 6.5},  {128, 64, 0.395, 0.706, 2.53},  {64, 64, 0.283, 0.442, 1.33},
    {64, 128, 0.365, 0.678, 5.48},  {192, 192, 0.894, 1.23, 6.33},
};
constexpr int kTileCount = static_cast<int>(sizeof(kTiles) / sizeof(kTiles[0]));
constexpr int kTile64x64 = 8, kTile64x128 = 9;  // their places in kTiles

inline Plan tile_plan(int M, int N, int K, bool split_ok) {
  Plan best{0, 0, 0, 1, K, 0};
  double best_t = -1.0;
  for (int i = 0; i < kTileCount; ++i) try_tile(kTileModel, kTiles[i], i, M, N, K, split_ok, best, best_t);
  return best;
}

// M <= 64: the skinny plan or a 64-row tile of 64 (4 waves, two workgroups per
// CU) or 128 columns (4 waves, one per CU). The skinny plan is modelled as
//   1.26 + max(1, W / 256) x (n x step + base) [+ the split],
// n slices per wave, `step` by workgroup shape (kSkinnyShapes) times a factor by
// row tiles, `base` by row tiles (M <= 16, <= 32, <= 64). Where no skinny grid
// fits one workgroup per CU (N > 32768), a tile runs at every M: of N 128256, K
// 4096 at M = 16 the grid of 8 x 1 waves took 180 us, 64 x 128 177. Fitted like
// kTiles, to 755 (M, N, K), M = 1 ... 64: the pick is 0.8% slower than the fastest
// of the three kinds on average. Against a plan that took the fewest weight bytes per
// workgroup from M = 32 on: 0.986 of the time, more than 5% slower at 15 sizes,
// none of them a projection (2.4% at most). Llama-3-8B gate_up (N 28672, K
// 4096) at M = 1 / 64 41.7 / 51.0 -> 39.9 / 43.8, head at M = 1 / 16 / 64 192 / 200 /
// 221 -> 169 / 177 / 183.
constexpr TimeModel kDecodeModel{2.37, 9.55e6, 8.76};
constexpr TileShape kDecodeTiles[] = {{64, 64, 0.377, 0.377, 2.05}, {64, 128, 0.680, 0.680, 2.55}};
constexpr double kSkinnyStep[] = {0.631, 0.527, 0.622, 0.764, 1.35, 0.589};  // as kSkinnyShapes
constexpr double kSkinnyRows[] = {1.0, 1.59, 1.62};
constexpr double kSkinnyBase[] = {1.71, 1.80, 2.53};

inline Plan decode_plan(int M, int N, int K, bool split_ok) {
  const SkinnyPlan p = skinny_plan(M, N, K, split_ok);
  Plan best{-1, p.wn, p.wk, p.splits, p.k_split, 0};
  if (K <= 0) return best;
  double best_t = -1.0;
  if (skinny_plan_unsplit(M, N, K).wn > 0) {
    const int rows = p.mt / 2;  // row tiles 1, 2, 4
    double step = 0.0;
    for (int i = 0; i < kSkinnyShapeCount; ++i)
      if (kSkinnyShapes[i][0] == p.wn) step = kSkinnyStep[i] * kSkinnyRows[rows];
    const double n = static_cast<double>((p.k_split + kLdsBK - 1) / kLdsBK) / p.wk;
    const double rounds = static_cast<double>(ceil_div64(N, 16 * p.wn) * p.splits) / kSkinnyCus;
    best_t = 1.26 + std::max(1.0, rounds) * (n * step + kSkinnyBase[rows]) + split_us(kDecodeModel, p.splits, M, N);
  }
  try_tile(kDecodeModel, kDecodeTiles[0], kTile64x64, M, N, K, split_ok, best, best_t);
  try_tile(kDecodeModel, kDecodeTiles[1], kTile64x128, M, N, K, split_ok, best, best_t);
  return best;
}

// What a call of one size runs with the workspace of `full` and with less: a plan
// that does not split is the same in both, so its results do not depend on the
// workspace. A function of the sizes alone, kept per thread in a small
// direct-mapped table: a call asks for it twice (workspace, launch), and its
// evaluation (0.3-1 us of host time) shows where the kernel takes less than
// its launch.
struct CallPlan {
  int M, N, K;  // M = 0: an empty entry
  Plan full, unsplit;
};

inline CallPlan make_call_plan(int M, int N, int K) {
  const auto plan = M > 64 ? tile_plan : decode_plan;
  const Plan full = plan(M, N, K, true);
  return CallPlan{M, N, K, full, full.splits > 1 ? plan(M, N, K, false) : full};
}

inline const CallPlan& call_plan(int M, int N, int K) {
  constexpr unsigned kEntries = 64;
  static thread_local CallPlan table[kEntries];
  const unsigned h = static_cast<unsigned>(M) * 0x9E3779B1u ^ static_cast<unsigned>(N) * 0x85EBCA77u ^
                     static_cast<unsigned>(K) * 0xC2B2AE3Du;
  CallPlan& c = table[(h >> 16) % kEntries];
  if (c.M != M || c.N != N || c.K != K) c = make_call_plan(M, N, K);
  return c;
}

// Launches C = A B^T (+ bias) with the plan for (M, N, K) and the workspace
// given. With deferred_splits != nullptr, a plan that splits K stops after the
// main kernel, leaving splits x M x N fp32 partial tiles (no bias) in the
// workspace for the caller to sum in split order, and reports the split count
// there (1: C was written directly). dma_ok: the row strides allow the LDS-DMA
// kernel's 32-bit offsets (M <= 64 then keeps to the skinny kernel without).
template <typename E>
hipError_t launch(const uint16_t* A, const uint16_t* B, const uint16_t* bias, uint16_t* C, int M, int N, int K,
                  int lda, int ldb, int ldc, void* workspace, int64_t workspace_bytes, hipStream_t s,
                  int* deferred_splits, bool dma_ok) {
  const auto fits = [&](const Plan& q) {
    return q.splits == 1 || (workspace != nullptr && plan_workspace_bytes(q, M, N) <= workspace_bytes);
  };
  const CallPlan& c = call_plan(M, N, K);
  Plan p = fits(c.full) ? c.full : c.unsplit;
  if (!dma_ok) {
    SkinnyPlan k = skinny_plan(M, N, K, true);
    p = Plan{-1, k.wn, k.wk, k.splits, k.k_split, 0};
    if (!fits(p)) {
      k = skinny_plan(M, N, K, false);
      p = Plan{-1, k.wn, k.wk, k.splits, k.k_split, 0};
    }
  }
  if (deferred_splits != nullptr) *deferred_splits = p.splits;
  float* part = p.splits > 1 ? static_cast<float*>(workspace) : nullptr;
  if (p.shape >= 0)
    return tile_launchers<E>()[p.shape](A, B, bias, C, M, N, K, lda, ldb, ldc, s, part, p.splits, p.k_split,
                                        deferred_splits == nullptr, p.rot_step);
  const dim3 g2(static_cast<unsigned>(ceil_div64(N, 16 * p.wn)), static_cast<unsigned>(p.splits));
#define DK_SKINNY_LDS(MT_, WN_, WK_)                                                                                   \
  case MT_ * 100 + WN_ * 10 + WK_:                                                                                     \
    hipLaunchKernelGGL((gemm_skinny_lds_kernel<E, MT_, WN_, WK_, DK_SKINNY_DEPTH>), g2, dim3(WN_ * WK_ * kWave), 0, s, \
                       A, B, bias, C, M, N, K, lda, ldb, ldc, part, p.k_split);                                        \
    break;
#define DK_SKINNY_MT(MT_)                                                                             \
  DK_SKINNY_LDS(MT_, 1, 8) DK_SKINNY_LDS(MT_, 2, 4) DK_SKINNY_LDS(MT_, 4, 2) DK_SKINNY_LDS(MT_, 6, 2) \
  DK_SKINNY_LDS(MT_, 7, 2) DK_SKINNY_LDS(MT_, 8, 1)
  switch ((M <= 16 ? 1 : (M <= 32 ? 2 : 4)) * 100 + p.wn * 10 + p.wk) {
    DK_SKINNY_MT(1)
    DK_SKINNY_MT(2)
    DK_SKINNY_MT(4)
    default: return hipErrorInvalidValue;  // not a shape the plans produce
  }
#undef DK_SKINNY_MT
#undef DK_SKINNY_LDS
  if (part != nullptr && deferred_splits == nullptr) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    launch_splitk_reduce<E>(part, p.splits, M, N, bias, C, ldc, s);
  }
  return hipGetLastError();
}

}  // namespace gemm
}  // namespace dk

namespace {

int gemm_tn_checked(int dtype, const void* A, const void* B, const void* bias, void* C, int M, int N, int K, int lda,
                    int ldb, int ldc, void* workspace, int64_t workspace_bytes, void* stream,
                    int* deferred_splits = nullptr) {
  using namespace dk;
  clear_error();
  if (dtype != DK_FLOAT16 && dtype != DK_BFLOAT16)
    return fail("gemm_tn: expected float16 or bfloat16, got dtype code %d", dtype);
  if (M < 0 || N < 0 || K < 0) return fail("gemm_tn: M, N and K must be non-negative");
  if (M == 0 || N == 0) return hipSuccess;
  // A lone row's stride is never used: take the row length. Otherwise a row
  // stride below the row length would overlap rows, cut the last rows off the
  // load descriptors' extents (read as zeros) and write C out of bounds.
  if (M == 1) {
    lda = K;
    ldc = N;
  }
  if (N == 1) ldb = K;
  if (lda < K || ldb < K || ldc < N)
    return fail("gemm_tn: row strides must be at least the row lengths (lda, ldb >= K, ldc >= N)");
  if (K % 8 != 0 || lda % 8 != 0 || ldb % 8 != 0)
    return fail("gemm_tn: K and row strides of a/b must be multiples of 8");
  if (!aligned_to(A, 16) || !aligned_to(B, 16)) return fail("gemm_tn: a and b must be 16-byte aligned");
  if (C == nullptr || (K > 0 && (A == nullptr || B == nullptr))) return fail("gemm_tn: pointers must not be NULL");
  if (workspace != nullptr && !aligned_to(workspace, 16)) return fail("gemm_tn: workspace must be 16-byte aligned");
  if (workspace_bytes < 0) return fail("gemm_tn: workspace_bytes must be non-negative");
  if (M > 64 && ceil_div64(M, 64) * ceil_div64(N, 64) >= (int64_t{1} << 31)) return fail("gemm_tn: M x N is too large");
  const bool dma_ok = int64_t{256} * std::max(lda, ldb) * 2 < (int64_t{1} << 31);
  if (M > 64 && !dma_ok) return fail("gemm_tn: row strides too large for 32-bit buffer offsets");
  if (M <= 64 && (static_cast<int64_t>(M) * lda * 2 >= (int64_t{1} << 31) || int64_t{16} * ldb * 2 >= (int64_t{1} << 31)))
    return fail("gemm_tn: row strides too large for 32-bit buffer offsets");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto* a = static_cast<const uint16_t*>(A);
  const auto* b = static_cast<const uint16_t*>(B);
  const auto* bi = static_cast<const uint16_t*>(bias);
  auto* c = static_cast<uint16_t*>(C);
  const hipError_t e =
      dtype == DK_BFLOAT16
          ? gemm::launch<Bf16>(a, b, bi, c, M, N, K, lda, ldb, ldc, workspace, workspace_bytes, s, deferred_splits,
                               dma_ok)
          : gemm::launch<F16>(a, b, bi, c, M, N, K, lda, ldb, ldc, workspace, workspace_bytes, s, deferred_splits,
                              dma_ok);
  return static_cast<int>(e);
}

}  // namespace

extern "C" int dk_gemm_tn(int dtype, const void* A, const void* B, const void* bias, void* C, int M, int N, int K,
                          int lda, int ldb, int ldc, void* stream) {
  return gemm_tn_checked(dtype, A, B, bias, C, M, N, K, lda, ldb, ldc, nullptr, 0, stream);
}

extern "C" int64_t dk_gemm_tn_workspace_bytes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return dk::gemm::plan_workspace_bytes(dk::gemm::call_plan(M, N, K).full, M, N);
}

namespace {

// The plan of a call; nullptr for sizes that are refused.
const dk::gemm::Plan* plan_of(const char* op, int M, int N, int K, int with_workspace, const int* out) {
  dk::clear_error();
  if (out == nullptr) {
    dk::fail("%s: the output must not be NULL", op);
    return nullptr;
  }
  if (M <= 0 || N <= 0 || K < 0) {
    dk::fail("%s: M and N must be positive, K non-negative", op);
    return nullptr;
  }
  const dk::gemm::CallPlan& c = dk::gemm::call_plan(M, N, K);
  return with_workspace != 0 ? &c.full : &c.unsplit;
}

}  // namespace

extern "C" int dk_gemm_tn_plan(int M, int N, int K, int with_workspace, int* plan) {
  const dk::gemm::Plan* p = plan_of("gemm_tn_plan", M, N, K, with_workspace, plan);
  if (p == nullptr) return hipErrorInvalidValue;
  plan[0] = p->shape >= 0 ? dk::gemm::kTiles[p->shape].bm : p->wn;
  plan[1] = p->shape >= 0 ? dk::gemm::kTiles[p->shape].bn : p->wk;
  plan[2] = p->splits;
  plan[3] = p->k_split;
  return hipSuccess;
}

extern "C" int dk_gemm_tn_tile(int M, int N, int K, int with_workspace, int* tile) {
  const dk::gemm::Plan* p = plan_of("gemm_tn_tile", M, N, K, with_workspace, tile);
  if (p == nullptr) return hipErrorInvalidValue;
  tile[0] = p->shape >= 0 ? dk::gemm::kTiles[p->shape].bm : p->wn;
  tile[1] = p->shape >= 0 ? dk::gemm::kTiles[p->shape].bn : p->wk;
  tile[2] = p->splits;
  tile[3] = p->rot_step;
  return hipSuccess;
}

extern "C" int dk_gemm_tn_ws(int dtype, const void* A, const void* B, const void* bias, void* C, int M, int N, int K,
                             int lda, int ldb, int ldc, void* workspace, int64_t workspace_bytes, void* stream) {
  return gemm_tn_checked(dtype, A, B, bias, C, M, N, K, lda, ldb, ldc, workspace, workspace_bytes, stream);
}

// gemm_tn followed by fused_add_rms_norm on its output, with the split-K sum
// of decode-size plans done inside the norm's kernel (one launch fewer, the
// GEMM output never written before the norm). Results equal dk_gemm_tn_ws into
// `out` followed by dk_fused_add_rms_norm(out, residual, weight, eps) bit for
// bit; rows whose norm cannot take its vector path run exactly that pair.
extern "C" int dk_gemm_tn_add_rms_norm(int dtype, const void* A, const void* B, const void* bias, void* out,
                                       void* residual, const void* weight, float eps, int M, int N, int K, int lda,
                                       int ldb, int ld_out, int ld_res, void* workspace, int64_t workspace_bytes,
                                       void* stream) {
  using namespace dk;
  clear_error();
  if (dtype != DK_FLOAT16 && dtype != DK_BFLOAT16)
    return fail("gemm_tn_add_rms_norm: expected float16 or bfloat16, got dtype code %d", dtype);
  if (M < 0 || N < 0 || K < 0) return fail("gemm_tn: M, N and K must be non-negative");
  if (M == 0 || N == 0) return hipSuccess;
  if (out == nullptr || residual == nullptr || weight == nullptr)
    return fail("gemm_tn_add_rms_norm: out, residual and weight must not be NULL");
  if (ld_out < N || ld_res < N) return fail("gemm_tn_add_rms_norm: row strides of out and residual must be >= N");
  const bool fused = fused_add_rms_norm_vectorizable(N, ld_out, ld_res, out, residual, weight);
  int splits = 1;
  const int rc = gemm_tn_checked(dtype, A, B, bias, out, M, N, K, lda, ldb, ld_out, workspace, workspace_bytes,
                                 stream, fused ? &splits : nullptr);
  if (rc != hipSuccess) return rc;
  if (splits > 1)
    return launch_splitk_fused_add_rms_norm(dtype, static_cast<const float*>(workspace), splits, bias, out, ld_out,
                                            residual, ld_res, weight, M, N, eps, static_cast<hipStream_t>(stream));
  return dk_fused_add_rms_norm(dtype, out, residual, weight, M, N, ld_out, ld_res, eps, stream);
}

namespace {

int gemm_tn_rope_cache(const char* op, int dtype, const void* A, const void* B, const void* bias, void* C, int M, int N,
                       int K, int lda, int ldb, int ldc, const dk_rotary_params* r, const dk_cache_write_params* c,
                       bool fp8, float k_scale, float v_scale, void* workspace, int64_t workspace_bytes,
                       void* stream) {
  using namespace dk;
  clear_error();
  if (dtype != DK_FLOAT16 && dtype != DK_BFLOAT16) return fail("%s: expected float16 or bfloat16, got dtype code %d", op, dtype);
  if (M < 0 || N < 0 || K < 0) return fail("gemm_tn: M, N and K must be non-negative");
  if (M == 0 || N == 0) return hipSuccess;
  if (C == nullptr) return fail("gemm_tn: pointers must not be NULL");
  hipStream_t s = static_cast<hipStream_t>(stream);
  // Everything is checked before the GEMM runs, so a bad rotary / cache
  // argument leaves C untouched.
  if (const int rc = rotary_and_cache_on_rows(op, r, c, dtype, fp8, k_scale, v_scale, nullptr, 1, bias, C, ldc, M, N,
                                              true, s))
    return rc;
  int splits = 1;
  const int rc = gemm_tn_checked(dtype, A, B, bias, C, M, N, K, lda, ldb, ldc, workspace, workspace_bytes, stream,
                                 &splits);
  if (rc != hipSuccess) return rc;
  return rotary_and_cache_on_rows(op, r, c, dtype, fp8, k_scale, v_scale,
                                  splits > 1 ? static_cast<const float*>(workspace) : nullptr, splits, bias, C, ldc, M, N,
                                  false, s);
}

}  // namespace

// gemm_tn into C (e.g. a fused q | k | v projection) followed by
// rotary_embedding_and_cache on q / k / v views of C's rows; a plan that
// splits K forms each token's row of C from the partial tiles inside the
// rotary / cache kernel (one launch fewer). Results equal dk_gemm_tn_ws then
// dk_rotary_embedding_and_cache bit for bit.
extern "C" int dk_gemm_tn_rotary_embedding_and_cache(int dtype, const void* A, const void* B, const void* bias, void* C,
                                                     int M, int N, int K, int lda, int ldb, int ldc,
                                                     const dk_rotary_params* r, const dk_cache_write_params* c,
                                                     void* workspace, int64_t workspace_bytes, void* stream) {
  return gemm_tn_rope_cache("gemm_tn_rotary_embedding_and_cache", dtype, A, B, bias, C, M, N, K, lda, ldb, ldc, r, c,
                            false, 1.0f, 1.0f, workspace, workspace_bytes, stream);
}

// The same into fp8 (e4m3fn) caches (dk_rotary_embedding_and_cache_fp8).
extern "C" int dk_gemm_tn_rotary_embedding_and_cache_fp8(int dtype, const void* A, const void* B, const void* bias,
                                                         void* C, int M, int N, int K, int lda, int ldb, int ldc,
                                                         const dk_rotary_params* r, const dk_cache_write_params* c,
                                                         float k_scale, float v_scale, void* workspace,
                                                         int64_t workspace_bytes, void* stream) {
  return gemm_tn_rope_cache("gemm_tn_rotary_embedding_and_cache_fp8", dtype, A, B, bias, C, M, N, K, lda, ldb, ldc, r,
                            c, true, k_scale, v_scale, workspace, workspace_bytes, stream);
}
