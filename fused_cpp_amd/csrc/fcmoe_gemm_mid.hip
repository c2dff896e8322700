// fcmoe_gemm_mid.hip -- grouped GEMM on 64-row tiles for layers of little work.
//
// A layer whose active experts hold a few hundred MB of weights at most, or
// whose experts see some tens of rows, is bound by latency: the 128- and
// 256-row LDS tiles give it a few dozen workgroups, each walking K with two
// chunks in flight, and the 16-row tiles re-read an expert's weights for every
// 16 rows. Here:
//   * a workgroup is 4 waves and one row tile of at most 64 rows; each wave
//     holds all the tile's rows (FM = 4 fragments) against 2 channel tiles (a
//     gate/up pair, or 2 neighbouring tiles), so a weight byte is read once per
//     row tile, by one wave, straight into a register ring;
//   * the rows' K chunk is staged in LDS by buffer_load ... lds and read by the
//     4 waves;
//   * D - 1 chunks (7; W8A16 5) of both are in flight per wave, so that K is
//     walked at HBM latency / 7 per chunk even by a lone workgroup, and two or
//     three workgroups share a CU;
//   * loads past the last chunk fall outside the buffer resource or are not
//     issued: nothing is moved for them.
// The epilogues are the grouped GEMM's own (fcmoe_gemm_common.h).
#include <utility>

#include "fcmoe_gemm_common.h"

namespace fcmoe {

namespace {

constexpr int kMidWaves = 4;
constexpr int kMidFM = 4;  // 16-row fragments per tile
constexpr int kMidFN = 2;  // channel tiles per wave
constexpr int kMidBufWord3 = 0x00020000;
constexpr int kMidXcds = 8;
typedef __attribute__((address_space(3))) void* mid_lds_ptr;

// s_waitcnt vmcnt(N), the other counters unconstrained (gfx9 encoding)
template <int N>
__device__ __forceinline__ void mid_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// A rows are 64 bytes per K chunk (32 bf16 or 64 int8 elements); W8A16 rows
// are 128 (64 bf16 elements against 64 int8 weights).
template <bool I8, int EPI, int BPOL>
__global__ __launch_bounds__(kMidWaves * kWave) void grouped_gemm_mid_kernel(GemmParams p, int n_blocks) {
#if __HIP_DEVICE_COMPILE__
  constexpr bool PAIR = epi_pair(EPI);
  constexpr bool W8 = epi_w8(EPI);
  constexpr int FM = kMidFM, FN = kMidFN, BM = 16 * FM;
  constexpr int D = W8 ? 6 : 8;
  constexpr int AROW = W8 ? 128 : 64;
  constexpr int ABYTES = BM * AROW;
  constexpr int LA = ABYTES / 1024 / kMidWaves;  // A loads (1 KB) per wave and chunk
  static_assert(LA * 1024 * kMidWaves == ABYTES, "the waves' A loads cover the stage");
  constexpr int OPS = LA + FN;  // vector-memory ops per chunk and wave
  typedef typename Acc<I8>::type AccT;
  // One LDS object: the A stages, then the epilogue's per-row and per-channel
  // values (a second one would cost the K loop its counted waits).
  constexpr int NT = kMidWaves * FN;  // channel tiles per workgroup
  static_assert(NT * 16 <= kMidWaves * kWave && BM <= kMidWaves * kWave, "one value per thread");
  constexpr int THREADS = kMidWaves * kWave;
  __shared__ __attribute__((aligned(1024))) uint8_t sa[D * ABYTES + 12 * THREADS];
  float* const meta_rs = (float*)(sa + D * ABYTES);
  int* const meta_orow = (int*)(sa + D * ABYTES + 4 * THREADS);
  float* const meta_cs = (float*)(sa + D * ABYTES + 8 * THREADS);

  // The dispatcher deals workgroups to the XCDs round-robin; workgroup b runs
  // item b / 8 of a contiguous range owned by XCD b % 8, tiles last-first with
  // a tile's channel blocks side by side: its A rows, and the weights that the
  // row tiles of one expert share, are then re-read from that XCD's L2.
  const int count = *p.tile_count;
  const int total = count * n_blocks;
  const int x = (int)blockIdx.x % kMidXcds, k = (int)blockIdx.x / kMidXcds;
  const int q = total / kMidXcds, rem = total % kMidXcds;
  if (k >= q + (x < rem ? 1 : 0)) return;
  const int item = x * q + (x < rem ? x : rem) + k;
  const int tile = count - 1 - item / n_blocks;
  const int nb = item % n_blocks;
  const int expert = p.tiles[2 * tile];
  const int m0 = p.tiles[2 * tile + 1];
  const int rows_left = p.counts[expert] - m0;
  const int rows = rows_left < BM ? rows_left : BM;
  const int pos0 = p.offsets[expert] + m0;

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int nch = (int)p.k_chunks;
  const int64_t total_tiles = (int64_t)p.n_groups * p.n_tiles;
  int64_t gtile[FN];
  bool tvalid[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    if constexpr (PAIR) {
      const int64_t pr = (int64_t)nb * kMidWaves + wave;
      tvalid[j] = pr < p.n_tiles;
      gtile[j] = (j == 0 ? 0 : p.n_tiles) + pr;
    } else {
      gtile[j] = ((int64_t)nb * kMidWaves + wave) * FN + j;
      tvalid[j] = gtile[j] < total_tiles;
    }
  }

  // ---- A: load u of this wave is 1 KB of the stage: 16 rows x 64 bytes, unit
  // v of row r at slot v ^ ((r >> 2) & 3), or 8 rows x 128 bytes, unit v of
  // row r at slot v ^ ((r >> 1) & 7); the 16 rows of a fragment read then fall
  // on distinct banks. Rows past the tile's rows load from past the buffer
  // resource (zeros, nothing moved; the load still counts in vmcnt).
  const int64_t lda_bytes = p.lda * (I8 ? 1 : 2);
  const __amdgpu_buffer_rsrc_t rsrc_a =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.a), (short)0, 0x7ffffff0, kMidBufWord3);
  uint32_t voff_a[LA];
#pragma unroll
  for (int u = 0; u < LA; ++u) {
    const int g = wave * LA + u;
    const int r = W8 ? g * 8 + lane / 8 : g * 16 + lane / 4;
    const int unit = W8 ? (lane % 8) ^ ((r >> 1) & 7) : (lane % 4) ^ ((lane >> 4) & 3);
    const int pos = pos0 + (r < rows ? r : rows - 1);
    const int64_t arow = p.row_map ? (int64_t)p.row_map[pos] : (int64_t)pos;
    voff_a[u] = r < rows ? (uint32_t)(arow * lda_bytes + unit * 16) : 0x80000040u;
  }
  // ---- weights: one resource over the expert, the tile and chunk in the
  // scalar offset
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const uint8_t*)p.w + (int64_t)expert * p.w_expert_bytes), (short)0, (int)p.w_expert_bytes,
      kMidBufWord3);
  const int voff_b = lane * 16;
  int soff_b[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j)
    soff_b[j] = __builtin_amdgcn_readfirstlane((int)((tvalid[j] ? gtile[j] : 0) * p.k_chunks * 1024));

  const int frag = W8 ? (lane % 16) * 128 + (((2 * (lane / 16)) ^ ((lane % 16) >> 1)) * 16)
                      : (lane % 16) * 64 + (((lane / 16) ^ ((lane % 16) >> 2)) * 16);
  const int dhi = (frag ^ 16) - frag;  // W8A16: the row's second unit of the chunk's 16-byte weight piece

  // ---- the epilogue's row scales, output rows and channel scales: loaded
  // ahead of the ring (thread t: row t, channel slot t) and kept in LDS. Loaded
  // by the epilogue, each fragment's would wait for the stores of the one
  // before it, and W13's row scale is a dependent pair of loads (W8A8 TP rank
  // T=200 60 -> 55 us, 8x512 T=1000 52 -> 39).
  constexpr bool ROUTE = epi_route(EPI), COLS = epi_col_scale(EPI);
  const int mt = (int)threadIdx.x;
  const int mpos = pos0 + (mt < rows ? mt : rows - 1);
  int m_row = mpos, m_orow = mpos;
  float m_rs = 0.0f, m_cs = 0.0f;
  if constexpr (EPI == kEpiW13SwigluI8) {
    if (p.row_map) m_row = p.row_map[mpos];
    m_rs = p.scale_row[m_row];
  }
  if constexpr (EPI == kEpiW2RouteI8) m_rs = p.scale_row[mpos];
  if constexpr (ROUTE) m_orow = p.sorted_routes[mpos];
  if constexpr (COLS) {
    // slot t / 16: wave t / 16 / FN's tile (t / 16) % FN
    const int sw = mt / 16 / FN, sj = (mt / 16) % FN;
    const int64_t g = PAIR ? sj : 0;
    const int64_t cin = (PAIR ? (int64_t)nb * kMidWaves + sw : ((int64_t)nb * kMidWaves + sw) * FN + sj) * 16 + mt % 16;
    m_cs = p.scale_col[(int64_t)expert * p.n + g * p.n_half + (sw < kMidWaves && cin < p.n_half ? cin : 0)];
  }

  v4i bq[D][FN];
  AccT acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = AccT{0, 0, 0, 0};

  // Chunk t into ring slot `slot`: the A stage, then the weights, in this
  // order (the wait counts assume it). Past the last chunk: the last chunk
  // again (never read).
  auto issue = [&](int t, auto slot_c) {
    constexpr int slot = decltype(slot_c)::value;
    const int c = t < nch ? t : nch - 1;
#pragma unroll
    for (int u = 0; u < LA; ++u)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (mid_lds_ptr)(sa + slot * ABYTES + (wave * LA + u) * 1024), 16,
                                               voff_a[u], c * AROW, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < FN; ++j)
      bq[slot][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, voff_b, soff_b[j] + c * 1024, BPOL));
    __builtin_amdgcn_sched_barrier(0);
  };
  [&]<int... S>(std::integer_sequence<int, S...>) {
    (issue(S, std::integral_constant<int, S>{}), ...);
  }(std::make_integer_sequence<int, D - 1>{});

  // Published by the K loop's first barrier, with one chunk the only one: the
  // writes end here (lgkmcnt(0); the ring's loads stay in flight), as the
  // loop's barriers wait for none. Every thread writes its entry (the
  // epilogue reads the first BM and 16 NT): in a conditional block the loads
  // would be sunk into it, behind the ring, and drain it.
  meta_rs[mt] = m_rs;
  meta_orow[mt] = m_orow;
  meta_cs[mt] = m_cs;
  __builtin_amdgcn_s_waitcnt(0xC07F);

  // The closing scheduling barrier keeps the MFMAs, and with them the waits
  // for this wave's fragment reads, ahead of the next chunk's workgroup
  // barrier, past which the stage may be overwritten.
  auto compute = [&](auto slot_c) {
    constexpr int slot = decltype(slot_c)::value;
    const uint8_t* st = sa + slot * ABYTES + frag;
    if constexpr (W8) {
      v4i lo[FN], hi[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) i8x16_to_bf16(bq[slot][j], lo[j], hi[j]);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const v4i a0 = *(const v4i*)(st + i * 2048), a1 = *(const v4i*)(st + i * 2048 + dhi);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          acc[i][j] = mfma(__builtin_bit_cast(v8bf, a0), __builtin_bit_cast(v8bf, lo[j]), acc[i][j]);
          acc[i][j] = mfma(__builtin_bit_cast(v8bf, a1), __builtin_bit_cast(v8bf, hi[j]), acc[i][j]);
        }
      }
    } else {
      v4i af[FM];
#pragma unroll
      for (int i = 0; i < FM; ++i) af[i] = *(const v4i*)(st + i * 1024);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          if constexpr (I8)
            acc[i][j] = mfma(af[i], bq[slot][j], acc[i][j]);
          else
            acc[i][j] = mfma(__builtin_bit_cast(v8bf, af[i]), __builtin_bit_cast(v8bf, bq[slot][j]), acc[i][j]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Whole rings, then the rest, whose chunks are all in flight when the loop
  // ends: its steps issue nothing and each waits for one chunk fewer. (The
  // loop stays free of conditional steps, which would make the compiler drain
  // the weight registers at its header.)
  int t0 = 0;
  for (; t0 + D <= nch; t0 += D) {
    [&]<int... S>(std::integer_sequence<int, S...>) {
      ((mid_wait_vmcnt<OPS * (D - 2)>(), __builtin_amdgcn_s_barrier(),
        issue(t0 + S + D - 1, std::integral_constant<int, (S + D - 1) % D>{}),
        compute(std::integral_constant<int, S>{})),
       ...);
    }(std::make_integer_sequence<int, D>{});
  }
  auto rest = [&](auto slot_c) {
    constexpr int slot = decltype(slot_c)::value;
    mid_wait_vmcnt<OPS * (D - 2 - slot)>();
    __builtin_amdgcn_s_barrier();
    compute(slot_c);
  };
  [&]<int... S>(std::integer_sequence<int, S...>) {
    ((t0 + S < nch ? rest(std::integral_constant<int, S>{}) : void()), ...);
  }(std::make_integer_sequence<int, D - 1>{});
  mid_wait_vmcnt<0>();

  const EpiMeta meta{(lds_cfloat_ptr)meta_rs, (lds_cint_ptr)meta_orow, (lds_cfloat_ptr)meta_cs, wave * FN};
  gemm_epilogue<I8, EPI, FM, FN, true>(p, acc, gtile, tvalid, 0, rows, pos0, expert, lane, meta);
#endif
}

template <bool I8, int EPI>
int launch_mid(const GemmParams& p, int64_t max_tiles, hipStream_t stream) {
  constexpr bool PAIR = epi_pair(EPI);
  const int64_t units = PAIR ? p.n_tiles : (int64_t)p.n_groups * p.n_tiles;
  const int64_t n_blocks = ceil_div(units, (int64_t)kMidWaves * (PAIR ? 1 : kMidFN));
  const int64_t grid = round_up(max_tiles * n_blocks, kMidXcds);
  if (grid <= 0) return FCMOE_OK;
  if (grid > INT32_MAX) return fail(FCMOE_EINVAL, "grouped gemm grid too large");
  if (p.k_chunks <= 0) return fail(FCMOE_EINVAL, "grouped gemm: empty K");
  if (p.weights_once)
    hipLaunchKernelGGL((grouped_gemm_mid_kernel<I8, EPI, 2>), dim3((unsigned)grid), dim3(kMidWaves * kWave), 0, stream,
                       p, (int)n_blocks);
  else
    hipLaunchKernelGGL((grouped_gemm_mid_kernel<I8, EPI, 0>), dim3((unsigned)grid), dim3(kMidWaves * kWave), 0, stream,
                       p, (int)n_blocks);
  return check_launch("grouped_gemm_mid");
}

}  // namespace

int gemm_mid_launch(int epi, const GemmParams& p, int64_t max_tiles, hipStream_t stream) {
  switch (epi) {
    case kEpiW13SwigluI8:
      return launch_mid<true, kEpiW13SwigluI8>(p, max_tiles, stream);
    case kEpiW2RouteI8:
      return launch_mid<true, kEpiW2RouteI8>(p, max_tiles, stream);
    case kEpiW13ActBf16:
      return launch_mid<false, kEpiW13ActBf16>(p, max_tiles, stream);
    case kEpiRawF32Bias:
      return launch_mid<false, kEpiRawF32Bias>(p, max_tiles, stream);
    case kEpiW2RouteBf16:
      return launch_mid<false, kEpiW2RouteBf16>(p, max_tiles, stream);
    case kEpiW13ActW8:
      return launch_mid<false, kEpiW13ActW8>(p, max_tiles, stream);
    case kEpiW2RouteW8:
      return launch_mid<false, kEpiW2RouteW8>(p, max_tiles, stream);
    default:
      return fail(FCMOE_EINVAL, "unsupported 64-row epilogue");
  }
}

}  // namespace fcmoe
