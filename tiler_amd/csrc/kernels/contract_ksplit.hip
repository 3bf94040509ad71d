// ---------------------------------------------------------------------------
// bf16 contraction with the k loop split over the waves of a workgroup, for
// the products that leave the 128-tiles' chip idle: m <= 64 (decode shapes,
// *_skinny{1..4}) and the m of a prompt chunk (*_k{MB}x{NB}).  Any m and n, k
// a multiple of 8, 16-byte aligned operands; 128 rows of k below 2^32 bytes, or
// the *_skinny{1..4}_l forms (kLong), whose lanes carry 64-bit addresses.
//
// A workgroup owns a tile of 16 MB x 16 NB outputs and each of its W waves the
// whole tile over its own 64-deep chunks of k (wave w chunks w, w + W, ...).
// A wave moves its chunk's rows global -> LDS with buffer_load_dwordx4 ... lds
// into a slot of its own, reads the fragments once, refills the slot with its
// next chunk, and runs the MFMAs while that lands.  No barrier until the end:
// a wave waits for its own loads only, every operand byte staged is read by
// one wave once, and nearly W slots per CU stay in flight.  The partial tiles
// fold in LDS in a fixed order, then SiLU, one bf16 narrowing, and 16-byte
// stores of whole row chunks.
//
// LDS rows are 128 bytes, chunk c of row r at c ^ ((r >> 1) & 7), as in the
// staged form.  Loading the fragments straight into registers instead (16 rows
// x 64 bytes per load, so neighbouring lanes are in different lines) reached
// 32 bytes/ns per CU where this layout reaches ~80 (64 x 4096 x 4096 20.2
// against 10.6 us, 300 x 4096 x 4096 36 against 17.5).
//
// Bound by the operand fill: k (MB + NB) 32 bytes per tile at ~80 bytes/ns per
// CU (20 TB/s over the chip; 300 x 4096 x 4096: 2.33 M L2 requests of 128 bytes,
// 298 MB, 81% of them hits).  The smaller tiles fill more CUs and read more.
// Before (16 waves, fragments in registers, m <= 64; 128-tiles above) and now,
// us: 1 x 4096 x 4096 9.4 / 8.4, 48 x 4096 x 4096 19.1 / 9.8, 128 x 4096 x 4096
// 45.7 / 12.0, 200 x 1024 x 1024 14.0 / 4.3, 300 x 4096 x 4096 46 / 18,
// 512 x 4096 x 4096 45 / 25.
namespace {

typedef __attribute__((address_space(1))) void global_void;

template <int MB, int NB, int W, bool kSilu, bool kLong = false>
__device__ __forceinline__ void contract_bf16_ksplit_body(const uint16_t* __restrict__ a,
                                                          const uint16_t* __restrict__ b, uint32_t m, uint32_t n,
                                                          uint32_t k, uint16_t* __restrict__ c) {
  constexpr int kBlocks = MB * NB, kLoads = 2 * (MB + NB);
  constexpr int R = W % 4 == 0 && kBlocks <= 36 ? 4 : 2;  // partial tiles that meet in LDS
  static_assert(W % R == 0 && W > R - 1, "the waves fold onto R partial tiles");
  constexpr uint32_t kRow = NB * 16 + 8;              // bf16 elements per staged C row
  constexpr uint32_t kSlot = kLoads * 512u;           // bf16 elements of a wave's slot
  constexpr uint32_t kStage = W * kSlot * 2u, kRed = R * kBlocks * 1024u, kC = MB * 16 * kRow * 2u;
  constexpr uint32_t kBytes = kStage > kRed ? (kStage > kC ? kStage : kC) : (kRed > kC ? kRed : kC);
  // (6 x 4 blocks fold onto 96 KiB; onto two partial tiles, 80, a workgroup that
  // has its CU to itself took 8.7 against 8.1 us, 1300 x 1001 x 512.)
  static_assert(kLoads * W > 80 || kBlocks > 20 || kBytes <= 80 * 1024,
                "the planner counts on two workgroups of such a tile to a CU");
  __shared__ __attribute__((aligned(1024))) uint16_t smem[kBytes / 2];
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t tiles_m = (m + MB * 16 - 1) / (MB * 16), tiles_n = (n + NB * 16 - 1) / (NB * 16);
  // Panels of B in groups of eight, one per XCD, and the tiles of a panel in
  // consecutive slots of it; fewer than eight panels: row-major.
  uint32_t tm, tn;
  if (tiles_n >= 8) {
    const uint32_t place = blockIdx.x >> 3;
    tm = place % tiles_m;
    tn = place / tiles_m * 8u + (blockIdx.x & 7u);
  } else {
    tm = blockIdx.x % tiles_m;
    tn = blockIdx.x / tiles_m;
  }
  if (tn >= tiles_n) return;
  const uint32_t m0 = tm * MB * 16, n0 = tn * NB * 16;
  const uint32_t rows = m - m0 < MB * 16u ? m - m0 : MB * 16u, cols = n - n0 < NB * 16u ? n - n0 : NB * 16u;
  const __amdgpu_buffer_rsrc_t pa =
      __builtin_amdgcn_make_buffer_rsrc((void*)(a + (uint64_t)m0 * k), (short)0, rows * k * 2u, 0x00020000);
  const __amdgpu_buffer_rsrc_t pb =
      __builtin_amdgcn_make_buffer_rsrc((void*)(b + (uint64_t)n0 * k), (short)0, cols * k * 2u, 0x00020000);
  // Load j of an operand fills rows 8 j .. 8 j + 7 of its slot: lane i the
  // 16-byte chunk i % 8 of row 8 j + i / 8, from chunk (i % 8) ^ ((row >> 1) & 7).
  uint32_t vbase[2];
#pragma unroll
  for (uint32_t o = 0; o < 2; ++o)
    vbase[o] = (o * 8u + (lane >> 3)) * k * 2u + ((lane & 7u) ^ (o * 4u + (lane >> 4))) * 16u;
  uint16_t* const slot = smem + wave * kSlot;
  // kLong: the rows past the last read the last one (never stored) and the
  // chunks past k read chunk 0 (zeroed below), where a buffer would give zeros.
  auto row_piece = [&](const uint16_t* panel, uint32_t panel_rows, uint32_t j, uint32_t chunk) {
    const uint32_t row = j * 8u + (lane >> 3), e = chunk * 64u + ((lane & 7u) ^ ((row >> 1) & 7u)) * 8u;
    return (global_void*)(panel + (uint64_t)(row < panel_rows ? row : panel_rows - 1u) * k + (e < k ? e : 0u));
  };
  auto issue = [&](uint32_t chunk) {
    if constexpr (kLong) {
#pragma unroll
      for (int j = 0; j < 2 * NB; ++j)
        __builtin_amdgcn_global_load_lds(row_piece(b + (uint64_t)n0 * k, cols, j, chunk),
                                         (lds_void*)(slot + (2 * MB + j) * 512), 16, 0, 0);
#pragma unroll
      for (int j = 0; j < 2 * MB; ++j)
        __builtin_amdgcn_global_load_lds(row_piece(a + (uint64_t)m0 * k, rows, j, chunk),
                                         (lds_void*)(slot + j * 512), 16, 0, 0);
      return;
    }
    const uint32_t at = chunk * 128u;
#pragma unroll
    for (int j = 0; j < 2 * NB; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(pb, (lds_void*)(slot + (2 * MB + j) * 512), 16,
                                               vbase[j & 1] + (at + (j >> 1) * 32u * k), 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 2 * MB; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(pa, (lds_void*)(slot + j * 512), 16,
                                               vbase[j & 1] + (at + (j >> 1) * 32u * k), 0, 0, 0);
  };
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const uint32_t frow = lane & 15u, grp = lane >> 4, swz = frow >> 1;
  const uint32_t chunks = (k + 63u) >> 6, ragged = k & 63u;
  if (wave < chunks) issue(wave);
  for (uint32_t ch = wave; ch < chunks; ch += W) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    u32x4 fa[2][MB], fb[2][NB];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint32_t chunk = ((uint32_t)s * 4u + grp) ^ swz;
      const uint16_t* q = slot + frow * 64u + chunk * 8u;
#pragma unroll
      for (int j = 0; j < NB; ++j) fb[s][j] = *reinterpret_cast<const u32x4*>(q + (MB + j) * 1024);
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[s][i] = *reinterpret_cast<const u32x4*>(q + i * 1024);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (ch + W < chunks) issue(ch + W);
    if (ragged && ch == chunks - 1) {  // past k: zeros in both operands
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if ((uint32_t)s * 32u + grp * 8u >= ragged) {
#pragma unroll
          for (int i = 0; i < MB; ++i) fa[s][i] = u32x4{0, 0, 0, 0};
#pragma unroll
          for (int j = 0; j < NB; ++j) fb[s][j] = u32x4{0, 0, 0, 0};
        }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(fa[s][i]), as_bf16x8(fb[s][j]), acc[i][j], 0,
                                                              0, 0);
  }
  // The waves' partial tiles fold onto R of them in LDS (fixed order), then
  // each wave finishes its share of the blocks.
  f32x4* const red = reinterpret_cast<f32x4*>(smem);
  auto add = [](const f32x4 x, const f32x4 y) { return f32x4{x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w}; };
  auto put = [&]() {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) red[((wave % R) * kBlocks + i * NB + j) * 64u + lane] = acc[i][j];
  };
  __syncthreads();
#pragma unroll
  for (int w0 = W - R; w0 >= R; w0 -= R) {
    if (wave >= (uint32_t)w0 && wave < (uint32_t)(w0 + R)) put();
    __syncthreads();
    if (wave >= (uint32_t)(w0 - R) && wave < (uint32_t)w0) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = add(acc[i][j], red[((wave % R) * kBlocks + i * NB + j) * 64u + lane]);
    }
    if (w0 > R) __syncthreads();
  }
  if (wave < (uint32_t)R) put();
  __syncthreads();
  constexpr int kMine = (kBlocks + W - 1) / W;
  uint32_t mine[kMine][2];
#pragma unroll
  for (int x = 0; x < kMine; ++x) {
    const uint32_t q = wave + x * W;
    if (q < (uint32_t)kBlocks) {
      f32x4 t = add(red[q * 64u + lane], red[(kBlocks + q) * 64u + lane]);
      if constexpr (R == 4)
        t = add(t, add(red[(2 * kBlocks + q) * 64u + lane], red[(3 * kBlocks + q) * 64u + lane]));
      if (kSilu) {
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] = tiler::silu_for_bf16(t[r]);
      }
      mine[x][0] = tiler::bf16_pack2_rne(t[0], t[1]);
      mine[x][1] = tiler::bf16_pack2_rne(t[2], t[3]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int x = 0; x < kMine; ++x) {
    const uint32_t q = wave + x * W;
    if (q < (uint32_t)kBlocks) {
      uint16_t* d = smem + (q / NB * 16u + grp * 4u) * kRow + q % NB * 16u + frow;
      d[0] = (uint16_t)mine[x][0];
      d[kRow] = (uint16_t)(mine[x][0] >> 16);
      d[2 * kRow] = (uint16_t)mine[x][1];
      d[3 * kRow] = (uint16_t)(mine[x][1] >> 16);
    }
  }
  __syncthreads();
  uint16_t* out = c + (uint64_t)m0 * n + n0;
  if ((n & 7u) == 0 && ((uintptr_t)c & 15u) == 0) {  // uniform: whole 16-byte chunks
    for (uint32_t q = threadIdx.x; q < MB * 16u * NB * 2u; q += 64u * W) {
      const uint32_t r = q / (NB * 2u), x = q % (NB * 2u) * 8u;
      if (r < rows && x < cols)
        *reinterpret_cast<u32x4*>(out + (uint64_t)r * n + x) = *reinterpret_cast<const u32x4*>(smem + r * kRow + x);
    }
  } else {
    for (uint32_t q = threadIdx.x; q < MB * 16u * NB * 16u; q += 64u * W) {
      const uint32_t r = q / (NB * 16u), x = q % (NB * 16u);
      if (r < rows && x < cols) out[(uint64_t)r * n + x] = smem[r * kRow + x];
    }
  }
}

}  // namespace

#define TILER_CONTRACT_KSPLIT(NAME, MB, NB, W, SILU, LONG)                                           \
  extern "C" __global__ void __launch_bounds__(64 * W, (W + 3) / 4)                                   \
      NAME(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint32_t m, uint32_t n,     \
           uint32_t k, uint16_t* __restrict__ c) {                                                    \
    contract_bf16_ksplit_body<MB, NB, W, SILU, LONG>(a, b, m, n, k, c);                               \
  }                                                                                                   \
  extern "C" __global__ void __launch_bounds__(64 * W, (W + 3) / 4)                                   \
      NAME##_b(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint32_t m, uint32_t n, \
               uint32_t k, uint16_t* __restrict__ c, tiler_geom::BatchGeometry g) {                   \
    uint64_t oa, ob, oc;                                                                              \
    batch_offsets(g, blockIdx.y, oa, ob, oc);                                                         \
    contract_bf16_ksplit_body<MB, NB, W, SILU, LONG>(a + oa, b + ob, m, n, k, c + oc);                \
  }
#define TILER_CONTRACT_KSPLIT_BOTH(FORM, MB, NB, W)                                                   \
  TILER_CONTRACT_KSPLIT(tiler_contract_bf16_##FORM, MB, NB, W, false, false)                          \
  TILER_CONTRACT_KSPLIT(tiler_contract_bf16_silu_##FORM, MB, NB, W, true, false)
#define TILER_CONTRACT_KSPLIT_LONG(FORM, MB)                                                          \
  TILER_CONTRACT_KSPLIT(tiler_contract_bf16_##FORM##_l, MB, 1, 8, false, true)                        \
  TILER_CONTRACT_KSPLIT(tiler_contract_bf16_silu_##FORM##_l, MB, 1, 8, true, true)
TILER_CONTRACT_KSPLIT_BOTH(skinny1, 1, 1, 8)
TILER_CONTRACT_KSPLIT_BOTH(skinny2, 2, 1, 8)
TILER_CONTRACT_KSPLIT_BOTH(skinny3, 3, 1, 8)
TILER_CONTRACT_KSPLIT_BOTH(skinny4, 4, 1, 8)
TILER_CONTRACT_KSPLIT_LONG(skinny1, 1)
TILER_CONTRACT_KSPLIT_LONG(skinny2, 2)
TILER_CONTRACT_KSPLIT_LONG(skinny3, 3)
TILER_CONTRACT_KSPLIT_LONG(skinny4, 4)
TILER_CONTRACT_KSPLIT_BOTH(k2x2, 2, 2, 8)
TILER_CONTRACT_KSPLIT_BOTH(k2x4, 2, 4, 8)
TILER_CONTRACT_KSPLIT_BOTH(k3x4, 3, 4, 8)
TILER_CONTRACT_KSPLIT_BOTH(k4x4, 4, 4, 4)
TILER_CONTRACT_KSPLIT_BOTH(k5x4, 5, 4, 8)
TILER_CONTRACT_KSPLIT_BOTH(k6x4, 6, 4, 4)
TILER_CONTRACT_KSPLIT_BOTH(k4x8, 4, 8, 4)
TILER_CONTRACT_KSPLIT_BOTH(k6x8, 6, 8, 4)
