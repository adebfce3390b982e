// Many-token GEMM on int8 weights: C[token][row] = scale[row] * sum_k x[token][k] q[row][k] for hundreds or thousands
// of tokens (the drafter's prompt projection), where the products and not the weight bytes are the work.
//
// A workgroup of four waves owns a tile of 2 SR row strips x 2 ST token blocks (16 rows, 16 tokens each) and one band of
// K; wave (wr, wt) holds SR x ST accumulators of v_mfma_f32_16x16x32_f16. 64 columns a step come into one slot of a
// three-slot LDS ring by direct-to-LDS loads, two steps ahead of the products:
//   weights  the tile-major copy's 1 KB (strip, chunk) tiles as they are, still int8 (half the LDS bytes of fp16; each
//            wave widens its SR strips in registers, once for all ST token blocks);
//   x        row-major fp16, 8 tokens x 128 bytes per load (whole lines); lane l brings 16-byte piece (l % 8) ^ (l / 8)
//            of token l / 8, so token t's piece q lies in slot q ^ (t % 8) of its row and an operand read (16 tokens, one
//            piece each) covers every bank.
// Tiles are dealt to the XCDs in runs of neighbours (8 token tiles by consecutive row tiles), so one XCD's L2 serves the
// x and weight tiles that its workgroups share. K goes in `bands` shares when the tiles alone would leave CUs idle; band
// b's scaled sums go to y + b n N and the consumer (the norm kernel) adds them in order.
//
// Bound by the matrix cores and the LDS reads that feed them (per 64 columns a wave reads 12 KB for 32 products). Measured:
// 2048 tokens x 2048 rows x 10240 columns 86.8 us (0.99 PFLOP/s; torch's fp16 product of that shape 89.7 us), 2048 x 4096
// x 2048 41 us; a 2048-position prompt projection 3.14 ms in 128 chunks of 16 tokens -> 0.22 ms, 400 positions 601 -> 127
// us, 17 positions 108 -> 91 us.
//
// GS: per-128-column group scales: a group's two chunks go to fresh accumulators, scaled in fp32 and added in group order
// (as in the verify GEMM); the scales of a chunk's group ride in its ring slot, one copy per wave.
#include "common.h"
#include "dspark.h"
#include "dspark_internal.h"

namespace dspark {

constexpr int WIDE_SLOTS = 3;

template <int SR, int ST, bool GS>
__global__ __launch_bounds__(256, 2) void gemm_wide_kernel(GemmWideParams p) {
  constexpr int RS = 2 * SR, TB = 2 * ST;                 // strips and token blocks of the tile
  constexpr int XOFF = RS * 1024, SOFF = XOFF + TB * 2048;  // x and group scales in a slot
  constexpr int SLOT = SOFF + (GS ? 4 * 256 : 0);
  constexpr int UNITS = RS + 2 * TB, LPW = UNITS / 4 + (GS ? 1 : 0);  // loads a step, and per wave
  static_assert(UNITS % 4 == 0 && WIDE_SLOTS == 3, "every wave issues the same loads; the loop below is unrolled by 3");
  __shared__ __attribute__((aligned(16))) char slot0[SLOT], slot1[SLOT], slot2[SLOT];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave & 1, wt = wave >> 1;
  // Workgroup -> tile: XCD x (workgroups x, x + 8, ...) takes run x of the tiles in order (band, 8 token tiles, row tile,
  // token tile)
  const int RT = p.N / (16 * RS), TT = (p.n + 16 * TB - 1) / (16 * TB), total = RT * TT * p.bands;
  const int run = (total + 7) / 8;
  const int id = (int)(blockIdx.x % 8) * run + (int)(blockIdx.x / 8);
  if ((int)(blockIdx.x / 8) >= run || id >= total) return;
  const int band = id / (RT * TT), r = id % (RT * TT);
  const int tg = r / (RT * 8), width = min(8, TT - 8 * tg), rr = r - tg * RT * 8;
  const int strip0 = rr / width * RS, t0 = (8 * tg + rr % width) * 16 * TB;
  const int chunks = p.K / 64;
  const int c0 = min(chunks, band * p.band_chunks), nc = min(chunks, c0 + p.band_chunks) - c0;  // (>= 1)

  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, (short)0, (int)((size_t)p.N * p.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc((void*)p.x, (short)0, (int)((size_t)p.n * p.K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(GS ? p.gscale : p.scale), (short)0, (int)(GS ? (size_t)p.K / 128 * p.N * 2 : (size_t)p.N * 2), 0x00020000);
  // chunk c0 + k into `slot`: unit u < RS is a weight tile, the others 8 token rows each (tokens past the last read the
  // last: their products are never stored)
  uint32_t off[UNITS / 4];
#pragma unroll
  for (int i = 0; i < UNITS / 4; ++i) {
    const int u = wave + 4 * i;
    if (u < RS) {
      off[i] = (uint32_t)(((size_t)(strip0 + u) * chunks + c0) * 1024 + lane * 16);
    } else {
      const int t = min(t0 + 8 * (u - RS) + (lane >> 3), p.n - 1);
      off[i] = (uint32_t)(((size_t)t * p.K + (size_t)c0 * 64) * 2 + (((lane & 7) ^ (lane >> 3)) * 16));
    }
  }
  auto issue = [&](int k, char* slot) {
#pragma unroll
    for (int i = 0; i < UNITS / 4; ++i) {
      const int u = wave + 4 * i;
      const bool isw = u < RS;
      char* dst = isw ? slot + u * 1024 : slot + XOFF + (u - RS) * 1024;
      const uint32_t o = off[i] + (uint32_t)k * (isw ? 1024u : 128u);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(isw ? rw : rx, (__attribute__((address_space(3))) void*)dst, 16, o, 0, 0,
                                               0);
    }
    if constexpr (GS)  // two rows' scales per lane (lanes past the tile's rows load nothing)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (__attribute__((address_space(3))) void*)(slot + SOFF + wave * 256), 4,
          2 * lane < 16 * RS ? (uint32_t)(((size_t)((c0 + k) >> 1) * p.N + strip0 * 16 + 2 * lane) * 2) : 0x80000000u, 0,
          0, 0);
  };

  f32x4 acc[SR][ST], grp[GS ? SR : 1][GS ? ST : 1];
  const f32x4 z4 = {0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < SR; ++s)
#pragma unroll
    for (int t = 0; t < ST; ++t) {
      acc[s][t] = z4;
      if constexpr (GS) grp[s][t] = z4;
    }
  // x piece q = 2 g + h of the lane's token (rows 16 tb + n; the slot's rows start at a multiple of 8 tokens)
  const int xq0 = n * 128 + (((2 * g) ^ (n & 7)) * 16), xq1 = n * 128 + (((2 * g + 1) ^ (n & 7)) * 16);
  auto step = [&](int k, const char* cur, char* nxt) {
    ring_barrier<LPW>();  // chunk k is in LDS; every wave is done with chunk k - 1 (its slot is nxt)
    issue(min(k + 2, nc - 1), nxt);
    half8 a[SR][2];
    half4 gs[GS ? SR : 1];  // (read every step: under the branch below the compiler would drain every load first)
#pragma unroll
    for (int s = 0; s < SR; ++s) {
      if constexpr (GS)
        gs[s] = *reinterpret_cast<const half4*>(cur + SOFF + wave * 256 + ((wr * SR + s) * 16 + 4 * g) * 2);
      const u32x4 w = *reinterpret_cast<const u32x4*>(cur + (wr * SR + s) * 1024 + lane * 16);
      a[s][0] = i8x8_to_half8(w[0], w[1]);
      a[s][1] = i8x8_to_half8(w[2], w[3]);
    }
#pragma unroll
    for (int t = 0; t < ST; ++t) {
      const char* xb = cur + XOFF + (wt * ST + t) * 2048;
      const half8 b0 = *reinterpret_cast<const half8*>(xb + xq0), b1 = *reinterpret_cast<const half8*>(xb + xq1);
#pragma unroll
      for (int s = 0; s < SR; ++s) {
        f32x4& d = GS ? grp[GS ? s : 0][GS ? t : 0] : acc[s][t];
        d = mfma16x16x32(a[s][0], b0, d);
        d = mfma16x16x32(a[s][1], b1, d);
      }
    }
    if constexpr (GS) {
      if (((c0 + k) & 1) || k + 1 == nc) {  // the group's last chunk
#pragma unroll
        for (int s = 0; s < SR; ++s) {
#pragma unroll
          for (int t = 0; t < ST; ++t) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[s][t][i] = fmaf(grp[s][t][i], (float)gs[s][i], acc[s][t][i]);
            grp[s][t] = z4;
          }
        }
      }
    }
  };
  // Every step issues a chunk (past the band's end its last one again, into a slot nobody reads), so the loop has no
  // branches and the compiler can count the loads in flight: with them it drained every load before the first reads.
  issue(0, slot0);
  issue(min(1, nc - 1), slot1);
  int k = 0;
  for (; k + 3 <= nc; k += 3) {
    step(k, slot0, slot2);
    step(k + 1, slot1, slot0);
    step(k + 2, slot2, slot1);
  }
  if (k < nc) step(k, slot0, slot2);
  if (k + 1 < nc) step(k + 1, slot1, slot0);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
#pragma unroll
  for (int s = 0; s < SR; ++s) {
    const int row = (strip0 + wr * SR + s) * 16 + 4 * g;
    f32x4 sc = {1, 1, 1, 1};
    if constexpr (!GS) {
      const half4 h = ldg(reinterpret_cast<const half4*>(p.scale + row));
      sc = f32x4{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
    }
#pragma unroll
    for (int t = 0; t < ST; ++t) {
      const int tok = t0 + (wt * ST + t) * 16 + n;
      if (tok < p.n) *reinterpret_cast<f32x4*>(p.y + ((size_t)band * p.n + tok) * p.N + row) = acc[s][t] * sc;
    }
  }
}

// 128 x 128 tiles once those give every CU about one (each weight widened in registers serves 64 tokens of the wave),
// else 64 x 64; K in bands until there are two workgroups per CU, each keeping 8 chunks (16 with group scales: whole
// groups), and the bands within the caller's buffer.
bool gemm_wide_plan(int n, int N, int K, bool gs, int max_bands, GemmWideParams* p) {
  if (n < 1 || N % 128 || K % (gs ? 128 : 64)) return false;
  if ((int64_t)n * K * 2 > GEMM_WIDE_MAX_BYTES || (int64_t)N * K > GEMM_WIDE_MAX_BYTES) return false;
  const int chunks = K / 64;
  auto tiles = [&](int d) { return (N / d) * ((n + d - 1) / d); };
  p->tile = tiles(128) >= 192 ? 128 : 64;
  int bands = 1;
  while (2 * bands <= max_bands && tiles(p->tile) * bands * 2 <= 512 && chunks / (2 * bands) >= 8) bands *= 2;
  p->band_chunks = (chunks + bands - 1) / bands;
  if (gs) p->band_chunks += p->band_chunks & 1;  // bands start on whole groups
  p->bands = (chunks + p->band_chunks - 1) / p->band_chunks;
  p->n = n;
  p->N = N;
  p->K = K;
  return true;
}

int gemm_wide_launch(const GemmWideParams& p, hipStream_t s) {
  if (!p.x || !p.w || !p.y || !p.scale == !p.gscale || p.bands < 1 || (p.tile != 64 && p.tile != 128)) return DSPARK_EINVAL;
  const int total = (p.N / p.tile) * ((p.n + p.tile - 1) / p.tile) * p.bands;
  const dim3 grid((total + 7) / 8 * 8), block(256);
  if (p.tile == 128) {
    if (p.gscale)
      hipLaunchKernelGGL((gemm_wide_kernel<4, 4, true>), grid, block, 0, s, p);
    else
      hipLaunchKernelGGL((gemm_wide_kernel<4, 4, false>), grid, block, 0, s, p);
  } else {
    if (p.gscale)
      hipLaunchKernelGGL((gemm_wide_kernel<2, 2, true>), grid, block, 0, s, p);
    else
      hipLaunchKernelGGL((gemm_wide_kernel<2, 2, false>), grid, block, 0, s, p);
  }
  return (int)hipGetLastError();
}

}  // namespace dspark
