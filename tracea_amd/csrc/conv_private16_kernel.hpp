// Convolution on 16x16x32 MFMAs for launches of few output pixels (a batch of one or a few images, gfx950): small output
// tiles, the K axis split over the waves of a workgroup, every wave on a private ring of tiles.
//
// Same arithmetic as the reference's kernel_main (src/emitter/cuda/conv.rs:153-331):
// out[n,ho,wo,k] = epilogue(sum_{r,s,c} x[n, ho*sh-ph+r*dh, wo*sw-pw+s*dw, c] * w[k,r,s,c]), fp32 accumulation,
// zero padding; the sum is formed as one partial sum per wave, added in wave order at the end.
//
// A workgroup takes 8 XR output pixels by 16 NB filters and all of K = R*S*C; its waves take the 64-channel pieces of K
// in turn (with C a multiple of 64 a piece lies inside one tap and the tap's offsets are scalars).  A piece is 8 XR
// pixel rows and 16 NB filter rows of 128 bytes, requested straight into the wave's ring of DEPTH stages, 8 rows per
// direct-to-LDS load; pixels outside the image are requested out of range and read as zeros.  No wave waits for
// another before the partial sums meet in LDS.  What bounds such a launch is latency -- the launch itself (1.8 us),
// one round trip for the first pieces, the pieces of a wave one after the other, the tail -- so the tiles are small
// enough to put a workgroup on most CUs and K is cut WAVES ways instead of over workgroups, which needs a second
// kernel or a ticket and two more round trips through memory.
// Layout and swizzle of a stage: 128-byte rows, 16-byte column XOR (row / 2) & 7, filters first.
#pragma once
#include "contraction_kernel.hpp"

namespace tracea_amd {

// GEN: any multiple of 8 channels.  A 16-byte column of a piece still lies inside one tap, but the columns of a piece lie in
// several: tap and channel are worked out per lane, once for each of the two columns its rows are swizzled to.
template <int DT, int WAVES, int XR, int NB, int DEPTH, bool GEN>
__global__ void __launch_bounds__(WAVES * 64) conv_private16_kernel(const ContractionCore args) {
  constexpr int BM = 8 * XR, BN = 16 * NB, MB = XR / 2, NT = WAVES * 64;
  constexpr int BR = 2 * NB, REQS = BR + XR, STAGE = REQS * 1024;
  constexpr int NBLK = (MB * NB + WAVES - 1) / WAVES;  // blocks of the output a wave finishes
  static_assert(XR % 2 == 0 && (DEPTH - 1) * REQS < 64, "vmcnt is a 6-bit counter");
  static_assert(DEPTH * STAGE >= MB * NB * 1024, "the partial sums of a wave lie in its ring");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  asm volatile("" ::"s"(args.A), "s"(args.B), "s"(args.M), "s"(args.N), "s"(args.K), "s"(args.a_bytes), "s"(args.b_bytes), "s"(args.grid_n),
               "s"(args.h_in), "s"(args.w_in), "s"(args.c_in), "s"(args.h_out), "s"(args.w_out), "s"(args.s_sz), "s"(args.epi.n_ops));
  asm volatile("" ::"s"(args.stride_h), "s"(args.stride_w), "s"(args.pad_h), "s"(args.pad_w), "s"(args.dil_h), "s"(args.dil_w),
               "s"(args.hw_m), "s"(args.hw_s), "s"(args.w_m), "s"(args.w_s), "s"(args.sc_m), "s"(args.sc_s), "s"(args.c_m), "s"(args.c_s),
               "s"(args.gn_m), "s"(args.gn_s));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  int tile_m, tile_n;
  fast_divmod((int)blockIdx.x, args.gn_m, args.gn_s, args.grid_n, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int M = args.M, N = args.N, K = args.K, C = args.c_in, w_in = args.w_in;
  __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)args.A, 0, (int)args.a_bytes, 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)args.B, 0, (int)args.b_bytes, 0x00020000);
  constexpr unsigned OOB = 0x80000000u;

  // load i of a tensor: row 8 i + lane / 8, 16-byte slot lane % 8
  unsigned b_voff[BR];
#pragma unroll
  for (int i = 0; i < BR; ++i) {
    const int row = i * 8 + (lane >> 3);
    b_voff[i] = n0 + row < N ? (unsigned)((n0 + row) * (int)args.ldb + ((lane & 7) ^ ((row >> 1) & 7)) * 8) * 2 : OOB;
  }
  int pix[XR], hi0[XR], wi0[XR];  // byte offset of the pixel under tap (0, 0), its row and column
#pragma unroll
  for (int i = 0; i < XR; ++i) {
    const int row = i * 8 + (lane >> 3), m = m0 + row;
    int img, rem, ho, wo;
    fast_divmod(m < M ? m : M - 1, args.hw_m, args.hw_s, args.h_out * args.w_out, img, rem);
    fast_divmod(rem, args.w_m, args.w_s, args.w_out, ho, wo);
    hi0[i] = m < M ? ho * args.stride_h - args.pad_h : -(1 << 28);
    wi0[i] = wo * args.stride_w - args.pad_w;
    pix[i] = (((img * args.h_in + ho * args.stride_h - args.pad_h) * w_in + wi0[i]) * C + (GEN ? 0 : ((lane & 7) ^ ((row >> 1) & 7)) * 8)) * 2;
  }
  unsigned char *const ring = smem + wave * (DEPTH * STAGE);
  const int pieces = GEN ? (K + 63) / 64 : K / 64;
  auto request = [&](int t, int slot) __attribute__((always_inline)) {
    const int p = wave + WAVES * t;
    const bool live = p < pieces;
    const int k0 = live ? p * 64 : 0;
    // (rows of even and odd loads: the swizzle of a row repeats every 16 rows)
    constexpr int NK = GEN ? 2 : 1;
    int dh[NK], dw[NK], off[NK];
    bool in[NK];
#pragma unroll
    for (int e = 0; e < NK; ++e) {
      const int k = GEN ? k0 + ((lane & 7) ^ ((e * 4 + (lane >> 4)) & 7)) * 8 : k0;
      int rf, rem, sf, ci;
      fast_divmod(k, args.sc_m, args.sc_s, args.s_sz * C, rf, rem);
      fast_divmod(rem, args.c_m, args.c_s, C, sf, ci);
      dh[e] = rf * args.dil_h;
      dw[e] = sf * args.dil_w;
      off[e] = ((dh[e] * w_in + dw[e]) * C + ci) * 2;
      in[e] = GEN ? live & (k < K) : live;
    }
    unsigned char *dst = ring + slot * STAGE;
#pragma unroll
    for (int i = 0; i < BR; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (__attribute__((address_space(3))) void *)(dst + i * 1024), 16,
                                               (int)(in[i % NK] ? b_voff[i] : OOB), k0 * 2, 0, 0);
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      const bool ok = in[i % NK] & ((unsigned)(hi0[i] + dh[i % NK]) < (unsigned)args.h_in) & ((unsigned)(wi0[i] + dw[i % NK]) < (unsigned)w_in);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void *)(dst + (BR + i) * 1024), 16,
                                               (int)(ok ? (unsigned)(pix[i] + off[i % NK]) : OOB), 0, 0, 0);
    }
  };
#pragma unroll
  for (int t = 0; t < DEPTH; ++t) request(t, t);

  // The chain's operands travel under the main loop: per-channel vectors into a table (a thread's entries), the first
  // residual of the blocks this wave will finish into registers.
  const ChainPlan plan = chain_plan(args.epi);
  constexpr int TAB = TRACEA_MAX_EPILOGUE_OPS * 2 * BN, TPT = (TAB + NT - 1) / NT;
  float tabr[TPT];
#pragma unroll
  for (int i = 0; i < TPT; ++i) tabr[i] = 0.0f;
  if (plan.n_ops > 0) {
#pragma unroll
    for (int i = 0; i < TPT; ++i) {
      const int idx = tid + i * NT;
      if (idx < TAB) tabr[i] = chain_table_value(args.epi, idx / (2 * BN), (idx / BN) & 1, n0 + idx % BN, N);
    }
  }
  float res[NBLK][4];
  auto block_row = [&](int x) { return m0 + ((wave + x * WAVES) / NB) * 16 + r; };
  auto block_col = [&](int x) { return n0 + ((wave + x * WAVES) % NB) * 16 + q * 4; };
  if (plan.res_index >= 0) {
#pragma unroll
    for (int x = 0; x < NBLK; ++x) {
      const int m = block_row(x), n = block_col(x);
      if (wave + x * WAVES < MB * NB && m < M && n < N) load_as_float<4>(plan.res_ptr, plan.res_dtype, (long long)m * plan.res_ld + n, N - n, res[x]);
    }
  }

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int FLIGHT = (DEPTH - 1) * REQS;
  constexpr int WAIT_PIECE = 0x0f70 | (FLIGHT & 15) | ((FLIGHT >> 4) << 14);
  const unsigned frag = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)ring + r * 128 + ((q ^ ((r >> 1) & 7)) << 4);
  const int mine = (pieces - wave + WAVES - 1) / WAVES;  // pieces wave, wave + WAVES, ...
  int slot = 0;
  for (int t = 0; t < mine; ++t) {
    __builtin_amdgcn_s_waitcnt(WAIT_PIECE);
    const unsigned at = frag + slot * STAGE;
    u32x4 fb[2][NB], fa[2][MB];
    // (the reads are instructions with their own wait: through a pointer the compiler waits for every request in flight)
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // (column 4 h + q: the swizzle's exclusive-or leaves bit 2 to the half)
      const unsigned p = at ^ (h * 64);
#pragma unroll
      for (int j = 0; j < NB; ++j) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[h][j]) : "v"(p), "i"(j * 2048) : "memory");
#pragma unroll
      for (int i = 0; i < MB; ++i) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[h][i]) : "v"(p), "i"((NB + i) * 2048) : "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < NB; ++j) asm volatile("" : "+v"(fb[h][j]));
#pragma unroll
      for (int i = 0; i < MB; ++i) asm volatile("" : "+v"(fa[h][i]));
    }
    request(t + DEPTH, slot);
    slot = slot + 1 == DEPTH ? 0 : slot + 1;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = Mfma16<DT>::run(fb[h][j], fa[h][i], acc[i][j]);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // (requests past the end of K still write zeros to the ring)
  f32x4 *part = (f32x4 *)smem;  // the partial sums of wave w: part[w * PITCH + block * 64 + lane]
  constexpr int PITCH = DEPTH * STAGE / 16;
  float *const table = (float *)(smem + WAVES * DEPTH * STAGE);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) part[wave * PITCH + (i * NB + j) * 64 + lane] = acc[i][j];
#pragma unroll
  for (int i = 0; i < TPT; ++i)
    if (tid + i * NT < TAB) table[tid + i * NT] = tabr[i];
  __syncthreads();
#pragma unroll
  for (int x = 0; x < NBLK; ++x) {
    const int b = wave + x * WAVES;
    if (b >= MB * NB) break;
    f32x4 sum = part[b * 64 + lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += part[w * PITCH + b * 64 + lane];
    const int m = block_row(x), n = block_col(x);
    if (m >= M || n >= N) continue;
    float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    const float *tab = table + (n - n0);
#pragma nounroll
    for (int o = 0; o < plan.n_ops; ++o) {
      const int kind = (int)((plan.kinds >> (4 * o)) & 15u);
      if (kind == TRACEA_EPI_OP_RELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = fmaxf(0.0f, v[e]);
      } else if (kind == TRACEA_EPI_OP_RESIDUAL_ADD && o == plan.res_index) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] + res[x][e];
      } else if (kind == TRACEA_EPI_OP_BIAS_ADD || kind == TRACEA_EPI_OP_SCALE_SHIFT || kind == TRACEA_EPI_OP_BATCHNORM ||
                 kind == TRACEA_EPI_OP_BIAS_ADD_SILU) {
        const f32x4 a = *(const f32x4 *)(tab + (o * 2) * BN), s = *(const f32x4 *)(tab + (o * 2 + 1) * BN);  // s: zeros for a bias
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (kind == TRACEA_EPI_OP_BIAS_ADD) v[e] = v[e] + a[e];
          else if (kind == TRACEA_EPI_OP_BIAS_ADD_SILU) {
            const float y = v[e] + a[e];
            v[e] = y / (1.0f + expf(-y));
          } else v[e] = v[e] * a[e] + s[e];
        }
      } else {
        apply_epilogue_one<4>(v, m, n, N - n, args.epi.ops[o]);  // GELU, SiLU, a second residual
      }
    }
    store_from_float<4>(args.C, args.out_dtype, (long long)m * args.ldc + n, N - n, v);
  }
}

template <int WAVES, int BM, int BN, int DEPTH>
int launch_conv_private16(const ContractionArgs &a, bool conv, int dtype, bool b_ncontig, hipStream_t stream) {
  constexpr int XR = BM / 8, NB = BN / 16;
  constexpr int lds = WAVES * DEPTH * (2 * NB + XR) * 1024 + TRACEA_MAX_EPILOGUE_OPS * 2 * BN * 4;
  static_assert(lds <= 160 * 1024, "rings and table must fit LDS");
  if (!conv || b_ncontig || a.c_in % 8 != 0 || a.a_bytes == 0 || a.b_bytes == 0 || a.grid_m != (a.M + BM - 1) / BM ||
      a.grid_n != (a.N + BN - 1) / BN)
    return (int)hipErrorInvalidValue;
  const dim3 grid((unsigned)(a.grid_m * a.grid_n)), block(WAVES * 64);
#define TRACEA_LAUNCH_CP(DTV, GENV)                                                                          \
  do {                                                                                                     \
    auto kfn = conv_private16_kernel<DTV, WAVES, XR, NB, DEPTH, GENV>;                                     \
    static bool attr_done = false;                                                                         \
    if (!attr_done) {                                                                                      \
      hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds); \
      if (e != hipSuccess) return (int)e;                                                                  \
      attr_done = true;                                                                                    \
    }                                                                                                      \
    hipLaunchKernelGGL(kfn, grid, block, lds, stream, a);                                                  \
    return (int)hipGetLastError();                                                                         \
  } while (0)
  const bool gen = a.c_in % 64 != 0;
  if (dtype == DT_F16) { if (gen) TRACEA_LAUNCH_CP(DT_F16, true); else TRACEA_LAUNCH_CP(DT_F16, false); }
  else { if (gen) TRACEA_LAUNCH_CP(DT_BF16, true); else TRACEA_LAUNCH_CP(DT_BF16, false); }
  return (int)hipErrorInvalidValue;
#undef TRACEA_LAUNCH_CP
}

}  // namespace tracea_amd
