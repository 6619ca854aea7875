// Half-precision product of a few rows: C[M,N] = chain(A[M,K] . B[K,N]), M <= 48.  One decoding step or a small batch
// through a linear layer: bound by reading B once.
//
// A workgroup of four waves takes 16, 32 or 64 columns of C and all of K; the waves take the 64-deep pieces of K in turn
// and multiply them into partial sums of their own with v_mfma_f32_16x16x32 (16 channels of B by 16 rows of A), added
// through LDS in wave order at the end: no barrier before that, every wave runs through its pieces alone.  A piece
// travels into a ring of DEPTH stages private to the wave with direct-to-LDS loads in runs of 64 or 128 bytes (lanes side
// by side on a row: the address path takes a 64-byte run of neighbouring lanes per cycle; fetched straight into the
// MFMA's register layout, where neighbouring lanes lie in different rows, a kilobyte took 64 cycles instead of 16,
// and M 16 N 4096 K 4096 10.8 us instead of 8.9).  B then comes at 3.8 TB/s for N = K = 4096 and at 5.1 TB/s for
// N 16384 K 8192 (268 MB in 52 us), what a large copy reaches on this device.
#include "contraction_kernel.hpp"

namespace tracea_amd {

// WAVES: waves of the workgroup; NB: blocks of 16 columns of C; XR: load instructions for the rows of A of a piece (8 rows each)
template <int DT, int WAVES, int NB, int XR, int DEPTH, bool KN>
__global__ void __launch_bounds__(WAVES * 64) gemm_rows_kernel(const ContractionArgs args) {
  constexpr int MB = (XR + 1) / 2;       // blocks of 16 rows
  constexpr int BR = 2 * NB, REQS = BR + XR;  // load instructions per piece: the channels of B, then the rows of A
  constexpr int STAGE = REQS * 1024;
  static_assert((DEPTH - 1) * REQS < 64, "vmcnt is a 6-bit counter");
  static_assert(DEPTH * STAGE >= MB * NB * 1024, "the partial sums of a wave lie in its ring");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  // KN with rows of 64 bytes: the two workgroups that share the 128-byte lines of B go to one XCD (ids are dealt round-robin)
  constexpr bool PAIRED = KN && NB == 2;
  const int bid = blockIdx.x;
  const int tile = PAIRED ? (bid & ~15) + (bid & 7) * 2 + ((bid >> 3) & 1) : bid;
  const int n0 = tile * (16 * NB);
  if (PAIRED && n0 >= args.N) return;  // (the grid is a multiple of 16)
  const int M = args.M, N = args.N, K = args.K;
  const long long z = (long long)blockIdx.z;
  __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)((const unsigned short *)args.A + z * args.batch_a), 0, (int)args.a_bytes, 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)((const unsigned short *)args.B + z * args.batch_b), 0, (int)args.b_bytes, 0x00020000);
  // rows past the end, like columns of K past the end, are requested out of range and read as zeros
  constexpr unsigned OOB = 0x80000000u;
  // load instruction i of a tensor: row 8 i + lane / 8, 16-byte slot lane % 8, which holds the piece's column
  // (lane % 8) ^ (row / 2): 16 rows at one column then lie in 16 different bank groups
  constexpr int NI = XR > BR ? XR : BR;
  // KN: a piece of B is 64 k rows of 16 NB channels, CB 16-byte columns each; fragments are fetched with transposing
  // reads, whose half-waves take 4 rows of two groups 8 rows apart: the swizzle spreads those over the banks
  constexpr int CB = 2 * NB, ROWB = 32 * NB, RPI = 64 / CB;
  auto swz = [](int krow) { return (NB == 4 ? ((krow >> 1) & 1) << 2 : 0) ^ (((krow >> 3) & 1) << 1); };
  unsigned b_voff[BR], a_voff[XR];
  int kcol[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int row = i * 8 + (lane >> 3);
    kcol[i] = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    if (i < BR) {
      if constexpr (KN) {
        const int krow = i * RPI + lane / CB, n = n0 + (((lane % CB) ^ swz(krow)) << 3);
        b_voff[i] = n < N ? (unsigned)(krow * args.ldb + n) * 2 : OOB;
      } else {
        b_voff[i] = n0 + row < N ? (unsigned)((n0 + row) * args.ldb + kcol[i]) * 2 : OOB;
      }
    }
    if (i < XR) a_voff[i] = row < M ? (unsigned)(row * args.lda + kcol[i]) * 2 : OOB;
  }
  unsigned char *const ring = smem + wave * (DEPTH * STAGE);
  auto request = [&](int t, int slot) __attribute__((always_inline)) {
    const int k0 = (wave + WAVES * t) * 64;
    unsigned char *dst = ring + slot * STAGE;
#pragma unroll
    for (int i = 0; i < BR; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (__attribute__((address_space(3))) void *)(dst + i * 1024), 16,
                                               (int)(k0 + (KN ? i * RPI + lane / CB : kcol[i]) < K ? b_voff[i] : OOB),
                                               k0 < K ? (int)(KN ? (long long)k0 * args.ldb * 2 : k0 * 2) : 0, 0, 0);
#pragma unroll
    for (int i = 0; i < XR; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void *)(dst + (BR + i) * 1024), 16,
                                               (int)(k0 + kcol[i] < K ? a_voff[i] : OOB), k0 < K ? k0 * 2 : 0, 0, 0);
  };
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int FLIGHT = (DEPTH - 1) * REQS;
  constexpr int WAIT_PIECE = 0x0f70 | (FLIGHT & 15) | ((FLIGHT >> 4) << 14);
  const unsigned frag = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)ring + r * 128 + ((q ^ ((r >> 1) & 7)) << 4);
  unsigned tr[KN ? NB : 1];
  if constexpr (KN) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int krow = q * 8 + (r >> 2), c = j * 2 + ((r & 3) >> 1);
      tr[j] = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)ring + krow * ROWB + ((c ^ swz(krow)) << 4) + (r & 1) * 8;
    }
  }
  const int pieces = (K + 63) / 64;
  const int mine = (pieces - wave + WAVES - 1) / WAVES;  // pieces wave, wave + WAVES, ...
#pragma unroll
  for (int t = 0; t < DEPTH; ++t) request(t, t);
  int slot = 0;
  for (int t = 0; t < mine; ++t) {
    __builtin_amdgcn_s_waitcnt(WAIT_PIECE);
    // (the reads are instructions with their own wait: through a pointer the compiler waits for every request in flight)
    const unsigned at = frag + slot * STAGE;
    u32x4 fb[2][NB], fa[2][MB];
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // (column 4 h + q: the swizzle's exclusive-or leaves bit 2 to the half)
      const unsigned p = at ^ (h * 64);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        if constexpr (KN) {
          u32x2 lo, hi;
          asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(tr[j] + slot * STAGE), "i"(h * 32 * ROWB) : "memory");
          asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(tr[j] + slot * STAGE), "i"((h * 32 + 4) * ROWB) : "memory");
          fb[h][j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        } else {
          asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[h][j]) : "v"(p), "i"(j * 2048) : "memory");
        }
      }
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
  f32x4 *part = (f32x4 *)smem;  // the partial sums of wave w: part[w * (DEPTH * STAGE / 16) + block * 64 + lane]
  constexpr int PITCH = DEPTH * STAGE / 16;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) part[wave * PITCH + (i * NB + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  // lane of block (i, j): row 16 i + r, channels n0 + 16 j + 4 q .. + 3
  for (int b = wave; b < MB * NB; b += WAVES) {
    const int m = (b / NB) * 16 + r, n = n0 + (b % NB) * 16 + q * 4;
    f32x4 sum = part[b * 64 + lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += part[w * PITCH + b * 64 + lane];
    if (m < M && n < N) {
      float v[4] = {sum[0], sum[1], sum[2], sum[3]};
      const long long row = z * args.batch_rows + m;
      apply_epilogue<4>(v, row, n, N - n, args.epi);
      store_from_float<4>(args.C, args.out_dtype, row * args.ldc + n, N - n, v);
    }
  }
}

template <int DT, int WAVES, int NB, int XR, int DEPTH, bool KN>
static int launch_rows(const ContractionArgs &a, hipStream_t stream) {
  // (+ 1 KB: an odd number of 8-row loads leaves the last block's upper 8 rows to be read from what lies behind)
  constexpr int lds = WAVES * DEPTH * (2 * NB + XR) * 1024 + 1024;
  if constexpr (lds > 160 * 1024) return (int)hipErrorInvalidValue;
  auto kfn = gemm_rows_kernel<DT, WAVES, NB, XR, DEPTH, KN>;
  static bool attr_done = false;
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
    attr_done = true;
  }
  unsigned tiles = (unsigned)((a.N + 16 * NB - 1) / (16 * NB));
  if (KN && NB == 2) tiles = (tiles + 15) & ~15u;
  const dim3 grid(tiles, 1, (unsigned)(a.batch > 1 ? a.batch : 1)), block(WAVES * 64);
  hipLaunchKernelGGL(kfn, grid, block, lds, stream, a);
  return (int)hipGetLastError();
}

// LO, HI: the least and most 8-row loads for A this form is compiled for
template <int DT, int NB, int DEPTH, bool KN, int LO, int HI>
static int launch_rows_of(const ContractionArgs &a, hipStream_t stream) {
  const int xr = (a.M + 7) / 8;
  if constexpr (LO < HI) {
    if (xr > LO) return launch_rows_of<DT, NB, DEPTH, KN, LO + 1, HI>(a, stream);
  }
  return launch_rows<DT, 4, NB, LO, DEPTH, KN>(a, stream);
}

// Which form (us in replayed graphs, bias, three sets of operands in turn; the 64x64 tiles split along K in brackets):
//   K-contiguous B: 16 columns per workgroup, so that N = 4096 fills the device (M 16 N 4096 K 4096 8.9 [13.8], M 48
//   10.8 [14.1], M 1 N 1024 K 1024 3.1 [7.4]); a third stage where a workgroup walks a long K over few rows (M 16 N
//   1024 K 8192 8.7 against 9.7 with two, but M 16 N 16384 K 1024 9.0 against 8.3).  With more than 16 rows the
//   re-reads of A outweigh B: 64 columns per workgroup wherever two thirds of the CUs still get one (M 48 N 16384 K 8192
//   61 against 75 [74], M 24 N 11008 K 4096 19.0 against 20.1 [31.0]; M 32 N 8192 K 2048 11.3 against 10.2).
//   N-contiguous B: 64 columns (128-byte rows) under the same condition (M 16 N 16384 K 8192 55 [66]), else 32 (M 16 N
//   4096 K 4096 12.5 [14.3], M 32 N 1024 K 1024 4.6 [7.8]).
// Eight waves instead of four, 32 columns of a K-contiguous B and deeper rings were never ahead by more than 2 %.
static bool wide_tiles(const ContractionArgs &a, int cus) {
  return (long long)((a.N + 63) / 64) * (a.batch > 1 ? a.batch : 1) * 3 >= 2ll * cus;
}

bool gemm_rows_pays(const ContractionArgs &a, bool b_ncontig, int cus) {
  if (a.M > kGemmRowsMax) return false;
  if (wide_tiles(a, cus)) return true;
  // few workgroups and a long K: the tile kernels spread K over more of them (N-contiguous: M 16 N 1024 K 8192 20.5
  // us here against 11.2, M 48 N 4096 K 4096 15.6 against 14.4, M 43 N 8376 K 768 13.2 against 11.2)
  if (b_ncontig) return a.K <= 4096 && a.M <= 32;
  // more than 32 rows: A's re-reads make a workgroup as long as the tile kernels' and a second round of them shows
  // (M 48 N 4528 K 2232, 283 workgroups, 12.3 us against 12.0)
  if (a.M > 32 && (long long)((a.N + 15) / 16) * (a.batch > 1 ? a.batch : 1) > cus) return false;
  return a.K <= 8192 || (long long)((a.N + 15) / 16) * (a.batch > 1 ? a.batch : 1) * 2 >= cus;
}

template <int DT>
static int launch_rows_type(const ContractionArgs &a, bool b_ncontig, int cus, hipStream_t stream) {
  const bool wide = wide_tiles(a, cus);
  if (b_ncontig) return wide ? launch_rows_of<DT, 4, 2, true, 1, 6>(a, stream) : launch_rows_of<DT, 2, 2, true, 1, 6>(a, stream);
  if (wide && a.M > 16) return launch_rows_of<DT, 4, 2, false, 3, 6>(a, stream);
  if (a.K >= 4096 && a.M <= 16) return launch_rows_of<DT, 1, 3, false, 1, 2>(a, stream);
  return launch_rows_of<DT, 1, 2, false, 1, 6>(a, stream);
}

int launch_gemm_rows(const ContractionArgs &a, int dtype, bool b_ncontig, int cus, hipStream_t stream) {
  if (a.M < 1 || a.M > kGemmRowsMax || a.a_bytes == 0 || a.b_bytes == 0) return (int)hipErrorInvalidValue;
  return dtype == DT_F16 ? launch_rows_type<DT_F16>(a, b_ncontig, cus, stream) : launch_rows_type<DT_BF16>(a, b_ncontig, cus, stream);
}

}  // namespace tracea_amd
