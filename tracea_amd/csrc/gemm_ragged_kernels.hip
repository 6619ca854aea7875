// Half-precision product of operands at any element alignment: C[M,N] = chain(A[M,K] . B[K,N]), A by rows, B by rows or
// by columns, rows of any length and pitch (M 1000 N 900 K 1030: no row but the first starts on 16 bytes).
//
// Direct-to-LDS loads want their 16-byte pieces aligned, so tiles come through registers: 16-byte loads at the elements'
// own alignment, DEPTH K tiles ahead of the one being multiplied, written to one of two LDS stages when their turn
// comes.  One barrier per K tile; nothing waits for a load that was not requested DEPTH tiles earlier.  Two groups of
// four waves may share a tile: they take the K tiles in turn, each with stages and sums of its own, added through LDS at
// the end.  M 1000 N 900 K 1030 11.8 us (f16, replayed graph) against 24.7 from padded copies of both operands.
//
// Bound by the walk over K: nine rounds per group at that size, each a store to LDS, a barrier and a multiply, with the
// matrix pipe busy for 8 % of the launch and a third of the wave cycles waiting on an instruction.  Of that the address
// path is about 3 us: a load off a dword takes a cycle per lane where an aligned one takes four lanes (M = N = 100, K 5000
// on one workgroup per CU and four groups: 0.19 us per K tile on rows that start on a dword, 0.38 off it).
// Aligned loads of the dwords around a piece, joined in registers, cost the same cycles again (32 us against 33 there,
// 43 against 33 with one group).
//
// Reads stay inside the operand's extent ((rows - 1) * pitch + row length, at least 8 elements): a piece that would
// pass the end is read from the last 8 elements and shifted into place, elements of A and rows of B behind K are
// cleared (a product with whatever lies there could be NaN), columns of B behind N reach only columns never stored.
#include "contraction_kernel.hpp"

namespace tracea_amd {

typedef u32x4 u32x4_any __attribute__((aligned(2)));  // 16 bytes at any element

// p's elements s .. 7 moved to the front (zeros or anything else behind them), s < 8
__device__ __forceinline__ u32x4 drop_front(u32x4 p, unsigned s) {
  const u32x4 h = {__builtin_amdgcn_alignbit(p[1], p[0], 16), __builtin_amdgcn_alignbit(p[2], p[1], 16),
                   __builtin_amdgcn_alignbit(p[3], p[2], 16), p[3] >> 16};
  p = (s & 1) ? h : p;
  const u32x4 w = {p[1], p[2], p[3], 0u};
  p = (s & 2) ? w : p;
  const u32x4 d = {p[2], p[3], 0u, 0u};
  return (s & 4) ? d : p;
}
// the first `keep` elements of p, zeros behind them
__device__ __forceinline__ u32x4 keep_front(u32x4 p, int keep) {
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = keep >= 2 * i + 2 ? p[i] : keep == 2 * i + 1 ? p[i] & 0xffffu : 0u;
  return p;
}

// LDS of a group: its two stages, and in their place at the end its sums, T rows of T + 4 floats
constexpr int ragged_group_bytes(int t) { return t * (t + 4) * 4 > t * 512 ? t * (t + 4) * 4 : t * 512; }

// T: rows and columns of the tile; WN: waves side by side (two rows of them); KN: B by rows (else by columns)
template <int DT, int T, int WN, int GROUPS, int DEPTH, bool KN>
__global__ void __launch_bounds__(GROUPS * WN * 128) gemm_ragged_kernel(const ContractionCore args) {
  constexpr int GT = WN * 128;                // threads of a group
  constexpr int NP = T * 8 / GT;              // 16-byte pieces per thread, operand and K tile of 64
  constexpr int OPERAND = T * 128, STAGE = 2 * OPERAND;
  constexpr int TM = T / 2, TN = T / WN, NBM = TM / 16, NBN = TN / 16;  // a wave's share of the tile, in 16x16 blocks
  constexpr int CB = T / 8, ROWB = T * 2;     // KN: 16-byte columns and bytes of a k row of B
  constexpr int NT = GROUPS * GT, PITCH = T + 4;
  constexpr int GROUP_BYTES = ragged_group_bytes(T);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x % GT, lane = threadIdx.x & 63, wave = tid >> 6;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
  const int wm = wave & 1, wn = wave >> 1, r = lane & 15, q = lane >> 4;
  int tile_m, tile_n;
  tile_coordinates(args, tile_m, tile_n);
  const int m0 = tile_m * T, n0 = tile_n * T;
  const int M = args.M, N = args.N, K = args.K;
  const unsigned short *A = (const unsigned short *)args.A, *B = (const unsigned short *)args.B;
  // (extents below 2 GiB: element offsets in 32 bits)
  const unsigned a_last = args.a_bytes / 2 - 8, b_last = args.b_bytes / 2 - 8;  // where the last whole piece starts
  const unsigned lda = (unsigned)args.lda, ldb = (unsigned)args.ldb;

  // B by rows: the swizzle of the transposing reads' tiles (see the kernel for products of a few rows); else, as for A,
  // 16 rows at one column lie in 16 different bank groups
  auto swz_kn = [](int krow) { return (T == 64 ? ((krow >> 1) & 1) << 2 : (krow & 3) << 2) ^ (((krow >> 3) & 1) << 1); };
  auto swz = [](int row) { return (row >> 1) & 7; };
  unsigned a_off[NP], b_off[NP], a_dst[NP], b_dst[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = tid + i * GT, row = p >> 3, c = p & 7;
    a_off[i] = (unsigned)min(m0 + row, M - 1) * lda + c * 8;
    a_dst[i] = row * 128 + ((c ^ swz(row)) << 4);
    if constexpr (KN) {
      const int krow = p / CB, cn = p % CB;
      b_off[i] = (unsigned)krow * ldb + n0 + cn * 8;
      b_dst[i] = OPERAND + krow * ROWB + ((cn ^ swz_kn(krow)) << 4);
    } else {
      b_off[i] = (unsigned)min(n0 + row, N - 1) * ldb + c * 8;
      b_dst[i] = OPERAND + a_dst[i];
    }
  }
  const int kcol = (tid & 7) * 8;

  u32x4 ra[DEPTH][NP], rb[DEPTH][NP];
  auto offset_a = [&](int i, int k0) { return a_off[i] + (unsigned)k0; };
  auto offset_b = [&](int i, int k0) { return b_off[i] + (KN ? (unsigned)k0 * ldb : (unsigned)k0); };
  auto load = [&](int slot, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      ra[slot][i] = *(const u32x4_any *)(A + min(offset_a(i, k0), a_last));
      rb[slot][i] = *(const u32x4_any *)(B + min(offset_b(i, k0), b_last));
    }
  };
  auto store = [&](int slot, unsigned char *dst, int k0) __attribute__((always_inline)) {
    u32x4 va[NP], vb[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      va[i] = ra[slot][i];
      vb[i] = rb[slot][i];
    }
    if (k0 + 72 > K) {  // (a row of B within 8 elements of the end may need the shift in front of the last tile)
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const unsigned oa = offset_a(i, k0), ob = offset_b(i, k0);
        va[i] = keep_front(drop_front(va[i], oa - min(oa, a_last)), K - k0 - kcol);
        vb[i] = keep_front(drop_front(vb[i], ob - min(ob, b_last)), KN ? (k0 + (tid + i * GT) / CB < K ? 8 : 0) : K - k0 - kcol);
      }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      *(u32x4 *)(dst + a_dst[i]) = va[i];
      *(u32x4 *)(dst + b_dst[i]) = vb[i];
    }
  };

  f32x4 acc[NBM][NBN];
#pragma unroll
  for (int i = 0; i < NBM; ++i)
#pragma unroll
    for (int j = 0; j < NBN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  unsigned char *const stages = smem + group * GROUP_BYTES;
  const int frag = r * 128 + ((q ^ swz(r)) << 4);  // (wave tiles start on multiples of 16 rows)
  int tr[NBN];
  if constexpr (KN) {
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
      const int krow = q * 8 + (r >> 2), c = (wn * TN + j * 16) / 8 + ((r & 3) >> 1);
      tr[j] = OPERAND + krow * ROWB + ((c ^ swz_kn(krow)) << 4) + (r & 1) * 8;
    }
  }
  auto multiply = [&](const unsigned char *st) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // 32 of the tile's 64 k (column 4 h + q: the swizzle's exclusive-or leaves bit 2 to h)
      u32x4 fa[NBM], fb[NBN];
#pragma unroll
      for (int i = 0; i < NBM; ++i) fa[i] = *(const u32x4 *)(st + (wm * TM + i * 16) * 128 + (frag ^ (h * 64)));
#pragma unroll
      for (int j = 0; j < NBN; ++j) {
        if constexpr (KN) {
          const unsigned char *p = st + tr[j] + h * 32 * ROWB;
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(p + 4 * ROWB));
          const u32x2 lo2 = __builtin_bit_cast(u32x2, lo), hi2 = __builtin_bit_cast(u32x2, hi);
          fb[j] = u32x4{lo2[0], lo2[1], hi2[0], hi2[1]};
        } else {
          fb[j] = *(const u32x4 *)(st + OPERAND + (wn * TN + j * 16) * 128 + (frag ^ (h * 64)));
        }
      }
#pragma unroll
      for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j) acc[i][j] = Mfma16<DT>::run(fb[j], fa[i], acc[i][j]);
    }
  };

  // group g takes K tiles g, g + GROUPS, ...; every group runs the same number of rounds (the barriers are the
  // workgroup's), with tiles of zeros behind the last one
  const int rounds = ((K + 63) / 64 + GROUPS - 1) / GROUPS;
  auto k_of = [&](int t) { return min(t * GROUPS + group, rounds * GROUPS) * 64; };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(d, k_of(d));
  auto round = [&](auto slot_c, int t) __attribute__((always_inline)) {
    constexpr int slot = decltype(slot_c)::value;
    unsigned char *st = stages + (t & 1) * STAGE;
    store(slot, st, k_of(t));
    load(slot, k_of(t + DEPTH));
    // the stage is written (nobody reads it: its last readers passed the previous barrier); the loads stay in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    multiply(st);
  };
  static_assert(DEPTH == 2 || DEPTH == 4, "the unrolled rounds below");
  for (int t = 0; t < rounds;) {
    round(std::integral_constant<int, 0>{}, t);
    if (++t >= rounds) break;
    round(std::integral_constant<int, 1>{}, t);
    if constexpr (DEPTH == 4) {
      if (++t >= rounds) break;
      round(std::integral_constant<int, 2>{}, t);
      if (++t >= rounds) break;
      round(std::integral_constant<int, 3>{}, t);
    }
    ++t;
  }
  __syncthreads();
  // sums of group g: T rows of PITCH floats over its stages; lane of block (i, j): row 16 i + r, channels 16 j + 4 q .. + 3
  float *sums = (float *)stages + (wm * TM + r) * PITCH + wn * TN + q * 4;
#pragma unroll
  for (int i = 0; i < NBM; ++i)
#pragma unroll
    for (int j = 0; j < NBN; ++j) *(f32x4 *)(sums + i * 16 * PITCH + j * 16) = acc[i][j];
  __syncthreads();
#pragma nounroll
  for (int p = threadIdx.x; p < T * (T / 8); p += NT) {
    const int row = p / (T / 8), n = n0 + (p % (T / 8)) * 8, m = m0 + row;
    if (m >= M || n >= N) continue;
    const float *src = (const float *)smem + row * PITCH + (p % (T / 8)) * 8;
    f32x4 lo = *(const f32x4 *)src, hi = *(const f32x4 *)(src + 4);
#pragma unroll
    for (int g = 1; g < GROUPS; ++g) {
      lo += *(const f32x4 *)(src + g * (GROUP_BYTES / 4));
      hi += *(const f32x4 *)(src + g * (GROUP_BYTES / 4) + 4);
    }
    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    apply_epilogue<8>(v, m, n, N - n, args.epi);
    store_from_float<8>(args.C, args.out_dtype, (long long)m * args.ldc + n, N - n, v);
  }
}

template <int DT, int T, int WN, int GROUPS, int DEPTH, bool KN>
static int launch_one(const ContractionArgs &a, hipStream_t stream) {
  constexpr int lds = GROUPS * ragged_group_bytes(T);
  auto kfn = gemm_ragged_kernel<DT, T, WN, GROUPS, DEPTH, KN>;
  static bool attr_done = false;
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
    attr_done = true;
  }
  hipLaunchKernelGGL(kfn, dim3((unsigned)(a.grid_m * a.grid_n)), dim3(GROUPS * WN * 128), lds, stream, a);
  return (int)hipGetLastError();
}

template <int DT, bool KN>
static int launch_form(const ContractionArgs &a, int tile, int groups, hipStream_t stream) {
  if (tile == 128) return launch_one<DT, 128, 4, 1, 2, KN>(a, stream);
  return groups == 2 ? launch_one<DT, 64, 2, 2, 4, KN>(a, stream) : launch_one<DT, 64, 2, 1, 4, KN>(a, stream);
}

template <int DT>
static int launch_type(const ContractionArgs &a, bool b_ncontig, int tile, int groups, hipStream_t stream) {
  return b_ncontig ? launch_form<DT, true>(a, tile, groups, stream) : launch_form<DT, false>(a, tile, groups, stream);
}

int launch_gemm_ragged(const ContractionArgs &a, int dtype, bool b_ncontig, int tile, int groups, hipStream_t stream) {
  if (a.M < 1 || a.N < 1 || a.K < 1 || a.a_bytes < 16 || a.b_bytes < 16) return (int)hipErrorInvalidValue;
  return dtype == DT_F16 ? launch_type<DT_F16>(a, b_ncontig, tile, groups, stream) : launch_type<DT_BF16>(a, b_ncontig, tile, groups, stream);
}

// The same for fp32, A and B by rows: K tiles of 32 through registers, DEPTH ahead, 64x64 of C per group of four waves, a wave
// 32x32 of it on 32x32x2 MFMAs.  An MFMA's two k are its lane halves': half g takes k 16 g + j of the tile in MFMA j,
// so that a lane reads four of them from a row of A at once.  1000x900x1030 28.9 us (replayed graph) against 42.8 from padded
// copies of both operands, 33x65x16 6.4 against 11.0.  Bound by the walk over K: 0.7 us per K tile and group where a CU
// has one workgroup, of which the MFMAs' issue is 0.43.  Four groups measured level with two (1000x900x1030).
//
// Reads stay inside the extents ((rows - 1) * pitch + row length, at least 4 elements) as above.
typedef f32x4 f32x4_any __attribute__((aligned(4)));

__device__ __forceinline__ f32x4 drop_front(f32x4 p, unsigned s) {
  const f32x4 h = {p[1], p[2], p[3], 0.0f};
  p = (s & 1) ? h : p;
  const f32x4 w = {p[2], p[3], 0.0f, 0.0f};
  return (s & 2) ? w : p;
}
__device__ __forceinline__ f32x4 keep_front(f32x4 p, int keep) {
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = i < keep ? p[i] : 0.0f;
  return p;
}

template <int GROUPS>
__global__ void __launch_bounds__(GROUPS * 256) gemm_ragged_f32_kernel(const ContractionCore args) {
  constexpr int T = 64, GT = 256, NP = 2, DEPTH = 4, NT = GROUPS * GT;
  constexpr int A_PITCH = 36;                  // floats: 16 rows at one column lie in 16 different groups of four banks
  constexpr int A_FLOATS = T * A_PITCH, STAGE = A_FLOATS + 32 * T, GROUP_FLOATS = 2 * STAGE;
  constexpr int PITCH = T + 4;
  static_assert(T * PITCH <= GROUP_FLOATS, "a group's sums go over its stages");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x % GT, lane = threadIdx.x & 63, wave = tid >> 6;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
  const int wm = wave & 1, wn = wave >> 1, r = lane & 31, g = lane >> 5;
  int tile_m, tile_n;
  tile_coordinates(args, tile_m, tile_n);
  const int m0 = tile_m * T, n0 = tile_n * T;
  const int M = args.M, N = args.N, K = args.K;
  const float *A = (const float *)args.A, *B = (const float *)args.B;
  const unsigned a_last = args.a_bytes / 4 - 4, b_last = args.b_bytes / 4 - 4;  // where the last whole piece starts
  const unsigned ldb = (unsigned)args.ldb;

  unsigned a_off[NP], b_off[NP], a_dst[NP], b_dst[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = tid + i * GT, row = p >> 3, krow = p >> 4, cn = (p & 15) * 4;
    a_off[i] = (unsigned)min(m0 + row, M - 1) * (unsigned)args.lda + (p & 7) * 4;
    a_dst[i] = row * A_PITCH + (p & 7) * 4;
    b_off[i] = (unsigned)krow * ldb + n0 + cn;
    // (the two halves of a wave read rows 16 apart: the lower 16 rows have their two 32 columns exchanged)
    b_dst[i] = A_FLOATS + krow * T + (cn ^ ((krow >> 4) << 5));
  }
  const int kcol = (tid & 7) * 4;

  f32x4 ra[DEPTH][NP], rb[DEPTH][NP];
  auto load = [&](int slot, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      ra[slot][i] = *(const f32x4_any *)(A + min(a_off[i] + (unsigned)k0, a_last));
      rb[slot][i] = *(const f32x4_any *)(B + min(b_off[i] + (unsigned)k0 * ldb, b_last));
    }
  };
  auto store = [&](int slot, float *dst, int k0) __attribute__((always_inline)) {
    f32x4 va[NP], vb[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      va[i] = ra[slot][i];
      vb[i] = rb[slot][i];
    }
    if (k0 + 36 > K) {  // (a row of B within 4 elements of the end may need the shift in front of the last tile)
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const unsigned oa = a_off[i] + (unsigned)k0, ob = b_off[i] + (unsigned)k0 * ldb;
        va[i] = keep_front(drop_front(va[i], oa - min(oa, a_last)), K - k0 - kcol);
        vb[i] = keep_front(drop_front(vb[i], ob - min(ob, b_last)), k0 + ((tid + i * GT) >> 4) < K ? 4 : 0);
      }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      *(f32x4 *)(dst + a_dst[i]) = va[i];
      *(f32x4 *)(dst + b_dst[i]) = vb[i];
    }
  };

  f32x16 acc[4] = {};  // four chains of MFMAs: none waits for the one before, and the sums round less
  float *const stages = (float *)smem + group * GROUP_FLOATS;
  const int fa_at = (wm * 32 + r) * A_PITCH + g * 16;
  const int fb_at = A_FLOATS + g * 16 * T + ((wn * 32 + r) ^ (g << 5));
  auto multiply = [&](const float *st) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 fa = *(const f32x4 *)(st + fa_at + j * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(st[fb_at + (j * 4 + e) * T], fa[e], acc[e], 0, 0, 0);
    }
  };

  const int rounds = ((K + 31) / 32 + GROUPS - 1) / GROUPS;  // the same for every group, tiles of zeros behind the last one
  auto k_of = [&](int t) { return min(t * GROUPS + group, rounds * GROUPS) * 32; };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(d, k_of(d));
  auto round = [&](auto slot_c, int t) __attribute__((always_inline)) {
    constexpr int slot = decltype(slot_c)::value;
    float *st = stages + (t & 1) * STAGE;
    store(slot, st, k_of(t));
    load(slot, k_of(t + DEPTH));
    // (as above: the stage's last readers passed the previous barrier, the loads stay in flight)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    multiply(st);
  };
  for (int t = 0; t < rounds; ++t) {
    round(std::integral_constant<int, 0>{}, t);
    if (++t >= rounds) break;
    round(std::integral_constant<int, 1>{}, t);
    if (++t >= rounds) break;
    round(std::integral_constant<int, 2>{}, t);
    if (++t >= rounds) break;
    round(std::integral_constant<int, 3>{}, t);
  }
  __syncthreads();
  // a lane's registers 4 i .. 4 i + 3: row r, columns 8 i + 4 g .. + 3 of the wave's 32x32
  const f32x16 sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  float *sums = stages + (wm * 32 + r) * PITCH + wn * 32 + g * 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) *(f32x4 *)(sums + i * 8) = f32x4{sum[4 * i], sum[4 * i + 1], sum[4 * i + 2], sum[4 * i + 3]};
  __syncthreads();
#pragma nounroll
  for (int p = threadIdx.x; p < T * (T / 4); p += NT) {
    const int row = p / (T / 4), n = n0 + (p % (T / 4)) * 4, m = m0 + row;
    if (m >= M || n >= N) continue;
    const float *src = (const float *)smem + row * PITCH + (p % (T / 4)) * 4;
    f32x4 s = *(const f32x4 *)src;
#pragma unroll
    for (int o = 1; o < GROUPS; ++o) s += *(const f32x4 *)(src + o * GROUP_FLOATS);
    float v[4] = {s[0], s[1], s[2], s[3]};
    apply_epilogue<4>(v, m, n, N - n, args.epi);
    store_from_float<4>(args.C, args.out_dtype, (long long)m * args.ldc + n, N - n, v);
  }
}

template <int GROUPS>
static int launch_f32_one(const ContractionArgs &a, hipStream_t stream) {
  constexpr int lds = GROUPS * 2 * (64 * 36 + 32 * 64) * 4;
  auto kfn = gemm_ragged_f32_kernel<GROUPS>;
  static bool attr_done = false;
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
    attr_done = true;
  }
  hipLaunchKernelGGL(kfn, dim3((unsigned)(a.grid_m * a.grid_n)), dim3(GROUPS * 256), lds, stream, a);
  return (int)hipGetLastError();
}

int launch_gemm_ragged_f32(const ContractionArgs &a, int groups, hipStream_t stream) {
  if (a.M < 1 || a.N < 1 || a.K < 1 || a.a_bytes < 16 || a.b_bytes < 16) return (int)hipErrorInvalidValue;
  return groups == 2 ? launch_f32_one<2>(a, stream) : launch_f32_one<1>(a, stream);
}

}  // namespace tracea_amd
