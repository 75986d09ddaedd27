// Contraction with few rows (token-by-token decoding): C[m, n] as in
// hf_mmad.h with M up to about 128, where the 256x256 tiles of the ring
// kernels leave most of the chip idle (N = 4096 gives 16 workgroups).
//
// Such a call reads its weights once and multiplies little, so what bounds it
// is how fast every CU can pull its share of A and B through its LDS.  A
// workgroup owns 16 or 32 columns and its waves split K, so N = 4096 gives
// every CU one, nothing is read twice by a workgroup and no sum crosses
// workgroups.  int8 sums are exact in any order; f32 sums are one partial sum
// per wave over its K slices, added in wave order.
// Measured, W8A8 at N = K = 4096, B [N, K], against 40 us for the 256x256
// ring: M = 16 4.75 us (an empty launch is 2.3; 16.8 MB of weights are 3.3 us
// at the rate of a large copy), M = 32 5.1, M = 64 6.1, M = 128 8.5; bf16 7.1,
// 7.6, 8.4, 11.9 us.  B [K, N] at M = 16: 9.2 us (16-byte pieces of each
// k-row).  Loading the operands straight into registers instead (16 rows x
// 64 bytes per load) took 5.8, 7.6 and 11.3 us at M = 16, 32 and 64.
#pragma once
#include "hf_mmad.h"

namespace hf {

typedef float v4f __attribute__((ext_vector_type(4)));

// 16x16 matrix-core step over 64 bytes of K: lane l feeds 16 bytes of row
// (column) l % 16 at byte 16 (l / 16); accumulator register r of lane l is
// row 4 (l / 16) + r, column l % 16.
template <int MK> struct Mfma16;
template <> struct Mfma16<MK_I8> {
  using acc_t = v4i;
  using scalar_t = int32_t;
  __device__ __forceinline__ static acc_t run(v4i a, v4i b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma16<MK_BF16> {
  using acc_t = v4f;
  using scalar_t = float;
  __device__ __forceinline__ static acc_t run(v4i a, v4i b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  }
};
template <> struct Mfma16<MK_F16> {
  using acc_t = v4f;
  using scalar_t = float;
  __device__ __forceinline__ static acc_t run(v4i a, v4i b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
  }
};

// One workgroup of NW waves owns 16 MT rows x 16 NT columns of C.  Wave w
// takes the 128-byte K slices w, w + NW, ... with a ring of S slots of its
// own in LDS, filled by LDS DMA: no barrier before the final sum, and the
// ring of every wave is in flight at once.
// A is [M, K]; B is [N, K], or [K, N] with BKN (N a multiple of 16 bytes); K
// spans a multiple of 64 bytes.
//   Row-major operand: a DMA instruction carries 8 rows x 128 bytes, whole
//     lines; granule g (16 bytes) of row r at position g ^ ((r >> 1) & 7) of
//     the row, so the 16 rows of a fragment read hit 16 bank groups.
//   B [K, N]: a slice is 128 (16-bit: 64) k-rows of 16 NT columns as they
//     lie; transposing LDS reads (as in hf_mmad.h) form the operand.
//     Granule g of k-row r is at g ^ skn_swz(r): the k-rows of one transposing
//     read (8 bytes, or 4 of 16-bit) on different bank groups.
// Grid: 8 * ceil(ceil(N / (16 NT)) / 8) workgroups per row tile; workgroup b
// runs on XCD b % 8 and each XCD takes consecutive column tiles, so that one
// L2 fetches the lines of a [K, N] B that neighbouring tiles share.
template <int MK, typename Epi, bool BKN, int MT, int NT, int NW, typename ElemT, typename Args>
__device__ __forceinline__ void mmad_skinny(const ElemT *__restrict__ A, const ElemT *__restrict__ B,
                                            typename Epi::out_t *__restrict__ out, int64_t M, int64_t N, int64_t K,
                                            const Args &P) {
  using Op = Mfma16<MK>;
  using acc_t = typename Op::acc_t;
  using scalar_t = typename Op::scalar_t;
  constexpr int ESZ = sizeof(ElemT), TM = 16 * MT, TN = 16 * NT;
  constexpr int SLOT = 2048 * (MT + NT), DA = 2 * MT, DPS = 2 * (MT + NT); // bytes and DMA instructions per slice
  constexpr int SMAX = 160 * 1024 / (NW * SLOT), S = SMAX < 5 ? SMAX : 5;
  static_assert(S >= 2, "the ring does not fit the LDS");
  static_assert(NW * MT * NT * 1024 <= NW * S * SLOT, "partial sums reuse the ring");
  __shared__ __attribute__((aligned(1024))) char lds[NW * S * SLOT];
  const int tn = (int)((N + TN - 1) / TN), per = (tn + 7) / 8;
  const int b = (int)blockIdx.x % (8 * per);
  const int tj = b % 8 * per + b / 8;
  if (tj >= tn) return;
  const int64_t m0 = (int64_t)((int)blockIdx.x / (8 * per)) * TM, n0 = (int64_t)tj * TN;
  const int64_t Kb = K * ESZ;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
  const int ns = (int)((Kb + 127) / 128);          // K slices; the last may be half a slice
  const int n = ns > wave ? (ns - wave + NW - 1) / NW : 0; // this wave's
  const bool half = Kb % 128 != 0;
  const char *Ab = reinterpret_cast<const char *>(A), *Bb = reinterpret_cast<const char *>(B);

  constexpr int LPR = NT * ESZ, G = LPR;          // B [K, N]: lanes (granules) per k-row
  auto skn_swz = [](int kr) { return ESZ == 1 ? (G == 4 ? (kr >> 2) & 3 : 0) : (G == 8 ? ((kr >> 1) & 3) << 1 : 0); };
  // DMA d of a slice: this lane's source as an offset from the slice's
  // wave-uniform base (rows and columns past the end re-read valid ones,
  // whose results are not stored), and whether it lies in the second half
  // of the slice (a half slice re-reads the first: those bytes are not
  // multiplied)
  uint32_t dofs[DPS];
  bool hi[DPS];
#pragma unroll
  for (int d = 0; d < DPS; ++d) {
    if (d < DA || !BKN) {
      const int r = 8 * (d < DA ? d : d - DA) + lane / 8, g = (lane % 8) ^ ((r >> 1) & 7);
      const int64_t rows = d < DA ? M : N, row0 = d < DA ? m0 : n0;
      const int64_t row = row0 + r < rows ? row0 + r : rows - 1;
      dofs[d] = (uint32_t)((row - row0) * Kb + g * 16);
      hi[d] = g >= 4;
    } else {
      const int kr = (d - DA) * (64 / LPR) + lane / LPR, g = (lane % LPR) ^ skn_swz(kr);
      int64_t col = n0 + g * (16 / ESZ);
      col = col + 16 / ESZ <= N ? col : N - 16 / ESZ;
      dofs[d] = (uint32_t)((kr * N + col) * ESZ);
      hi[d] = kr >= 64 / ESZ;
    }
  }
  const uint32_t back_b = BKN ? (uint32_t)(64 * N) : 64u; // from the second half of a slice to the first
  const char *const a0 = Ab + m0 * Kb, *const b0 = BKN ? Bb : Bb + n0 * Kb;
  const int64_t bstep = BKN ? 128 * N : 128;
  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)&lds[0] + (uint32_t)(wave * S * SLOT);
  auto issue = [&](int i) { // the wave's i-th slice into slot i % S
    const int s = wave + i * NW;
    const uint32_t slot = ring + (uint32_t)(i % S * SLOT);
    const bool tail = half && s == ns - 1;
#pragma unroll
    for (int d = 0; d < DPS; ++d) {
      uint32_t off = dofs[d];
      if (tail && hi[d]) off -= d < DA ? 64u : back_b;
      mmd_dma16_off(d < DA ? a0 + (int64_t)s * 128 : b0 + (int64_t)s * bstep, off,
                    __builtin_amdgcn_readfirstlane(slot + (uint32_t)(d * 1024)));
    }
  };

  acc_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = acc_t{};

  // 16-byte fragments of a slot: k-block kb (64 bytes of K), 16-row tile t
  const int q = lane / 16, j16 = lane % 16;
  auto frag = [&](uint32_t base, int t, int kb) -> v4i {
    const int r = 16 * t + j16, g = 4 * kb + q;
    return *(__attribute__((address_space(3))) const v4i *)(uintptr_t)(base + (uint32_t)((8 * r + (g ^ ((r >> 1) & 7))) * 16));
  };
  auto frag_kn = [&](uint32_t base, int t, int kb) -> v4i {
    typedef int v2i_ __attribute__((ext_vector_type(2)));
    typedef short v4s_ __attribute__((ext_vector_type(4)));
    v4i f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v2i_ x;
      if constexpr (ESZ == 1) {
        const int kr = 64 * kb + 16 * q + 8 * h + j16 / 2;
        const uint32_t at = base + (uint32_t)((kr * LPR + (t ^ skn_swz(kr))) * 16 + 8 * (j16 % 2));
        x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i_ *)(uintptr_t)at);
      } else {
        const int kr = 32 * kb + 8 * q + 4 * h + j16 / 4;
        const uint32_t at = base + (uint32_t)((kr * LPR + ((2 * t + (j16 % 4) / 2) ^ skn_swz(kr))) * 16 + 8 * (j16 % 2));
        x = __builtin_bit_cast(v2i_, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s_ *)(uintptr_t)at));
      }
      f[2 * h] = x.x;
      f[2 * h + 1] = x.y;
    }
    return f;
  };
  // waits until at most `ahead` slices are in flight
  auto wait_ahead = [&](int ahead) {
    if (ahead >= S - 1) { mmd_wait_vm<(S - 1) * DPS>(); return; }
    if constexpr (S > 4) if (ahead == 3) { mmd_wait_vm<3 * DPS>(); return; }
    if constexpr (S > 3) if (ahead == 2) { mmd_wait_vm<2 * DPS>(); return; }
    if constexpr (S > 2) if (ahead == 1) { mmd_wait_vm<DPS>(); return; }
    mmd_wait_vm<0>();
  };

#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < n) issue(i);
#pragma unroll 1
  for (int i = 0; i < n; ++i) {
    wait_ahead(n - 1 - i);
    const uint32_t slot = ring + (uint32_t)(i % S * SLOT);
    v4i fa[2][MT], fb[2][NT];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int t = 0; t < MT; ++t) fa[kb][t] = frag(slot, t, kb);
#pragma unroll
      for (int t = 0; t < NT; ++t) fb[kb][t] = BKN ? frag_kn(slot + DA * 1024, t, kb) : frag(slot + DA * 1024, t, kb);
    }
    if (i + S < n) {
      // the slot has been read (the fragments are in registers) before it is filled again
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue(i + S);
    }
    const bool tail = half && wave + i * NW == ns - 1;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
      if (kb == 0 || !tail) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int u = 0; u < NT; ++u) acc[t][u] = Op::run(fa[kb][t], fb[kb][u], acc[t][u]);
      }
  }
  __syncthreads(); // every wave is done with its ring

  // partial sums [wave][16x16 tile][lane][4 rows], then one output element
  // per thread and step: consecutive threads take consecutive columns
  acc_t *red = reinterpret_cast<acc_t *>(lds);
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < NT; ++u) red[((wave * MT + t) * NT + u) * 64 + lane] = acc[t][u];
  __syncthreads();
  const scalar_t *rs = reinterpret_cast<const scalar_t *>(lds);
#pragma unroll 4
  for (int o = threadIdx.x; o < TM * TN; o += NW * 64) {
    const int r = o / TN, c = o % TN, rr = r % 16;
    const int64_t m = m0 + r, nn = n0 + c;
    if (m >= M || nn >= N) continue;
    const int at = ((r / 16 * NT + c / 16) * 64 + rr / 4 * 16 + c % 16) * 4 + rr % 4;
    scalar_t s = rs[at];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += rs[w * MT * NT * 256 + at];
    out[m * N + nn] = Epi::apply(s, m, nn, Epi::row(m, P), Epi::col(nn, P), P);
  }
}

} // namespace hf
