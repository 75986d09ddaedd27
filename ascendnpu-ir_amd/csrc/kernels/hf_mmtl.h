// Contraction tiles smaller than the 256x256 of hf_mmad.h, for shapes with
// too few of those to fill the chip (one 256x256 tile per CU needs M N of
// 4096 x 4096).
//
// Such a call is bound by what a CU pulls through its LDS: (TM + TN) K bytes
// per tile.  Measured parts of a 128x128 tile's 128-byte step (4 waves, W8A8):
// DMA alone 0.31 us (105 GB/s per CU), fragment reads and multiplies alone
// 0.41 us, together 0.58 us.  So tiles are as large as still gives every CU
// one (pickTile in the lowering holds the measured times).  W8A8 at N = K =
// 4096, before (256x256 ring) and after: M = 333 43 -> 13.8 us, M = 512 41.6
// -> 15.5, M = 1024 41.9 -> 24.5, M = 2048 46 -> 40.7; bf16 74 -> 24.7, 74 ->
// 26.9, 74 -> 41, 78 -> 72.6 us; block-scaled fp8 M = 128 49 -> 13.9 us, M =
// 1024 55 -> 30 us, fp4 32 -> 8.7 and 39 -> 19 us.
// Reading the next half slice's (or slice's) fragments under the multiplies
// and spreading the DMAs between them changed these by -3 .. +15 %: the
// other waves of the CU fill the gaps already.
#pragma once
#include "hf_mmsk.h"

namespace hf {

// Waits until at most `ahead` (< S) groups of CNT memory operations are in flight.
template <int S, int CNT> __device__ __forceinline__ void mmt_wait_ahead(int ahead) {
  if constexpr (S > 1) {
    if (ahead >= S - 1) { mmd_wait_vm<(S - 1) * CNT>(); return; }
    mmt_wait_ahead<S - 1, CNT>(ahead);
  } else {
    mmd_wait_vm<0>();
  }
}

// A wave-uniform pointer in scalar registers, as mmd_dma16_off's base has to be:
// the compiler selects between two of them in vector registers at times.
__device__ __forceinline__ const char *mmt_uniform(const char *p) {
  const uint64_t u = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return reinterpret_cast<const char *>((uint64_t)hi << 32 | lo);
}

// One workgroup of WM x WN waves per TM x TN tile of C; wave (wm, wn) holds
// TM / WM rows and TN / WN columns as 32x32 matrix-core tiles.  K advances in
// slices of 128 bytes (the last may be half) through a ring of S stages:
// step s waits for its slice, passes the one barrier of the step (which also
// says that everyone has read slice s - 1), refills the slot of slice s - 1
// with slice s + S - 1 and multiplies slice s.
// KG > 1: a stage holds KG slices and KG groups of WM x WN waves multiply one
// each, so that there are as many times fewer barriers and waits, and more
// waves to fill them; the groups' partial sums meet in LDS at the end.  It
// pays while a CU has one tile (N = K = 4096, 64x64 KG 1 -> 2 at M = 200: W8A8
// 11.8 -> 10.9 us, bf16 20.6 -> 17.5) and, of a [K, N] B, against the two
// resident narrower tiles too (M = 333: W8A8 64x64 KG 1 -> 64x128 KG 2 16.0 ->
// 14.8 us, bf16 27 -> 24); of an [N, K] B those are as fast (13.5 against 14.6,
// 23.8 against 23.6).
// Operands as in hf_mmad.h: A [M, K] row-major; B [N, K] row-major, or
// [K, N] with BKN.  Row-major slices: granule g (16 bytes) of row r at
// position g ^ ((r >> 1) & 7).  K-major slices: k-rows of TN columns as they
// lie, granule g of k-row r at g ^ swz(r), where swz spreads the k-rows that
// one transposing read (two groups of 16 lanes) touches over the 16 bank
// groups and leaves the granule bits apart that tell those groups.
// Block-scaled kinds: SA [M, K/32], SB [N, K/32] e8m0 bytes ride the ring,
// 4 (fp4: 8) bytes per row and stage.
template <int MK, typename Epi, bool BKN, int TM, int TN, int WM, int WN, int S, int KG = 1, typename ElemT, typename Args>
__device__ __forceinline__ void mmad_tile(const ElemT *__restrict__ A, const ElemT *__restrict__ B,
                                          typename Epi::out_t *__restrict__ out, int64_t M, int64_t N, int64_t K, const Args &P,
                                          const uint8_t *__restrict__ SA = nullptr, const uint8_t *__restrict__ SB = nullptr) {
  constexpr bool MX = mk_is_mx(MK), FP4 = mk_is_fp4(MK);
  constexpr int NWD = FP4 ? 2 : 1; // scale words per row per stage
  static_assert(!MX || BKN, "block-scaled operands come with B [K, N]");
  using Op = typename std::conditional<MX, MfmaMx<(MX ? MK : MK_MX)>, MfmaOp<(MX ? MK_I8 : MK)>>::type;
  using acc_t = typename Op::acc_t;
  using O = typename Epi::out_t;
  constexpr int ESZ = sizeof(ElemT), NWG = WM * WN, NW = NWG * KG, IT = TM / WM / 32, JT = TN / WN / 32;
  constexpr int SL = (TM + TN) * 128, SLOT = KG * SL;                         // bytes of a slice, of a stage
  constexpr int DA = TM / 8, DS = (TM + TN) / 8, DT = KG * DS;                // DMA instructions: A, slice, stage
  static_assert(!MX || KG == 1, "block-scaled kinds: one slice per stage");
  static_assert(DT % NW == 0, "every wave issues as many DMA instructions");
  constexpr int DW = DT / NW;                                               // per wave and stage
  constexpr int SCE = (TM + TN + 63) / 64 * 64;                               // scale entries: A rows, B columns, padding
  constexpr int SCI = MX ? SCE / 64 * NWD : 0, SCW = (SCI + NW - 1) / NW; // scale DMAs (64 entries) per stage, per wave
  constexpr int DPS = DW + SCW;
  constexpr int SCB = MX ? SCE * 4 * NWD : 0; // scale bytes per stage
  constexpr int LDSB = S * (SLOT + SCB);
  static_assert(LDSB <= 160 * 1024 && S >= 3 && (S - 1) * DPS < 64, "ring");
  __shared__ __attribute__((aligned(1024))) char lds[LDSB];
  const int tmt = (int)((M + TM - 1) / TM), tnt = (int)((N + TN - 1) / TN);
  // consecutive column tiles (all row tiles of them) per XCD: workgroup b
  // runs on XCD b % 8 (the grid may hold more than 8 per workgroups)
  const int per = (tnt * tmt + 7) / 8, lin = (int)blockIdx.x % 8 * per + (int)blockIdx.x / 8;
  if ((int)blockIdx.x / 8 >= per || lin >= tnt * tmt) return;
  const int ti = lin % tmt, tj = lin / tmt;
  const int64_t m0 = (int64_t)ti * TM, n0 = (int64_t)tj * TN;
  const int64_t Kb = K * ESZ;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
  const int kg = wave / NWG, wm = wave % NWG / WN, wn = wave % WN; // K group, place in the tile
  const int nslices = (int)((Kb + 127) / 128), nsteps = (nslices + KG - 1) / KG;
  const bool half = Kb % 128 != 0;
  const char *Ab = reinterpret_cast<const char *>(A), *Bb = reinterpret_cast<const char *>(B);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)&lds[0];

  constexpr int G = TN * ESZ / 16, RPI = 64 / G > 0 ? 64 / G : 1; // B [K, N]: granules per k-row, k-rows per DMA
  static_assert(!BKN || G <= 64, "a DMA instruction carries whole k-rows");
  auto swz = [](int kr) {
    if constexpr (ESZ == 1) return G >= 16 ? ((kr & 7) << 1) | ((kr >> 3) & 1) : G == 8 ? ((kr >> 1) & 3) << 1 : G == 4 ? ((kr >> 2) & 1) << 1 : 0;
    else return G >= 16 ? (kr & 3) << 2 : G == 8 ? ((kr >> 1) & 1) << 2 : 0;
  };
  // this lane's source of the wave's DMA d, as an offset from the operand's
  // base of the slice; rows and columns past the end re-read valid ones; in
  // a half slice the second half re-reads the first (those k are not
  // multiplied)
  uint32_t dofs[DW];
  uint32_t back[DW];
#pragma unroll
  for (int d = 0; d < DW; ++d) {
    const int x = KG == 1 ? wave + d * NW : (wave + d * NW) % DS; // instruction of its slice (A first)
    const bool isA = x < DA;
    const int64_t rows = isA ? M : N, row0 = isA ? m0 : n0;
    if (isA || !BKN) {
      const int r = 8 * (isA ? x : x - DA) + lane / 8, g = (lane % 8) ^ ((r >> 1) & 7);
      const int64_t row = row0 + r < rows ? row0 + r : rows - 1;
      dofs[d] = (uint32_t)((row - row0) * Kb + g * 16);
      back[d] = g >= 4 ? 64u : 0u;
    } else {
      const int kr = (x - DA) * RPI + lane / G, g = (lane % G) ^ swz(kr);
      int64_t col = n0 + g * (16 / ESZ);
      col = col + 16 / ESZ <= N ? col : N - 16 / ESZ;
      dofs[d] = (uint32_t)((kr * N + col) * ESZ);
      back[d] = kr >= 64 / ESZ ? (uint32_t)(64 * N) : 0u;
    }
  }
  // each instruction's slice of the stage in flight next, its address and step
  const char *src[DW];
  int64_t step[DW];
  int next[DW];
#pragma unroll
  for (int d = 0; d < DW; ++d) {
    const int y = wave + d * NW, x = KG == 1 ? y : y % DS;
    next[d] = KG == 1 ? 0 : y / DS;
    step[d] = x < DA || !BKN ? 128 : 128 * N;
    if (next[d] >= nslices) next[d] = nslices - 1; // (a slice past the end: the last again, not multiplied)
    src[d] = mmt_uniform((x < DA ? Ab + m0 * Kb : BKN ? Bb : Bb + n0 * Kb) + next[d] * step[d]);
  }
  auto issue = [&](int s) { // s = 0, 1, 2, ...
    const uint32_t slot = lds0 + (uint32_t)(s % S * SLOT);
#pragma unroll
    for (int d = 0; d < DW; ++d) {
      mmd_dma16_off(src[d], half && next[d] == nslices - 1 ? dofs[d] - back[d] : dofs[d],
                    __builtin_amdgcn_readfirstlane(slot + (uint32_t)((wave + d * NW) * 1024)));
      const int adv = KG == 1 || next[d] + KG < nslices ? KG : nslices - 1 - next[d];
      src[d] += adv * step[d];
      next[d] += adv;
    }
    if constexpr (MX) {
#pragma unroll
      for (int d = 0; d < SCW; ++d) {
        int x = wave + d * NW; // (block of 64 entries) * NWD + word; surplus instructions repeat the last
        x = x < SCI ? x : SCI - 1;
        const int blk = x / NWD, w = x % NWD, e = 64 * blk + lane;
        const bool isA = e < TM;
        const int64_t rows = isA ? M : N;
        int64_t row = isA ? m0 + e : n0 + (e - TM);
        row = row < rows ? row : rows - 1;
        mmd_dma4((isA ? SA : SB) + row * (K / (32 / NWD)) + 4 * NWD * (int64_t)s + 4 * w,
                 __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(S * SLOT + s % S * SCB + (w * SCE + 64 * blk) * 4)));
      }
    }
  };

  acc_t acc[IT][JT];
#pragma unroll
  for (int i = 0; i < IT; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[i][j] = acc_t{};

  // fragment of k-block kb (32 bytes of K) of the 32-row block at row r0
  auto frag = [&](uint32_t base, int r0, int kb) -> v4i {
    const int r = r0 + lane % 32, g = 2 * kb + lane / 32;
    return *(__attribute__((address_space(3))) const v4i *)(uintptr_t)(base + (uint32_t)((8 * r + (g ^ ((r >> 1) & 7))) * 16));
  };
  auto frag_kn = [&](uint32_t base, int c0, int kb) -> v4i {
    typedef int v2i_ __attribute__((ext_vector_type(2)));
    typedef short v4s_ __attribute__((ext_vector_type(4)));
    const int q = lane / 16, j = lane % 16;
    v4i f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v2i_ x;
      if constexpr (ESZ == 1) {
        const int kr = kb * 32 + 16 * (q / 2) + 8 * h + j / 2, g = c0 / 16 + q % 2;
        x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
            (__attribute__((address_space(3))) v2i_ *)(uintptr_t)(base + (uint32_t)((kr * G + (g ^ swz(kr))) * 16 + 8 * (j % 2))));
      } else {
        const int kr = kb * 16 + 8 * (q / 2) + 4 * h + j / 4, g = c0 / 8 + 2 * (q % 2) + (j % 4) / 2;
        x = __builtin_bit_cast(v2i_, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4s_ *)(uintptr_t)(base + (uint32_t)((kr * G + (g ^ swz(kr))) * 16 + 8 * (j % 2)))));
      }
      f[2 * h] = x.x;
      f[2 * h + 1] = x.y;
    }
    return f;
  };

#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < nsteps) issue(s);
#pragma unroll 1
  for (int s = 0; s < nsteps; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    // slices s + 1 .. min(s + S - 2, nsteps - 1) may be in flight
    mmt_wait_ahead<S - 1, DPS>(nsteps - 1 - s);
    __syncthreads();
    if (s + S - 1 < nsteps) issue(s + S - 1);
    const uint32_t slot = lds0 + (uint32_t)(s % S * SLOT + kg * SL);
    const bool tail = half && s * KG + kg == nslices - 1;
    if (KG > 1 && s * KG + kg >= nslices) continue; // (no barrier follows in the loop body)
    uint32_t sa[IT][NWD], sb[JT][NWD];
    if constexpr (MX) {
      // this lane's scale words: byte 2 h (fp4: byte 2 kk of word h) is the
      // scale of its k in half h
      const uint32_t sc = lds0 + (uint32_t)(S * SLOT + s % S * SCB);
      auto word = [&](int row, int w) {
        return *(__attribute__((address_space(3))) const uint32_t *)(uintptr_t)(sc + (uint32_t)((w * SCE + row) * 4)) >> (8 * (lane / 32));
      };
#pragma unroll
      for (int w = 0; w < NWD; ++w) {
#pragma unroll
        for (int i = 0; i < IT; ++i) sa[i][w] = word(wm * (TM / WM) + 32 * i + lane % 32, w);
#pragma unroll
        for (int j = 0; j < JT; ++j) sb[j][w] = word(TM + wn * (TN / WN) + 32 * j + lane % 32, w);
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) { // the two halves of the slice
      if (h == 1 && tail) break;
      v4i fa[2][IT], fb[2][JT];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int i = 0; i < IT; ++i) fa[kk][i] = frag(slot, wm * (TM / WM) + 32 * i, 2 * h + kk);
#pragma unroll
        for (int j = 0; j < JT; ++j)
          fb[kk][j] = BKN ? frag_kn(slot + DA * 1024, wn * (TN / WN) + 32 * j, 2 * h + kk)
                          : frag(slot + DA * 1024, wn * (TN / WN) + 32 * j, 2 * h + kk);
      }
      if constexpr (MX && !FP4) {
#pragma unroll
        for (int i = 0; i < IT; ++i)
#pragma unroll
          for (int j = 0; j < JT; ++j) {
            const v8i a8 = mx_cat(fa[0][i], fa[1][i]), b8 = mx_cat(fb[0][j], fb[1][j]);
            acc[i][j] = h == 0 ? Op::template run<0>(a8, b8, acc[i][j], (int)sa[i][0], (int)sb[j][0])
                               : Op::template run<2>(a8, b8, acc[i][j], (int)sa[i][0], (int)sb[j][0]);
          }
      } else {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int i = 0; i < IT; ++i)
#pragma unroll
            for (int j = 0; j < JT; ++j) {
              if constexpr (!FP4)
                acc[i][j] = Op::run(fa[kk][i], fb[kk][j], acc[i][j]);
              else
                acc[i][j] = kk == 0 ? Op::template run<0>(mx_lo(fa[0][i]), mx_lo(fb[0][j]), acc[i][j], (int)sa[i][h], (int)sb[j][h])
                                    : Op::template run<2>(mx_lo(fa[1][i]), mx_lo(fb[1][j]), acc[i][j], (int)sa[i][h], (int)sb[j][h]);
            }
      }
    }
  }

  if constexpr (KG > 1) {
    // the other K groups' partial sums through the ring, added in K order
    static_assert((KG - 1) * TM * TN * 4 <= LDSB, "partial sums");
    acc_t *red = reinterpret_cast<acc_t *>(lds);
    __syncthreads();
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < IT; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) red[(((kg - 1) * NWG + wm * WN + wn) * IT * JT + i * JT + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int q = 0; q < KG - 1; ++q)
#pragma unroll
        for (int i = 0; i < IT; ++i)
#pragma unroll
          for (int j = 0; j < JT; ++j) acc[i][j] += red[((q * NWG + wm * WN + wn) * IT * JT + i * JT + j) * 64 + lane];
    }
  }
  // outputs through the (now free) ring into row-major 16-byte stores;
  // accumulator register r of a 32x32 tile is row 8 (r / 4) + 4 (lane / 32) +
  // r % 4, column lane % 32.  PASS rows at a time when the tile does not fit.
  constexpr int RS = TN * (int)sizeof(O) + 16, CPR = TN * (int)sizeof(O) / 16, EPC = 16 / (int)sizeof(O);
  constexpr int NP = TM * RS <= LDSB ? 1 : 2, RP = TM / NP; // passes, rows per pass
  static_assert(RP * RS <= LDSB && (NP == 1 || WM % 2 == 0), "epilogue stage");
#pragma unroll 1
  for (int h = 0; h < NP; ++h) {
    __syncthreads();
    if (kg == 0 && (NP == 1 || wm / (WM / NP) == h)) {
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        typename Epi::row_t rv[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t m = m0 + wm * (TM / WM) + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
          rv[r] = Epi::row(m < M ? m : M - 1, P);
        }
#pragma unroll
        for (int j = 0; j < JT; ++j) {
          const int col = wn * (TN / WN) + j * 32 + lane % 32;
          const int64_t n = n0 + col;
          const typename Epi::col_t cv = Epi::col(n < N ? n : N - 1, P);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = wm * (TM / WM) + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
            const int64_t m = m0 + row;
            // rows and columns past C are staged (from clamped operand indices) but never stored
            *reinterpret_cast<O *>(lds + (row - h * RP) * RS + col * (int)sizeof(O)) =
                Epi::apply(acc[i][j][r], m < M ? m : M - 1, n < N ? n : N - 1, rv[r], cv, P);
          }
        }
      }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < RP * CPR; c += NW * 64) {
      const int row = c / CPR, ch = c % CPR;
      const int64_t m = m0 + h * RP + row, n = n0 + (int64_t)ch * EPC;
      if (m >= M) continue;
      const v4i v = *reinterpret_cast<const v4i *>(lds + row * RS + ch * 16);
      if (n + EPC <= N && (N % EPC == 0)) {
        __builtin_nontemporal_store(v, reinterpret_cast<v4i *>(out + m * N + n));
      } else {
        const O *e = reinterpret_cast<const O *>(&v);
        for (int k = 0; k < EPC && n + k < N; ++k) out[m * N + n + k] = e[k];
      }
    }
  }
}

// Block-scaled entry, arguments as mmad_mx of hf_mmad.h.
template <int MK, typename Epi, int TM, int TN, int WM, int WN, int S, typename Args>
__device__ __forceinline__ void mmad_mx(const uint8_t *A, const uint8_t *B, const uint8_t *SA, const uint8_t *SB,
                                        typename Epi::out_t *out, int64_t M, int64_t N, int64_t K, const Args &P) {
  mmad_tile<MK, Epi, true, TM, TN, WM, WN, S>(A, B, out, M, N, K, P, SA, SB);
}

} // namespace hf
