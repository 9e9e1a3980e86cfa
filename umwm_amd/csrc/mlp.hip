// BF16 MFMA kernels of the surrogate network (mlp.hpp): the training GEMM
// with operand-layout and epilogue variants (the loss among them), the
// inference GEMM, and the Adam step that reduces the gradients' partials.
//
// MFMA operand layout (32x32x16): lane l supplies A(m = l%32, k = 8(l/32)
// + j) and B(k = 8(l/32) + j, n = l%32), j = 0..7; accumulator register i
// of lane l holds C(m = 8(i/4) + 4(l/32) + i%4, n = l%32).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <random>
#include <string>

#include "bufio.hpp"
#include "common.hpp"
#include "mlp.hpp"

namespace umwm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int BK = 32;  // K tile of the inference GEMM

// Training GEMM.  A step's products are small (2048 x 512 x 1344 and down to
// 2048 x 512 x 512): the time is the chain of K tiles, not the MFMA rate, so
// a workgroup takes only 64 x 64 of C (256 workgroups for 2048 x 512, one a
// compute unit, where 128 x 128 blocks left three quarters of them idle),
// steps K by 64 and keeps two tiles in registers ahead of the one in LDS.
// Wave (wm, wn) of its four owns 32 x 32 as one accumulator of the 32x32x16
// MFMA.
//
// An operand lies in LDS as it lies in memory, k-contiguous rows ([m][k], one
// 16-byte read per MFMA operand; 144-byte rows put 16 lanes on distinct
// banks) or m- or n-contiguous rows ([k][m]: the products over the batch and
// the weights in the backward pass), which ds_read_tr16_b64 transposes as it
// reads: a group of 16 lanes reads 4 k rows of 16 values, lane i the 8 bytes
// of row i / 4 at value 4 (i % 4), and receives value i of the 4 rows
// (192-byte rows put a half wave on distinct banks).  Turning the operand on
// its way into LDS took a 2-byte store per value.
//
// One training step of 2048 rows through 1335-512-512-512-1332 took 790 us
// (GEMMs 430 of them), now 179 us of kernels (138).
constexpr int TT = 64;             // block of C and K tile
constexpr int LMK = TT + 8, LKM = TT + 32;

template <int KMAJOR>
struct Tile64 {
  static constexpr int LD = KMAJOR ? LKM : LMK;
  // the 8 k values of this lane's row: r0 the wave's first row of C, ks the
  // 16-wide K step
  static __device__ __forceinline__ bf16x8 frag(const bf16* t, int r0, int ks, int lane) {
    if constexpr (KMAJOR) {
      typedef __attribute__((address_space(3))) bf16x4 lds4;
      const int g = lane >> 4, i = lane & 15;
      const bf16* q = t + (ks * 16 + 8 * (g >> 1) + (i >> 2)) * LD + r0 + 16 * (g & 1) + 4 * (i & 3);
      const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4*)q);
      const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4*)(q + 4 * LD));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
      return *(const bf16x8*)(t + (r0 + (lane & 31)) * LD + ks * 16 + (lane >> 5) * 8);
    }
  }
};

// The bias gradient beside the products over the batch: the sums over k of
// A(m, k), which lies as [k][m].  A workgroup takes 32 m: 8 groups of its
// threads add every 8th k each, one after the other, then the 8 sums are added
// in order.  A chain of K / 8 additions whose loads are what it waits for, so
// they go out 32 at a time.
constexpr int kSumCols = 32, kSumRows = 8;

// workgroups of the sums, a whole number on each XCD
__host__ __device__ inline int bias_blocks(int M) {
  return ((M + kSumCols - 1) / kSumCols + 7) / 8 * 8;
}

__device__ __forceinline__ void bias_sum(const GemmArgs& g, float* part) {
  const int c = (int)threadIdx.x % kSumCols, rg = (int)threadIdx.x / kSumCols;
  const int m = (int)blockIdx.x * kSumCols + c;
  float s = 0.f;
  if (m < g.M) {
    const bf16* a = g.A + m;
    int k = rg;
    for (; k + 31 * kSumRows < g.K; k += 32 * kSumRows) {
      bf16 v[32];
#pragma unroll
      for (int i = 0; i < 32; ++i) v[i] = a[(int64_t)(k + i * kSumRows) * g.lda];
#pragma unroll
      for (int i = 0; i < 32; ++i) s += (float)v[i];
    }
    for (; k < g.K; k += kSumRows) s += (float)a[(int64_t)k * g.lda];
  }
  part[rg * kSumCols + c] = s;
  __syncthreads();
  if (rg == 0 && m < g.M) {
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < kSumRows; ++q) t += part[q * kSumCols + c];
    g.asum[m] = t;
  }
}

template <int AL, int BL, int EP>
__global__ __launch_bounds__(256, 2) void k_gemm(GemmArgs g, int ntm, int ntn, int nz) {
  using TA = Tile64<AL == A_KM>;
  using TB = Tile64<BL == B_KN>;
  __shared__ __attribute__((aligned(16))) bf16 As[2][TT * TA::LD];
  __shared__ __attribute__((aligned(16))) bf16 Bs[2][TT * TB::LD];
  int b = (int)blockIdx.x, nb = (int)gridDim.x;
  if constexpr (EP == EP_PART) {
    // the first workgroups sum the bias gradient beside the products
    const int sums = bias_blocks(g.M);
    if (b < sums) {
      bias_sum(g, reinterpret_cast<float*>(As));
      return;
    }
    b -= sums;
    nb -= sums;
  }
  // blocks sharing rows of A and of the K range run on one XCD (workgroups go
  // round-robin over the 8), whose L2 then holds them
  const int per = nb / 8;
  const int t = b % 8 * per + b / 8;
  if (t >= ntm * ntn * nz) return;
  const int tz = t / (ntm * ntn), tm = t / ntn % ntm, tn = t % ntn;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int wm = w >> 1, wn = w & 1;
  const int m0 = tm * TT, n0 = tn * TT;
  const int kb = tz * g.kchunk, ke = min(g.K, kb + g.kchunk);
  // Chunks of 16 bytes, two of each operand a thread and K tile, through a
  // buffer resource at the tile's first byte: rows past M or N and k past the
  // range read from beyond it, which gives 0 (a masked load would make the
  // compiler wait for every load in flight).  A chunk never straddles the
  // end: K, and M or N on their contiguous axis, are multiples of 8 (checked
  // by gemm()).
  constexpr uint32_t kOut = 0x80000000u;  // beyond every resource
  uint32_t oa[2], ob[2];
  int ka[2], kbv[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int q = tid + c * 256, r = q >> 3, x = (q & 7) * 8;
    const bool ina = AL == A_MK ? m0 + r < g.M : m0 + x < g.M;
    const bool inb = BL == B_NK ? n0 + r < g.N : n0 + x < g.N;
    oa[c] = ina ? (uint32_t)(r * g.lda + x) * 2u : kOut;
    ob[c] = inb ? (uint32_t)(r * g.ldb + x) * 2u : kOut;
    ka[c] = AL == A_MK ? x : r;
    kbv[c] = BL == B_NK ? x : r;
  }
  struct Stage {
    bf16x8 a[2], b[2];
  };
  auto gload = [&](Stage& S, int k0) {
    const rsrc_t rA = make_rsrc(AL == A_MK ? g.A + (int64_t)m0 * g.lda + k0
                                           : g.A + (int64_t)k0 * g.lda + m0, kOut);
    const rsrc_t rB = make_rsrc(BL == B_NK ? g.B + (int64_t)n0 * g.ldb + k0
                                           : g.B + (int64_t)k0 * g.ldb + n0, kOut);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      S.a[c] = __builtin_bit_cast(bf16x8, bld16<float>(rA, k0 + ka[c] < ke ? oa[c] : kOut));
      S.b[c] = __builtin_bit_cast(bf16x8, bld16<float>(rB, k0 + kbv[c] < ke ? ob[c] : kOut));
    }
  };
  auto sstore = [&](const Stage& S, int buf) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int q = tid + c * 256, r = q >> 3, x = (q & 7) * 8;
      *(bf16x8*)&As[buf][r * TA::LD + x] = S.a[c];
      *(bf16x8*)&Bs[buf][r * TB::LD + x] = S.b[c];
    }
  };
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  auto mfma = [&](int buf) {
#pragma unroll
    for (int ks = 0; ks < TT / 16; ++ks)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TA::frag(As[buf], wm * 32, ks, lane),
                                                    TB::frag(Bs[buf], wn * 32, ks, lane), acc, 0, 0, 0);
  };
  // K tile u in LDS buffer u % 2; tiles past the range load zeros
  Stage st[2];
  gload(st[0], kb);
  gload(st[1], kb + TT);
  sstore(st[0], 0);
  gload(st[0], kb + 2 * TT);
  __syncthreads();
#pragma unroll 1
  for (int k0 = kb; k0 < ke; k0 += 2 * TT) {
    sstore(st[1], 1);
    gload(st[1], k0 + 3 * TT);
    mfma(0);
    __syncthreads();
    sstore(st[0], 0);
    gload(st[0], k0 + 4 * TT);
    mfma(1);  // all zero past an odd number of tiles
    __syncthreads();
  }
  // epilogue
  [[maybe_unused]] double loss = 0;
  const int n = n0 + wn * 32 + (lane & 31);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int m = m0 + wm * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
    if (m >= g.M || n >= g.N) continue;
    const float v = acc[i];
    const int64_t o = (int64_t)m * g.ldc + n;
    if constexpr (EP == EP_GELU) {
      const float z = v + g.bias[n];
      g.Zout[o] = (bf16)z;
      ((bf16*)g.C)[o] = (bf16)gelu_f(z);
    } else if constexpr (EP == EP_F32) {
      ((float*)g.C)[o] = v + g.bias[n];
    } else if constexpr (EP == EP_LOSS) {
      float gr = 0.f;
      if (n < g.nout) {
        const float d = v + g.bias[n] - g.target[o];
        gr = 2.f * d * g.inv;
        loss += (double)d * d * g.inv;
      }
      ((bf16*)g.C)[o] = (bf16)gr;
    } else if constexpr (EP == EP_DGELU) {
      ((bf16*)g.C)[o] = (bf16)(v * gelu_grad_f((float)g.Zin[(int64_t)m * g.ldz + n]));
    } else {
      static_assert(EP == EP_PART, "training epilogues");
      ((float*)g.C)[(int64_t)tz * g.M * g.ldc + o] = v;
    }
  }
  if constexpr (EP == EP_LOSS) {
    __shared__ double wsum[4];
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_down(loss, off, 64);
    if (lane == 0) wsum[w] = loss;
    __syncthreads();
    if (tid == 0) atomicAdd(g.loss, wsum[0] + wsum[1] + wsum[2] + wsum[3]);
  }
}

// Inference GEMM.  A workgroup of 4 waves (2 x 2) computes a BMT x BNT
// block of C, each wave a (BMT/2) x (BNT/2) part as TA x TB tiles of the
// 32x32x16 MFMA (8 tiles: each 16-byte LDS read feeds 8/6 of an MFMA, the
// training GEMM's 2 x 2 wave tiles feed one).  bf16 A operands use 256 x
// 128 blocks; the spectrum operand uses 128 x 256, so that its ln /
// normalise / bf16 transform, done once per column block, is repeated
// over 2 column blocks of the 512 hidden outputs rather than 4.  The K
// loop steps by 32 with two tiles staged in registers ahead.  Blocks are
// numbered so that the blocks sharing one A block (or, for the transposed
// last layer, one B block) land on the same XCD back to back (workgroups
// go round-robin over the 8 XCDs): the shared operand then comes from that
// XCD's L2 after the first read.
//
// A_SPEC stages the first layer's input from the spectrum (fp32, points
// contiguous): each thread loads BMT/64 points x 8 inputs as 8 vector
// reads (a wave reads BMT x 4 bytes contiguous per input row), forms
// ln e, normalises, rounds to bf16 and writes each point's 8 inputs as
// one 16-byte LDS row segment.
constexpr int ILDK = BK + 8;

template <int AM, int BMT>
struct InfStage;
template <int BMT>
struct InfStage<A_MK, BMT> {
  bf16x8 a[BMT / 64];
};
template <int BMT>
struct InfStage<A_SPEC, BMT> {
  using V = float __attribute__((ext_vector_type(BMT / 64)));
  V a[8];
};

template <int AM, int EP, int BMT, int BNT>
__global__ __launch_bounds__(256, 2) void k_gemm_inf(GemmArgs g, int ntm, int ntn, int nmajor) {
  constexpr int TA = BMT / 64, TB = BNT / 64;  // MFMA tiles per wave
  constexpr int CA = BMT / 64, CB = BNT / 64;  // 16-byte bf16 chunks per thread per K tile
  constexpr int PPT = BMT / 64;                // A_SPEC: points per thread
  static_assert(TA * TB == 8 && (BMT == 256 || BMT == 128), "block shapes 256x128, 128x256");
  // one LDS array: the A and B tiles of the K loop, then the epilogue's
  // staging rows
  __shared__ __attribute__((aligned(16))) bf16 lds[2 * (BMT + BNT) * ILDK];
  bf16(*const As)[BMT][ILDK] = reinterpret_cast<bf16(*)[BMT][ILDK]>(lds);
  bf16(*const Bs)[BNT][ILDK] = reinterpret_cast<bf16(*)[BNT][ILDK]>(lds + 2 * BMT * ILDK);
  // XCD-aware tile order (the grid is padded to a multiple of 8): row
  // blocks outer (the blocks of one A block adjacent) or, with nmajor,
  // column blocks outer (the blocks of one B block adjacent)
  const int nt = ntm * ntn, per = (int)(gridDim.x / 8);
  const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (t >= nt) return;
  const int tm = nmajor ? t % ntm : t / ntn, tn = nmajor ? t / ntm : t % ntn;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  const int m0 = tm * BMT, n0 = tn * BNT;
  const int K = g.K;
  struct Stage {
    InfStage<AM, BMT> a;
    bf16x8 b[CB];
  };
  Stage st[2];  // two K tiles in flight
  // A_SPEC: this thread's PPT points and (wave-uniform) 8-input group
  [[maybe_unused]] const int smc = (tid & 63) * PPT;
  [[maybe_unused]] const int skg = __builtin_amdgcn_readfirstlane(tid >> 6) * 8;
  // A_SPEC: the largest |normalised input| of each of its points
  [[maybe_unused]] float zabs[PPT] = {};
  // Every load stays inside its operand and none is conditional (a
  // masked load would make the compiler wait for every load in flight
  // before the next LDS store): K is a multiple of 64 (checked by
  // gemm_infer()), so the K tiles hold no partial 16-byte chunk; rows past
  // M or N read row M - 1 or N - 1 again, and their results are never
  // stored; a spectrum vector lies wholly inside its row or wholly past it
  // (lde, the chunk start and the points per thread all multiples of 4 or
  // of PPT) and reads 0 there.  Points past M feed only their own rows of
  // C.
  // bf16 operands through buffer resources: each thread's 16-byte chunks
  // keep a fixed 32-bit byte offset (row, column within the K tile), and the
  // K tile's position is the scalar offset (gemm_infer() checks that the
  // operands span less than 2 GiB)
  [[maybe_unused]] const rsrc_t rA =
      make_rsrc(AM == A_MK ? (const void*)g.A : (const void*)g.B,
                AM == A_MK ? (uint32_t)((int64_t)g.M * g.lda * 2) : 0u);
  const rsrc_t rB = make_rsrc(g.B, (uint32_t)((int64_t)g.N * g.ldb * 2));
  [[maybe_unused]] uint32_t offA[CA];
  uint32_t offB[CB];
#pragma unroll
  for (int c = 0; c < CA; ++c) {
    const int q = tid + c * 256;
    if constexpr (AM == A_MK)
      offA[c] = (uint32_t)(((int64_t)min(m0 + (q >> 2), g.M - 1) * g.lda + (q & 3) * 8) * 2);
  }
#pragma unroll
  for (int c = 0; c < CB; ++c) {
    const int q = tid + c * 256;
    offB[c] = (uint32_t)(((int64_t)min(n0 + (q >> 2), g.N - 1) * g.ldb + (q & 3) * 8) * 2);
  }
  auto gload = [&](Stage& S, int k0) {
    if constexpr (AM == A_MK) {
#pragma unroll
      for (int c = 0; c < CA; ++c)
        S.a.a[c] = __builtin_bit_cast(bf16x8, bld16<float>(rA, offA[c], (uint32_t)k0 * 2u));
    } else {
      // one buffer resource per input row (scalar registers: the row is
      // wave-uniform) covering this block's columns of the row; a vector
      // past the row's end (the last row of the spectrum only) reads 0,
      // and rows past the inputs (K padding) get an empty resource
      const SpecOperand& sa = g.sa;
      const int kb = k0 + skg;
      const uint32_t voff = (uint32_t)smc * 4u;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int k = kb + i;
        const bool spec = k < sa.nb, in = k < sa.nb + 3;
        const int kk = in ? k : sa.nb;
        const float* row = spec ? sa.e + (int64_t)k * sa.lde : sa.ext + (int64_t)(kk - sa.nb) * sa.ldx;
        const int cols = spec ? sa.cols : (int)sa.ldx;
        const rsrc_t r = make_rsrc(row + m0, in ? (uint32_t)std::min(cols - m0, BMT) * 4u : 0u);
        if constexpr (PPT == 4) {
          S.a.a[i] = bld16<float>(r, voff);
        } else {
          S.a.a[i] = __builtin_bit_cast(typename InfStage<AM, BMT>::V,
                                        __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, 0, 0));
        }
      }
    }
#pragma unroll
    for (int c = 0; c < CB; ++c)
      S.b[c] = __builtin_bit_cast(bf16x8, bld16<float>(rB, offB[c], (uint32_t)k0 * 2u));
  };
  auto sstore = [&](const Stage& S, int buf, int k0) {
    if constexpr (AM == A_MK) {
#pragma unroll
      for (int c = 0; c < CA; ++c) {
        const int q = tid + c * 256;
        *(bf16x8*)&As[buf][q >> 2][(q & 3) * 8] = S.a.a[c];
      }
    } else {
      const SpecOperand& sa = g.sa;
      const int kb = k0 + skg;
      bf16x8 o[PPT];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int k = kb + i;
        float x[PPT];
#pragma unroll
        for (int c = 0; c < PPT; ++c) x[c] = S.a.a[i][c];
        if (k < sa.nb) {
          // (ln e - mu) is = log2(e) (ln 2 is) - mu is: the hardware log2
          // and one fma per input (wave-uniform constants per k)
          const float is = sa.is[k], a = is * 0.6931471805599453f, c0 = -sa.mu[k] * is;
#pragma unroll
          for (int c = 0; c < PPT; ++c) {
            x[c] = fmaf(__builtin_amdgcn_logf(fmaxf(x[c], 1e-30f)), a, c0);
            zabs[c] = fmaxf(zabs[c], fabsf(x[c]));
          }
        }
#pragma unroll
        for (int c = 0; c < PPT; ++c) o[c][i] = (bf16)x[c];
      }
#pragma unroll
      for (int c = 0; c < PPT; ++c) *(bf16x8*)&As[buf][smc + c][skg] = o[c];
    }
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const int q = tid + c * 256;
      *(bf16x8*)&Bs[buf][q >> 2][(q & 3) * 8] = S.b[c];
    }
  };
  f32x16 acc[TA][TB];
#pragma unroll
  for (int a = 0; a < TA; ++a)
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
  auto mfma = [&](int buf) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int kk = ks * 16 + (lane >> 5) * 8;
      bf16x8 fa[TA], fb[TB];
#pragma unroll
      for (int a = 0; a < TA; ++a)
        fa[a] = *(const bf16x8*)&As[buf][wm * (BMT / 2) + a * 32 + (lane & 31)][kk];
#pragma unroll
      for (int b = 0; b < TB; ++b)
        fb[b] = *(const bf16x8*)&Bs[buf][wn * (BNT / 2) + b * 32 + (lane & 31)][kk];
#pragma unroll
      for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a], fb[b], acc[a][b], 0, 0, 0);
    }
  };
  // K tiles 0 .. nkt-1 of BK (nkt even: K a multiple of 64); tile u lives
  // in LDS buffer u % 2, odd tiles wait in st[0], even ones in st[1].  Each
  // step stores the next tile, refills its stage three tiles ahead and
  // multiplies the current one.  Loads and stores are unconditional (tile
  // indices past the end are clamped to the last tile, whose reload and
  // restore change nothing): a load under a branch leaves the compiler
  // unsure which stage's loads are the newest, and it then waits for all of
  // them before each LDS store.
  const int nkt = K / BK, last = nkt - 1;
  auto tile = [&](int u) { return min(u, last) * BK; };
  gload(st[0], 0);
  sstore(st[0], 0, 0);
  gload(st[0], tile(1));
  gload(st[1], tile(2));
  __syncthreads();
#pragma unroll 1
  for (int u = 0; u + 1 < nkt; u += 2) {
    sstore(st[0], 1, tile(u + 1));
    gload(st[0], tile(u + 3));
    mfma(0);
    __syncthreads();
    sstore(st[1], 0, tile(u + 2));
    gload(st[1], tile(u + 4));
    mfma(1);
    __syncthreads();
  }
  if constexpr (AM == A_SPEC) {
    // the first column of blocks reports each point's zmax verdict (inputs
    // are at least 1e-30 before the log, so no normalised input is NaN)
    if (tn == 0) {
#pragma unroll
      for (int c = 0; c < PPT; ++c)
        if (!(zabs[c] <= g.sa.zmax) && m0 + smc + c < g.M) atomicAnd(g.sa.ok + m0 + smc + c, 0);
    }
  }
  // Epilogue through LDS: each wave writes its part of C in 64 x 64 pieces
  // into its own LDS region (the MFMA layout puts one column per lane),
  // then reads rows back 16 bytes per lane, so that every store to C is a
  // whole 128-byte row segment.  Scattered 2-byte stores of the MFMA layout
  // ran at about 0.6 TB/s and made the output-heavy last layer store-bound.
  constexpr int SLD = 64 + 8;  // staging row, padded
  static_assert(4 * 64 * SLD <= 2 * (BMT + BNT) * ILDK, "staging fits in the LDS array");
  __syncthreads();  // every wave done with the K loop's tiles
  bf16(*stg)[SLD] = reinterpret_cast<bf16(*)[SLD]>(lds) + w * 64;
  bf16* const C = static_cast<bf16*>(g.C);
#pragma unroll
  for (int pr = 0; pr < TA / 2; ++pr)
#pragma unroll
    for (int pc = 0; pc < TB / 2; ++pc) {
#pragma unroll
      for (int aa = 0; aa < 2; ++aa)
#pragma unroll
        for (int bb = 0; bb < 2; ++bb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int r = aa * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3), c = bb * 32 + (lane & 31);
            // indices of the epilogue's vectors, clamped: rows past M and
            // columns past N are staged but never stored
            const int m = min(m0 + wm * (BMT / 2) + pr * 64 + r, g.M - 1);
            const int n = min(n0 + wn * (BNT / 2) + pc * 64 + c, g.N - 1);
            const float v = acc[2 * pr + aa][2 * pc + bb][i];
            float y;
            if constexpr (EP == EP_GELU) {
              y = gelu_fast_f(v + g.bias[n]);
            } else if constexpr (EP == EP_BF16_BM) {
              y = v + g.bias[m];
            } else {
              static_assert(EP == EP_SUR, "inference epilogues: GELU, BF16_BM, SUR");
              // exp(x) - 1 with the hardware exp2: its cancellation near
              // x = 0 costs relative precision only where dm^2 - 1 is below
              // 1e-4, which moves dm^2 by less than bf16 resolves
              const float x = fminf(g.osd[m] * (v + g.bias[m]) + g.omu[m], 30.f);
              y = __builtin_amdgcn_exp2f(1.4426950408889634f * x) - 1.f;
            }
            stg[r][c] = (bf16)y;
          }
      // LDS accesses of one wave complete in order: the rows read below are
      // the ones written above, by any lane of the wave
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const int q = it * 64 + lane, r = q >> 3, cc = (q & 7) * 8;
        const int m = m0 + wm * (BMT / 2) + pr * 64 + r, n = n0 + wn * (BNT / 2) + pc * 64 + cc;
        const bf16x8 v = *(const bf16x8*)&stg[r][cc];
        if (m < g.M) {
          bf16* dst = C + (int64_t)m * g.ldc + n;
          if (n + 8 <= g.N) {
            *(bf16x8*)dst = v;
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (n + e < g.N) dst[e] = v[e];
          }
        }
      }
    }
}

// A layer's weight gradient from the partials of the products over the batch,
// added in order (the result does not depend on scheduling), and its bias
// gradient: the first n elements are the weights, the next nbias the biases.
struct LayerParts {
  const float *pw, *pb;  // [splits][n], [nbias]
  int splits;
  int64_t n;
  int nbias;
};
__device__ __forceinline__ float part_sum(const LayerParts& a, int64_t i) {
  if (i >= a.n) return a.pb[i - a.n];
  float s = 0.f;
  for (int k = 0; k < a.splits; ++k) s += a.pw[k * a.n + i];
  return s;
}

__global__ void k_reduce_parts(LayerParts a, float* __restrict__ gw, float* __restrict__ gb) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n + a.nbias) return;
  const float s = part_sum(a, i);
  if (i < a.n) gw[i] = s; else gb[i - a.n] = s;
}

// The Adam step of one layer straight from the partials, with the bf16 copy
// of the new weights.  Bound by its 4 + splits reads and 3.5 writes a weight;
// as a reduction, two Adam launches and a conversion the gradient and the
// weights went through memory three times.
__global__ void k_adam(LayerParts a, MlpLayerDev L, AdamStep h) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n + a.nbias) return;
  const float gi = part_sum(a, i);
  const bool wt = i < a.n;
  const int64_t q = wt ? i : i - a.n;
  float* const p = wt ? L.w : L.b;
  float* const m = wt ? L.mw : L.mb;
  float* const v = wt ? L.vw : L.vb;
  const float mi = h.b1 * m[q] + (1.f - h.b1) * gi;
  const float vi = h.b2 * v[q] + (1.f - h.b2) * gi * gi;
  m[q] = mi;
  v[q] = vi;
  const float x = p[q] - h.lr * (mi * h.c1) / (sqrtf(vi * h.c2) + h.eps);
  p[q] = x;
  if (wt) L.wb[q] = (bf16)x;
}

__global__ void k_to_bf16(const float* __restrict__ a, bf16* __restrict__ b, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (bf16)a[i];
}

inline dim3 grid_for(int64_t n, int t = 256) { return dim3((unsigned)((n + t - 1) / t)); }

// K range of one split, in whole steps of 32 (K tiles end where it ends)
inline int gemm_chunk(int K, int splits) {
  const int k = (K + std::max(1, splits) - 1) / std::max(1, splits);
  return (k + 31) / 32 * 32;
}

}  // namespace

int gemm(int alay, int blay, int ep, const GemmArgs& g0, int splits, hipStream_t s) {
  GemmArgs g = g0;
  if (g.M <= 0 || g.N <= 0 || g.K <= 0) return 0;
  // 16-byte chunks: K and the contiguous axis of transposed operands must
  // be multiples of 8, and so must the leading dimensions
  if (g.K % 8 || g.lda % 8 || g.ldb % 8 || (alay == A_KM && g.M % 8) || (blay == B_KN && g.N % 8))
    return fail(UMWM_ERR_ARGUMENT, "gemm: K, lda, ldb (and M or N when transposed) must be "
                                   "multiples of 8");
  if (g.lda > (1 << 23) || g.ldb > (1 << 23))
    return fail(UMWM_ERR_SIZE, "gemm: an operand's rows are longer than 8 M values");
  if (ep != EP_PART) splits = 1;
  g.kchunk = gemm_chunk(g.K, splits);
  const int nz = (g.K + g.kchunk - 1) / g.kchunk;
  const int ntm = (g.M + TT - 1) / TT, ntn = (g.N + TT - 1) / TT;
  const int64_t nt = (int64_t)ntm * ntn * nz;
  if (nt > (1ll << 30)) return fail(UMWM_ERR_SIZE, "gemm: too many tiles");
  const dim3 grid((unsigned)((nt + 7) / 8 * 8 + (ep == EP_PART ? bias_blocks(g.M) : 0)));
#define UMWM_GEMM(AL_, BL_, EP_)                                                            \
  if (alay == AL_ && blay == BL_ && ep == EP_) {                                            \
    hipLaunchKernelGGL((k_gemm<AL_, BL_, EP_>), grid, dim3(256), 0, s, g, ntm, ntn, nz);    \
  } else
  UMWM_GEMM(A_MK, B_NK, EP_GELU)
  UMWM_GEMM(A_MK, B_NK, EP_F32)
  UMWM_GEMM(A_MK, B_NK, EP_LOSS)
  UMWM_GEMM(A_MK, B_KN, EP_DGELU)
  UMWM_GEMM(A_KM, B_KN, EP_PART)
  return fail(UMWM_ERR_ARGUMENT, "gemm: unsupported operands and epilogue");
#undef UMWM_GEMM
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UMWM_ERR_HIP, std::string("gemm: ") + hipGetErrorString(e));
  return 0;
}

int gemm_infer(int amode, int ep, const GemmArgs& g, hipStream_t s) {
  if (g.M <= 0 || g.N <= 0 || g.K <= 0) return 0;
  if (g.K % (2 * BK) || g.ldb % 8 || g.ldc % 8 || (amode == A_MK && g.lda % 8) ||
      reinterpret_cast<uintptr_t>(g.C) % 16)
    return fail(UMWM_ERR_ARGUMENT, "gemm_infer: K a multiple of 64, lda, ldb and ldc of 8, C "
                                   "16-byte aligned");
  if ((int64_t)g.N * g.ldb * 2 >= (1ll << 31) || (amode == A_MK && (int64_t)g.M * g.lda * 2 >= (1ll << 31)))
    return fail(UMWM_ERR_SIZE, "gemm_infer: an operand spans 2 GiB or more; use smaller chunks");
  if (amode == A_SPEC) {
    const SpecOperand& a = g.sa;
    if (!a.e || !a.mu || !a.is || !a.ext || !a.ok || a.nb < 1 || a.nb + 3 > g.K ||
        a.lde % 4 || a.ldx % 4 || a.cols < g.M || a.cols % 4 || a.ldx < g.M ||
        reinterpret_cast<uintptr_t>(a.e) % 16 || reinterpret_cast<uintptr_t>(a.ext) % 16)
      return fail(UMWM_ERR_ARGUMENT, "gemm_infer: bad spectrum operand");
  }
  // the spectrum operand takes 128 x 256 blocks, bf16 operands 256 x 128
  const int bm = amode == A_SPEC ? 128 : 256, bn = amode == A_SPEC ? 256 : 128;
  const int ntm = (g.M + bm - 1) / bm, ntn = (g.N + bn - 1) / bn;
  const int64_t nt = (int64_t)ntm * ntn;
  if (nt > (1ll << 30)) return fail(UMWM_ERR_SIZE, "gemm_infer: too many tiles");
  const dim3 grid((unsigned)((nt + 7) / 8 * 8));
  // the transposed last layer (EP_SUR, EP_BF16_BM) has few row blocks (the
  // outputs) and many column blocks (the points): column blocks outer, so
  // that the row blocks of one activation block share it in L2
  const int nmajor = ep == EP_GELU ? 0 : 1;
#define UMWM_INF(AM_, EP_, BM_, BN_) \
  hipLaunchKernelGGL((k_gemm_inf<AM_, EP_, BM_, BN_>), grid, dim3(256), 0, s, g, ntm, ntn, nmajor)
  if (amode == A_MK && ep == EP_GELU) UMWM_INF(A_MK, EP_GELU, 256, 128);
  else if (amode == A_SPEC && ep == EP_GELU) UMWM_INF(A_SPEC, EP_GELU, 128, 256);
  else if (amode == A_MK && ep == EP_SUR) UMWM_INF(A_MK, EP_SUR, 256, 128);
  else if (amode == A_MK && ep == EP_BF16_BM) UMWM_INF(A_MK, EP_BF16_BM, 256, 128);
  else return fail(UMWM_ERR_ARGUMENT, "gemm_infer: unsupported operand/epilogue pair");
#undef UMWM_INF
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UMWM_ERR_HIP, std::string("gemm_infer: ") + hipGetErrorString(e));
  return 0;
}

Mlp::~Mlp() {
  for (void* p : allocs) (void)hipFree(p);
}

namespace {
template <typename U>
U* dalloc(Mlp& m, size_t n) {
  void* p = nullptr;
  if (hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(U)) != hipSuccess) return nullptr;
  m.allocs.push_back(p);
  return static_cast<U*>(p);
}
inline int pad8(int v) { return (v + 7) / 8 * 8; }
inline int pad64(int v) { return (v + 63) / 64 * 64; }
}  // namespace

int mlp_create(const std::vector<int>& dims, uint64_t seed, int rows, Mlp& m) {
  const int nl = (int)dims.size() - 1;
  if (nl < 1 || rows < 1) return fail(UMWM_ERR_ARGUMENT, "mlp: need >= 1 layer and >= 1 row");
  m.nin = dims.front();
  m.nout = dims.back();
  m.cap_rows = rows;
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  size_t part = 0;
  for (int l = 0; l < nl; ++l) {
    MlpLayerDev L{};
    // inputs padded to an even number of 32-wide K tiles of the inference
    // GEMM (a hidden layer's outputs are the next layer's inputs), the
    // network's outputs to 8
    L.K = pad64(dims[l]);
    L.N = l + 1 < nl ? pad64(dims[l + 1]) : pad8(dims[l + 1]);
    const size_t nw = (size_t)L.N * L.K;
    L.w = dalloc<float>(m, nw); L.b = dalloc<float>(m, L.N); L.wb = dalloc<bf16>(m, nw);
    L.gw = dalloc<float>(m, nw); L.gb = dalloc<float>(m, L.N);
    L.mw = dalloc<float>(m, nw); L.vw = dalloc<float>(m, nw);
    L.mb = dalloc<float>(m, L.N); L.vb = dalloc<float>(m, L.N);
    if (!L.vb) return fail(UMWM_ERR_NOMEM, "mlp: device allocation failed");
    // He-uniform for the GELU layers, Glorot-uniform for the linear output;
    // padding rows and columns zero
    const double fan_in = dims[l], fan_out = dims[l + 1];
    const double a = l + 1 < nl ? std::sqrt(6.0 / fan_in) : std::sqrt(6.0 / (fan_in + fan_out));
    std::vector<float> hw(nw, 0.f), zero(nw, 0.f), zb(L.N, 0.f);
    for (int n = 0; n < dims[l + 1]; ++n)
      for (int k = 0; k < dims[l]; ++k) hw[(size_t)n * L.K + k] = (float)(a * U(rng));
    UMWM_HIP_TRY(hipMemcpy(L.w, hw.data(), nw * 4, hipMemcpyHostToDevice));
    for (float* p : {L.gw, L.mw, L.vw}) UMWM_HIP_TRY(hipMemcpy(p, zero.data(), nw * 4, hipMemcpyHostToDevice));
    for (float* p : {L.b, L.gb, L.mb, L.vb}) UMWM_HIP_TRY(hipMemcpy(p, zb.data(), L.N * 4, hipMemcpyHostToDevice));
    m.L.push_back(L);
    part = std::max(part, nw);
  }
  // activation buffers
  m.x = dalloc<bf16>(m, (size_t)rows * m.L[0].K);
  int wmax = m.L[0].K;
  for (int l = 0; l + 1 < nl; ++l) {
    m.z.push_back(dalloc<bf16>(m, (size_t)rows * m.L[l].N));
    m.h.push_back(dalloc<bf16>(m, (size_t)rows * m.L[l].N));
    wmax = std::max(wmax, m.L[l].N);
  }
  wmax = std::max(wmax, m.L.back().N);
  m.y = dalloc<float>(m, (size_t)rows * m.L.back().N);
  m.dy = dalloc<bf16>(m, (size_t)rows * m.L.back().N);
  m.da = dalloc<bf16>(m, (size_t)rows * wmax);
  m.db = dalloc<bf16>(m, (size_t)rows * wmax);
  // split-K partials: at most 32 splits of the largest weight matrix; and the
  // longest bias gradient
  m.part_elems = part * 32;
  m.part = dalloc<float>(m, m.part_elems);
  m.partb = dalloc<float>(m, (size_t)wmax);
  m.loss_acc = dalloc<double>(m, 1);
  if (!m.loss_acc || !m.part || !m.partb || !m.db) return fail(UMWM_ERR_NOMEM, "mlp: device allocation failed");
  if (int rc = mlp_sync_bf16(m, nullptr)) return rc;
  UMWM_HIP_TRY(hipDeviceSynchronize());
  return 0;
}

int mlp_sync_bf16(Mlp& m, hipStream_t s) {
  for (auto& L : m.L) {
    const int64_t nw = (int64_t)L.N * L.K;
    hipLaunchKernelGGL(k_to_bf16, grid_for(nw), dim3(256), 0, s, (const float*)L.w, L.wb, nw);
  }
  UMWM_HIP_TRY(hipGetLastError());
  return 0;
}

int mlp_forward(Mlp& m, int rows, hipStream_t s, const float* t, double* loss) {
  if (rows > m.cap_rows) return fail(UMWM_ERR_SIZE, "mlp: more rows than the buffers hold");
  const int nl = (int)m.L.size();
  const bf16* in = m.x;
  for (int l = 0; l < nl; ++l) {
    const MlpLayerDev& L = m.L[l];
    GemmArgs g{};
    g.A = in; g.lda = L.K;
    g.B = L.wb; g.ldb = L.K;
    g.M = rows; g.N = L.N; g.K = L.K;
    g.bias = L.b;
    g.ldc = L.N;
    int ep = EP_GELU;
    if (l + 1 < nl) {
      g.C = m.h[l]; g.Zout = m.z[l];
      in = m.h[l];
    } else if (t) {
      ep = EP_LOSS;
      g.C = m.dy; g.target = t; g.loss = loss; g.nout = m.nout;
      g.inv = 1.f / ((float)rows * (float)m.nout);
    } else {
      ep = EP_F32;
      g.C = m.y;
    }
    if (int rc = gemm(A_MK, B_NK, ep, g, 1, s)) return rc;
  }
  return 0;
}

int mlp_backward(Mlp& m, int rows, hipStream_t s, const AdamStep* adam) {
  if (rows % 8) return fail(UMWM_ERR_ARGUMENT, "mlp: training rows must be a multiple of 8");
  const int nl = (int)m.L.size();
  const bf16* dz = m.dy;
  bf16* bufs[2] = {m.da, m.db};
  int pb = 0;
  for (int l = nl - 1; l >= 0; --l) {
    const MlpLayerDev& L = m.L[l];
    const bf16* a = l == 0 ? m.x : m.h[l - 1];
    const int64_t nw = (int64_t)L.N * L.K;
    // weight gradient over the batch, split over rows so that the small
    // output (N x K) still fills the GPU.  The splits set the order of the
    // sums and with it the last bits of the gradients, which Adam's normalised
    // step turns into differences of 6e-4 in the weights after sixteen steps:
    // the rule counts blocks of 128 x 128 whatever the GEMM's own are.
    const int tiles = ((L.N + 127) / 128) * ((L.K + 127) / 128);
    int splits = std::max(1, std::min(rows / 256, (1024 + tiles - 1) / tiles));
    splits = std::min<int>(std::min(splits, 32), (int)(m.part_elems / nw));
    GemmArgs g{};
    g.A = dz; g.lda = L.N;       // A(m = out, k = row) = dz[row][out]
    g.B = a; g.ldb = L.K;        // B(k = row, n = in) = a[row][in]
    g.M = L.N; g.N = L.K; g.K = rows;
    g.C = m.part; g.ldc = L.K;
    g.asum = m.partb;
    if (int rc = gemm(A_KM, B_KN, EP_PART, g, splits, s)) return rc;
    if (l > 0) {
      // d a_{l-1} = dz W_l, times gelu'(z_{l-1})
      GemmArgs d{};
      d.A = dz; d.lda = L.N;      // A(m = row, k = out)
      d.B = L.wb; d.ldb = L.K;    // B(k = out, n = in) = W[out][in]
      d.M = rows; d.N = L.K; d.K = L.N;
      d.C = bufs[pb]; d.ldc = L.K;
      d.Zin = m.z[l - 1]; d.ldz = L.K;
      if (int rc = gemm(A_MK, B_KN, EP_DGELU, d, 1, s)) return rc;
      dz = bufs[pb];
      pb ^= 1;
    }
    // after the product that reads the weights
    const int chunk = gemm_chunk(rows, splits);
    const LayerParts p{m.part, m.partb, (rows + chunk - 1) / chunk, nw, L.N};
    if (adam)
      hipLaunchKernelGGL(k_adam, grid_for(nw + L.N), dim3(256), 0, s, p, L, *adam);
    else
      hipLaunchKernelGGL(k_reduce_parts, grid_for(nw + L.N), dim3(256), 0, s, p, L.gw, L.gb);
    UMWM_HIP_TRY(hipGetLastError());
  }
  return 0;
}

int mlp_train_step(Mlp& m, const float* t, int rows, float lr, double* loss, hipStream_t s) {
  m.step += 1;
  AdamStep h{lr, 0.9f, 0.999f, 1e-8f, 0.f, 0.f};
  h.c1 = 1.f / (1.f - std::pow(h.b1, (float)m.step));
  h.c2 = 1.f / (1.f - std::pow(h.b2, (float)m.step));
  if (int rc = mlp_forward(m, rows, s, t, loss)) return rc;
  return mlp_backward(m, rows, s, &h);
}

namespace {
// Hidden layers 1.. and the transposed last layer of an inference pass
// whose first hidden layer already ran into m.h[0].
int infer_rest(Mlp& m, int rows, bf16* out, int64_t ldo, hipStream_t s, const float* omu,
               const float* osd) {
  const int nl = (int)m.L.size();
  const bf16* in = m.h[0];
  for (int l = 1; l + 1 < nl; ++l) {
    const MlpLayerDev& L = m.L[l];
    GemmArgs g{};
    g.A = in; g.lda = L.K;
    g.B = L.wb; g.ldb = L.K;
    g.M = rows; g.N = L.N; g.K = L.K;
    g.bias = L.b;
    g.C = m.h[l]; g.ldc = L.N;
    if (int rc = gemm_infer(A_MK, EP_GELU, g, s)) return rc;
    in = m.h[l];
  }
  // out[o][j] = sum_k W[o][k] h[j][k] + b[o]: the network's outputs of point
  // j along a contiguous row per output (the spectra's [bin][point] layout)
  const MlpLayerDev& L = m.L.back();
  GemmArgs g{};
  g.A = L.wb; g.lda = L.K;
  g.B = in; g.ldb = L.K;
  g.M = m.nout; g.N = rows; g.K = L.K;
  g.bias = L.b;
  g.C = out; g.ldc = ldo;
  if (omu && osd) {
    g.omu = omu; g.osd = osd;
    return gemm_infer(A_MK, EP_SUR, g, s);
  }
  return gemm_infer(A_MK, EP_BF16_BM, g, s);
}
}  // namespace

int mlp_infer_transposed(Mlp& m, int rows, bf16* out, int64_t ldo, hipStream_t s,
                         const float* omu, const float* osd) {
  if (rows > m.cap_rows) return fail(UMWM_ERR_SIZE, "mlp: more rows than the buffers hold");
  if (m.L.size() < 2) return fail(UMWM_ERR_ARGUMENT, "mlp: inference needs a hidden layer");
  const MlpLayerDev& L = m.L[0];
  GemmArgs g{};
  g.A = m.x; g.lda = L.K;
  g.B = L.wb; g.ldb = L.K;
  g.M = rows; g.N = L.N; g.K = L.K;
  g.bias = L.b;
  g.C = m.h[0]; g.ldc = L.N;
  if (int rc = gemm_infer(A_MK, EP_GELU, g, s)) return rc;
  return infer_rest(m, rows, out, ldo, s, omu, osd);
}

int mlp_infer_spectrum(Mlp& m, const SpecOperand& in, int rows, bf16* out, int64_t ldo,
                       hipStream_t s, const float* omu, const float* osd) {
  if (rows > m.cap_rows) return fail(UMWM_ERR_SIZE, "mlp: more rows than the buffers hold");
  if (m.L.size() < 2) return fail(UMWM_ERR_ARGUMENT, "mlp: inference needs a hidden layer");
  const MlpLayerDev& L = m.L[0];
  if (in.nb + 3 != m.nin) return fail(UMWM_ERR_ARGUMENT, "mlp: spectrum operand width");
  GemmArgs g{};
  g.sa = in;
  g.B = L.wb; g.ldb = L.K;
  g.M = rows; g.N = L.N; g.K = L.K;
  g.bias = L.b;
  g.C = m.h[0]; g.ldc = L.N;
  if (int rc = gemm_infer(A_SPEC, EP_GELU, g, s)) return rc;
  return infer_rest(m, rows, out, ldo, s, omu, osd);
}

}  // namespace umwm
