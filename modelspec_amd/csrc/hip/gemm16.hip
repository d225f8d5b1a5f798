// The mixed-precision GEMMs on the f16 MFMA of gfx950 (v_mfma_f32_16x16x32_f16, f32 accumulation),
// reading the operands' f16 copies straight from HBM into LDS.
#include "gemm_common.h"
#include "lds_util.h"

#include <algorithm>

namespace msx::hk {

// ---------------------------------------------------------------------------------------------
// Operand K tiles of BK halves move from global memory into an NS-stage LDS ring (global_load_lds):
//   - an operand contiguous along K (KC) is staged [row][BK], the 16-byte chunk ch of row r at slot
//     ch ^ swz(r); an MFMA fragment (row c, K 8 q .. 8 q + 7 of lane c + 16 q) is one ds_read_b128;
//   - an operand contiguous along its rows is staged [K][row], as it lies in memory, the chunk ch of
//     K row k at slot ch ^ ksw(k); a fragment is two ds_read_b64_tr_b16: in each 16-lane group source
//     lane l reads 4 rows at K row k0 + l / 4, and after the transpose lane c holds row base + c at K
//     k0 .. k0 + 3.
// Both XORs are laid out for the lane groups the LDS serves together: a ds_read_b128 takes lanes 0-3,
// 12-15, 20-27 in one pass and 4-11, 16-19, 28-31 in the next (and so for lanes 32-63), a transposed
// read lanes 0-31 and 32-63. With the slots spread over 16 consecutive lanes instead, half of the LDS
// cycles were bank conflicts (SQ_LDS_BANK_CONFLICT / SQ_LDS_IDX_ACTIVE over BERT-base's step 0.50, now
// 0.03 to 0.06, the output's way through LDS included).
// BK 64 loads whole 128-byte lines of a KC operand: the loads alone of 16384 x 768 x 3072 take 56 us
// against 71 with 64-byte rows (BK 32).
//
// The MFMA takes B's fragment first (C^T tiles): a lane holds output row 16 i + c, columns 16 j + 4 q
// .. + 3. Rows and columns past the edges repeat the last (never stored); the K past the end of the
// last tile is zeroed in both operands' fragments, so K needs no alignment or padding.
//
// The fragments' LDS reads are inline assembly, the wait for them in the same block: the compiler
// would wait for the global->LDS loads in flight before a transposed read.
namespace {
#define MSX_RK(O, P, S, U) "ds_read_b128 %" #O ", %[" #P "] offset:" #U "*%[" #S "]\n"
#define MSX_RT(L, H, P, S) "ds_read_b64_tr_b16 %" #L ", %[" #P "]\nds_read_b64_tr_b16 %" #H ", %[" #P "] offset:%[" #S "]\n"
#define MSX_RWAIT "s_waitcnt lgkmcnt(0)"
[[maybe_unused]] __device__ __forceinline__ v8h join8(v4s16 lo, v4s16 hi) {
  const v4h16 a = __builtin_bit_cast(v4h16, lo), b = __builtin_bit_cast(v4h16, hi);
  return v8h{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// I + J fragments. A KC operand: one address, 16-row blocks S bytes apart; else one address
// a fragment, its second read S bytes further (four K rows).
template <int I, int J, bool AKC, bool BKC, int SA, int SB, int NA, int NB>
__device__ __forceinline__ void read_frags(const uint32_t (&pa)[NA], const uint32_t (&pb)[NB], v8h (&fa)[I], v8h (&fb)[J]) {
#if defined(__HIP_DEVICE_COMPILE__)
  // The tiles and layouts written out below: any other would compile to no read at all.
  static_assert((I == 8 && J == 3 && (AKC || !BKC)) || (I == 4 && J == 4) || (I == 2 && (J == 2 || J == 1)),
                "no fragment reads for this tile and layout");
  [[maybe_unused]] v4s16 la[I], ha[I], lb[J], hb[J];
  if constexpr (I == 8 && J == 3 && AKC && BKC)
    asm volatile(
        MSX_RK(0, pa, sa, 0) MSX_RK(1, pa, sa, 1) MSX_RK(2, pa, sa, 2) MSX_RK(3, pa, sa, 3) MSX_RK(4, pa, sa, 4)
        MSX_RK(5, pa, sa, 5) MSX_RK(6, pa, sa, 6) MSX_RK(7, pa, sa, 7) MSX_RK(8, pb, sb, 0) MSX_RK(9, pb, sb, 1)
        MSX_RK(10, pb, sb, 2) MSX_RWAIT
        :
        "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fa[2]), "=&v"(fa[3]), "=&v"(fa[4]), "=&v"(fa[5]), "=&v"(fa[6]),
        "=&v"(fa[7]), "=&v"(fb[0]), "=&v"(fb[1]), "=&v"(fb[2])
        :
        [pa] "v"(pa[0]), [pb] "v"(pb[0]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 8 && J == 3 && AKC && !BKC)
    asm volatile(
        MSX_RK(0, pa, sa, 0) MSX_RK(1, pa, sa, 1) MSX_RK(2, pa, sa, 2) MSX_RK(3, pa, sa, 3) MSX_RK(4, pa, sa, 4)
        MSX_RK(5, pa, sa, 5) MSX_RK(6, pa, sa, 6) MSX_RK(7, pa, sa, 7) MSX_RT(8, 9, pb0, sb) MSX_RT(10, 11, pb1, sb)
        MSX_RT(12, 13, pb2, sb) MSX_RWAIT
        :
        "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fa[2]), "=&v"(fa[3]), "=&v"(fa[4]), "=&v"(fa[5]), "=&v"(fa[6]),
        "=&v"(fa[7]), "=&v"(lb[0]), "=&v"(hb[0]), "=&v"(lb[1]), "=&v"(hb[1]), "=&v"(lb[2]), "=&v"(hb[2])
        :
        [pa] "v"(pa[0]), [pb0] "v"(pb[0]), [pb1] "v"(pb[1]), [pb2] "v"(pb[2]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 8 && J == 3 && !AKC && !BKC)
    asm volatile(
        MSX_RT(0, 1, pa0, sa) MSX_RT(2, 3, pa1, sa) MSX_RT(4, 5, pa2, sa) MSX_RT(6, 7, pa3, sa) MSX_RT(8, 9, pa4, sa)
        MSX_RT(10, 11, pa5, sa) MSX_RT(12, 13, pa6, sa) MSX_RT(14, 15, pa7, sa) MSX_RT(16, 17, pb0, sb)
        MSX_RT(18, 19, pb1, sb) MSX_RT(20, 21, pb2, sb) MSX_RWAIT
        :
        "=&v"(la[0]), "=&v"(ha[0]), "=&v"(la[1]), "=&v"(ha[1]), "=&v"(la[2]), "=&v"(ha[2]), "=&v"(la[3]),
        "=&v"(ha[3]), "=&v"(la[4]), "=&v"(ha[4]), "=&v"(la[5]), "=&v"(ha[5]), "=&v"(la[6]), "=&v"(ha[6]),
        "=&v"(la[7]), "=&v"(ha[7]), "=&v"(lb[0]), "=&v"(hb[0]), "=&v"(lb[1]), "=&v"(hb[1]), "=&v"(lb[2]), "=&v"(hb[2])
        :
        [pa0] "v"(pa[0]), [pa1] "v"(pa[1]), [pa2] "v"(pa[2]), [pa3] "v"(pa[3]), [pa4] "v"(pa[4]), [pa5] "v"(pa[5]),
        [pa6] "v"(pa[6]), [pa7] "v"(pa[7]), [pb0] "v"(pb[0]), [pb1] "v"(pb[1]), [pb2] "v"(pb[2]), [sa] "i"(SA),
        [sb] "i"(SB)
        : "memory");
  if constexpr (I == 4 && J == 4 && AKC && BKC)
    asm volatile(
        MSX_RK(0, pa, sa, 0) MSX_RK(1, pa, sa, 1) MSX_RK(2, pa, sa, 2) MSX_RK(3, pa, sa, 3) MSX_RK(4, pb, sb, 0)
        MSX_RK(5, pb, sb, 1) MSX_RK(6, pb, sb, 2) MSX_RK(7, pb, sb, 3) MSX_RWAIT
        :
        "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fa[2]), "=&v"(fa[3]), "=&v"(fb[0]), "=&v"(fb[1]), "=&v"(fb[2]), "=&v"(fb[3])
        :
        [pa] "v"(pa[0]), [pb] "v"(pb[0]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 4 && J == 4 && AKC && !BKC)
    asm volatile(
        MSX_RK(0, pa, sa, 0) MSX_RK(1, pa, sa, 1) MSX_RK(2, pa, sa, 2) MSX_RK(3, pa, sa, 3) MSX_RT(4, 5, pb0, sb)
        MSX_RT(6, 7, pb1, sb) MSX_RT(8, 9, pb2, sb) MSX_RT(10, 11, pb3, sb) MSX_RWAIT
        :
        "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fa[2]), "=&v"(fa[3]), "=&v"(lb[0]), "=&v"(hb[0]), "=&v"(lb[1]),
        "=&v"(hb[1]), "=&v"(lb[2]), "=&v"(hb[2]), "=&v"(lb[3]), "=&v"(hb[3])
        :
        [pa] "v"(pa[0]), [pb0] "v"(pb[0]), [pb1] "v"(pb[1]), [pb2] "v"(pb[2]), [pb3] "v"(pb[3]), [sa] "i"(SA),
        [sb] "i"(SB)
        : "memory");
  if constexpr (I == 4 && J == 4 && !AKC && BKC)
    asm volatile(
        MSX_RT(0, 1, pa0, sa) MSX_RT(2, 3, pa1, sa) MSX_RT(4, 5, pa2, sa) MSX_RT(6, 7, pa3, sa) MSX_RK(8, pb, sb, 0)
        MSX_RK(9, pb, sb, 1) MSX_RK(10, pb, sb, 2) MSX_RK(11, pb, sb, 3) MSX_RWAIT
        :
        "=&v"(la[0]), "=&v"(ha[0]), "=&v"(la[1]), "=&v"(ha[1]), "=&v"(la[2]), "=&v"(ha[2]), "=&v"(la[3]),
        "=&v"(ha[3]), "=&v"(fb[0]), "=&v"(fb[1]), "=&v"(fb[2]), "=&v"(fb[3])
        :
        [pa0] "v"(pa[0]), [pa1] "v"(pa[1]), [pa2] "v"(pa[2]), [pa3] "v"(pa[3]), [pb] "v"(pb[0]), [sa] "i"(SA),
        [sb] "i"(SB)
        : "memory");
  if constexpr (I == 4 && J == 4 && !AKC && !BKC)
    asm volatile(
        MSX_RT(0, 1, pa0, sa) MSX_RT(2, 3, pa1, sa) MSX_RT(4, 5, pa2, sa) MSX_RT(6, 7, pa3, sa) MSX_RT(8, 9, pb0, sb)
        MSX_RT(10, 11, pb1, sb) MSX_RT(12, 13, pb2, sb) MSX_RT(14, 15, pb3, sb) MSX_RWAIT
        :
        "=&v"(la[0]), "=&v"(ha[0]), "=&v"(la[1]), "=&v"(ha[1]), "=&v"(la[2]), "=&v"(ha[2]), "=&v"(la[3]),
        "=&v"(ha[3]), "=&v"(lb[0]), "=&v"(hb[0]), "=&v"(lb[1]), "=&v"(hb[1]), "=&v"(lb[2]), "=&v"(hb[2]),
        "=&v"(lb[3]), "=&v"(hb[3])
        :
        [pa0] "v"(pa[0]), [pa1] "v"(pa[1]), [pa2] "v"(pa[2]), [pa3] "v"(pa[3]), [pb0] "v"(pb[0]), [pb1] "v"(pb[1]),
        [pb2] "v"(pb[2]), [pb3] "v"(pb[3]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 2 && J == 2 && AKC && BKC)
    asm volatile(
        MSX_RK(0, pa, sa, 0) MSX_RK(1, pa, sa, 1) MSX_RK(2, pb, sb, 0) MSX_RK(3, pb, sb, 1) MSX_RWAIT
        :
        "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fb[0]), "=&v"(fb[1])
        :
        [pa] "v"(pa[0]), [pb] "v"(pb[0]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 2 && J == 2 && AKC && !BKC)
    asm volatile(
        MSX_RK(0, pa, sa, 0) MSX_RK(1, pa, sa, 1) MSX_RT(2, 3, pb0, sb) MSX_RT(4, 5, pb1, sb) MSX_RWAIT
        :
        "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(lb[0]), "=&v"(hb[0]), "=&v"(lb[1]), "=&v"(hb[1])
        :
        [pa] "v"(pa[0]), [pb0] "v"(pb[0]), [pb1] "v"(pb[1]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 2 && J == 2 && !AKC && BKC)
    asm volatile(
        MSX_RT(0, 1, pa0, sa) MSX_RT(2, 3, pa1, sa) MSX_RK(4, pb, sb, 0) MSX_RK(5, pb, sb, 1) MSX_RWAIT
        :
        "=&v"(la[0]), "=&v"(ha[0]), "=&v"(la[1]), "=&v"(ha[1]), "=&v"(fb[0]), "=&v"(fb[1])
        :
        [pa0] "v"(pa[0]), [pa1] "v"(pa[1]), [pb] "v"(pb[0]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 2 && J == 2 && !AKC && !BKC)
    asm volatile(
        MSX_RT(0, 1, pa0, sa) MSX_RT(2, 3, pa1, sa) MSX_RT(4, 5, pb0, sb) MSX_RT(6, 7, pb1, sb) MSX_RWAIT
        :
        "=&v"(la[0]), "=&v"(ha[0]), "=&v"(la[1]), "=&v"(ha[1]), "=&v"(lb[0]), "=&v"(hb[0]), "=&v"(lb[1]), "=&v"(hb[1])
        :
        [pa0] "v"(pa[0]), [pa1] "v"(pa[1]), [pb0] "v"(pb[0]), [pb1] "v"(pb[1]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 2 && J == 1 && AKC && BKC)
    asm volatile(
        MSX_RK(0, pa, sa, 0) MSX_RK(1, pa, sa, 1) MSX_RK(2, pb, sb, 0) MSX_RWAIT
        :
        "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fb[0])
        :
        [pa] "v"(pa[0]), [pb] "v"(pb[0]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 2 && J == 1 && AKC && !BKC)
    asm volatile(
        MSX_RK(0, pa, sa, 0) MSX_RK(1, pa, sa, 1) MSX_RT(2, 3, pb0, sb) MSX_RWAIT
        :
        "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(lb[0]), "=&v"(hb[0])
        :
        [pa] "v"(pa[0]), [pb0] "v"(pb[0]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 2 && J == 1 && !AKC && BKC)
    asm volatile(
        MSX_RT(0, 1, pa0, sa) MSX_RT(2, 3, pa1, sa) MSX_RK(4, pb, sb, 0) MSX_RWAIT
        :
        "=&v"(la[0]), "=&v"(ha[0]), "=&v"(la[1]), "=&v"(ha[1]), "=&v"(fb[0])
        :
        [pa0] "v"(pa[0]), [pa1] "v"(pa[1]), [pb] "v"(pb[0]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (I == 2 && J == 1 && !AKC && !BKC)
    asm volatile(
        MSX_RT(0, 1, pa0, sa) MSX_RT(2, 3, pa1, sa) MSX_RT(4, 5, pb0, sb) MSX_RWAIT
        :
        "=&v"(la[0]), "=&v"(ha[0]), "=&v"(la[1]), "=&v"(ha[1]), "=&v"(lb[0]), "=&v"(hb[0])
        :
        [pa0] "v"(pa[0]), [pa1] "v"(pa[1]), [pb0] "v"(pb[0]), [sa] "i"(SA), [sb] "i"(SB)
        : "memory");
  if constexpr (!AKC)
#pragma unroll
    for (int u = 0; u < I; ++u) fa[u] = join8(la[u], ha[u]);
  if constexpr (!BKC)
#pragma unroll
    for (int u = 0; u < J; ++u) fb[u] = join8(lb[u], hb[u]);
#endif
}
#undef MSX_RK
#undef MSX_RT
#undef MSX_RWAIT

// GELU and its gradient for values that leave as f16: x s and g (s + x s'), s = 1 / (1 + exp(-v)),
// v = 2 sqrt(2/pi) (x + 0.044715 x^3), on the hardware exp2 and reciprocal (1 ulp each). Against 64 bits
// over x of N(0, 1): 4.7e-8 and 6.6e-8 in f32, where d_gelu and d_gelu_grad have 4.6e-8 and 5.7e-8; rounded
// to f16 2.0649e-4 and 2.0755e-4 with either.
constexpr float kGeluA = -2.0f * 0.797884560802865f * 1.4426950408889634f, kGeluB = kGeluA * 0.044715f;
__device__ __forceinline__ float gelu16(float x) {
  const float e = __builtin_amdgcn_exp2f(x * __builtin_fmaf(kGeluB, x * x, kGeluA));  // exp(-v)
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu_grad16(float x, float g) {
  const float x2 = x * x;
  const float e = __builtin_amdgcn_exp2f(fminf(x * __builtin_fmaf(kGeluB, x2, kGeluA), 126.0f));
  const float s = __builtin_amdgcn_rcpf(1.0f + e), r = e * s;  // r = 1 - s
  const float slope = __builtin_fmaf(6.0f * 0.797884560802865f * 0.044715f, x2, 2.0f * 0.797884560802865f);
  return s * __builtin_fmaf(x * r, slope, 1.0f) * g;
}

// Output columns col .. col + 7 of a row, staged in LDS at src: the epilogue, then the f32 and f16
// outputs. v8: rows of whole 16-byte f16 groups (and 32-byte f32 ones). FAST: the GELU gate above,
// for a problem whose output and pre-activation are f16.
struct Out16Tile {
  float* out;
  _Float16* out16;
  int64_t m, n, ld, zero_to;
  bool more, v8, fast;
};
__device__ __forceinline__ void put8(const Out16Tile& o, const GemmEpi& epi, const float* src, int64_t row, int64_t col) {
  const int64_t at = row * o.ld + col;
  if (!o.v8 || col + 7 >= o.n) {
#pragma unroll 1
    for (int u = 0; u < 8 && col + u < o.zero_to; ++u) {
      const float x = col + u < o.n ? (o.more ? gemm_epilogue(epi, src[u], row, col + u, o.ld) : src[u]) : 0.0f;
      if (o.out) o.out[at + u] = x;
      if (o.out16) o.out16[at + u] = _Float16(x);
    }
    return;
  }
  v4f a = *reinterpret_cast<const v4f*>(src), b = *reinterpret_cast<const v4f*>(src + 4);
  float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  auto load8 = [](const float* p, float (&x)[8]) {
    const v4f lo = *reinterpret_cast<const v4f*>(p), hi = *reinterpret_cast<const v4f*>(p + 4);
#pragma unroll
    for (int u = 0; u < 4; ++u) { x[u] = lo[u]; x[4 + u] = hi[u]; }
  };
  auto store8 = [](float* p, const float (&x)[8]) {
    *reinterpret_cast<v4f*>(p) = v4f{x[0], x[1], x[2], x[3]};
    *reinterpret_cast<v4f*>(p + 4) = v4f{x[4], x[5], x[6], x[7]};
  };
  auto store8h = [](_Float16* p, const float (&x)[8]) {
    *reinterpret_cast<v8h*>(p) = v8h{_Float16(x[0]), _Float16(x[1]), _Float16(x[2]), _Float16(x[3]),
                                     _Float16(x[4]), _Float16(x[5]), _Float16(x[6]), _Float16(x[7])};
  };
  if (o.more) {
    float x[8];
    if (epi.bias) {
      load8(epi.bias + col, x);
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = v[u] + x[u];
    }
    if (epi.act == EPI_GELU || epi.act == EPI_RELU) {
      if (epi.pre16) store8h(epi.pre16 + at, v);
      else if (epi.pre_out) store8(epi.pre_out + at, v);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v[u] = epi.act == EPI_RELU ? (v[u] > 0.0f ? v[u] : 0.0f) : o.fast ? gelu16(v[u]) : d_gelu(v[u]);
    } else if (epi.act == EPI_GELU_GRAD || epi.act == EPI_RELU_GRAD) {
      if (epi.pre16) {
        const v8h h = *reinterpret_cast<const v8h*>(epi.pre16 + at);
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = float(h[u]);
      } else {
        load8(epi.pre_in + at, x);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v[u] = epi.act == EPI_RELU_GRAD ? (x[u] > 0.0f ? v[u] : 0.0f)
                                        : o.fast ? gelu_grad16(x[u], v[u]) : d_gelu_grad(x[u], v[u]);
    }
    if (epi.addend) {
      load8(epi.addend + at, x);
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = x[u] + v[u];
    }
    if (epi.drop_token)
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = epi_drop(epi, v[u], at + u);
  }
  if (o.out) store8(o.out + at, v);
  if (o.out16) store8h(o.out16 + at, v);
}
}  // namespace

struct Gemm16Dims {
  int64_t m, n, k, lda, ldb, ldc, kchunk, zero_to;
  bool v8;
};

// A BM x BN output tile by WGM x WGN waves (I x J MFMA blocks a wave). SUMS: 1, the row sums of op(A)
// over K; 2, the column sums of op(B) (a bias gradient), from the fragments.
//   PP (eight waves, two a SIMD): the waves of the first half multiply while those of the second read
// their next fragments, one barrier apart, so the matrix cores of a SIMD always have one wave's
// products (256 x 192 tiles, one block a CU). Otherwise one barrier a K tile, and the blocks of a CU
// (four of 128 x 128) cover each other's waits.
//   The output leaves through LDS in rows of 16-byte groups, one compact loop of the epilogue: written
// out per accumulator its code was 250 KB and fell out of the instruction cache (16384 x 3072 x 768
// with GELU: 151 us, now 112).
template <int BM, int BN, int WGM, int WGN, int BK, int NS, bool AKC, bool BKC, int SUMS, bool PP>
__global__ __launch_bounds__(64 * WGM * WGN, WGM * WGN == 8 ? 2 : 4) void k_gemm_lds16(GemmPtrs ptrs, Gemm16Dims d, GemmOrder order) {
  constexpr int W = WGM * WGN, KS = BK / 32;
  constexpr int CPR = BK / 8, RPI = 64 / CPR;  // KC tiles: 16-byte chunks a row, rows a load instruction
  constexpr int WTM = BM / WGM, WTN = BN / WGN, I = WTM / 16, J = WTN / 16;
  constexpr int SA = BM * BK, SB = BN * BK, SS = SA + SB;   // halves a stage
  constexpr int PA = SA / 512 / W, PB = SB / 512 / W, LPT = PA + PB;  // a wave's 1 KB load instructions a tile
  static_assert(SA % (512 * W) == 0 && SB % (512 * W) == 0, "whole load instructions a wave");
  static_assert(!PP || (W == 8 && WGM == 2), "two groups of four waves");
  constexpr int LW = WTN + 4, RING = NS * SS * 2;
  // Output rows a wave stages at a time: as many as fit the ring (and a little more).
  constexpr int PR = WTM >= 64 && W * 64 * LW * 4 <= RING + 12 * 1024 ? 64 : WTM >= 32 ? 32 : 16;
  constexpr int STAGE_OUT = W * PR * LW * 4;
  __shared__ __align__(1024) char smem[RING > STAGE_OUT ? RING : STAGE_OUT];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Consecutive blocks go to the 8 XCDs in turn; each XCD takes a contiguous run of the tile order.
  const uint32_t per = gridDim.x / 8, tg = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (tg >= order.tiles * uint32_t(ptrs.count)) return;
  const int qp = int(tg / order.tiles);
  const uint32_t t0 = tg - uint32_t(qp) * order.tiles;
  const uint32_t tz = t0 / (order.mt * order.nt), tr = t0 % (order.mt * order.nt);
  const uint32_t tm = order.m_fastest ? tr % order.mt : tr / order.nt;
  const uint32_t tn = order.m_fastest ? tr / order.mt : tr % order.nt;
  const int64_t M = d.m, N = d.n;
  const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;
  const int64_t kbeg = int64_t(tz) * d.kchunk, kend = d.k < kbeg + d.kchunk ? d.k : kbeg + d.kchunk;
  const int klen = int(kend - kbeg), tiles = (klen + BK - 1) / BK;
  const int left = klen - (tiles - 1) * BK;  // K of the last tile
  const int wm = (wave / WGN) * WTM, wn = (wave % WGN) * WTN;
  auto swz = [](int r) { return BK == 32 ? -(r >> 2) & 3 : r & 7; };
  auto ksw = [](int R, int k) {
    const int b = ((k >> 3) ^ (k >> 4)) & 1;
    return R % 128 == 0 ? 2 * (k & 3) | 8 * b : R >= 64 ? 2 * ((k & 3) ^ b) : 2 * b;
  };
  // A lane's byte offset of load instruction t from the tile's first row and K, and that of the last
  // K tile, where chunks and K rows past the end repeat the first.
  auto offsets = [&](bool kc, int R, int t, int64_t first, int64_t rows, int64_t ld, uint32_t& v, uint32_t& tail) {
    if (kc) {
      const int r = t * RPI + lane / CPR, ch = (lane % CPR) ^ swz(r);
      const int64_t row = first + r < rows ? r : rows - 1 - first;
      v = uint32_t(row * ld + 8 * ch) * 2;
      tail = uint32_t(row * ld + (8 * ch < left ? 8 * ch : 0)) * 2;
    } else {
      const int RQ = R / 8, at = t * 64 + lane, kr = at / RQ, slot = at % RQ;
      int64_t col = 8 * (slot ^ ksw(R, kr));
      if (first + col >= rows) col = ((rows - 1) & ~int64_t(7)) - first;
      v = uint32_t(kr * ld + col) * 2;
      tail = uint32_t((kr < left ? kr : 0) * ld + col) * 2;
    }
  };
  uint32_t vA[PA], vB[PB], tA[PA], tB[PB];
#pragma unroll
  for (int h = 0; h < PA; ++h) offsets(AKC, BM, wave * PA + h, m0, M, d.lda, vA[h], tA[h]);
#pragma unroll
  for (int h = 0; h < PB; ++h) offsets(BKC, BN, wave * PB + h, n0, N, d.ldb, vB[h], tB[h]);
  const int64_t sA = (AKC ? int64_t(BK) : BK * d.lda) * 2, sB = (BKC ? int64_t(BK) : BK * d.ldb) * 2;
  const int64_t oA = (AKC ? m0 * d.lda + kbeg : kbeg * d.lda + m0) * 2;
  const int64_t oB = (BKC ? n0 * d.ldb + kbeg : kbeg * d.ldb + n0) * 2;
  const char* gA = reinterpret_cast<const char*>(ptrs.a16[qp]) + oA;
  const char* gB = reinterpret_cast<const char*>(ptrs.b16[qp]) + oB;
  // K segments: the tiles are loaded in ascending order; at a segment's first tile its operands take
  // over (kseg a multiple of BK, one problem, no split).
  int seg = 0, seg_end = ptrs.ksegs > 1 ? int(ptrs.kseg / BK) : 1 << 30;
  auto issue = [&](int t) {
    if (t == seg_end) {
      ++seg;
      gA = reinterpret_cast<const char*>(ptrs.a16[seg]) + oA - t * sA;
      gB = reinterpret_cast<const char*>(ptrs.b16[seg]) + oB - t * sB;
      seg_end += int(ptrs.kseg / BK);
    }
    char* st = smem + (t % NS) * (SS * 2);
    const char* a = gA + t * sA;
    const char* b = gB + t * sB;
    const bool last = t + 1 == tiles;
#pragma unroll
    for (int h = 0; h < PA; ++h) load_lds16(a + (last ? tA[h] : vA[h]), st + (wave * PA + h) * 1024);
#pragma unroll
    for (int h = 0; h < PB; ++h) load_lds16(b + (last ? tB[h] : vB[h]), st + SA * 2 + (wave * PB + h) * 1024);
  };
  v4f acc[I][J];
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  // Fragment addresses in stage 0, K step 0.
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)(smem)));
  auto frag_at = [&](bool kc, int R, int w, int u, uint32_t base) {
    if (kc) return base + uint32_t((w + c) * (2 * BK) + 16 * (q ^ swz(c)));
    const int k = 8 * q + c / 4, row = w + 16 * u + 4 * (c % 4);
    return base + uint32_t((k * R + ((row / 8) ^ ksw(R, k)) * 8 + row % 8) * 2);
  };
  constexpr int NPA = AKC ? 1 : I, NPB = BKC ? 1 : J;
  uint32_t pA[NPA], pB[NPB];
#pragma unroll
  for (int u = 0; u < NPA; ++u) pA[u] = frag_at(AKC, BM, wm, u, lds0);
#pragma unroll
  for (int u = 0; u < NPB; ++u) pB[u] = frag_at(BKC, BN, wn, u, lds0 + SA * 2);
  // Sums over K by the waves of the first wave column (row) of the first tile column (row).
  constexpr int SN = SUMS == 1 ? I : SUMS == 2 ? J : 1;
  float ksum[SN];
#pragma unroll
  for (int u = 0; u < SN; ++u) ksum[u] = 0.0f;
  const bool sum_wave = SUMS == 1 ? wn == 0 && tn == 0 : SUMS == 2 ? wm == 0 && tm == 0 : false;
  v8h fa[I], fb[J];
  auto read = [&](int t, int ks) {
    // K step ks: chunk 4 ks + q of a KC row (its slot's XOR), or 32 ks K rows further.
    const uint32_t off = uint32_t(t % NS) * (SS * 2);
    uint32_t xa[NPA], xb[NPB];
#pragma unroll
    for (int u = 0; u < NPA; ++u) xa[u] = AKC ? (pA[u] ^ (64 * ks)) + off : pA[u] + off + ks * (64 * BM);
#pragma unroll
    for (int u = 0; u < NPB; ++u) xb[u] = BKC ? (pB[u] ^ (64 * ks)) + off : pB[u] + off + ks * (64 * BN);
    read_frags<I, J, AKC, BKC, AKC ? 32 * BK : 8 * BM, BKC ? 32 * BK : 8 * BN>(xa, xb, fa, fb);
    if (left < BK && t + 1 == tiles) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool in = 32 * ks + 8 * q + e < left;
#pragma unroll
        for (int i = 0; i < I; ++i) fa[i][e] = in ? fa[i][e] : _Float16(0.0f);
#pragma unroll
        for (int j = 0; j < J; ++j) fb[j][e] = in ? fb[j][e] : _Float16(0.0f);
      }
    }
  };
  auto multiply = [&]() {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
    if (SUMS != 0 && sum_wave) {
      // v_dot2_f32_f16 against (1, 1): two halves added into the f32 sum a VALU op.
      typedef _Float16 v2h_ __attribute__((ext_vector_type(2)));
      const v2h_ one{_Float16(1.0f), _Float16(1.0f)};
#pragma unroll
      for (int u = 0; u < SN; ++u) {
        const v8h x = SUMS == 1 ? fa[u % I] : fb[u % J];
#pragma unroll
        for (int e = 0; e < 4; ++e) ksum[u] = __builtin_amdgcn_fdot2(v2h_{x[2 * e], x[2 * e + 1]}, one, ksum[u], false);
      }
    }
  };
  // Waits until this wave's loads of tile t have landed, with those of tiles below `issued` issued.
  auto landed = [&](int t, int issued) {
    if (issued - 1 - t >= NS - 2) wait_vm((NS - 2) * LPT);
    else wait_vm(0);
  };
  const int pre = tiles < NS - 1 ? tiles : NS - 1;
  for (int t = 0; t < pre; ++t) issue(t);
  if constexpr (PP) {
    // The second group runs one barrier behind: while one group is between its reads and its second
    // barrier, the other is between its barriers' other pair. A stage is overwritten by loads issued
    // after the barrier that follows both groups' last read of it; a tile's loads are waited for by
    // each wave before the last barrier ahead of the first group's first read of it.
    landed(0, pre);
    __builtin_amdgcn_s_barrier();
    if (wave >= 4) __builtin_amdgcn_s_barrier();
#pragma unroll 1
    for (int t = 0; t < tiles; ++t) {
      if (t + NS - 1 < tiles) issue(t + NS - 1);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        read(t, ks);
        if (ks == KS - 1 && t + 1 < tiles) landed(t + 1, t + NS < tiles ? t + NS : tiles);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_setprio(1);
        __builtin_amdgcn_sched_barrier(0);
        multiply();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (wave < 4) __builtin_amdgcn_s_barrier();
  } else {
    // The barrier follows every wave's reads of tile t - 1, whose stage the loads then overwrite.
#pragma unroll 1
    for (int t = 0; t < tiles; ++t) {
      landed(t, t + NS - 1 < tiles ? t + NS - 1 : tiles);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (t + NS - 1 < tiles) issue(t + NS - 1);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        read(t, ks);
        multiply();
      }
    }
  }
  __syncthreads();  // every wave is past its last read of the ring before any stages output over it
  float* __restrict__ ws = ptrs.ws[qp];
  const GemmEpi epi = ptrs.epi[qp];
  const bool more = !ws && (epi.bias || epi.act != EPI_NONE || epi.addend || epi.drop_token);
  const Out16Tile o{ws ? ws + int64_t(tz) * M * N : ptrs.c[qp], ws ? nullptr : ptrs.c16[qp], M, N, ws ? N : d.ldc,
                    ws ? N : d.zero_to, more, d.v8, !ptrs.c[qp] && epi.pre16};
  float* mine = reinterpret_cast<float*>(smem) + wave * (PR * LW);
  constexpr int CH = WTN / 8;  // 8-column groups a row
#pragma unroll
  for (int ps = 0; ps < WTM / PR; ++ps) {
#pragma unroll
    for (int i = 0; i < PR / 16; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j)
        *reinterpret_cast<v4f*>(mine + (16 * i + c) * LW + 16 * j + 4 * q) = acc[ps * (PR / 16) + i][j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll 1
    for (int e = lane; e < PR * CH; e += 64) {
      const int rl = e / CH, cc = (e % CH) * 8;
      const int64_t row = m0 + wm + ps * PR + rl, col = n0 + wn + cc;
      if (row < M && col < o.zero_to) put8(o, epi, mine + rl * LW + cc, row, col);
    }
    __builtin_amdgcn_wave_barrier();
  }
  if constexpr (SUMS != 0) {
    // The lane groups q hold disjoint K: added across them (a fixed order), written by group 0.
#pragma unroll
    for (int u = 0; u < SN; ++u) {
      ksum[u] += __shfl_xor(ksum[u], 16, 64);
      ksum[u] += __shfl_xor(ksum[u], 32, 64);
    }
    float* colsum = ptrs.colsum[qp];
    if (sum_wave && q == 0 && colsum) {
      const int64_t base = SUMS == 1 ? m0 + wm : n0 + wn, width = SUMS == 1 ? M : N;
      float* dst = colsum + (ws ? int64_t(tz) * width : 0);
#pragma unroll
      for (int u = 0; u < SN; ++u) {
        const int64_t at = base + 16 * u + c;
        if (at < width) dst[at] = ksum[u];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// A lane's offset from its tile's first row and K is 32 bits of bytes: up to 255 rows of a KC operand,
// 63 of another. K, in 32 bits too, is counted up to the end of its last tile.
bool gemm16_takes(int64_t lda, bool akc, int64_t ldb, bool bkc, int64_t k) {
  auto pitch = [](int64_t ld, bool kc) { return ld % 8 == 0 && ld <= (int64_t(1) << (kc ? 23 : 25)); };
  return pitch(lda, akc) && pitch(ldb, bkc) && k <= INT32_MAX - 63;
}
bool gemm16_layout(const GemmArgs& o) { return gemm16_takes(o.lda, !o.ta, o.ldb, o.tb, o.k); }

// Split-K of a mixed-precision product. A deferred one (a weight gradient, its slices summed by the
// batched finalize) takes up to 1024 128 x 128 tiles; its slices keep 3200 K of a K of 8192 or more
// (BERT-base's 16384: five slices, so that the 48 256 x 192 tiles of a 768 x 3072 gradient, or of the
// four 768 x 768 ones of a layer in one launch, come to 240 blocks), 512 of a shorter one. Another is
// split only where K is 8192 or more and its tiles would leave the chip idle (the decoder's input
// gradient, 2880 x 768 over 30522: 48 tiles in five slices); shorter ones take smaller tiles instead
// (2048 x 256 over 1024: 64 x 64 tiles 9.0 us, split 128 x 128 tiles and their sum 26).
Split16 gemm16_split(int64_t m, int64_t n, int64_t k, bool defer) {
  const int64_t tiles = ((m + 127) / 128) * ((n + 127) / 128), wide = ((m + 255) / 256) * ((n + 191) / 192);
  int64_t split = 1;
  if (defer && tiles < 256) split = std::min((1023 + tiles) / tiles, k / (k >= 8192 ? 3200 : 512));
  else if (!defer && tiles < 256 && k >= 8192) split = std::min((255 + wide) / wide, k / 2048);
  if (split < 1) split = 1;
  Split16 p;
  p.chunk = ((k + split - 1) / split + 63) / 64 * 64;
  p.split = int((k + p.chunk - 1) / p.chunk);
  return p;
}

bool gemm16(hipStream_t s, const GemmArgs* list, int count, const GemmPtrs& ptrs, int split, int64_t chunk) {
  const GemmArgs& g = list[0];
  auto al16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool akc = !g.ta, bkc = g.tb, segs = ptrs.ksegs > 1;
  if (!gemm16_layout(g)) return false;
  const int operands = segs ? ptrs.ksegs : count;
  for (int q = 0; q < operands; ++q)
    if (!ptrs.a16[q] || !ptrs.b16[q] || !al16(ptrs.a16[q]) || !al16(ptrs.b16[q])) return false;
  if (segs && (count != 1 || split != 1 || ptrs.kseg % 64 != 0)) return false;
  // 32-byte f32 groups and 16-byte f16 groups of the output rows.
  bool v8 = true;
  for (int q = 0; q < count; ++q) {
    const GemmArgs& o = list[q];
    v8 = v8 && (ptrs.ws[q] ? (o.n % 4 == 0 && al16(ptrs.ws[q]))
                           : (o.ldc % 8 == 0 && al16(o.c) && al16(o.c16) && al16(o.bias) && al16(o.addend) &&
                              al16(o.pre_in) && al16(o.pre_out) && al16(o.pre16)));
  }
  const Gemm16Dims dims{g.m, g.n, g.k, g.lda, g.ldb, g.ldc, split > 1 ? chunk : g.k, g.pad_c ? g.ldc : g.n, v8};
  const int sums = g.colsum ? (g.sum_a ? 1 : 2) : 0;
  auto blocks = [&](int bm, int bn) { return ((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * split * count; };
  GemmOrder order{};
  dim3 grid;
  auto plan = [&](int bm, int bn) {
    const int64_t all = blocks(bm, bn);
    if (all > (int64_t(1) << 30)) bad("gemm has too many tiles");
    order = GemmOrder{uint32_t((g.m + bm - 1) / bm), uint32_t((g.n + bn - 1) / bn), uint32_t(all / count),
                      g.n * g.k >= g.m * g.k};
    grid = dim3(unsigned((all + 7) / 8 * 8));
  };
  // The tile, from timings of the BERT shapes on one MI355X (us):
  //   few blocks: 64 x 32 while every block has a CU of its own (64 x 768 x 3072: 17.8 against 18.7 with
  //   64 x 64 and 40 with 128 x 128 tiles), else 64 x 64 while 128 x 128 would leave CUs idle (2048 x
  //   1024 x 256: 8.5 against 16.2);
  //   256 x 192 (a K tile of 64 takes a CU 1.40) against 128 x 128 (0.576 for each block of a CU), by
  //   their rounds: 16384 x 768 x 3072 71 against 83, 16384 x 768 x 768 27 against 28.5, but 2816 x 768
  //   x 768 x 3 26 against 20. An activation's epilogue leaves one block a CU idle matrix cores
  //   (16384 x 3072 x 768 with GELU 124 against 112): it stays on 128 x 128.
#define MSX_GO16(BM, BN, WGM, WGN, BK, NS, AK, BK_, S, PP)                                                          \
  do {                                                                                                              \
    plan(BM, BN);                                                                                                   \
    MSX_LAUNCH((k_gemm_lds16<BM, BN, WGM, WGN, BK, NS, AK, BK_, S, PP>), grid, dim3(64 * WGM * WGN), 0, s, ptrs, dims, order); \
    return true;                                                                                                    \
  } while (0)
  const int64_t b128 = blocks(128, 128), wide = blocks(256, 192);
  const bool pp = b128 >= 256 && g.act == EPI_NONE && (akc || !bkc) && (!sums || (!akc && !bkc)) &&
                  double((wide + 255) / 256) * 1.40 < double((b128 + 255) / 256) * 0.576;
  if (pp) {
    if (akc && bkc) MSX_GO16(256, 192, 2, 4, 64, 2, true, true, 0, true);
    if (akc) MSX_GO16(256, 192, 2, 4, 64, 2, true, false, 0, true);
    if (sums == 1) MSX_GO16(256, 192, 2, 4, 64, 2, false, false, 1, true);
    if (sums == 2) MSX_GO16(256, 192, 2, 4, 64, 2, false, false, 2, true);
    MSX_GO16(256, 192, 2, 4, 64, 2, false, false, 0, true);
  }
#define MSX_GO16_S(BM, BN, BK, NS, AK, BK_)                                \
  if (sums == 1) MSX_GO16(BM, BN, 2, 2, BK, NS, AK, BK_, 1, false);        \
  else if (sums == 2) MSX_GO16(BM, BN, 2, 2, BK, NS, AK, BK_, 2, false);   \
  else MSX_GO16(BM, BN, 2, 2, BK, NS, AK, BK_, 0, false)
#define MSX_GO16_T(BM, BN, BK, NS)                                   \
  if (akc && bkc) { MSX_GO16_S(BM, BN, BK, NS, true, true); }        \
  else if (akc) { MSX_GO16_S(BM, BN, BK, NS, true, false); }         \
  else if (bkc) { MSX_GO16_S(BM, BN, BK, NS, false, true); }         \
  else { MSX_GO16_S(BM, BN, BK, NS, false, false); }
  if (blocks(64, 32) <= 256) {
    MSX_GO16_T(64, 32, 64, 4)
  } else if (b128 < 256) {
    MSX_GO16_T(64, 64, 64, 2)
  } else {
    MSX_GO16_T(128, 128, 32, 2)
  }
#undef MSX_GO16_T
#undef MSX_GO16_S
#undef MSX_GO16
  return true;
}

}  // namespace msx::hk
