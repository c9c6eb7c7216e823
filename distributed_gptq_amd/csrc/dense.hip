// Dense product C = A B^T on gfx950 MFMA: A (M x K) and B (N x K) bf16 or
// fp16 with the contraction contiguous, fp32 accumulation, C (M x N) rounded
// once to A's type.
#include <type_traits>

#include "mfma_lds.hpp"

namespace gptq {
namespace {

// One workgroup of 4 waves (one per SIMD) per C tile of 256 x 32 NBJ; wave w
// owns the 128 x 16 NBJ block (w / 2, w % 2) as 8 x NBJ MFMA 16x16 blocks (at
// the power limit the chip runs these products ~5% faster than with 32x32
// blocks).  Stages of 64 k alternate between two LDS buffers, filled by
// buffer_load ... lds: an LDS row is the 128 bytes (eight 16-byte chunks, one
// cache line) of one matrix row, chunk c at slot c ^ row_sig(row), so that the
// fragment reads hit distinct banks.
//
// Schedule, per stage of two halves (32 k each), one register set per half:
//   * the second half's fragments are read under the first MFMAs; a barrier
//     then frees the stage's buffer, and the copies of the stage two ahead go
//     into it, spread over the MFMAs up to the second barrier;
//   * before that a wave waits for its copies of the next stage (issued one
//     and a half stages ago), after it the next stage's first half is read
//     under the last MFMAs.
// The barriers are bare: the compiler's own would also wait for the copies.
//
// Bound by the matrix units at the power limit.  Measured alone (bf16 / fp16,
// us): 8192^3 728 / 756 (1511 TFLOP/s in bf16), 4096 x 4096 x 14336 302 / 317
// (1591), 2048 x 28672 x 4096 347 / 364 (1388).  On the way (bf16, 8192^3):
// 32-k stages (64-byte rows, half cache lines) with 32x32 MFMAs 854, with 16x16
// MFMAs 810; the scalar address work after a barrier instead of before it cost
// a tenth of a stage.
constexpr int kBK = 64;
constexpr int kRowBytes = kBK * 2;
constexpr int kTileM = 256;
constexpr int kOperandBytes = 256 * kRowBytes;

__shared__ __attribute__((aligned(1024))) uint8_t g_d0[2][kOperandBytes];
__shared__ __attribute__((aligned(1024))) uint8_t g_d1[2][kOperandBytes];

template <int B>
__device__ __forceinline__ uint8_t* dbuf(int op) {
  return B == 0 ? &g_d0[op][0] : &g_d1[op][0];
}
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
// (generic -> LDS address-space casts have to be C-style; an LDS pointer keeps
// the epilogue's accesses ds instructions)
__device__ __forceinline__ lds_u8* dbuf_of(int wave) {
  lds_u8* p0 = (lds_u8*)&g_d0[0][0];
  lds_u8* p1 = (lds_u8*)&g_d1[0][0];
  return (wave & 2 ? p1 : p0) + (wave & 1) * kOperandBytes;
}

// A 128-bit LDS read serves 16 lanes at a time, in groups of lanes 0-3,
// 12-15, 20-23, 24-27 (and the complement, and both 32 lanes up): with lane l
// on row l % 16, chunk l / 16, this puts a group on 16 distinct bank quads.
__device__ __forceinline__ int row_sig(int row) { return (row >> 1) & 7; }

struct DenseArgs {
  const uint16_t* A;
  const uint16_t* B;
  uint16_t* C;
  const void* bias;     // N values or null
  const int32_t* inexact;  // kPlaneFlags ints: all zero -> the third B plane is zero everywhere (or null)
  int64_t lda, ldb, ldc;
  int M, N;
  int ks;               // contraction of one (A plane, B plane) segment, a multiple of kBK
  int aplanes, bplanes;
  int bias_dtype;
  int ntm, ntn;         // tiles of 256 x 256
  int full;             // workgroups below this take whole tiles, the rest halves of the tiles after them
};

// Tile t in band order: bands of up to 8 tile rows walked column by column,
// so that 32 consecutive tiles (one XCD's share of a round) read 8 panels of
// A and 4 of B.
__device__ __forceinline__ void dense_coords(int t, int ntm, int ntn, int& tm, int& tn) {
  const int band = 8 * ntn;
  const int b = t / band, r0 = 8 * b;
  const int h = ntm - r0 < 8 ? ntm - r0 : 8;
  const int u = t - b * band;
  tn = u / h;
  tm = r0 + (u - tn * h);
}

__device__ __forceinline__ bool nonfinite16(uint32_t h, bool bf16) {
  return bf16 ? (h & 0x7F80u) == 0x7F80u : (h & 0x7C00u) == 0x7C00u;
}

// OUT_BF16: C's type (A's own unless A is split into planes)
//
// With planes, a tile with an infinite or NaN result is multiplied again, the
// first planes alone, and its infinite and NaN sums replace those results: an
// infinity times a zero low plane is no term of the product, and the first
// planes are zero, infinite or NaN where the whole values are (down to bf16's
// subnormals).  A finite sum that only rounds to an infinity stays.  This costs
// one plane pair more: the gradient of 1024 x 4096 x 4096, bf16, takes 172 us
// with one infinity in each row or all NaN and 122 us without (4-bit weights;
// summed again one element at a time it took 148 ms).
template <bool kBF16, bool kOutBF16, bool kPlanes, int NBJ>
__device__ __forceinline__ void dense_tile(const DenseArgs& a, int m0, int n0, int bplanes) {
  constexpr int NM = 8 * NBJ;  // MFMAs per half
  constexpr int NF = 8 + NBJ;  // fragments per half
  constexpr int NC = 8 + NBJ;  // copies per wave and stage

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int wm = (wave >> 1) * 128, wn = (wave & 1) * 16 * NBJ;

  // copy role: copy k of this wave fills LDS rows 8 (wave + 4k) .. + 7 of A
  // (k < 8) or B; lane l lands on row l / 8, slot l % 8
  const int64_t rowa = a.lda * 2, rowb = a.ldb * 2;
  uint32_t voff[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int row = 8 * (wave + 4 * (k < 8 ? k : k - 8)) + (lane >> 3);
    voff[k] = static_cast<uint32_t>(row * (k < 8 ? rowa : rowb) + ((lane & 7) ^ row_sig(row)) * 16);
  }
  const uint16_t* baseA = a.A + static_cast<int64_t>(m0) * a.lda;
  const uint16_t* baseB = a.B + static_cast<int64_t>(n0) * a.ldb;
  const int rowsA = a.M - m0 < kTileM ? a.M - m0 : kTileM;
  const int rowsB = a.N - n0 < 32 * NBJ ? a.N - n0 : 32 * NBJ;
  const uint32_t recA = static_cast<uint32_t>(rowsA * rowa), recB = static_cast<uint32_t>(rowsB * rowb);

  // fragment role: lane l holds row l % 16, k 8 (l / 16) .. + 7 of a half.
  // Offsets for buffer 0, and the same 64 KB up for buffer 1 (opaque, and
  // subtracted again below), so that a read's constant part fits the
  // instruction's 16-bit offset instead of costing an add.
  const int frow = lane & 15;
  int aoff[2][2], boff[2][2];  // [half][buffer]
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int foff = frow * kRowBytes + ((4 * h + (lane >> 4)) ^ row_sig(frow)) * 16;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      aoff[h][u] = wm * kRowBytes + foff + u * 65536;
      boff[h][u] = wn * kRowBytes + foff + u * 65536;
      asm volatile("" : "+v"(aoff[h][u]), "+v"(boff[h][u]));
    }
  }

  int ap = kPlanes ? a.aplanes : 1, bp = kPlanes ? bplanes : 1;
  for (bool again = false;; again = true) {
    // the stage being copied: byte offsets of its first column of A and B and
    // the record counts (zero past the end: nothing is fetched).  Segment s
    // multiplies A plane s % ap with B plane s / ap.  The descriptors
    // stay fixed and the columns go through the scalar offset; a row past the
    // matrix is past the records whether the hardware counts that offset in the
    // bounds check or not.
    const int nst = ap * bp * (a.ks / kBK);
    const int seg = 2 * a.ks;
    struct Src {
      int oa, ob;
      uint32_t na, nb;
    };
    int f_k = 0, f_a = 0, f_b = 0;  // bytes: in the segment, of the A and the B plane
    const int f_aend = ap * seg, f_bend = bp * seg;
    auto front = [&]() {
      Src s;
      s.oa = f_a + f_k;
      s.ob = f_b + f_k;
      s.na = f_b < f_bend ? recA : 0u;
      s.nb = f_b < f_bend ? recB : 0u;
      f_k += kRowBytes;
      const bool wrap = f_k >= seg;
      f_k = wrap ? 0 : f_k;
      f_a = wrap ? f_a + seg : f_a;
      const bool next = f_a >= f_aend;
      f_a = next ? 0 : f_a;
      f_b = next ? f_b + seg : f_b;
      return s;
    };
    auto copy = [&](const Src& s, auto bsel, auto ksel) {
      constexpr int B = decltype(bsel)::value, k = decltype(ksel)::value;
      if constexpr (k < 8)
        lds_copy16(baseA, s.na, dbuf<B>(0) + (wave + 4 * k) * 1024, voff[k], s.oa);
      else
        lds_copy16(baseB, s.nb, dbuf<B>(1) + (wave + 4 * (k - 8)) * 1024, voff[k], s.ob);
    };

    f32x4 acc[8][NBJ];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < NBJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    u32x4 fr[2][NF];  // [half][A0..A7, B0..]
    // fragment f of half h of buffer B, in the order the MFMAs need them: A0, all of B, A1..A7
    auto read = [&](auto bsel, auto hsel, auto fsel) {
      constexpr int B = decltype(bsel)::value, h = decltype(hsel)::value, f = decltype(fsel)::value;
      constexpr int idx = f == 0 ? 0 : f <= NBJ ? f + 7 : f - NBJ;
      const lds_u8* p = idx < 8 ? (const lds_u8*)dbuf<B>(0) + (aoff[h][B] + (idx * 16 * kRowBytes - B * 65536))
                                : (const lds_u8*)dbuf<B>(1) + (boff[h][B] + ((idx - 8) * 16 * kRowBytes - B * 65536));
      fr[h][idx] = *(const lds_u32x4*)p;
    };
    // B's rows first: a lane's accumulators then run along n (C's contiguous side)
    auto mfma = [&](auto msel) {
      constexpr int h = decltype(msel)::value / NM, m = decltype(msel)::value % NM;
      mfma16_asm<kBF16>(acc[m / NBJ][m % NBJ], fr[h][8 + m % NBJ], fr[h][m / NBJ]);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;

    constexpr int kFree = NF + 4;            // MFMAs before the barrier that frees the buffer
    constexpr int kNext = 2 * NM - NF - 4;   // MFMAs before the next stage's first reads
    constexpr int kEvery = (kNext - kFree) / NC;
    Src src;  // of the stage being copied
    auto stage = [&](auto bsel) {
      constexpr int B = decltype(bsel)::value;
      using Bn = std::integral_constant<int, 1 - B>;
      // the scalar work for this stage's copies sits under these MFMAs (after
      // the barrier it would hold up the MFMA pipe)
      src = front();
      sfor<0, kFree>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        mfma(mc);
        if constexpr (m < NF) read(bsel, I1{}, mc);
      });
      sfor<0, kFree>([&](auto mc) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr (decltype(mc)::value < NF) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x004, 2, 0);
      });
      asm volatile("" : "+s"(src.oa), "+s"(src.ob), "+s"(src.na), "+s"(src.nb), "+s"(f_k), "+s"(f_a), "+s"(f_b));
      __builtin_amdgcn_sched_barrier(0);
      wait_lgkm<0>();
      bare_barrier();
      __builtin_amdgcn_sched_barrier(0);
      sfor<kFree, kNext>([&](auto mc) {
        constexpr int m = decltype(mc)::value - kFree;
        mfma(mc);
        if constexpr (m % kEvery == 0 && m / kEvery < NC) copy(src, bsel, std::integral_constant<int, m / kEvery>{});
      });
      sfor<kFree, kNext>([&](auto mc) {
        constexpr int m = decltype(mc)::value - kFree;
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr (m % kEvery == 0 && m / kEvery < NC) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      });
      __builtin_amdgcn_sched_barrier(0);
      wait_vm<NC>();
      bare_barrier();
      __builtin_amdgcn_sched_barrier(0);
      sfor<kNext, 2 * NM>([&](auto mc) {
        constexpr int m = decltype(mc)::value - kNext;
        mfma(mc);
        if constexpr (m < NF) read(Bn{}, I0{}, std::integral_constant<int, m>{});
      });
      sfor<kNext, 2 * NM>([&](auto mc) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr (decltype(mc)::value - kNext < NF) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      });
      __builtin_amdgcn_sched_barrier(0);
    };

    src = front();
    sfor<0, NC>([&](auto kc) { copy(src, I0{}, kc); });
    src = front();
    sfor<0, NC>([&](auto kc) { copy(src, I1{}, kc); });
    wait_vm<NC>();
    bare_barrier();
    __builtin_amdgcn_sched_barrier(0);
    sfor<0, NF>([&](auto fc) { read(I0{}, I0{}, fc); });
    // two stages per trip, one per buffer; a stage past the end multiplies zeros
    // (zero-record copies), which leaves the sums unchanged
    for (int t = 0; t < nst; t += 2) {
      stage(I0{});
      stage(I1{});
    }
    // no copy may still be writing LDS, and no wave reading it, when the
    // epilogue reuses the buffers
    wait_vm<0>();
    wait_lgkm<0>();
    bare_barrier();
    mfma_settle();
    if (kPlanes && again) {  // zeros in place of what stays as it is
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j) {
          asm volatile("" : "+a"(acc[i][j]));
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][e] = fabsf(acc[i][j][e]) < INFINITY ? 0.0f : acc[i][j][e];
          asm volatile("" : "+a"(acc[i][j]));
        }
    }

    // Epilogue through LDS, each wave in a buffer of its own: lane l, register
    // v of block (i, j) is row 16i + l % 16, column 16j + 4 (l / 16) + v.  Rows
    // of 32 NBJ bytes in 16-byte chunks, chunk c at c ^ (row % chunks), then
    // 16-byte stores along C's rows.
    // (el: the lane, opaque, so that the addresses are not kept through the loop)
    int el = lane;
    if constexpr (kPlanes) asm volatile("" : "+v"(el));
    constexpr int kChunks = 2 * NBJ;
    constexpr int kRB = kChunks * 16;
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
    lds_u8* own = dbuf_of(wave);
#pragma unroll
    for (int j = 0; j < NBJ; ++j) {
      float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (a.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = n0 + wn + 16 * j + 4 * (el >> 4) + e;
          b[e] = load_elem(a.bias, n < a.N ? n : a.N - 1, a.bias_dtype);
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // (stays in AGPRs up to here: with all blocks copied out at the start a
        // spill of one of them was placed before the wait states)
        asm volatile("" : "+a"(acc[i][j]));
        f32x4 y = acc[i][j];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] += b[e];
        const int row = 16 * i + (el & 15);
        lds_u8* at = own + row * kRB + (((2 * j + (el >> 5)) ^ (row & (kChunks - 1))) * 16) + ((el >> 4) & 1) * 8;
        *(lds_u32x2*)at =
            kOutBF16 ? u32x2{pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3])}
                     : u32x2{pack_f16(y[0], y[1]), pack_f16(y[2], y[3])};
      }
    }
    wave_sync();
    constexpr int kRows = 64 / kChunks;  // rows per pass
    const int chunk = el % kChunks;
    const int n = n0 + wn + 8 * chunk;
    bool redo = false;
    for (int it = 0; it < 128 / kRows; ++it) {
      const int row = it * kRows + el / kChunks;
      const int m = m0 + wm + row;
      u32x4 v = *(const lds_u32x4*)(own + row * kRB + ((chunk ^ (row & (kChunks - 1))) * 16));
      if (m >= a.M || n >= a.N) continue;
      u32x4* out = reinterpret_cast<u32x4*>(a.C + static_cast<int64_t>(m) * a.ldc + n);
      if constexpr (kPlanes) {
        const u32x4 old = again ? *out : v;  // (written by this thread)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t mask = 0xFFFFu << (16 * (e & 1));
          const bool bad = nonfinite16((old[e / 2] >> (16 * (e & 1))) & 0xFFFFu, kOutBF16);
          redo = redo || bad;
          if (!bad || (v[e / 2] & mask) == 0) v[e / 2] = (v[e / 2] & ~mask) | (old[e / 2] & mask);
        }
      }
      *out = v;
    }
    // (also the barrier before the buffers are filled again)
    if (!kPlanes || again || !__syncthreads_or(redo)) break;
    wait_vm<0>();  // the stores, which the waits for copies would count
    ap = bp = 1;
  }
}

constexpr int kPlaneFlags = 256;

template <bool kBF16, bool kOutBF16, bool kPlanes>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void dense_nt_k(DenseArgs a) {
  // each round of 256 workgroups (the last one with what is left) is permuted
  // so that XCD x (workgroups x, x + 8, ...) runs consecutive tiles
  int b = blockIdx.x;
  {
    const int r0 = b & ~255, x = b & 7, q = (b & 255) >> 3;
    const int w = static_cast<int>(gridDim.x) - r0 < 256 ? static_cast<int>(gridDim.x) - r0 : 256;
    b = r0 + x * (w >> 3) + (x < (w & 7) ? x : (w & 7)) + q;
  }
  int bplanes = a.bplanes;
  if (kPlanes && a.inexact) {
    int any = 0;
#pragma unroll
    for (int i = 0; i < kPlaneFlags / 64; ++i) any |= a.inexact[i * 64 + (threadIdx.x & 63)];
    bplanes = __ballot(any != 0) != 0 ? 3 : 2;
  }
  bplanes = __builtin_amdgcn_readfirstlane(bplanes);
  int tm, tn;
  if (b < a.full) {
    dense_coords(b, a.ntm, a.ntn, tm, tn);
    dense_tile<kBF16, kOutBF16, kPlanes, 8>(a, tm * 256, tn * 256, bplanes);
  } else {
    const int h = b - a.full;
    dense_coords(a.full + h / 2, a.ntm, a.ntn, tm, tn);
    const int n0 = tn * 256 + (h & 1) * 128;
    if (n0 < a.N) dense_tile<kBF16, kOutBF16, kPlanes, 4>(a, tm * 256, n0, bplanes);
  }
}

// fp16 -> two bf16 planes side by side (M x 2N): 11 bits are 8 and 3, exact;
// an infinity or NaN has a zero low plane
__global__ __launch_bounds__(256) void split_fp16_k(const uint16_t* __restrict__ x, int64_t n8, int64_t M, int64_t N,
                                                    uint16_t* __restrict__ out) {
  const int64_t total = M * n8;
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < total; i += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t m = i / n8, c = (i - m * n8) * 8;
    const u32x4 v = *reinterpret_cast<const u32x4*>(x + m * N + c);
    u32x4 hi, lo;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t h2 = 0, l2 = 0;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float f = f16_bits_to_f32(static_cast<uint16_t>(v[d] >> (16 * e)));
        const uint16_t h = f32_to_bf16_bits(f);
        const float r = f - bf16_bits_to_f32(h);
        const uint16_t l = (h & 0x7F80u) == 0x7F80u ? 0 : f32_to_bf16_bits(r);
        h2 |= static_cast<uint32_t>(h) << (16 * e);
        l2 |= static_cast<uint32_t>(l) << (16 * e);
      }
      hi[d] = h2;
      lo[d] = l2;
    }
    *reinterpret_cast<u32x4*>(out + m * 2 * N + c) = hi;
    *reinterpret_cast<u32x4*>(out + m * 2 * N + N + c) = lo;
  }
}

}  // namespace
}  // namespace gptq

using namespace gptq;

extern "C" int gptq_matmul_nt(const void* A, int64_t lda, const void* B, int64_t ldb, int dtype, int64_t M, int64_t N,
                              int64_t K, int aplanes, int bplanes, const int32_t* inexact, const void* bias,
                              int bias_dtype, void* C, int64_t ldc, int out_dtype, gptq_stream_t stream) {
  clear_error();
  GPTQ_REQUIRE(A && B && C, GPTQ_ERR_ARG, "matmul_nt: null pointer");
  GPTQ_REQUIRE((dtype == GPTQ_F16 || dtype == GPTQ_BF16) && (out_dtype == GPTQ_F16 || out_dtype == GPTQ_BF16) &&
                   (!bias || valid_dtype(bias_dtype)), GPTQ_ERR_DTYPE, "matmul_nt: bad dtype");
  GPTQ_REQUIRE(aplanes >= 1 && aplanes <= 2 && bplanes >= 1 && bplanes <= 3, GPTQ_ERR_ARG, "matmul_nt: bad planes");
  GPTQ_REQUIRE((aplanes * bplanes == 1 && !inexact && dtype == out_dtype) || (dtype == GPTQ_BF16 && bplanes == 3),
               GPTQ_ERR_ARG, "matmul_nt: planes are bf16");
  GPTQ_REQUIRE(M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && ldc % 8 == 0 &&
                   lda >= aplanes * K && ldb >= bplanes * K && ldc >= N && M <= (1 << 24) && N <= (1 << 24) &&
                   K <= (1 << 24) && lda < (1 << 22) && ldb < (1 << 22),
               GPTQ_ERR_SHAPE, "matmul_nt: bad shape M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
  GPTQ_REQUIRE(reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(C) % 16 == 0, GPTQ_ERR_ARG, "matmul_nt: operands must be 16-byte aligned");
  DenseArgs a;
  a.A = static_cast<const uint16_t*>(A);
  a.B = static_cast<const uint16_t*>(B);
  a.C = static_cast<uint16_t*>(C);
  a.bias = bias;
  a.inexact = inexact;
  a.lda = lda; a.ldb = ldb; a.ldc = ldc;
  a.M = static_cast<int>(M); a.N = static_cast<int>(N); a.ks = static_cast<int>(K);
  a.aplanes = aplanes; a.bplanes = bplanes; a.bias_dtype = bias_dtype;
  a.ntm = static_cast<int>(cdiv(M, 256)); a.ntn = static_cast<int>(cdiv(N, 256));
  const int64_t tiles = static_cast<int64_t>(a.ntm) * a.ntn;
  GPTQ_REQUIRE(tiles < (int64_t(1) << 28), GPTQ_ERR_SHAPE, "matmul_nt: too many tiles");
  const int rest = static_cast<int>(tiles % 256);
  a.full = static_cast<int>(rest <= 128 ? tiles - rest : tiles);
  const dim3 grid(static_cast<unsigned>(a.full + 2 * (tiles - a.full)));
  hipStream_t st = as_hip(stream);
  if (bplanes > 1 && out_dtype == GPTQ_BF16)
    hipLaunchKernelGGL((dense_nt_k<true, true, true>), grid, dim3(256), 0, st, a);
  else if (bplanes > 1)
    hipLaunchKernelGGL((dense_nt_k<true, false, true>), grid, dim3(256), 0, st, a);
  else if (dtype == GPTQ_BF16)
    hipLaunchKernelGGL((dense_nt_k<true, true, false>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((dense_nt_k<false, false, false>), grid, dim3(256), 0, st, a);
  return check_launch("matmul_nt");
}

extern "C" int gptq_split_planes(const void* x, int64_t M, int64_t N, void* out, gptq_stream_t stream) {
  clear_error();
  GPTQ_REQUIRE(x && out, GPTQ_ERR_ARG, "split_planes: null pointer");
  GPTQ_REQUIRE(M > 0 && N > 0 && N % 8 == 0, GPTQ_ERR_SHAPE, "split_planes: bad shape");
  GPTQ_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0, GPTQ_ERR_ARG,
               "split_planes: operands must be 16-byte aligned");
  const int64_t blocks = std::min<int64_t>(cdiv(M * (N / 8), 256), 8192);
  hipLaunchKernelGGL(split_fp16_k, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, as_hip(stream),
                     static_cast<const uint16_t*>(x), N / 8, M, N, static_cast<uint16_t*>(out));
  return check_launch("split_planes");
}
