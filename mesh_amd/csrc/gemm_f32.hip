// Grouped float32 products on the bf16 matrix cores of gfx950:
//   C[e] = act(A[e] . B[e]^T),  or A[e]^T . B[e] (weight gradients)
// (the float32 configuration of layers.dense_product / layers.dense in
// mesh_tensorflow/transformer/moe.py:469-486 and of their gradients).
#include <type_traits>
#include <utility>

#include "common.h"

namespace mesh_moe {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// ---------------------------------------------------------------------------
// Every float32 is the sum of three bf16 terms, x = x1 + x2 + x3: x1 is x
// rounded to bf16, x2 the remainder rounded, and what is left then has at most
// 8 significant bits, which bf16 holds exactly down to 2^-133, the last bit of its
// denormals.  A product a b is then the sum of nine exact products, of which
// a2 b3, a3 b2 and a3 b3, together at most 2^-24 |a b| (2^-28 on average), are left
// out; the other six run on v_mfma_f32_16x16x32_bf16, which adds exact products into float32: 96 cycles
// of the matrix pipe for 16 x 16 outputs and k = 32 instead of 256 of
// v_mfma_f32_32x32x2_f32.  The six are summed by themselves, small ones first, and
// added to the accumulator once per 32 k, which rounds a sixteenth as often as
// those did.  Error against float64 (relative 2-norm; before, with float32 MFMAs,
// in brackets): K = 512 0.9e-7 (4.1e-7), 2048 1.3e-7 (4.1e-7), 3072 1.9e-7 (9.9e-7),
// weight gradients from 320 rows 0.75e-7 (3.2e-7), 16000 rows 2.5e-7 (11e-7).
//
// Measured (us, float32 MFMAs -> here): 8 experts x 320 rows, 512 -> 2048 64 -> 39,
// 2048 -> 512 66 -> 42, their weight gradients 54 -> 34; 4096 x 4096, K = 1024 303
// -> 174 (1.18 PFLOP/s of bf16 products, what a large product reaches here); 64 x
// 160 rows, 512 -> 2048 241 -> 132; 33 rows x 128, K = 4096, 32 experts 50 -> 28.
// Bound by the bf16 matrix pipes (and the power cap) in large launches; in small
// ones by the latency of a block's first loads and of its last stores, and by
// making terms, 12 vector instructions per pair of values, which run beside the
// MFMAs.  What stays behind is reductions of few K tiles (K = 200 and 260: 8.4 ->
// 9.0 and 6.8 -> 7.3).
//
// A sum with an infinity, a NaN or an overflow in it is not what the terms give
// (inf - inf, inf * 0).  Whatever such an operand touches comes out as an
// infinity or a NaN.  A block that finds one among its sums makes its tile again on
// v_mfma_f32_16x16x4_f32, operands straight from memory.  So does one with an operand
// whose third term is not whole (a value below 2^-110), which one more instruction per
// pair of values finds out (1 % of a launch).  8 x 1024 rows, K = 2048, 512 columns:
// 113 us, 440 with NaN everywhere; weight gradients of these sizes 129 and 313.  (A
// chain of multiply-adds per element took 15400 and 16600.)
//
// TM x TN MFMA tiles per wavefront; WN wavefronts along N times WK wavefronts
// that share out the k of every K tile and add up their sums in the end.  All
// wavefronts of a block work on the same 16 TM rows of A: their terms are made
// once, on the way from registers into LDS ([3][rows][BK] bf16, rows padded by 16
// bytes so that fragment reads and writes spread over all banks).  A
// wavefront's 16 TN columns of B belong to it and its WK partners alone: its
// lanes load them straight from memory in operand layout and make the terms in
// registers.  Both operands of K tile t + 2 are on their way in registers, and
// the terms of tile t + 1 are made beside the MFMAs of tile t.
//
// k is taken in an order of its own, the same for both operands: 16-byte piece
// p of a group of 32 k holds k = 4 p .. 4 p + 3 and 16 + 4 p .. 16 + 4 p + 3, so
// that the loads of a row are 64 bytes wide.
//
// KMAJOR: the reduction index is the outermost one of both operands (A [K][R],
// B [K][N], token rows summed over); a lane's 8 k of a column are 8 loads, each
// contiguous over the wavefront.
// ---------------------------------------------------------------------------
template <int TM_, int TN_, int WN_, int WK_>
struct SplitCfg {
  static constexpr int TM = TM_, TN = TN_, WN = WN_, WK = WK_;
  static constexpr int THREADS = 64 * WN * WK;
  static constexpr int BM = 16 * TM, BN = 16 * TN * WN;
  static constexpr int BK = WK > 1 ? 32 * WK : 32;
  static constexpr int LDR = BK + 8;           // bf16 per LDS row
  static constexpr int PLANE = BM * LDR;       // one term of the A tile
  static constexpr int STAGE = 3 * PLANE;
  static constexpr int CHUNKS = BK / 8;        // 16-byte pieces per row
  static constexpr int A_PIECES = BM * CHUNKS;
  // per thread; where they do not come out even, some pieces are done twice
  static constexpr int A_CHUNKS = (A_PIECES + THREADS - 1) / THREADS;
  static constexpr int KS = BK / 32 / WK;      // MFMA steps of a wavefront
  static constexpr size_t LOOP_BYTES = 2ull * STAGE * sizeof(bf16_t);
  static constexpr size_t SUM_BYTES =
      (size_t)(WK - 1) * WN * TM * TN * 256 * sizeof(float);
  static constexpr size_t LDS_BYTES =
      LOOP_BYTES > SUM_BYTES ? LOOP_BYTES : SUM_BYTES;
};

template <typename F, int... I>
__device__ __forceinline__ void for_each_index(
    F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
// f(0), ..., f(COUNT - 1) with constant arguments
template <int COUNT, typename F>
__device__ __forceinline__ void for_each_index(F f) {
  for_each_index(f, std::make_integer_sequence<int, COUNT>());
}

// The three terms of two values, a's in the low halves.  `lost` collects the third
// terms' bits: they are whole if its low half stays 0.  (The remainders by
// v_dot2c_f32_bf16 would be one instruction each instead of two, but it waits for
// the matrix pipe: 8 of them and 2 MFMAs take as long as both by themselves.)
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&t)[3],
                                           uint32_t& lost) {
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    t[n] = f32x2_to_bf16x2(a, b);
    if (n == 2) {
      // (in C++ the compiler collects the values of many pairs before it ors them)
      asm("v_or3_b32 %0, %0, %1, %2" : "+v"(lost) : "v"(a), "v"(b));
      break;
    }
    a = a - __uint_as_float(t[n] << 16);            // exact
    b = b - __uint_as_float(t[n] & 0xffff0000u);
  }
}
// the terms of 8 values as MFMA operands
__device__ __forceinline__ void split_terms(const float (&f)[8], uint4 (&t)[3],
                                            uint32_t& lost) {
  uint32_t w[4][3];
#pragma unroll
  for (int p = 0; p < 4; ++p) split_pair(f[2 * p], f[2 * p + 1], w[p], lost);
#pragma unroll
  for (int n = 0; n < 3; ++n)
    t[n] = make_uint4(w[0][n], w[1][n], w[2][n], w[3][n]);
}

// mask_src (shape of C): elements whose mask_src element is not positive become
// 0, the others are multiplied by mask_scale.
__device__ __forceinline__ float finish_f32(float v, bool relu, bool masked,
                                            float m, float mask_scale) {
  if (relu) v = fmaxf(v, 0.f);
  if (masked) v = m > 0.f ? v * mask_scale : 0.f;
  return v;
}

// The sums of TM x TN MFMA tiles from (row0, col0) on, straight from the operands of an
// expert, on float32 MFMAs; the wavefronts wk of WK share k.  Any sizes.
template <int TM, int TN, int WK, bool KMAJOR>
__device__ __forceinline__ void sums_from_operands(
    const float* __restrict__ Ae, const float* __restrict__ Be, int R, int N, int K,
    int row0, int col0, int wk, f32x4_t (&acc)[TM][TN]) {
  const int lane = threadIdx.x & 63;
  // two MFMAs of 4 k at a time, which the wavefronts that share k take in turn: the
  // q-th has k = 8 g + 2 (lane / 16) + q, with KMAJOR 8 g + 4 q + lane / 16
  constexpr int NQ = 2;
  const int groups = (K + 7) / 8;
  int64_t a_at[TM], b_at[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
    a_at[i] = (int64_t)min(row0 + i * 16 + (lane & 15), R - 1) * (KMAJOR ? 1 : K);
#pragma unroll
  for (int j = 0; j < TN; ++j)
    b_at[j] = (int64_t)min(col0 + j * 16 + (lane & 15), N - 1) * (KMAJOR ? 1 : K);
  float fa[TM][NQ], fb[TN][NQ];
  // (past the end of k: zeros in both operands)
  auto load = [&](int g) {
    if constexpr (KMAJOR) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int k = 8 * g + 4 * q + (lane >> 4);
        const int64_t kk = min(k, K - 1);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const float v = Ae[kk * R + a_at[i]];
          fa[i][q] = k < K ? v : 0.f;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const float v = Be[kk * N + b_at[j]];
          fb[j][q] = k < K ? v : 0.f;
        }
      }
    } else {
      const int k = 8 * g + 2 * (lane >> 4), kk = min(k, K - 2);
      auto load2 = [&](const float* p, float (&f)[NQ]) {
        const float2 v = *reinterpret_cast<const float2*>(p);
        f[0] = k < K ? v.x : 0.f;
        f[1] = k < K ? v.y : 0.f;
      };
#pragma unroll
      for (int i = 0; i < TM; ++i) load2(Ae + a_at[i] + kk, fa[i]);
#pragma unroll
      for (int j = 0; j < TN; ++j) load2(Be + b_at[j] + kk, fb[j]);
    }
  };
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
  load(wk);
  for (int g = wk; g < groups; g += WK) {
    float ca[TM][NQ], cb[TN][NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
#pragma unroll
      for (int i = 0; i < TM; ++i) ca[i][q] = fa[i][q];
#pragma unroll
      for (int j = 0; j < TN; ++j) cb[j][q] = fb[j][q];
    }
    load(g + WK);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(cb[j][q], ca[i][q],
                                                           acc[i][j], 0, 0, 0);
  }
}

template <int TM, int TN, int WN, int WK, int RAW, bool KMAJOR>
__global__ __launch_bounds__(64 * WN * WK) void grouped_gemm_f32_split_kernel(
    const float* __restrict__ A, const float* __restrict__ B,
    float* __restrict__ Cout, int R, int N, int K, int tiles_m, int tiles_n,
    int relu, const float* __restrict__ mask_src, float mask_scale) {
  using Cfg = SplitCfg<TM, TN, WN, WK>;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, LDR = Cfg::LDR;
  constexpr int KS = Cfg::KS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  bf16_t* As = reinterpret_cast<bf16_t*>(smem_raw);   // [2][3][BM][LDR]
  __shared__ int again;           // the sums are made again
  if (threadIdx.x == 0) again = 0;
  // an XCD works on a contiguous range of tiles, which share weight panels
  const int nblk = gridDim.x;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int logical = xcd * (nblk >> 3) + min(xcd, nblk & 7) + local;
  const int tiles_per_e = tiles_m * tiles_n;
  const int e = logical / tiles_per_e;
  const int rem = logical - e * tiles_per_e;
  const int tn = rem / tiles_m, tm = rem - tn * tiles_m;
  const int row0 = tm * BM, col0 = tn * BN;
  const float* Ae = A + (int64_t)e * R * K;
  const float* Be = B + (int64_t)e * N * K;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wk = wave / WN, wn = wave % WN;

  // Where this thread's loads lie relative to the K tile's corner (element
  // (row0, k0) of A, (col0, k0) of B), in bytes.  Rows past the end are read as
  // the last one and not stored.
  auto k_of_piece = [](int c) { return (c >> 2) * 32 + (c & 3) * 4; };
  uint32_t a_off[Cfg::A_CHUNKS], b_off[KS][TN];
  int a_lds[Cfg::A_CHUNKS], a_k[Cfg::A_CHUNKS], b_k[KS];
#pragma unroll
  for (int i = 0; i < Cfg::A_CHUNKS; ++i) {
    const int c = (tid + i * Cfg::THREADS) % Cfg::A_PIECES;
    const int r = KMAJOR ? c % BM : c / Cfg::CHUNKS;
    const int piece = KMAJOR ? c / BM : c % Cfg::CHUNKS;
    const uint32_t row = min(row0 + r, R - 1) - row0;
    a_k[i] = k_of_piece(piece);
    a_off[i] = 4u * (KMAJOR ? (uint32_t)a_k[i] * R + row : row * K + a_k[i]);
    a_lds[i] = r * LDR + piece * 8;
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    b_k[s] = k_of_piece((wk * KS + s) * 4 + (lane >> 4));
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int c = (wn * TN + j) * 16 + (lane & 15);
      const uint32_t col = min(col0 + c, N - 1) - col0;
      b_off[s][j] = 4u * (KMAJOR ? (uint32_t)b_k[s] * N + col : col * K + b_k[s]);
    }
  }
  // 8 values of one row: k .. k + 3 and k + 16 .. k + 19 from `at` on
  auto load8 = [&](const float* corner, uint32_t off, int rows, float (&f)[8]) {
    const char* p = reinterpret_cast<const char*>(corner);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (KMAJOR) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          f[4 * h + q] = *reinterpret_cast<const float*>(
              p + (int64_t)(16 * h + q) * rows * 4 + off);
      } else {
        const float4 v = *reinterpret_cast<const float4*>(p + 64 * h + off);
        f[4 * h] = v.x; f[4 * h + 1] = v.y; f[4 * h + 2] = v.z; f[4 * h + 3] = v.w;
      }
    }
  };
  const float* a_corner = Ae + (KMAJOR ? (int64_t)row0 : (int64_t)row0 * K);
  const float* b_corner = Be + (KMAJOR ? (int64_t)col0 : (int64_t)col0 * K);
  const int nk = K / BK;          // whole K tiles, at least one
  // first k of K tile kt; past the whole tiles, the last BK of k
  auto k_first = [&](int kt) { return (int64_t)min(kt * BK, K - BK); };
  float a_raw[RAW][Cfg::A_CHUNKS][8], b_raw[RAW][KS][TN][8];
  auto load_tile = [&](int kt, auto slot_c) {
    constexpr int SLOT = decltype(slot_c)::value;
    const int64_t k0 = k_first(kt);
    const float* ac = a_corner + (KMAJOR ? k0 * R : k0);
    const float* bc = b_corner + (KMAJOR ? k0 * N : k0);
#pragma unroll
    for (int i = 0; i < Cfg::A_CHUNKS; ++i)
      load8(ac, a_off[i], R, a_raw[SLOT % RAW][i]);
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < TN; ++j) load8(bc, b_off[s][j], N, b_raw[SLOT % RAW][s][j]);
  };
  uint4 b_terms[2][KS][TN][3];
  uint32_t lost = 0;
  // the terms of a loaded tile: A's into stage `slot`, B's into registers
  auto make_terms = [&](auto slot_c) {
    constexpr int SLOT = decltype(slot_c)::value;
#pragma unroll
    for (int i = 0; i < Cfg::A_CHUNKS; ++i) {
      uint4 t[3];
      split_terms(a_raw[SLOT % RAW][i], t, lost);
#pragma unroll
      for (int n = 0; n < 3; ++n)
        *reinterpret_cast<uint4*>(As + SLOT * Cfg::STAGE + n * Cfg::PLANE +
                                  a_lds[i]) = t[n];
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        split_terms(b_raw[SLOT % RAW][s][j], b_terms[SLOT][s][j], lost);
  };

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
  // The products of the K tile in stage / registers SLOT.  With NEXT, the terms of
  // the other slot's loaded tile are made on the way, a pair of values at a time
  // between the MFMAs, and each piece's registers are loaded again with tile
  // `ahead`.
  auto products = [&](auto slot_c, auto next_c, int ahead) {
    constexpr int SLOT = decltype(slot_c)::value, OTHER = SLOT ^ 1;
    constexpr bool NEXT = decltype(next_c)::value;
    // (the small products first)
    constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};
    constexpr int MFMAS = 6 * TM * TN * KS;
    constexpr int GROUPS = Cfg::A_CHUNKS + KS * TN, PAIRS = 4 * GROUPS;
    const int64_t k0 = k_first(ahead);
    const float* ac = a_corner + (KMAJOR ? k0 * R : k0);
    const float* bc = b_corner + (KMAJOR ? k0 * N : k0);
    const bf16_t* src = As + SLOT * Cfg::STAGE + (lane & 15) * LDR +
                        (wk * KS * 4 + (lane >> 4)) * 8;
    // the terms of row tile at % TM in MFMA step at / TM
    bf16x8_t af[2][3];
    auto read = [&](int at) {
#pragma unroll
      for (int n = 0; n < 3; ++n)
        af[at & 1][n] = *reinterpret_cast<const bf16x8_t*>(
            src + n * Cfg::PLANE + at % TM * 16 * LDR + at / TM * 32);
    };
    uint32_t w[3][4];
    auto work = [&](auto at_c) {
      constexpr int g = decltype(at_c)::value >> 2, p = decltype(at_c)::value & 3;
      constexpr bool of_a = g < Cfg::A_CHUNKS;
      constexpr int ga = of_a ? g : 0, gb = of_a ? 0 : g - Cfg::A_CHUNKS;
      constexpr int s = gb / TN, j = gb % TN;
      float(&raw)[8] = of_a ? a_raw[OTHER % RAW][ga] : b_raw[OTHER % RAW][s][j];
      uint32_t t[3];
      split_pair(raw[2 * p], raw[2 * p + 1], t, lost);
#pragma unroll
      for (int n = 0; n < 3; ++n) w[n][p] = t[n];
      if constexpr (p == 3) {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
          const uint4 v = make_uint4(w[n][0], w[n][1], w[n][2], w[n][3]);
          if constexpr (of_a)
            *reinterpret_cast<uint4*>(As + OTHER * Cfg::STAGE + n * Cfg::PLANE +
                                      a_lds[ga]) = v;
          else
            b_terms[OTHER][s][j][n] = v;
        }
        if constexpr (of_a) load8(ac, a_off[ga], R, raw);
        else load8(bc, b_off[s][j], N, raw);
      }
    };
    // the products of 32 k, added to the accumulators while the next row tile's
    // are on their way
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t sum[2][TN];
    auto add = [&](int at, int j) { acc[at % TM][j] += sum[at & 1][j]; };
    read(0);
    for_each_index<MFMAS>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value;
      constexpr int j = m % TN, p = m / TN % 6, at = m / (TN * 6), i = at % TM,
                    s = at / TM;
      constexpr int ta = TA[p], tb = TB[p];
      if constexpr (m % (TN * 6) == 0 && at + 1 < TM * KS) read(at + 1);
      sum[at & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8_t, b_terms[SLOT][s][j][tb]), af[at & 1][ta],
          p == 0 ? zero : sum[at & 1][j], 0, 0, 0);
      if constexpr (at > 0 && p == 1) add(at - 1, j);
      if constexpr (NEXT) {
        constexpr int from = PAIRS * m / MFMAS, to = PAIRS * (m + 1) / MFMAS;
        for_each_index<to - from>([&](auto at_c) {
          work(std::integral_constant<int, from + decltype(at_c)::value>());
        });
        __builtin_amdgcn_sched_barrier(0);
      }
    });
#pragma unroll
    for (int j = 0; j < TN; ++j) add(TM * KS - 1, j);
  };
  // LDS writes and reads of every wavefront are done; loads stay in flight
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  load_tile(0, S0());
  if constexpr (RAW == 2) load_tile(1, S1());
  make_terms(S0());
  load_tile(RAW, S0());
  barrier();
  // (the stage written here was read in the step before, whose readers have
  // passed the barrier at its end; past the end it is written for nobody)
  for (int kt = 0; kt + 1 < nk; kt += 2) {
    products(S0(), std::true_type(), kt + 1 + RAW);
    barrier();
    products(S1(), std::true_type(), kt + 2 + RAW);
    barrier();
  }
  if (nk & 1) {
    products(S0(), std::false_type(), 0);
    barrier();
  }
  if (nk * BK < K) {
    // the last BK of k are in the raw registers: the whole tiles' share of them
    // becomes zeros in A
    const int old = (nk + 1) * BK - K;
#pragma unroll
    for (int i = 0; i < Cfg::A_CHUNKS; ++i)
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (a_k[i] + (q >> 2) * 16 + (q & 3) < old) a_raw[0][i][q] = 0.f;
    make_terms(S0());
    barrier();
    products(S0(), std::false_type(), 0);
    barrier();
  }
  // 0 x is 0 only for finite x
  float test[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        test[r] = __builtin_fmaf(acc[i][j][r], 0.f, test[r]);
  if (!(test[0] + test[1] + test[2] + test[3] == 0.f) || (lost & 0xffffu) != 0)
    again = 1;
  auto sums_again = [&]() {
    sums_from_operands<TM, TN, WK, KMAJOR>(Ae, Be, R, N, K, row0,
                                           col0 + wn * TN * 16, wk, acc);
  };
  if constexpr (WK == 1) {
    __syncthreads();
    if (again) sums_again();
  } else {
    // [wk - 1][wn][TM][TN][4][64], where the stages were
    float* parts = reinterpret_cast<float*>(smem_raw);
    constexpr int SUB = TM * TN * 256, PART = WN * SUB;
    auto store_part = [&]() {
      if (wk == 0) return;
      float* dst = parts + (wk - 1) * PART + wn * SUB + lane;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            dst[((i * TN + j) * 4 + r) * 64] = acc[i][j][r];
    };
    store_part();
    __syncthreads();
    if (again) {
      sums_again();
      store_part();
      __syncthreads();
    }
    if (wk > 0) return;
#pragma unroll
    for (int w = 0; w < WK - 1; ++w) {
      const float* src = parts + w * PART + wn * SUB + lane;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[i][j][r] += src[((i * TN + j) * 4 + r) * 64];
    }
  }
  float* Ce = Cout + (int64_t)e * R * N;
  const float* mask = mask_src == nullptr ? nullptr : mask_src + (int64_t)e * R * N;
  const int col_w = col0 + wn * TN * 16;
  const int m_l = lane & 15, n_l = (lane >> 4) * 4;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int grow = row0 + i * 16 + m_l, gcol = col_w + j * 16 + n_l;
      if (grow < R && gcol < N) {
        const int64_t c = (int64_t)grow * N + gcol;
        const float4 m = mask == nullptr
                             ? make_float4(1.f, 1.f, 1.f, 1.f)
                             : *reinterpret_cast<const float4*>(mask + c);
        const bool masked = mask != nullptr;
        *reinterpret_cast<float4*>(Ce + c) = make_float4(
            finish_f32(acc[i][j][0], relu, masked, m.x, mask_scale),
            finish_f32(acc[i][j][1], relu, masked, m.y, mask_scale),
            finish_f32(acc[i][j][2], relu, masked, m.z, mask_scale),
            finish_f32(acc[i][j][3], relu, masked, m.w, mask_scale));
      }
    }
}

template <int TM, int TN, int WN, int WK, int RAW>
static int launch_split(const float* A, const float* B, float* C, int E, int R,
                        int N, int K, bool kmajor, bool relu,
                        const float* mask_src, float mask_scale, hipStream_t st) {
  using Cfg = SplitCfg<TM, TN, WN, WK>;
  const int tiles_m = (R + Cfg::BM - 1) / Cfg::BM;
  const int tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  const int64_t blocks = (int64_t)tiles_m * tiles_n * E;
  MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: too many tiles (%lld)", (long long)blocks);
  auto k = kmajor ? grouped_gemm_f32_split_kernel<TM, TN, WN, WK, RAW, true>
                  : grouped_gemm_f32_split_kernel<TM, TN, WN, WK, RAW, false>;
  MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
  k<<<(unsigned)blocks, Cfg::THREADS, Cfg::LDS_BYTES, st>>>(
      A, B, C, R, N, K, tiles_m, tiles_n, relu ? 1 : 0, mask_src, mask_scale);
  MOE_CHECK_LAUNCH("expert_ffn (float32 in bf16 terms)");
  return 0;
}

// Block tiles and what a launch of one costs: a + n b us for n = blocks per
// compute unit (rounded up), plus (c + n d) us per K tile.  Fitted to 38 products
// of 1 to 64 experts, 33 to 8192 rows, K 36 to 16000, both layouts, each with
// every tile (root mean square of the deviations 6 to 10 %, 18 % for the smallest
// tile); the tile the fit picks is 0.6 % slower than the best one on average and 10 %
// at worst.  Large tiles spend less on making terms (each value of A once per
// column tile, of B once per row tile), small ones waste less on rows that do not
// fill a tile and on the last round; the wavefronts of the small ones share out
// k, so that every SIMD has work.
struct SplitTile {
  int rows, cols, k;
  decltype(&launch_split<8, 2, 8, 1, 1>) launch;
  double a, b, c, d;
};
template <int TM, int TN, int WN, int WK, int RAW>
static constexpr SplitTile split_tile(double a, double b, double c, double d) {
  using Cfg = SplitCfg<TM, TN, WN, WK>;
  return {Cfg::BM, Cfg::BN, Cfg::BK, launch_split<TM, TN, WN, WK, RAW>, a, b, c, d};
}
static const SplitTile split_tiles[] = {
    split_tile<8, 2, 8, 1, 1>(0.0, 5.93, 0.0, 2.08),     // 128 x 256
    split_tile<10, 2, 8, 1, 1>(0.0, 6.23, 0.0, 2.76),    // 160 x 256
    split_tile<10, 2, 4, 2, 1>(0.33, 7.41, 0.0, 2.98),   // 160 x 128
    split_tile<4, 2, 4, 2, 1>(1.71, 3.89, 0.0, 1.39),    // 64 x 128
    split_tile<5, 2, 2, 4, 1>(1.27, 5.19, 0.0, 2.01),    // 80 x 64
    split_tile<6, 2, 2, 4, 1>(0.86, 5.74, 0.0, 2.18),    // 96 x 64
    split_tile<2, 2, 1, 8, 1>(1.71, 3.12, 0.10, 1.36),   // 32 x 32
    split_tile<1, 2, 1, 4, 2>(4.10, 0.34, 0.0, 0.59),    // 16 x 32
    split_tile<2, 2, 2, 2, 1>(3.39, 0.52, 0.13, 0.58),   // 32 x 64
    split_tile<6, 2, 8, 1, 1>(0.0, 5.35, 0.0, 1.75),     // 96 x 256
    split_tile<4, 2, 8, 1, 1>(0.0, 4.97, 0.0, 1.35),     // 64 x 256
    split_tile<4, 2, 4, 1, 1>(1.85, 2.07, 0.26, 0.68),   // 64 x 128, K tiles of 32
    split_tile<1, 2, 4, 1, 2>(2.90, 0.50, 0.13, 0.48)};  // 16 x 128

// The offsets of a tile's loads are 32 bits: of its rows' k, or (kmajor) of its k's
// rows, the last of which lies 20 below the K tile's end.
static bool split_tile_fits(const SplitTile& t, int R, int N, int K, bool kmajor) {
  const int64_t most = 1LL << 30;
  return kmajor ? (int64_t)(t.k - 20) * (R > N ? R : N) + 256 <= most
                : (int64_t)(t.rows > t.cols ? t.rows : t.cols) * K <= most;
}

// Weight gradients of rows too long for that (from 89 million elements on): a
// wavefront per 32 x 32 outputs, bound by memory.
__global__ __launch_bounds__(64) void f32_long_rows_kernel(
    const float* __restrict__ A, const float* __restrict__ B,
    float* __restrict__ Cout, int R, int N, int K, int tiles_m) {
  const int tm = blockIdx.x % tiles_m, tn = blockIdx.x / tiles_m, e = blockIdx.y;
  f32x4_t acc[2][2];
  sums_from_operands<2, 2, 1, true>(A + (int64_t)e * R * K, B + (int64_t)e * N * K,
                                    R, N, K, tm * 32, tn * 32, 0, acc);
  const int lane = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = tm * 32 + i * 16 + (lane & 15);
      const int col = tn * 32 + j * 16 + (lane >> 4) * 4;
      if (row < R && col < N)
        *reinterpret_cast<f32x4_t*>(Cout + ((int64_t)e * R + row) * N + col) =
            acc[i][j];
    }
}

bool f32_gemm_applies(int R, int N, int K) {
  const int most = 0x7fffffff - 1024;    // (room for the indexes of a last tile)
  return R >= 32 && N >= 32 && K >= 32 && R <= most && N <= most && K <= most;
}

int f32_gemm(const float* A, const float* B, float* C, int E, int R, int N, int K,
             bool kmajor, bool relu, const float* mask_src, float mask_scale,
             hipStream_t st) {
  const int cus = compute_units();
  if (cus == 0) return MESH_MOE_E_HIP;
  const SplitTile* best = nullptr;
  double best_cost = 0;
  for (const SplitTile& t : split_tiles) {
    if (t.k > K || !split_tile_fits(t, R, N, K, kmajor)) continue;
    const int64_t blocks = (int64_t)E * ((R + t.rows - 1) / t.rows) *
                           ((N + t.cols - 1) / t.cols);
    const double n = (double)((blocks + cus - 1) / cus);
    const double cost =
        t.a + n * t.b + (double)((K + t.k - 1) / t.k) * (t.c + n * t.d);
    if (best == nullptr || cost < best_cost) {
      best = &t;
      best_cost = cost;
    }
  }
  if (best != nullptr)
    return best->launch(A, B, C, E, R, N, K, kmajor, relu, mask_src, mask_scale, st);
  if (!kmajor)
    return f32_gemm_stable(A, B, C, E, R, N, K, relu, mask_src, mask_scale, st);
  const int64_t tiles_m = ((int64_t)R + 31) / 32, tiles_n = ((int64_t)N + 31) / 32;
  MOE_REQUIRE(!relu && mask_src == nullptr, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: no activation on sums of rows");
  MOE_REQUIRE(tiles_m * tiles_n <= 0x7fffffffLL && E <= 65535,
              MESH_MOE_E_UNSUPPORTED, "expert_ffn: too many tiles (%lld)",
              (long long)(tiles_m * tiles_n));
  f32_long_rows_kernel<<<dim3((unsigned)(tiles_m * tiles_n), (unsigned)E), 64, 0,
                         st>>>(A, B, C, R, N, K, (int)tiles_m);
  MOE_CHECK_LAUNCH("expert_ffn (float32, long rows)");
  return 0;
}

// ---------------------------------------------------------------------------
// Few rows per expert (fewer than 32), C[e] = act(A[e] . B[e]^T): small batches, whose
// time is that of reading the weights.  A wavefront takes all rows and 16 TN columns and
// walks k by itself on v_mfma_f32_16x16x4_f32, whose sums are a chain of multiply-adds in
// ascending k: the bits of grouped_gemm_simple_kernel, which had these products on 64 x
// 64 tiles of plain multiply-adds.  (So a hidden tensor that is kept for a gradient has
// one set of sums, see below.)  A lane loads 16 bytes, four consecutive k of its row; an
// MFMA wants one k of each lane group, so the four registers and the four groups change
// places (v_permlane32_swap, v_permlane16_swap).  DEPTH groups of 16 k are on their way.
// A layer of 85 tokens, 8 experts, 832 -> 1664 -> 832 (21 rows each) 364 -> 89 us, of
// which the two products are 18 and 32; 407 tokens, 48 experts, 640 -> 2560, a training
// step 1558 -> 587, its four products 82 to 123 us for 315 MB of weights each.  What is
// left to the read rate is rows of one stride that all wavefronts walk in step (another
// first k per wavefront would be another order of the sums).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void swap_groups(float (&v)[4]) {
  auto swap32 = [](float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b),
                                                    false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  };
  auto swap16 = [](float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b),
                                                    false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  };
  swap32(v[0], v[2]);
  swap32(v[1], v[3]);
  swap16(v[0], v[1]);
  swap16(v[2], v[3]);
}

template <int RT, int TN>
__global__ __launch_bounds__(256) void f32_few_rows_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ Cout,
    int R, int N, int K, int col_blocks, int relu, const float* __restrict__ mask_src,
    float mask_scale) {
  constexpr int DEPTH = RT + TN == 2 ? 10 : RT + TN == 3 ? 8 : 6;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = blockIdx.x / col_blocks;
  const int col0 = ((blockIdx.x - e * col_blocks) * 4 + wave) * 16 * TN;
  if (col0 >= N) return;
  const int c = lane & 15, g = lane >> 4;
  // (rows and columns past the end are read as the last one and not stored)
  const float *a_row[RT], *b_row[TN];
#pragma unroll
  for (int i = 0; i < RT; ++i)
    a_row[i] = A + ((int64_t)e * R + min(16 * i + c, R - 1)) * K;
#pragma unroll
  for (int j = 0; j < TN; ++j)
    b_row[j] = B + ((int64_t)e * N + min(col0 + 16 * j + c, N - 1)) * K;
  f32x4_t a_raw[DEPTH][RT], b_raw[DEPTH][TN];
  auto load = [&](int chunk, auto slot_c) {
    constexpr int SLOT = decltype(slot_c)::value;
    const int k = min(16 * chunk + 4 * g, K - 4);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      b_raw[SLOT][j] = *reinterpret_cast<const f32x4_t*>(b_row[j] + k);
#pragma unroll
    for (int i = 0; i < RT; ++i)
      a_raw[SLOT][i] = *reinterpret_cast<const f32x4_t*>(a_row[i] + k);
  };
  f32x4_t acc[RT][TN];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
  auto multiply = [&](int chunk, auto slot_c, auto whole_c) {
    constexpr int SLOT = decltype(slot_c)::value;
    constexpr bool WHOLE = decltype(whole_c)::value;
    float a[RT][4], b[TN][4];
    const bool mine = 16 * chunk + 4 * g < K;
    auto take = [&](f32x4_t v, float (&to)[4]) {
      // (the four values stay together till here: taken apart where they are loaded,
      // the compiler waits for them there)
      asm volatile("" : "+v"(v));
      to[0] = v[0]; to[1] = v[1]; to[2] = v[2]; to[3] = v[3];
      if constexpr (!WHOLE)
#pragma unroll
        for (int q = 0; q < 4; ++q) to[q] = mine ? to[q] : 0.f;
      swap_groups(to);
    };
#pragma unroll
    for (int i = 0; i < RT; ++i) take(a_raw[SLOT][i], a[i]);
#pragma unroll
    for (int j = 0; j < TN; ++j) take(b_raw[SLOT][j], b[j]);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][q], a[i][q], acc[i][j],
                                                           0, 0, 0);
  };
  // (a branch between the loads would wait for all of them)
  const int chunks = (K + 15) / 16;
  int first = 0;
  for_each_index<DEPTH>([&](auto u) { load(decltype(u)::value, u); });
  for (; first + DEPTH <= K / 16; first += DEPTH)
    for_each_index<DEPTH>([&](auto u) {
      const int chunk = first + decltype(u)::value;
      multiply(chunk, u, std::true_type());
      load(chunk + DEPTH, u);
      __builtin_amdgcn_sched_barrier(0);
    });
  for_each_index<DEPTH>([&](auto u) {
    const int chunk = first + decltype(u)::value;
    if (chunk < chunks) multiply(chunk, u, std::false_type());
  });
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row = 16 * i + c, col = col0 + 16 * j + 4 * g;
      if (row >= R || col >= N) continue;
      const int64_t at = ((int64_t)e * R + row) * N + col;
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = acc[i][j][q];
        if (relu) v[q] = v[q] > 0.f ? v[q] : 0.f;
      }
      if (mask_src != nullptr) {
        const float4 m = *reinterpret_cast<const float4*>(mask_src + at);
        const float mv[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[q] = finish_f32(v[q], false, true, mv[q], mask_scale);
      }
      *reinterpret_cast<float4*>(Cout + at) = make_float4(v[0], v[1], v[2], v[3]);
    }
}

bool f32_few_rows_applies(int R, int N, int K) {
  return R >= 1 && R < 32 && N >= 16 && K >= 16 && N % 4 == 0 && K % 4 == 0;
}

int f32_few_rows(const float* A, const float* B, float* C, int E, int R, int N, int K,
                 bool relu, const float* mask_src, float mask_scale, hipStream_t st) {
  const int cus = compute_units();
  if (cus == 0) return MESH_MOE_E_HIP;
  // two column tiles per wavefront, which share the rows' loads, once every SIMD has two
  // wavefronts anyway
  const bool two = (int64_t)E * ((N + 15) / 16) >= (int64_t)16 * cus;
  const int col_blocks = (N + (two ? 127 : 63)) / (two ? 128 : 64);
  const int64_t blocks = (int64_t)E * col_blocks;
  MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: too many tiles (%lld)", (long long)blocks);
  auto run = [&](auto k) {
    k<<<(unsigned)blocks, 256, 0, st>>>(A, B, C, R, N, K, col_blocks, relu ? 1 : 0,
                                        mask_src, mask_scale);
    MOE_CHECK_LAUNCH("expert_ffn (float32, few rows)");
    return 0;
  };
  if (R <= 16) return two ? run(f32_few_rows_kernel<1, 2>) : run(f32_few_rows_kernel<1, 1>);
  return two ? run(f32_few_rows_kernel<2, 2>) : run(f32_few_rows_kernel<2, 1>);
}

// Their weight gradients, C[e] = A[e]^T . B[e] over fewer than 32 rows (A [K][R], B
// [K][N]): bound by the stores.  A wavefront makes 64 x 64 outputs from one load of 16
// bytes per operand and four rows; the register of a load picks the column, so that a
// lane ends up with four consecutive outputs and a store is four whole rows of 256 bytes.
// The sums are chains of multiply-adds over 16 or 32 rows (zeros behind the last one):
// the bits of grouped_gemm_simple_kernel on transposed copies, which these were before.
// 48 experts, 10 rows, 640 x 2560: 65 us, 4.8 TB/s.
template <int KS>
__global__ __launch_bounds__(256) void f32_few_k_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ Cout,
    int R, int N, int K, int tiles_m, int tiles_n) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles = tiles_m * tiles_n, e = blockIdx.x / tiles;
  const int rem = blockIdx.x - e * tiles, tm = rem / tiles_n, tn = rem - tm * tiles_n;
  const int row0 = tm * 64, col0 = (tn * 4 + wave) * 64;
  if (col0 >= N) return;
  const int c = lane & 15, g = lane >> 4;
  const float* a_at = A + (int64_t)e * K * R + min(row0 + 4 * c, R - 4);
  const float* b_at = B + (int64_t)e * K * N + min(col0 + 4 * c, N - 4);
  float4 a[KS], b[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int64_t k = min(4 * s + g, K - 1);
    a[s] = *reinterpret_cast<const float4*>(a_at + k * R);
    b[s] = *reinterpret_cast<const float4*>(b_at + k * N);
  }
  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const bool there = 4 * s + g < K;
    const float av[4] = {there ? a[s].x : 0.f, there ? a[s].y : 0.f,
                         there ? a[s].z : 0.f, there ? a[s].w : 0.f};
    const float bv[4] = {there ? b[s].x : 0.f, there ? b[s].y : 0.f,
                         there ? b[s].z : 0.f, there ? b[s].w : 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
  }
  const int col = col0 + 4 * c;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 16 * g + 4 * r + i;
      if (row < R && col < N)
        *reinterpret_cast<float4*>(Cout + ((int64_t)e * R + row) * N + col) =
            make_float4(acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]);
    }
}

bool f32_few_k_applies(int R, int N, int K) {
  return K >= 1 && K < 32 && R >= 16 && N >= 16 && R % 4 == 0 && N % 4 == 0;
}

int f32_few_k(const float* A, const float* B, float* C, int E, int R, int N, int K,
              hipStream_t st) {
  const int64_t tiles_m = ((int64_t)R + 63) / 64, tiles_n = ((int64_t)N + 255) / 256;
  MOE_REQUIRE((int64_t)E * tiles_m <= 0x7fffffffLL / tiles_n, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: too many tiles (%lld a expert)", (long long)(tiles_m * tiles_n));
  const unsigned blocks = (unsigned)(E * tiles_m * tiles_n);
  auto k = K <= 16 ? f32_few_k_kernel<4> : f32_few_k_kernel<8>;
  k<<<blocks, 256, 0, st>>>(A, B, C, R, N, K, (int)tiles_m, (int)tiles_n);
  MOE_CHECK_LAUNCH("expert_ffn (float32, sums over few rows)");
  return 0;
}

// ---------------------------------------------------------------------------
// Sums that do not change: v_mfma_f32_32x32x2_f32, true float32 operands, the
// order of k and the tiles these products have always had.
//
// For the hidden tensor of ReLU experts in a training step (mesh_moe_expert_ffn_kept).
// Its ReLU lets a unit through or not by the sign of a sum, about one in ten million of
// these sums is 0 up to rounding, and a unit that switches moves its column of the
// weight gradient by up to 0.6 of the gradient's root mean square.  With other rounding
// a few units of a step would switch, so that steps of two versions could not be
// compared; the more exact kernel above is as good an answer, and not the same one.
// The price: 60 us instead of 41 (8 experts x 320 rows, 512 -> 2048), and that a step
// without gradients rounds h otherwise.  Hidden tensors that are made projection by
// projection (dense layers, experts with dropout or several factors) have the sums of
// the kernel above.
// Also for short reductions of little work, which are faster here.
//
// Four wavefronts; K step 32.  The weight tile is the MFMA's first operand, so a
// lane ends up with 4 consecutive output columns per register group.  One MFMA
// consumes k = 2 s + (lane / 32) for step s; a lane instead takes the four
// consecutive k = 8 u + 4 (lane / 32) + j for steps 4 u + j, which makes its operand
// reads 16 bytes wide.  Tiles are staged through registers into LDS rows of 32 + 4
// floats.  K % 4 == 0 and N % 4 == 0.
//
// Bound by the float32 matrix pipes, of whose 64 cycles an MFMA the loop keeps 60 to
// 75 % busy.  Three (128 x 128 tiles: two) K tiles are on their way in registers, and
// the barrier does not wait for them.  8 experts x 320 rows, 5.4 GFLOP (34 us at the
// peak): 512 -> 2048 62 us, 2048 -> 512 67 us.
//
// TM x TN: MFMA tiles per wavefront.  WM x WN x WK: the wavefronts' grid; the
// WK wavefronts of a sub-tile share out the k of every staged tile and add up
// their sums in the end, so a small tile keeps all four matrix pipes busy.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

template <int TM, int TN, int WM, int WN, int WK>
struct F32Cfg {
  static_assert(WM * WN * WK == 4, "four wavefronts");
  static constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN, BK = 32,
                       THREADS = 256;
  // floats per LDS row and per stage of an operand
  static constexpr int LDR = BK + 4;
  static constexpr int STAGE_A = BM * LDR, STAGE_B = BN * LDR;
  static constexpr int CPR = BK / 4;      // 16-byte chunks per staged row
  // K tiles loaded ahead
  static constexpr int PF = BM * BN >= 128 * 128 ? 2 : 3;
  static constexpr int A_CHUNKS = BM * BK / 4 / THREADS;
  static constexpr int B_CHUNKS = BN * BK / 4 / THREADS;
  static constexpr size_t LDS_BYTES =
      2ull * (STAGE_A + STAGE_B) * sizeof(float);
  static_assert(LDS_BYTES >= (WK - 1) * WM * WN * TM * TN * 1024 * sizeof(float),
                "the partial sums of the other wavefronts fit");
};

template <int TM, int TN, int WM, int WN, int WK>
__global__ __launch_bounds__(256) void grouped_gemm_f32_mfma_kernel(
    const float* __restrict__ A, const float* __restrict__ B,
    float* __restrict__ Cout, int R, int N, int K, int tiles_m, int tiles_n,
    int relu, const float* __restrict__ mask_src, float mask_scale) {
  using Cfg = F32Cfg<TM, TN, WM, WN, WK>;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK;
  constexpr int LDR = Cfg::LDR, CPR = Cfg::CPR, PF = Cfg::PF;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  float* As = reinterpret_cast<float*>(smem_raw);  // [2][STAGE_A]
  float* Bs = As + 2 * Cfg::STAGE_A;               // [2][STAGE_B]
  const int nblk = gridDim.x;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int logical = xcd * (nblk >> 3) + min(xcd, nblk & 7) + local;
  const int tiles_per_e = tiles_m * tiles_n;
  const int e = logical / tiles_per_e;
  const int rem = logical - e * tiles_per_e;
  const int tn = rem / tiles_m, tm = rem - tn * tiles_m;
  const int row0 = tm * BM, col0 = tn * BN;
  const float* Ae = A + (int64_t)e * R * K;
  const float* Be = B + (int64_t)e * N * K;
  float* Ce = Cout + (int64_t)e * R * N;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wk = wave / (WM * WN), wmn = wave % (WM * WN);
  const int wm = wmn / WN, wn = wmn % WN;

  // PF K tiles are on their way in registers beside the one in LDS.  Chunk c of
  // an operand tile whose first row is `first` of `rows`; addresses are clamped
  // into the operand, what lies past the end of k becomes 0 on its way into LDS.
  uint4 areg[PF][Cfg::A_CHUNKS], breg[PF][Cfg::B_CHUNKS];
  auto load_chunk = [&](const float* src, int c, int first, int rows, int k0) {
    const int r = c / CPR, off = (c % CPR) * 4;
    return *reinterpret_cast<const uint4*>(
        src + (int64_t)min(first + r, rows - 1) * K + min(k0 + off, K - 4));
  };
  auto load_global = [&](int k0, auto slot_c) {
    constexpr int SLOT = decltype(slot_c)::value;
#pragma unroll
    for (int i = 0; i < Cfg::A_CHUNKS; ++i)
      areg[SLOT][i] = load_chunk(Ae, tid + i * Cfg::THREADS, row0, R, k0);
#pragma unroll
    for (int i = 0; i < Cfg::B_CHUNKS; ++i)
      breg[SLOT][i] = load_chunk(Be, tid + i * Cfg::THREADS, col0, N, k0);
  };
  auto store_chunk = [&](float* dst, int c, uint4 v, int k0) {
    const int r = c / CPR, off = (c % CPR) * 4;
    if (k0 + BK > K && k0 + off >= K) v = make_uint4(0, 0, 0, 0);
    *reinterpret_cast<uint4*>(dst + r * LDR + off) = v;
  };
  auto store_lds = [&](int buf, int k0, auto slot_c) {
    constexpr int SLOT = decltype(slot_c)::value;
#pragma unroll
    for (int i = 0; i < Cfg::A_CHUNKS; ++i)
      store_chunk(As + buf * Cfg::STAGE_A, tid + i * Cfg::THREADS, areg[SLOT][i],
                  k0);
#pragma unroll
    for (int i = 0; i < Cfg::B_CHUNKS; ++i)
      store_chunk(Bs + buf * Cfg::STAGE_B, tid + i * Cfg::THREADS, breg[SLOT][i],
                  k0);
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int nk = (K + BK - 1) / BK;
  // where this lane's operands start: a row and four k, of its wavefront's k
  constexpr int US = BK / 8 / WK;                  // groups of 8 k a wavefront
  const int frag_row = lane & 31, frag_k = (lane >> 5) * 4 + wk * US * 8;
  const int a_at = (wm * 32 * TM + frag_row) * LDR + frag_k;
  const int b_at = (wn * 32 * TN + frag_row) * LDR + frag_k;
  auto fragment = [&](const float* src, int tile, int u) {
    return *reinterpret_cast<const float4*>(src + tile * 32 * LDR + u * 8);
  };
  auto step = [&](int kt, auto slot_c) {
    const int buf = kt & 1;
    // (the other stage may still be read by wavefronts one step behind; this
    // one's readers passed the barrier of the step before)
    store_lds(buf, kt * BK, slot_c);
    load_global((kt + PF) * BK, slot_c);
    // the LDS writes of every wavefront are done; the loads stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const float* as = As + buf * Cfg::STAGE_A + a_at;
    const float* bs = Bs + buf * Cfg::STAGE_B + b_at;
#pragma unroll
    for (int u = 0; u < US; ++u) {
      float4 af[TM], bfr[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = fragment(as, i, u);
#pragma unroll
      for (int j = 0; j < TN; ++j) bfr[j] = fragment(bs, j, u);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const float a = q == 0 ? af[i].x : q == 1 ? af[i].y
                            : q == 2 ? af[i].z : af[i].w;
            const float b = q == 0 ? bfr[j].x : q == 1 ? bfr[j].y
                            : q == 2 ? bfr[j].z : bfr[j].w;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b, a, acc[i][j],
                                                             0, 0, 0);
          }
      }
    }
  };
  load_global(0, std::integral_constant<int, 0>());
  load_global(BK, std::integral_constant<int, 1>());
  if constexpr (PF > 2) load_global(2 * BK, std::integral_constant<int, PF - 1>());
  for (int kt = 0; kt < nk; kt += PF) {
    step(kt, std::integral_constant<int, 0>());
    if (kt + 1 < nk) step(kt + 1, std::integral_constant<int, 1>());
    if constexpr (PF > 2)
      if (kt + 2 < nk) step(kt + 2, std::integral_constant<int, PF - 1>());
  }
  if constexpr (WK > 1) {
    // [wk - 1][sub-tile][TM][TN][16][64], where the stages were
    __syncthreads();
    float* parts = reinterpret_cast<float*>(smem_raw);
    constexpr int SUB = TM * TN * 1024, PLANE = WM * WN * SUB;
    if (wk > 0) {
      float* dst = parts + (wk - 1) * PLANE + wmn * SUB + lane;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            dst[((i * TN + j) * 16 + r) * 64] = acc[i][j][r];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int w = 0; w < WK - 1; ++w) {
      const float* src = parts + w * PLANE + wmn * SUB + lane;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[i][j][r] += src[((i * TN + j) * 16 + r) * 64];
    }
  }
  const int m_l = lane & 31, n_l = (lane >> 5) * 4;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int grow = row0 + (wm * TM + i) * 32 + m_l;
        const int gcol = col0 + (wn * TN + j) * 32 + 8 * q + n_l;
        if (grow < R && gcol < N) {
          float4 v = make_float4(acc[i][j][4 * q + 0], acc[i][j][4 * q + 1],
                                 acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
          const int64_t at = (int64_t)grow * N + gcol;
          if (relu) {
            v.x = fmaxf(v.x, 0.f); v.y = fmaxf(v.y, 0.f);
            v.z = fmaxf(v.z, 0.f); v.w = fmaxf(v.w, 0.f);
          }
          if (mask_src != nullptr) {
            const float4 m = *reinterpret_cast<const float4*>(
                mask_src + (int64_t)e * R * N + at);
            v = make_float4(finish_f32(v.x, false, true, m.x, mask_scale),
                            finish_f32(v.y, false, true, m.y, mask_scale),
                            finish_f32(v.z, false, true, m.z, mask_scale),
                            finish_f32(v.w, false, true, m.w, mask_scale));
          }
          *reinterpret_cast<float4*>(Ce + at) = v;
        }
      }
}

template <int TM, int TN, int WM, int WN, int WK>
static int launch_f32_mfma_tile(const float* A, const float* B, float* C, int E,
                                int R, int N, int K, bool relu,
                                const float* mask_src, float mask_scale,
                                hipStream_t st) {
  using Cfg = F32Cfg<TM, TN, WM, WN, WK>;
  const int tiles_m = (R + Cfg::BM - 1) / Cfg::BM;
  const int tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  const int64_t blocks = (int64_t)tiles_m * tiles_n * E;
  MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: too many tiles (%lld)", (long long)blocks);
  auto k = grouped_gemm_f32_mfma_kernel<TM, TN, WM, WN, WK>;
  MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
  k<<<(unsigned)blocks, Cfg::THREADS, Cfg::LDS_BYTES, st>>>(
      A, B, C, R, N, K, tiles_m, tiles_n, relu ? 1 : 0, mask_src, mask_scale);
  MOE_CHECK_LAUNCH("expert_ffn (float32 mfma)");
  return 0;
}

// Block tile of the float32 kernel.  The kernel is bound by the float32 matrix
// pipes (a 32 x 32 x 2 MFMA takes 64 cycles), so its time is rounds of tiles
// over the compute units times the tile's area; small launches want small tiles
// (less padding of the row count, fewer idle compute units in the last round).
// The smallest two pay for it with more LDS and cache traffic per product: the
// weights.  Measured at 8 experts x 320 rows, per launch (us), in the order of
// the table: 512 -> 2048 83, 71, 62, 67, 73; 2048 -> 512 151, 85, 85, 73, 67.
int f32_gemm_stable(const float* A, const float* B, float* C, int E, int R, int N,
                    int K, bool relu, const float* mask_src, float mask_scale,
                    hipStream_t st) {
  const int cus = compute_units();
  if (cus == 0) return MESH_MOE_E_HIP;
  static const int shapes[5][2] = {{128, 128}, {64, 128}, {64, 64}, {32, 64},
                                   {32, 32}};
  static const double weight[5] = {1.0, 1.0, 1.0, 1.08, 1.18};
  int best = 0;
  double best_cost = 0;
  int64_t best_tiles = 0;
  for (int i = 0; i < 5; ++i) {
    const int bm = shapes[i][0], bn = shapes[i][1];
    const int64_t tiles = (int64_t)E * ((R + bm - 1) / bm) * ((N + bn - 1) / bn);
    const double cost = (double)((tiles + cus - 1) / cus) * bm * bn * weight[i];
    // a smaller tile when it saves time by this count, or costs the same while
    // the larger one leaves compute units with fewer than two blocks to overlap
    if (i == 0 || cost < 0.95 * best_cost ||
        (cost <= best_cost && best_tiles < 2 * (int64_t)cus)) {
      best = i;
      best_cost = cost;
      best_tiles = tiles;
    }
  }
#define MOE_F32_TILE(...)                                                      \
  launch_f32_mfma_tile<__VA_ARGS__>(A, B, C, E, R, N, K, relu, mask_src,       \
                                    mask_scale, st)
  switch (best) {
    case 0: return MOE_F32_TILE(2, 2, 2, 2, 1);
    case 1: return MOE_F32_TILE(1, 2, 2, 2, 1);
    case 2: return MOE_F32_TILE(1, 1, 2, 2, 1);
    case 3: return MOE_F32_TILE(1, 1, 1, 2, 2);
    default: return MOE_F32_TILE(1, 1, 1, 1, 4);
  }
#undef MOE_F32_TILE
}

}  // namespace mesh_moe
