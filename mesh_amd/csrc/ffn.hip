// Expert feed-forward as a grouped GEMM for gfx950:
//   h[e] = act(expert_in[e] . wi[e]),  y[e] = h[e] . wo[e]
// Replaces layers.dense_product "wi" + layers.dense "wo" of
// mesh_tensorflow/transformer/moe.py:469-486 (hierarchical layer: :765-774).
//
// Both GEMMs are "TN": A [R, K] and the packed weight B [N, K] are
// K-contiguous, C [R, N] = A . B^T.  The bf16 kernel uses
// v_mfma_f32_32x32x16_bf16 with LDS double buffering; float32 has its own file
// (gemm_f32.hip), odd shapes use a plain FMA tile kernel.
#include <type_traits>

#include "common.h"

namespace mesh_moe {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

// ---------------------------------------------------------------------------
// bf16 MFMA kernel.
// Block tile BM x BN, K step BK, 4 wavefronts in a 2 x 2 grid, each owning a
// (BM/2) x (BN/2) sub-tile made of 32 x 32 MFMA tiles.  LDS rows hold BK bf16
// plus 8 bf16 of padding, which makes the 16-byte fragment reads of
// consecutive rows hit disjoint banks.
//
// The weight tile is fed as the MFMA "A" operand and the activation tile as
// "B", i.e. each MFMA produces a 32(n) x 32(m) block of C^T.  Per lane l the
// operands are row/column l%32 with k = 8*(l/32)..+7, and accumulator register
// r holds n = 8*(r/4) + 4*(l/32) + r%4 for m = l%32: four consecutive output
// columns per lane, which the epilogue packs into one 8-byte LDS write.  The
// finished tile is staged in LDS and written out with 16-byte row-contiguous
// stores.
// ---------------------------------------------------------------------------
template <int BM, int BN, int BK>
struct GemmCfg {
  static constexpr int THREADS = 256;
  static constexpr int LDK = BK + 8;  // padded LDS row, in bf16
  static constexpr int WTM = BM / 2, WTN = BN / 2;
  static constexpr int TM = WTM / 32, TN = WTN / 32;
  static constexpr int CPR = BK / 8;  // 16-byte chunks per tile row
  static constexpr int A_CHUNKS = BM * CPR / THREADS;
  static constexpr int B_CHUNKS = BN * CPR / THREADS;
  static constexpr int LDC = BN + 4;  // padded row of the staged C tile
  static constexpr size_t LOOP_BYTES = 2ull * (BM + BN) * LDK * sizeof(bf16_t);
  static constexpr size_t EPI_BYTES = (size_t)BM * LDC * sizeof(bf16_t);
  static constexpr size_t LDS_BYTES =
      LOOP_BYTES > EPI_BYTES ? LOOP_BYTES : EPI_BYTES;
};

// relu commutes with the rounding (which keeps the sign; -0 and +0 both end as
// +0), so it is applied to the float32 accumulators
__device__ __forceinline__ uint32_t pack2_bf16(float a, float b, bool relu) {
  if (relu) {
    a = fmaxf(a, 0.f);
    b = fmaxf(b, 0.f);
  }
  return f32x2_to_bf16x2(a, b);
}

template <int BM, int BN, int BK, bool RELU, bool OUT_F32 = false>
__global__ __launch_bounds__(256) void grouped_gemm_bf16_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
    void* __restrict__ Cvoid, int R, int N, int K, int tiles_m, int tiles_n,
    int64_t a_stride) {
  bf16_t* Cout = reinterpret_cast<bf16_t*>(Cvoid);
  using Cfg = GemmCfg<BM, BN, BK>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  bf16_t* As = reinterpret_cast<bf16_t*>(smem_raw);  // [2][BM][LDK]
  bf16_t* Bs = As + 2 * BM * Cfg::LDK;               // [2][BN][LDK]

  // Workgroups are handed to the 8 XCDs round-robin (block b runs on XCD
  // b % 8) and each XCD has its own L2.  Renumber so that every XCD works on a
  // contiguous range of logical tiles; logical tiles walk the M tiles of one
  // (expert, N tile), so the tiles resident on an XCD at one time share a few
  // weight panels and all of the expert's activation rows through that L2.
  const int nblk = gridDim.x;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int q = nblk >> 3, rmd = nblk & 7;
  const int logical = xcd * q + min(xcd, rmd) + local;
  const int tiles_per_e = tiles_m * tiles_n;
  const int e = logical / tiles_per_e;
  const int rem = logical - e * tiles_per_e;
  const int tn = rem / tiles_m;
  const int tm = rem - tn * tiles_m;
  const int row0 = tm * BM, col0 = tn * BN;
  // (a_stride: elements from one expert's rows to the next one's, 0 where all
  // experts read the same rows)
  const bf16_t* Ae = A + e * a_stride;
  const bf16_t* Be = B + (int64_t)e * N * K;
  bf16_t* Ce = Cout + (int64_t)e * R * N;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // global -> register staging (rows clamped; the K tail reads zeros)
  uint4 areg[Cfg::A_CHUNKS], breg[Cfg::B_CHUNKS];
  auto load_global = [&](int k0) {
#pragma unroll
    for (int i = 0; i < Cfg::A_CHUNKS; ++i) {
      int c = tid + i * Cfg::THREADS;
      int r = c / Cfg::CPR, kc = c % Cfg::CPR;
      int gr = min(row0 + r, R - 1);
      int gk = k0 + kc * 8;
      uint4 v = *reinterpret_cast<const uint4*>(Ae + (int64_t)gr * K + min(gk, K - 8));
      areg[i] = gk < K ? v : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < Cfg::B_CHUNKS; ++i) {
      int c = tid + i * Cfg::THREADS;
      int r = c / Cfg::CPR, kc = c % Cfg::CPR;
      int gr = min(col0 + r, N - 1);
      int gk = k0 + kc * 8;
      uint4 v = *reinterpret_cast<const uint4*>(Be + (int64_t)gr * K + min(gk, K - 8));
      breg[i] = gk < K ? v : make_uint4(0, 0, 0, 0);
    }
  };
  auto store_lds = [&](int buf) {
    bf16_t* as = As + buf * BM * Cfg::LDK;
    bf16_t* bs = Bs + buf * BN * Cfg::LDK;
#pragma unroll
    for (int i = 0; i < Cfg::A_CHUNKS; ++i) {
      int c = tid + i * Cfg::THREADS;
      int r = c / Cfg::CPR, kc = c % Cfg::CPR;
      *reinterpret_cast<uint4*>(as + r * Cfg::LDK + kc * 8) = areg[i];
    }
#pragma unroll
    for (int i = 0; i < Cfg::B_CHUNKS; ++i) {
      int c = tid + i * Cfg::THREADS;
      int r = c / Cfg::CPR, kc = c % Cfg::CPR;
      *reinterpret_cast<uint4*>(bs + r * Cfg::LDK + kc * 8) = breg[i];
    }
  };

  f32x16_t acc[Cfg::TM][Cfg::TN];
#pragma unroll
  for (int i = 0; i < Cfg::TM; ++i)
#pragma unroll
    for (int j = 0; j < Cfg::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int nk = (K + BK - 1) / BK;
  load_global(0);
  store_lds(0);
  __syncthreads();
  const int frag_row = lane & 31;
  const int frag_k = (lane >> 5) * 8;
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) load_global((kt + 1) * BK);
    const bf16_t* as = As + buf * BM * Cfg::LDK + (wm * Cfg::WTM + frag_row) * Cfg::LDK + frag_k;
    const bf16_t* bs = Bs + buf * BN * Cfg::LDK + (wn * Cfg::WTN + frag_row) * Cfg::LDK + frag_k;
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bf16x8_t af[Cfg::TM], bfr[Cfg::TN];
#pragma unroll
      for (int i = 0; i < Cfg::TM; ++i)
        af[i] = *reinterpret_cast<const bf16x8_t*>(as + i * 32 * Cfg::LDK + kk * 16);
#pragma unroll
      for (int j = 0; j < Cfg::TN; ++j)
        bfr[j] = *reinterpret_cast<const bf16x8_t*>(bs + j * 32 * Cfg::LDK + kk * 16);
#pragma unroll
      for (int i = 0; i < Cfg::TM; ++i)
#pragma unroll
        for (int j = 0; j < Cfg::TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[j], af[i], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) store_lds(buf ^ 1);
    __syncthreads();
  }

  const int m_l = lane & 31;
  const int n_l = (lane >> 5) * 4;
  if (OUT_F32) {
    // float32 result (attention logits, which the reference keeps in float32):
    // every lane owns 4 consecutive columns per register group
    float* Cf = reinterpret_cast<float*>(Cvoid) + (int64_t)e * R * N;
#pragma unroll
    for (int i = 0; i < Cfg::TM; ++i) {
#pragma unroll
      for (int j = 0; j < Cfg::TN; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int grow = row0 + wm * Cfg::WTM + i * 32 + m_l;
          const int gcol = col0 + wn * Cfg::WTN + j * 32 + 8 * q + n_l;
          if (grow < R && gcol < N) {
            float4 v = make_float4(acc[i][j][4 * q + 0], acc[i][j][4 * q + 1],
                                   acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
            if (RELU) {
              v.x = fmaxf(v.x, 0.f); v.y = fmaxf(v.y, 0.f);
              v.z = fmaxf(v.z, 0.f); v.w = fmaxf(v.w, 0.f);
            }
            *reinterpret_cast<float4*>(Cf + (int64_t)grow * N + gcol) = v;
          }
        }
      }
    }
    return;
  }
  // epilogue: round (and relu), stage the tile in LDS, coalesced stores
  bf16_t* Cs = reinterpret_cast<bf16_t*>(smem_raw);  // [BM][LDC]
#pragma unroll
  for (int i = 0; i < Cfg::TM; ++i) {
#pragma unroll
    for (int j = 0; j < Cfg::TN; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = wm * Cfg::WTM + i * 32 + m_l;
        const int col = wn * Cfg::WTN + j * 32 + 8 * q + n_l;
        uint2 v;
        v.x = pack2_bf16(acc[i][j][4 * q + 0], acc[i][j][4 * q + 1], RELU);
        v.y = pack2_bf16(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3], RELU);
        *reinterpret_cast<uint2*>(Cs + row * Cfg::LDC + col) = v;
      }
    }
  }
  __syncthreads();
  constexpr int CPR_C = BN / 8;  // 16-byte chunks per output row
#pragma unroll 4
  for (int c = tid; c < BM * CPR_C; c += Cfg::THREADS) {
    const int r = c / CPR_C, cc = (c % CPR_C) * 8;
    const int grow = row0 + r, gcol = col0 + cc;
    if (grow < R && gcol < N) {
      const uint2* s = reinterpret_cast<const uint2*>(Cs + r * Cfg::LDC + cc);
      uint2 lo = s[0], hi = s[1];
      *reinterpret_cast<uint4*>(Ce + (int64_t)grow * N + gcol) =
          make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
  }
}

// ---------------------------------------------------------------------------
// bf16 MFMA kernel for a few rows per expert (decoding steps, small batches):
// the launch is a stream over the weights.
//
// A block owns 16 NT columns of one expert and all of its rows (MT tiles of 16);
// its wavefronts cut the reduction into contiguous parts and add their sums in
// LDS, in wavefront order.  Operands go from global memory to registers as the
// instruction (16 x 16 x 32) wants them: lane l brings row l % 16, 16 bytes at k =
// 8 (l / 16), i.e. 64-byte pieces of 16 rows per load.  That is a quarter of what
// the load path can do for whole lines and four times what the weights need
// (each weight byte is read by one block, once); the tokens come from the L2.
// No LDS in the loop, no barrier: a wavefront has U (MT + NT) loads in flight.
// 32 rows: 1024 x 1024 6.5 us, 1024 x 4096 6.9, 4096 x 1024 15.8; the 128 x 128
// tile kernel, one block per 128 columns walking all of K: 20.4, 20.7, 69.9.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

template <int MT, int NT>
__global__ __launch_bounds__(1024) void skinny_gemm_bf16_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
    bf16_t* __restrict__ C, int R, int N, int K, int groups_n, int relu,
    int64_t a_stride) {
  constexpr int U = MT <= 2 ? 4 : 2;       // k steps of 32 loaded together
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int waves = blockDim.x >> 6;
  const int e = blockIdx.x / groups_n, n0 = (blockIdx.x - e * groups_n) * 16 * NT;
  const int r16 = lane & 15, kq = (lane >> 4) * 8;
  const bf16_t* bp[NT];
  const bf16_t* ap[MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    bp[j] = B + ((int64_t)e * N + min(n0 + 16 * j + r16, N - 1)) * K + kq;
#pragma unroll
  for (int i = 0; i < MT; ++i)
    ap[i] = A + e * a_stride + (int64_t)min(16 * i + r16, R - 1) * K + kq;
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[i][j][q] = 0.f;
  const int steps = K / 32;
  const int s1 = (int)((int64_t)steps * (wave + 1) / waves);
  int s = (int)((int64_t)steps * wave / waves);
  auto block_of = [&](auto u_tag) {
    constexpr int UU = decltype(u_tag)::value;
    bf16x8_t bf[UU][NT], af[UU][MT];
#pragma unroll
    for (int u = 0; u < UU; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        bf[u][j] = __builtin_nontemporal_load(
            reinterpret_cast<const bf16x8_t*>(bp[j] + (s + u) * 32));
#pragma unroll
    for (int u = 0; u < UU; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i)
        af[u][i] = *reinterpret_cast<const bf16x8_t*>(ap[i] + (s + u) * 32);
#pragma unroll
    for (int u = 0; u < UU; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              bf[u][j], af[u][i], acc[i][j], 0, 0, 0);
    s += UU;
  };
  while (s + U <= s1) block_of(std::integral_constant<int, U>{});
  while (s < s1) block_of(std::integral_constant<int, 1>{});
  // lane: row 16 i + l % 16, columns 16 j + 4 (l / 16) ..
  f32x4_t* part = reinterpret_cast<f32x4_t*>(smem_raw);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      part[(wave * (MT * NT) + i * NT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  for (int t = wave; t < MT * NT; t += waves) {
    f32x4_t sum = part[t * 64 + lane];
    for (int w = 1; w < waves; ++w) {
      const f32x4_t v = part[(w * (MT * NT) + t) * 64 + lane];
#pragma unroll
      for (int q = 0; q < 4; ++q) sum[q] += v[q];
    }
    const int row = t / NT * 16 + r16, col = n0 + t % NT * 16 + (lane >> 4) * 4;
    if (row < R && col < N) {
      uint2 v;
      v.x = pack2_bf16(sum[0], sum[1], relu != 0);
      v.y = pack2_bf16(sum[2], sum[3], relu != 0);
      *reinterpret_cast<uint2*>(C + ((int64_t)e * R + row) * N + col) = v;
    }
  }
}

// ---------------------------------------------------------------------------
// Direct global -> LDS loads, which feed the K loops of the kernels below
// (global_load_lds_dwordx4): every lane names its own 16 global bytes and the
// wavefront's 64 x 16 bytes land contiguously in LDS without passing through
// registers.
//
// One load instruction fetches 8 rows x 128 bytes (BK = 64 bf16): 8 consecutive
// lanes read one full 128-byte line of a row, which is what the memory
// pipeline coalesces best (lanes that stride across rows run ~4x slower).
// LDS therefore holds plain 128-byte rows, and bank conflicts are avoided by
// an XOR swizzle of the 16-byte chunk index applied on the GLOBAL side: the
// lane that fills LDS slot (row, p) loads chunk p ^ swz(row), with
// swz(row) = (row & 7) ^ ((row >> 3) & 1).  The MFMA fragment read of 16
// consecutive rows at one chunk then touches 16 distinct 16-byte columns of a
// 256-byte window (and any 8 consecutive rows 8 distinct columns of 128 bytes).
// Requires K % 64 == 0 and per-expert operand sizes below 2^30 elements.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void lds_void_t;
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;
typedef const __attribute__((address_space(1))) void glb_void_t;

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  // s_waitcnt with expcnt / lgkmcnt left at "no wait"
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void lds_write_b64_asm(uint32_t addr, u32x2_t v) {
  asm volatile("ds_write_b64 %0, %1" :: "v"(addr), "v"(v) : "memory");
}
// Four 16-byte reads, 8192 bytes apart, and the wait for them: in one asm, whose
// outputs then hold what the compiler takes them for.
__device__ __forceinline__ void lds_read_lines(u32x4_t (&p)[4], uint32_t at) {
  asm volatile("ds_read_b128 %0, %4\n\t"
               "ds_read_b128 %1, %4 offset:8192\n\t"
               "ds_read_b128 %2, %4 offset:16384\n\t"
               "ds_read_b128 %3, %4 offset:24576\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2]), "=&v"(p[3])
               : "v"(at)
               : "memory");
}

__device__ __forceinline__ int lds_swizzle(int row) {
  return (row & 7) ^ ((row >> 3) & 1);
}

// ---------------------------------------------------------------------------
// bf16 MFMA kernel for 256 x 256 tiles with SPREAD direct-to-LDS loads.
//
// 8 wavefronts in a 2 x 4 grid, two per SIMD, each a 128 x 64 sub-tile = 4 x 2
// MFMA tiles; operand roles as in the first kernel of this file.  What shapes
// the kernel is when the loads are issued.  A wavefront that issues its eight
// loads of a K tile back to back sits in that burst for ~0.7 us (the memory
// pipeline accepts them only as fast as earlier requests drain), and because
// the wavefronts of a block hand over together, the MFMA pipes idle meanwhile.
// Here the 160 KB of LDS hold two slots for the token tile and THREE for the
// weight tile, which lets the loads of tile t+2 ride on the MFMA steps of
// tile t, pinned between its MFMAs:
//
//   step 0:            weight loads 0,1 of tile t+2   (two tiles ahead)
//   step 1, step 2:    weight load 2 / weight load 3 of tile t+2
//   step 3 (after the hand-over barrier that frees their slot, behind the
//           first fragment reads of tile t+1): the four token loads of tile t+2
//
// vmcnt counts in issue order, so the hand-over of tile t waits with vmcnt(4):
// everything up to the token loads of tile t+1 has landed, the four weight
// loads of tile t+2 stay in flight.
// ---------------------------------------------------------------------------
// Two ds_read_b64_tr_b16 at byte offsets OFF and OFF + 2048 from LDS address
// `addr` (see the K-major variant of the ring kernel).
template <int OFF>
__device__ __forceinline__ void lds_read_tr16_pair(uint32_t addr, i16x4_t& lo,
                                                   i16x4_t& hi) {
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2"
               : "=v"(lo) : "v"(addr), "n"(OFF));
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2"
               : "=v"(hi) : "v"(addr), "n"(OFF + 2048));
}

// ---------------------------------------------------------------------------
// bf16 MFMA kernel for few rows per expert and many experts (a decoding step's
// experts): the launch is a stream over the weights, every byte of which one
// block reads once.
//
// Block tile: all rows of an expert (MT tiles of 32) x 128 columns, K step 64,
// 4 wavefronts of 32 columns each, direct-to-LDS loads (whole 128-byte lines,
// the same swizzled LDS image as above) into a ring of NS slots: NS - 1 K
// tiles in flight per block, two blocks per compute unit.  One barrier per K
// tile: it publishes the oldest tile and frees the slot that the next loads go
// to.
//
// row_map (optional, [E, R]): the slot -> token map.  An expert without an
// occupied slot is left out, its rows of C unwritten (nothing reads them).
// With `gather` row r of expert e is A[row_map[e, r]], zeros where that is
// negative.
//
// 64 experts, 512 MB of weights: 4 rows each 89 - 93 us (5.8 - 6.0 TB/s), 32 rows
// 100, 64 rows 107 (K = 1024) and 113 (K = 4096); the 128 x 128 register-staged
// kernel before: 112 / 123 at 4 rows, 106 at 32, 110 / 130 at 64.  (8
// wavefronts and 256 columns: the same at 4 rows, 121 / 106 at 64.  65 to 128
// rows: 149 / 124 at 128 against 134 / 139 of the 128 x 128 kernel, which keeps
// them.)
// ---------------------------------------------------------------------------
template <int MT>        // tiles of 32 rows
struct StreamCfg {
  static constexpr int BN = 128, BK = 64, ROW_BYTES = BK * 2;
  static constexpr int A_BYTES = 32 * MT * ROW_BYTES, B_BYTES = BN * ROW_BYTES;
  static constexpr int SLOT_BYTES = A_BYTES + B_BYTES;
  static constexpr int NS = 80 * 1024 / SLOT_BYTES;
  static constexpr size_t LDS_BYTES = (size_t)NS * SLOT_BYTES;
  static constexpr int LOADS = MT + 4;     // per wavefront and K tile
  static_assert(NS >= 3, "a ring");
};

template <int MT, bool MAPPED>
__global__ __launch_bounds__(256) void stream_gemm_bf16_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
    bf16_t* __restrict__ C, int R, int N, int K, int tiles_n, int relu,
    const int32_t* __restrict__ row_map, int gather,
    const bf16_t* __restrict__ zero_row,
    int64_t a_stride) {
  using Cfg = StreamCfg<MT>;
  constexpr int BN = Cfg::BN, BK = Cfg::BK, NS = Cfg::NS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int e = blockIdx.x / tiles_n, tn = blockIdx.x - e * tiles_n;
  const int col0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bf16_t* asrc[MT];
  const bf16_t* bsrc[4];
  bool any = !MAPPED;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int row = (wave + 4 * j) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ lds_swizzle(row);
    const bf16_t* base = A + e * a_stride + (int64_t)min(row, R - 1) * K;
    if constexpr (MAPPED) {
      const int src = row_map[(int64_t)e * R + min(row, R - 1)];
      any |= src >= 0;
      if (gather) base = src >= 0 ? A + (int64_t)src * K : zero_row;
    }
    asrc[j] = base + chunk * 8;
  }
  if constexpr (MAPPED) {
    if (!__syncthreads_or(any)) return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = (wave + 4 * j) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ lds_swizzle(row);
    bsrc[j] = B + ((int64_t)e * N + min(col0 + row, N - 1)) * K + chunk * 8;
  }
  const int nk = K / BK;
  // Blocks start their walk along K at different K tiles: rows of a weight
  // matrix are a power of two apart in many models, and blocks in step would
  // all read from the same few memory channels (64 experts of 1024 x 4096, 4
  // rows: 113 us in step, 90 like this).
  // (Past the end of K a tile is fetched again into a slot nobody reads: every
  // K tile then has the same number of loads in flight behind it.)
  const int first = (int)((blockIdx.x * 5u) % (unsigned)nk);
  auto issue = [&](int kt, int slot) {
    int t = min(kt, nk - 1) + first;
    t = t >= nk ? t - nk : t;
    const int at = t * BK;
    unsigned char* sa = smem_raw + slot * Cfg::SLOT_BYTES;
    unsigned char* sb = sa + Cfg::A_BYTES;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_global_load_lds((glb_void_t*)(bsrc[j] + at),
                                       (lds_void_t*)(sb + (wave + 4 * j) * 1024),
                                       16, 0, 0);
#pragma unroll
    for (int j = 0; j < MT; ++j)
      __builtin_amdgcn_global_load_lds((glb_void_t*)(asrc[j] + at),
                                       (lds_void_t*)(sa + (wave + 4 * j) * 1024),
                                       16, 0, 0);
  };
  f32x16_t acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
#pragma unroll
  for (int t = 0; t < NS - 1; ++t) issue(t, t);
  const int fr = lane & 31, fc = lane >> 5;
  int slot = 0, free_slot = NS - 1;
  for (int kt = 0; kt < nk; ++kt) {
    // the oldest tile has landed, and this wavefront's reads of the slot that
    // is about to be loaded again have returned: the multiplications that use
    // them need not be issued yet
    wait_vmcnt<(NS - 2) * Cfg::LOADS>();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(kt + NS - 1, free_slot);
    const unsigned char* sa = smem_raw + slot * Cfg::SLOT_BYTES;
    const unsigned char* sb = sa + Cfg::A_BYTES + wave * 32 * Cfg::ROW_BYTES;
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      const int at = fr * Cfg::ROW_BYTES + (((kk * 2 + fc) ^ lds_swizzle(fr)) * 16);
      const bf16x8_t b = *reinterpret_cast<const bf16x8_t*>(sb + at);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(
            sa + i * 32 * Cfg::ROW_BYTES + at);
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, acc[i], 0, 0, 0);
      }
    }
    free_slot = slot;
    slot = slot + 1 == NS ? 0 : slot + 1;
  }
  // no direct-to-LDS load may outlive the block
  wait_vmcnt<0>();
  // lane: row 32 i + l % 32, columns 8 q + 4 (l / 32) .. of the wavefront's 32
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row = i * 32 + fr;
    if (row >= R) continue;
    bf16_t* dst = C + ((int64_t)e * R + row) * N + col0 + wave * 32 + fc * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (col0 + wave * 32 + fc * 4 + 8 * q < N) {
        uint2 v;
        v.x = pack2_bf16(acc[i][4 * q], acc[i][4 * q + 1], relu != 0);
        v.y = pack2_bf16(acc[i][4 * q + 2], acc[i][4 * q + 3], relu != 0);
        *reinterpret_cast<uint2*>(dst + 8 * q) = v;
      }
  }
}

struct RingCfg {
  static constexpr int BM = 256, BN = 256, BK = 64, WM = 2, WN = 4;
  static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / 32, TN = WTN / 32;
  static constexpr int ROW_BYTES = BK * 2;
  static constexpr int A_INSTR = (BM / 8) / WAVES, B_INSTR = (BN / 8) / WAVES;
  static constexpr int A_BYTES = BM * ROW_BYTES, B_BYTES = BN * ROW_BYTES;
  static constexpr int A_SLOTS = 2, B_SLOTS = 3;
  static constexpr int B_BASE = A_SLOTS * A_BYTES;
  static constexpr size_t LOOP_BYTES = (size_t)A_SLOTS * A_BYTES + (size_t)B_SLOTS * B_BYTES;
  static constexpr size_t LDS_BYTES = LOOP_BYTES;  // the output is staged inside
  static_assert(A_INSTR == 4 && B_INSTR == 4, "load schedule assumes 4 + 4");
  // row tiles of at most DEEP_ROWS rows: three slots for the token tile too
  static constexpr int DEEP_ROWS = 160, DEEP_A_BYTES = DEEP_ROWS * ROW_BYTES;
  static_assert(3 * DEEP_A_BYTES + B_SLOTS * B_BYTES <= LDS_BYTES, "three slots");
};

// Position of tile `rem` of an expert where its row tiles are many: 32
// consecutive logical tiles (what an XCD holds at any moment) form a block of 8
// row tiles x 4 column tiles: 12 operand panels for 32 tiles.  With the plain
// order they would be 32 row tiles of one column tile: 33 panels, every row
// panel fetched once per column tile.  Blocks follow each other along N, so the
// next 32 tiles share the 8 row panels.  (8 row tiles: both orders are the
// same.)  Leaves (tm, tn) alone where it does not apply.
__device__ __forceinline__ void ring_tile_blocks(int rem, int tiles_m,
                                                 int tiles_n, int& tm, int& tn) {
  if (tiles_m > 8 && (tiles_m & 7) == 0 && (tiles_n & 3) == 0) {
    const int sup = rem >> 5, within = rem & 31;
    const int per_row = tiles_n >> 2;
    const int sm = sup / per_row, sn = sup - sm * per_row;
    tm = sm * 8 + (within & 7);
    tn = sn * 4 + (within >> 3);
  }
}

// GATHER: the rows of expert e's first operand are not A[e][r] but rows of a
// shared token matrix, A[row_map[e * R + r]] (row_map < 0: the all-zero row
// `zero_row`): the dispatch of the Mixture-of-Experts layer folded into the
// first expert GEMM's loads.
//
// KMAJOR: both operands are stored with the reduction index outermost,
// A[e][k][r] and B[e][k][n] (C = A^T . B, the weight gradients of the expert
// einsums: the reduction runs over token rows).  A K tile is then 64 rows of
// 256 consecutive elements; it goes to LDS as it lies in memory (row k at byte
// 512 k, the 64-byte units of a row XOR-ed with k % 4 against bank
// conflicts) and the MFMA operands, which need 8 consecutive k per lane, are
// read with ds_read_b64_tr_b16: within 16 lanes, lane t addresses the 8 bytes
// at (row t / 4, elements 4 (t % 4) ..) of a 4 x 16 block and lane i receives
// the block's column i.  R, N multiples of 8.  With k_extent, expert e's
// reduction stops after its first k_extent[e] rows, rounded up to a K tile
// (rows up to there must hold finite values in one operand and zeros in the
// other); k_extent[e] == 0 gives an all-zero result.  K need not be a
// multiple of the K tile: the rows of the last tile past K come from a zero
// buffer.
//
// MASKED: element (e, r, n) of the result is stored as zero unless
// mask_src[e][r][n] > 0 (the backward of a ReLU whose output is mask_src,
// applied while the tile is written out).  The elements that stay are
// multiplied by mask_scale and rounded again (the backward of a dropout in
// front of the ReLU's consumer: where the stored activation is positive the
// element was kept, and its noise is 1 / keep_prob).
//
// LISTED: only the tiles named in tile_list[0 .. tile_list[-1]) are computed
// (logical tile numbers in ascending order, their count in the element before
// the list): an expert whose occupied rows were moved to the front of its row
// range needs no tiles for the rest (see mesh_moe_compact_expert_ffn).
// (Skipping, inside an expert's last listed tile, the 32-row pieces of a
// wavefront's sub-tile that lie past the occupied rows -- about a tenth of the
// multiply-adds with 1024 +- 32 rows per expert -- made the launches 2 to 5 %
// slower; so did letting only the wavefronts of a tile's empty second half
// skip their multiply-adds, with the flag carried in the list entry: 5 %
// slower, although nothing was added to the path of the full tiles but a
// second copy of the K loop next to it.)
//
// TAILS (row tiles of `tile_rows` <= 256 rows, see ring_tile_rows, and a last
// one that may hold fewer): a wavefront multiplies only 32-row pieces that hold
// rows -- their count is the same for the whole K loop, so the wavefront runs
// the copy of the loop written for that count (0 to 4 pieces; with 0 it only
// loads and meets the barriers).  The two wavefronts of a SIMD own the upper
// and the lower half of the LDS tile; the tile's pieces are dealt out evenly
// between them (rows 0 .. 32 p0 - 1 to the upper half, the others to the lower),
// so that neither waits for the other at the hand-overs.  (Numbering the
// experts' last row tiles after all full ones separates the row tiles that
// share a weight panel: with 400 rows per expert the weights were then read
// twice from memory and the launches took 14 % longer.)
//
// DEEP (TAILS with row tiles of at most 160 rows): three token slots of 160 rows
// instead of two of 256, and all seven loads of K tile t + 2 in steps 0 to 2 of K tile
// t.  A low tile's MFMAs take half a microsecond a K tile, less than a load takes from
// memory; with two slots the token loads wait for the hand-over that frees theirs and
// are due at the next one.  (Loads alone, without the products: 32 x 640 rows, 4096 ->
// 1024 159 of 168 us.)  Back to back, two slots / three, the same bits: 32 x 640 rows,
// 4096 -> 1024 170 / 154 us; 64 x 320, 1024 -> 4096 197 / 183; 16 x 256, 4096 -> 1024
// 52 / 41.5; 5000 rows, 1280 -> 1280 21.7 / 20.5; 16 x 708, 3072 -> 768 52.3 / 50.0.
// (Weights ahead of the tokens, or the last load behind the hand-over: 1 to 3 % slower;
// all loads in the first two steps: no change, as for the weights of the higher tiles.)
// 512 bytes that stay zero (nothing writes them): where a K-major tile reaches
// past the last reduction row, its rows are loaded from here, and so is the second
// K tile of a reduction that has one
static __device__ __attribute__((aligned(256))) bf16_t ring_zero_row[256];

// A reduction in up to three parts (SEGMENTS), C = A0 . B0^T + A1 . B1^T + ...: K is one
// part's, and part i of an operand lies where its K tiles, counted through, are off by
// a_at[i] and b_at[i] elements.
struct RingSegments {
  int count = 1, tiles = 0;       // parts, K tiles of each
  int64_t a_at[3] = {}, b_at[3] = {};
};

// (the pieces of the kernel are lambdas over its registers: one that the compiler
// left out of line would move them to memory)
#define RING_INLINE __attribute__((always_inline))

template <bool RELU, bool GATHER = false, bool KMAJOR = false,
          bool MASKED = false, bool LISTED = false, bool TAILS = false,
          bool SPLIT = false, bool DEEP = false, bool SEGMENTS = false>
__global__ __launch_bounds__(RingCfg::THREADS) void grouped_gemm_bf16_ring_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
    bf16_t* __restrict__ Cout, int R, int N, int K, int tiles_m, int tiles_n,
    int total_tiles, const int32_t* __restrict__ row_map,
    const bf16_t* __restrict__ zero_row,
    const bf16_t* __restrict__ mask_src,
    const int32_t* __restrict__ tile_list,
    const int32_t* __restrict__ row_count,
    float mask_scale, float* __restrict__ partial,
    int whole_tiles, int split, int tile_rows, int64_t a_stride,
    RingSegments segments) {
  using Cfg = RingCfg;
  // row_count [E], optional: KMAJOR kernels take it as the reduction extent
  // per expert (k_extent)
  const int32_t* k_extent = KMAJOR ? row_count : nullptr;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, WN = Cfg::WN;
  static_assert(!DEEP || (TAILS && !KMAJOR && !LISTED && !SPLIT), "low row tiles");
  static_assert(!SEGMENTS || (TAILS && !KMAJOR && !GATHER && !LISTED && !MASKED), "");
  constexpr int A_BYTES = DEEP ? Cfg::DEEP_A_BYTES : Cfg::A_BYTES;
  constexpr int A_SLOTS = DEEP ? 3 : Cfg::A_SLOTS;
  // loads of a token tile per wavefront (DEEP: the third is half a one)
  constexpr int A_LOADS = DEEP ? 3 : Cfg::A_INSTR;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  // PERSISTENT blocks: one per CU, each walks a strided list of tiles, whose K tiles
  // follow each other without a gap: the loads of a tile's last two K tiles are the
  // next tile's first (see last_tile).  Block b runs on XCD b % 8.  The P = blocks / 8 blocks of an XCD
  // hold P consecutive logical tiles at any moment (shared panels in its L2),
  // and consecutive groups of P tiles go to consecutive XCDs: the whole chip
  // then works on the same one or two experts, whose token panels every XCD
  // re-reads from the memory-side cache, instead of on eight experts at once
  // (1 % faster than giving each XCD a contiguous eighth of the tiles).
  const int nblk = gridDim.x;
  if constexpr (LISTED) total_tiles = tile_list[-1];
  // TAILS: in its round k a block takes the tile k places further (cyclically)
  // among its XCD's P tiles of the round, so that it meets every row tile of
  // the experts in turn, full and partly empty ones: with a fixed place and an
  // even number of row tiles half of the blocks would only ever get the cheap
  // last row tiles and run ahead of the blocks they share weight panels with.
  const int xcd_tiles = nblk >> 3;
  int round_first = (blockIdx.x & 7) * xcd_tiles, place = blockIdx.x >> 3;
  const int tile = round_first + place;
  if (tile >= total_tiles) return;
  // the block's tile of the round after the last one asked for
  auto following_tile = [&]() {
    round_first += nblk;
    if (TAILS) place = place + 1 == xcd_tiles ? 0 : place + 1;
    return round_first + place;
  };

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int tiles_per_e = tiles_m * tiles_n;

  // what the K loop and the output of a tile need to know about it
  struct Tile {
    // K tiles of its reduction: all of K, or with k_extent (KMAJOR) the expert's
    // first k_extent[e] reduction rows only
    int nk;
    int empty;           // k_extent[e] == 0: the result is zero
    int unit;            // SPLIT: its place among the partial results (-1: a whole tile)
    int row0, col0;
    bf16_t* out;         // the expert's rows of C
    // TAILS: 32-row pieces of this wavefront's sub-tile that hold rows of the
    // tile, and of the sub-tiles of the upper half
    int pieces, pieces0;
  };

  // the tile that is being loaded: two K tiles ahead of the one that is multiplied
  const bf16_t *Ae, *Be;
  // Where a load's 16 bytes lie: a part that is the same for the wavefront, in
  // scalar registers, and this lane's.  Load j fills the rows 8 (wave + WAVES j) + l / 8
  // of an LDS tile (KMAJOR: 2 (wave + WAVES j) + l / 32).
  //   a_row[j]   GATHER: the row of A (negative: zero_row); else (not KMAJOR) the
  //              bytes to this lane's chunk of its row
  //   a_lane, b_lane   KMAJOR: elements to this lane's chunk in the pair of rows;
  //              else b_lane: bytes to its chunk in the eight rows
  //   b_row[j]   not KMAJOR: elements to the first of the eight rows
  uint32_t a_row[A_LOADS], a_lane = 0, b_lane = 0;
  int b_row[Cfg::B_INSTR];
  int kt0 = 0;           // SPLIT: its first K tile
  // first row of row tile tm, and the place in it of LDS tile row `row`
  auto tile_row0 = [&](int tm) { return TAILS ? tm * tile_rows : tm * BM; };
  auto tile_pieces0 = [&](int tm) {
    const int valid = min(tile_rows, R - tm * tile_rows);
    return (((valid + 31) >> 5) + 1) >> 1;
  };
  // (rows that are not multiplied: a row of the tile that another lane loads)
  auto row_in_tile = [&](int row, int p0, int tm) {
    if (!TAILS) return row;
    const int last = min(tile_rows, R - tm * tile_rows) - 1;
    if (DEEP) return min(row, last);
    return row >= BM / 2 ? min(row - BM / 2 + 32 * p0, last)
                         : min(row, min(32 * p0 - 1, last));
  };
  // LDS row that lane l's 16 bytes of load j belong to
  auto lds_row = [&](int j, int l) {
    return DEEP && j == 2 ? 128 + wave * 4 + ((l & 31) >> 3)
                          : (wave + Cfg::WAVES * j) * 8 + (l >> 3);
  };
  // logical tile -> expert, row tile, column tile
  auto tile_coords = [&](int logical, int& e, int& tm, int& tn) RING_INLINE {
    e = logical / tiles_per_e;
    const int rem = logical - e * tiles_per_e;
    tn = rem / tiles_m;
    tm = rem - tn * tiles_m;
    if (!LISTED) ring_tile_blocks(rem, tiles_m, tiles_n, tm, tn);
  };
  // the chunk that goes to 16-byte position l % 8 of the lane's rows: rows
  // 8 (wave + 8 j) + l / 8, whose swizzle does not depend on j
  static_assert(Cfg::WAVES % 2 == 0, "the swizzle of a lane's rows");
  auto chunk_of = [&](int l) {
    return ((l & 7) ^ lds_swizzle(wave * 8 + (l >> 3))) * 8;
  };
  const int a_chunk = chunk_of(lane);
  // (DEEP: of load 2, whose rows are four per wavefront)
  auto chunk2_of = [&](int l) { return ((l & 7) ^ lds_swizzle(lds_row(2, l))) * 8; };
  const int a_chunk2 = DEEP ? chunk2_of(lane) : 0;
  if constexpr (!KMAJOR) b_lane = (uint32_t)((lane >> 3) * K + a_chunk) * 2;
  // (What a step of the tile loop outside its K loop computes from the lane index, it
  // computes from a copy that the compiler cannot see through: done once ahead of
  // the tile loop it would be live across the K loop, which has no registers to
  // spare.)
  auto lane_again = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  // GATHER: the slot -> token map entries of the four rows this lane loads in a
  // tile.  They are asked for a whole tile ahead of their use.
  int map_src[A_LOADS];
  auto fetch_map = [&](int logical) RING_INLINE {
    if constexpr (GATHER) {
      int e, tm, tn;
      tile_coords(logical, e, tm, tn);
      const int p0 = TAILS ? tile_pieces0(tm) : 0;
      const int s_lane = lane_again();
#pragma unroll
      for (int j = 0; j < A_LOADS; ++j) {
        const int row = row_in_tile(lds_row(j, s_lane), p0, tm);
        map_src[j] = row_map[(int64_t)e * R + min(tile_row0(tm) + row, R - 1)];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // (logical: an entry of the tile list where there is one)
  auto set_tile = [&](int logical) RING_INLINE {
    Tile t;
    const int s_lane = lane_again();
    int part = 0;
    t.unit = -1;
    if constexpr (SPLIT) {
      const int unit = logical - whole_tiles;
      if (unit >= 0) {
        t.unit = unit;
        const int split_tiles = (total_tiles - whole_tiles) / split;
        part = unit / split_tiles;
        logical = whole_tiles + unit - part * split_tiles;
      }
    }
    int e, tm, tn;
    tile_coords(logical, e, tm, tn);
    if constexpr (TAILS) {
      const int valid = min(tile_rows, R - tm * tile_rows);
      const int blocks = (valid + 31) >> 5;
      t.pieces0 = (blocks + 1) >> 1;
      t.pieces = wm == 0 ? t.pieces0 : blocks - t.pieces0;
    } else {
      t.pieces0 = t.pieces = Cfg::TM;
    }
    const int row0 = t.row0 = tile_row0(tm);
    const int col0 = t.col0 = tn * BN;
    int nk = KMAJOR ? (K + BK - 1) / BK : K / BK;
    if constexpr (SEGMENTS) nk *= segments.count;
    t.empty = false;
    if constexpr (KMAJOR && !SPLIT) {
      if (k_extent != nullptr) {
        const int used = k_extent[e];
        t.empty = used == 0;
        nk = max(1, min(nk, (used + BK - 1) / BK));
      }
    }
    if constexpr (SPLIT) {
      kt0 = 0;
      if (t.unit >= 0) {
        const int all = nk;
        kt0 = (int)((int64_t)all * part / split);
        nk = (int)((int64_t)all * (part + 1) / split) - kt0;
        if (nk == 0) {     // fewer K tiles than parts
          nk = 1;
          kt0 = 0;
          t.empty = true;
        }
      }
    }
    t.nk = nk;
    // (a_stride 0: all experts read the same rows, -1: each its own)
    if constexpr (GATHER) Ae = A;
    else if constexpr (LISTED || MASKED) Ae = A + (int64_t)e * R * K;
    else Ae = A + e * (a_stride < 0 ? (int64_t)R * K : a_stride);
    Be = B + (int64_t)e * N * K;
    t.out = Cout + (int64_t)e * R * N;
    if constexpr (KMAJOR) {
      // lane l fills 16-byte position l % 32 of its row with the chunk that
      // belongs there under the unit swizzle
      const int p = s_lane & 31, k_row = wave * 2 + (s_lane >> 5);
      const int chunk = ((((p >> 2) ^ (k_row & 3)) << 2) | (p & 3)) * 8;
      // (TAILS: what lies past the tile's rows is not multiplied; its lanes
      // fetch the tile's last piece again)
      const int row_chunk = TAILS ? min(chunk, tile_rows - 8) : chunk;
      a_lane = k_row * R + min(row0 + row_chunk, R - 8);
      b_lane = k_row * N + min(col0 + chunk, N - 8);
    } else {
#pragma unroll
      for (int j = 0; j < A_LOADS; ++j) {
        const int row = lds_row(j, s_lane);
        if constexpr (GATHER)
          a_row[j] = map_src[j];
        else
          a_row[j] = (uint32_t)(min(row0 + row_in_tile(row, t.pieces0, tm), R - 1) * K +
                                (DEEP && j == 2 ? chunk2_of(s_lane)
                                                : chunk_of(s_lane))) * 2;
      }
#pragma unroll
      for (int j = 0; j < Cfg::B_INSTR; ++j)
        // (N % 8 == 0: eight rows exist or they do not)
        b_row[j] = min(col0 + (wave + Cfg::WAVES * j) * 8, N - 8) * K;
    }
    return t;
  };
  // load j of the token (A, two slots at LDS offset 0, DEEP: three) / weight (B,
  // three slots behind them) tile kt; `zeros`: of a K tile of zeros instead
  constexpr int B_BASE = A_SLOTS * A_BYTES;
  // KMAJOR: load j of a tile fills reduction rows 2 (wave + WAVES j) and + 1
  // (lanes 32-63) of it; past the last reduction row they are zeros
  auto kmajor_past_end = [&](int kt, int j) {
    return (kt0 + kt) * BK + (wave + Cfg::WAVES * j) * 2 + (lane >> 5) >= K;
  };
  auto kmajor_row = [&](int kt, int j) {
    return (int64_t)((kt0 + kt) * BK + Cfg::WAVES * j * 2);
  };
  // SEGMENTS: elements from where K tile kt would follow K tile 0 to where it lies
  auto segment_of = [&](int kt) {
    return kt < segments.tiles ? 0 : kt < 2 * segments.tiles ? 1 : 2;
  };
  auto load_a = [&](int kt, int slot, int j, bool zeros = false) RING_INLINE {
    const bf16_t* src;
    const int64_t jump = SEGMENTS ? segments.a_at[segment_of(kt)] : 0;
    if constexpr (KMAJOR)
      src = Ae + kmajor_row(kt, j) * R + a_lane;
    else if constexpr (GATHER)
      src = ((int)a_row[j] < 0 ? zero_row : Ae + (int64_t)(int)a_row[j] * K) +
            ((DEEP && j == 2 ? a_chunk2 : a_chunk) + kt * BK);
    else
      src = (const bf16_t*)((const char*)(Ae + (jump + kt * BK)) + a_row[j]);
    if (zeros || (KMAJOR && kmajor_past_end(kt, j)))
      src = ring_zero_row + ((KMAJOR ? lane : lane_again()) & 31) * 8;
    if (DEEP && j == 2) {
      if (lane < 32)
        __builtin_amdgcn_global_load_lds(
            (glb_void_t*)src,
            (lds_void_t*)(smem_raw + slot * A_BYTES + 128 * Cfg::ROW_BYTES +
                          wave * 512), 16, 0, 0);
      return;
    }
    __builtin_amdgcn_global_load_lds(
        (glb_void_t*)src,
        (lds_void_t*)(smem_raw + slot * A_BYTES +
                      (wave + Cfg::WAVES * j) * 1024), 16, 0, 0);
  };
  auto load_b = [&](int kt, int slot, int j, bool zeros = false) RING_INLINE {
    const bf16_t* src;
    const int64_t jump = SEGMENTS ? segments.b_at[segment_of(kt)] : 0;
    if constexpr (KMAJOR)
      src = Be + kmajor_row(kt, j) * N + b_lane;
    else
      src = (const bf16_t*)((const char*)(Be + b_row[j] + (jump + kt * BK)) + b_lane);
    if (zeros || (KMAJOR && kmajor_past_end(kt, j)))
      src = ring_zero_row + ((KMAJOR ? lane : lane_again()) & 31) * 8;
    __builtin_amdgcn_global_load_lds(
        (glb_void_t*)src,
        (lds_void_t*)(smem_raw + B_BASE + slot * Cfg::B_BYTES +
                      (wave + Cfg::WAVES * j) * 1024), 16, 0, 0);
  };

  f32x16_t acc[Cfg::TM][Cfg::TN];

  const int fr = lane & 31, fc = lane >> 5;
  int a_frag[BK / 16], b_frag[BK / 16];
  // KMAJOR: byte offset of this lane's 8 bytes for 32-column block n of its
  // wavefront's sub-tile, at step 0 / first half: a_frag[n], b_frag[n].  The rows
  // of the tile lie in LDS as they do in memory: the lower half's pieces (TAILS)
  // follow the upper half's.
  auto kmajor_inner = [&]() {
    const int t = lane & 15, g = lane >> 4;
    return ((g & 1) * 16 + 4 * (t & 3)) * 2 + ((g >> 1) * 8 + (t >> 2)) * 512;
  };
  auto set_a_frag = [&](int pieces0) {
    const int first = wm == 0 ? 0 : pieces0;
#pragma unroll
    for (int n = 0; n < Cfg::TM; ++n)
      a_frag[n] = (((first + n) ^ ((lane & 15) >> 2)) * 64) + kmajor_inner();
  };
  if constexpr (KMAJOR) {
    static_assert(Cfg::TM <= BK / 16 && Cfg::TN <= BK / 16, "offset arrays");
    if constexpr (!TAILS) set_a_frag(Cfg::TM);
#pragma unroll
    for (int n = 0; n < Cfg::TN; ++n)
      b_frag[n] =
          (((wn * Cfg::TN + n) ^ ((lane & 15) >> 2)) * 64) + kmajor_inner();
  } else {
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      const int col = ((kk * 2 + fc) ^ lds_swizzle(fr)) * 16;
      a_frag[kk] = ((DEEP ? 0 : wm * Cfg::WTM) + fr) * Cfg::ROW_BYTES + col;
      b_frag[kk] = (wn * Cfg::WTN + fr) * Cfg::ROW_BYTES + col;
    }
  }
  constexpr int KSTEPS = BK / 16;
  bf16x8_t fa[2][Cfg::TM], fb[2][Cfg::TN];
  // 8 consecutive k of one column of a K-major tile: two transposed reads at
  // LDS byte address `at` + 8192 kk (+ 2048 for the second four).  Written as
  // asm because the compiler puts a vmcnt(0) in front of the builtin form (it
  // takes the read for a possible LDS store racing the direct-to-LDS loads),
  // which would drain the loads that are meant to stay in flight.  The
  // compiler therefore does not know when the data arrives: wait_frags()
  // (lgkmcnt(0)) stands before the MFMAs that use it.
  const uint32_t lds0 = (uint32_t)(size_t)(lds_void_t*)smem_raw;
  auto read_tr = [&](uint32_t at, int kk) RING_INLINE {
    i16x4_t lo, hi;
    switch (kk) {
      case 0: lds_read_tr16_pair<0>(at, lo, hi); break;
      case 1: lds_read_tr16_pair<8192>(at, lo, hi); break;
      case 2: lds_read_tr16_pair<16384>(at, lo, hi); break;
      default: lds_read_tr16_pair<24576>(at, lo, hi); break;
    }
    return __builtin_bit_cast(
        bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto wait_frags = [&]() RING_INLINE {
    if constexpr (KMAJOR) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0) only
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // DEEP: the lower half's rows follow the upper half's pieces
  int a_half = 0;
  // token fragment of piece n / weight fragment n of MFMA step kk
  auto read_a = [&](int aslot, int kk, int n) RING_INLINE -> bf16x8_t {
    if constexpr (KMAJOR)
      return read_tr(lds0 + aslot * A_BYTES + a_frag[n], kk);
    else
      return *reinterpret_cast<const bf16x8_t*>(
          smem_raw + (aslot * A_BYTES + a_half) + a_frag[kk] +
          n * 32 * Cfg::ROW_BYTES);
  };
  auto read_b = [&](int bslot, int kk, int n) RING_INLINE -> bf16x8_t {
    if constexpr (KMAJOR)
      return read_tr(lds0 + B_BASE + bslot * Cfg::B_BYTES + b_frag[n], kk);
    else
      return *reinterpret_cast<const bf16x8_t*>(
          smem_raw + B_BASE + bslot * Cfg::B_BYTES + b_frag[kk] +
          n * 32 * Cfg::ROW_BYTES);
  };
  // fragment read n of a step: 0..TM-1 token rows, TM..TM+TN-1 weight rows
  auto read_frag = [&](int aslot, int bslot, int kk, int buf, int n) RING_INLINE {
    if (n < Cfg::TM) fa[buf][n] = read_a(aslot, kk, n);
    else fb[buf][n - Cfg::TM] = read_b(bslot, kk, n - Cfg::TM);
  };
  // (first: the sums begin)
  auto mfma = [&](int buf, int n, bool first = false) RING_INLINE {
    const int i = n / Cfg::TN, j = n % Cfg::TN;
    const f32x16_t none = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                           0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        fb[buf][j], fa[buf][i], first ? none : acc[i][j], 0, 0, 0);
  };
  // with NA of the wavefront's TM row pieces in use: is fragment read n /
  // MFMA n of a step needed?
  auto frag_used = [](int na, int n) {
    return na > 0 && (n >= Cfg::TM || n < na);
  };
  auto mfma_used = [](int na, int n) { return n / Cfg::TN < na; };
  // nothing moves across: the instruction order below is the issue order
  auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };
  // fragment reads in the order the MFMAs (token tile i = n / TN outer, weight
  // tile j = n % TN inner) first need them: a0 b0 b1 a1 a2 a3
  constexpr int RD[6] = {0, Cfg::TM, Cfg::TM + 1, 1, 2, 3};

  // Output lines: 16 bytes per lane, eight rows of 128 bytes per store.  `base`
  // is the first of the eight rows, `rows` how many of them are rows of the output
  // (what the buffer's range drops; a store leaves in any case, the waits count
  // on that), line_at this lane's place, out of range where the columns end.
  constexpr int STORES = 4;       // per 32-row piece
  constexpr uint32_t OUTSIDE = 0x80000000u;    // (8 rows of N < 2^25 end before)
  auto store_line = [&](u32x4_t v, bf16_t* base, int rows, uint32_t line_at)
      RING_INLINE {
    rows = max(rows, 0);
    asm("" : "+s"(rows));    // (scalar: not one clamp in the vector unit)
    const int bytes = min(rows, 8) * N * 2;
    __builtin_amdgcn_raw_buffer_store_b128(
        v, __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00027000), line_at,
        0, 0);
  };
  // slots of the K tile that is multiplied, and the K tile (of the tile that is
  // being loaded) that its loads fetch
  int aslot = 0, bslot = 0, lk = 2;
  // FIRST: K tile 0
  auto next_a_slot = [&](int slot) {
    if constexpr (A_SLOTS == 2) return slot ^ 1;
    else return slot == A_SLOTS - 1 ? 0 : slot + 1;
  };
  auto k_tile = [&](auto first_tag, auto na_tag) RING_INLINE {
    constexpr bool FIRST = decltype(first_tag)::value;
    constexpr int NA = decltype(na_tag)::value;      // row pieces in use
    auto rd = [&](int as, int bs, int kk, int buf, int n) {
      if (frag_used(NA, n)) read_frag(as, bs, kk, buf, n);
    };
    int kk_now = 0;
    auto mm = [&](int buf, int n) {
      if (mfma_used(NA, n)) mfma(buf, n, FIRST && kk_now == 0);
    };
    const int bnext = bslot == 2 ? 0 : bslot + 1;       // slot of the next K tile
    const int bnext2 = bnext == 2 ? 0 : bnext + 1;      // of the one after it
    const int anext = next_a_slot(aslot), anext2 = next_a_slot(anext);
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) {
      const int cur = kk & 1, nxt = cur ^ 1;
      kk_now = kk;
      // The loads a step carries.  Two token slots: the four weight loads of the K
      // tile after the next over steps 0..2, all four token loads of it in step 3,
      // behind the hand-over barrier that frees their slot (a full K tile ahead of
      // use).  DEEP: all seven of them over steps 0..2, into slots that the hand-over
      // barrier of the K tile before freed (step 3 carries none).
      auto load = [&](int which) {
        if constexpr (DEEP) {
          const int n = 2 * kk + which;       // 0 .. 6
          if (kk == 3) return;
          if (n < 3) load_a(lk, anext2, n);
          else load_b(lk, bnext2, n - 3);
          return;
        }
        if (which > 1 && kk < 3) return;
        if (kk == 0) load_b(lk, bnext2, which);
        if (kk == 1 && which == 0) load_b(lk, bnext2, 2);
        if (kk == 2 && which == 0) load_b(lk, bnext2, 3);
        if (kk == 3) load_a(lk, aslot, which);
      };
      if (kk + 1 < KSTEPS) {
        // 6 fragment reads of step kk+1 (in the order its MFMAs need them),
        // 2 loads, 8 MFMAs of step kk
        fence();
        wait_frags();
        rd(aslot, bslot, kk + 1, nxt, RD[0]);
        rd(aslot, bslot, kk + 1, nxt, RD[1]);
        mm(cur, 0); fence();
        rd(aslot, bslot, kk + 1, nxt, RD[2]);
        mm(cur, 1); fence();
        load(0);
        mm(cur, 2); fence();
        rd(aslot, bslot, kk + 1, nxt, RD[3]);
        mm(cur, 3); fence();
        rd(aslot, bslot, kk + 1, nxt, RD[4]);
        mm(cur, 4); fence();
        load(1);
        mm(cur, 5); fence();
        rd(aslot, bslot, kk + 1, nxt, RD[5]);
        mm(cur, 6); fence();
        if (DEEP && kk == 2) { load(2); fence(); }
        mm(cur, 7); fence();
      } else {
        // this lane holds the last step's fragments (lgkmcnt 0); everything but the
        // loads of tile kt+2 that are out has landed: the four weight loads, whose
        // token loads follow this barrier (vmcnt 4), DEEP all seven (vmcnt 7)
        fence();
        constexpr int AHEAD = DEEP ? A_LOADS + Cfg::B_INSTR : Cfg::B_INSTR;
        __builtin_amdgcn_s_waitcnt((AHEAD & 15) | (0 << 8) | (7 << 4));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fence();
        // fragment reads first: a load right behind the barrier would queue
        // up with the other wavefronts' and hold this one's MFMAs back
#pragma unroll
        for (int n = 0; n < 6; ++n) {
          rd(anext, bnext, 0, nxt, RD[n]);
          if (n >= 2) load(n - 2);
          mm(cur, n); fence();
        }
        mm(cur, 6); fence();
        mm(cur, 7); fence();
      }
    }
    aslot = anext;
    bslot = bnext;
    ++lk;
  };

  // The last K tile of a tile, its output, and the hand-over to the next tile.
  //
  // The K tile is multiplied piece by piece (32 rows of the wavefront's sub-tile):
  // step 0 of all pieces, then steps 1 to 3 of one after the other, and while the
  // matrix pipe is at piece i + 1, piece i is rounded (and relu), turned round in
  // LDS and stored, 16 bytes per lane and whole 128-byte lines.  Each wavefront
  // turns its pieces round by itself, without barriers, in the four kilobytes of
  // the free weight slot that its own loads of the next tile's K tile 1 fill
  // afterwards.  By then K tile 0 of the next tile has been on its way for a whole K
  // tile, so the matrix pipes go on with it at once, and the stores have that
  // much time before anything waits for them.
  //
  // A tile's output used to be staged by all wavefronts in two passes behind block
  // barriers, with the ring drained and nothing multiplied, 6.5 us a tile.  Before and
  // now, back to back: 16384 rows, 1024 -> 4096 126 -> 118 us, -> 1024 34.4 -> 31.3;
  // 16 x 705 rows, 768 -> 3072 62 -> 53; 64 x 512 rows, 1024 -> 4096 270 -> 260; weight
  // gradients of 64 x 512 rows 312 -> 293.  Without stores and staging the same
  // launches take 103, 26.6, 46, 229 and 229.  (A compute unit's 128 KB take 4.7 us when
  // the whole chip stores, 2.7 if they stay in the L2s.)  Twelve of the sixteen stores
  // held back for the next three K tiles are no faster.  Turned round in registers
  // (v_permlane32_swap, v_permlane16_swap) instead of LDS a store covers rows of 64
  // bytes, which cost the L2 1.4 times as long: weight gradients 293 -> 309.
  const uint32_t lds_base = (uint32_t)(size_t)(lds_void_t*)smem_raw;
  // The fragments of a tile's first step: read right behind the hand-over, or (TAILS:
  // the wavefront's pieces in the next tile are another copy of the code) ahead of
  // its first K tile.
  auto first_frags = [&](int as, int bs, int na) RING_INLINE {
#pragma unroll
    for (int n = 0; n < 6; ++n)
      if (frag_used(na, RD[n])) read_frag(as, bs, 0, 0, RD[n]);
  };
  auto last_tile = [&](const Tile& t, const Tile& after, bool has_next,
                       auto na_tag) RING_INLINE {
    constexpr int NA = decltype(na_tag)::value;
    constexpr int TN = Cfg::TN;
    static_assert(Cfg::TM == 4 && TN == 2 && KSTEPS == 4 && Cfg::WTN == 64,
                  "a piece is 32 rows of 128 bytes");
    const int bnext = bslot == 2 ? 0 : bslot + 1;       // K tile 0 of the next tile
    const int bfree = bnext == 2 ? 0 : bnext + 1;       // K tile 1: free till then
    const int anext = next_a_slot(aslot), afree = next_a_slot(anext);
    bf16x8_t ga[2][KSTEPS - 1], gb[KSTEPS - 1][TN];
    auto mm = [&](int i, int n) {
      const int kk = n / TN, j = n % TN;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gb[kk][j], ga[i & 1][kk],
                                                          acc[i][j], 0, 0, 0);
    };
    const int e_lane = lane_again();
    // Writes: row l % 32, 8-byte unit 2 c + l / 32 of it at unit (2 c + l / 32) ^
    // (2 (row % 8) + row / 8 % 2); reads: row 8 n + l / 8, chunk l % 8, whose two
    // units are exchanged where n is odd.  Both spread over all banks.
    const uint32_t stage = lds_base + B_BASE + bfree * Cfg::B_BYTES + wave * 1024;
    const int w_row = e_lane & 31;
    const uint32_t w_at =
        stage + (w_row >> 3) * (Cfg::WAVES * 1024) + (w_row & 7) * 128 +
        (((e_lane >> 5) ^ ((w_row & 7) * 2) ^ ((w_row >> 3) & 1)) * 8);
    const int r_row = e_lane >> 3, r_chunk = e_lane & 7;
    const uint32_t r_at = stage + r_row * 128 + ((r_chunk ^ r_row) * 16);
    const int first_row = t.row0 + (wm == 0 ? 0 : TAILS ? 32 * t.pieces0 : Cfg::WTM);
    const int end_row = TAILS ? min(R, t.row0 + tile_rows) : R;
    const int col = t.col0 + wn * Cfg::WTN + r_chunk * 8;
    bf16_t* const out = t.out + (int64_t)first_row * N + t.col0 + wn * Cfg::WTN;
    const uint32_t line_at =
        col < N ? (uint32_t)(r_row * N + r_chunk * 8) * 2 : OUTSIDE;
    u32x4_t mask[2][MASKED ? STORES : 1];
    auto load_mask = [&](int i) {
      if constexpr (MASKED) {
        const bf16_t* m = mask_src + (t.out - Cout) + min(col, N - 8);
#pragma unroll
        for (int n = 0; n < STORES; ++n)
          mask[i & 1][n] = *reinterpret_cast<const u32x4_t*>(
              m + (int64_t)min(first_row + 32 * i + 8 * n + r_row, R - 1) * N);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    const bool part = SPLIT && t.unit >= 0;
    // piece i, two of its eight groups of 4 columns per lane
    auto put = [&](int i, int g) {
      if (part) return;
#pragma unroll
      for (int c = 2 * g; c < 2 * g + 2; ++c) {
        const int j = c >> 2, q = c & 3;
        u32x2_t v;
        v.x = pack2_bf16(acc[i][j][4 * q + 0], acc[i][j][4 * q + 1], RELU);
        v.y = pack2_bf16(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3], RELU);
        lds_write_b64_asm(w_at ^ (16 * c), v);
      }
    };
    u32x4_t line[STORES];
    auto get = [&]() {
      if (!part) lds_read_lines(line, r_at);
    };
    // line n of piece i as it goes to memory
    auto finished = [&](int i, int n) {
      u32x4_t v = line[n];
      if (n & 1) v = __builtin_shufflevector(v, v, 2, 3, 0, 1);
      if constexpr (MASKED) {
        const u32x4_t hm = mask[i & 1][n];
        if (mask_scale != 1.0f) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            v[q] = f32x2_to_bf16x2(
                __builtin_bit_cast(float, v[q] << 16) * mask_scale,
                __builtin_bit_cast(float, v[q] & 0xffff0000u) * mask_scale);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t keep =
              (__builtin_bit_cast(float, hm[q] << 16) > 0.f ? 0xffffu : 0u) |
              (__builtin_bit_cast(float, hm[q] & 0xffff0000u) > 0.f
                   ? 0xffff0000u : 0u);
          v[q] &= keep;
        }
      }
      return v;
    };
    auto store = [&](int i) {
      if (part) {
        // a part of a tile's reduction: the accumulators as they lie, 16
        // bytes per lane and register group; split_reduce_kernel adds the
        // parts and knows the layout
        float* dst = partial + (int64_t)t.unit * (BM * BN) +
                     (wave * 64 + e_lane) * 4;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(
                dst + ((i * TN + j) * 4 + q) * (Cfg::THREADS * 4)) =
                make_float4(acc[i][j][4 * q + 0], acc[i][j][4 * q + 1],
                            acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
        return;
      }
#pragma unroll
      for (int n = 0; n < STORES; ++n) {
        store_line(finished(i, n), out + (int64_t)(32 * i + 8 * n) * N,
                   end_row - first_row - 32 * i - 8 * n, line_at);
      }
    };
    auto zero_if_empty = [&](int i) {
      if constexpr (KMAJOR || SPLIT) {
        // an expert without reduction rows: its one K tile held rows that
        // nobody wrote
        if (t.empty) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
        }
      }
    };

    if constexpr (NA > 0) {
      // step 0 of all pieces; meanwhile the fragments of piece 0's step 1
      fence();
      wait_frags();
      ga[0][0] = read_a(aslot, 1, 0);
#pragma unroll
      for (int j = 0; j < TN; ++j) gb[0][j] = read_b(bslot, 1, j);
      fence();
#pragma unroll
      for (int m = 0; m < NA * TN; ++m) { mfma(0, m); fence(); }
      load_mask(0);
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        fence();
        wait_frags();
        if (i == 0) {
          // (the fragments of piece 0's steps 2 and 3)
#pragma unroll
          for (int kk = 2; kk < KSTEPS; ++kk) {
            ga[0][kk - 1] = read_a(aslot, kk, 0);
#pragma unroll
            for (int j = 0; j < TN; ++j) gb[kk - 1][j] = read_b(bslot, kk, j);
          }
          fence();
        }
        mm(i, 0); fence();
        mm(i, 1); fence();
        if (i == 0) wait_frags();
        if (i + 1 < NA) {
#pragma unroll
          for (int kk = 1; kk < KSTEPS; ++kk)
            ga[(i + 1) & 1][kk - 1] = read_a(aslot, kk, i + 1);
          fence();
        }
        if (i > 0) { zero_if_empty(i - 1); put(i - 1, 0); put(i - 1, 1); }
        mm(i, 2); fence();
        if (i > 0) { put(i - 1, 2); put(i - 1, 3); }
        mm(i, 3); fence();
        if (i > 0) get();
        mm(i, 4); fence();
        if (i > 0) store(i - 1);
        mm(i, 5); fence();
        if (i + 1 < NA) load_mask(i + 1);
      }
    }
    // Hand-over: the fragments of this tile are in registers, and all but the
    // stores that came after the loads of the next tile's K tile 0 are done.
    fence();
    constexpr int LATER = NA > 1 ? STORES * (NA - 1) : 0;
    __builtin_amdgcn_s_waitcnt((LATER & 15) | (0 << 8) | (7 << 4));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fence();
    // (K tile 1 as a number that the compiler does not know: it would keep K tile 0's
    // addresses to add to)
    int kt1 = 1;
    asm volatile("" : "+s"(kt1));
    if (has_next) {
#pragma unroll
      for (int j = 0; j < A_LOADS; ++j) load_a(kt1, afree, j, after.nk < 2);
    }
    fence();
    if constexpr (!TAILS) first_frags(anext, bnext, Cfg::TM);
    fence();
    if constexpr (NA > 0) {
      zero_if_empty(NA - 1);
#pragma unroll
      for (int g = 0; g < 4; ++g) put(NA - 1, g);
      get();
      store(NA - 1);
    }
    wait_frags();
    fence();
    if (has_next) {
#pragma unroll
      for (int j = 0; j < 4; ++j) load_b(kt1, bfree, j, after.nk < 2);
    }
    fence();
    aslot = anext;
    bslot = bnext;
    lk = 2;
  };

  // The block's next tile and the one after it: their numbers in the list where
  // there is one, read ahead of their use.
  auto entry_of = [&](int number) {
    if constexpr (LISTED) return tile_list[min(number, total_tiles - 1)];
    else return number;
  };
  Tile t = [&]() {
    const int entry = entry_of(tile);
    fetch_map(entry);
    return set_tile(entry);
  }();
  int next = following_tile(), next2 = following_tile();
  int next_entry = entry_of(next), next2_entry = entry_of(next2);
  if (next < total_tiles) fetch_map(next_entry);
#pragma unroll
  for (int j = 0; j < A_LOADS; ++j) load_a(0, 0, j);
#pragma unroll
  for (int j = 0; j < 4; ++j) load_b(0, 0, j);
#pragma unroll
  for (int j = 0; j < 4; ++j) load_b(1, 1, j, t.nk < 2);
#pragma unroll
  for (int j = 0; j < A_LOADS; ++j) load_a(1, 1, j, t.nk < 2);
  // K tile 0 has landed: only tile 1 may still be in flight
  wait_vmcnt<A_LOADS + Cfg::B_INSTR>();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if constexpr (!TAILS) first_frags(0, 0, Cfg::TM);
  wait_frags();
  for (;;) {
    if constexpr (KMAJOR && TAILS) set_a_frag(t.pieces0);
    if constexpr (DEEP) a_half = wm == 0 ? 0 : t.pieces0 * 32 * Cfg::ROW_BYTES;
    const bool has_next = next < total_tiles;
    Tile after = t;
    auto tile_pass = [&](auto na_tag) RING_INLINE {
      if constexpr (TAILS) {
        first_frags(aslot, bslot, decltype(na_tag)::value);
        wait_frags();
      }
      // The loads of the last two K tiles are the next tile's.  (Its map entries are
      // older than the eight loads of a K tile that are in flight.  Without a next
      // tile they are the first of this one again, which nobody reads.)
      auto advance = [&]() RING_INLINE {
        if (has_next) {
          if constexpr (GATHER) wait_vmcnt<A_LOADS + Cfg::B_INSTR>();
          after = set_tile(next_entry);
          if (next2 < total_tiles) fetch_map(next2_entry);
        }
        lk = 0;
      };
      if (t.nk > 2) {
        k_tile(std::true_type{}, na_tag);
        for (int kt = 1; kt < t.nk - 2; ++kt) k_tile(std::false_type{}, na_tag);
        advance();
        k_tile(std::false_type{}, na_tag);
      } else {
        // (two K tiles at least: the second of one holds zeros)
        advance();
        k_tile(std::true_type{}, na_tag);
      }
      last_tile(t, after, has_next, na_tag);
    };
    if constexpr (TAILS) {
      switch (t.pieces) {
        case 0: tile_pass(std::integral_constant<int, 0>{}); break;
        case 1: tile_pass(std::integral_constant<int, 1>{}); break;
        case 2: tile_pass(std::integral_constant<int, 2>{}); break;
        case 3: tile_pass(std::integral_constant<int, 3>{}); break;
        default: tile_pass(std::integral_constant<int, DEEP ? 3 : Cfg::TM>{}); break;
      }
    } else {
      tile_pass(std::integral_constant<int, Cfg::TM>{});
    }
    if (!has_next) break;
    t = after;
    next = next2;
    next_entry = next2_entry;
    next2 = following_tile();
    next2_entry = entry_of(next2);
  }
  // no direct-to-LDS load may outlive the block
  wait_vmcnt<0>();
}

#undef RING_INLINE

// Sums the parts of the split tiles of a ring launch, in part order, rounds
// once and writes the tiles.  One block per (tile, MFMA tile of the
// wavefronts); the parts lie in accumulator order (see the kernel above).
__global__ __launch_bounds__(RingCfg::THREADS) void split_reduce_kernel(
    const float* __restrict__ partial, bf16_t* __restrict__ Cout, int R, int N,
    int tiles_m, int tiles_n, int whole_tiles, int split_tiles, int split) {
  using Cfg = RingCfg;
  constexpr int GROUPS = Cfg::TM * Cfg::TN;
  const int t = blockIdx.x / GROUPS, ij = blockIdx.x - t * GROUPS;
  const int tiles_per_e = tiles_m * tiles_n;
  const int logical = whole_tiles + t;
  const int e = logical / tiles_per_e, rem = logical - e * tiles_per_e;
  int tn = rem / tiles_m, tm = rem - tn * tiles_m;
  ring_tile_blocks(rem, tiles_m, tiles_n, tm, tn);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  const int i = ij / Cfg::TN, j = ij - i * Cfg::TN;
  float4 sum[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) sum[q] = make_float4(0.f, 0.f, 0.f, 0.f);
  const float* src = partial + (int64_t)t * (Cfg::BM * Cfg::BN) +
                     (int64_t)ij * 4 * (Cfg::THREADS * 4) + tid * 4;
  const int64_t part_stride = (int64_t)split_tiles * (Cfg::BM * Cfg::BN);
#pragma unroll 2
  for (int p = 0; p < split; ++p, src += part_stride) {
    float4 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = *reinterpret_cast<const float4*>(src + q * (Cfg::THREADS * 4));
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      sum[q].x += v[q].x; sum[q].y += v[q].y;
      sum[q].z += v[q].z; sum[q].w += v[q].w;
    }
  }
  const int row = tm * Cfg::BM + wm * Cfg::WTM + i * 32 + (lane & 31);
  const int col = tn * Cfg::BN + wn * Cfg::WTN + j * 32 + (lane >> 5) * 4;
  if (row >= R) return;
  bf16_t* dst = Cout + ((int64_t)e * R + row) * N + col;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (col + 8 * q < N)
      *reinterpret_cast<uint2*>(dst + 8 * q) =
          make_uint2(f32x2_to_bf16x2(sum[q].x, sum[q].y),
                     f32x2_to_bf16x2(sum[q].z, sum[q].w));
}

// ---------------------------------------------------------------------------
// Plain FMA tile kernel (float32, and bf16 shapes the MFMA kernel rejects):
// 64 x 64 tile, 16-deep K step, each thread a 4 x 4 patch, float32 accumulate
// in k order.
// ---------------------------------------------------------------------------
template <typename T, bool RELU, typename TO = T>
__global__ __launch_bounds__(256) void grouped_gemm_simple_kernel(
    const T* __restrict__ A, const T* __restrict__ B, TO* __restrict__ Cout,
    int R, int N, int K, int tiles_m, int tiles_n) {
  __shared__ float As[16][64 + 4];
  __shared__ float Bs[16][64 + 4];
  const int tiles_per_e = tiles_m * tiles_n;
  const int e = blockIdx.x / tiles_per_e;
  const int rem = blockIdx.x - e * tiles_per_e;
  const int tn = rem / tiles_m, tm = rem - tn * tiles_m;
  const int row0 = tm * 64, col0 = tn * 64;
  const T* Ae = A + (int64_t)e * R * K;
  const T* Be = B + (int64_t)e * N * K;
  TO* Ce = Cout + (int64_t)e * R * N;
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
  for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int c = tid + i * 256;
      int r = c >> 4, k = c & 15;
      int gr = row0 + r, gc = col0 + r, gk = k0 + k;
      As[k][r] = (gr < R && gk < K) ? load_f32<T>(Ae + (int64_t)gr * K + gk) : 0.f;
      Bs[k][r] = (gc < N && gk < K) ? load_f32<T>(Be + (int64_t)gc * K + gk) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int row = row0 + ty * 4 + i;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      int col = col0 + tx * 4 + j;
      if (row < R && col < N) {
        float v = round_to<TO>(acc[i][j]);
        if (RELU) v = v > 0.f ? v : 0.f;
        store_f32<TO>(Ce + (int64_t)row * N + col, v);
      }
    }
  }
}

// In-place activation on an already rounded tensor, for the activations that
// are not fused into the GEMM epilogue (everything except relu / linear).
template <typename T>
__global__ __launch_bounds__(256) void activation_kernel(T* __restrict__ h,
                                                         int64_t n, int act) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += stride)
    store_f32<T>(h + i, apply_activation(load_f32<T>(h + i), act));
}

// out = act(pre), element by element (what activation_kernel does in place).
template <typename T>
__global__ __launch_bounds__(256) void activation_copy_kernel(
    const T* __restrict__ pre, T* __restrict__ out, int64_t n, int act) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += stride)
    store_f32<T>(out + i, apply_activation(load_f32<T>(pre + i), act));
}

// dh = dh * scale (when given), then dh = (h > 0) ? dh : 0 for ReLU experts --
// the hidden dropout and the ReLU of the forward pass seen from behind (h is
// the stored, already rounded activation: positive iff the pre-activation
// rounded to a positive value and the element was not dropped).
// (const_scale: one factor for every element that stays, in place of a scale
// tensor -- a dropout's noise where the ReLU mask already says which elements
// were kept.)
template <typename T>
__global__ __launch_bounds__(256) void hidden_grad_kernel(
    T* __restrict__ dh, const T* __restrict__ h, const T* __restrict__ scale,
    bool relu, int64_t n, float const_scale) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    if (relu && !(load_f32<T>(h + i) > 0.f)) {
      dh[i] = (T)0;
    } else if (scale) {
      store_f32<T>(dh + i, load_f32<T>(dh + i) * load_f32<T>(scale + i));
    } else if (const_scale != 1.0f) {
      store_f32<T>(dh + i, load_f32<T>(dh + i) * const_scale);
    }
  }
}

// h = h * factor (when given), then dropout: noise = (u < keep) ? inv_keep : 0,
// h = h * noise, each product rounded once to T.
template <typename T>
__global__ __launch_bounds__(256) void hidden_product_kernel(
    T* __restrict__ h, const T* __restrict__ factor,
    const T* __restrict__ uniform, float keep, float inv_keep,
    T* __restrict__ noise_out, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    float v = load_f32<T>(h + i);
    if (factor) {
      store_f32<T>(h + i, v * load_f32<T>(factor + i));
      v = load_f32<T>(h + i);
    }
    if (uniform) {
      const float noise = load_f32<T>(uniform + i) < keep ? inv_keep : 0.f;
      store_f32<T>(h + i, v * noise);
      if (noise_out) store_f32<T>(noise_out + i, noise);
    } 
  }
}

// d(act(v)) / dv in float32, from the pre-activation v.
__device__ __forceinline__ float activation_derivative(float v, int act) {
  switch (act) {
    case MESH_MOE_ACT_RELU:
      return v > 0.f ? 1.0f : 0.0f;
    case MESH_MOE_ACT_GELU: {
      const float k = 0.7978845608028654f;
      const float t = tanhf(k * (v + 0.044715f * v * v * v));
      const float du = k * (1.0f + 3.0f * 0.044715f * v * v);
      return 0.5f * (1.0f + t) + 0.5f * v * (1.0f - t * t) * du;
    }
    case MESH_MOE_ACT_SIGMOID: {
      const float sg = 1.0f / (1.0f + expf(-v));
      return sg * (1.0f - sg);
    }
    case MESH_MOE_ACT_TANH: {
      const float t = tanhf(v);
      return 1.0f - t * t;
    }
    case MESH_MOE_ACT_SWISH: {
      const float sg = 1.0f / (1.0f + expf(-v));
      return sg + v * sg * (1.0f - sg);
    }
    default:
      return 1.0f;
  }
}

// dpre = dh * factor * act'(pre), float32 arithmetic, one rounding.
template <typename T>
__global__ __launch_bounds__(256) void activation_backward_kernel(
    const T* __restrict__ dh, const T* __restrict__ pre,
    const T* __restrict__ factor, T* __restrict__ dpre, int64_t n, int act) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    float g = load_f32<T>(dh + i);
    if (factor) g *= load_f32<T>(factor + i);
    store_f32<T>(dpre + i, g * activation_derivative(load_f32<T>(pre + i), act));
  }
}

// The same for bf16 with 16-byte accesses: 8 elements per thread and step.
__global__ __launch_bounds__(256) void activation_backward_bf16x8_kernel(
    const uint4* __restrict__ dh, const uint4* __restrict__ pre,
    const uint4* __restrict__ factor, uint4* __restrict__ dpre, int64_t n8,
    int act) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
       i += stride) {
    const uint4 g4 = load_streaming(dh + i), p4 = load_streaming(pre + i);
    uint4 f4 = make_uint4(0, 0, 0, 0);
    if (factor) f4 = load_streaming(factor + i);
    const uint32_t g[4] = {g4.x, g4.y, g4.z, g4.w}, p[4] = {p4.x, p4.y, p4.z, p4.w};
    const uint32_t f[4] = {f4.x, f4.y, f4.z, f4.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float g0 = __uint_as_float(g[j] << 16), g1 = __uint_as_float(g[j] & 0xffff0000u);
      if (factor) {
        g0 *= __uint_as_float(f[j] << 16);
        g1 *= __uint_as_float(f[j] & 0xffff0000u);
      }
      o[j] = f32x2_to_bf16x2(
          g0 * activation_derivative(__uint_as_float(p[j] << 16), act),
          g1 * activation_derivative(__uint_as_float(p[j] & 0xffff0000u), act));
    }
    store_streaming(dpre + i, make_uint4(o[0], o[1], o[2], o[3]));
  }
}

// hidden_grad_kernel, hidden_product_kernel and activation_kernel for bf16
// with 16-byte accesses (8 elements per thread and step; the same arithmetic
// and the same roundings element by element).
__global__ __launch_bounds__(256) void hidden_grad_bf16x8_kernel(
    uint4* __restrict__ dh, const uint4* __restrict__ h,
    const uint4* __restrict__ scale, bool relu, int64_t n8,
    float const_scale) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
       i += stride) {
    float d[8], hv[8], sc[8];
    unpack16(load_streaming(dh + i), d, bf16_t());
    if (relu) unpack16(load_streaming(h + i), hv, bf16_t());
    if (scale) unpack16(load_streaming(scale + i), sc, bf16_t());
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (relu && !(hv[j] > 0.f)) d[j] = 0.f;
      else if (scale) d[j] = d[j] * sc[j];
      else d[j] = d[j] * const_scale;
    }
    store_streaming(dh + i, pack16(d, bf16_t()));
  }
}

__global__ __launch_bounds__(256) void hidden_product_bf16x8_kernel(
    uint4* __restrict__ h, const uint4* __restrict__ factor,
    const uint4* __restrict__ uniform, float keep, float inv_keep,
    uint4* __restrict__ noise_out, int64_t n8) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
       i += stride) {
    float v[8], f[8], u[8], nz[8];
    unpack16(load_streaming(h + i), v, bf16_t());
    if (factor) {
      unpack16(load_streaming(factor + i), f, bf16_t());
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = round_to<bf16_t>(v[j] * f[j]);
    }
    if (uniform) {
      unpack16(load_streaming(uniform + i), u, bf16_t());
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        nz[j] = u[j] < keep ? inv_keep : 0.f;
        v[j] = v[j] * nz[j];
      }
      if (noise_out) store_streaming(noise_out + i, pack16(nz, bf16_t()));
    }
    store_streaming(h + i, pack16(v, bf16_t()));
  }
}

// (out may be the input: in place)
__global__ __launch_bounds__(256) void activation_bf16x8_kernel(
    const uint4* h, uint4* out, int64_t n8, int act) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
       i += stride) {
    float v[8];
    unpack16(load_streaming(h + i), v, bf16_t());
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = apply_activation(v[j], act);
    store_streaming(out + i, pack16(v, bf16_t()));
  }
}

static bool x8_applies(int64_t n, int dtype, const void* a, const void* b,
                       const void* c, const void* d = nullptr) {
  return dtype == MESH_MOE_BF16 && n % 8 == 0 &&
         (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d) & 15) == 0;
}
static int elementwise_blocks(int64_t n) {
  return (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
}

// dh = dh * scale, then the ReLU mask of h (hidden_grad_kernel's contract)
static int launch_hidden_grad(void* dh, const void* h, const void* scale,
                              bool relu, int64_t n, int dtype, hipStream_t st,
                              float const_scale = 1.0f) {
  if (x8_applies(n, dtype, dh, h, scale))
    hidden_grad_bf16x8_kernel<<<elementwise_blocks(n / 8), 256, 0, st>>>(
        (uint4*)dh, (const uint4*)h, (const uint4*)scale, relu, n / 8,
        const_scale);
  else if (dtype == MESH_MOE_F32)
    hidden_grad_kernel<float><<<elementwise_blocks(n), 256, 0, st>>>(
        (float*)dh, (const float*)h, (const float*)scale, relu, n, const_scale);
  else
    hidden_grad_kernel<bf16_t><<<elementwise_blocks(n), 256, 0, st>>>(
        (bf16_t*)dh, (const bf16_t*)h, (const bf16_t*)scale, relu, n,
        const_scale);
  MOE_CHECK_LAUNCH("hidden gradient (mask / scale)");
  return 0;
}

// h = act(h) in place
static int launch_activation(void* h, int64_t n, int act, int dtype,
                             hipStream_t st) {
  if (x8_applies(n, dtype, h, nullptr, nullptr))
    activation_bf16x8_kernel<<<elementwise_blocks(n / 8), 256, 0, st>>>(
        (const uint4*)h, (uint4*)h, n / 8, act);
  else if (dtype == MESH_MOE_F32)
    activation_kernel<float><<<elementwise_blocks(n), 256, 0, st>>>((float*)h, n,
                                                                    act);
  else
    activation_kernel<bf16_t><<<elementwise_blocks(n), 256, 0, st>>>((bf16_t*)h,
                                                                     n, act);
  MOE_CHECK_LAUNCH("activation");
  return 0;
}

// Compute units of the current device (one persistent block per CU: a block
// takes all of a CU's LDS); 0 on failure.
int compute_units() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) !=
            hipSuccess || n < 1) {
      set_error("cannot query the number of compute units");
      return 0;
    }
    cus = n;
  }
  return cus;
}

template <int BM, int BN, int BK>
static int launch_mfma(const bf16_t* A, const bf16_t* B, bf16_t* C, int E,
                       int R, int N, int K, bool relu, hipStream_t st,
                       int64_t a_stride) {
  using Cfg = GemmCfg<BM, BN, BK>;
  const int tiles_m = (R + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int64_t blocks = (int64_t)tiles_m * tiles_n * E;
  MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: too many tiles (%lld)", (long long)blocks);
  if (relu) {
    auto k = grouped_gemm_bf16_kernel<BM, BN, BK, true>;
    MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
    k<<<(unsigned)blocks, 256, Cfg::LDS_BYTES, st>>>(A, B, C, R, N, K, tiles_m,
                                                      tiles_n, a_stride);
  } else {
    auto k = grouped_gemm_bf16_kernel<BM, BN, BK, false>;
    MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
    k<<<(unsigned)blocks, 256, Cfg::LDS_BYTES, st>>>(A, B, C, R, N, K, tiles_m,
                                                      tiles_n, a_stride);
  }
  MOE_CHECK_LAUNCH("expert_ffn (mfma)");
  return 0;
}

constexpr int SKINNY_ROWS = 128;
// Columns of a block of the kernel for few rows and few columns.
static int skinny_columns(int E, int N) {
  return (int64_t)E * ((N + 15) / 16) <= compute_units() ? 16 : 32;
}

static int launch_skinny(const bf16_t* A, const bf16_t* B, bf16_t* C, int E,
                         int R, int N, int K, bool relu, hipStream_t st,
                         int64_t a_stride) {
  // 16 columns per block while no compute unit gets a second block, else 32
  // (half the token reads)
  const int nt = skinny_columns(E, N) / 16;
  const int groups_n = (N + 16 * nt - 1) / (16 * nt);
  const int64_t blocks = (int64_t)E * groups_n;
  MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: too many tiles (%lld)", (long long)blocks);
  // wavefronts along the reduction: 16 per compute unit in all, while each
  // keeps 4 steps of 32
  int waves = 2;
  while (waves < 16 && blocks * waves < 4096 && K / 32 / (2 * waves) >= 4)
    waves *= 2;
  int mt = (R + 15) / 16;              // 1, 2, 3, 4, 6 or 8 tiles of 16 rows
  mt = mt == 5 || mt == 7 ? mt + 1 : mt;
  while (waves * mt * nt > 128) waves /= 2;    // 128 KB of LDS
  const size_t lds = (size_t)waves * mt * nt * 64 * 16;
  auto run = [&](auto k) -> int {
    MOE_ALLOW_LDS(k, lds);
    k<<<(unsigned)blocks, 64 * waves, lds, st>>>(A, B, C, R, N, K, groups_n,
                                                 relu ? 1 : 0, a_stride);
    MOE_CHECK_LAUNCH("expert_ffn (mfma, few rows)");
    return 0;
  };
#define MOE_SKINNY(MT_)                                                        \
  return nt == 2 ? run(skinny_gemm_bf16_kernel<MT_, 2>)                        \
                 : run(skinny_gemm_bf16_kernel<MT_, 1>)
  switch (mt) {
    case 1: MOE_SKINNY(1);
    case 2: MOE_SKINNY(2);
    case 3: MOE_SKINNY(3);
    case 4: MOE_SKINNY(4);
    case 6: MOE_SKINNY(6);
    default: MOE_SKINNY(8);
  }
#undef MOE_SKINNY
}

// The two kernels for a few rows per expert.  The skinny one cuts the reduction
// so that every compute unit has work; it is the faster one while no unit gets a
// second block of 32 columns (blocks that do not fit in one round, each with all
// of the token rows to read, cost up to twice the tile kernels' time: 128 rows,
// 16000 x 4096: 135 us, 128 x 128 tiles 75).  Above, up to 64 rows, the stream of
// whole lines.  us, one expert, K = 4096, by columns: 16 a block / 32 a block /
// stream / best tile kernel:
//    64 rows   4096: 25, 28, 33, 57   8192: 46, 29, 34, 58  10240: 66, 52, 34, 57
//    96 rows   4096: 30, 36, -, 56    8192: 55, 37, -, 57   10240: 84, 70, -, 57
//   128 rows   4096: 37, 47, -, 56    8192: 70, 48, -, 57   10240: 102, 91, -, 57
// Above 96 rows, blocks of 32 columns win with long reductions only (8192 columns,
// K = 1024: 16.2, tiles 14.8; 2048: 27, 32).  Reductions that the stream does not
// take (K % 64 != 0) keep to 32 columns a block (64 rows, 16000 x 1024: 16, 128 x
// 128 tiles 22).
constexpr int STREAM_ROWS = 64;
static bool skinny_rounds(int E, int N) {
  return (int64_t)E * ((N + 31) / 32) <= compute_units();
}
// a 128-column tile for half of the compute units
static bool many_column_tiles(int E, int N) {
  return (int64_t)E * ((N + 127) / 128) * 2 >= compute_units();
}
static bool skinny_applies(int E, int R, int N, int K) {
  if (compute_units() == 0 || N % 16 != 0 || K % 32 != 0 || R > SKINNY_ROWS ||
      many_column_tiles(E, N))
    return false;
  if (R <= STREAM_ROWS) return skinny_rounds(E, N) || K % 64 != 0;
  return skinny_rounds(E, N) &&
         (R <= 96 || K > 1024 || skinny_columns(E, N) == 16);
}
// From 49 rows on, 128 x 128 tiles are faster for short reductions of few columns
// in more than one block per compute unit: they keep an expert's column tiles, which
// share its rows, on one die (64 rows: 200 experts, 512 columns, K = 128 13.0 us
// against 15.5, 512 29 against 32; 64 experts, 1024 columns, K = 256 12.1, 13.5).
static bool stream_applies(int E, int R, int N, int K) {
  const bool tiles_faster = R > 48 && K <= 512 && N <= 1024 &&
                            (int64_t)E * ((N + 127) / 128) > compute_units();
  return compute_units() > 0 && R <= STREAM_ROWS && K % 64 == 0 && N % 8 == 0 &&
         (many_column_tiles(E, N) || !skinny_rounds(E, N)) && !tiles_faster;
}

// row_map / gather / zero_row: see the kernel (null: rows as they lie)
static int launch_stream(const bf16_t* A, const bf16_t* B, bf16_t* C, int E,
                         int R, int N, int K, bool relu, hipStream_t st,
                         const int32_t* row_map = nullptr, bool gather = false,
                         const bf16_t* zero_row = nullptr,
                         int64_t a_stride = -1) {
  if (a_stride < 0) a_stride = (int64_t)R * K;
  auto run = [&](auto k, auto cfg) -> int {
    using Cfg = decltype(cfg);
    const int tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
    const int64_t blocks = (int64_t)E * tiles_n;
    MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
                "expert_ffn: too many tiles (%lld)", (long long)blocks);
    MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
    k<<<(unsigned)blocks, 256, Cfg::LDS_BYTES, st>>>(
        A, B, C, R, N, K, tiles_n, relu ? 1 : 0, row_map, gather ? 1 : 0,
        zero_row, a_stride);
    MOE_CHECK_LAUNCH("expert_ffn (mfma, few rows per expert)");
    return 0;
  };
#define MOE_STREAM(MT_)                                                        \
  return row_map != nullptr                                                    \
             ? run(stream_gemm_bf16_kernel<MT_, true>, StreamCfg<MT_>())       \
             : run(stream_gemm_bf16_kernel<MT_, false>, StreamCfg<MT_>())
  if (R <= 32) MOE_STREAM(1);
  MOE_STREAM(2);
#undef MOE_STREAM
}

// C[e] [R, N] = A[e]^T . B[e] with A[e] [K, R] and B[e] [K, N] (both with the
// reduction index outermost); true if the K-major ring kernel takes the shape.
static bool kmajor_path_applies(const void* A, const void* B, const void* C,
                                int R, int N, int K, int dtype) {
  return dtype == MESH_MOE_BF16 && K >= 1 &&
         R % 8 == 0 && N % 8 == 0 && R >= 128 && N >= 128 &&
         R < (1 << 25) && N < (1 << 25) &&   // 32-bit offsets within 32 rows
         (int64_t)R * K < (1LL << 31) && (int64_t)N * K < (1LL << 31) &&
         (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15) == 0;
}

// A weight gradient of few tiles and a long reduction (a dense layer's: one
// "expert", every token of the batch) leaves most compute units idle, each
// busy one walking the whole reduction: the K tiles of the last, partly filled
// round of tiles are then cut into `split` parts, which are units of work of
// their own (SPLIT), and split_reduce_kernel adds the parts.  Measured for 768 x
// 768 from 16000 rows (9 tiles of 250 K tiles), both launches: 277 us in one
// part, 81 in 4, 46 in 10, 40 in 14 - 20, 42 in 28; 768 x 3072 (36 tiles): 275
// in one, 97 in 4, 84 in 7.  The count comes from what these runs and those at
// 512 x 512 x 4000 and 1024 x 4096 x 2000 fit: 1.15 us per K tile, 0.07 us per part (256
// KB written and read back), 7 us for the second launch.
struct SplitPlan {
  int whole_tiles = 0;   // tiles computed whole, before the split ones
  int split = 1;         // parts of each of the others (1: none is split)
  size_t bytes = 0;      // scratch for the parts
};
static SplitPlan kmajor_split_plan(int E, int R, int N, int K) {
  using Cfg = RingCfg;
  SplitPlan plan;
  const int64_t tiles = (int64_t)((R + Cfg::BM - 1) / Cfg::BM) *
                        ((N + Cfg::BN - 1) / Cfg::BN) * E;
  const int cus = compute_units();
  if (cus == 0 || tiles > 0x7fffffffLL) return plan;
  const int tail = (int)(tiles % cus), nk = (K + Cfg::BK - 1) / Cfg::BK;
  if (tail == 0) return plan;
  const double per_k_tile = 1.15, per_part = 0.07, second_launch = 7.0;
  double best = nk * per_k_tile;
  for (int split = 2; split * tail <= cus && split <= nk; ++split) {
    const double cost = ((nk + split - 1) / split) * per_k_tile +
                        split * tail * per_part + second_launch;
    if (cost < best) {
      best = cost;
      plan.split = split;
    }
  }
  if (plan.split == 1) return plan;
  plan.whole_tiles = (int)tiles - tail;
  plan.bytes = (size_t)tail * plan.split * Cfg::BM * Cfg::BN * sizeof(float);
  return plan;
}

// Persistent blocks of a ring launch: always a multiple of 8, so that the XCDs
// hold runs of consecutive tiles, which share operand panels; blocks without a
// tile end at once.  (Dealt out one by one, 180 tiles -- 30 experts, 384 x 512,
// K = 1024 -- took 28.3 us, 252 tiles 36.6; now 23 and 24.)
static unsigned ring_blocks(int64_t tiles, int cus) {
  return (unsigned)(((tiles < cus ? tiles : cus) + 7) / 8 * 8);
}

// Rows per row tile (a multiple of 32, at most 256) for R rows per expert.
// The persistent blocks take whole rounds of tiles, so what counts is rounds
// times the time of a tile, and a tile of fewer 32-row pieces is cheaper: about
// 0.40 + 0.13 per piece us per K tile (0.20 + 0.14 with three token slots, no less than
// 0.6 and 0.5) and 5 us outside the K loop, 4.5 of a single piece.  Rows are spread
// evenly over the row tiles: 640 rows per expert are three tiles of 224 or four of 160,
// not 256 + 256 + 128.  In more than one round the row tiles of an expert do not run
// side by side, and each reads its weights again: no less than 9 TB/s takes for all of
// them.  (Without that term three low tiles in two rounds were chosen over one tile in
// one where the weights set the pace: 32 x 240 rows, 2304 -> 1152 68 us, one tile 58;
// 32 x 166, 4608 -> 1152 125 and 99.  One round of low tiles reads them once from
// memory: 12 x 152, 4608 -> 1536 61 in tiles of 64, 64 in tiles of 96.  70 products
// whose tiles of 32 rows fit into one round, which 64 were chosen for: with K below
// 1600 all are 4 to 8 % faster in 32, 2 x 570 rows, 832 -> 384 9.6 us and 8.9; others
// between 17 % faster and 3.5 % slower.)  Of 394 products of 1 to 128 experts, 128 to
// 16000 rows, K and N 512 to 8192, timed with every height from 64 on, the rule's
// choice is 0.3 % slower than the best one on average, by more than 3 % in 16 and by 9
// % at worst (24 x 417 rows, 8192 -> 2048: 224 rows 370 us, 128 338).  Tiles of 256 and
// a shorter last one -> the rule's choice (both sides bit-identical):
//   32 x 640 rows, 4096 x 1024 (160 rows; of 224 186 us)       197 -> 155 us
//   16 x 708 rows, 768 x 3072 (192 rows) / 3072 x 768 (160)  67 / 56 -> 53 / 51
//   8 x 900 rows, 1536 x 4608 (192 rows)                        111 -> 93
//   64 x 320 rows, 1024 x 4096 (160 rows; of 128 206 us)       200 -> 182
//   16 x 700 rows, 512 x 512 (96 rows)                         14.1 -> 10.7
//   5000 rows, 1280 x 1280 (128 rows)                          26.6 -> 20.4
// In launches of three rounds of 256-row tiles and more the power limiter sets the pace,
// and low tiles move more bytes per product: the terms for three token slots then count
// 1.10 times.  (24 such products timed without that factor, 160 or 128 rows against the
// 192 to 256 that the terms give the others: chosen for less than a tenth they were 1 to
// 13 % slower, 16 x 1408 rows, 1920 -> 7680 563 -> 606 us, 48 x 501, 7296 -> 2624 869 ->
// 982; for more, 1 % slower to 4 % faster.)
// K-major operands (weight gradients; R is then a width, K the rows summed over):
// 0.48 + 0.12 per piece us per K tile, 3.3 + 0.75 per piece outside the K loop, whose
// share is larger there (reductions of few K tiles; from 16 x 704 and 1280 rows, and
// the same remark: in 12 timed since, 64 to 1280 rows, the rule's choice was the fastest
// or within 2 % of it):
//   16 x 704 rows, 768 x 3072 / 3072 x 768 (192 rows)       65 / 63 -> 51.5 / 52
//   16 x 1280 rows, 768 x 3072 (192 rows)                       105 -> 85
//   24 x 512 rows, 512 x 1536 (192 rows)                       32.5 -> 27.2
//   12 x 1000 rows, 1280 x 2560 (224 rows)                     85.1 -> 76.9
// and the rule stays with 256 where that is the fastest (64 x 512 rows, 1024 x 4096
// 287, 224 rows 301; 8 x 640 rows, 1024 x 4096 41.4, 192 rows 45).
static int ring_tile_rows(int E, int R, int N, int K, int cus,
                          bool kmajor = false) {
  const int tiles_n = (N + RingCfg::BN - 1) / RingCfg::BN;
  const int nk = (K + RingCfg::BK - 1) / RingCfg::BK;
  const bool long_launch =
      (int64_t)E * ((R + RingCfg::BM - 1) / RingCfg::BM) * tiles_n >= 3 * (int64_t)cus;
  const double weights_once = (double)E * N * K * sizeof(bf16_t) / 9e6;
  int best_rows = RingCfg::BM;
  double best = 0;
  for (int rows = RingCfg::BM; rows >= 32; rows -= 32) {
    const int tiles_m = (R + rows - 1) / rows;
    const int even = ((R + tiles_m - 1) / tiles_m + 31) / 32 * 32;
    const int64_t tiles = (int64_t)E * ((R + even - 1) / even) * tiles_n;
    const int pieces = even / 32;
    const bool deep = !kmajor && even <= RingCfg::DEEP_ROWS;
    const double per_k_tile = kmajor ? 0.48 + 0.12 * pieces
                              : deep ? 0.20 + 0.14 * pieces
                                     : 0.40 + 0.13 * pieces;
    const double least = deep ? 0.5 : 0.6;
    const double outside = kmajor ? 3.3 + 0.75 * pieces : pieces == 1 ? 4.5 : 5.0;
    const double limited = deep && long_launch ? 1.10 : 1.0;
    double cost = limited * (double)((tiles + cus - 1) / cus) *
                  (nk * (per_k_tile < least ? least : per_k_tile) + outside);
    if (!kmajor && tiles > cus && cost < tiles_m * weights_once)
      cost = tiles_m * weights_once;
    if (rows == RingCfg::BM || cost < 0.98 * best) {
      best = cost;
      best_rows = even;
    }
  }
  return best_rows;
}

// scratch: kmajor_split_plan(...).bytes for the parts (null: nothing is split;
// with k_extent nothing is)
static int launch_ring_kmajor(const bf16_t* A, const bf16_t* B, bf16_t* C,
                              int E, int R, int N, int K, hipStream_t st,
                              const int32_t* k_extent = nullptr,
                              void* scratch = nullptr, int64_t a_stride = -1) {
  using Cfg = RingCfg;
  const int cus = compute_units();
  if (cus == 0) return MESH_MOE_E_HIP;
  const SplitPlan plan =
      scratch == nullptr || k_extent != nullptr ? SplitPlan()
                                                : kmajor_split_plan(E, R, N, K);
  const int tile_rows =
      plan.split > 1 ? Cfg::BM : ring_tile_rows(E, R, N, K, cus, true);
  const int tiles_m = (R + tile_rows - 1) / tile_rows;
  const int tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  const int64_t tiles = (int64_t)tiles_m * tiles_n * E;
  MOE_REQUIRE(tiles <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn_backward: too many tiles (%lld)", (long long)tiles);
  const unsigned blocks = ring_blocks(tiles, cus);
  if (plan.split > 1) {
    const int tail = (int)tiles - plan.whole_tiles;
    const int units = plan.whole_tiles + tail * plan.split;
    const unsigned split_blocks = ring_blocks(units, cus);
    auto k = grouped_gemm_bf16_ring_kernel<false, false, true, false, false,
                                           false, true>;
    MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
    k<<<split_blocks, Cfg::THREADS, Cfg::LDS_BYTES, st>>>(
        A, B, C, R, N, K, tiles_m, tiles_n, units, nullptr, nullptr, nullptr,
        nullptr, nullptr, 1.0f, (float*)scratch, plan.whole_tiles, plan.split,
        Cfg::BM, a_stride, RingSegments());
    MOE_CHECK_LAUNCH("expert_ffn_backward (mfma, K-major operands, split)");
    split_reduce_kernel<<<(unsigned)tail * Cfg::TM * Cfg::TN, Cfg::THREADS, 0,
                          st>>>((const float*)scratch, C, R, N, tiles_m,
                                tiles_n, plan.whole_tiles, tail, plan.split);
    MOE_CHECK_LAUNCH("expert_ffn_backward (sum of the parts)");
    return 0;
  }
  auto run = [&](auto k) -> int {
    MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
    k<<<blocks, Cfg::THREADS, Cfg::LDS_BYTES, st>>>(
        A, B, C, R, N, K, tiles_m, tiles_n, (int)tiles, nullptr, nullptr,
        nullptr, nullptr, k_extent, 1.0f, nullptr, 0, 1, tile_rows, a_stride,
        RingSegments());
    MOE_CHECK_LAUNCH("expert_ffn_backward (mfma, K-major operands)");
    return 0;
  };
  if (tile_rows != Cfg::BM)
    return run(grouped_gemm_bf16_ring_kernel<false, false, true, false, false,
                                             true>);
  return run(grouped_gemm_bf16_ring_kernel<false, false, true>);
}

static int launch_ring(const bf16_t* A, const bf16_t* B, bf16_t* C, int E,
                       int R, int N, int K, bool relu, hipStream_t st,
                       const int32_t* row_map = nullptr,
                       const bf16_t* zero_row = nullptr,
                       const bf16_t* mask_src = nullptr,
                       const int32_t* tile_list = nullptr,
                       float mask_scale = 1.0f, int64_t a_stride = -1,
                       const RingSegments& segments = RingSegments()) {
  using Cfg = RingCfg;
  const int cus = compute_units();
  if (cus == 0) return MESH_MOE_E_HIP;
  // (listed tiles are 256 rows high)
  const int tile_rows =
      tile_list != nullptr ? Cfg::BM
                           : ring_tile_rows(E, R, N, K * segments.count, cus);
  const int tiles_m = (R + tile_rows - 1) / tile_rows;
  const int tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  const int64_t tiles = (int64_t)tiles_m * tiles_n * E;
  MOE_REQUIRE(tiles <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: too many tiles (%lld)", (long long)tiles);
  MOE_REQUIRE(mask_src == nullptr || (!relu && row_map == nullptr),
              MESH_MOE_E_ARG,
              "expert_ffn: masked result with relu or gathered rows");
  const unsigned blocks = ring_blocks(tiles, cus);
  auto run = [&](auto k) -> int {
    MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
    k<<<blocks, Cfg::THREADS, Cfg::LDS_BYTES, st>>>(
        A, B, C, R, N, K, tiles_m, tiles_n, (int)tiles, row_map, zero_row,
        mask_src, tile_list, nullptr, mask_scale, nullptr, 0, 1, tile_rows,
        a_stride, segments);
    MOE_CHECK_LAUNCH("expert_ffn (mfma, 256-column direct-to-LDS tiles)");
    return 0;
  };
#define MOE_RING(RELU_, GATHER_, MASKED_, LISTED_, TAILS_)                     \
  run(grouped_gemm_bf16_ring_kernel<RELU_, GATHER_, false, MASKED_, LISTED_,   \
                                    TAILS_>)
#define MOE_RING_DEEP(RELU_, GATHER_, MASKED_)                                 \
  run(grouped_gemm_bf16_ring_kernel<RELU_, GATHER_, false, MASKED_, false,     \
                                    true, false, true>)
  if (tile_list != nullptr) {
    if (mask_src != nullptr) return MOE_RING(false, false, true, true, false);
    // the first GEMM gathers its rows, the second does not
    if (row_map != nullptr)
      return relu ? MOE_RING(true, true, false, true, false)
                  : MOE_RING(false, true, false, true, false);
    return relu ? MOE_RING(true, false, false, true, false)
                : MOE_RING(false, false, false, true, false);
  }
  // row tiles of fewer than 256 rows, or an expert's last one partly empty: the
  // instantiation that skips empty 32-row pieces
  const bool tails = R % tile_rows != 0 || tile_rows != Cfg::BM;
  const bool deep = tile_rows <= Cfg::DEEP_ROWS;
  if (segments.count > 1)       // (whole tiles too)
    return deep ? run(grouped_gemm_bf16_ring_kernel<false, false, false, false, false,
                                                    true, false, true, true>)
                : run(grouped_gemm_bf16_ring_kernel<false, false, false, false, false,
                                                    true, false, false, true>);
#define MOE_RING_T(RELU_, GATHER_, MASKED_)                                    \
  (deep    ? MOE_RING_DEEP(RELU_, GATHER_, MASKED_)                            \
   : tails ? MOE_RING(RELU_, GATHER_, MASKED_, false, true)                    \
           : MOE_RING(RELU_, GATHER_, MASKED_, false, false))
  if (mask_src != nullptr) return MOE_RING_T(false, false, true);
  if (row_map != nullptr)
    return relu ? MOE_RING_T(true, true, false) : MOE_RING_T(false, true, false);
  return relu ? MOE_RING_T(true, false, false) : MOE_RING_T(false, false, false);
#undef MOE_RING_T
#undef MOE_RING_DEEP
#undef MOE_RING
}

template <typename T>
static int launch_simple(const T* A, const T* B, T* C, int E, int R, int N,
                         int K, bool relu, hipStream_t st) {
  const int tiles_m = (R + 63) / 64, tiles_n = (N + 63) / 64;
  const int64_t blocks = (int64_t)tiles_m * tiles_n * E;
  MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn: too many tiles (%lld)", (long long)blocks);
  if (relu)
    grouped_gemm_simple_kernel<T, true><<<(unsigned)blocks, 256, 0, st>>>(
        A, B, C, R, N, K, tiles_m, tiles_n);
  else
    grouped_gemm_simple_kernel<T, false><<<(unsigned)blocks, 256, 0, st>>>(
        A, B, C, R, N, K, tiles_m, tiles_n);
  MOE_CHECK_LAUNCH("expert_ffn (fma)");
  return 0;
}

static bool ring_shape(int R, int N, int K) {
  return N >= 256 && R >= 128 && K % 64 == 0 && N % 8 == 0 &&
         (int64_t)N * K < (1LL << 31);
}
// Products for which the 128 x 128 tiles are no slower than the ring's 256 columns
// (same bits):
// short reductions in at most two blocks per compute unit (the ring's first loads and
// the output of its last tile, which has no next one beside it, take longer than the K
// loop: 16 experts, 512 x 1024, K = 64 8.2 against 9.9 us; 30 experts, 384 x 512, K = 64
// 8.0, 8.3; from three blocks on the ring wins: 30 x 640 x 512, K = 128 11.2, 8.7), and
// one row tile per expert in a few blocks per compute unit, where a ring tile of 128
// rows has no second row tile to share its weights with.  (There the lines were drawn
// when a ring tile's output was staged behind its K loop, 64 experts, 128 x 1024: K = 256
// 14.8 against 17.2 us, K = 1024 33.9, 38.5; the ring is now as fast or a little faster
// on this side of them: 11.7, 10.9; 26.6, 26.1; 256 experts, 128 x 512, K = 512 32.7,
// 31.7.)
static bool small_tiles_apply(int E, int R, int N, int K) {
  const int64_t tiles =
      (int64_t)E * ((R + 127) / 128) * ((N + 127) / 128);
  const int cus = compute_units();
  if (R <= 128 && tiles > cus) return tiles <= 2 * cus || K <= 512;
  return (K <= 128 && tiles <= 2 * cus) || (K <= 256 && tiles <= cus);
}
// The calls that fold the dispatch into their first GEMM decline row counts
// whose whole 256-row tiles would be more than a fifth padding.  (The line was drawn
// for tiles of 256 rows; it has not been measured with lower ones.)
static bool ring_path_applies(int R, int N, int K) {
  const int pad256 = (R + 255) / 256 * 256, pad128 = (R + 127) / 128 * 128;
  return ring_shape(R, N, K) && pad128 * 5 >= pad256 * 4;
}

// f32_gemm and f32_gemm_stable take these operands
static bool f32_nt_applies(const void* A, const void* B, const void* C, int R,
                           int N, int K) {
  return K % 4 == 0 && N % 4 == 0 && f32_gemm_applies(R, N, K) &&
         ((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) % 16 == 0;
}

// C[e] = act(A[e] . B[e]^T) for every expert.
// relu_mask_src (same shape and dtype as C): the kernels that can zero the
// elements of C whose mask_src element is not positive while they write C do so
// and set *mask_applied; otherwise the caller runs the mask as a pass of its own.
static int grouped_gemm(const void* A, const void* B, void* C, int E, int R,
                        int N, int K, int act, int dtype, hipStream_t st,
                        const void* relu_mask_src = nullptr,
                        bool* mask_applied = nullptr, float mask_scale = 1.0f,
                        bool shared_a = false) {
  const bool relu = act == MESH_MOE_ACT_RELU;
  // shared_a (bf16 on the matrix cores only): one A [R, K] for all experts
  const int64_t a_stride = shared_a ? 0 : (int64_t)R * K;
  int rc;
  if (mask_applied) *mask_applied = false;
  if (dtype == MESH_MOE_F32) {
    if (f32_nt_applies(A, B, C, R, N, K)) {
      const bool masks = relu_mask_src != nullptr && mask_applied != nullptr &&
                         !relu && ((uintptr_t)relu_mask_src % 16) == 0;
      // Short reductions of little work: making the terms costs more than they save
      // (2 x 1000 rows, 260 -> 100 6.7 against 7.3 us in terms, 33 rows, 36 -> 64 4.3
      // and 4.6; 64 rows, 512 -> 512 8.1 and 6.6, 24 x 40 rows, 256 -> 1024 13.2 and
      // 11.5).
      const float* mask = masks ? (const float*)relu_mask_src : nullptr;
      if (K < 320 && (double)E * R * N * K < 1.2e8)
        rc = f32_gemm_stable((const float*)A, (const float*)B, (float*)C, E, R, N, K,
                             relu, mask, mask_scale, st);
      else
        rc = f32_gemm((const float*)A, (const float*)B, (float*)C, E, R, N, K, false,
                      relu, mask, mask_scale, st);
      if (masks) *mask_applied = rc == 0;
    } else if (f32_few_rows_applies(R, N, K) &&
               ((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) % 16 == 0) {
      const bool masks = relu_mask_src != nullptr && mask_applied != nullptr &&
                         !relu && ((uintptr_t)relu_mask_src % 16) == 0;
      rc = f32_few_rows((const float*)A, (const float*)B, (float*)C, E, R, N, K, relu,
                        masks ? (const float*)relu_mask_src : nullptr, mask_scale, st);
      if (masks) *mask_applied = rc == 0;
    } else
      rc = launch_simple<float>((const float*)A, (const float*)B, (float*)C, E,
                                R, N, K, relu, st);
  } else {
    const bool mfma_ok =
        (K % 8 == 0) && (N % 8 == 0) &&
        (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) % 16 == 0);
    const bool masks = relu_mask_src != nullptr && mask_applied != nullptr &&
                       !relu && ((uintptr_t)relu_mask_src % 16) == 0;
    if (!mfma_ok)
      rc = launch_simple<bf16_t>((const bf16_t*)A, (const bf16_t*)B,
                                 (bf16_t*)C, E, R, N, K, relu, st);
    else if (stream_applies(E, R, N, K))
      rc = launch_stream((const bf16_t*)A, (const bf16_t*)B, (bf16_t*)C, E, R,
                         N, K, relu, st, nullptr, false, nullptr, a_stride);
    else if (skinny_applies(E, R, N, K))
      rc = launch_skinny((const bf16_t*)A, (const bf16_t*)B, (bf16_t*)C, E, R,
                         N, K, relu, st, a_stride);
    else if (ring_shape(R, N, K) && (int64_t)R * K < (1LL << 31) &&
             (masks || !small_tiles_apply(E, R, N, K))) {
      // 256-column tiles in persistent blocks of 8 wavefronts (two per SIMD),
      // the loads spread over the MFMA steps
      rc = launch_ring((const bf16_t*)A, (const bf16_t*)B, (bf16_t*)C, E, R, N,
                       K, relu, st, nullptr, nullptr,
                       masks ? (const bf16_t*)relu_mask_src : nullptr, nullptr,
                       masks ? mask_scale : 1.0f, a_stride);
      if (masks) *mask_applied = rc == 0;
    } else if (R >= 1024 && N >= 1024 && !small_tiles_apply(E, R, N, K))
      rc = launch_mfma<256, 256, 64>((const bf16_t*)A, (const bf16_t*)B,
                                     (bf16_t*)C, E, R, N, K, relu, st, a_stride);
    else
      rc = launch_mfma<128, 128, 64>((const bf16_t*)A, (const bf16_t*)B,
                                     (bf16_t*)C, E, R, N, K, relu, st, a_stride);
  }
  if (rc != 0) return rc;
  if (act != MESH_MOE_ACT_RELU && act != MESH_MOE_ACT_LINEAR)
    return launch_activation(C, (int64_t)E * R * N, act, dtype, st);
  return 0;
}

// C[e] = A[e]^T . B[e] in float32, A [K, R] and B [K, N]: what f32_gemm and f32_few_k take
// with operands as they lie.
static bool f32_kmajor_applies(const void* A, const void* B, const void* C,
                               int R, int N, int K, int dtype) {
  return dtype == MESH_MOE_F32 && R % 4 == 0 && N % 4 == 0 &&
         (f32_gemm_applies(R, N, K) || f32_few_k_applies(R, N, K)) &&
         ((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) % 16 == 0;
}
static int f32_kmajor(const void* A, const void* B, void* C, int E, int R, int N, int K,
                      hipStream_t st) {
  if (f32_few_k_applies(R, N, K))
    return f32_few_k((const float*)A, (const float*)B, (float*)C, E, R, N, K, st);
  return f32_gemm((const float*)A, (const float*)B, (float*)C, E, R, N, K, true, false,
                  nullptr, 1.f, st);
}

// Batched C[e] = A[e] . B[e]^T for the other source files (attention): `dtype`
// operands, `dtype` result or, with out_f32, a float32 result.
int batched_gemm_nt(const void* A, const void* B, void* C, int E, int R, int N,
                    int K, int dtype, bool out_f32, hipStream_t st) {
  if (dtype == MESH_MOE_F32 || !out_f32)
    return grouped_gemm(A, B, C, E, R, N, K, MESH_MOE_ACT_LINEAR, dtype, st);
  if (!(K % 8 == 0 && N % 8 == 0 &&
        (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) % 16 == 0))) {
    // shapes the matrix-core kernel does not take (e.g. a key / value size
    // that is not a multiple of 8): the plain tile kernel, bf16 in, float32 out
    const int tiles_m = (R + 63) / 64, tiles_n = (N + 63) / 64;
    const int64_t blocks = (int64_t)tiles_m * tiles_n * E;
    MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
                "batched_gemm_nt: too many tiles (%lld)", (long long)blocks);
    grouped_gemm_simple_kernel<bf16_t, false, float>
        <<<(unsigned)blocks, 256, 0, st>>>((const bf16_t*)A, (const bf16_t*)B,
                                           (float*)C, R, N, K, tiles_m, tiles_n);
    MOE_CHECK_LAUNCH("batched_gemm_nt (fma, float32 result)");
    return 0;
  }
  using Cfg = GemmCfg<128, 128, 64>;
  const int tiles_m = (R + 127) / 128, tiles_n = (N + 127) / 128;
  const int64_t blocks = (int64_t)tiles_m * tiles_n * E;
  MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "batched_gemm_nt: too many tiles (%lld)", (long long)blocks);
  auto k = grouped_gemm_bf16_kernel<128, 128, 64, false, true>;
  MOE_ALLOW_LDS(k, Cfg::LDS_BYTES);
  k<<<(unsigned)blocks, 256, Cfg::LDS_BYTES, st>>>(
      (const bf16_t*)A, (const bf16_t*)B, C, R, N, K, tiles_m, tiles_n,
      (int64_t)R * K);
  MOE_CHECK_LAUNCH("batched_gemm_nt (mfma, float32 result)");
  return 0;
}

}  // namespace mesh_moe

using namespace mesh_moe;

static int expert_ffn(const void* expert_in, const void* wi_packed,
                      const void* wo_packed, void* h, void* y, int E, int R, int M,
                      int H, int N, int activation, int dtype, void* stream,
                      bool hidden_kept) {
  MOE_REQUIRE(expert_in && wi_packed && wo_packed && h && y, MESH_MOE_E_ARG,
              "expert_ffn: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG, "expert_ffn: bad dtype %d",
              dtype);
  MOE_REQUIRE(E >= 1 && R >= 1 && M >= 1 && H >= 1 && N >= 1, MESH_MOE_E_ARG,
              "expert_ffn: bad sizes E=%d R=%d M=%d H=%d N=%d", E, R, M, H, N);
  MOE_REQUIRE(activation >= MESH_MOE_ACT_LINEAR &&
                  activation <= MESH_MOE_ACT_SWISH,
              MESH_MOE_E_ARG, "expert_ffn: unknown activation %d", activation);
  hipStream_t st = (hipStream_t)stream;
  int rc;
  if (hidden_kept && dtype == MESH_MOE_F32 && activation == MESH_MOE_ACT_RELU &&
      f32_nt_applies(expert_in, wi_packed, h, R, H, M))
    rc = f32_gemm_stable((const float*)expert_in, (const float*)wi_packed,
                         (float*)h, E, R, H, M, true, nullptr, 1.f, st);
  else
    rc = grouped_gemm(expert_in, wi_packed, h, E, R, H, M, activation, dtype, st);
  if (rc != 0) return rc;
  return grouped_gemm(h, wo_packed, y, E, R, N, H, MESH_MOE_ACT_LINEAR, dtype,
                      st);
}

extern "C" int mesh_moe_expert_ffn(const void* expert_in, const void* wi_packed,
                                   const void* wo_packed, void* h, void* y,
                                   int E, int R, int M, int H, int N,
                                   int activation, int dtype, void* stream) {
  return expert_ffn(expert_in, wi_packed, wo_packed, h, y, E, R, M, H, N,
                    activation, dtype, stream, false);
}

extern "C" int mesh_moe_expert_ffn_kept(const void* expert_in,
                                        const void* wi_packed,
                                        const void* wo_packed, void* h, void* y,
                                        int E, int R, int M, int H, int N,
                                        int activation, int dtype, void* stream) {
  return expert_ffn(expert_in, wi_packed, wo_packed, h, y, E, R, M, H, N,
                    activation, dtype, stream, true);
}

namespace mesh_moe {

// ---------------------------------------------------------------------------
// Dispatch folded into the first expert GEMM: slot -> token map.
// ---------------------------------------------------------------------------
// threads first, first + stride, ... of those that clear the map
__device__ __forceinline__ void clear_slot_map(int32_t* map, int64_t n,
                                               bf16_t* zero_row, int m,
                                               int64_t first, int64_t stride) {
  for (int64_t i = first; i < n; i += stride) map[i] = -1;
  for (int64_t i = first; i < m; i += stride) zero_row[i] = 0;
}

__global__ void slot_map_clear_kernel(int32_t* map, int64_t n, bf16_t* zero_row,
                                      int m) {
  clear_slot_map(map, n, zero_row, m,
                 (int64_t)blockIdx.x * blockDim.x + threadIdx.x,
                 (int64_t)gridDim.x * blockDim.x);
}

// one thread per (token, choice): a kept choice whose activation-dtype gate is
// not 0 owns slot [idx][g][pos] (transformer/moe.py:1510-1511: the dispatch
// tensor is the combine tensor cast to bool)
__global__ void slot_map_kernel(const int32_t* __restrict__ idx,
                                const int32_t* __restrict__ pos,
                                const float* __restrict__ gate,
                                const uint8_t* __restrict__ kept,
                                int32_t* __restrict__ map, int64_t tokens,
                                int S, int C, int64_t rows_per_expert) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= tokens * 2) return;
  if (!kept[i] || round_to<bf16_t>(gate[i]) == 0.0f) return;
  const int64_t t = i >> 1;
  const int64_t g = t / S;
  map[(int64_t)idx[i] * rows_per_expert + g * C + pos[i]] = (int32_t)t;
}

// The same map in one launch where the fill counts are there: the first blocks take a
// thread per (token, choice), the next ones 1 << lane_bits threads (at most a
// wavefront) per (group, expert) for its empty slots, which are the last ones, and the
// last one the row of zeros.  Bound by being a launch: 16 x 1024 tokens, 32 experts 5.6
// us, in two launches 5.5 each.  (One thread per (group, expert) is a chain of stores
// where slots are mostly empty: 2 x 4096 tokens that all prefer one or two of 16 experts,
// 700 slots each, 19.5 us, now 2.7.)
__global__ __launch_bounds__(256) void slot_map_fill_kernel(
    const int32_t* __restrict__ idx, const int32_t* __restrict__ pos,
    const float* __restrict__ gate, const uint8_t* __restrict__ kept,
    const int32_t* __restrict__ fill, int32_t* __restrict__ map, int64_t tokens, int S,
    int G, int E, int C, bf16_t* __restrict__ zero_row, int m, int pair_blocks,
    int expert_blocks, int lane_bits) {
  const int block = blockIdx.x, tid = threadIdx.x;
  if (block < pair_blocks) {
    const int64_t i = (int64_t)block * 256 + tid;
    if (i >= tokens * 2 || !kept[i]) return;
    const int64_t t = i >> 1, g = t / S;
    map[((int64_t)idx[i] * G + g) * C + pos[i]] =
        round_to<bf16_t>(gate[i]) == 0.0f ? -1 : (int32_t)t;
  } else if (block < pair_blocks + expert_blocks) {
    const int64_t i = ((int64_t)(block - pair_blocks) * 256 + tid) >> lane_bits;
    if (i >= (int64_t)G * E) return;
    const int64_t g = i / E, e = i - g * E;
    const int lanes = 1 << lane_bits;
    for (int slot = fill[i] + (tid & (lanes - 1)); slot < C; slot += lanes)
      map[(e * G + g) * C + slot] = -1;
  } else {
    for (int i = tid; i < m; i += 256) zero_row[i] = 0;
  }
}

// The same map in one launch for few rows per expert (at most STREAM_ROWS) and at
// most MAP_SCAN_TOKENS tokens: a block per expert looks through the whole record
// for its slots, 128 tokens a round.  From about 512 tokens on that takes longer
// than the launch it saves, and with the map in two launches the call takes longer
// than a dispatch and the two products (64 experts of 256 -> 512 -> 256: 256 tokens
// 15.1 us, two launches 16.1, dispatch 14.0 to 16; 2048 tokens 28, 21, 19; 16384
// tokens 64, 21, 21.  64 experts of 1024 -> 4096 -> 1024, 1024 tokens: two launches
// 219, dispatch 213).
constexpr int MAP_SCAN_TOKENS = 512;
__global__ __launch_bounds__(256) void slot_map_rows_kernel(
    const int32_t* __restrict__ idx, const int32_t* __restrict__ pos,
    const float* __restrict__ gate, const uint8_t* __restrict__ kept,
    int32_t* __restrict__ map, int tokens, int S, int C, int rows,
    bf16_t* zero_row, int m) {
  __shared__ int32_t own[STREAM_ROWS];
  const int e = blockIdx.x, tid = threadIdx.x;
  if (tid < rows) own[tid] = -1;
  if (e == 0)
    for (int i = tid; i < m; i += 256) zero_row[i] = 0;
  __syncthreads();
  for (int i = tid; i < tokens * 2; i += 256) {
    if (idx[i] != e || !kept[i] || round_to<bf16_t>(gate[i]) == 0.0f) continue;
    const int t = i >> 1;
    own[t / S * C + pos[i]] = t;
  }
  __syncthreads();
  if (tid < rows) map[(int64_t)e * rows + tid] = own[tid];
}

// ---------------------------------------------------------------------------
// Compacted rows: expert e's occupied slots, groups in order, slots in order,
// become rows 0 .. rows_used[e] - 1 of its row range.
//
// Two launches prepare a call's GEMMs: compact_rows_kernel (the row offsets, and
// the map cleared) and compact_map_kernel (the map from the offsets, and both
// GEMMs' tile lists); the backward takes one (compact_lists_kernel).  Each is
// bound by being a launch, about 5 us.  As a launch per task they were five and
// three: 32768 tokens, 64 experts, 572 -> 566 us a pass, and 2253 -> 2233 in
// training with one choice per token.
// ---------------------------------------------------------------------------
// The sum of v over the threads before this one; `total` over all.  (Callers
// synchronise before they use wave_sums, NT / 64 values, again.)
template <int NT>
__device__ __forceinline__ int block_prefix(int v, int* wave_sums, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int sum = v;
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int before = __shfl_up(sum, d);
    if (lane >= d) sum += before;
  }
  if (lane == 63) wave_sums[wave] = sum;
  __syncthreads();
  int first = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    const int s = wave_sums[w];
    if (w < wave) first += s;
    total += s;
  }
  return first + sum - v;
}

// Blocks 0 .. E - 1: row_offsets[e][g] = sum over g' < g of fill[g'][e].  The
// blocks behind them clear the map.
__global__ __launch_bounds__(256) void compact_rows_kernel(
    const int32_t* __restrict__ fill, int32_t* __restrict__ row_offsets,
    int32_t* __restrict__ rows_used, int G, int E, int32_t* __restrict__ map,
    int64_t n_map, bf16_t* __restrict__ zero_row, int m) {
  __shared__ int wave_sums[4];
  const int e = blockIdx.x, tid = threadIdx.x;
  if (e >= E) {
    clear_slot_map(map, n_map, zero_row, m, (int64_t)(e - E) * 256 + tid,
                   (int64_t)((int)gridDim.x - E) * 256);
    return;
  }
  const int per = (G + 255) / 256;
  const int g0 = min(G, tid * per), g1 = min(G, g0 + per);
  int sum = 0;
  for (int g = g0; g < g1; ++g) sum += fill[(int64_t)g * E + e];
  int total;
  int run = block_prefix<256>(sum, wave_sums, total);
  if (tid == 0) rows_used[e] = total;
  for (int g = g0; g < g1; ++g) {
    row_offsets[(int64_t)e * G + g] = run;
    run += fill[(int64_t)g * E + e];
  }
}

// The tiles that hold occupied rows, in the order of the full tile numbering
// ((expert, N tile, M tile), M tile fastest), of up to two GEMMs over the same
// rows: list[-1] = their number.  E <= 1024 (a thread per expert).
constexpr int LIST_THREADS = 1024;
struct TileLists {
  int32_t* list[2];
  int tiles_n[2];
  int E, tiles_m, bm;
  int parts;             // blocks per list
};
// a block per 8 tiles a thread, no more than a list needs and at most 16
static int tile_list_parts(int E, int tiles_m, int tn1, int tn2) {
  const int64_t tiles = (int64_t)E * tiles_m * (tn1 > tn2 ? tn1 : tn2);
  const int64_t parts = (tiles + 8 * LIST_THREADS - 1) / (8 * LIST_THREADS);
  return (int)(parts < 16 ? parts : 16);
}
// block `block` of 2 L.parts; used: the occupied rows of expert threadIdx.x
__device__ __forceinline__ void write_tile_list(const TileLists& L, int used,
                                                int block) {
  __shared__ int32_t mt[LIST_THREADS], pre[LIST_THREADS];
  __shared__ int wave_sums[LIST_THREADS / 64];
  const int tid = threadIdx.x, part = block >> 1;
  const bool second = (block & 1) != 0;
  int32_t* list = second ? L.list[1] : L.list[0];
  const int tiles_n = second ? L.tiles_n[1] : L.tiles_n[0];
  const int own = tid < L.E ? min(L.tiles_m, (used + L.bm - 1) / L.bm) : 0;
  int total_m;
  pre[tid] = block_prefix<LIST_THREADS>(own, wave_sums, total_m);
  mt[tid] = own;
  if (part == 0 && tid == 0) list[-1] = total_m * tiles_n;
  __syncthreads();
  const int64_t total = (int64_t)L.E * tiles_n * L.tiles_m;
  for (int64_t at = (int64_t)part * LIST_THREADS + tid; at < total;
       at += (int64_t)L.parts * LIST_THREADS) {
    const int i = (int)at;
    const int tm = i % L.tiles_m, rest = i / L.tiles_m;
    const int tn = rest % tiles_n, e = rest / tiles_n;
    if (tm < mt[e]) list[tiles_n * pre[e] + tn * mt[e] + tm] = i;
  }
}

// Blocks 0 .. 2 parts - 1: the tile lists.  Behind them one thread per (token,
// choice), as slot_map_kernel, onto the compacted rows.
__global__ __launch_bounds__(LIST_THREADS) void compact_map_kernel(
    const int32_t* __restrict__ idx, const int32_t* __restrict__ pos,
    const float* __restrict__ gate, const uint8_t* __restrict__ kept,
    const int32_t* __restrict__ row_offsets,
    const int32_t* __restrict__ rows_used, int32_t* __restrict__ map,
    int64_t tokens, int S, int G, int64_t rows_per_expert, TileLists lists) {
  const int list_blocks = 2 * lists.parts, tid = threadIdx.x;
  if ((int)blockIdx.x < list_blocks) {
    write_tile_list(lists, tid < lists.E ? rows_used[tid] : 0, blockIdx.x);
    return;
  }
  const int64_t i = (int64_t)(blockIdx.x - list_blocks) * LIST_THREADS + tid;
  if (i >= tokens * 2) return;
  if (!kept[i] || round_to<bf16_t>(gate[i]) == 0.0f) return;
  const int64_t t = i >> 1;
  const int64_t g = t / S;
  const int e = idx[i];
  map[(int64_t)e * rows_per_expert + row_offsets[(int64_t)e * G + g] + pos[i]] =
      (int32_t)t;
}

// The backward's tile lists, and rows_used[e] from the row offsets of the last
// group and its fill count.
__global__ __launch_bounds__(LIST_THREADS) void compact_lists_kernel(
    const int32_t* __restrict__ fill, const int32_t* __restrict__ row_offsets,
    int32_t* __restrict__ rows_used, int G, TileLists lists) {
  const int e = threadIdx.x;
  int used = 0;
  if (e < lists.E)
    used = row_offsets[(int64_t)e * G + G - 1] +
           fill[(int64_t)(G - 1) * lists.E + e];
  if (blockIdx.x == 0 && e < lists.E) rows_used[e] = used;
  write_tile_list(lists, used, blockIdx.x);
}

// The conditions of mesh_moe_dispatched_expert_ffn and mesh_moe_compact_expert_ffn on
// sizes (operands are to lie on 16 bytes besides)
static bool dispatched_sizes_fit(int G, int S, int C, int dtype) {
  return dtype == MESH_MOE_BF16 && (int64_t)G * C <= 0x7fffffffLL &&
         (int64_t)G * S <= 0x7fffffffLL;
}
bool dispatched_few_rows(int G, int S, int E, int C, int M, int H) {
  const int64_t rows = (int64_t)G * C;
  return rows <= STREAM_ROWS && (int64_t)G * S <= MAP_SCAN_TOKENS &&
         stream_applies(E, (int)rows, H, M) && many_column_tiles(E, H);
}
bool dispatched_ffn_shapes(int G, int S, int E, int C, int M, int H, int dtype) {
  return dispatched_sizes_fit(G, S, C, dtype) &&
         (dispatched_few_rows(G, S, E, C, M, H) || ring_path_applies(G * C, H, M));
}
bool compact_ffn_shapes(int G, int S, int E, int C, int M, int H, int N, int dtype) {
  return dispatched_sizes_fit(G, S, C, dtype) && E <= 1024 &&
         ring_path_applies(G * C, H, M) && ring_path_applies(G * C, N, H) &&
         (int64_t)G * C * H < (1LL << 31);    // h's offsets within an expert
}
// Two choices per token fill nearly all slots.  Compacted rows then save a tile nowhere,
// the empty slots only move to the end of each expert's rows: 1.5 % faster forward, 1 %
// forward and backward (64 experts of 2048 slots, 4096 -> 16384) where an expert's slots
// are whole tiles.  Of others the padded layout shortens an expert's last row tile.
bool top2_compacts(int G, int C) { return (int64_t)G * C % RingCfg::BM == 0; }

}  // namespace mesh_moe

extern "C" int mesh_moe_top2_compacts(int G, int C) {
  return top2_compacts(G, C) ? 1 : 0;
}

extern "C" size_t mesh_moe_dispatched_expert_ffn_workspace_bytes(int G, int E,
                                                                 int C, int M) {
  if (G < 1 || E < 1 || C < 1 || M < 1) return 0;
  return sizeof(int32_t) * (size_t)E * G * C + sizeof(bf16_t) * (size_t)M + 512;
}

namespace mesh_moe {

SlotMap slot_map_in(void* workspace, int G, int E, int C, int M) {
  auto up = [](uintptr_t q) { return (q + 255) & ~(uintptr_t)255; };
  SlotMap slots;
  slots.map = (int32_t*)up((uintptr_t)workspace);
  slots.zero_row = (bf16_t*)up((uintptr_t)(slots.map + (size_t)E * G * C));
  slots.zeros = M;
  return slots;
}

int dispatched_ffn(const void* x, const int32_t* idx, const int32_t* pos,
                   const float* gate, const uint8_t* kept, const int32_t* fill,
                   bool map_made, const void* wi_packed, const void* wo_packed, void* h,
                   void* y, void* workspace, size_t workspace_bytes, int G, int S,
                   int E, int C, int M, int H, int N, int activation, int dtype,
                   void* stream, int outer) {
  MOE_REQUIRE(x && idx && pos && gate && kept && wi_packed && wo_packed && h &&
                  y && workspace, MESH_MOE_E_ARG,
              "dispatched_expert_ffn: null pointer");
  MOE_REQUIRE(G >= 1 && S >= 1 && E >= 1 && C >= 1 && M >= 1 && H >= 1 && N >= 1,
              MESH_MOE_E_ARG, "dispatched_expert_ffn: bad sizes");
  MOE_REQUIRE(activation >= MESH_MOE_ACT_LINEAR &&
                  activation <= MESH_MOE_ACT_SWISH,
              MESH_MOE_E_ARG, "dispatched_expert_ffn: unknown activation %d",
              activation);
  MOE_REQUIRE(outer >= 1 && G % outer == 0 && (int64_t)E * outer <= 0x7fffffff,
              MESH_MOE_E_ARG, "dispatched_expert_ffn: %d groups in %d outer parts", G,
              outer);
  // outer > 1: every expert has that many kernels, one for G / outer groups in a row, and
  // its rows lie in that order anyway
  const int64_t rows = (int64_t)G / outer * C;
  const bool few_rows = outer == 1 && dispatched_few_rows(G, S, E, C, M, H) &&
                        ((uintptr_t)wo_packed | (uintptr_t)y) % 16 == 0;
  MOE_REQUIRE(dispatched_sizes_fit(G, S, C, dtype) &&
                  (few_rows || ring_path_applies((int)rows, H, M)) &&
                  (((uintptr_t)x | (uintptr_t)wi_packed | (uintptr_t)h) % 16 == 0),
              MESH_MOE_E_UNSUPPORTED,
              "dispatched_expert_ffn: needs bf16 and a first GEMM that one of "
              "the direct-to-LDS kernels takes (rows=%lld M=%d H=%d)",
              (long long)rows, M, H);
  MOE_REQUIRE(workspace_bytes >=
                  mesh_moe_dispatched_expert_ffn_workspace_bytes(G, E, C, M),
              MESH_MOE_E_ARG, "dispatched_expert_ffn: workspace too small");
  hipStream_t st = (hipStream_t)stream;
  const int R = (int)rows;
  const SlotMap slots = slot_map_in(workspace, G, E, C, M);
  int32_t* map = slots.map;
  bf16_t* zero_row = slots.zero_row;
  const bool relu = activation == MESH_MOE_ACT_RELU;
  if (few_rows) {
    if (!map_made) {
      slot_map_rows_kernel<<<E, 256, 0, st>>>(idx, pos, gate, kept, map, G * S, S,
                                              C, R, zero_row, M);
      MOE_CHECK_LAUNCH("dispatched_expert_ffn (slot map, few rows)");
    }
    int rc = launch_stream((const bf16_t*)x, (const bf16_t*)wi_packed,
                           (bf16_t*)h, E, R, H, M, relu, st, map, true,
                           zero_row);
    if (rc != 0) return rc;
    if (!relu && activation != MESH_MOE_ACT_LINEAR) {
      // (also over the rows of experts that were left out: nothing reads them)
      rc = launch_activation(h, (int64_t)E * R * H, activation, dtype, st);
      if (rc != 0) return rc;
    }
    if (stream_applies(E, R, N, H))
      return launch_stream((const bf16_t*)h, (const bf16_t*)wo_packed,
                           (bf16_t*)y, E, R, N, H, false, st, map);
    return grouped_gemm(h, wo_packed, y, E, R, N, H, MESH_MOE_ACT_LINEAR, dtype,
                        st);
  }
  const int64_t pairs = (int64_t)G * S * 2;
  const int pair_blocks = (int)((pairs + 255) / 256);
  if (fill != nullptr) {
    int lane_bits = 0;
    while (lane_bits < 6 && 1 << lane_bits < C) ++lane_bits;
    const int expert_blocks = (int)((((int64_t)G * E << lane_bits) + 255) / 256);
    slot_map_fill_kernel<<<(unsigned)(pair_blocks + expert_blocks + 1), 256, 0, st>>>(
        idx, pos, gate, kept, fill, map, (int64_t)G * S, S, G, E, C, zero_row, M,
        pair_blocks, expert_blocks, lane_bits);
    MOE_CHECK_LAUNCH("dispatched_expert_ffn (slot map)");
  } else {
    const int64_t n_map = (int64_t)E * G * C;
    const unsigned cb = (unsigned)((n_map + 255) / 256 < 4096 ? (n_map + 255) / 256
                                                              : 4096);
    slot_map_clear_kernel<<<cb, 256, 0, st>>>(map, n_map, zero_row, M);
    MOE_CHECK_LAUNCH("dispatched_expert_ffn (clear)");
    slot_map_kernel<<<(unsigned)pair_blocks, 256, 0, st>>>(
        idx, pos, gate, kept, map, (int64_t)G * S, S, C, (int64_t)G * C);
    MOE_CHECK_LAUNCH("dispatched_expert_ffn (slot map)");
  }
  int rc = launch_ring((const bf16_t*)x, (const bf16_t*)wi_packed, (bf16_t*)h,
                       E * outer, R, H, M, relu, st, map, zero_row);
  if (rc != 0) return rc;
  if (!relu && activation != MESH_MOE_ACT_LINEAR) {
    rc = launch_activation(h, (int64_t)E * outer * R * H, activation, dtype, st);
    if (rc != 0) return rc;
  }
  return grouped_gemm(h, wo_packed, y, E * outer, R, N, H, MESH_MOE_ACT_LINEAR, dtype,
                      st);
}

}  // namespace mesh_moe

extern "C" int mesh_moe_dispatched_expert_ffn(
    const void* x, const int32_t* idx, const int32_t* pos, const float* gate,
    const uint8_t* kept, const void* wi_packed, const void* wo_packed, void* h,
    void* y, void* workspace, size_t workspace_bytes, int G, int S, int E, int C,
    int M, int H, int N, int activation, int dtype, void* stream) {
  return dispatched_ffn(x, idx, pos, gate, kept, nullptr, false, wi_packed, wo_packed,
                        h, y, workspace, workspace_bytes, G, S, E, C, M, H, N,
                        activation, dtype, stream);
}

// (The inner level of the hierarchical layer, forward: the dispatch in front of its
// experts wrote and read every slot row once more.  8 x 16 experts, 40960 tokens of 2048
// in 40 groups, 71 us of 3570.)
extern "C" int mesh_moe_dispatched_outer_expert_ffn(
    const void* x, const int32_t* idx, const int32_t* pos, const float* gate,
    const uint8_t* kept, const int32_t* fill, const void* wi_packed,
    const void* wo_packed, void* h, void* y, void* workspace, size_t workspace_bytes,
    int G, int S, int E, int C, int outer, int M, int H, int N, int activation, int dtype,
    void* stream) {
  return dispatched_ffn(x, idx, pos, gate, kept, fill, false, wi_packed, wo_packed, h, y,
                        workspace, workspace_bytes, G, S, E, C, M, H, N, activation,
                        dtype, stream, outer);
}

static size_t compact_ffn_tiles(int E, int R, int H, int N) {
  const size_t tm = (size_t)(R + RingCfg::BM - 1) / RingCfg::BM;
  return (size_t)E * tm * ((size_t)(H + RingCfg::BN - 1) / RingCfg::BN +
                           (size_t)(N + RingCfg::BN - 1) / RingCfg::BN);
}

extern "C" size_t mesh_moe_compact_expert_ffn_workspace_bytes(int G, int E,
                                                              int C, int M,
                                                              int H, int N) {
  if (G < 1 || E < 1 || C < 1 || M < 1 || H < 1 || N < 1) return 0;
  const int64_t rows = (int64_t)G * C;
  if (rows > 0x7fffffffLL) return 0;
  return sizeof(int32_t) * ((size_t)E * rows + (size_t)E +
                            compact_ffn_tiles(E, (int)rows, H, N) + 2 * 64) +
         sizeof(bf16_t) * (size_t)M + 6 * 256;
}

extern "C" int mesh_moe_compact_expert_ffn(
    const void* x, const int32_t* idx, const int32_t* pos, const float* gate,
    const uint8_t* kept, const int32_t* fill, const void* wi_packed,
    const void* wo_packed, void* h, void* y, int32_t* row_offsets,
    const void* hidden_uniform, float keep_prob, void* noise_out,
    void* workspace, size_t workspace_bytes, int G, int S, int E, int C, int M,
    int H, int N, int activation, int dtype, void* stream) {
  MOE_REQUIRE(x && idx && pos && gate && kept && fill && wi_packed &&
                  wo_packed && h && y && row_offsets && workspace,
              MESH_MOE_E_ARG, "compact_expert_ffn: null pointer");
  MOE_REQUIRE(!noise_out || hidden_uniform, MESH_MOE_E_ARG,
              "compact_expert_ffn: noise_out without hidden_uniform");
  MOE_REQUIRE(!hidden_uniform || (keep_prob > 0.f && keep_prob <= 1.f),
              MESH_MOE_E_ARG, "compact_expert_ffn: keep_prob %g outside (0, 1]",
              (double)keep_prob);
  MOE_REQUIRE(G >= 1 && S >= 1 && E >= 1 && C >= 1 && M >= 1 && H >= 1 && N >= 1,
              MESH_MOE_E_ARG, "compact_expert_ffn: bad sizes");
  MOE_REQUIRE(activation >= MESH_MOE_ACT_LINEAR &&
                  activation <= MESH_MOE_ACT_SWISH,
              MESH_MOE_E_ARG, "compact_expert_ffn: unknown activation %d",
              activation);
  const int64_t rows = (int64_t)G * C;
  MOE_REQUIRE(compact_ffn_shapes(G, S, E, C, M, H, N, dtype) &&
                  (((uintptr_t)x | (uintptr_t)wi_packed | (uintptr_t)wo_packed |
                    (uintptr_t)h | (uintptr_t)y) % 16 == 0),
              MESH_MOE_E_UNSUPPORTED,
              "compact_expert_ffn: needs bf16, at most 1024 experts and GEMMs "
              "the 256 x 256 direct-to-LDS kernel takes (rows=%lld M=%d H=%d "
              "N=%d)", (long long)rows, M, H, N);
  MOE_REQUIRE(workspace_bytes >= mesh_moe_compact_expert_ffn_workspace_bytes(
                                     G, E, C, M, H, N),
              MESH_MOE_E_ARG, "compact_expert_ffn: workspace too small");
  hipStream_t st = (hipStream_t)stream;
  const int R = (int)rows;
  auto up = [](uintptr_t q) { return (q + 255) & ~(uintptr_t)255; };
  int32_t* map = (int32_t*)up((uintptr_t)workspace);
  int32_t* rows_used = (int32_t*)up((uintptr_t)(map + (size_t)E * R));
  const int tiles_m = (R + RingCfg::BM - 1) / RingCfg::BM;
  const int tn1 = (H + RingCfg::BN - 1) / RingCfg::BN;
  const int tn2 = (N + RingCfg::BN - 1) / RingCfg::BN;
  // each list is preceded by its length (and padding up to 256 bytes)
  int32_t* list1 = (int32_t*)up((uintptr_t)(rows_used + E)) + 64;
  int32_t* list2 = (int32_t*)up((uintptr_t)(list1 + (size_t)E * tiles_m * tn1)) + 64;
  bf16_t* zero_row = (bf16_t*)up((uintptr_t)(list2 + (size_t)E * tiles_m * tn2));
  const int64_t n_map = (int64_t)E * R;
  const unsigned cb = (unsigned)((n_map + 255) / 256 < 4096 ? (n_map + 255) / 256
                                                            : 4096);
  compact_rows_kernel<<<(unsigned)E + cb, 256, 0, st>>>(
      fill, row_offsets, rows_used, G, E, map, n_map, zero_row, M);
  MOE_CHECK_LAUNCH("compact_expert_ffn (row offsets)");
  const TileLists lists = {{list1, list2}, {tn1, tn2}, E, tiles_m, RingCfg::BM,
                           tile_list_parts(E, tiles_m, tn1, tn2)};
  const int64_t pairs = (int64_t)G * S * 2;
  compact_map_kernel<<<(unsigned)(2 * lists.parts +
                                  (pairs + LIST_THREADS - 1) / LIST_THREADS),
                       LIST_THREADS, 0, st>>>(
      idx, pos, gate, kept, row_offsets, rows_used, map, (int64_t)G * S, S, G,
      rows, lists);
  MOE_CHECK_LAUNCH("compact_expert_ffn (slot map, tile lists)");
  const bool relu = activation == MESH_MOE_ACT_RELU;
  int rc = launch_ring((const bf16_t*)x, (const bf16_t*)wi_packed, (bf16_t*)h,
                       E, R, H, M, relu, st, map, zero_row, nullptr, list1);
  if (rc != 0) return rc;
  if (!relu && activation != MESH_MOE_ACT_LINEAR) {
    // (the pass also runs over the rows no listed tile wrote: they hold
    // unspecified values before and after, and nothing reads them)
    rc = launch_activation(h, (int64_t)E * R * H, activation, dtype, st);
    if (rc != 0) return rc;
  }
  if (hidden_uniform != nullptr) {
    // the hidden dropout, element for element of the [E, G*C, H] buffer (the
    // noise of a slot is the one drawn at its compacted row)
    rc = mesh_moe_hidden_product(h, nullptr, hidden_uniform, keep_prob,
                                 noise_out, (int64_t)E * R * H, dtype, stream);
    if (rc != 0) return rc;
  }
  return launch_ring((const bf16_t*)h, (const bf16_t*)wo_packed, (bf16_t*)y, E,
                     R, N, H, false, st, nullptr, nullptr, nullptr, list2);
}

extern "C" int mesh_moe_expert_linear(const void* a, const void* w_packed,
                                      void* y, int E, int R, int K, int N,
                                      int activation, int dtype, void* stream) {
  MOE_REQUIRE(a && w_packed && y, MESH_MOE_E_ARG, "expert_linear: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG, "expert_linear: bad dtype %d",
              dtype);
  MOE_REQUIRE(E >= 1 && R >= 1 && K >= 1 && N >= 1, MESH_MOE_E_ARG,
              "expert_linear: bad sizes E=%d R=%d K=%d N=%d", E, R, K, N);
  MOE_REQUIRE(activation >= MESH_MOE_ACT_LINEAR &&
                  activation <= MESH_MOE_ACT_SWISH,
              MESH_MOE_E_ARG, "expert_linear: unknown activation %d",
              activation);
  return grouped_gemm(a, w_packed, y, E, R, N, K, activation, dtype,
                      (hipStream_t)stream);
}

extern "C" int mesh_moe_hidden_product(void* h, const void* factor,
                                       const void* uniform, float keep_prob,
                                       void* noise_out, int64_t n, int dtype,
                                       void* stream) {
  MOE_REQUIRE(h, MESH_MOE_E_ARG, "hidden_product: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG,
              "hidden_product: bad dtype %d", dtype);
  MOE_REQUIRE(n >= 1, MESH_MOE_E_ARG, "hidden_product: bad size n=%lld",
              (long long)n);
  MOE_REQUIRE(!noise_out || uniform, MESH_MOE_E_ARG,
              "hidden_product: noise_out without uniform");
  MOE_REQUIRE(!uniform || (keep_prob > 0.f && keep_prob <= 1.f), MESH_MOE_E_ARG,
              "hidden_product: keep_prob %g outside (0, 1]", (double)keep_prob);
  if (!factor && !uniform) return 0;
  hipStream_t st = (hipStream_t)stream;
  const int blocks = (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
  if (x8_applies(n, dtype, h, factor, uniform, noise_out)) {
    const float keep = round_bf16_host(keep_prob);
    hidden_product_bf16x8_kernel<<<elementwise_blocks(n / 8), 256, 0, st>>>(
        (uint4*)h, (const uint4*)factor, (const uint4*)uniform, keep,
        round_bf16_host(1.f / keep), (uint4*)noise_out, n / 8);
  } else if (dtype == MESH_MOE_F32) {
    hidden_product_kernel<float><<<blocks, 256, 0, st>>>(
        (float*)h, (const float*)factor, (const float*)uniform, keep_prob,
        1.f / keep_prob, (float*)noise_out, n);
  } else {
    // the threshold and 1 / keep_prob are scalars of the activation dtype
    const float keep = round_bf16_host(keep_prob);
    hidden_product_kernel<bf16_t><<<blocks, 256, 0, st>>>(
        (bf16_t*)h, (const bf16_t*)factor, (const bf16_t*)uniform, keep,
        round_bf16_host(1.f / keep), (bf16_t*)noise_out, n);
  }
  MOE_CHECK_LAUNCH("hidden_product");
  return 0;
}

extern "C" int mesh_moe_activation(const void* pre, void* out, int64_t n,
                                   int activation, int dtype, void* stream) {
  MOE_REQUIRE(pre && out, MESH_MOE_E_ARG, "activation: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG, "activation: bad dtype %d",
              dtype);
  MOE_REQUIRE(n >= 1, MESH_MOE_E_ARG, "activation: bad size n=%lld",
              (long long)n);
  MOE_REQUIRE(activation >= MESH_MOE_ACT_LINEAR &&
                  activation <= MESH_MOE_ACT_SWISH,
              MESH_MOE_E_ARG, "activation: unknown activation %d", activation);
  hipStream_t st = (hipStream_t)stream;
  const int blocks = (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
  if (x8_applies(n, dtype, pre, out, nullptr))
    activation_bf16x8_kernel<<<elementwise_blocks(n / 8), 256, 0, st>>>(
        (const uint4*)pre, (uint4*)out, n / 8, activation);
  else if (dtype == MESH_MOE_F32)
    activation_copy_kernel<float><<<blocks, 256, 0, st>>>(
        (const float*)pre, (float*)out, n, activation);
  else
    activation_copy_kernel<bf16_t><<<blocks, 256, 0, st>>>(
        (const bf16_t*)pre, (bf16_t*)out, n, activation);
  MOE_CHECK_LAUNCH("activation");
  return 0;
}

extern "C" int mesh_moe_activation_backward(const void* dh, const void* pre,
                                            const void* factor, void* dpre,
                                            int64_t n, int activation,
                                            int dtype, void* stream) {
  MOE_REQUIRE(dh && pre && dpre, MESH_MOE_E_ARG,
              "activation_backward: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG,
              "activation_backward: bad dtype %d", dtype);
  MOE_REQUIRE(n >= 1, MESH_MOE_E_ARG, "activation_backward: bad size n=%lld",
              (long long)n);
  MOE_REQUIRE(activation >= MESH_MOE_ACT_LINEAR &&
                  activation <= MESH_MOE_ACT_SWISH,
              MESH_MOE_E_ARG, "activation_backward: unknown activation %d",
              activation);
  hipStream_t st = (hipStream_t)stream;
  const int blocks = (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
  if (dtype == MESH_MOE_F32)
    activation_backward_kernel<float><<<blocks, 256, 0, st>>>(
        (const float*)dh, (const float*)pre, (const float*)factor,
        (float*)dpre, n, activation);
  else if (n % 8 == 0 &&
           (((uintptr_t)dh | (uintptr_t)pre | (uintptr_t)factor |
             (uintptr_t)dpre) % 16) == 0) {
    const int64_t n8 = n / 8;
    const int vb = (int)((n8 + 255) / 256 < 16384 ? (n8 + 255) / 256 : 16384);
    activation_backward_bf16x8_kernel<<<vb, 256, 0, st>>>(
        (const uint4*)dh, (const uint4*)pre, (const uint4*)factor, (uint4*)dpre,
        n8, activation);
  } else
    activation_backward_kernel<bf16_t><<<blocks, 256, 0, st>>>(
        (const bf16_t*)dh, (const bf16_t*)pre, (const bf16_t*)factor,
        (bf16_t*)dpre, n, activation);
  MOE_CHECK_LAUNCH("activation_backward");
  return 0;
}

extern "C" size_t mesh_moe_expert_linear_backward_workspace_bytes(int E, int R,
                                                                  int K, int N,
                                                                  int dtype) {
  if (E < 1 || R < 1 || K < 1 || N < 1 || !valid_dtype(dtype)) return 0;
  const size_t transposed =
      ((size_t)E * R * K + (size_t)E * R * N) * dtype_size(dtype) + 2 * 256;
  const size_t parts = kmajor_split_plan(E, K, N, R).bytes + 256;
  return transposed > parts ? transposed : parts;
}

extern "C" int mesh_moe_expert_linear_backward(
    const void* a, const void* dy, const void* w, void* da, void* dw,
    const void* da_relu_mask, int E, int R, int K, int N, int dtype,
    void* workspace, size_t workspace_bytes, void* stream) {
  MOE_REQUIRE(a && dy && w && dw && workspace, MESH_MOE_E_ARG,
              "expert_linear_backward: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG,
              "expert_linear_backward: bad dtype %d", dtype);
  MOE_REQUIRE(E >= 1 && R >= 1 && K >= 1 && N >= 1, MESH_MOE_E_ARG,
              "expert_linear_backward: bad sizes E=%d R=%d K=%d N=%d", E, R, K,
              N);
  MOE_REQUIRE(workspace_bytes >=
                  mesh_moe_expert_linear_backward_workspace_bytes(E, R, K, N,
                                                                  dtype),
              MESH_MOE_E_ARG, "expert_linear_backward: workspace too small");
  hipStream_t st = (hipStream_t)stream;
  auto up = [](uintptr_t v) { return (v + 255) & ~(uintptr_t)255; };
  int rc;
  if (da != nullptr) {
    // da = dy . w^T  (w in its variable layout [E, K, N] is K-contiguous here);
    // a ReLU mask rides on the stores of this GEMM where its kernel can
    bool masked = false;
    rc = grouped_gemm(dy, w, da, E, R, K, N, MESH_MOE_ACT_LINEAR, dtype, st,
                      da_relu_mask, &masked);
    if (rc != 0) return rc;
    if (da_relu_mask != nullptr && !masked) {
      rc = launch_hidden_grad(da, da_relu_mask, nullptr, true,
                              (int64_t)E * R * K, dtype, st);
      if (rc != 0) return rc;
    }
  }
  // dw [E, K, N] = a^T . dy: the reduction runs over the rows of both operands
  if (kmajor_path_applies(a, dy, dw, K, N, R, dtype))
    return launch_ring_kmajor((const bf16_t*)a, (const bf16_t*)dy, (bf16_t*)dw,
                              E, K, N, R, st, nullptr,
                              (void*)up((uintptr_t)workspace));
  if (f32_kmajor_applies(a, dy, dw, K, N, R, dtype))
    return f32_kmajor(a, dy, dw, E, K, N, R, st);
  const size_t es = dtype_size(dtype);
  unsigned char* tr_a = (unsigned char*)up((uintptr_t)workspace);
  unsigned char* tr_dy =
      (unsigned char*)up((uintptr_t)(tr_a + (size_t)E * R * K * es));
  rc = mesh_moe_pack_weights(a, tr_a, E, R, K, dtype, dtype, stream);
  if (rc != 0) return rc;
  rc = mesh_moe_pack_weights(dy, tr_dy, E, R, N, dtype, dtype, stream);
  if (rc != 0) return rc;
  return grouped_gemm(tr_a, tr_dy, dw, E, K, N, R, MESH_MOE_ACT_LINEAR, dtype,
                      st);
}

// Elements of the scratch mesh_moe_expert_ffn_backward needs: dh [E,R,H], one
// [E,H,R] transpose buffer (h^T, then dh^T) and one [E,max(M,N),R] buffer
// (dy^T, then expert_in^T).
static size_t ffn_backward_elems(int E, int R, int M, int H, int N) {
  const size_t mn = (size_t)(M > N ? M : N);
  return (size_t)E * R * H * 2 + (size_t)E * R * mn;
}

extern "C" size_t mesh_moe_expert_ffn_backward_workspace_bytes(int E, int R,
                                                               int M, int H,
                                                               int N,
                                                               int dtype) {
  if (E < 1 || R < 1 || M < 1 || H < 1 || N < 1 || !valid_dtype(dtype))
    return 0;
  const size_t p1 = kmajor_split_plan(E, H, N, R).bytes;
  const size_t p2 = kmajor_split_plan(E, M, H, R).bytes;
  const size_t hidden = (size_t)E * R * H * dtype_size(dtype);
  const size_t parts = hidden + (p1 > p2 ? p1 : p2) + 2 * 256;
  const size_t transposed =
      ffn_backward_elems(E, R, M, H, N) * dtype_size(dtype) + 3 * 256;
  return transposed > parts ? transposed : parts;
}

extern "C" int mesh_moe_expert_ffn_backward(
    const void* expert_in, const void* h, const void* dy, const void* wi,
    const void* wo, const void* dh_scale, float dh_keep_prob,
    void* dexpert_in, void* dwi, void* dwo, int E, int R,
    int M, int H, int N, int activation, int dtype, void* workspace,
    size_t workspace_bytes, void* stream) {
  MOE_REQUIRE(expert_in && h && dy && wi && wo && dexpert_in && dwi && dwo &&
                  workspace, MESH_MOE_E_ARG,
              "expert_ffn_backward: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG,
              "expert_ffn_backward: bad dtype %d", dtype);
  MOE_REQUIRE(E >= 1 && R >= 1 && M >= 1 && H >= 1 && N >= 1, MESH_MOE_E_ARG,
              "expert_ffn_backward: bad sizes E=%d R=%d M=%d H=%d N=%d", E, R,
              M, H, N);
  MOE_REQUIRE(activation == MESH_MOE_ACT_RELU ||
                  activation == MESH_MOE_ACT_LINEAR, MESH_MOE_E_UNSUPPORTED,
              "expert_ffn_backward: only relu and linear experts (got %d): the "
              "other activations need the pre-activation, which is not kept",
              activation);
  MOE_REQUIRE(dh_keep_prob >= 0.f && dh_keep_prob <= 1.f, MESH_MOE_E_ARG,
              "expert_ffn_backward: dh_keep_prob=%g outside [0, 1] (0: no "
              "dropout, or a noise tensor alone describes it)",
              (double)dh_keep_prob);
  MOE_REQUIRE(workspace_bytes >= mesh_moe_expert_ffn_backward_workspace_bytes(
                                     E, R, M, H, N, dtype),
              MESH_MOE_E_ARG, "expert_ffn_backward: workspace too small");
  const size_t es = dtype_size(dtype);
  auto up = [](uintptr_t v) { return (v + 255) & ~(uintptr_t)255; };
  unsigned char* dh = (unsigned char*)up((uintptr_t)workspace);
  unsigned char* tr_h = (unsigned char*)up((uintptr_t)(dh + (size_t)E * R * H * es));
  unsigned char* tr_mn = (unsigned char*)up((uintptr_t)(tr_h + (size_t)E * R * H * es));
  hipStream_t st = (hipStream_t)stream;
  int rc;
  // dh = dy . wo^T  (wo in its variable layout [E, H, N] is K-contiguous here)
  // (the ReLU mask rides on the stores of this GEMM where its kernel can)
  // With a dropout whose keep probability is known, a ReLU expert's noise need
  // not be read: where the stored activation is positive the element was kept
  // and its noise is 1 / keep_prob (as mesh_moe_hidden_product rounds it).
  const bool relu_act = activation == MESH_MOE_ACT_RELU;
  const bool noise_by_mask =
      relu_act && dh_keep_prob > 0.f && dh_keep_prob < 1.f;
  // 1 / keep_prob as mesh_moe_hidden_product has it
  const float mask_scale =
      !noise_by_mask ? 1.f
      : dtype == MESH_MOE_BF16
          ? round_bf16_host(1.f / round_bf16_host(dh_keep_prob))
          : 1.f / dh_keep_prob;
  bool masked = false;
  rc = grouped_gemm(dy, wo, dh, E, R, H, N, MESH_MOE_ACT_LINEAR, dtype, st,
                    relu_act && (!dh_scale || noise_by_mask) ? h : nullptr,
                    &masked, mask_scale);
  if (rc != 0) return rc;
  if (!masked && (relu_act || dh_scale)) {
    rc = launch_hidden_grad(dh, h, noise_by_mask ? nullptr : dh_scale, relu_act,
                            (int64_t)E * R * H, dtype, st, mask_scale);
    if (rc != 0) return rc;
  }
  // dexpert_in = dh . wi^T  (wi in its variable layout [E, M, H])
  rc = grouped_gemm(dh, wi, dexpert_in, E, R, M, H, MESH_MOE_ACT_LINEAR, dtype,
                    st);
  if (rc != 0) return rc;
  // dwo [E, H, N] = h^T . dy and dwi [E, M, H] = expert_in^T . dh: the
  // reduction runs over token rows, the outermost index of both operands
  if (kmajor_path_applies(h, dy, dwo, H, N, R, dtype) &&
      kmajor_path_applies(expert_in, dh, dwi, M, H, R, dtype)) {
    // (the parts of split reductions lie behind dh)
    rc = launch_ring_kmajor((const bf16_t*)h, (const bf16_t*)dy, (bf16_t*)dwo,
                            E, H, N, R, st, nullptr, tr_h);
    if (rc != 0) return rc;
    return launch_ring_kmajor((const bf16_t*)expert_in, (const bf16_t*)dh,
                              (bf16_t*)dwi, E, M, H, R, st, nullptr, tr_h);
  }
  if (f32_kmajor_applies(h, dy, dwo, H, N, R, dtype) &&
      f32_kmajor_applies(expert_in, dh, dwi, M, H, R, dtype)) {
    rc = f32_kmajor(h, dy, dwo, E, H, N, R, st);
    if (rc != 0) return rc;
    return f32_kmajor(expert_in, dh, dwi, E, M, H, R, st);
  }
  // otherwise: both operands transposed to token-contiguous copies first
  rc = mesh_moe_pack_weights(h, tr_h, E, R, H, dtype, dtype, stream);
  if (rc != 0) return rc;
  rc = mesh_moe_pack_weights(dy, tr_mn, E, R, N, dtype, dtype, stream);
  if (rc != 0) return rc;
  rc = grouped_gemm(tr_h, tr_mn, dwo, E, H, N, R, MESH_MOE_ACT_LINEAR, dtype,
                    st);
  if (rc != 0) return rc;
  // dwi [E, M, H] = expert_in^T . dh
  rc = mesh_moe_pack_weights(expert_in, tr_mn, E, R, M, dtype, dtype, stream);
  if (rc != 0) return rc;
  rc = mesh_moe_pack_weights(dh, tr_h, E, R, H, dtype, dtype, stream);
  if (rc != 0) return rc;
  return grouped_gemm(tr_mn, tr_h, dwi, E, M, H, R, MESH_MOE_ACT_LINEAR, dtype,
                      st);
}

// ---------------------------------------------------------------------------
// Backward of the expert feed-forward on COMPACTED rows (the row order of
// mesh_moe_compact_expert_ffn): the two GEMMs whose result has token rows
// (dh, dexpert_in) compute only the row tiles that hold occupied slots, the
// two weight-gradient GEMMs reduce over every expert's occupied rows only.
// ---------------------------------------------------------------------------
static bool compact_backward_applies(int G, int E, int C, int M, int H, int N) {
  if (G < 1 || E < 1 || E > 1024 || C < 1 || M < 1 || H < 1 || N < 1)
    return false;
  const int64_t rows = (int64_t)G * C;
  if (rows > 0x7fffffffLL) return false;
  const int R = (int)rows;
  return ring_path_applies(R, H, N) && ring_path_applies(R, M, H) &&
         kmajor_path_applies(nullptr, nullptr, nullptr, H, N, R,
                             MESH_MOE_BF16) &&
         kmajor_path_applies(nullptr, nullptr, nullptr, M, H, R, MESH_MOE_BF16);
}

extern "C" size_t mesh_moe_compact_expert_ffn_backward_workspace_bytes(
    int G, int E, int C, int M, int H, int N) {
  if (!compact_backward_applies(G, E, C, M, H, N)) return 0;
  const size_t R = (size_t)G * C;
  const size_t tm = (R + RingCfg::BM - 1) / RingCfg::BM;
  const size_t tiles = (size_t)E * tm *
                       ((size_t)(H + RingCfg::BN - 1) / RingCfg::BN +
                        (size_t)(M + RingCfg::BN - 1) / RingCfg::BN);
  return sizeof(bf16_t) * (size_t)E * R * H +
         sizeof(int32_t) * ((size_t)E + tiles + 2 * 64) + 5 * 256;
}

extern "C" int mesh_moe_compact_expert_ffn_backward(
    const void* expert_in, const void* h, const void* dy, const void* wi,
    const void* wo, const void* dh_scale, float dh_keep_prob,
    const int32_t* fill, const int32_t* row_offsets, void* dexpert_in,
    void* dwi, void* dwo, int G, int E, int C, int M, int H, int N,
    int activation, int dtype, void* workspace, size_t workspace_bytes,
    void* stream) {
  MOE_REQUIRE(expert_in && h && dy && wi && wo && fill && row_offsets &&
                  dexpert_in && dwi && dwo && workspace, MESH_MOE_E_ARG,
              "compact_expert_ffn_backward: null pointer");
  MOE_REQUIRE(G >= 1 && E >= 1 && C >= 1 && M >= 1 && H >= 1 && N >= 1,
              MESH_MOE_E_ARG, "compact_expert_ffn_backward: bad sizes");
  MOE_REQUIRE(activation == MESH_MOE_ACT_RELU ||
                  activation == MESH_MOE_ACT_LINEAR, MESH_MOE_E_UNSUPPORTED,
              "compact_expert_ffn_backward: only relu and linear experts (got "
              "%d)", activation);
  MOE_REQUIRE(dh_keep_prob >= 0.f && dh_keep_prob <= 1.f, MESH_MOE_E_ARG,
              "compact_expert_ffn_backward: dh_keep_prob=%g outside [0, 1]",
              (double)dh_keep_prob);
  MOE_REQUIRE(dtype == MESH_MOE_BF16 &&
                  compact_backward_applies(G, E, C, M, H, N) &&
                  (((uintptr_t)expert_in | (uintptr_t)h | (uintptr_t)dy |
                    (uintptr_t)wi | (uintptr_t)wo | (uintptr_t)dexpert_in |
                    (uintptr_t)dwi | (uintptr_t)dwo) % 16 == 0),
              MESH_MOE_E_UNSUPPORTED,
              "compact_expert_ffn_backward: needs bf16, at most 1024 experts "
              "and shapes the 256 x 256 direct-to-LDS kernels take (rows=%lld "
              "M=%d H=%d N=%d)", (long long)G * C, M, H, N);
  MOE_REQUIRE(workspace_bytes >=
                  mesh_moe_compact_expert_ffn_backward_workspace_bytes(
                      G, E, C, M, H, N),
              MESH_MOE_E_ARG, "compact_expert_ffn_backward: workspace too small");
  hipStream_t st = (hipStream_t)stream;
  const int R = G * C;
  auto up = [](uintptr_t q) { return (q + 255) & ~(uintptr_t)255; };
  bf16_t* dh = (bf16_t*)up((uintptr_t)workspace);
  int32_t* rows_used = (int32_t*)up((uintptr_t)(dh + (size_t)E * R * H));
  const int tiles_m = (R + RingCfg::BM - 1) / RingCfg::BM;
  const int tn_h = (H + RingCfg::BN - 1) / RingCfg::BN;
  const int tn_m = (M + RingCfg::BN - 1) / RingCfg::BN;
  int32_t* list_h = (int32_t*)up((uintptr_t)(rows_used + E)) + 64;
  int32_t* list_m =
      (int32_t*)up((uintptr_t)(list_h + (size_t)E * tiles_m * tn_h)) + 64;
  const TileLists lists = {{list_h, list_m}, {tn_h, tn_m}, E, tiles_m,
                           RingCfg::BM,
                           tile_list_parts(E, tiles_m, tn_h, tn_m)};
  compact_lists_kernel<<<2 * lists.parts, LIST_THREADS, 0, st>>>(
      fill, row_offsets, rows_used, G, lists);
  MOE_CHECK_LAUNCH("compact_expert_ffn_backward (tile lists)");
  // dh = dy . wo^T on the listed row tiles, the ReLU mask on its stores (the
  // rows of a listed tile past the expert's occupied ones have h = 0 and
  // dy = 0)
  // (a ReLU expert's dropout noise follows from the stored activation: see
  // mesh_moe_expert_ffn_backward)
  const bool noise_by_mask = activation == MESH_MOE_ACT_RELU &&
                             dh_keep_prob > 0.f && dh_keep_prob < 1.f;
  const float mask_scale =
      noise_by_mask ? round_bf16_host(1.f / round_bf16_host(dh_keep_prob)) : 1.f;
  const bool mask_on_stores =
      activation == MESH_MOE_ACT_RELU && (!dh_scale || noise_by_mask);
  int rc = launch_ring(
      (const bf16_t*)dy, (const bf16_t*)wo, dh, E, R, H, N, false, st, nullptr,
      nullptr, mask_on_stores ? (const bf16_t*)h : nullptr, list_h, mask_scale);
  if (rc != 0) return rc;
  if (dh_scale != nullptr && !mask_on_stores) {
    // the dropout's noise (and the ReLU mask) as a pass over the buffer, as in
    // mesh_moe_expert_ffn_backward; rows outside the listed tiles hold
    // unspecified values before and after
    rc = launch_hidden_grad(dh, h, dh_scale, activation == MESH_MOE_ACT_RELU,
                            (int64_t)E * R * H, dtype, st);
    if (rc != 0) return rc;
  }
  // dexpert_in = dh . wi^T on the listed row tiles
  rc = launch_ring(dh, (const bf16_t*)wi, (bf16_t*)dexpert_in, E, R, M, H,
                   false, st, nullptr, nullptr, nullptr, list_m);
  if (rc != 0) return rc;
  // dwo = h^T . dy and dwi = expert_in^T . dh over the occupied rows
  rc = launch_ring_kmajor((const bf16_t*)h, (const bf16_t*)dy, (bf16_t*)dwo, E,
                          H, N, R, st, rows_used);
  if (rc != 0) return rc;
  return launch_ring_kmajor((const bf16_t*)expert_in, dh, (bf16_t*)dwi, E, M,
                            H, R, st, rows_used);
}

// Several dense layers of one input: y[e] = a . w[e].  The experts of a grouped product
// that all read the same rows (a_stride 0).  What bounds a projection of few rows is its
// launch and a chip that one product does not fill: three products of 32 rows,
// 1024 -> 1024, 14.6 us one by one and 5.4 in one launch, of 1024 rows, 768 -> 768,
// 31.6 and 12.6, of 4096 rows 40.5 and 21.8, of 16384 rows, 1024 -> 1024 (256 tiles of
// the ring each), 100.6 and 95.3.
extern "C" int mesh_moe_shared_linear(const void* a, const void* w_packed, void* y,
                                      int E, int R, int K, int N, int dtype,
                                      void* stream) {
  MOE_REQUIRE(a && w_packed && y, MESH_MOE_E_ARG, "shared_linear: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG, "shared_linear: bad dtype %d",
              dtype);
  MOE_REQUIRE(E >= 1 && R >= 1 && K >= 1 && N >= 1, MESH_MOE_E_ARG,
              "shared_linear: bad sizes E=%d R=%d K=%d N=%d", E, R, K, N);
  MOE_REQUIRE(dtype == MESH_MOE_BF16 && K % 8 == 0 && N % 8 == 0 &&
                  ((uintptr_t)a | (uintptr_t)w_packed | (uintptr_t)y) % 16 == 0,
              MESH_MOE_E_UNSUPPORTED,
              "shared_linear: needs bf16, sizes that are multiples of 8 and 16-byte "
              "alignment (K=%d N=%d dtype=%d)", K, N, dtype);
  return grouped_gemm(a, w_packed, y, E, R, N, K, MESH_MOE_ACT_LINEAR, dtype,
                      (hipStream_t)stream, nullptr, nullptr, 1.0f, true);
}

extern "C" size_t mesh_moe_shared_linear_backward_workspace_bytes(int E, int R,
                                                                  int K, int N) {
  if (E < 1 || R < 1 || K < 1 || N < 1) return 0;
  return kmajor_split_plan(E, K, N, R).bytes + 256;
}

// Their weight gradients: dw[e] = a^T . dy[e].  Nine tiles of 256 x 256 (768 -> 768) leave
// most of the chip idle or are cut along a reduction that is then written and read as
// partial sums; three times as many tiles need a third of the cuts.  With the three
// products for dx: 4096 rows, 768 -> 768, 109.9 us one by one and 73.2, 16384 rows,
// 1024 -> 1024, 260.5 and 206.9.
extern "C" int mesh_moe_shared_linear_backward(const void* a, const void* dy,
                                               void* dw, int E, int R, int K, int N,
                                               int dtype, void* workspace,
                                               size_t workspace_bytes,
                                               void* stream) {
  MOE_REQUIRE(a && dy && dw && workspace, MESH_MOE_E_ARG,
              "shared_linear_backward: null pointer");
  MOE_REQUIRE(E >= 1 && R >= 1 && K >= 1 && N >= 1, MESH_MOE_E_ARG,
              "shared_linear_backward: bad sizes E=%d R=%d K=%d N=%d", E, R, K, N);
  MOE_REQUIRE(kmajor_path_applies(a, dy, dw, K, N, R, dtype),
              MESH_MOE_E_UNSUPPORTED,
              "shared_linear_backward: needs bf16, K and N multiples of 8 and at "
              "least 128, 16-byte alignment (K=%d N=%d dtype=%d)", K, N, dtype);
  MOE_REQUIRE(workspace_bytes >=
                  mesh_moe_shared_linear_backward_workspace_bytes(E, R, K, N),
              MESH_MOE_E_ARG, "shared_linear_backward: workspace too small");
  void* parts = (void*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  return launch_ring_kmajor((const bf16_t*)a, (const bf16_t*)dy, (bf16_t*)dw, E, K,
                            N, R, (hipStream_t)stream, nullptr, parts, 0);
}

// The gradient of that input, dx = sum over e of dy[e] . w[e]^T, as one product whose
// reduction has E parts, added in float32.  One by one every part is written, and read
// again by a sum of its own that rounds it: three parts of 16000 rows, 768 -> 768, are
// three products of 24 us and two sums of 12, and a training step of such a block took
// 1924 us, now 1888.  What other kernels than the ring make (few rows, short reductions)
// is left to them.
extern "C" int mesh_moe_shared_linear_backward_input_supported(int E, int R, int K,
                                                               int N, int dtype) {
  return dtype == MESH_MOE_BF16 && (E == 2 || E == 3) && R >= 1 && K >= 1 && N >= 1 &&
         ring_shape(R, K, N) && (int64_t)R * N < (1LL << 31) &&
         (int64_t)N * E <= 0x7fffffff && !stream_applies(1, R, K, N * E) &&
         !skinny_applies(1, R, K, N * E) && !small_tiles_apply(1, R, K, N * E);
}

extern "C" int mesh_moe_shared_linear_backward_input(const void* dy,
                                                     const void* const* w, void* dx,
                                                     int E, int R, int K, int N,
                                                     int dtype, void* stream) {
  MOE_REQUIRE(dy && w && dx, MESH_MOE_E_ARG,
              "shared_linear_backward_input: null pointer");
  MOE_REQUIRE(mesh_moe_shared_linear_backward_input_supported(E, R, K, N, dtype),
              MESH_MOE_E_UNSUPPORTED,
              "shared_linear_backward_input: needs bf16, two or three layers and a "
              "product of the 256-column tiles (E=%d R=%d K=%d N=%d dtype=%d)", E, R, K,
              N, dtype);
  uintptr_t bits = (uintptr_t)dy | (uintptr_t)dx;
  RingSegments parts;
  parts.count = E;
  parts.tiles = N / RingCfg::BK;
  for (int i = 0; i < E; ++i) {
    MOE_REQUIRE(w[i], MESH_MOE_E_ARG, "shared_linear_backward_input: null pointer");
    bits |= (uintptr_t)w[i];
    parts.a_at[i] = (int64_t)i * R * N - (int64_t)i * N;
    parts.b_at[i] = ((intptr_t)w[i] - (intptr_t)w[0]) / (intptr_t)sizeof(bf16_t) -
                    (int64_t)i * N;
  }
  MOE_REQUIRE(bits % 16 == 0, MESH_MOE_E_UNSUPPORTED,
              "shared_linear_backward_input: operands off 16 bytes");
  return launch_ring((const bf16_t*)dy, (const bf16_t*)w[0], (bf16_t*)dx, 1, R, K, N,
                     false, (hipStream_t)stream, nullptr, nullptr, nullptr, nullptr,
                     1.0f, -1, parts);
}
