// Router projection and top-2 gating (softmax, expert choice, capacity
// positions, balancing loss) for gfx950.
//
// Follows _top_2_gating, mesh_tensorflow/transformer/moe.py:1384-1496, with the
// float32 operation order of mtf.softmax (ops.py:5493-5541) and mtf.top_1
// (ops.py:4937-4940).  The dense [G,S,E] masks and the S x S cumsum matmul
// (ops.py:2761-2781) are replaced by a per-token record and integer counting.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "common.h"

namespace mesh_moe {

// ---------------------------------------------------------------------------
// Router logits: logits[b,t,e] = sum_m x[b,t,m] * w[b,m,e] (+ bias[e]), float32
// multiply-adds in the order of m.
//
// A wavefront makes 16 tokens x 16 experts on v_mfma_f32_16x16x4_f32, which
// adds its four products one after the other: the sums have the bits of fmaf in
// the order of m.  Operands come straight from memory, PF groups of 16 columns
// ahead; the wavefronts of a block share the token rows, one expert tile each.
// VEC: a lane loads four consecutive columns of its token and the four lanes that
// hold a token's 16 trade them (the MFMA wants column 4 j + lane / 16).
//
// Bound by the chain of MFMAs, 8 cycles per column, and the first loads.  Measured
// (us), in brackets one thread per token and a few experts with the operands
// through LDS, which waited for every LDS read: 2048 tokens x 512, 8 experts 7.0
// (11.8), 64 experts 9.3 (43); 64 x 1024, 64 experts 13.5 (82); 16384 x 1024, 128
// experts 88 (577); 4000 x 320, 24 experts 6.6 (16.6); bf16, 20000 x 700, 64 experts
// 38 (259).
// ---------------------------------------------------------------------------
constexpr int RL_MAX_EXPERTS = 128;      // of a router_logits call
typedef __attribute__((ext_vector_type(4))) float rl_f32x4_t;

template <typename T>
__device__ __forceinline__ void load_f32x4(const T* p, float (&v)[4]);
template <>
__device__ __forceinline__ void load_f32x4<float>(const float* p,
                                                  float (&v)[4]) {
  const float4 q = *reinterpret_cast<const float4*>(p);
  v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
}
template <>
__device__ __forceinline__ void load_f32x4<bf16_t>(const bf16_t* p,
                                                   float (&v)[4]) {
  const uint2 q = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(q.x << 16); v[1] = __uint_as_float(q.x & 0xffff0000u);
  v[2] = __uint_as_float(q.y << 16); v[3] = __uint_as_float(q.y & 0xffff0000u);
}

template <typename T, bool VEC>
__global__ __launch_bounds__(256) void router_logits_kernel(
    const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ bias, float* __restrict__ logits,
    int64_t tokens, int M, int E) {
  constexpr int PF = 8;
  const int b = blockIdx.z;
  const int64_t t0 = (int64_t)blockIdx.x * 16;
  const int lane = threadIdx.x & 63, col = lane & 15, h = lane >> 4;
  const int e0 = (blockIdx.y * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 16;
  if (e0 >= E) return;
  // tokens and experts past the end are read as the last ones, not stored
  const T* xt = x + ((int64_t)b * tokens + min(t0 + col, tokens - 1)) * M;
  const T* we = w + (int64_t)b * M * E + min(e0 + col, E - 1);
  float xr[PF][4], wr[PF][4];
  // a group of 16 columns: WHOLE, or with what lies past M clamped
  const T* xh = xt + (VEC ? 4 * h : h);
  const T* wh = we + (int64_t)h * E;
  auto load = [&](int k0, float (&xv)[4], float (&wv)[4], auto whole_c) {
    constexpr bool WHOLE = decltype(whole_c)::value;
    if (VEC) {
      load_f32x4<T>(WHOLE ? xh + k0 : xt + min(k0 + 4 * h, M - 4), xv);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xv[j] = load_f32<T>(WHOLE ? xh + k0 + 4 * j
                                  : xt + min(k0 + 4 * j + h, M - 1));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      wv[j] = load_f32<T>(WHOLE ? wh + (int64_t)(k0 + 4 * j) * E
                                : we + (int64_t)min(k0 + 4 * j + h, M - 1) * E);
  };
  rl_f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int k0, float (&xv)[4], float (&wv)[4], auto whole_c) {
    constexpr bool WHOLE = decltype(whole_c)::value;
    if (VEC) {
      auto swap = [](auto fn, float& p, float& q) {
        const auto r = fn(__float_as_uint(p), __float_as_uint(q));
        p = __uint_as_float(r[0]);
        q = __uint_as_float(r[1]);
      };
      auto swap32 = [](uint32_t p, uint32_t q) {
        return __builtin_amdgcn_permlane32_swap(p, q, false, false);
      };
      auto swap16 = [](uint32_t p, uint32_t q) {
        return __builtin_amdgcn_permlane16_swap(p, q, false, false);
      };
      swap(swap32, xv[0], xv[2]);
      swap(swap32, xv[1], xv[3]);
      swap(swap16, xv[0], xv[1]);
      swap(swap16, xv[2], xv[3]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = WHOLE || k0 + 4 * j + h < M;      // past M: 0 * 0
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? wv[j] : 0.f,
                                                 in ? xv[j] : 0.f, acc, 0, 0, 0);
    }
  };
  using Whole = std::true_type;
  using Rest = std::false_type;
#pragma unroll
  for (int u = 0; u < PF; ++u) load(u * 16, xr[u], wr[u], Rest());
  int k0 = 0;
  for (; k0 + 32 * PF <= M; k0 += 16 * PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      multiply(k0 + 16 * u, xr[u], wr[u], Whole());
      load(k0 + 16 * (u + PF), xr[u], wr[u], Whole());
    }
  }
  for (; k0 < M; k0 += 16 * PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      if (k0 + 16 * u < M) multiply(k0 + 16 * u, xr[u], wr[u], Rest());
      if (k0 + 16 * (u + PF) < M)
        load(k0 + 16 * (u + PF), xr[u], wr[u], Rest());
    }
  }
  const int64_t t = t0 + col;
  if (t >= tokens) return;
  float* out = logits + ((int64_t)b * tokens + t) * E;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int e = e0 + 4 * h + r;
    if (e < E) out[e] = bias ? acc[r] + bias[e] : acc[r];
  }
}

// ---------------------------------------------------------------------------
// Router logits on the matrix cores (bf16 inputs, packed router weights
// wp[b][e][m]).  logits^T tile = wp tile (experts as MFMA rows) x x tile (tokens
// as MFMA columns): lane l ends up with token l % 32 of its wavefront and, per
// 32-expert tile, experts 8*(r/4) + 4*(l/32) + r%4 in accumulator register r.
// bf16 x bf16 products are exact in float32, so this is the float32 matmul of
// the reference on bf16-rounded operands up to summation order.
//
// A block is 4 wavefronts x 32 tokens; x and wp K tiles (64 deep) are brought
// into a three-slot LDS ring by global_load_lds_dwordx4 with the same
// 128-byte-row XOR swizzle as the expert GEMM.  The kernel is bound by reading
// x once from HBM.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(8))) __bf16 rl_bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float rl_f32x16_t;
typedef __attribute__((address_space(3))) void rl_lds_void_t;
typedef const __attribute__((address_space(1))) void rl_glb_void_t;

// Cache-policy operand of the direct-to-LDS loads of the token tile: the
// non-temporal hint.  Every token row is read exactly once by these kernels;
// with the hint the fused router kernel runs 8 % faster (0.121 -> 0.112 ms at
// 65536 tokens x 4096).  The router weights keep the default policy: every
// block re-reads them from the L2.
constexpr int RL_STREAMING = 2;

__device__ __forceinline__ int rl_swizzle(int row) {
  return (row & 7) ^ ((row >> 3) & 1);
}

// Writes a block's 128 x E logits as whole rows.  The matrix cores leave a
// token's row spread over two lanes in groups of four experts (v[j][4 q + r]
// = expert 32 j + 8 q + 4 (lane / 32) + r of token wave * 32 + lane % 32);
// stored straight from there a store instruction writes 32-byte pieces 4 E
// bytes apart, the 128-byte lines reach the L2 in quarters and the 16.8 MB of
// logits of 65536 tokens x 64 experts cost 10 us.  Here the values go through
// LDS (stage: [128][E + 4] floats, any earlier use of it over) and leave as
// consecutive 16-byte pieces, whole lines per instruction (the 16.8 MB then
// cost 2 us).  rows: how many of the block's 128 tokens exist; out: their
// first row.  Ends with a barrier: the caller may reuse `stage` at once.
template <int NT, typename V>  // V: float[16] or a 16-float vector
__device__ __forceinline__ void store_logits_rows(const V (&v)[NT],
                                                  float* stage, int E,
                                                  float* __restrict__ out,
                                                  int rows) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ld = E + 4;
  float* row = stage + (wave * 32 + (lane & 31)) * ld;
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e0 = j * 32 + 8 * q + 4 * (lane >> 5);
      if (e0 < E)
        *reinterpret_cast<float4*>(row + e0) = make_float4(
            v[j][4 * q], v[j][4 * q + 1], v[j][4 * q + 2], v[j][4 * q + 3]);
    }
  __syncthreads();
  const int per_row = E >> 2;                    // 16-byte pieces per row
  for (int c = tid; c < rows * per_row; c += (int)blockDim.x) {
    const int r = c / per_row, piece = c - r * per_row;
    store_streaming(reinterpret_cast<uint4*>(out + (int64_t)r * E + piece * 4),
                    *reinterpret_cast<const uint4*>(stage + r * ld + piece * 4));
  }
  __syncthreads();
}

template <int NT>  // number of 32-expert tiles: E <= 32 * NT
__global__ __launch_bounds__(256) void router_mfma_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ wp,
    const float* __restrict__ bias, float* __restrict__ logits, int tokens,
    int M, int E) {
  constexpr int TOK = 128, BK = 64, ROWB = 128;
  constexpr int X_BYTES = TOK * ROWB, W_BYTES = NT * 32 * ROWB;
  constexpr int STAGE = X_BYTES + W_BYTES;
  extern __shared__ __attribute__((aligned(16))) unsigned char rl_smem[];
  const int b = blockIdx.y;
  const int t0 = blockIdx.x * TOK;
  const bf16_t* xb = x + (int64_t)b * tokens * M;
  const bf16_t* wb = wp + (int64_t)b * E * M;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // load instruction q covers tile rows 8q..8q+7; lane l fills slot
  // (row 8q + l/8, column l%8) and fetches chunk (l%8) ^ swizzle(row)
  int x_off[4], w_off[NT];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = (wave + 4 * j) * 8 + (lane >> 3);
    x_off[j] = min(t0 + row, tokens - 1) * M + (((lane & 7) ^ rl_swizzle(row)) * 8);
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int row = (wave + 4 * j) * 8 + (lane >> 3);
    w_off[j] = min(row, E - 1) * M + (((lane & 7) ^ rl_swizzle(row)) * 8);
  }
  // Block b walks the K tiles starting at tile b % nk and wraps around: the
  // blocks run in step, and with rows a power of two apart all of them asking
  // for the same 128-byte column of their rows at the same moment lands on
  // few memory channels (measured: 20 % slower).
  const int nk = M / BK;
  const int rot = (int)(blockIdx.x % (unsigned)nk);
  auto issue = [&](int kt, int slot) {
    unsigned char* sx = rl_smem + slot * STAGE;
    unsigned char* sw = sx + X_BYTES;
    int kq = kt + rot;
    if (kq >= nk) kq -= nk;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_global_load_lds(
          (rl_glb_void_t*)(xb + kq * BK + x_off[j]),
          (rl_lds_void_t*)(sx + (wave + 4 * j) * 1024), 16, 0, RL_STREAMING);
#pragma unroll
    for (int j = 0; j < NT; ++j)
      __builtin_amdgcn_global_load_lds(
          (rl_glb_void_t*)(wb + kq * BK + w_off[j]),
          (rl_lds_void_t*)(sw + (wave + 4 * j) * 1024), 16, 0, 0);
  };

  rl_f32x16_t acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;

  const int fr = lane & 31, fc = lane >> 5;
  int x_frag[4], w_frag[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int col = ((kk * 2 + fc) ^ rl_swizzle(fr)) * 16;
    x_frag[kk] = (wave * 32 + fr) * ROWB + col;
    w_frag[kk] = fr * ROWB + col;
  }
  // Three slots, two K tiles in flight: the loop is bound by the latency of
  // one round trip to HBM per K tile, so what it moves per second is the bytes
  // it keeps in flight.  vmcnt retires in issue order: leaving the newest
  // tile's 4 + NT loads outstanding means tile kt has landed.  Passing the
  // barrier of step kt also means every wavefront has finished reading slot
  // (kt - 1) % 3, which the loads of tile kt + 2 then overwrite.
  issue(0, 0);
  if (nk > 1) issue(1, 1);
  int slot = 0;
  for (int kt = 0; kt < nk; ++kt) {
    if (kt + 1 < nk)
      __builtin_amdgcn_s_waitcnt(0x0070 | (4 + NT));  // vmcnt(4+NT) lgkmcnt(0)
    else
      __builtin_amdgcn_s_waitcnt(0x0070);             // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + 2 < nk) issue(kt + 2, slot == 0 ? 2 : slot - 1);
    const unsigned char* sx = rl_smem + slot * STAGE;
    slot = slot == 2 ? 0 : slot + 1;
    const unsigned char* sw = sx + X_BYTES;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const rl_bf16x8_t xf = *reinterpret_cast<const rl_bf16x8_t*>(sx + x_frag[kk]);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const rl_bf16x8_t wf =
            *reinterpret_cast<const rl_bf16x8_t*>(sw + w_frag[kk] + j * 32 * ROWB);
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, xf, acc[j], 0, 0, 0);
      }
    }
  }
  __syncthreads();  // every wavefront is done with the ring: reuse it
  if (bias != nullptr) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        // E % 4 == 0, so the four experts are in range together
        const int e0 = min(j * 32 + 8 * q + 4 * (lane >> 5), E - 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[j][4 * q + r] += bias[e0 + r];
      }
  }
  store_logits_rows<NT>(acc, reinterpret_cast<float*>(rl_smem), E,
                        logits + ((int64_t)b * tokens + t0) * E,
                        min(TOK, tokens - t0));
}

// The same products for few tokens, in the same order (the bits of router_mfma_kernel): a
// wavefront per 32 tokens and 32 experts, operands straight into registers.  A block of
// 128 tokens that has the whole chip to itself is bound by its chain of K tiles, a
// barrier and a round trip each; here two batches of four K tiles are in flight and
// nobody waits for another wavefront: 64 tokens of 4096, 64 experts 31.9 -> 16.4 us.
__global__ __launch_bounds__(64) void router_few_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ wp,
    const float* __restrict__ bias, float* __restrict__ logits, int tokens,
    int M, int E) {
  constexpr int BK = 64, TILES = 4;
  const int lane = threadIdx.x, fr = lane & 31, fc = lane >> 5;
  const int t0 = blockIdx.x * 32, e0 = blockIdx.y * 32, b = blockIdx.z;
  const int tok = t0 + fr;
  const bf16_t* xr = x + ((int64_t)b * tokens + min(tok, tokens - 1)) * M + fc * 8;
  const bf16_t* wr = wp + ((int64_t)b * E + min(e0 + fr, E - 1)) * M + fc * 8;
  const int nk = M / BK;
  const int rot = (t0 / 128) % nk;            // where router_mfma_kernel starts
  struct Batch { rl_bf16x8_t x[TILES * 4], w[TILES * 4]; };
  auto load = [&](Batch& f, int kt) {
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      int kq = min(kt + i, nk - 1) + rot;     // (past the end: read, not used)
      if (kq >= nk) kq -= nk;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        f.x[i * 4 + kk] =
            *reinterpret_cast<const rl_bf16x8_t*>(xr + kq * BK + kk * 16);
        f.w[i * 4 + kk] =
            *reinterpret_cast<const rl_bf16x8_t*>(wr + kq * BK + kk * 16);
      }
    }
  };
  rl_f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  auto multiply = [&](const Batch& f, int kt) {
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      if (kt + i >= nk) return;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[i * 4 + kk],
                                                      f.x[i * 4 + kk], acc, 0, 0, 0);
    }
  };
  Batch even, odd;
  int kt = 0;
  load(even, 0);
  for (; kt + 2 * TILES < nk; kt += 2 * TILES) {
    load(odd, kt + TILES);
    multiply(even, kt);
    load(even, kt + 2 * TILES);
    multiply(odd, kt + TILES);
  }
  if (kt + TILES < nk) {
    load(odd, kt + TILES);
    multiply(even, kt);
    multiply(odd, kt + TILES);
  } else {
    multiply(even, kt);
  }
  if (tok >= tokens) return;
  float* out = logits + ((int64_t)b * tokens + tok) * E;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = e0 + 8 * q + 4 * fc;        // E % 4 == 0: all four or none
    if (e >= E) continue;
    float4 v = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2],
                           acc[4 * q + 3]);
    if (bias != nullptr) {
      v.x += bias[e]; v.y += bias[e + 1]; v.z += bias[e + 2]; v.w += bias[e + 3];
    }
    *reinterpret_cast<float4*>(out + e) = v;
  }
}

// ---------------------------------------------------------------------------
// Gating step 1: per token softmax, top-2, gate normalisation, second-place
// policy; per block column sums of the balancing-loss proxies.
// Grid (blocks per group, G).
// ---------------------------------------------------------------------------
// Accesses that are coherent across the GPU's compute dies without a cache
// flush.  Each die (XCD) has its own L2; an ordinary store may sit there, and
// an ordinary load may hit a stale line there, until a device-scope fence
// writes back / invalidates that whole L2 -- too expensive to issue from
// every block of a kernel whose other blocks are still streaming through the
// same L2.  A relaxed atomic store / load at device scope is a write-through
// store / a load that bypasses lines the L2 cannot vouch for.  The blocks of
// the single-launch gating kernel exchange their data only through these:
// the writer waits until its stores have completed (vmcnt 0) before it bumps
// the arrival counter, the reader loads after it has seen the counter.
template <typename T>
__device__ __forceinline__ void st_dev(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T ld_dev(const T* p) {
  return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long pack_i2(int a, int b) {
  return (unsigned long long)(unsigned)a | ((unsigned long long)(unsigned)b << 32);
}
__device__ __forceinline__ unsigned long long pack_f2(float a, float b) {
  return pack_i2((int)__float_as_uint(a), (int)__float_as_uint(b));
}
// this wavefront's global stores (and loads) have completed
__device__ __forceinline__ void wait_stores() {
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0), nothing else
  asm volatile("" ::: "memory");
}

struct GateParams {
  int G, S, E, C;
  int policy;
  float threshold;      // float32(threshold)            (moe.py:1460)
  float inv_threshold;  // float32(1 / max(thr, 1e-9))   (moe.py:1465)
  int use_second_place_loss;
  int num_microbatches;
  int importance_from_slot_gate;  // importance = 0.5*((w>0.5)+(w>0))
  int tt;    // tokens per block of step 1
  int nblk;  // blocks per group of step 1
  int router;          // ROUTER_TOP2 or ROUTER_SWITCH
  int has_importance;  // switch loss: the proxy is masked per token
  int use_z_loss;      // switch: add z_loss_coef * z_loss (moe.py:1253-1266)
  float z_loss_coef;
  int rank_by_gate;    // switch_max: slots by descending gate (moe.py:1033-1039)
};

constexpr int ROUTER_TOP2 = 0;    // _top_2_gating, moe.py:1312-1513
constexpr int ROUTER_SWITCH = 1;  // _switch_gating, moe.py:1176-1309
constexpr int GSUM = 4;  // floats per group: loss term 1, term 2, #(imp==1), z
// Largest group every gating entry accepts (the reference's moe_group_size
// defaults to 1024, moe.py:139).  The capacity kernel keeps a group's expert
// ids in LDS (6 bytes per token) and the one-launch tail keeps slot prefixes
// in 16 bits: both rely on it.
constexpr int GATE_MAX_GROUP = 16384;

// bit 0 of the step-1 `kept` byte: the token competes for a slot (mask_k after
// importance and policy); bit 1 (second choice only): mask_2 before the policy,
// which is what the second-place loss counts (moe.py:1430).

// ---------------------------------------------------------------------------
// gate_select_kernel's work for the projection kernel, straight from the
// matrix-core accumulators: 256 threads, 128 tokens, two lanes per token.
// After the 32x32x16 MFMAs lane l of a wavefront holds, for token l % 32 and per
// 32-expert tile j, the logits of experts 32 j + 8 q + 4 (l / 32) + r (q, r =
// 0..3): lanes l and l + 32 together hold the token's whole row, in alternating
// groups of four experts.  Each lane does the exponentials of its half (two per
// expert, the bulk of the work); every float32 sum still runs in expert order
// (the running sum changes lanes after every group of four) and a tie between
// the two lanes' arg-max candidates goes to the lower expert, so every
// per-token result is bit for bit that of gate_select_kernel.  The probabilities
// go to LDS (tile [128][ld], ld % 4 == 0) for the per-block column sums of the
// loss, which are split over four row ranges; colpart: LDS [4][E] floats.
// ---------------------------------------------------------------------------
template <int NT, typename IT>
__device__ __forceinline__ void gate_select_acc_tile(
    const float (&xin)[NT][16], float* tile, float* isone, int ld, int g,
    int blk, int t0, const IT* __restrict__ importance,
    const float* __restrict__ second_uniform, const GateParams& p,
    int32_t* __restrict__ idx, int32_t* __restrict__ pos,
    float* __restrict__ gate, uint8_t* __restrict__ kept,
    float* __restrict__ part1, float* __restrict__ part2, int16_t* ch,
    float* colpart) {
  constexpr int NTOK = 128;
  const int E = p.E, S = p.S;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5;
  const int tok = wave * 32 + (lane & 31);
  const bool sw = p.router == ROUTER_SWITCH;
  float* row = tile + tok * ld;
  const int64_t t = (int64_t)g * S + t0 + tok;
  // As the matrix cores leave them, register group (j, q) of the lower lane of
  // a token's pair holds experts 32 j + 8 q + 0..3 and the upper lane's
  // + 4..7: a sum in expert order changes lanes after every four experts.
  // With an even number of 32-expert blocks the pair first trades registers
  // (v_permlane32_swap: the upper half of one register against the lower half
  // of another), after which the lower lane holds the whole of block 2 jp in
  // its groups (2 jp, q), (2 jp + 1, q) -- experts 8 q + 0..3 and 8 q + 4..7 --
  // and the upper lane the whole of block 2 jp + 1: a sum in expert order then
  // changes lanes once per 32 experts.
  constexpr bool SWAPPED = NT % 2 == 0;
  float x[NT][16];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) x[j][i] = xin[j][i];
  if constexpr (SWAPPED) {
#pragma unroll
    for (int jp = 0; jp < NT / 2; ++jp)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const auto sw2 = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(x[2 * jp][i]), __float_as_uint(x[2 * jp + 1][i]),
            false, false);
        x[2 * jp][i] = __uint_as_float(sw2[0]);
        x[2 * jp + 1][i] = __uint_as_float(sw2[1]);
      }
  }
  // first expert of this lane's group (j, q); the group exists if it is < E
  auto first = [&](int j, int q) {
    return SWAPPED ? ((j & ~1) + half) * 32 + 8 * q + 4 * (j & 1)
                   : j * 32 + 8 * q + 4 * half;
  };
  // calls fn(j, q) for the lane's groups in ascending expert order
  auto for_groups = [&](auto fn) {
    if constexpr (SWAPPED) {
#pragma unroll
      for (int jp = 0; jp < NT / 2; ++jp)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          fn(2 * jp, q);
          fn(2 * jp + 1, q);
        }
    } else {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) fn(j, q);
    }
  };
  // the partner's candidate wins if it is larger, or equal with a lower index
  auto take_other = [&](float mine, int mi, float other, int oi) {
    return other > mine || (other == mine && oi < mi);
  };
  // a float32 sum over the experts in index order: the lanes of a pair take
  // turns, the running value changing lanes when the next expert lives in the
  // other lane
  auto ordered_sum = [&](const float (&v)[NT][16]) {
    float s = 0.f;
    if constexpr (SWAPPED) {
#pragma unroll
      for (int jp = 0; jp < NT / 2; ++jp)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          if (half == hh) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
              for (int jj = 0; jj < 2; ++jj)
                if (first(2 * jp + jj, q) < E) {
#pragma unroll
                  for (int r = 0; r < 4; ++r) s += v[2 * jp + jj][4 * q + r];
                }
          }
          s = __shfl_xor(s, 32);
        }
    } else {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bool mine = first(j, q) < E;
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            if (half == hh && mine) {
#pragma unroll
              for (int r = 0; r < 4; ++r) s += v[j][4 * q + r];
            }
            s = __shfl_xor(s, 32);
          }
        }
    }
    return __shfl(s, lane & 31);      // the lower lane holds the final value
  };

  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (first(j, q) < E) {
#pragma unroll
        for (int r = 0; r < 4; ++r) m = fmaxf(m, x[j][4 * q + r]);   // reduce_max
      }
  m = fmaxf(m, __shfl_xor(m, 32));
  const float negm = -m;
  float pr[NT][16];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) pr[j][i] = expf(x[j][i] + negm);    // exp
  const float ssum = ordered_sum(pr);                                // reduce_sum
  const float neglse = -(logf(ssum) + m);                            // log + max
  float g1 = -1.f;
  int i1 = 0;
  for_groups([&](int j, int q) {
    if (first(j, q) < E) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pe = expf(x[j][4 * q + r] + neglse);   // exp(log_softmax)
        pr[j][4 * q + r] = pe;
        if (pe > g1) { g1 = pe; i1 = first(j, q) + r; }    // first argmax
      }
      *reinterpret_cast<float4*>(row + first(j, q)) = make_float4(
          pr[j][4 * q], pr[j][4 * q + 1], pr[j][4 * q + 2], pr[j][4 * q + 3]);
    }
  });
  {
    const float og = __shfl_xor(g1, 32);
    const int oi = __shfl_xor(i1, 32);
    if (take_other(g1, i1, og, oi)) { g1 = og; i1 = oi; }
  }
  bool sel1 = true;
  if (sw && second_uniform != nullptr) {
    // policy "sample": first arg-max of the caller's choice logits
    const float* cl = second_uniform + t * E;
    float best = -INFINITY;
    int bi = E;
    for_groups([&](int j, int q) {
      if (first(j, q) < E) {
        const float4 c4 = *reinterpret_cast<const float4*>(cl + first(j, q));
        const float cv[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (bi == E || cv[r] > best) { best = cv[r]; bi = first(j, q) + r; }
      }
    });
    const float ob = __shfl_xor(best, 32);
    const int oi = __shfl_xor(bi, 32);
    if (take_other(best, bi, ob, oi)) bi = oi;
    i1 = bi;
    __syncthreads();           // the partner's half of the row is in LDS
    g1 = row[i1];
  }
  float qscale = 0.f, zterm = 0.f;
  if (sw) {
    if (importance != nullptr)
      sel1 = (load_f32<IT>(importance + t) == 1.0f);
    if (!sel1) g1 = g1 * 0.0f;
    if (half == 0) {
      st_dev(reinterpret_cast<unsigned long long*>(idx + t * 2), pack_i2(i1, 0));
      st_dev(reinterpret_cast<unsigned long long*>(gate + t * 2),
             pack_f2(g1, 0.0f));
    } else {
      st_dev(reinterpret_cast<uint16_t*>(kept + t * 2),
             (uint16_t)((sel1 ? 1 : 0) | 2));
      if (ch == nullptr) {
        *reinterpret_cast<int2*>(pos + t * 2) = make_int2(0, 0);
      } else {
        ch[tok] = sel1 ? (int16_t)i1 : (int16_t)-1;
        ch[NTOK + tok] = -1;
        ch[2 * NTOK + tok] = (int16_t)i1;
      }
      isone[tok] = 1.0f;
    }
    const float lse = -neglse;
    zterm = sel1 ? lse * lse : 0.0f;
  } else {
    bool sel2 = true;
    if (importance != nullptr) {
      float imp = load_f32<IT>(importance + t);
      if (p.importance_from_slot_gate)
        imp = 0.5f * ((imp > 0.5f ? 1.0f : 0.0f) + (imp > 0.0f ? 1.0f : 0.0f));
      sel1 = (imp == 1.0f);
      sel2 = (imp > 0.0f);
    }
    if (!sel1) g1 = g1 * 0.0f;
    // gates_without_top_1 = raw_gates * (1 - mask_1), in place; its first argmax
    float g2 = -1.f;
    int i2 = 0;
    for_groups([&](int j, int q) {
      if (first(j, q) < E) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int e = first(j, q) + r;
          const float keep = (sel1 && e == i1) ? 0.0f : 1.0f;
          const float qv = pr[j][4 * q + r] * keep;
          pr[j][4 * q + r] = qv;
          if (qv > g2) { g2 = qv; i2 = e; }
        }
      }
    });
    {
      const float og = __shfl_xor(g2, 32);
      const int oi = __shfl_xor(i2, 32);
      if (take_other(g2, i2, og, oi)) { g2 = og; i2 = oi; }
    }
    const float denom = (g1 + g2) + 1e-9f;
    const float r = 1.0f / denom;
    const float g1n = g1 * r, g2n = g2 * r;
    const bool sel2_loss = sel2;
    if (p.policy == MESH_MOE_SECOND_NONE) {
      sel2 = false;
    } else if (p.policy == MESH_MOE_SECOND_THRESHOLD) {
      sel2 = sel2 && (g2n > p.threshold);
    } else if (p.policy == MESH_MOE_SECOND_RANDOM) {
      sel2 = sel2 && (second_uniform[t] < g2n * p.inv_threshold);
    }
    if (half == 0) {
      st_dev(reinterpret_cast<unsigned long long*>(idx + t * 2), pack_i2(i1, i2));
      st_dev(reinterpret_cast<unsigned long long*>(gate + t * 2),
             pack_f2(g1n, g2n));
    } else {
      st_dev(reinterpret_cast<uint16_t*>(kept + t * 2), (uint16_t)(
          (sel1 ? 1 : 0) | ((sel2 ? 1 : 0) | (sel2_loss ? 2 : 0)) << 8));
      if (ch == nullptr) {
        *reinterpret_cast<int2*>(pos + t * 2) = make_int2(0, 0);
      } else {
        ch[tok] = sel1 ? (int16_t)i1 : (int16_t)-1;
        ch[NTOK + tok] = sel2 ? (int16_t)i2 : (int16_t)-1;
        ch[2 * NTOK + tok] = sel2_loss ? (int16_t)i2 : (int16_t)-1;
      }
      isone[tok] = sel1 ? 1.0f : 0.0f;
    }
    if (p.use_second_place_loss)
      qscale = 1.0f / (ordered_sum(pr) + 1e-9f);            // moe.py:1433-1434
  }
  __syncthreads();
  // column sums over the block's tokens, four row ranges per column
  auto column_sums = [&](int ncol, bool weighted, float* out) {
    for (int i = tid; i < 4 * ncol; i += blockDim.x) {
      const int e = i % ncol, q4 = i / ncol;
      float acc = 0.f;
      // (the reads of a batch fly together; the additions keep their order)
      const float* col = tile + q4 * (NTOK / 4) * ld + e;
      const float* one = isone + q4 * (NTOK / 4);
#pragma unroll 8
      for (int r = 0; r < NTOK / 4; ++r)
        acc += weighted ? col[r * ld] * one[r] : col[r * ld];
      colpart[q4 * ncol + e] = acc;
    }
    __syncthreads();
    for (int e = tid; e < ncol; e += blockDim.x)
      st_dev(out + ((int64_t)g * p.nblk + blk) * E + e,
             ((colpart[e] + colpart[ncol + e]) + colpart[2 * ncol + e]) +
                 colpart[3 * ncol + e]);
  };
  column_sums(E, true, part1);       // density_1_proxy: p * (imp == 1)
  if (sw) {
    // z-loss: column 0 = sum of logsumexp^2 over the tokens of importance 1,
    // column 1 = how many those are
    __syncthreads();
    if (half == 0) {
      row[0] = zterm;
      row[1] = sel1 ? 1.0f : 0.0f;
    }
    __syncthreads();
    column_sums(2, false, part2);
  } else if (p.use_second_place_loss) {
    // the proxy of the second-place loss: (gates without the first) / their sum
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (first(j, q) < E)
          *reinterpret_cast<float4*>(row + first(j, q)) = make_float4(
              pr[j][4 * q] * qscale, pr[j][4 * q + 1] * qscale,
              pr[j][4 * q + 2] * qscale, pr[j][4 * q + 3] * qscale);
    __syncthreads();
    column_sums(E, false, part2);
  }
}

// ---------------------------------------------------------------------------
// Step 1 from logits in memory.  A block of 1024 threads has LANES lanes per token;
// lane l does the exponentials and comparisons of experts l, l + LANES, ...  The two
// sums over a token's experts that decide its gates still run in expert order, read
// back from LDS (every lane of the token runs the same chain), and a tie between two
// lanes' candidates goes to the lower expert: the per-token results do not depend on
// the split.  One thread per token walking its row was a chain of four passes of E
// dependent steps, and 256 tokens per block left most compute units without one:
// 64 tokens of 64 experts 17.6 -> 8.2 us with sixteen lanes, 6 groups of 1500 tokens,
// 16 experts 16.5 -> 6.8 us.
// Launches that fill the chip anyway pay for what the lanes of a token do alike (the
// chain), the more of it the fewer experts there are.  The whole gating in us, 16 / 8
// / 4 lanes (one thread per token before): 65536 tokens, 16 experts 28.9, 22.7, 23.5
// (28), 64 experts 36, 32, 34; 131072 tokens, 16 experts 44, 36, 32; 524288 tokens, 8
// experts 141, 106, 92 (94), 16 experts 138, 99, 88 (93), 32 experts 150, 127, 129
// (113), 64 experts 184, 161, 171, 128 experts 310, 280, 271.
// ---------------------------------------------------------------------------
constexpr int SELECT_THREADS = 1024;

// Tokens per block of step 1 from logits in memory: SELECT_THREADS / LANES.  (The
// probabilities of 128 tokens lie in LDS twice per compute unit up to 128 experts.)
static int select_tokens(int G, int S, int E) {
  const int64_t tokens = (int64_t)G * S;
  if (tokens < 65536 || E > 128) return 64;
  return tokens >= 131072 && E <= 24 ? 256 : 128;
}

__host__ __device__ constexpr int select_row_floats(int E) {
  return (E + 3) / 4 * 4 + 4;            // 16-byte rows, odd in units of 16 bytes
}                                        // for E = 8 n

// Where step 1 leaves the records and the partial sums of the loss.  RECORD_TAIL: another
// block of the launch reads them (device-scope stores, see st_dev); the choices also go
// to ch [3][TOKENS] in LDS (-1: not competing; the third: what the loss counts), and
// `pos` is left to gate_rank_block.  RECORD_LDS: the same block finishes them; idx [64][2],
// gate [64][2], ch and the parts [E] are LDS, pos and kept are left to it.
constexpr int RECORD_MEMORY = 0, RECORD_TAIL = 1, RECORD_LDS = 2;
template <typename IT, int LANES, int RECORD = RECORD_MEMORY>
__device__ __forceinline__ void gate_select_block(
    const float* logits, const IT* importance, const float* second_uniform,
    const GateParams& p, int32_t* idx, int32_t* pos, float* gate, uint8_t* kept,
    float* part1, float* part2, float* smem, int16_t* ch = nullptr) {
  constexpr int TOKENS = SELECT_THREADS / LANES;
  const int E = p.E, S = p.S;
  const int ld = select_row_floats(E);
  float* tile = smem;                                  // [TOKENS][ld]
  float* isone = tile + TOKENS * ld;            // [TOKENS]
  float* cols = isone + TOKENS;                 // [SELECT_THREADS]
  const int g = blockIdx.y, blk = blockIdx.x;
  const int t0 = blk * TOKENS;
  const int ntok = min(TOKENS, S - t0);
  const int tid = threadIdx.x, lane = tid % LANES;
  const int tok = tid / LANES;
  const bool live = tok < ntok;
  // experts this lane walks: none for a token that does not exist
  const int e_end = live ? E : 0;
  const int64_t t = (int64_t)g * S + t0 + (live ? tok : 0);
  // A block that has the chip to itself reads its logits from memory once, where they fit
  // REGS registers, and several experts of a sum at a time.  (gate_logits_kernel has no
  // registers to spare: 2 x 1024 tokens, 8 experts 11.6 us, with the same 12.4.)
  constexpr bool ALONE = RECORD == RECORD_LDS;
  constexpr int REGS = ALONE ? 8 : 1;
  const float* src = logits + t * E;
  const bool in_regs = ALONE && E <= REGS * LANES;
  float x[REGS];
#pragma unroll
  for (int i = 0; i < REGS; ++i)
    x[i] = in_regs && lane + i * LANES < e_end ? src[lane + i * LANES] : -INFINITY;
  // fn(expert, logit) for the experts of this lane, in ascending order
  auto for_logits = [&](auto fn) {
    if (in_regs) {
#pragma unroll
      for (int i = 0; i < REGS; ++i)
        if (lane + i * LANES < e_end) fn(lane + i * LANES, x[i]);
    } else {
      for (int e = lane; e < e_end; e += LANES) fn(e, src[e]);
    }
  };
  float* row = tile + tok * ld;
  const bool sw = p.router == ROUTER_SWITCH;
  // the token's record (by one lane of a token that exists): choices, gates, the two
  // `kept` bytes and what the loss counts
  auto write_record = [&](int i1, int i2, float g1, float g2, unsigned k1,
                          unsigned k2, int third) {
    if constexpr (RECORD == RECORD_LDS) {
      idx[tok * 2] = i1;
      idx[tok * 2 + 1] = i2;
      gate[tok * 2] = g1;
      gate[tok * 2 + 1] = g2;
      ch[tok] = (k1 & 1) ? (int16_t)i1 : (int16_t)-1;
      ch[TOKENS + tok] = (k2 & 1) ? (int16_t)i2 : (int16_t)-1;
      ch[2 * TOKENS + tok] = (int16_t)third;
    } else if constexpr (RECORD == RECORD_TAIL) {
      st_dev(reinterpret_cast<unsigned long long*>(idx + t * 2), pack_i2(i1, i2));
      st_dev(reinterpret_cast<unsigned long long*>(gate + t * 2), pack_f2(g1, g2));
      st_dev(reinterpret_cast<uint16_t*>(kept + t * 2), (uint16_t)(k1 | k2 << 8));
      ch[tok] = (k1 & 1) ? (int16_t)i1 : (int16_t)-1;
      ch[TOKENS + tok] = (k2 & 1) ? (int16_t)i2 : (int16_t)-1;
      ch[2 * TOKENS + tok] = (int16_t)third;
    } else {
      idx[t * 2 + 0] = i1;
      idx[t * 2 + 1] = i2;
      pos[t * 2 + 0] = 0;
      pos[t * 2 + 1] = 0;
      gate[t * 2 + 0] = g1;
      gate[t * 2 + 1] = g2;
      kept[t * 2 + 0] = (uint8_t)k1;
      kept[t * 2 + 1] = (uint8_t)k2;
    }
  };
  auto write_part = [&](float* at, float v) {
    if constexpr (RECORD == RECORD_TAIL) st_dev(at, v);
    else *at = v;
  };
  const int64_t part_at = RECORD == RECORD_LDS ? 0 : ((int64_t)g * p.nblk + blk) * E;

  float m = -INFINITY;
  for_logits([&](int, float v) { m = fmaxf(m, v); });
#pragma unroll
  for (int d = 1; d < LANES; d *= 2) m = fmaxf(m, __shfl_xor(m, d));
  const float negm = -m;                                    // reduce_max
  for_logits([&](int e, float v) { row[e] = expf(v + negm); });
  __syncthreads();
  // exp, reduce_sum: in expert order
  float s = 0.f;
  if (live) {
    int e = 0;
    auto add4 = [&](int at) {
      const float4 v = *reinterpret_cast<const float4*>(row + at);
      s += v.x; s += v.y; s += v.z; s += v.w;
    };
    if constexpr (ALONE) {
#pragma unroll 4
      for (; e + 4 <= E; e += 4) add4(e);
    } else {
      for (; e + 4 <= E; e += 4) add4(e);
    }
    for (; e < E; ++e) s += row[e];
  }
  __syncthreads();
  // the larger value, of equal ones the lower expert
  auto first_max = [&](float& v, int& i) {
#pragma unroll
    for (int d = 1; d < LANES; d *= 2) {
      const float v2 = __shfl_xor(v, d);
      const int i2 = __shfl_xor(i, d);
      if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
    }
  };
  const float neglse = -(logf(s) + m);                      // log + max
  float g1 = -1.f;
  int i1 = 0;
  for_logits([&](int e, float v) {
    const float pe = expf(v + neglse);                      // exp(log_softmax)
    row[e] = pe;
    if (pe > g1) { g1 = pe; i1 = e; }                       // first argmax
  });
  first_max(g1, i1);
  __syncthreads();
  bool sel1 = live;
  float qscale = 0.f;
  if (sw) {
    if (second_uniform != nullptr) {
      // policy "sample" (moe.py:1213-1216): the expert is the first arg-max of
      // the caller's choice logits [G,S,E] (router logits plus Gumbel noise
      // times the temperature, ops.py:5070-5086), which arrive through the
      // pointer the top-2 mode uses for its uniform samples; the gate is the
      // softmax probability of that expert (mtf.gather of raw_gates)
      const float* ch = second_uniform + t * E;
      float best = -INFINITY;
      i1 = 0;
      for (int e = lane; e < e_end; e += LANES) {
        const float v = ch[e];
        if (v > best) { best = v; i1 = e; }
      }
      first_max(best, i1);
      // (nothing compares greater than a NaN in the first place)
      if (live && ch[0] != ch[0]) i1 = 0;
      if (live) g1 = row[i1];
    }
    // one choice, raw probability as the gate (moe.py:1207-1228); the load
    // balancing loss counts every token's arg-max (density_1 is taken
    // before the importance mask, moe.py:1224) and an unmasked proxy
    if (live && importance != nullptr)
      sel1 = (load_f32<IT>(importance + t) == 1.0f);
    if (!sel1) g1 = g1 * 0.0f;
    if (live && lane == 0) {
      // (bit 1: counted by density_1)
      write_record(i1, 0, g1, 0.0f, (sel1 ? 1u : 0u) | 2u, 0u, i1);
      isone[tok] = 1.0f;
    }
  } else {
    bool sel2 = live;
    if (live && importance != nullptr) {
      float imp = load_f32<IT>(importance + t);
      if (p.importance_from_slot_gate)                      // moe.py:725-727
        imp = 0.5f * ((imp > 0.5f ? 1.0f : 0.0f) + (imp > 0.0f ? 1.0f : 0.0f));
      sel1 = (imp == 1.0f);                                 // moe.py:1402-1404
      sel2 = (imp > 0.0f);                                  // moe.py:1411
    }
    if (!sel1) g1 = g1 * 0.0f;
    // gates_without_top_1 = raw_gates * (1 - mask_1); its first argmax.
    const int masked = sel1 ? i1 : -1;                      // 1 + (-mask_1)
    float g2 = -1.f;
    int i2 = 0;
    for (int e = lane; e < e_end; e += LANES) {
      const float q = row[e] * (e == masked ? 0.0f : 1.0f);
      if (q > g2) { g2 = q; i2 = e; }
    }
    first_max(g2, i2);
    if (p.use_second_place_loss && live) {
      float qsum = 0.f;
      for (int e = 0; e < E; ++e) qsum += row[e] * (e == masked ? 0.0f : 1.0f);
      qscale = 1.0f / (qsum + 1e-9f);                       // moe.py:1433-1434
    }
    const float denom = (g1 + g2) + 1e-9f;                  // moe.py:1413
    const float r = 1.0f / denom;                           // reciprocal
    const float g1n = g1 * r, g2n = g2 * r;
    const bool sel2_loss = sel2;
    if (live && lane == 0) {
      if (p.policy == MESH_MOE_SECOND_NONE) {
        sel2 = false;
      } else if (p.policy == MESH_MOE_SECOND_THRESHOLD) {
        sel2 = sel2 && (g2n > p.threshold);
      } else if (p.policy == MESH_MOE_SECOND_RANDOM) {
        sel2 = sel2 && (second_uniform[t] < g2n * p.inv_threshold);
      }
      write_record(i1, i2, g1n, g2n, sel1 ? 1u : 0u,
                   (sel2 ? 1u : 0u) | (sel2_loss ? 2u : 0u), sel2_loss ? i2 : -1);
      isone[tok] = sel1 ? 1.0f : 0.0f;
    }
  }
  // sums over the block's tokens, per expert: part[e] = sum of tile[r][e] *
  // (weights ? weights[r] : 1); the rows in up to 16 ranges, whose
  // sums are added in order
  auto column_sums = [&](const float* weights, float* part) {
    int el = 2;
    while (el < E) el *= 2;
    const int ranges = min(16, SELECT_THREADS / el);
    const int e = tid % el, c = tid / el;
    const int per = TOKENS / ranges;
    __syncthreads();
    if (e < E && c < ranges) {
      float a = 0.f;
      for (int r = c * per; r < min(ntok, (c + 1) * per); ++r)
        a += weights != nullptr ? tile[r * ld + e] * weights[r]
                                : tile[r * ld + e];
      cols[c * el + e] = a;
    }
    __syncthreads();
    if (tid < E) {
      float a = 0.f;
      if constexpr (ALONE) {
#pragma unroll 8
        for (int k = 0; k < ranges; ++k) a += cols[k * el + tid];
      } else {
        for (int k = 0; k < ranges; ++k) a += cols[k * el + tid];
      }
      write_part(part + part_at + tid, a);
    }
  };
  // density_1_proxy partial: sum over the block's tokens of p * (imp == 1)
  column_sums(isone, part1);
  if (sw) {
    // per-block sums for the z-loss: column 0 = sum of logsumexp^2 over the
    // tokens with importance 1, column 1 = how many those are
    __syncthreads();
    if (lane == 0) {
      const float lse = -neglse;                            // reduce_logsumexp
      cols[tok] = sel1 ? lse * lse : 0.0f;                  // moe.py:1256-1259
      cols[TOKENS + tok] = sel1 ? 1.0f : 0.0f;
    }
    __syncthreads();
    if (tid < 2) {
      float a = 0.f;
      for (int r = 0; r < ntok; ++r) a += cols[tid * TOKENS + r];
      write_part(part2 + part_at + tid, a);
    }
  } else if (p.use_second_place_loss) {
    __syncthreads();
    for (int e = lane; e < e_end; e += LANES)
      row[e] = (row[e] * (sel1 && e == i1 ? 0.0f : 1.0f)) * qscale;
    column_sums(nullptr, part2);
  }
}

template <typename IT, int LANES>
__global__ __launch_bounds__(SELECT_THREADS) void gate_select_kernel(
    const float* __restrict__ logits, const IT* __restrict__ importance,
    const float* __restrict__ second_uniform, GateParams p,
    int32_t* __restrict__ idx, int32_t* __restrict__ pos,
    float* __restrict__ gate, uint8_t* __restrict__ kept,
    float* __restrict__ part1, float* __restrict__ part2) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  gate_select_block<IT, LANES>(logits, importance, second_uniform, p, idx, pos,
                               gate, kept, part1, part2, smem);
}

// ---------------------------------------------------------------------------
// Capacity positions and the loss inside the projection kernel's launch.
//
// Every block ranks the choices of its own 128 tokens (gate_rank_tile: per
// expert a wavefront ballot over 64 tokens and the number of set bits below
// the lane, then the count of the block's other half) and publishes its
// per-expert counts.  The block of a group that arrives last at the group's
// counter (gate_group_tail) turns the counts into each block's first slot per
// expert, finishes every token of the group (slot = first slot of its block +
// rank in the block; second choices behind the kept first choices), writes
// `fill` and the group's loss term; the group that finishes last adds the
// terms up.  Nobody waits for anybody, so the scheme does not depend on which
// blocks are resident together.
//
// A counter is a 64-bit word: call number << 16 | arrivals.  A word that does
// not carry the current call's number counts as zero, so the workspace may
// hold anything when the call starts; the last arrival leaves zero behind.
// ---------------------------------------------------------------------------
struct GateParams;
template <bool COHERENT>
__device__ __forceinline__ void gate_loss_value(const GateParams& p,
                                                const float* gsum, float* loss);

struct FusedTail {
  int32_t* bcnt;              // [G][nblk][3][E] per-block counts
  unsigned long long* gctr;   // [G] arrivals per group
  unsigned long long* fctr;   // [1] groups done
  float* gsum;                // [G][GSUM]
  int32_t* fill;              // [G][E]
  float* loss;                // [1]
  unsigned long long call;    // number of this call, < 2^48, never 0
};

// Puts a counter word into this call's state "no arrivals yet", whatever it holds: zero
// where the last arrival of a call left it, anything where the workspace's memory has
// served something else since (between two passes of a training step it has).  One
// thread of a block that arrives at the word itself; it hands the returned word to
// counter_settle once its work is done (nobody waits for it before) and arrives behind
// that.
__device__ __forceinline__ unsigned long long counter_prepare(
    unsigned long long* word, unsigned long long call) {
  return __hip_atomic_exchange(word, call << 16, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}

// Puts back the arrivals that came before counter_prepare.  Until then the word counts
// too few, so no arrival takes itself for the last one, and this block's own arrival is
// still to come.
__device__ __forceinline__ void counter_settle(unsigned long long* word,
                                               unsigned long long call,
                                               unsigned long long prepared) {
  if ((prepared >> 16) == call)
    (void)__hip_atomic_fetch_add(word, prepared & 0xffffu, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
}

// true for the last of `expected` arrivals; one thread per arrival.  The
// common case is one fetch-add on a word that counter_prepare stamped long
// ago.  An arrival that finds another stamp (its add then changed a word
// nobody relies on) installs the stamp itself or, if somebody else just did,
// adds again: every arrival ends with exactly one successful operation on a
// word that carries this call's stamp.
__device__ __forceinline__ bool arrive_is_last(unsigned long long* word,
                                               unsigned long long call,
                                               unsigned expected) {
  unsigned long long old = __hip_atomic_fetch_add(
      word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((old >> 16) == call) return (unsigned)((old + 1) & 0xffffu) == expected;
  old = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (;;) {
    if ((old >> 16) == call) {
      old = __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
      return (unsigned)((old + 1) & 0xffffu) == expected;
    }
    const unsigned long long seen = atomicCAS(word, old, (call << 16) | 1ull);
    if (seen == old) return expected == 1u;
    old = seen;
  }
}

// Ranks of the block's choices.  ch [3][128] int16 in LDS as written by
// gate_select_kernel; wcnt [3][2][E] int32 in LDS.  Wavefront w ranks choice
// w / 2 of tokens 64 (w % 2) ..; with `loss2` wavefronts 0 and 1 also count
// the third array.  A lane's rank is the number of lower lanes of its
// wavefront that name the same expert.  Writes pos (rank within the block)
// for competing choices, 0 otherwise, and the block's counts to
// bcnt_blk [3][E].
__device__ __forceinline__ void gate_rank_tile(
    const int16_t* ch, int32_t* wcnt, int E, bool loss2, int64_t tok0,
    int32_t* __restrict__ pos, int32_t* __restrict__ bcnt_blk) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = wave >> 1, half = wave & 1;
  // bits an expert id has
  const int nbits = 32 - __builtin_clz((unsigned)max(E - 1, 1));
  // The lanes of this wavefront that name the same expert as this lane, from
  // one ballot per bit of the id (instead of one per expert): a lane keeps the
  // lanes whose bit equals its own.  id < 0: not competing, matches nobody.
  auto same_choice = [&](int id) {
    unsigned long long match = __ballot(id >= 0);
    for (int b = 0; b < nbits; ++b) {
      const bool bit = ((id >> b) & 1) != 0;
      const unsigned long long mb = __ballot(bit);
      match &= bit ? mb : ~mb;
    }
    return id >= 0 ? match : 0ull;
  };
  const unsigned long long before =
      lane == 0 ? 0ull : (~0ull >> (64 - lane));      // the lanes below this one
  auto clear_counts = [&](int32_t* dst) {
    for (int e = lane; e < E; e += 64) dst[e] = 0;
  };
  const int mine = ch[c * 128 + half * 64 + lane];
  int32_t* my_cnt = wcnt + (c * 2 + half) * E;
  clear_counts(my_cnt);
  const unsigned long long match = same_choice(mine);
  int rank = (int)__popcll(match & before);
  // the first lane of every expert's choosers writes the expert's count (LDS
  // keeps a wavefront's writes in program order: after the clearing)
  if (mine >= 0 && rank == 0) my_cnt[mine] = (int)__popcll(match);
  if (loss2 && c == 0) {
    const int third = ch[2 * 128 + half * 64 + lane];
    int32_t* cnt3 = wcnt + (4 + half) * E;
    clear_counts(cnt3);
    const unsigned long long m3 = same_choice(third);
    if (third >= 0 && (m3 & before) == 0ull) cnt3[third] = (int)__popcll(m3);
  }
  __syncthreads();
  if (half == 1 && mine >= 0) rank += wcnt[(c * 2) * E + mine];
  st_dev(pos + (tok0 + half * 64 + lane) * 2 + c, mine >= 0 ? rank : 0);
  for (int i = tid; i < 3 * E; i += blockDim.x) {
    const int cc = i / E, e = i - cc * E;
    st_dev(bcnt_blk + i, (cc < 2 || loss2) ? wcnt[(cc * 2) * E + e] +
                                                 wcnt[(cc * 2 + 1) * E + e]
                                           : 0);
  }
}

// Ranks of the choices of a block of 64 tokens: gate_rank_tile with one wavefront per
// choice.  ch [3][64] and cnt [3][E] in LDS; `live` tokens exist; ranked(token, choice,
// rank among the block's choosers of that expert).
template <typename F>
__device__ __forceinline__ void gate_rank_choices(const int16_t* ch, int32_t* cnt, int E,
                                                  bool loss2, int live, F&& ranked) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < 3 * E; i += blockDim.x) cnt[i] = 0;
  __syncthreads();
  if (wave < 2 || (wave == 2 && loss2)) {
    const int nbits = 32 - __builtin_clz((unsigned)max(E - 1, 1));
    const int mine = lane < live ? ch[wave * 64 + lane] : -1;
    // the lanes that name the same expert
    unsigned long long match = __ballot(mine >= 0);
    for (int b = 0; b < nbits; ++b) {
      const bool bit = ((mine >> b) & 1) != 0;
      const unsigned long long with = __ballot(bit);
      match &= bit ? with : ~with;
    }
    const unsigned long long before = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const int rank = (int)__popcll(match & before);
    if (mine >= 0 && rank == 0) cnt[wave * E + mine] = (int)__popcll(match);
    if (wave < 2 && lane < live) ranked(lane, wave, mine >= 0 ? rank : 0);
  }
  __syncthreads();
}
__device__ __forceinline__ void gate_rank_block(
    const int16_t* ch, int32_t* cnt, int E, bool loss2, int live, int64_t tok0,
    int32_t* pos, int32_t* bcnt_blk) {
  gate_rank_choices(ch, cnt, E, loss2, live, [&](int token, int choice, int rank) {
    st_dev(pos + (tok0 + token) * 2 + choice, rank);
  });
  for (int i = threadIdx.x; i < 3 * E; i += blockDim.x) st_dev(bcnt_blk + i, cnt[i]);
}

// What the last block of group g does (all of its threads, 2 E at least; smem is the
// block's whole dynamic LDS, free by now).  Same results, bit for bit, as
// gate_capacity_kernel + gate_loss_kernel for slots in token order.  U: tokens per
// thread and trip; PB: blocks whose sums are fetched together; the group's blocks are
// 2^SHIFT tokens.  LONG: so are those of every further PB blocks.  (Without: one by
// one.  The loop over batches takes 44 registers in router_gate_kernel, whose groups
// seldom have more than 16 blocks of 128 tokens: 174 instead of 130 registers, two
// wavefronts per SIMD instead of three.)
template <int U, int PB, int SHIFT, bool LONG>
__device__ __forceinline__ void gate_group_tail(
    unsigned char* smem, const GateParams& p, const FusedTail& ft, int g,
    const int32_t* __restrict__ idx, int32_t* __restrict__ pos,
    float* __restrict__ gate, uint8_t* __restrict__ kept,
    const float* __restrict__ part1, const float* __restrict__ part2) {
  const int S = p.S, E = p.E, C = p.C, nblk = p.nblk;
  const int tid = threadIdx.x;
  const bool sw = p.router == ROUTER_SWITCH;
  const bool loss2 = p.use_second_place_loss != 0 || sw;
  // First slots per block and expert.  16 bits suffice: a prefix is at most
  // the number of tokens of the earlier blocks, below S <= GATE_MAX_GROUP
  // (every gating entry refuses larger groups).
  static_assert(GATE_MAX_GROUP <= 65535, "the block prefixes are 16 bits wide");
  uint16_t* pre1 = reinterpret_cast<uint16_t*>(smem);          // [nblk][E]
  uint16_t* pre2 = pre1 + (size_t)nblk * E;                    // [nblk][E]
  int32_t* tot = reinterpret_cast<int32_t*>(
      smem + (((size_t)nblk * E * 4 + 15) & ~(size_t)15));     // [3][E]
  float* prod = reinterpret_cast<float*>(tot + 3 * E);         // [2][E]
  float* misc = prod + 2 * E;                                  // [4]
  int* last_group = reinterpret_cast<int*>(misc + 4);          // [1] (+ 3 pad)
  const int32_t* bc = ft.bcnt + (int64_t)g * nblk * 3 * E;
  const int64_t base = (int64_t)g * S;
  // Everything here comes from other compute units' stores, i.e. from memory,
  // one round trip per dependent access: the loads of the three parts (token
  // records, partial sums of the loss, per-block counts) are issued together
  // before anything is used.
  int2 ex[U], rk[U];
  float2 gt[U];
  uint16_t kk[U];
  auto load_records = [&](int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * (int)blockDim.x;
      if (s < S) {
        const int64_t t = base + s;
        const unsigned long long e2 =
            ld_dev(reinterpret_cast<const unsigned long long*>(idx + t * 2));
        const unsigned long long r2 =
            ld_dev(reinterpret_cast<const unsigned long long*>(pos + t * 2));
        const unsigned long long g2 =
            ld_dev(reinterpret_cast<const unsigned long long*>(gate + t * 2));
        kk[u] = ld_dev(reinterpret_cast<const uint16_t*>(kept + t * 2));
        ex[u] = make_int2((int)(unsigned)e2, (int)(e2 >> 32));
        rk[u] = make_int2((int)(unsigned)r2, (int)(r2 >> 32));
        gt[u] = make_float2(__uint_as_float((unsigned)g2),
                            __uint_as_float((unsigned)(g2 >> 32)));
      }
    }
  };
  // Loads return in the order they were issued: the per-block counts, which
  // the prefixes below need first, go out before the (many more) record loads.
  auto load_counts = [&](int i, int b0, int (&cv)[PB]) {
    const int c = i / E, e = i - c * E;
#pragma unroll
    for (int b = 0; b < PB; ++b)
      cv[b] = (i < 3 * E && b0 + b < nblk && (c < 2 || loss2))
                  ? ld_dev(bc + ((int64_t)(b0 + b) * 3 + c) * E + e) : 0;
  };
  int cv0[PB];
  load_counts(tid, 0, cv0);
  // thread e < E sums column e of part1, threads E .. 2E-1 column e of part2
  // (second-place loss: E columns; switch: columns 0 and 1), in block order
  const int pcol = tid < E ? tid : tid - E;
  const bool sums1 = tid < E;
  const bool sums2 = !sums1 && tid < 2 * E && loss2 && (!sw || pcol < 2);
  const float* pcolumn = (sums1 ? part1 : part2) + (int64_t)g * nblk * E + pcol;
  float pv[PB];
  if (sums1 || sums2) {
#pragma unroll
    for (int b = 0; b < PB; ++b)
      pv[b] = b < nblk ? ld_dev(pcolumn + (int64_t)b * E) : 0.f;
  }
  load_records(tid);
  // first slot of every block per expert: exclusive prefix over the blocks
  for (int i = tid; i < 3 * E; i += blockDim.x) {
    const int c = i / E, e = i - c * E;
    if (c == 2 && !loss2) { tot[i] = 0; continue; }
    uint16_t* pre = c == 0 ? pre1 : pre2;
    int cv[PB];
    if (i == tid) {
#pragma unroll
      for (int b = 0; b < PB; ++b) cv[b] = cv0[b];
    } else {
      load_counts(i, 0, cv);
    }
    int run = 0;
#pragma unroll
    for (int b = 0; b < PB; ++b) {
      if (b < nblk) {
        if (c < 2) pre[b * E + e] = (uint16_t)run;
        run += cv[b];
      }
    }
    if constexpr (LONG) {
      for (int b0 = PB; b0 < nblk; b0 += PB) {
        load_counts(i, b0, cv);
#pragma unroll
        for (int b = 0; b < PB; ++b) {
          if (b0 + b < nblk) {
            if (c < 2) pre[(b0 + b) * E + e] = (uint16_t)run;
            run += cv[b];
          }
        }
      }
    } else {
      for (int b = PB; b < nblk; ++b) {
        const int v = ld_dev(bc + ((int64_t)b * 3 + c) * E + e);
        if (c < 2) pre[b * E + e] = (uint16_t)run;
        run += v;
      }
    }
    tot[i] = run;
  }
  float psum = 0.f;
  if (sums1 || sums2) {
#pragma unroll
    for (int b = 0; b < PB; ++b)
      if (b < nblk) psum += pv[b];
    if constexpr (LONG) {
      for (int b0 = PB; b0 < nblk; b0 += PB) {
#pragma unroll
        for (int b = 0; b < PB; ++b)
          pv[b] = b0 + b < nblk ? ld_dev(pcolumn + (int64_t)(b0 + b) * E) : 0.f;
#pragma unroll
        for (int b = 0; b < PB; ++b)
          if (b0 + b < nblk) psum += pv[b];
      }
    } else {
      for (int b = PB; b < nblk; ++b) psum += ld_dev(pcolumn + (int64_t)b * E);
    }
  }
  __syncthreads();
  // Per-expert outputs and the group's share of the balancing loss come first:
  // the group's arrival at the call's counter then travels while the records
  // are rewritten.
  if (sums2) {
    if (sw) misc[pcol] = psum;
    else prod[E + pcol] = psum;      // proxy of the second-place loss, for now
  }
  __syncthreads();
  if (tid < E) {
    const int t1 = tot[tid], t2 = tot[E + tid];
    const int k1 = min(t1, C);
    ft.fill[(int64_t)g * E + tid] = k1 + min(t2, C - k1);
    const float inv_s = (float)(1.0 / (double)S);
    const int dens = sw ? tot[2 * E + tid] : t1;
    prod[tid] = (psum * inv_s) * ((float)dens * inv_s);
    if (loss2 && !sw)
      prod[E + tid] = (prod[E + tid] * inv_s) * ((float)tot[2 * E + tid] * inv_s);
  }
  __syncthreads();
  if (tid == 0) {
    float s1 = 0.f, s2 = 0.f;
    for (int k = 0; k < E; ++k) s1 += prod[k];
    if (loss2 && !sw)
      for (int k = 0; k < E; ++k) s2 += prod[E + k];
    float* gs = ft.gsum + (int64_t)g * GSUM;
    st_dev(gs + 0, s1);
    st_dev(gs + 1, s2);
    st_dev(gs + 2, sw ? (E > 1 ? misc[1] : 0.f) : 0.f);
    st_dev(gs + 3, sw ? misc[0] : 0.f);
    st_dev(ft.gctr + g, 0ull);
    wait_stores();
    const bool last = arrive_is_last(ft.fctr, ft.call, (unsigned)p.G);
    if (last) st_dev(ft.fctr, 0ull);
    *last_group = last ? 1 : 0;
  }
  for (int s0 = tid; s0 < S; s0 += (int)blockDim.x * U) {
    if (s0 != tid) load_records(s0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * (int)blockDim.x;
      if (s >= S) continue;
      const int blk = s >> SHIFT;
      uint16_t kout = 0;
      if (kk[u] & 1) {
        const int slot = pre1[blk * E + ex[u].x] + rk[u].x;
        rk[u].x = slot;
        if (slot < C) kout |= 1; else gt[u].x = gt[u].x * 0.0f;
      } else {
        rk[u].x = 0;
        gt[u].x = gt[u].x * 0.0f;
      }
      if (kk[u] & 0x100) {
        const int slot = min(tot[ex[u].y], C) + pre2[blk * E + ex[u].y] + rk[u].y;
        rk[u].y = slot;
        if (slot < C) kout |= 0x100; else gt[u].y = gt[u].y * 0.0f;
      } else {
        rk[u].y = 0;
        gt[u].y = gt[u].y * 0.0f;
      }
      kk[u] = kout;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * (int)blockDim.x;
      if (s < S) {
        const int64_t t = base + s;
        *reinterpret_cast<int2*>(pos + t * 2) = rk[u];
        *reinterpret_cast<uint16_t*>(kept + t * 2) = kk[u];
        *reinterpret_cast<float2*>(gate + t * 2) = gt[u];
      }
    }
  }
  // The last group to finish turns the groups' terms into the loss: all
  // threads fetch them (one round trip instead of one per group), one thread
  // adds them in group order.
  __syncthreads();
  const bool finishes_call = *last_group != 0;
  __syncthreads();                 // (the staging below overwrites the flag)
  if (finishes_call) {
    float* stage = reinterpret_cast<float*>(smem);     // the prefixes are done with
    const int n = p.G * GSUM;
    if (n <= 8192) {
      for (int i = tid; i < n; i += (int)blockDim.x) stage[i] = ld_dev(ft.gsum + i);
      __syncthreads();
      if (tid == 0) gate_loss_value<false>(p, stage, ft.loss);
    } else if (tid == 0) {
      gate_loss_value<true>(p, ft.gsum, ft.loss);
    }
  }
}

// ---------------------------------------------------------------------------
// Router projection fused with gating step 1: the K loop of router_mfma_kernel,
// then the block's 128 x E logits go from the accumulators to LDS (never to
// HBM unless `logits` is given) and step 1 runs on them.  Needs the
// group size to be a multiple of 128 so that a block's tokens share a group.
// ---------------------------------------------------------------------------
template <int NT, typename IT>
__global__ __launch_bounds__(256) void router_gate_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ wp,
    const float* __restrict__ bias, float* __restrict__ logits,
    int64_t tokens_total, int M, const IT* __restrict__ importance,
    const float* __restrict__ second_uniform, GateParams p,
    int32_t* __restrict__ idx, int32_t* __restrict__ pos,
    float* __restrict__ gate, uint8_t* __restrict__ kept,
    float* __restrict__ part1, float* __restrict__ part2,
    int tokens_per_batch, FusedTail ft) {
  constexpr int TOK = 128, BK = 64, ROWB = 128;
  constexpr int X_BYTES = TOK * ROWB, W_BYTES = NT * 32 * ROWB;
  constexpr int STAGE = X_BYTES + W_BYTES;
  extern __shared__ __attribute__((aligned(16))) unsigned char rl_smem[];
  __shared__ int last_of_group;
  const int E = p.E;
  const int64_t tok0 = (int64_t)blockIdx.x * TOK;       // first token, flat
  unsigned long long gctr_was = 0, fctr_was = 0;
  if (ft.bcnt != nullptr && threadIdx.x == 0) {
    // the first block of a group stamps the group's counter for this call
    if (tok0 % p.S == 0) gctr_was = counter_prepare(ft.gctr + tok0 / p.S, ft.call);
    if (blockIdx.x == 0) fctr_was = counter_prepare(ft.fctr, ft.call);
  }
  const int b = (int)(tok0 / tokens_per_batch);         // router weight set
  const bf16_t* xb = x + tok0 * M;
  const bf16_t* wb = wp + (int64_t)b * E * M;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  int x_off[4], w_off[NT];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = (wave + 4 * j) * 8 + (lane >> 3);
    x_off[j] = row * M + (((lane & 7) ^ rl_swizzle(row)) * 8);
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int row = (wave + 4 * j) * 8 + (lane >> 3);
    w_off[j] = min(row, E - 1) * M + (((lane & 7) ^ rl_swizzle(row)) * 8);
  }
  // Block b walks the K tiles starting at tile b % nk and wraps around: the
  // blocks run in step, and with rows a power of two apart all of them asking
  // for the same 128-byte column of their rows at the same moment lands on
  // few memory channels (measured: 20 % slower).
  const int nk = M / BK;
  const int rot = (int)(blockIdx.x % (unsigned)nk);
  auto issue = [&](int kt, int slot) {
    unsigned char* sx = rl_smem + slot * STAGE;
    unsigned char* sw = sx + X_BYTES;
    int kq = kt + rot;
    if (kq >= nk) kq -= nk;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_global_load_lds(
          (rl_glb_void_t*)(xb + kq * BK + x_off[j]),
          (rl_lds_void_t*)(sx + (wave + 4 * j) * 1024), 16, 0, RL_STREAMING);
#pragma unroll
    for (int j = 0; j < NT; ++j)
      __builtin_amdgcn_global_load_lds(
          (rl_glb_void_t*)(wb + kq * BK + w_off[j]),
          (rl_lds_void_t*)(sw + (wave + 4 * j) * 1024), 16, 0, 0);
  };
  rl_f32x16_t acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
  const int fr = lane & 31, fc = lane >> 5;
  int x_frag[4], w_frag[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int col = ((kk * 2 + fc) ^ rl_swizzle(fr)) * 16;
    x_frag[kk] = (wave * 32 + fr) * ROWB + col;
    w_frag[kk] = fr * ROWB + col;
  }
  // Three slots, two K tiles in flight: the loop is bound by the latency of
  // one round trip to HBM per K tile, so what it moves per second is the bytes
  // it keeps in flight.  vmcnt retires in issue order: leaving the newest
  // tile's 4 + NT loads outstanding means tile kt has landed.  Passing the
  // barrier of step kt also means every wavefront has finished reading slot
  // (kt - 1) % 3, which the loads of tile kt + 2 then overwrite.
  issue(0, 0);
  if (nk > 1) issue(1, 1);
  int slot = 0;
  for (int kt = 0; kt < nk; ++kt) {
    if (kt + 1 < nk)
      __builtin_amdgcn_s_waitcnt(0x0070 | (4 + NT));  // vmcnt(4+NT) lgkmcnt(0)
    else
      __builtin_amdgcn_s_waitcnt(0x0070);             // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + 2 < nk) issue(kt + 2, slot == 0 ? 2 : slot - 1);
    const unsigned char* sx = rl_smem + slot * STAGE;
    slot = slot == 2 ? 0 : slot + 1;
    const unsigned char* sw = sx + X_BYTES;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const rl_bf16x8_t xf = *reinterpret_cast<const rl_bf16x8_t*>(sx + x_frag[kk]);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const rl_bf16x8_t wf =
            *reinterpret_cast<const rl_bf16x8_t*>(sw + w_frag[kk] + j * 32 * ROWB);
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, xf, acc[j], 0, 0, 0);
      }
    }
  }
  __syncthreads();  // every wavefront is done with the ring: reuse it

  // this lane's logits (+ bias), written out if the caller wants them
  float* tile = reinterpret_cast<float*>(rl_smem);
  const int ld = E + 4;
  float* isone = tile + TOK * ld;
  float xl[NT][16];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e0 = j * 32 + 8 * q + 4 * (lane >> 5);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[j][4 * q + r];
        if (e0 < E) {
          if (bias != nullptr) v += bias[e0 + r];
        } else {
          v = -INFINITY;     // not an expert: exp() = 0, never the maximum
        }
        xl[j][4 * q + r] = v;
      }
    }
  }
  if (logits != nullptr)
    store_logits_rows<NT>(xl, tile, E, logits + tok0 * E, TOK);
  const int g = (int)(tok0 / p.S);
  const int t0 = (int)(tok0 - (int64_t)g * p.S);
  int16_t* ch = reinterpret_cast<int16_t*>(isone + TOK);      // [3][TOK]
  int32_t* wcnt = reinterpret_cast<int32_t*>(ch + 3 * TOK);   // [3][2][E]
  float* colpart = reinterpret_cast<float*>(wcnt + 6 * E);    // [4][E]
  const int blk = t0 / TOK;
  // (one call for both uses: the selection is 64 exponentials per lane long,
  // and a second inlined copy is code the instruction cache has to fetch)
  gate_select_acc_tile<NT, IT>(
      xl, tile, isone, ld, g, blk, t0, importance, second_uniform, p, idx, pos,
      gate, kept, part1, part2, ft.bcnt == nullptr ? nullptr : ch, colpart);
  // without the tail's workspace, capacity positions and loss follow as
  // launches of their own
  if (ft.bcnt == nullptr) return;
  const bool loss2 = p.use_second_place_loss != 0 || p.router == ROUTER_SWITCH;
  gate_rank_tile(ch, wcnt, E, loss2, tok0, pos,
                 ft.bcnt + ((int64_t)g * p.nblk + blk) * 3 * E);
  // This block's records, counts and partial sums are out (write-through
  // stores, see st_dev): once every wavefront's stores have completed, one
  // thread arrives at the group's counter; the last block to arrive finishes
  // the group.
  if (threadIdx.x == 0) {
    if (tok0 % p.S == 0) counter_settle(ft.gctr + g, ft.call, gctr_was);
    if (blockIdx.x == 0) counter_settle(ft.fctr, ft.call, fctr_was);
  }
  wait_stores();
  __syncthreads();
  if (tid == 0)
    last_of_group =
        arrive_is_last(ft.gctr + g, ft.call, (unsigned)p.nblk) ? 1 : 0;
  __syncthreads();
  if (!last_of_group) return;
  gate_group_tail<8, 16, 7, false>(rl_smem, p, ft, g, idx, pos, gate, kept, part1, part2);
  (void)tokens_total;
}

// The balancing loss from the groups' terms; one thread.  COHERENT: the terms
// were written by other blocks of the same launch (see st_dev).
template <bool COHERENT>
__device__ __forceinline__ void gate_loss_value(const GateParams& p,
                                                const float* gsum_in,
                                                float* loss) {
  struct Terms {
    const float* q;
    __device__ float operator[](int i) const {
      return COHERENT ? ld_dev(q + i) : q[i];
    }
  } gsum = {gsum_in};
  float s1 = 0.f, s2 = 0.f;
  for (int g = 0; g < p.G; ++g) {
    s1 += gsum[g * GSUM];
    s2 += gsum[g * GSUM + 1];
  }
  const float inv_ge = (float)(1.0 / ((double)p.G * (double)p.E));
  const float ee = (float)((double)p.E * (double)p.E);
  float l;
  if (p.router == ROUTER_SWITCH) {
    if (p.has_importance) {
      // mean over [G,E,S] of proxy[g,e] * (imp[g,s] == 1) * density[g,e]
      // (moe.py:1229-1234): each group's term counts once per such token
      float sm = 0.f;
      for (int g = 0; g < p.G; ++g) sm += gsum[g * GSUM] * gsum[g * GSUM + 2];
      l = (sm * (float)(1.0 / ((double)p.G * (double)p.E * (double)p.S))) * ee;
    } else {
      l = (s1 * inv_ge) * ee;
    }
    if (p.num_microbatches > 1)
      l = l * (float)(1.0 / (double)p.num_microbatches);     // moe.py:1235-1238
    if (p.use_z_loss) {                                      // moe.py:1253-1266
      float z = 0.f, n = 0.f;
      for (int g = 0; g < p.G; ++g) {
        z += gsum[g * GSUM + 3];
        n += gsum[g * GSUM + 2];
      }
      const float mb = (float)(p.num_microbatches > 0 ? p.num_microbatches : 1);
      l = l + p.z_loss_coef * (z / (n * mb));
    }
    loss[0] = l;
    return;
  }
  l = (s1 * inv_ge) * ee;                                    // moe.py:1423-1424
  if (p.use_second_place_loss) l = l + ((s2 * inv_ge) * ee) * 0.5f;
  if (p.num_microbatches > 1)
    l = l * (float)(1.0 / (double)p.num_microbatches);       // moe.py:1439-1442
  loss[0] = l;
}

// ---------------------------------------------------------------------------
// Gating step 2: capacity positions for one group per block (moe.py:1472-1496).
// Thread (e = tid % EL, chunk = tid / EL) counts, over its chunk of the
// group's tokens, those whose choice is expert e; an exclusive prefix over the
// chunks gives the slot of each chunk's first chooser of e.  Then one thread
// per token adds the number of earlier choosers of its expert inside its own
// chunk: every lane runs the same short loop, where a walk per (expert, chunk)
// would have each wave step through every token of the chunk.  Second choices
// start after the kept first choices of the same expert.  The token's expert
// ids live in LDS as int16 (-1 = not competing).
// ---------------------------------------------------------------------------
constexpr int CAP_THREADS = 1024;

// How many of the eight int16 expert ids in v equal e (0 <= e < 1024; an id of
// -1, "not competing", never does).
__device__ __forceinline__ int cap_match8(const uint4& v, int e) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  const uint32_t ue = (uint32_t)e;
  int n = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    n += ((w[j] & 0xffffu) == ue ? 1 : 0) + ((w[j] >> 16) == ue ? 1 : 0);
  return n;
}

// Number of entries of ch[s_begin, s_end) equal to e; with `vec` the range
// starts 16-byte aligned and is read eight ids at a time, up to the next
// multiple of eight.
__device__ __forceinline__ int cap_count(const int16_t* ch, int s_begin,
                                         int s_end, int e, bool vec) {
  int c = 0, s = s_begin;
  if (vec) {
    for (; s + 8 <= s_end; s += 8)
      c += cap_match8(*reinterpret_cast<const uint4*>(ch + s), e);
    const int n = s_end - s;             // of the next eight only the first n
    if (n > 0) {
      const uint4 v = *reinterpret_cast<const uint4*>(ch + s);
      auto only = [&](uint32_t w, int at) {
        return n >= at + 2 ? w : n == at + 1 ? w | 0xffff0000u : 0xffffffffu;
      };
      c += cap_match8(make_uint4(only(v.x, 0), only(v.y, 2), only(v.z, 4),
                                 only(v.w, 6)), e);
    }
    return c;
  }
  for (; s < s_end; ++s) c += (ch[s] == e);
  return c;
}

__device__ __forceinline__ void gate_capacity_group(
    const GateParams& p, const int32_t* idx, int32_t* pos, float* gate,
    uint8_t* kept, int32_t* fill, const float* part1, const float* part2,
    float* gsum, int el, int ss, float* loss, int32_t* smem_i, int g) {
  const int S = p.S, E = p.E, C = p.C;
  int32_t* cnt = smem_i;                        // [nchunks][el] = CAP_THREADS
  int32_t* pre = cnt + CAP_THREADS;             // [nchunks][el]: first slots
  int32_t* tot = pre + CAP_THREADS;             // [3][el]: total1,total2,loss2
  float* prod = reinterpret_cast<float*>(tot + 3 * el);  // [2][el]
  int16_t* c1 = reinterpret_cast<int16_t*>(prod + 2 * el);  // [ss], ss >= S
  int16_t* c2 = c1 + ss;                                     // [ss]
  int16_t* c2l = c2 + ss;                                    // [ss] (loss only)
  // first-choice gates of the group, for the by-gate slot order; float-aligned
  // because 3 * ss int16 may end on an odd 2-byte boundary
  float* gl = reinterpret_cast<float*>(c2l + ss + (ss & 1));  // [S]
  // by-gate order only: the first-choice gates listed per expert (token order
  // within an expert), every token's place in that list, the experts' first
  // places
  float* lg = gl + S;                                         // [S]
  int32_t* lpos = reinterpret_cast<int32_t*>(lg + S);         // [S]
  int32_t* ebase = lpos + S;                                  // [el]
  const int tid = threadIdx.x;
  const int64_t base = (int64_t)g * S;
  const bool sw = p.router == ROUTER_SWITCH;
  // a third count per expert: the second-place loss's mask_2 before the
  // policy (top-2), or every token's arg-max for density_1 (switch)
  const bool loss2 = p.use_second_place_loss != 0 || sw;
  for (int s = tid; s < S; s += CAP_THREADS) {
    int64_t t = base + s;
    int a = idx[t * 2], b = idx[t * 2 + 1];
    uint8_t k1 = kept[t * 2], k2 = kept[t * 2 + 1];
    c1[s] = (k1 & 1) ? (int16_t)a : (int16_t)-1;
    c2[s] = (k2 & 1) ? (int16_t)b : (int16_t)-1;
    if (sw) c2l[s] = (k1 & 2) ? (int16_t)a : (int16_t)-1;
    else if (loss2) c2l[s] = (k2 & 2) ? (int16_t)b : (int16_t)-1;
    if (p.rank_by_gate) gl[s] = gate[t * 2];
  }
  __syncthreads();
  const int e = tid % el;
  const int chunk = tid / el;
  const int nchunks = CAP_THREADS / el;
  // 16-byte reads of the id arrays: c1 starts 8192 + 20 * el bytes into LDS,
  // c2 and c2l ss and 2 ss ids later, a chunk clen ids after the previous one
  const bool vec = (el % 4 == 0) && (ss % 8 == 0);
  int clen = (S + nchunks - 1) / nchunks;
  if (vec) clen = (clen + 7) / 8 * 8;
  const int s_begin = min(S, chunk * clen);
  const int s_end = min(S, s_begin + clen);
  // The prefix over the chunks in two levels of about sqrt(nchunks) each
  // (nchunks and q are powers of two): one walk over all of them by all 1024
  // threads was much of the kernel (2 groups of 1024 tokens, 8 experts: 15.6 ->
  // 10.1 us; 6 groups of 1500, 16 experts, ids now padded for wide reads: 18.3
  // -> 14.2 us).
  int q = 1;
  while (q * q < nchunks) q *= 2;
  const int super = chunk / q;

  int count1 = 0;  // kept first choices of expert e (valid after choice 0)
  for (int choice = 0; choice < 2; ++choice) {
    const int16_t* ch = choice == 0 ? c1 : c2;
    cnt[chunk * el + e] = cap_count(ch, s_begin, s_end, e, vec);
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll 4
    for (int k = super * q; k < (super + 1) * q; ++k) {
      const int v = cnt[k * el + e];
      total += v;
      if (k < chunk) before += v;
    }
    if (chunk == super * q) pre[super * el + e] = total;
    __syncthreads();
    total = 0;
#pragma unroll 4
    for (int k = 0; k < nchunks / q; ++k) {
      const int v = pre[k * el + e];
      total += v;
      if (k < super) before += v;
    }
    __syncthreads();
    pre[chunk * el + e] = before + (choice == 0 ? 0 : count1);
    if (chunk == 0 && e < E) tot[choice * el + e] = total;
    if (choice == 0) count1 = min(total, C);
    __syncthreads();
    const bool by_gate = p.rank_by_gate && choice == 0;
    if (by_gate) {
      if (tid == 0) {
        int run = 0;
        for (int k = 0; k < E; ++k) { ebase[k] = run; run += tot[k]; }
      }
      __syncthreads();
    }
    for (int s = tid; s < S; s += CAP_THREADS) {
      const int ex = ch[s];
      if (ex < 0) continue;
      const int ck = s / clen;
      const int slot = pre[ck * el + ex] + cap_count(ch, ck * clen, s, ex, vec);
      if (by_gate) {
        // not the slot yet: the token's place among its expert's choosers
        lpos[s] = ebase[ex] + slot;
        lg[ebase[ex] + slot] = gl[s];
        continue;
      }
      const int64_t t = base + s;
      const bool ok = slot < C;
      pos[t * 2 + choice] = slot;
      kept[t * 2 + choice] = ok ? 1 : 0;
      if (!ok) gate[t * 2 + choice] = gate[t * 2 + choice] * 0.0f;
    }
    __syncthreads();
  }
  if (p.rank_by_gate) {
    // switch_max: expert e keeps its C choosers with the largest gate; slot =
    // rank by (gate descending, token ascending), the order of tf.math.top_k
    for (int s = tid; s < S; s += CAP_THREADS) {
      const int ex = c1[s];
      if (ex < 0) continue;
      const float gs = gl[s];
      const int mine = lpos[s], first = ebase[ex], last = first + tot[ex];
      int rank = 0;
      for (int j = first; j < last; ++j) {
        const float g2 = lg[j];
        rank += (g2 > gs || (g2 == gs && j < mine)) ? 1 : 0;
      }
      const int64_t t = base + s;
      const bool ok = rank < C;
      pos[t * 2] = rank;
      kept[t * 2] = ok ? 1 : 0;
      if (!ok) gate[t * 2] = gs * 0.0f;
    }
  }
  // tokens that did not compete: mask_k_flat = 0 -> gate_k * 0, kept = 0
  for (int s = tid; s < S; s += CAP_THREADS) {
    int64_t t = base + s;
    if (c1[s] < 0) { kept[t * 2] = 0; gate[t * 2] = gate[t * 2] * 0.0f; }
    if (c2[s] < 0) {
      kept[t * 2 + 1] = 0;
      gate[t * 2 + 1] = gate[t * 2 + 1] * 0.0f;
    }
  }
  if (loss2) {
    cnt[chunk * el + e] = cap_count(c2l, s_begin, s_end, e, vec);
    __syncthreads();
    if (chunk == 0 && e < E) {
      int total = 0;
#pragma unroll 8
      for (int k = 0; k < nchunks; ++k) total += cnt[k * el + e];
      tot[2 * el + e] = total;
    }
    __syncthreads();
  }
  // per-expert outputs and the group's share of the balancing loss.  The
  // per-block partial sums of the select step are summed in block order; they
  // come through LDS (`cnt` is free now), nchunks blocks at a time, so that
  // the loads of one batch fly together instead of one after the other, and while
  // the batch before is added.  (Blocks of 64 tokens are four times as many as they
  // were: 4 groups of 16384 tokens, 64 experts, one choice per token, slots by token
  // 365 us with blocks of 256 tokens, 380 of 64, 358 of 64 with loads ahead.)
  float* stage = reinterpret_cast<float*>(cnt);          // [nchunks][el]
  auto sum_blocks = [&](const float* part) {
    float acc = 0.f;
    auto load = [&](int bb) {
      return bb < p.nblk && e < E ? part[((int64_t)g * p.nblk + bb) * E + e] : 0.f;
    };
    float v = load(chunk);
    for (int b0 = 0; b0 < p.nblk; b0 += nchunks) {
      __syncthreads();
      stage[chunk * el + e] = v;
      v = load(b0 + nchunks + chunk);          // while this batch is added
      __syncthreads();
      const int n = min(nchunks, p.nblk - b0);
      if (tid < E) {
#pragma unroll 8
        for (int k = 0; k < n; ++k) acc += stage[k * el + tid];
      }
    }
    return acc;                                          // valid for tid < E
  };
  const float proxy = sum_blocks(part1);
  float proxy2 = 0.f, zsum = 0.f, n_one_sum = 0.f;
  if (loss2 && !sw) proxy2 = sum_blocks(part2);
  if (sw) {
    // columns 0 and 1 of part2: sum of logsumexp^2 and the number of tokens of
    // importance 1; thread e sums column e
    const float colsum = sum_blocks(part2);
    __syncthreads();
    if (tid < 2) stage[tid] = colsum;
    __syncthreads();
    zsum = stage[0];
    n_one_sum = E > 1 ? stage[1] : 0.f;
    __syncthreads();
  }
  if (tid < E) {
    const int t1 = tot[tid], t2 = tot[el + tid];
    const int k1 = min(t1, C);
    fill[(int64_t)g * E + tid] = k1 + min(t2, C - k1);
    const float inv_s = (float)(1.0 / (double)S);
    // density_1: competing first choices (top-2, moe.py:1420-1423) or every
    // token's arg-max (switch, moe.py:1224-1225)
    const int dens = sw ? tot[2 * el + tid] : t1;
    prod[tid] = (proxy * inv_s) * ((float)dens * inv_s);
    if (loss2 && !sw)
      prod[el + tid] = (proxy2 * inv_s) * ((float)tot[2 * el + tid] * inv_s);
  }
  __syncthreads();
  if (tid == 0) {
    float s1 = 0.f, s2 = 0.f;
#pragma unroll 8
    for (int k = 0; k < E; ++k) s1 += prod[k];
    if (loss2 && !sw)
#pragma unroll 8
      for (int k = 0; k < E; ++k) s2 += prod[el + k];
    gsum[g * GSUM] = s1;
    gsum[g * GSUM + 1] = s2;
    gsum[g * GSUM + 2] = sw ? n_one_sum : 0.f;
    gsum[g * GSUM + 3] = sw ? zsum : 0.f;
    // a single group's block needs no launch after it for the loss
    if (p.G == 1) gate_loss_value<false>(p, gsum, loss);
  }
}

__global__ __launch_bounds__(CAP_THREADS) void gate_capacity_kernel(
    GateParams p, const int32_t* __restrict__ idx, int32_t* __restrict__ pos,
    float* __restrict__ gate, uint8_t* __restrict__ kept,
    int32_t* __restrict__ fill, const float* __restrict__ part1,
    const float* __restrict__ part2, float* __restrict__ gsum, int el, int ss,
    float* __restrict__ loss) {
  extern __shared__ __attribute__((aligned(16))) int32_t smem_i[];
  gate_capacity_group(p, idx, pos, gate, kept, fill, part1, part2, gsum, el, ss,
                      loss, smem_i, blockIdx.x);
}

// Both steps for a group that is one block of gate_select_kernel, slots by gate: what
// step 1 wrote is read back by the same block.  (No pointer is __restrict__ here.)  Each
// step alone is bound by being a launch.
template <typename IT, int LANES>
__global__ __launch_bounds__(SELECT_THREADS) void gate_small_groups_kernel(
    const float* logits, const IT* importance, const float* second_uniform,
    GateParams p, int32_t* idx, int32_t* pos, float* gate, uint8_t* kept,
    int32_t* fill, float* part1, float* part2, float* gsum, int el, int ss,
    float* loss) {
  static_assert(SELECT_THREADS == CAP_THREADS, "one block does both steps");
  extern __shared__ __attribute__((aligned(16))) float smem[];
  gate_select_block<IT, LANES>(logits, importance, second_uniform, p, idx, pos,
                               gate, kept, part1, part2, smem);
  __syncthreads();
  gate_capacity_group(p, idx, pos, gate, kept, fill, part1, part2, gsum, el, ss,
                      loss, reinterpret_cast<int32_t*>(smem), blockIdx.y);
}

// Everything for one group of at most 64 tokens, slots in token order, in one block: the
// records, ranks and sums stay in LDS until they are final.  With `map` also what the
// first expert product asks for: the token of every slot, -1 for empty ones (a kept
// choice whose bf16 gate is 0 owns none, as in slot_map_rows_kernel), and a row of m
// zeros.  Same results, bit for bit, as gate_select_kernel + gate_capacity_kernel.
// Bound by being a launch and a chain of block barriers.  Both steps in one block, the
// second on what the first left in memory / here: 32 tokens, 32 experts 10.0 / 6.4 us,
// 64 of 64 11.8 / 8.3, 17 of 128 13.1 / 8.9; the slot map was another launch, 3.4 to 4.9.
template <typename IT>
__global__ __launch_bounds__(SELECT_THREADS) void gate_one_group_kernel(
    const float* __restrict__ logits, const IT* __restrict__ importance,
    const float* __restrict__ second_uniform, GateParams p, int32_t* __restrict__ idx,
    int32_t* __restrict__ pos, float* __restrict__ gate, uint8_t* __restrict__ kept,
    int32_t* __restrict__ fill, float* __restrict__ loss, int32_t* __restrict__ map,
    bf16_t* __restrict__ zero_row, int m) {
  constexpr int LANES = 16, TOKENS = SELECT_THREADS / LANES;
  static_assert(TOKENS == 64, "gate_rank_choices");
  extern __shared__ __attribute__((aligned(16))) float smem[];
  __shared__ int32_t ids[TOKENS * 2], rank[TOKENS * 2];
  __shared__ float gates[TOKENS * 2], terms[GSUM];
  __shared__ int16_t ch[3 * TOKENS];
  const int E = p.E, S = p.S, C = p.C, tid = threadIdx.x;
  const bool sw = p.router == ROUTER_SWITCH;
  const bool loss2 = p.use_second_place_loss != 0 || sw;
  float* part1 = smem + TOKENS * select_row_floats(E) + TOKENS + SELECT_THREADS;  // [E]
  float* part2 = part1 + E;                                        // [max(E, 2)]
  int32_t* cnt = reinterpret_cast<int32_t*>(part2 + max(E, 2));    // [3][E]
  float* prod = reinterpret_cast<float*>(cnt + 3 * E);             // [2][E]
  if (map != nullptr)
    for (int i = tid; i < m; i += SELECT_THREADS) zero_row[i] = 0;
  gate_select_block<IT, LANES, RECORD_LDS>(logits, importance, second_uniform, p, ids,
                                           nullptr, gates, nullptr, part1, part2, smem,
                                           ch);
  __syncthreads();
  gate_rank_choices(ch, cnt, E, loss2, S, [&](int token, int choice, int r) {
    rank[token * 2 + choice] = r;
  });
  if (tid < S * 2) {
    const int t = tid >> 1, choice = tid & 1;
    const int e = ids[tid];
    const bool competes = ch[choice * TOKENS + t] >= 0;
    int slot = rank[tid];
    if (choice == 1 && competes) slot += min(cnt[e], C);
    const bool ok = competes && slot < C;
    const float v = ok ? gates[tid] : gates[tid] * 0.0f;
    idx[tid] = e;
    pos[tid] = slot;
    gate[tid] = v;
    kept[tid] = ok ? 1 : 0;
    if (map != nullptr && ok)
      map[(int64_t)e * C + slot] = round_to<bf16_t>(v) == 0.0f ? -1 : t;
  }
  if (tid < E) {
    const int t1 = cnt[tid], t2 = cnt[E + tid];
    const int k1 = min(t1, C), used = k1 + min(t2, C - k1);
    fill[tid] = used;
    const float inv_s = (float)(1.0 / (double)S);
    // density_1: competing first choices (top-2) or every token's arg-max (switch)
    const int dens = sw ? cnt[2 * E + tid] : t1;
    prod[tid] = (part1[tid] * inv_s) * ((float)dens * inv_s);
    if (loss2 && !sw)
      prod[E + tid] = (part2[tid] * inv_s) * ((float)cnt[2 * E + tid] * inv_s);
    if (map != nullptr)
      for (int slot = used; slot < C; ++slot) map[(int64_t)tid * C + slot] = -1;
  }
  __syncthreads();
  if (tid == 0) {
    float s1 = 0.f, s2 = 0.f;
#pragma unroll 8
    for (int k = 0; k < E; ++k) s1 += prod[k];
    if (loss2 && !sw)
#pragma unroll 8
      for (int k = 0; k < E; ++k) s2 += prod[E + k];
    terms[0] = s1;
    terms[1] = s2;
    terms[2] = sw && E > 1 ? part2[1] : 0.f;
    terms[3] = sw ? part2[0] : 0.f;
    gate_loss_value<false>(p, terms, loss);
  }
}

// Both steps and the loss from logits in memory, groups of any number of blocks of 64
// tokens: every block ranks its own tokens, and the last one of a group finishes it as
// in router_gate_kernel.  Apart, the three launches are a chain of round trips, and
// step 2 counts the tokens of a whole group in one block.  Kernel times apart / in one,
// whatever the workspace held: 2 x 1024 tokens, 8 experts 6.5 + 11.3 + 2.5 / 13.7 us, 6 x
// 1500, 16 experts 7.1 + 14 + 3.3 / 17.6.  (With counters that the arrivals themselves had
// to put into this call's state, two more round trips: 16.5 and 24.5.)
template <typename IT>
__global__ __launch_bounds__(SELECT_THREADS) void gate_logits_kernel(
    const float* __restrict__ logits, const IT* __restrict__ importance,
    const float* __restrict__ second_uniform, GateParams p, int32_t* idx,
    int32_t* pos, float* gate, uint8_t* kept, float* part1, float* part2,
    FusedTail ft) {
  constexpr int LANES = 16, TOKENS = SELECT_THREADS / LANES;
  static_assert(TOKENS == 64, "gate_rank_block");
  extern __shared__ __attribute__((aligned(16))) float smem[];
  __shared__ int last_of_group;
  const int g = blockIdx.y, blk = blockIdx.x, tid = threadIdx.x;
  // the first block of a group stamps the group's counter for this call
  unsigned long long gctr_was = 0, fctr_was = 0;
  if (tid == 0) {
    if (blk == 0) gctr_was = counter_prepare(ft.gctr + g, ft.call);
    if (blk == 0 && g == 0) fctr_was = counter_prepare(ft.fctr, ft.call);
  }
  float* cols = smem + TOKENS * select_row_floats(p.E) + TOKENS;
  int32_t* cnt = reinterpret_cast<int32_t*>(cols + SELECT_THREADS);   // [3][E]
  int16_t* ch = reinterpret_cast<int16_t*>(cnt + 3 * p.E);            // [3][TOKENS]
  gate_select_block<IT, LANES, RECORD_TAIL>(logits, importance, second_uniform, p, idx,
                                            pos, gate, kept, part1, part2, smem, ch);
  const bool loss2 = p.use_second_place_loss != 0 || p.router == ROUTER_SWITCH;
  const int64_t tok0 = (int64_t)g * p.S + blk * TOKENS;
  gate_rank_block(ch, cnt, p.E, loss2, min(TOKENS, p.S - blk * TOKENS), tok0, pos,
                  ft.bcnt + ((int64_t)g * p.nblk + blk) * 3 * p.E);
  if (tid == 0) {
    if (blk == 0) counter_settle(ft.gctr + g, ft.call, gctr_was);
    if (blk == 0 && g == 0) counter_settle(ft.fctr, ft.call, fctr_was);
  }
  wait_stores();
  __syncthreads();
  if (tid == 0)
    last_of_group =
        arrive_is_last(ft.gctr + g, ft.call, (unsigned)p.nblk) ? 1 : 0;
  __syncthreads();
  if (!last_of_group) return;
  gate_group_tail<2, 16, 6, true>(reinterpret_cast<unsigned char*>(smem), p, ft, g, idx,
                                  pos, gate, kept, part1, part2);
}

__global__ void gate_loss_kernel(GateParams p, const float* __restrict__ gsum,
                                 float* __restrict__ loss) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  gate_loss_value<false>(p, gsum, loss);
}

}  // namespace mesh_moe

using namespace mesh_moe;

template <int NT>
static int launch_router_mfma(const bf16_t* x, const bf16_t* wp,
                              const float* bias, float* logits, int batch,
                              int tokens, int M, int E, hipStream_t st) {
  const size_t smem = 3 * (128 * 128 + (size_t)NT * 32 * 128);
  auto k = router_mfma_kernel<NT>;
  MOE_ALLOW_LDS(k, smem);
  dim3 grid((unsigned)((tokens + 127) / 128), (unsigned)batch);
  k<<<grid, 256, smem, st>>>(x, wp, bias, logits, tokens, M, E);
  MOE_CHECK_LAUNCH("router_logits (mfma)");
  return 0;
}

// Whether a wavefront per 32 tokens and 32 experts beats a block per 128 tokens: while at
// most two wavefronts share a compute unit.  In us, block / wavefront: 64 tokens of 1024,
// 32 experts 7.6 / 6.0, 64 experts 9.9 / 6.0; 64 tokens of 4096, 64 experts 31.9 / 16.4;
// 2048 tokens of 2048, 128 experts 27.4 / 10.0; 32 tokens of 64, 128 experts 3.6 / 3.0; two
// per unit: 8192 tokens of 1024, 64 experts 11.4 / 10.9, of 4096 34.6 / 32.7; three and
// four: 3 x 8192 of 1088, 16 experts 12.8 / 14.3, 8192 of 2048, 128 experts 28.2 / 32.3.
static bool router_few_applies(int batch, int64_t tokens, int E) {
  return batch * ((tokens + 31) / 32) * ((E + 31) / 32) <=
         2 * (int64_t)compute_units();
}

extern "C" int mesh_moe_router_logits(const void* x, const void* w,
                                      const void* w_packed, const float* bias,
                                      float* logits, int batch, int64_t tokens,
                                      int M, int E, int dtype, void* stream) {
  MOE_REQUIRE(x && w && logits, MESH_MOE_E_ARG, "router_logits: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG, "router_logits: bad dtype %d",
              dtype);
  MOE_REQUIRE(batch >= 1 && tokens >= 0 && M >= 1 && E >= 1, MESH_MOE_E_ARG,
              "router_logits: bad sizes batch=%d tokens=%lld M=%d E=%d", batch,
              (long long)tokens, M, E);
  MOE_REQUIRE(E <= RL_MAX_EXPERTS, MESH_MOE_E_UNSUPPORTED,
              "router_logits: E=%d > %d", E, RL_MAX_EXPERTS);
  MOE_REQUIRE(batch <= 65535, MESH_MOE_E_UNSUPPORTED,
              "router_logits: batch=%d > 65535", batch);
  if (tokens == 0) return 0;
  if (dtype == MESH_MOE_BF16 && w_packed != nullptr && M % 64 == 0 &&
      E % 4 == 0 && tokens * (int64_t)M < (1LL << 31) &&
      (((uintptr_t)x | (uintptr_t)w_packed | (uintptr_t)logits) % 16 == 0)) {
    const bf16_t* xb = (const bf16_t*)x;
    const bf16_t* wp = (const bf16_t*)w_packed;
    hipStream_t s2 = (hipStream_t)stream;
    if (router_few_applies(batch, tokens, E)) {
      dim3 grid((unsigned)((tokens + 31) / 32), (unsigned)((E + 31) / 32),
                (unsigned)batch);
      router_few_kernel<<<grid, 64, 0, s2>>>(xb, wp, bias, logits, (int)tokens, M,
                                             E);
      MOE_CHECK_LAUNCH("router_logits (mfma, few tokens)");
      return 0;
    }
    if (E <= 32)
      return launch_router_mfma<1>(xb, wp, bias, logits, batch, (int)tokens, M, E, s2);
    if (E <= 64)
      return launch_router_mfma<2>(xb, wp, bias, logits, batch, (int)tokens, M, E, s2);
    return launch_router_mfma<4>(xb, wp, bias, logits, batch, (int)tokens, M, E, s2);
  }
  const int tiles = (E + 15) / 16, waves = tiles < 4 ? tiles : 4;
  const int64_t blocks = (tokens + 15) / 16;
  MOE_REQUIRE(blocks <= 0x7fffffffLL, MESH_MOE_E_UNSUPPORTED,
              "router_logits: too many tokens (%lld)", (long long)tokens);
  dim3 grid((unsigned)blocks, (unsigned)((tiles + waves - 1) / waves),
            (unsigned)batch);
  hipStream_t st = (hipStream_t)stream;
  const bool vec = M % 4 == 0 && (uintptr_t)x % (4 * dtype_size(dtype)) == 0;
  auto run = [&](auto kern, const auto* xp, const auto* wp) {
    kern<<<grid, 64 * waves, 0, st>>>(xp, wp, bias, logits, tokens, M, E);
  };
  if (dtype == MESH_MOE_F32)
    run(vec ? router_logits_kernel<float, true> : router_logits_kernel<float, false>,
        (const float*)x, (const float*)w);
  else
    run(vec ? router_logits_kernel<bf16_t, true>
            : router_logits_kernel<bf16_t, false>,
        (const bf16_t*)x, (const bf16_t*)w);
  MOE_CHECK_LAUNCH("router_logits");
  return 0;
}

// Gating steps 2 and 3 (capacity positions, balancing loss) for every group.
static int launch_loss(const GateParams& p, const float* gsum, float* loss,
                       hipStream_t st) {
  if (p.G == 1) return 0;                // a single group's block made it
  gate_loss_kernel<<<1, 64, 0, st>>>(p, gsum, loss);
  MOE_CHECK_LAUNCH("gate_loss");
  return 0;
}

// LDS of gate_capacity_group, its padded numbers of experts and of tokens.
static size_t capacity_lds(const GateParams& p, int& el, int& ss) {
  el = 2;
  while (el < p.E) el *= 2;
  // the id arrays padded to multiples of eight ids, for 16-byte reads, unless
  // a group as large as LDS takes leaves no room for it
  auto lds_bytes = [&](size_t ss) {
    return sizeof(int32_t) * (2 * CAP_THREADS + 3 * (size_t)el) +
           sizeof(float) * 2 * (size_t)el + sizeof(int16_t) * (3 * ss + 1) +
           (p.rank_by_gate ? sizeof(float) * (3 * (size_t)p.S + el) : 0);
  };
  const int padded = (p.S + 7) / 8 * 8;
  ss = lds_bytes(padded) <= 160 * 1024 ? padded : p.S;
  return lds_bytes(ss);
}

static int launch_capacity_and_loss(const GateParams& p, int32_t* idx,
                                    int32_t* pos, float* gate, uint8_t* kept,
                                    int32_t* fill, float* loss,
                                    const float* part1, const float* part2,
                                    float* gsum, hipStream_t st) {
  int el, ss;
  const size_t smem = capacity_lds(p, el, ss);
  MOE_ALLOW_LDS(gate_capacity_kernel, smem);
  gate_capacity_kernel<<<p.G, CAP_THREADS, smem, st>>>(
      p, idx, pos, gate, kept, fill, part1, part2, gsum, el, ss, loss);
  MOE_CHECK_LAUNCH("gate_capacity");
  return launch_loss(p, gsum, loss, st);
}

static int check_gating_args(int G, int S, int E, int C, int policy,
                             const float* second_uniform,
                             const void* importance, int importance_dtype,
                             size_t workspace_bytes) {
  MOE_REQUIRE(G >= 1 && S >= 1 && C >= 1, MESH_MOE_E_ARG,
              "top2_gating: bad sizes G=%d S=%d C=%d", G, S, C);
  MOE_REQUIRE(E >= 2 && E <= 512, MESH_MOE_E_UNSUPPORTED,
              "top2_gating: E=%d outside [2, 512]", E);
  MOE_REQUIRE(S <= GATE_MAX_GROUP, MESH_MOE_E_UNSUPPORTED,
              "top2_gating: group size S=%d > %d", S, GATE_MAX_GROUP);
  MOE_REQUIRE(G <= 65535, MESH_MOE_E_UNSUPPORTED, "top2_gating: G=%d > 65535",
              G);
  MOE_REQUIRE(policy >= MESH_MOE_SECOND_ALL && policy <= MESH_MOE_SECOND_RANDOM,
              MESH_MOE_E_ARG, "top2_gating: unknown policy %d", policy);
  MOE_REQUIRE(policy != MESH_MOE_SECOND_RANDOM || second_uniform,
              MESH_MOE_E_ARG,
              "top2_gating: policy RANDOM needs second_uniform samples");
  MOE_REQUIRE(!importance || valid_dtype(importance_dtype), MESH_MOE_E_ARG,
              "top2_gating: bad importance dtype %d", importance_dtype);
  MOE_REQUIRE(workspace_bytes >= mesh_moe_gating_workspace_bytes(G, S, E),
              MESH_MOE_E_ARG, "top2_gating: workspace too small (%zu < %zu)",
              workspace_bytes, mesh_moe_gating_workspace_bytes(G, S, E));
  return 0;
}

static GateParams make_gate_params(int G, int S, int E, int C, int policy,
                                   double threshold, int use_second_place_loss,
                                   int num_microbatches,
                                   int importance_from_slot_gate, int tt) {
  GateParams p;
  p.G = G; p.S = S; p.E = E; p.C = C;
  p.policy = policy;
  p.threshold = (float)threshold;
  p.inv_threshold = (float)(1.0 / (threshold > 1e-9 ? threshold : 1e-9));
  p.use_second_place_loss = use_second_place_loss ? 1 : 0;
  p.num_microbatches = num_microbatches;
  p.importance_from_slot_gate = importance_from_slot_gate ? 1 : 0;
  p.tt = tt;
  p.nblk = (S + tt - 1) / tt;
  p.router = ROUTER_TOP2;
  p.has_importance = 0;
  p.use_z_loss = 0;
  p.z_loss_coef = 0.f;
  p.rank_by_gate = 0;
  return p;
}

static GateParams make_switch_params(int G, int S, int E, int C,
                                     const void* importance, int slots_by_gate,
                                     int use_z_loss, double z_loss_coef,
                                     int num_microbatches, int tt) {
  GateParams p = make_gate_params(G, S, E, C, MESH_MOE_SECOND_NONE, 0.0, 0,
                                  num_microbatches, 0, tt);
  p.router = ROUTER_SWITCH;
  p.has_importance = importance != nullptr;
  p.use_z_loss = use_z_loss ? 1 : 0;
  p.z_loss_coef = (float)z_loss_coef;
  p.rank_by_gate = slots_by_gate ? 1 : 0;
  return p;
}

// LDS the last block of a group needs (gate_group_tail).
static size_t fused_tail_lds_bytes(int nblk, int E) {
  return (((size_t)nblk * E * 4 + 15) & ~(size_t)15) +
         sizeof(int32_t) * 3 * (size_t)E + sizeof(float) * (2 * (size_t)E + 8);
}

template <int NT, typename IT>
static int launch_router_gate(const bf16_t* x, const bf16_t* wp,
                              const float* bias, float* logits, int64_t tokens,
                              int M, const void* importance,
                              const float* second_uniform, const GateParams& p,
                              int32_t* idx, int32_t* pos, float* gate,
                              uint8_t* kept, float* part1, float* part2,
                              int tokens_per_batch, const FusedTail& ft,
                              hipStream_t st) {
  const size_t ring = 3 * (128 * 128 + (size_t)NT * 32 * 128);
  // logits tile, importance flags, choices, per-wavefront counts, column sums
  const size_t tile = sizeof(float) * (128 * (size_t)(p.E + 4) + 128) +
                      3 * 128 * sizeof(int16_t) +
                      6 * (size_t)p.E * sizeof(int32_t) +
                      4 * (size_t)p.E * sizeof(float);
  size_t smem = ring > tile ? ring : tile;
  if (ft.bcnt != nullptr) {
    const size_t tail = fused_tail_lds_bytes(p.nblk, p.E);
    smem = smem > tail ? smem : tail;
  }
  auto k = router_gate_kernel<NT, IT>;
  MOE_ALLOW_LDS(k, smem);
  k<<<(unsigned)(tokens / 128), 256, smem, st>>>(
      x, wp, bias, logits, tokens, M, (const IT*)importance, second_uniform, p,
      idx, pos, gate, kept, part1, part2, tokens_per_batch, ft);
  MOE_CHECK_LAUNCH("router_gate");
  return 0;
}

// Workspace: per-block partial sums of the loss (2 float arrays), the groups'
// terms, and for the single-launch kernel per-block counts (3 int32 arrays)
// and the arrival counters.
extern "C" size_t mesh_moe_gating_workspace_bytes(int G, int S, int E) {
  if (G < 1 || S < 1 || E < 1) return 0;
  const size_t nblk = (size_t)(S + 63) / 64;  // smallest token block of any path
  return sizeof(float) * (2 * (size_t)G * nblk * E + GSUM * (size_t)G) +
         sizeof(int32_t) * 3 * (size_t)G * nblk * E +
         sizeof(unsigned long long) * ((size_t)G + 1) + 3 * 256;
}

// Number of a single-launch gating call: the arrival counters in the
// workspace are read relative to it (see arrive_is_last).
static unsigned long long next_call_number() {
  static std::atomic<unsigned long long> counter{1};
  unsigned long long n = counter.fetch_add(1, std::memory_order_relaxed);
  return (n & ((1ull << 48) - 1)) | (1ull << 47);
}

// Whether the gating of one group can make the slot map of the first expert product.
namespace mesh_moe {
bool gating_makes_map(int G, int S) { return G == 1 && S <= 64; }
}  // namespace mesh_moe

// Gating from logits: step 1 (softmax / choices) then steps 2 and 3.
static int run_gating(const GateParams& p, const float* logits,
                      const void* importance, int importance_dtype,
                      const float* second_uniform, int32_t* idx, int32_t* pos,
                      float* gate, uint8_t* kept, int32_t* fill, float* loss,
                      void* workspace, hipStream_t st, const SlotMap& slots = {}) {
  const int G = p.G, E = p.E;
  uintptr_t wsp = ((uintptr_t)workspace + 255) & ~(uintptr_t)255;
  float* part1 = (float*)wsp;
  float* part2 = part1 + (size_t)G * p.nblk * E;
  float* gsum = part2 + (size_t)G * p.nblk * E;
  dim3 grid((unsigned)p.nblk, (unsigned)G);
  const size_t smem = sizeof(float) * ((size_t)p.tt * select_row_floats(E) +
                                       p.tt + SELECT_THREADS);
  auto run = [&](auto k, auto* imp) -> int {
    MOE_ALLOW_LDS(k, smem);
    k<<<grid, SELECT_THREADS, smem, st>>>(logits, imp, second_uniform, p, idx,
                                          pos, gate, kept, part1, part2);
    MOE_CHECK_LAUNCH("gate_select");
    return 0;
  };
  int el, ss;
  const size_t cap_smem = capacity_lds(p, el, ss);
  // A group of one block with nothing to wait for: one group (32 tokens, 32 experts
  // 6.4 us, with the tail of gate_logits_kernel 10.8; 64 of 64 8.3 and 13.1), or
  // slots by gate, which those two do not do, in up to 128 groups.  (Two to 128 groups:
  // kernel times of step 1, step 2 and the loss / in one launch 2 x 64 tokens, 16
  // experts 16.9 / 12.4 us, 32 x 40, 64 experts 20.6 / 16.8, 128 x 64, 128 experts 35.5 /
  // 24.6.)
  const bool one_group = gating_makes_map(G, p.S) && p.tt == 64 && !p.rank_by_gate;
  const bool one_block =
      one_group || (p.nblk == 1 && p.tt == 64 && p.rank_by_gate && G <= 128);
  MOE_REQUIRE(slots.map == nullptr || one_group, MESH_MOE_E_UNSUPPORTED,
              "gating: a slot map from more than one block of tokens");
  const size_t tail_smem = fused_tail_lds_bytes(p.nblk, E);
  const size_t select_smem = smem + sizeof(int32_t) * 3 * (size_t)E +
                             sizeof(int16_t) * 3 * 64;
  // One launch, finished by the last block of every group, while its blocks (one per
  // compute unit: 128 registers) are little more than one round of them, where groups
  // are single blocks, and where they are so long that one block per group for all of
  // step 2 is what takes the time.  Separate launches / one, us: 2 x 1024 tokens, 8
  // experts 15.5 / 12.2; 16 x 1000, 64 experts 22.5 / 16.3; 8 x 2048, 128 experts 52.5 /
  // 23.6; 48 x 333, 16 experts 20.8 / 17.7; 300 x 40 47 / 25; 16384 tokens 205 / 49; 6 x
  // 8192 192 / 55.  On the other side 24 x 1000, 8 experts 18.7 / 19.3; 32 x 1000 20.4 /
  // 33.6; 64 x 1000 30 / 46; 15 x 4096 40 / 52.  (In 64 registers, two blocks per
  // compute unit: 64 x 1000 38.5, 2 x 1024 13.8.)
  const int64_t all_blocks = (int64_t)G * p.nblk;
  const bool one_launch =
      p.tt == 64 && !p.rank_by_gate && !one_block && 2 * E <= SELECT_THREADS &&
      tail_smem <= 60 * 1024 &&
      G * GSUM <= 8192 &&      // (more groups' terms the last block reads one by one)
      (4 * all_blocks <= 5 * (int64_t)compute_units() || p.nblk == 1 || p.S >= 8192);
  auto run_lanes = [&](auto* imp) -> int {
    using IT = std::remove_const_t<std::remove_pointer_t<decltype(imp)>>;
    if (one_launch) {
      FusedTail ft;
      uintptr_t at = ((uintptr_t)(gsum + (size_t)G * GSUM) + 255) & ~(uintptr_t)255;
      ft.bcnt = (int32_t*)at;
      at = (at + sizeof(int32_t) * 3 * (size_t)G * p.nblk * E + 255) & ~(uintptr_t)255;
      ft.gctr = (unsigned long long*)at;
      ft.fctr = ft.gctr + G;
      ft.gsum = gsum;
      ft.fill = fill;
      ft.loss = loss;
      ft.call = next_call_number();
      auto k = gate_logits_kernel<IT>;
      // (the last block of all stages the groups' terms of the loss)
      const size_t terms = sizeof(float) * G * GSUM;
      const size_t both = std::max(std::max(select_smem, tail_smem), terms);
      MOE_ALLOW_LDS(k, both);
      k<<<grid, SELECT_THREADS, both, st>>>(logits, imp, second_uniform, p, idx, pos,
                                            gate, kept, part1, part2, ft);
      MOE_CHECK_LAUNCH("gate_logits");
      return 0;
    }
    if (one_group) {
      auto k = gate_one_group_kernel<IT>;
      // (the parts, counts and terms per expert behind what step 1 needs)
      const size_t lds = smem + sizeof(float) * (2 * (size_t)E + 3 * (size_t)E +
                                                 2 * (size_t)E);
      MOE_ALLOW_LDS(k, lds);
      k<<<1, SELECT_THREADS, lds, st>>>(logits, imp, second_uniform, p, idx, pos, gate,
                                        kept, fill, loss, slots.map, slots.zero_row,
                                        slots.zeros);
      MOE_CHECK_LAUNCH("gate_one_group");
      return 0;
    }
    if (one_block) {
      auto k = gate_small_groups_kernel<IT, SELECT_THREADS / 64>;
      const size_t both = smem > cap_smem ? smem : cap_smem;
      MOE_ALLOW_LDS(k, both);
      k<<<grid, SELECT_THREADS, both, st>>>(logits, imp, second_uniform, p, idx, pos,
                                         gate, kept, fill, part1, part2, gsum, el,
                                         ss, loss);
      MOE_CHECK_LAUNCH("gate_small_groups");
      return launch_loss(p, gsum, loss, st);
    }
    switch (p.tt) {
      case 64: return run(gate_select_kernel<IT, 16>, imp);
      case 128: return run(gate_select_kernel<IT, 8>, imp);
      default: return run(gate_select_kernel<IT, 4>, imp);
    }
  };
  const int rc = importance && importance_dtype == MESH_MOE_BF16
                     ? run_lanes((const bf16_t*)importance)
                     : run_lanes((const float*)importance);
  if (rc != 0 || one_block || one_launch) return rc;
  return launch_capacity_and_loss(p, idx, pos, gate, kept, fill, loss, part1,
                                  part2, gsum, st);
}

// Shape limits of the fused projection + gating kernel.
namespace mesh_moe {
bool fused_router_shapes(int M, int E, int S, int dtype) {
  return dtype == MESH_MOE_BF16 && M % 64 == 0 && E % 4 == 0 && E <= 128 &&
         S % 128 == 0;
}
}  // namespace mesh_moe

extern "C" int mesh_moe_fused_router_supported(int M, int E, int S, int dtype) {
  return fused_router_shapes(M, E, S, dtype) ? 1 : 0;
}

static int check_fused_router_args(const char* who, const void* x,
                                   const void* w_packed, int batch,
                                   int64_t tokens, int M, int dtype, int G,
                                   int S, int E) {
  MOE_REQUIRE(batch >= 1 && (int64_t)batch * tokens == (int64_t)G * S,
              MESH_MOE_E_ARG, "%s: batch*tokens=%lld != G*S=%lld", who,
              (long long)batch * tokens, (long long)G * S);
  // (the one-launch tail keeps per-block slot prefixes in 16 bits)
  MOE_REQUIRE(S <= GATE_MAX_GROUP, MESH_MOE_E_UNSUPPORTED,
              "%s: group size S=%d > %d", who, S, GATE_MAX_GROUP);
  MOE_REQUIRE(fused_router_shapes(M, E, S, dtype) && tokens % S == 0 &&
                  (int64_t)128 * M < (1LL << 31) &&
                  (((uintptr_t)x | (uintptr_t)w_packed) % 16 == 0),
              MESH_MOE_E_UNSUPPORTED,
              "%s: the fused kernel needs bf16, M %% 64 == 0, "
              "E %% 4 == 0, E <= 128, S %% 128 == 0 (M=%d E=%d S=%d dtype=%d); "
              "use router_logits + the logits-in gating call", who, M, E, S,
              dtype);
  return 0;
}

// Fused projection + gating step 1 (p.tt must be 128), then steps 2 and 3.
static int run_router_gating(const GateParams& p, const void* x,
                             const void* w_packed, const float* bias,
                             float* logits, int64_t tokens, int M,
                             const void* importance, int importance_dtype,
                             const float* second_uniform, int32_t* idx,
                             int32_t* pos, float* gate, uint8_t* kept,
                             int32_t* fill, float* loss, void* workspace,
                             hipStream_t st) {
  const int G = p.G, S = p.S, E = p.E;
  uintptr_t wsp = ((uintptr_t)workspace + 255) & ~(uintptr_t)255;
  float* part1 = (float*)wsp;
  float* part2 = part1 + (size_t)G * p.nblk * E;
  float* gsum = part2 + (size_t)G * p.nblk * E;
  const bf16_t* xb = (const bf16_t*)x;
  const bf16_t* wp = (const bf16_t*)w_packed;
  const int64_t total = (int64_t)G * S;
  const bool imp_bf16 = importance && importance_dtype == MESH_MOE_BF16;
  // Slots in token order: positions, fill and loss are finished inside the
  // same launch by the last block of each group.  Slots by gate (switch_max)
  // compare every pair of a group's tokens: the capacity kernel does that.
  FusedTail ft = {};
  const bool one_launch =
      !p.rank_by_gate && fused_tail_lds_bytes(p.nblk, E) <= 60 * 1024;
  if (one_launch) {
    auto up = [](uintptr_t q) { return (q + 255) & ~(uintptr_t)255; };
    ft.bcnt = (int32_t*)up((uintptr_t)(gsum + GSUM * (size_t)G));
    ft.gctr = (unsigned long long*)up(
        (uintptr_t)(ft.bcnt + 3 * (size_t)G * p.nblk * E));
    ft.fctr = ft.gctr + G;
    ft.gsum = gsum;
    ft.fill = fill;
    ft.loss = loss;
    ft.call = next_call_number();
  }
  int rc;
#define MOE_ROUTER_GATE(NT)                                                    \
  (imp_bf16 ? launch_router_gate<NT, bf16_t>(xb, wp, bias, logits, total, M,   \
                                             importance, second_uniform, p,    \
                                             idx, pos, gate, kept, part1,      \
                                             part2, (int)tokens, ft, st)       \
            : launch_router_gate<NT, float>(xb, wp, bias, logits, total, M,    \
                                            importance, second_uniform, p,     \
                                            idx, pos, gate, kept, part1,       \
                                            part2, (int)tokens, ft, st))
  if (E <= 32) rc = MOE_ROUTER_GATE(1);
  else if (E <= 64) rc = MOE_ROUTER_GATE(2);
  else rc = MOE_ROUTER_GATE(4);
#undef MOE_ROUTER_GATE
  if (rc != 0 || one_launch) return rc;
  return launch_capacity_and_loss(p, idx, pos, gate, kept, fill, loss, part1,
                                  part2, gsum, st);
}

// ---------------------------------------------------------------------------
// Scratch memory of mesh_moe_top2_gating_static_scratch: what the other gating
// calls take from the caller as `workspace`.  Every GPU holds its own copy of
// the array at its own address; in host code the array's name is only a
// handle for hipGetSymbolAddress, never a device address.
// ---------------------------------------------------------------------------
constexpr size_t STATIC_SCRATCH_BYTES = (size_t)MESH_MOE_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

constexpr int STATIC_SCRATCH_MAX_DEVICES = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[STATIC_SCRATCH_MAX_DEVICES] = {};

// Device address of `scratch` on the current device, looked up once per
// device; nullptr (error text set) if the runtime refuses.
static void* static_scratch_address() {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= STATIC_SCRATCH_MAX_DEVICES) {
    mesh_moe::set_error("static scratch: hipGetDevice gave device %d (%s)", dev,
                        hipGetErrorString(e));
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      mesh_moe::set_error("static scratch: hipGetSymbolAddress: %s",
                          hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

extern "C" int mesh_moe_top2_gating_static_scratch(
    const float* logits, const void* importance, int importance_dtype,
    int importance_from_slot_gate, const float* second_uniform, int G, int S,
    int E, int C, int policy, double threshold, int use_second_place_loss,
    int num_microbatches, int32_t* idx, int32_t* pos, float* gate,
    uint8_t* kept, int32_t* fill, float* loss, void* stream) {
  MOE_REQUIRE(G >= 1 && S >= 1 && E >= 1, MESH_MOE_E_ARG,
              "top2_gating_static_scratch: bad sizes G=%d S=%d E=%d", G, S, E);
  const size_t need = mesh_moe_gating_workspace_bytes(G, S, E);
  MOE_REQUIRE(need <= STATIC_SCRATCH_BYTES, MESH_MOE_E_UNSUPPORTED,
              "top2_gating_static_scratch: G=%d S=%d E=%d needs %zu bytes of "
              "scratch, the built-in buffer has %zu; use mesh_moe_top2_gating "
              "with a workspace", G, S, E, need, STATIC_SCRATCH_BYTES);
  void* ptr = static_scratch_address();
  if (ptr == nullptr) return MESH_MOE_E_HIP;
  return mesh_moe_top2_gating(logits, importance, importance_dtype,
                              importance_from_slot_gate, second_uniform, G, S,
                              E, C, policy, threshold, use_second_place_loss,
                              num_microbatches, idx, pos, gate, kept, fill,
                              loss, ptr, STATIC_SCRATCH_BYTES, stream);
}

namespace mesh_moe {
int top2_gating(const float* logits, const void* importance, int importance_dtype,
                int importance_from_slot_gate, const float* second_uniform, int G,
                int S, int E, int C, int policy, double threshold,
                int use_second_place_loss, int num_microbatches, int32_t* idx,
                int32_t* pos, float* gate, uint8_t* kept, int32_t* fill, float* loss,
                void* workspace, size_t workspace_bytes, void* stream,
                const SlotMap& slots) {
  MOE_REQUIRE(logits && idx && pos && gate && kept && fill && loss && workspace,
              MESH_MOE_E_ARG, "top2_gating: null pointer");
  if (int rc = check_gating_args(G, S, E, C, policy, second_uniform, importance,
                                 importance_dtype, workspace_bytes))
    return rc;
  GateParams p = make_gate_params(G, S, E, C, policy, threshold,
                                  use_second_place_loss, num_microbatches,
                                  importance_from_slot_gate,
                                  select_tokens(G, S, E));
  return run_gating(p, logits, importance, importance_dtype, second_uniform,
                    idx, pos, gate, kept, fill, loss, workspace,
                    (hipStream_t)stream, slots);
}
}  // namespace mesh_moe

extern "C" int mesh_moe_top2_gating(
    const float* logits, const void* importance, int importance_dtype,
    int importance_from_slot_gate, const float* second_uniform, int G, int S,
    int E, int C, int policy,
    double threshold, int use_second_place_loss, int num_microbatches,
    int32_t* idx, int32_t* pos, float* gate, uint8_t* kept, int32_t* fill,
    float* loss, void* workspace, size_t workspace_bytes, void* stream) {
  return top2_gating(logits, importance, importance_dtype, importance_from_slot_gate,
                     second_uniform, G, S, E, C, policy, threshold,
                     use_second_place_loss, num_microbatches, idx, pos, gate, kept,
                     fill, loss, workspace, workspace_bytes, stream, SlotMap());
}

extern "C" int mesh_moe_router_top2_gating(
    const void* x, const void* w_packed, const float* bias, float* logits,
    int batch, int64_t tokens, int M, int dtype, const void* importance,
    int importance_dtype, int importance_from_slot_gate,
    const float* second_uniform, int G, int S, int E, int C, int policy,
    double threshold, int use_second_place_loss, int num_microbatches,
    int32_t* idx, int32_t* pos, float* gate, uint8_t* kept, int32_t* fill,
    float* loss, void* workspace, size_t workspace_bytes, void* stream) {
  MOE_REQUIRE(x && w_packed && idx && pos && gate && kept && fill && loss &&
                  workspace, MESH_MOE_E_ARG, "router_top2_gating: null pointer");
  if (int rc = check_gating_args(G, S, E, C, policy, second_uniform, importance,
                                 importance_dtype, workspace_bytes))
    return rc;
  if (int rc = check_fused_router_args("router_top2_gating", x, w_packed, batch,
                                       tokens, M, dtype, G, S, E))
    return rc;
  GateParams p = make_gate_params(G, S, E, C, policy, threshold,
                                  use_second_place_loss, num_microbatches,
                                  importance_from_slot_gate, 128);
  return run_router_gating(p, x, w_packed, bias, logits, tokens, M, importance,
                           importance_dtype, second_uniform, idx, pos, gate,
                           kept, fill, loss, workspace, (hipStream_t)stream);
}

extern "C" int mesh_moe_switch_gating(
    const float* logits, const float* choice_logits, const void* importance,
    int importance_dtype, int G, int S, int E, int C, int slots_by_gate,
    int use_z_loss, double z_loss_coef,
    int num_microbatches, int32_t* idx, int32_t* pos, float* gate,
    uint8_t* kept, int32_t* fill, float* loss, void* workspace,
    size_t workspace_bytes, void* stream) {
  MOE_REQUIRE(logits && idx && pos && gate && kept && fill && loss && workspace,
              MESH_MOE_E_ARG, "switch_gating: null pointer");
  if (int rc = check_gating_args(G, S, E, C, MESH_MOE_SECOND_NONE, nullptr,
                                 importance, importance_dtype, workspace_bytes))
    return rc;
  GateParams p = make_switch_params(G, S, E, C, importance, slots_by_gate,
                                    use_z_loss, z_loss_coef, num_microbatches,
                                    select_tokens(G, S, E));
  return run_gating(p, logits, importance, importance_dtype, choice_logits,
                    idx, pos, gate, kept, fill, loss, workspace,
                    (hipStream_t)stream);
}

extern "C" int mesh_moe_router_switch_gating(
    const void* x, const void* w_packed, const float* bias, float* logits,
    int batch, int64_t tokens, int M, int dtype, const void* importance,
    int importance_dtype, int G, int S, int E, int C, int slots_by_gate,
    int use_z_loss, double z_loss_coef, int num_microbatches, int32_t* idx,
    int32_t* pos,
    float* gate, uint8_t* kept, int32_t* fill, float* loss, void* workspace,
    size_t workspace_bytes, void* stream) {
  MOE_REQUIRE(x && w_packed && idx && pos && gate && kept && fill && loss &&
                  workspace, MESH_MOE_E_ARG,
              "router_switch_gating: null pointer");
  if (int rc = check_gating_args(G, S, E, C, MESH_MOE_SECOND_NONE, nullptr,
                                 importance, importance_dtype, workspace_bytes))
    return rc;
  if (int rc = check_fused_router_args("router_switch_gating", x, w_packed,
                                       batch, tokens, M, dtype, G, S, E))
    return rc;
  GateParams p = make_switch_params(G, S, E, C, importance, slots_by_gate,
                                    use_z_loss, z_loss_coef, num_microbatches,
                                    128);
  return run_router_gating(p, x, w_packed, bias, logits, tokens, M, importance,
                           importance_dtype, nullptr, idx, pos, gate, kept,
                           fill, loss, workspace, (hipStream_t)stream);
}
