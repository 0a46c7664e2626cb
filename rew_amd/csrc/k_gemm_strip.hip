// bf16 GEMM for few rows or few tiles ("gemm_strip").
//
// The 256 x 256 kernel of k_gemm_lds.hip needs a few thousand rows: a decode
// step's 8 rows cost it the MFMAs of 256, and a product with fewer tiles
// than CUs leaves the chip idle however long its K is.  This kernel takes
// those products.  Output tile 32 R rows (R = 1 .. 5) x 128 columns (of two
// weight matrices in the SwiGLU mode), four waves side by side on 32 columns
// each, all R row blocks per wave, so the MFMAs follow the real row count;
// and the k range may be split over S workgroups whose fp32 partial tiles
// the last of them to finish adds up in split order (the result depends on S
// only, not on timing).
//
// What bounds it: up to about 64 rows the weight stream (every weight is
// read once), above that the MFMAs.  So many bytes have to be in flight per
// CU and the row padding has to be small.
//
// k-tiles of 64 move HBM -> LDS by buffer_load ... lds into a ring of NS
// stages, each its own __shared__ array (with run-time slots the compiler
// waits for every DMA before each fragment read):
//   * A: 32 R rows of 128 bytes, 16-byte chunk c of row r stored at
//     c ^ ((r >> 1) & 7) (the layout of k_gemm_lds.hip's pair stages);
//   * B: 64 k-rows of 256 bytes per matrix, chunk c of row k stored at
//     c ^ (4 (k & 3)), read untransposed with ds_read_b64_tr_b16.
// Past the last tile the requests go through a
// descriptor of zero records: they cost no memory traffic and keep the count
// of outstanding loads the same on every path.
//
// Measured (weights out of cache; K x N, before -> after): 14336 x 4096 at 8,
// 64, 300 and 1000 rows 443 -> 28, 449 -> 33, 451 -> 60, 460 -> 150 us;
// 4096 x 4096 at 8, 300, 1000 rows 120 -> 14, 131 -> 25, 131 -> 46 us; SwiGLU
// 4096 x 14336 at 8 rows 95 -> 52 us (4.5 TB/s of weights; a 1 GiB
// copy reaches 6.2 TB/s).
#include <cstdlib>
#include <cstring>

#include "kernels.h"
#include "vm_device.h"

namespace rew {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) bf16x8_t lds_bf16x8;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x4_t lds_u32x4;

constexpr int BK = 64;
constexpr int BN = 128;               // output columns per tile
constexpr int B_BYTES = BK * BN * 2;  // one matrix's k-tile

constexpr int waitcnt_imm(int vm, int lgkm) {
  return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | ((lgkm & 15) << 8);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  void* p = (void*)(uintptr_t)(((uint64_t)hi << 32) | lo);
  return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void buf_to_lds16(__amdgpu_buffer_rsrc_t r, uint32_t voff,
                                             uint32_t soff, lds_u8* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void block_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Partial tiles of split products and the arrivals per tile.  All launches
// of a device's context are ordered on its one stream and each leaves the
// counters at zero, so one array per device serves every launch (captured ones,
// which may run beside that stream, are not split).
constexpr int64_t kWsFloats = 12ll << 20;  // 48 MiB
constexpr int kMaxSplitTiles = 1024;
constexpr int kAgent = 16;  // cache policy sc1: agent-scope access
__device__ float g_strip_ws[kWsFloats];
__device__ int g_strip_count[kMaxSplitTiles];

struct StripArgs {
  int tiles_m, tiles_n;
  int splits;       // workgroups per tile along k
  int per;          // k-tiles per split
};

}  // namespace

template <int R, bool DUAL, int NS, int OCC>
__global__ void __launch_bounds__(256, OCC) gemm_strip_kernel(GemmSegs gs, StripArgs sa) {
  constexpr int NJ = DUAL ? 2 : 1;
  constexpr int A_BYTES = 32 * R * 128;
  constexpr int STAGE = A_BYTES + NJ * B_BYTES;
  constexpr int ND = R + 4 * NJ;  // DMA instructions per wave and k-tile
  static_assert((NS - 1) * ND <= 63, "vmcnt range");
  static_assert(NS >= 2 && NS <= 4, "ring stages");
#define REW_STRIP_STAGE(i) \
  __shared__ __attribute__((aligned(1024))) uint8_t L##i[NS > i ? STAGE : 16]
  REW_STRIP_STAGE(0);
  REW_STRIP_STAGE(1);
  REW_STRIP_STAGE(2);
  REW_STRIP_STAGE(3);
#undef REW_STRIP_STAGE
  // (The compiler ties an access to its array only through a few levels of
  // casts and additions, and a fragment read it cannot tie waits for every
  // DMA in flight: so LDS pointers throughout, and b_off below is kept whole.)
  auto ST = [&](int i) -> lds_u8* {
    return i == 0 ? (lds_u8*)L0 : i == 1 ? (lds_u8*)L1 : i == 2 ? (lds_u8*)L2 : (lds_u8*)L3;
  };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- tile: XCD-contiguous ranges; the row tiles of one column tile and
  // split are neighbours, so its weights reach an XCD's L2 once ------------
  const int total = sa.tiles_m * sa.tiles_n * sa.splits;
  int t;
  {
    const int x = blockIdx.x % 8, q = total / 8, rr = total % 8;
    t = x * q + (x < rr ? x : rr) + (int)blockIdx.x / 8;
  }
  const int tm = t % sa.tiles_m;
  int tn = (t / sa.tiles_m) % sa.tiles_n;
  const int split = t / (sa.tiles_m * sa.tiles_n);
  const int tile = tn * sa.tiles_m + tm;
  int seg = 0;
  while (seg + 1 < gs.n && tn >= gs.tn0[seg + 1]) ++seg;
  tn -= (int)gs.tn0[seg];
  const GemmArgs& g = gs.g[seg];
  const int64_t row0 = (int64_t)tm * 32 * R;
  const int m_rows = (int)min((int64_t)32 * R, g.M - row0);
  const int64_t n0 = (int64_t)tn * BN;
  const int K = (int)g.K;
  const int nk = (K + BK - 1) / BK;
  const int kt0 = split * sa.per;
  const int nt = min(sa.per, nk - kt0);  // >= 1 (the host's choice of splits)
  const bool tail = K % BK != 0;         // the product's last k-tile is partial

  // ---- per-lane DMA sources (byte offsets from the operands' bases) ---------
  // A block q of wave w: rows 8 (R w + q) + lane / 8, physical chunk lane % 8.
  // The *_t offsets serve the partial last k-tile: chunks (k-rows) past K
  // read the last one inside instead, and clear_tail zeroes them in LDS.
  uint32_t va[R], va_t[R], vb[4], vb_t[4];
  int a_kc[2], b_kr[4];
  const int kl = (nk - 1) * BK;  // first k of the last k-tile
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = 8 * (R * wave + q) + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    const int rr = r < m_rows ? r : m_rows - 1;
    va[q] = (uint32_t)(((row0 + rr) * g.a_sm + c * 8) * 2);
    va_t[q] = (uint32_t)(((row0 + rr) * g.a_sm + min(kl + c * 8, K - 8)) * 2);
  }
#pragma unroll
  for (int p = 0; p < 2; ++p)  // (r >> 1) & 7 = (4 (R w + q) + lane / 16) & 7
    a_kc[p] = ((lane & 7) ^ ((4 * p + (lane >> 4)) & 7)) * 8;
  const uint32_t b_kbytes = __builtin_amdgcn_readfirstlane((uint32_t)(g.b_sk * 2));
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    // B block 4 w + q: k-rows 4 (4 w + q) + lane / 16, physical chunk lane % 16
    const int kr = 4 * (4 * wave + q) + (lane >> 4);
    const int c = (lane & 15) ^ (4 * (kr & 3));
    int64_t col = n0 + c * 8;
    if (col > g.N - 8) col = g.N - 8;
    b_kr[q] = kr;
    vb[q] = (uint32_t)((kr * g.b_sk + col) * 2);
    vb_t[q] = (uint32_t)((min(kl + kr, K - 1) * g.b_sk + col) * 2);
  }
  // requests k-tile kt0 + i (i >= nt: nothing) into stage s
  auto issue = [&](lds_u8* s, int i) {
    const bool live = i < nt, last = tail && kt0 + i == nk - 1;
    const uint32_t bytes = live ? 0x7fffffffu : 0u;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(g.a, bytes);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(g.b, bytes);
    const uint32_t k0 = (uint32_t)(kt0 + i) * BK;
    const uint32_t sa_ = last || !live ? 0u : k0 * 2, sb_ = last || !live ? 0u : k0 * b_kbytes;
    lds_u8* pa = s + wave * R * 1024;
    lds_u8* pb = s + A_BYTES + wave * 4096;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const __amdgpu_buffer_rsrc_t rj = DUAL && j ? make_rsrc(g.b2, bytes) : rb;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        buf_to_lds16(rj, last ? vb_t[q] : vb[q], sb_, pb + (j * B_BYTES + q * 1024));
    }
#pragma unroll
    for (int q = 0; q < R; ++q) buf_to_lds16(ra, last ? va_t[q] : va[q], sa_, pa + q * 1024);
  };
  auto clear_tail = [&](lds_u8* s) {
    const u32x4_t z = {0, 0, 0, 0};
    lds_u8* pa = s + (wave * R * 1024 + lane * 16);
    lds_u8* pb = s + (A_BYTES + wave * 4096 + lane * 16);
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (kl + a_kc[(R * wave + q) & 1] >= K) *(lds_u32x4*)(pa + q * 1024) = z;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (kl + b_kr[q] >= K) {
        *(lds_u32x4*)(pb + q * 1024) = z;
        if constexpr (NJ > 1) *(lds_u32x4*)(pb + (B_BYTES + q * 1024)) = z;
      }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
  };

  // ---- fragment offsets -------------------------------------------------------
  const int a_row = lane & 31;
  int a_off[4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
    a_off[s] = a_row * 128 + (((2 * s + (lane >> 5)) ^ ((a_row >> 1) & 7)) * 16);
  int b_off;
  {
    const int g16 = lane >> 4, s16 = lane & 15;
    const int kr = 8 * (g16 >> 1) + (s16 >> 2);
    const int col = wave * 32 + 16 * (g16 & 1) + 4 * (s16 & 3);
    b_off = A_BYTES + kr * 256 + (((col >> 3) ^ (4 * (kr & 3))) * 16) + (col & 7) * 2;
    asm("" : "+v"(b_off));
  }

  f32x16_t acc[R][NJ];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  bf16x8_t fa[2][R], fb[2][NJ];
  auto read_frags = [&](lds_u8* s, int u, int slot) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int o = b_off + (j * B_BYTES + u * 4096);
      const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(s + o));
      const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(s + (o + 1024)));
      v4s both[2] = {lo, hi};
      __builtin_memcpy(&fb[slot][j], both, 16);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) fa[slot][i] = *(lds_bf16x8*)(s + (a_off[u] + i * 4096));
  };
  // B in the first operand: the block of C^T, so a lane holds row lane % 32
  // and runs of four consecutive columns (k_gemm_lds.hip)
  auto mfmas = [&](int slot) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[slot][j], fa[slot][i], acc[i][j],
                                                            0, 0, 0);
  };

  // ---- main loop ----------------------------------------------------------------
  // Step i (its first fragments already in slot 0): substeps 0 .. 2, each
  // behind the reads of the next; then tile i + 1 has landed and every wave
  // is done reading tile i, so the barrier frees its stage; the last
  // substep runs behind the reads of tile i + 1's first fragments.
  auto landed = [&](int j, int i) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 2) * ND, 0));
    if (tail && kt0 + i == nk - 1) clear_tail(ST(j));
    block_barrier();
  };
  auto step = [&](int j, int i) {
    lds_u8* s = ST(j);
    read_frags(s, 1, 1);
    mfmas(0);
    read_frags(s, 2, 0);
    mfmas(1);
    read_frags(s, 3, 1);
    mfmas(0);
    landed((j + 1) % NS, i + 1);
    read_frags(ST((j + 1) % NS), 0, 0);  // (past the last tile: never used)
    issue(s, i + NS);
    mfmas(1);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < NS - 1; ++i) issue(ST(i), i);
  landed(0, 0);
  read_frags(ST(0), 0, 0);
  issue(ST(NS - 1), NS - 1);
  // whole turns of the ring, then the rest: with an exit inside the turn the
  // compiler sees a path from there back into the loop and waits, at its
  // head, for the newest DMA
  int i = 0;
  for (; i + NS <= nt; i += NS) {
#pragma unroll
    for (int j = 0; j < NS; ++j) step(j, i + j);
  }
  if (i < nt) {
    step(0, i);
    if (NS > 2 && i + 1 < nt) {
      step(1, i + 1);
      if (NS > 3 && i + 2 < nt) step(2, i + 2);
    }
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));

  // ---- split products: partial tiles to memory, the last to arrive adds ------------
  const int lr = lane & 31;
  if (sa.splits > 1) {
    __attribute__((address_space(3))) int* s_last = (__attribute__((address_space(3))) int*)L0;
    constexpr uint32_t kTile = R * NJ * 4 * 256 * 16;  // bytes of a partial tile
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(g_strip_ws, (uint32_t)(kWsFloats * 4));
    const uint32_t ws = (uint32_t)(tile * sa.splits) * kTile;
    // rows past the matrix: an offset out of range (stores dropped, loads
    // zero, no traffic), so no branch splits a batch of accesses
    uint32_t wo[R];
#pragma unroll
    for (int i = 0; i < R; ++i)
      wo[i] = i * 32 + lr < m_rows ? (uint32_t)(i * NJ * 16384 + tid * 16) : 0x70000000u;
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x4_t v = {vm::as_u(acc[i][j][4 * q]), vm::as_u(acc[i][j][4 * q + 1]),
                             vm::as_u(acc[i][j][4 * q + 2]), vm::as_u(acc[i][j][4 * q + 3])};
          __builtin_amdgcn_raw_buffer_store_b128(v, rw, wo[i] + (uint32_t)((j * 4 + q) * 4096),
                                                 ws + split * kTile, kAgent);
        }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    __syncthreads();
    if (tid == 0) {
      // The partial values were stored past the L2 (agent scope) and every
      // wave waited for its stores before the barrier, and the last arrival
      // reads them past its own L2 again, so the count orders them without a
      // fence; a fence's cache write-back cost 0.6 to 6 us per product.
      const int n = __hip_atomic_fetch_add(&g_strip_count[tile], 1, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
      *s_last = n == sa.splits - 1;
      if (n == sa.splits - 1)
        __hip_atomic_store(&g_strip_count[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*s_last) return;
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    // U splits at a time (32 to 40 loads in flight per lane): each batch
    // costs a round trip past the L2
    constexpr int U = R * NJ >= 8 ? 1 : R * NJ >= 4 ? 2 : R * NJ == 2 ? 4 : 8;
#pragma unroll U
    for (int s = 0; s < sa.splits; ++s)
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(
                rw, wo[i] + (uint32_t)((j * 4 + q) * 4096), ws + s * kTile, kAgent);
#pragma unroll
            for (int x = 0; x < 4; ++x) acc[i][j][4 * q + x] += vm::as_f(v[x]);
          }
  }

  // ---- epilogue: four consecutive columns of one row per accumulator group -----------
  const int epi = DUAL ? (int)EPI_SWIGLU : g.epi;
  auto bf = [](uint16_t h) { return vm::as_f((uint32_t)h << 16); };
  uint16_t* C = (uint16_t*)g.c;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t n = n0 + wave * 32 + q * 8 + (lane >> 5) * 4;
    if (n >= g.N) continue;
    ushort4 bv = make_ushort4(0, 0, 0, 0), bv2 = bv;
    if (epi != EPI_NONE) bv = *(const ushort4*)((const uint16_t*)g.bias + n);
    if constexpr (DUAL) bv2 = *(const ushort4*)((const uint16_t*)g.bias2 + n);
    const float b1[4] = {bf(bv.x), bf(bv.y), bf(bv.z), bf(bv.w)};
    const float b2[4] = {bf(bv2.x), bf(bv2.y), bf(bv2.z), bf(bv2.w)};
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int row = i * 32 + lr;
      if (row >= m_rows) continue;
      const int64_t m = row0 + row;
      float y[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        y[x] = vm::round_bf16(acc[i][0][4 * q + x]);
        if (epi != EPI_NONE) y[x] = vm::round_bf16(y[x] + b1[x]);
      }
      uint16_t* dst = C + m * g.c_sm + n;
      if constexpr (DUAL) {
        // GatedFeedForward's gate, op by op in fp32 (gated_ffn.nim:46-67)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float u =
              vm::round_bf16(vm::round_bf16(acc[i][NJ - 1][4 * q + x]) + b2[x]);
          const float e = expf(-y[x]);
          const float den = 1.0f + e;
          const float sig = 1.0f / den;
          y[x] = y[x] * sig * u;
        }
      } else if (epi == EPI_BIAS_RES) {
        const ushort4 rv =
            *(const ushort4*)((const uint16_t*)g.res + m * g.res_sm + n);
        y[0] = bf(rv.x) + y[0];
        y[1] = bf(rv.y) + y[1];
        y[2] = bf(rv.z) + y[2];
        y[3] = bf(rv.w) + y[3];
      } else if (epi == EPI_BIAS_ROPE) {
        // applyRotate (rope.nim:56-108) on the two pairs
        const int64_t h = n / g.rope_D, d = n - h * g.rope_D;
        const int64_t b = m / g.rope_S, s = m - b * g.rope_S;
        const int64_t tb = b * g.rope_tb + s * g.rope_ts + h * g.rope_th + (d >> 1) * g.rope_ti;
#pragma unroll
        for (int x = 0; x < 4; x += 2) {
          const float co = g.rope_cos[tb + (x >> 1) * g.rope_ti];
          const float si = g.rope_sin[tb + (x >> 1) * g.rope_ti];
          const float x0 = y[x], x1 = y[x + 1];
          const float t1 = co * x0, t2 = si * x1, t3 = si * x0, t4 = co * x1;
          y[x] = t1 - t2;
          y[x + 1] = t3 + t4;
        }
        dst = C + b * g.out_b + s * g.out_s + h * g.out_h + d;
      }
      *(uint2*)dst = make_uint2(vm::bf16x2_bits(y[0], y[1]), vm::bf16x2_bits(y[2], y[3]));
    }
  }
}

// ---- host ------------------------------------------------------------------------------

namespace {

int64_t col_tiles(const GemmArgs& g) { return (g.N + BN - 1) / BN; }

// Row blocks per tile and splits of k, by an estimate of the time in
// microseconds (good enough to tell plans of one product apart; strip_time is
// the one to compare with another kernel).  Its terms are fits to measurements over 8 .. 2000 rows of
// K x N = 4096 x 4096, 14336 x 4096 and 4096 x 14336 (weights out of cache),
// which they meet within about 15 %:
//   * a k-tile of one workgroup per CU (more workgroups share the CU);
//   * the weights from HBM once (few workgroups keep too few bytes in flight:
//     8 rows x 14336 x 4096 took 52 / 35 / 28 us on 64 / 128 / 256 of them)
//     and, for each further row tile, from L2 at 13 TB/s;
//   * the sum of a split tile, several round trips past the L2 per row block;
//   * 4 us around them.
// K below 1024 is never split: there is little to gain, and the sum then
// runs in the order of the 256 x 256 kernel's.
StripPlan plan_for(const GemmArgs* segs, int n, int max_splits) {
  const int64_t M = segs[0].M, K = segs[0].K;
  const bool dual = segs[0].epi == EPI_SWIGLU;
  const int64_t nk = (K + BK - 1) / BK;
  StripPlan best;
  double best_us = 1e30;
  double weights = 0;
  for (int i = 0; i < n; ++i) {
    best.tiles_n += col_tiles(segs[i]);
    weights += (dual ? 4.0 : 2.0) * (double)K * (double)segs[i].N;
  }
  constexpr int kR[4] = {1, 2, 4, 5};
  constexpr double kTile[2][4] = {{0.28, 0.42, 0.65, 0.85}, {0.6, 0.8, 1.35, 1.5}};
  constexpr double kSum[2][4] = {{1, 3, 8, 12}, {0, 1, 12, 18}};
  for (int x = 0; x < 4; ++x) {
    const int64_t tm = (M + 32 * kR[x] - 1) / (32 * kR[x]), tiles = tm * best.tiles_n;
    const int64_t fit = kWsFloats / (tiles * 32 * kR[x] * BN * (dual ? 2 : 1));
    for (int64_t s = 1; s <= max_splits; ++s) {
      if (s > 1 && (K < 1024 || s > nk / 8 || s > fit || tiles > kMaxSplitTiles)) break;
      const int64_t per = (nk + s - 1) / s, wgs = tiles * s;
      const double fill = wgs > 256 ? (double)wgs / 256 : 1.0;
      const double loop = (double)per * kTile[dual][x] * fill;
      const double mem = weights / 8e6 + weights / (57e3 * (double)(wgs < 256 ? wgs : 256)) +
                         (double)(tm - 1) * weights / 13e6;
      const double us = 4 + (loop > mem ? loop : mem) + (s > 1 ? kSum[dual][x] : 0.0);
      if (us < best_us) {
        best_us = us;
        best.R = kR[x];
        best.per = (int)per;
        best.splits = (int)((nk + per - 1) / per);
        best.tiles_m = tm;
      }
    }
  }
  return best;
}

// Time of a plan, and of the 256 x 256 kernel for the same product, in
// microseconds: fits to both kernels' times over 8 .. 8000 rows, K 64 .. 14336
// and N 512 .. 128256, which they meet within 8 % (half of them) to 20 % (nine
// in ten).  A CU runs its workgroups' k-tiles one after another (two of them at
// once up to 64 rows) and pays a workgroup's start and end once per round; the
// 256 x 256 kernel likewise, a k-tile costing more with more CUs busy.
double strip_time(const StripPlan& p, int64_t K, double weights, bool dual) {
  constexpr double kTile[2][4] = {{0.230, 0.330, 0.510, 0.579}, {0.495, 0.579, 0.912, 1.094}};
  constexpr double kEnds[2][4] = {{4.1, 4.8, 6.8, 7.7}, {5.3, 7.3, 10.3, 11.3}};
  constexpr double kSum[2][4] = {{3.2, 4.0, 4.4, 6.1}, {4.2, 6.4, 7.9, 8.7}};
  const int x = p.R == 1 ? 0 : p.R == 2 ? 1 : p.R == 4 ? 2 : 3;
  const int64_t wgs = p.tiles_m * p.tiles_n * p.splits, slots = !dual && p.R <= 2 ? 512 : 256;
  const double loop = (double)((wgs + 255) / 256) * p.per * kTile[dual][x] +
                      (double)((wgs + slots - 1) / slots) * kEnds[dual][x];
  const double hbm = dual ? 6.5e6 : 5.5e6, wg = dual ? 58e3 : 102e3, l2 = dual ? 14e6 : 15.6e6;
  const double mem = weights / hbm + weights / (wg * (double)(wgs < slots ? wgs : slots)) +
                     (double)(p.tiles_m - 1) * weights / l2;
  return 3.8 + (loop > mem ? loop : mem) + (p.splits > 1 ? kSum[dual][x] : 0.0);
}
double tile256_time(int64_t tiles, int64_t K, double weights, bool dual) {
  const double busy = tiles <= 96 ? 0.0 : tiles >= 256 ? 1.0 : (double)(tiles - 96) / 160;
  const double step = dual ? 0.485 + 0.117 * busy : 0.48 + 0.04 * busy;  // 32 of K
  const double loop =
      (double)((tiles + 255) / 256) * ((dual ? 7.4 : 8.7) + (double)((K + 31) / 32) * step);
  return (dual ? 7.1 : 6.4) + (loop > weights / 4.8e6 ? loop : weights / 4.8e6);
}

template <int R, bool DUAL, int NS, int OCC>
void go(const GemmSegs& gs, const StripPlan& p, hipStream_t stream) {
  StripArgs sa{(int)p.tiles_m, (int)p.tiles_n, p.splits, p.per};
  const unsigned grid = (unsigned)(p.tiles_m * p.tiles_n * p.splits);
  hipLaunchKernelGGL((gemm_strip_kernel<R, DUAL, NS, OCC>), dim3(grid), dim3(256), 0, stream, gs,
                     sa);
}

}  // namespace

StripPlan gemm_strip_plan(const GemmArgs* segs, int n, int max_splits) {
  const StripPlan none;
  static const bool forced = std::getenv("REW_MI355X_GEMM_TILE") != nullptr;
  if (forced || n < 1 || n > kMaxSegs) return none;
  const GemmArgs& f = segs[0];
  if (f.batch != 1 || f.M <= 0) return none;
  const bool dual = f.epi == EPI_SWIGLU;
  constexpr int64_t kLim = (int64_t)1 << 31;
  int64_t tiles = 0;  // of the 256 x 256 kernel
  for (int i = 0; i < n; ++i) {
    const GemmArgs& g = segs[i];
    bool bkc;
    if (!gemm_lds_ok(g, &bkc) || bkc || (g.epi == EPI_SWIGLU) != dual) return none;
    if (g.epi == EPI_BIAS_RELU) return none;
    // 32-bit byte offsets from each operand's base
    if (((g.M - 1) * g.a_sm + g.K) * 2 >= kLim || ((g.K - 1) * g.b_sk + g.N) * 2 >= kLim)
      return none;
    tiles += (g.N + (dual ? 127 : 255)) / (dual ? 128 : 256);
  }
  tiles *= (f.M + 255) / 256;
  if (tiles >= 4096) return none;
  // Fewer than 96 of the 256 x 256 kernel's tiles otherwise go to the 128 x 128
  // kernel or, as SwiGLU, to the older 256 x 256 one, which no size measured had
  // faster (8 x 14336 x 4096: 443 us against 28 here; SwiGLU 1500 x 2048 x 1408:
  // 92 against 49).
  const StripPlan p = plan_for(segs, n, max_splits);
  if (tiles < 96 && n == 1) return p;
  // From there on the two estimates decide, where they differ by more than
  // their bias: the 256 x 256 kernel had every product of more than 256 rows
  // (us here / there: 1000 x 1024 x 8192 31 / 29, 600 x 4096 x 14336 121 / 83,
  // 3000 x 64 x 4096 26 / 17; SwiGLU 600 x 4096 x 14336 180 / 158, 300 x 4096 x
  // 14336 98 / 92), this one the few rows over many weights (16 x 4096 x 128256
  // 190 / 201, 8 x 1024 x 128256 52 / 66; SwiGLU 64 x 4096 x 14336 72 / 93).
  double weights = 0;
  for (int i = 0; i < n; ++i) weights += (dual ? 4.0 : 2.0) * (double)f.K * (double)segs[i].N;
  const double here = strip_time(p, f.K, weights, dual);
  const double there = tile256_time(tiles, f.K, weights, dual);
  return here < (dual && f.M > 64 ? 0.85 : 0.97) * there ? p : none;
}

bool being_captured(hipStream_t stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  REW_HIP(hipStreamIsCapturing(stream, &st));
  return st != hipStreamCaptureStatusNone;
}

void launch_gemm_strip(const GemmArgs* segs, int n, const StripPlan& p, hipStream_t stream) {
  GemmSegs gs;
  std::memset(&gs, 0, sizeof gs);
  gs.n = n;
  for (int i = 0; i < n; ++i) {
    gs.g[i] = segs[i];
    gs.tn0[i + 1] = gs.tn0[i] + col_tiles(segs[i]);
  }
  // NS stages fill the LDS: two workgroups per CU where 80 KiB hold enough
  if (segs[0].epi == EPI_SWIGLU) {
    if (p.R == 1) go<1, true, 4, 1>(gs, p, stream);
    else if (p.R == 2) go<2, true, 4, 1>(gs, p, stream);
    else if (p.R == 4) go<4, true, 3, 1>(gs, p, stream);
    else go<5, true, 3, 1>(gs, p, stream);
  } else {
    if (p.R == 1) go<1, false, 4, 2>(gs, p, stream);
    else if (p.R == 2) go<2, false, 3, 2>(gs, p, stream);
    else if (p.R == 4) go<4, false, 4, 1>(gs, p, stream);
    else go<5, false, 4, 1>(gs, p, stream);
  }
  REW_HIP(hipGetLastError());
}

}  // namespace rew
