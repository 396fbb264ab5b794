// qmlp_tiled.hip -- matrix-core GEMM kernels for many tokens (prefill chunks).
//
// Reference realisation being replaced: the prefill branch of Qwen36MLP -- the fused gate/up
// with SiLU on fp32 accumulators (docker/qwen-c2-graft/graft/mlp.py:440-456, rounded once,
// docs/real-text-2026-09-24.md:272-276) and the down projection with its prefill program config
// (mlp.py:539-611).
//
// Formulation: out^T[n, m] = sum_k W[n, k] x[m, k] on 32x32x16 products.  The weights are the
// matrix-core A operand: each of a block's 8 waves owns one 32-row unit (two packed 16-row tiles) of
// one matrix -- of both matrices in one gate/up variant -- and streams it through registers in the
// packed layout (bfp8 and bf4 dequantised exactly to fp16 in registers, bf16 used as is).  The tokens
// are the B operand: a block stages MG groups of 32 token rows, one 64-K step at a time, into a
// 3-slot LDS ring shared by all its waves.
//
// Pipeline per 64-K step s: compute step s from LDS slot s%3 and register stage s%3; issue the
// weight loads of step s+3 into that stage; write the B rows of step s+2 (requested one or three
// steps earlier, by the number of B register buffers) into slot (s+2)%3; one barrier.  The row
// exponents of a 256-K superblock (one 32-bit word per lane and row) are requested once per
// superblock, a superblock ahead.  Loads beyond the last step are clamped duplicates, so every
// weight and B load is unconditional.
//
// Epilogue (fp32 accumulators in registers): gate/up -> h = silu(g) * u rounded once (fp16 *
// 2^th for block-float, bf16 for bf16 weights); down -> out = residual + y.  Every output element is
// owned by one lane of one wave; a tile whose K range is split over a few blocks is finished by a
// second launch, which adds their fp32 partial tiles in K order (deterministic).
#include <algorithm>
#include <mutex>
#include <set>
#include <utility>

#include "qmlp_common.h"
#include "qmlp_internal.h"

namespace qmlp {

struct TlParams {
  const uint8_t* w0;
  const uint8_t* w1;
  const int* rowexp0;
  const int* rowexp1;
  const uint16_t* src;   // [M, K] B rows: fp16 * 2^tsrc[m] (block-float weights) or bf16
  int M, K, N, C;        // N output features, C = K / 256
  int nbm;               // token blocks
  int nfull;             // leading blocks that take one whole tile each
  int ntail;             // tiles that follow, split in K
  int ks;                // K pieces per split tile
  float* part;           // fp32 partial tiles, [split tile][piece][the block's outputs]
  int part_bytes;
  const int* tsrc;       // block-float: per-token exponent of src
  const int* tout;       // block-float gate/up: h16 = h * 2^tout[m]
  void* out;             // gate/up: h [M, N] 16-bit; down: out [M, N] bf16 or fp32
  const void* residual;  // down: [M, N] bf16 or fp32, may alias out
  int out_f32, res_f32;
};

// Runs steps s .. nst-1 of a block's K loop, unrolled by U (the period of the register stage and
// buffer rotation): step(k, s) runs step s, k = s % U (a constant of each unrolled copy).
template <int U, typename F>
__device__ __forceinline__ void run_steps(int s, int nst, F&& step) {
  for (; s + U <= nst; s += U)
#pragma unroll
    for (int k = 0; k < U; ++k) step(k, s + k);
  const int r = nst - s;
#pragma unroll
  for (int k = 0; k < U - 1; ++k)
    if (k < r) step(k, s + k);
}

// ---------------------------------------------------------------- kernel
//
// A operand from the packed layout as it stands: lane l = 32 hk + 16 ts + r takes row r of tile
// 2 P + ts and the packed chunks q = 2 hk and 2 hk + 1 of each K-step (K = 64 j + 32 hk + 0..31),
// i.e. the 16-byte slots of packed lanes 32 hk + r and 32 hk + 16 + r.  Product u (0..3) of the
// step takes the lane's values 8 u .. 8 u + 7 of those 32: K = 64 j + 32 hk + 8 u + (0..7) on the
// lanes whose A index half is hk.  The B fragment of product u therefore holds, in lane
// l = 32 hk + c, the K values 64 j + 32 hk + 8 u + (0..7) of token c of the group.
typedef float f32x16 __attribute__((ext_vector_type(16)));

// 16-byte LDS slot of product u's B fragment for lane l inside one group's 4 KB step image.  The
// 8 lanes 8a..8a+7 of a fragment read one aligned 128-byte run (a rotation of it), and the 8 slots
// one token row writes per step (all (u, hk) pairs) fall on distinct 16-byte bank groups.
__host__ __device__ inline uint32_t b32_slot(int u, int l) {
  return (uint32_t)(u * 64 + (l & ~7) + ((l + 2 * u + (l >> 5)) & 7));
}

template <int WF, int NM>
struct Tl32Stage {
  typename StepWord<WF>::type w[NM][WF ? 2 : 4];
};

// MODE, what the block's 8 waves own:
//   kDown: one 32-row unit of the down matrix each (256 features x MG x 32 tokens);
//   kPair: four units of gate (waves 0-3) and of up (waves 4-7); the two waves of a unit swap
//          halves of their sums through LDS at the end (128 features x MG x 32 tokens);
//   kBoth: one unit of gate and the same of up each (256 features x MG x 32 tokens).
// With one matrix per wave the accumulators leave registers for tiles of up to 224 tokens, and a
// gate/up tile is half as large; with both, each B fragment read from LDS feeds two products: 1.56
// us a step against twice 0.91 at 128 tokens, which large counts of tiles prefer.
//
// Bound by the matrix cores' power-limited rate and what the step adds around the products
// (dequantisation, LDS reads, vector memory return); with few tokens by the weights' arrival.
//
// Work (plan_tiles): blocks [0, nfull) each take one whole tile; blocks from nfull take K pieces of
// the ntail tiles that follow: ks consecutive blocks share a tile, piece q covering 64-K steps
// [q S / ks, (q + 1) S / ks) of its S.  The whole tiles come in complete rounds of resident blocks
// and the pieces start together as those rounds end, so the blocks reading one feature block's
// weights read the same K range at the same time (L2 reuse).  The pieces leave their partial tiles
// in the workspace for sum_kernel; no block ever waits for another, so the kernel cannot stall
// whatever else holds the CUs (other streams, other processes).
constexpr int kTlNWV = 8;  // waves per block

// The tile (or piece) of block b among P, so that each XCD (block b runs on XCD b % 8) takes one
// contiguous run of them, P / 8 or one more, whatever P is: neighbours share weights, or a split
// tile's partial tiles, in its L2.  With the runs only where P is a multiple of 8 and block order
// elsewhere, every XCD read every weight: bf16 gate/up of 4608 x 6400 at 259 tokens, 250 tiles,
// 81.8 us, with them 42.0; a count of 748 tiles at the 27B shape, bound by its products, 427.7 and
// 427.3.
__host__ __device__ constexpr int xcd_run(int b, int P) {
  return b % 8 * (P / 8) + (b % 8 < P % 8 ? b % 8 : P % 8) + b / 8;
}
constexpr bool xcd_runs_are_contiguous(int P) {
  int expect = 0;
  for (int x = 0; x < 8; ++x)
    for (int b = x; b < P; b += 8)
      if (xcd_run(b, P) != expect++) return false;
  return expect == P;
}
static_assert(xcd_runs_are_contiguous(1) && xcd_runs_are_contiguous(250) && xcd_runs_are_contiguous(255) &&
              xcd_runs_are_contiguous(256) && xcd_runs_are_contiguous(748));

// ---------------------------------------------------------------- outputs
//
// Four rows n .. n + 3 of token m, from the sums and their exponents (block-float weights).

// h = silu(g) * u, rounded once; eg, eu: row minus token exponents, to: h's exponent
template <int WF>
__device__ __forceinline__ void put_h(const TlParams& p, int m, int n, f32x4 g, f32x4 u, const int (&eg)[4],
                                      const int (&eu)[4], int to) {
  uint16_t o[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    float gv = g[v], uv = u[v];
    if constexpr (WF) {
      gv = __builtin_amdgcn_ldexpf(gv, eg[v]);
      uv = __builtin_amdgcn_ldexpf(uv, eu[v]);
    }
    const float hv = silu_mul(gv, uv);
    o[v] = WF ? f32_to_f16_bits(__builtin_amdgcn_ldexpf(hv, to)) : f32_to_bf16(hv);
  }
  *(u32x2*)((uint16_t*)p.out + (size_t)m * p.N + n) =
      u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
}

// The residual words of an output (bf16: the low two; fp32: all four; none: zero).
__device__ __forceinline__ u32x4 get_residual(const TlParams& p, int m, int n) {
  if (!p.residual) return u32x4{0u, 0u, 0u, 0u};
  if (p.res_f32) return *(const u32x4*)((const float*)p.residual + (size_t)m * p.N + n);
  const u32x2 w = *(const u32x2*)((const uint16_t*)p.residual + (size_t)m * p.N + n);
  return u32x4{w.x, w.y, 0u, 0u};
}

// out = residual + y * 2^e
template <int WF>
__device__ __forceinline__ void put_out(const TlParams& p, int m, int n, f32x4 y, const int (&e)[4], u32x4 res) {
  const f32x4 r = p.res_f32 ? __builtin_bit_cast(f32x4, res)
                            : f32x4{bf16_to_f32((uint16_t)(res.x & 0xffffu)), bf16_to_f32((uint16_t)(res.x >> 16)),
                                    bf16_to_f32((uint16_t)(res.y & 0xffffu)), bf16_to_f32((uint16_t)(res.y >> 16))};
#pragma unroll
  for (int v = 0; v < 4; ++v) y[v] = (WF ? __builtin_amdgcn_ldexpf(y[v], e[v]) : y[v]) + r[v];
  if (p.out_f32) {
    *(f32x4*)((float*)p.out + (size_t)m * p.N + n) = y;
  } else {
    const uint32_t o0 = f32_to_bf16(y[0]), o1 = f32_to_bf16(y[1]), o2 = f32_to_bf16(y[2]), o3 = f32_to_bf16(y[3]);
    *(u32x2*)((uint16_t*)p.out + (size_t)m * p.N + n) = u32x2{o0 | (o1 << 16), o2 | (o3 << 16)};
  }
}

enum { kDown = 0, kPair = 1, kBoth = 2 };

// LDS: the 3-slot B ring (kPair: later one or two swap buffers of 8 waves x 4 KB), then the exponents.
constexpr size_t kSwapBytes = 32 * 1024;
constexpr size_t tiled32_exp_offset(int MG, int MODE) {
  const size_t ring = (size_t)3 * MG * 4096, swap = MODE == kPair ? (MG > 2 ? 2 : 1) * kSwapBytes : 0;
  return ring > swap ? ring : swap;
}
constexpr size_t tiled32_lds(int MG, int MODE) {
  return tiled32_exp_offset(MG, MODE) + (size_t)((MODE == kBoth ? 512 : 256) + (MODE == kDown ? 1 : 2) * MG * 32) * 4;
}

template <int WF, int MG, int NBB, int MODE, bool ONCE>
__global__ __launch_bounds__(512) void tiled32_kernel(TlParams p) {
  constexpr int NWV = kTlNWV, NT = NWV * 64;
  constexpr int NM = MODE == kBoth ? 2 : 1;       // matrices of one wave
  constexpr int NMATS = MODE == kDown ? 1 : 2;    // matrices of the block
  constexpr int UNITS = NWV * NM / NMATS;         // 32-row units of the block in each matrix
  constexpr int ROWS = NMATS * UNITS * 32;        // row exponents of the block
  constexpr int SLOT = MG * 4096;     // LDS bytes of one 64-K step of B
  // 16-byte B chunks per thread per step; with an odd MG the last chunk of half the threads is
  // their one before it again (every load unconditional: with the upper waves' loads predicated
  // instead, bfp8 tiles of 5 groups were slower than tiles of 6)
  constexpr int NCH = MG * 256, CPT = (NCH + NT - 1) / NT;
  static_assert(MG >= 2, "at least one chunk per thread");
  constexpr int BLK = WF == 2 ? kBf4Block : (WF ? kBfp8Block : kBf16Block);
  constexpr uint32_t PART_BYTES = NWV * NM * MG * 16 * 64 * 4;  // one piece's partial tile
  extern __shared__ __align__(16) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool full = (int)blockIdx.x < p.nfull;
  const int b = full ? (int)blockIdx.x : (int)blockIdx.x - p.nfull;
  const int ks = full ? 1 : p.ks;
  const int L = xcd_run(b, full ? p.nfull : (int)gridDim.x - p.nfull);  // blocks sharing weights share an XCD
  const int tt = L / ks, q = L % ks;  // split tiles: index among them, piece
  if (!full && tt >= p.ntail) return;  // the pieces' rounding up to whole XCDs
  const int tile = full ? L : p.nfull + tt;
  const int bn = tile / p.nbm, bm = tile % p.nbm;
  const int m0 = bm * MG * 32;
  const int unit = wave % UNITS;
  const int pair = bn * UNITS + unit;  // the wave's 32-row unit (of each of its matrices)
  // The piece's 64-K steps [kb, kb + nst) (every step of the K range for a whole tile; pieces cut
  // at step granularity, so that they differ by one step at most) and the superblocks they touch,
  // [k0, k0 + nsb); ph: the first step's position inside its superblock.
  const int kst = p.C * kSteps;
  const int kb = q * kst / ks, nst = (q + 1) * kst / ks - kb;
  const int k0 = kb / kSteps, nsb = (kb + nst - 1) / kSteps - k0 + 1, ph = kb % kSteps;
  // The epilogue's exponents (the block's row exponents, its tokens' exponents)
  // staged in LDS after the B ring: requested first, written to LDS before the first barrier, read
  // after the last.  Kept out of the epilogue's global loads, which could not pass its stores.
  int* lexp = (int*)(lds + tiled32_exp_offset(MG, MODE));  // [ROWS], then [tsrc, tout][MG * 32]
  constexpr int NEXP = WF ? ROWS + NMATS * MG * 32 : 0;
  static_assert(NEXP <= 2 * NT, "two exponents per thread at most");
  int xval[2] = {0, 0};
  if constexpr (WF != 0) {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int i = (int)threadIdx.x + r * NT;
      if (i < ROWS) {
        const int* re = i < UNITS * 32 ? p.rowexp0 : p.rowexp1;
        xval[r] = re[bn * UNITS * 32 + (i & (UNITS * 32 - 1))];
      } else if (i < NEXP) {
        const int j = i - ROWS, mm = min(m0 + j % (MG * 32), p.M - 1);
        xval[r] = j < MG * 32 ? p.tsrc[mm] : p.tout[mm];
      }
    }
  }

  // B chunk c = threadIdx.x + i * NT: token row r = c / 8, K values 8 k8 .. 8 k8 + 7 of the step
  // (k8 = c % 8 = 4 hk + u).  Rows beyond M repeat row M - 1 (their outputs are not stored).
  // Every load goes through a buffer descriptor whose base is uniform (the block's token rows,
  // the wave's weight tiles): the lane's byte offset is a constant 32-bit register and the step's
  // offset a uniform scalar, so no load needs per-lane 64-bit address arithmetic.
  const int brows = min(MG * 32, p.M - m0);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const uint8_t*)p.src + (size_t)m0 * p.K * 2), 0, brows * p.K * 2, kBufferRsrcWord3);
  uint32_t goff[CPT], loff[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int ci = (int)threadIdx.x + i * NT, c = ci < NCH ? ci : ci - NT, r = c >> 3, k8 = c & 7;
    const int mr = min(r, brows - 1);
    goff[i] = (uint32_t)(mr * p.K + k8 * 8) * 2u;
    loff[i] = (uint32_t)(r >> 5) * 4096u + b32_slot(k8 & 3, 32 * (k8 >> 2) + (r & 31)) * 16u;
  }

  auto bload = [&](u32x4(&v)[CPT], int step) {
    const int so = (kb + min(step, nst - 1)) * 128;
#pragma unroll
      for (int i = 0; i < CPT; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b128(rb, goff[i], so, 0);
  };
  auto bstore = [&](const u32x4(&v)[CPT], int step) {
    uint8_t* slot = lds + (step % 3) * SLOT;
#pragma unroll
      for (int i = 0; i < CPT; ++i) *(u32x4*)(slot + loff[i]) = v[i];
  };

  const int hk = lane >> 5;
  const int tile_bytes = p.C * BLK;
  __amdgpu_buffer_rsrc_t wr[NM];  // the wave's two 16-row tiles (2 pair, 2 pair + 1) of each matrix
#pragma unroll
  for (int mat = 0; mat < NM; ++mat)
    wr[mat] = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((mat || (MODE == kPair && wave >= UNITS) ? p.w1 : p.w0) + (size_t)(2 * pair) * tile_bytes), 0,
        2 * tile_bytes, kBufferRsrcWord3);
  const uint32_t lp0 = (uint32_t)(32 * hk + (lane & 15)), lp1 = lp0 + 16u;
  const uint32_t wv = (uint32_t)((lane >> 4) & 1) * (uint32_t)tile_bytes;  // the lane's tile
  // Weights that several token blocks read stay in L2 for them; with one token block (ONCE) they are
  // read once and pass it by.  27B, eight layers in turn, us per layer without -> with: bf16 127.2 ->
  // 120.4 at 64 tokens and 139.2 -> 131.3 at 96; bfp8 79.8 -> 78.2 at 33, 83.1 -> 82.1 at 64 and 104.8 ->
  // 104.4 at 96 (its down launch alone is 0.6 us slower, the layer faster); bf4, whose down launch only
  // uses it, level: 76.0 / 76.2, 79.8 / 80.5 and 95.6 / 94.9.  Two or three layers in turn, which the
  // memory-side cache holds in part, differ by up to 6 us either way.  With several token blocks
  // 1-6 % slower.
  constexpr int POL = ONCE ? 2 : 0;  // buffer cache policy: non-temporal
  auto wload = [&](Tl32Stage<WF, NM>& st, int step) {
    const int sc = kb + min(step, nst - 1);
    const int bo = (sc >> 2) * BLK;
#pragma unroll
    for (int mat = 0; mat < NM; ++mat) {
      if constexpr (WF == 1) {
        const int so = bo + (sc & 3) * 1024;
        st.w[mat][0] = __builtin_amdgcn_raw_buffer_load_b128(wr[mat], wv + lp0 * 16u, so, POL);
        st.w[mat][1] = __builtin_amdgcn_raw_buffer_load_b128(wr[mat], wv + lp1 * 16u, so, POL);
      } else if constexpr (WF == 2) {
        const int so = bo + (sc & 2) * 512 + (sc & 1) * 8;
        st.w[mat][0] = __builtin_amdgcn_raw_buffer_load_b64(wr[mat], wv + lp0 * 16u, so, 0);
        st.w[mat][1] = __builtin_amdgcn_raw_buffer_load_b64(wr[mat], wv + lp1 * 16u, so, 0);
      } else {
        const int so = bo + (sc & 3) * 2048;
        st.w[mat][0] = __builtin_amdgcn_raw_buffer_load_b128(wr[mat], wv + lp0 * 16u, so, POL);
        st.w[mat][1] = __builtin_amdgcn_raw_buffer_load_b128(wr[mat], wv + 1024u + lp0 * 16u, so, POL);
        st.w[mat][2] = __builtin_amdgcn_raw_buffer_load_b128(wr[mat], wv + lp1 * 16u, so, POL);
        st.w[mat][3] = __builtin_amdgcn_raw_buffer_load_b128(wr[mat], wv + 1024u + lp1 * 16u, so, POL);
      }
    }
  };

  // Row exponents, once per superblock and one superblock ahead: the lane's words for its rows lp0
  // and lp1 of each matrix's tile (byte j: step j of the superblock).  Requested with every step's
  // weights they made 2 of a step's 5 vector memory instructions.
  uint32_t ecur[NM][2], enext[NM][2];
  auto eload = [&](uint32_t(&e)[NM][2], int sb) {
    if constexpr (WF != 0) {
      const int so = (k0 + min(sb, nsb - 1)) * BLK + (WF == 2 ? 2048 : 4096);
#pragma unroll
      for (int mat = 0; mat < NM; ++mat) {
        e[mat][0] = __builtin_amdgcn_raw_buffer_load_b32(wr[mat], wv + lp0 * 4u, so, 0);
        e[mat][1] = __builtin_amdgcn_raw_buffer_load_b32(wr[mat], wv + lp1 * 4u, so, 0);
      }
    }
  };
  auto erotate = [&](int sb) {  // after the last step of the piece's superblock sb
    if constexpr (WF != 0) {
#pragma unroll
      for (int mat = 0; mat < NM; ++mat)
#pragma unroll
        for (int c = 0; c < 2; ++c) ecur[mat][c] = enext[mat][c];
      eload(enext, sb + 2);
    }
  };

  f32x16 acc[NM][MG];
#pragma unroll
  for (int mat = 0; mat < NM; ++mat)
#pragma unroll
    for (int g = 0; g < MG; ++g)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mat][g][v] = 0.f;

  uint32_t bs[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) bs[u] = b32_slot(u, lane) * 16u;
  // kq = step % 4: the step's byte of the exponent word
  auto compute = [&](const Tl32Stage<WF, NM>& st, int step, int kq) {
    const uint8_t* slot = lds + (step % 3) * SLOT;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if constexpr (WF) {
        f16x8 a[NM][2];
#pragma unroll
        for (int mat = 0; mat < NM; ++mat) {
          if constexpr (WF == 2)
            dq16_bf4(st.w[mat][c].x, st.w[mat][c].y, scale_pair(ecur[mat][c], kq), a[mat][0], a[mat][1]);
          else
            dq16(st.w[mat][c], scale_pair(ecur[mat][c], kq), a[mat][0], a[mat][1]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int g = 0; g < MG; ++g) {
            const f16x8 b = __builtin_bit_cast(f16x8, *(const u32x4*)(slot + g * 4096 + bs[2 * c + h]));
#pragma unroll
            for (int mat = 0; mat < NM; ++mat)
              acc[mat][g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mat][h], b, acc[mat][g], 0, 0, 0);
          }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int g = 0; g < MG; ++g) {
            const bf16x8 b = __builtin_bit_cast(bf16x8, *(const u32x4*)(slot + g * 4096 + bs[2 * c + h]));
#pragma unroll
            for (int mat = 0; mat < NM; ++mat)
              acc[mat][g] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, st.w[mat][2 * c + h]),
                                                                    b, acc[mat][g], 0, 0, 0);
          }
      }
    }
  };

  // B rows travel global -> registers -> LDS: NBB = 3 B register buffers request step s+5 in
  // iteration s, NBB = 2 request step s+3 at the top of iteration s; weights of step s+3 are
  // requested right after step s's products; one barrier per step.
  constexpr int U = NBB == 3 ? 3 : 6;
  Tl32Stage<WF, NM> s0, s1, s2;
  u32x4 b0[CPT], b1[CPT], b2[CPT];
  bload(b0, 0);
  bload(b1, 1);
  eload(ecur, 0);
  wload(s0, 0);
  wload(s1, 1);
  wload(s2, 2);
  eload(enext, 1);
  bstore(b0, 0);
  bstore(b1, 1);
  bload(b2, 2);
  int s = 0;
  auto stage = [&](int i) -> Tl32Stage<WF, NM>& { return i == 0 ? s0 : (i == 1 ? s1 : s2); };
  if constexpr (WF != 0)
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if ((int)threadIdx.x + r * NT < NEXP) lexp[threadIdx.x + r * NT] = xval[r];
  if constexpr (NBB == 3) {
    bload(b0, 3);
    bload(b1, 4);
    __syncthreads();
    run_steps<U>(s, nst, [&](int k, int s) {
      Tl32Stage<WF, NM>& cur = stage(k % 3);
      u32x4(&bw)[CPT] = k % 3 == 0 ? b2 : (k % 3 == 1 ? b0 : b1);
      compute(cur, s, (s + ph) & 3);
      wload(cur, s + 3);
      bstore(bw, s + 2);
      bload(bw, s + 5);
      if (((s + ph) & 3) == 3) erotate((s + ph) / kSteps);
      __syncthreads();
    });
  } else {
    __syncthreads();
    run_steps<U>(s, nst, [&](int k, int s) {
      Tl32Stage<WF, NM>& cur = stage(k % 3);
      u32x4(&bnext)[CPT] = k % 2 == 0 ? b1 : b2;
      u32x4(&bwrite)[CPT] = k % 2 == 0 ? b2 : b1;
      bload(bnext, s + 3);
      compute(cur, s, (s + ph) & 3);
      // keeps the next weight loads behind the products: hoisted above them, their registers
      // make the compiler wait for every LDS read before its two products
      __builtin_amdgcn_sched_barrier(0);
      wload(cur, s + 3);
      bstore(bwrite, s + 2);
      if (((s + ph) & 3) == 3) erotate((s + ph) / kSteps);
      __syncthreads();
    });
  }

  // A split tile's pieces leave their partial tiles in their slots (tt, q); sum_kernel, the next
  // launch, adds them.
  auto own = [&](int mat, int g, int v4) {
    return f32x4{acc[mat][g][4 * v4], acc[mat][g][4 * v4 + 1], acc[mat][g][4 * v4 + 2], acc[mat][g][4 * v4 + 3]};
  };
  if (ks > 1) {
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(p.part, 0, p.part_bytes, kBufferRsrcWord3);
    const uint32_t slot = (uint32_t)(tt * ks + q) * PART_BYTES + (uint32_t)(wave * NM * MG * 256 + lane) * 16u;
#pragma unroll
    for (int mat = 0; mat < NM; ++mat)
#pragma unroll
      for (int g = 0; g < MG; ++g)
#pragma unroll
        for (int v4 = 0; v4 < 4; ++v4)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, own(mat, g, v4)), prs,
                                                 slot + (uint32_t)((mat * MG + g) * 4 + v4) * 1024u, 0, 0);
    return;
  }
  // Epilogue, one group of 32 tokens at a time.  Accumulator v of lane l holds row
  // 8 (v / 4) + 4 (l / 32) + v % 4 of the wave's 32-row unit for token l % 32 of the group.
  const int col = lane & 31, rq = (lane >> 5) * 4;
  const int* lrow = lexp + unit * 32 + rq;  // this lane's rows: + 8 vq + v (+ UNITS * 32 for up)
  const int* ltok = lexp + ROWS + col;      // this lane's token: + 32 g (+ MG * 32: tout)
  if constexpr (MODE == kDown) {
    // out = residual + y, y = acc * 2^(row exponent - token exponent).  The residual words of up
    // to four groups are requested together, ahead of their stores: one round trip, and none of
    // the loads waits behind a store.  (Requested before the K loop, their completion held up the
    // loop's first in-order waits: +5 us per block.)
    constexpr int RG = MG < 4 ? MG : 4;
#pragma unroll
    for (int g0 = 0; g0 < MG; g0 += RG) {
      u32x4 rres[RG][4];
#pragma unroll
      for (int i = 0; i < RG; ++i)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq)
          rres[i][vq] = get_residual(p, min(m0 + (g0 + i) * 32 + col, p.M - 1), pair * 32 + vq * 8 + rq);
#pragma unroll
      for (int i = 0; i < RG; ++i) {
        const int g = g0 + i;
        if (g >= MG) break;
        const int m = m0 + g * 32 + col;
        if (m >= p.M) continue;
        const int ts = WF ? ltok[32 * g] : 0;
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          int e[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) e[v] = WF ? lrow[8 * vq + v] - ts : 0;
          put_out<WF>(p, m, pair * 32 + vq * 8 + rq, own(0, g, vq), e, rres[i][vq]);
        }
      }
    }
  } else {
    // h = silu(g) * u, rounded once
    auto finish = [&](int g, const f32x4 (&gate)[4], const f32x4 (&up)[4]) {
      const int m = m0 + g * 32 + col;
      if (m >= p.M) return;
      const int ts = WF ? ltok[32 * g] : 0, to = WF ? ltok[MG * 32 + 32 * g] : 0;
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        int eg[4], eu[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          eg[v] = WF ? lrow[8 * vq + v] - ts : 0;
          eu[v] = WF ? lrow[UNITS * 32 + 8 * vq + v] - ts : 0;
        }
        put_h<WF>(p, m, pair * 32 + vq * 8 + rq, gate[vq], up[vq], eg, eu, to);
      }
    };
    if constexpr (MODE == kBoth) {
#pragma unroll
      for (int g = 0; g < MG; ++g) {
        f32x4 a[NM][4];
#pragma unroll
        for (int mat = 0; mat < NM; ++mat)
#pragma unroll
          for (int vq = 0; vq < 4; ++vq) a[mat][vq] = own(mat, g, vq);
        finish(g, a[0], a[NM - 1]);
      }
    } else {
      // The gate wave and the up wave of a unit swap groups through LDS (two buffers in turn, over
      // the B ring): of each two groups the gate wave finishes the first, the up wave the second.
      const bool up = wave >= UNITS;
#pragma unroll
      for (int g0 = 0; g0 < MG; g0 += 2) {
        f32x4* buf = (f32x4*)(lds + (size_t)(g0 & 2) / 2 * kSwapBytes) + lane;
        f32x4 a0[4], a1[4], o[4];
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          a0[vq] = own(0, g0, vq);
          a1[vq] = own(0, g0 + 1 < MG ? g0 + 1 : g0, vq);
          if (up || g0 + 1 < MG) buf[(wave * 4 + vq) * 64] = up ? a0[vq] : a1[vq];
        }
        __syncthreads();
        if (up && g0 + 1 >= MG) continue;
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) o[vq] = buf[((wave ^ UNITS) * 4 + vq) * 64];
        if (up)
          finish(g0 + 1, o, a1);
        else
          finish(g0, a0, o);
      }
    }
  }
}

// Adds the ks partial tiles of each split tile in K order and finishes its outputs: a block per
// (split tile, 32-row unit, group of 32 tokens), a wave per 8 rows, the lanes as in the tile's
// accumulators.  Bound by reading the partial tiles (once, every CU taking part); KB of them are
// requested at once, slots past the last piece beyond the descriptor's extent (they read as zero
// without touching memory), so every load is unconditional.
//
// As a launch of its own it costs its start, ~4 us, and needs no arrival counter, no wait for
// stores at the device level and no lone CU that adds a tile's pieces at the end: the last of a
// tile's blocks used to read all ks partial tiles.
template <int WF, int MODE>
__global__ __launch_bounds__(256) void sum_kernel(TlParams p, int mg) {
  constexpr int KB = 4, NM = MODE == kDown ? 1 : 2, UNITS = MODE == kPair ? 4 : 8;
  const int lane = threadIdx.x & 63, vq = threadIdx.x >> 6;
  const int g = blockIdx.x % mg, unit = blockIdx.x / mg % UNITS, tt = blockIdx.x / mg / UNITS;
  const int tile = p.nfull + tt, bn = tile / p.nbm, bm = tile % p.nbm;
  const int mr = (bm * mg + g) * 32 + (lane & 31), m = min(mr, p.M - 1);
  const int n = (bn * UNITS + unit) * 32 + vq * 8 + (lane >> 5) * 4;
  const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(p.part, 0, p.part_bytes, kBufferRsrcWord3);
  // a piece's slot: [wave][matrix of the wave][group][vq][lane]
  const uint32_t piece = (uint32_t)(kTlNWV * (MODE == kBoth ? 2 : 1) * mg) * 4096u;
  uint32_t off[NM];
#pragma unroll
  for (int mat = 0; mat < NM; ++mat) {
    const int w = MODE == kPair ? unit + mat * UNITS : unit, mw = MODE == kBoth ? mat : 0;
    off[mat] = (uint32_t)(tt * p.ks) * piece +
               (uint32_t)((((w * (MODE == kBoth ? 2 : 1) + mw) * mg + g) * 4 + vq) * 64 + lane) * 16u;
  }
  int er[NM][4], ts = 0, to = 0;
  u32x4 res = u32x4{0u, 0u, 0u, 0u};
  if constexpr (WF != 0) {
#pragma unroll
    for (int mat = 0; mat < NM; ++mat) {
      const u32x4 e = *(const u32x4*)((mat ? p.rowexp1 : p.rowexp0) + n);
#pragma unroll
      for (int v = 0; v < 4; ++v) er[mat][v] = (int)e[v];
    }
    ts = p.tsrc[m];
    if constexpr (MODE != kDown) to = p.tout[m];
  }
  if constexpr (MODE == kDown) res = get_residual(p, m, n);
  f32x4 sum[NM];
#pragma unroll
  for (int mat = 0; mat < NM; ++mat) sum[mat] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int r0 = 0; r0 < p.ks; r0 += KB) {
    f32x4 v[KB][NM];
#pragma unroll
    for (int r = 0; r < KB; ++r)
#pragma unroll
      for (int mat = 0; mat < NM; ++mat)
        v[r][mat] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       prs, r0 + r < p.ks ? off[mat] + (uint32_t)(r0 + r) * piece : 0xfffffff0u, 0, 0));
#pragma unroll
    for (int r = 0; r < KB; ++r)
#pragma unroll
      for (int mat = 0; mat < NM; ++mat) sum[mat] += v[r][mat];
  }
  if (mr >= p.M) return;
#pragma unroll
  for (int mat = 0; mat < NM; ++mat)
#pragma unroll
    for (int v = 0; v < 4; ++v) er[mat][v] = WF ? er[mat][v] - ts : 0;
  if constexpr (MODE == kDown)
    put_out<WF>(p, m, n, sum[0], er[0], res);
  else
    put_h<WF>(p, m, n, sum[0], sum[NM - 1], er[0], er[NM - 1], to);
}

// ---------------------------------------------------------------- host side

// What a launch of tiled32_kernel costs, in us, as measured on MI355X: 22 token counts from 33 to
// 2048 at the 27B shapes (H = 5120, I = 17408), every tile height and the splits within 1.4 x the
// best estimate, about 500 points per mode and format, fitted to 3-5 % rms with the points near the
// fastest weighted most.  The plans chosen are 0.7 % slower on average than the fastest measured there
// (0.9-2.1 % in a later run on another card, at most 12 %, below 100 tokens).  At other shapes
// (H = 1024-5120, I = 3072-16640, 48-2048 tokens) the estimates are up to a fifth too high, as tiles
// over a short K overlap their ends, and the plans are 0.3 (bf4), 1.0 (bf16) and 1.3 % (bfp8) slower
// than the fastest for gate/up, 1.2-1.7 and 3.5 % (bf16) for down, single ones by up to 24 %.
// kCostPair16's publish was fitted as 0 at the 27B shapes; at 3072 x 8192 that split tiles which
// whole ones beat, 58.9 against 45.3 us at 400 tokens and 44.1 against 34.0 at 259.  With .003 the
// bf16 gate/up plans are 1.1 % slower than the fastest on average over all shapes, 2.1 % with 0.
struct TileCost {
  float step[8];   // one 64-K step of a tile of MG groups (0: height not built)
  float tile;      // a tile's, or a piece's, start and end
  float launch;    // the launch's
  float tbps;      // TB/s at which weights nobody shares arrive
  float publish;   // writing and reading one group of one piece's matrix, spread over the CUs
  float add;       // one more piece in the sums of one group of one matrix
  float split;     // the second launch
  float cold;      // what a step takes longer where one token block reads every weight
};
constexpr TileCost kCostPair8{{0, 0, .53f, .75f, .92f, 1.15f, 1.33f, 1.55f}, 1.5f, 4.5f, 7.9f, .006f, .03f, 8.0f, .08f};
constexpr TileCost kCostPair4{{0, 0, .48f, .65f, .89f, 1.20f, 1.30f, 1.51f}, 0.9f, 4.0f, 7.3f, .007f, .07f, 3.7f, .01f};
constexpr TileCost kCostPair16{{0, 0, .57f, .78f, .92f, 1.13f, 1.26f, 1.46f}, 4.9f, 6.7f, 5.6f, .003f, .16f, 6.3f, .10f};
constexpr TileCost kCostBoth{{0, 0, 1.02f, 0, 1.60f, 0, 0, 0}, 3.2f, 0.0f, 7.3f, .009f, .04f, 3.1f, .09f};
constexpr TileCost kCostDown8{{0, 0, .53f, .75f, .93f, 1.16f, 1.36f, 1.61f}, 3.1f, 3.9f, 5.7f, .005f, .08f, 4.7f, .00f};
constexpr TileCost kCostDown16{{0, 0, .55f, .73f, .87f, 1.07f, 1.20f, 1.40f}, 5.9f, 6.1f, 7.9f, .006f, .05f, 6.0f, .09f};

// Largest K split of a tile, and how many rounds its pieces may take.
constexpr int kMaxKs = 12, kMaxSplitRounds = 4;

// Bytes of one K piece's partial tile (8 waves x nm 32-row units x mg groups of 32 tokens, fp32).
constexpr size_t split_part_bytes(int nm, int mg) { return (size_t)kTlNWV * nm * mg * 16 * 64 * 4; }

// Work of one projection: `nfull` whole tiles, then the remaining ntail tiles in ks pieces of their
// K range each.
struct TilePlan {
  int mode, mg;
  int nbm, nfull, ntail, ks;
  float cost;
};

// Adds the plans of one mode to `best` where they cost less.  For each tile height: every tile
// whole; every tile split; whole rounds of resident blocks (one per CU) whole and the remainder
// split.  Before heights and multi-round splits were weighed against each other -- tiles of 64 or
// 128 tokens, pieces within one round -- a count of tiles just above a round or a half round left
// up to half the chip idle (27B layer, interleaved: 201 tokens bf4 205 us, now 166; 777 tokens bf16
// 607, now 463; with sum_kernel 210 -> 159 and 614 -> 466).
static void plan_mode(int mode, const TileCost& c, int M, int N, int C, int fmt, int slots, size_t part_bytes,
                      TilePlan* best) {
  const int nm = mode == kBoth ? 2 : 1, kst = C * kSteps;
  const int nbn = N / (mode == kPair ? 128 : 256);
  const int blk = fmt == 2 ? kBf4Block : (fmt ? kBfp8Block : kBf16Block);
  const float step_mb = (float)(kTlNWV * nm * 2 * blk / kSteps) * 1e-6f;  // weights of a block's step
  for (int mg = 2; mg < 8; ++mg) {
    if (c.step[mg] == 0) continue;
    const int nbm = (M + mg * 32 - 1) / (mg * 32), T = nbn * nbm;
    // step(a): with a blocks at work, their distinct weights come from memory
    auto step = [&](int a) {
      return std::max(c.step[mg] + (nbm == 1 ? c.cold : 0.f), (float)a / (float)nbm * step_mb / c.tbps);
    };
    const float full = (float)kst * step(slots) + c.tile;  // a round of whole tiles
    auto whole = [&](int n) {
      const int rest = n % slots;
      return (float)(n / slots) * full + (rest ? (float)kst * step(std::max(rest, nbm)) + c.tile : 0.f);
    };
    auto take = [&](int nfull, int ntail, int ks, float cost) {
      if (cost < best->cost) *best = {mode, mg, nbm, nfull, ntail, ks, cost};
    };
    take(T, 0, 1, c.launch + whole(T));
    for (int lead = 0; lead < 2; ++lead) {
      const int nfull = lead ? T / slots * slots : 0, ntail = T - nfull;
      if (ntail == 0 || (lead && nfull == 0)) continue;
      for (int ks = 2; ks <= kMaxKs && ks <= kst; ++ks) {
        const long long P = (long long)ntail * ks;
        if (P > (long long)kMaxSplitRounds * slots || (size_t)P * split_part_bytes(nm, mg) > part_bytes) break;
        const int rounds = ((int)P + slots - 1) / slots;
        const float groups = (float)(mg * nm);
        take(nfull, ntail, ks,
             c.launch + whole(nfull) +
                 (float)rounds * ((float)((kst + ks - 1) / ks) * step(std::min((int)P, slots)) + c.tile) + c.split +
                 (float)P * groups * c.publish + (float)ks * groups * c.add);
      }
    }
  }
}

static TilePlan plan_tiles(bool down, int M, int N, int C, int fmt, int slots, size_t part_bytes) {
  TilePlan best{};
  best.cost = 1e30f;
  slots = std::max(slots, 1);
  if (down) {
    plan_mode(kDown, fmt ? kCostDown8 : kCostDown16, M, N, C, fmt, slots, part_bytes, &best);
  } else {
    plan_mode(kPair, fmt == 2 ? kCostPair4 : fmt ? kCostPair8 : kCostPair16, M, N, C, fmt, slots, part_bytes, &best);
    if (fmt) plan_mode(kBoth, kCostBoth, M, N, C, fmt, slots, part_bytes, &best);
  }
  return best;
}

// Sized for the most any plan uses (plan_mode bounds its pieces by it): constant in M, so that the
// workspace never shrinks as M grows.
size_t tiled_split_bytes(int M) { return M <= 32 ? 0 : (size_t)kSplitMaxSlots * split_part_bytes(2, 4); }

// Blocks of a plan's launch: the pieces rounded up to whole XCDs, so that consecutive ones share
// an XCD (at most 7 exit at once).
static int tile_blocks(const TilePlan& t) { return t.nfull + (t.ks > 1 ? (t.ntail * t.ks + 7) / 8 * 8 : 0); }

void plan_tiles_info(int M, int H, int I, int fmt, bool down, int num_cus, int* out8) {
  const size_t bytes = tiled_split_bytes(M);
  const TilePlan t = down ? plan_tiles(true, M, H, I / kSuperK, down_format(fmt), num_cus, bytes)
                          : plan_tiles(false, M, I, H / kSuperK, fmt, num_cus, bytes);
  out8[0] = t.mode == kPair ? 128 : 256;
  out8[1] = t.mg * 32;
  out8[2] = t.nfull + t.ntail;
  out8[3] = t.nfull;
  out8[4] = t.ks;
  out8[5] = tile_blocks(t);
  out8[6] = (int)split_part_bytes(t.mode == kBoth ? 2 : 1, t.mg);
  out8[7] = (int)bytes;
}

// Raises a kernel's dynamic LDS limit, once per kernel and device; thread-safe.
static int raise_lds_limit(const void* kern, size_t lds) {
  static std::mutex mu;
  static std::set<std::pair<const void*, int>> done;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return set_error(-7, "tiled32_kernel: no HIP device");
  std::lock_guard<std::mutex> lock(mu);
  if (done.count({kern, dev})) return 0;
  if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return set_error(-4, "tiled32_kernel: cannot enable %zu bytes of LDS", lds);
  done.insert({kern, dev});
  return 0;
}

template <int WF, int MODE, int MG, bool ONCE>
static int launch_tiled32(TlParams p, const TilePlan& t, hipStream_t s) {
  // B register buffers: three where the registers allow them; two for tall tiles, and for the bfp8
  // gate/up pair in one wave (three: 749 against 709-714 us at 2048 tokens, the compiler then waits
  // for every LDS read before its products).
  constexpr int NBB = MG >= 6 || (WF == 1 && MODE == kBoth) ? 2 : 3;
  auto kern = tiled32_kernel<WF, MG, NBB, MODE, ONCE>;
  constexpr size_t lds = tiled32_lds(MG, MODE);
  if (lds > 64 * 1024)
    if (int rc = raise_lds_limit((const void*)kern, lds)) return rc;
  p.nbm = t.nbm;
  p.nfull = t.nfull;
  p.ntail = t.ntail;
  p.ks = t.ks;
  constexpr int slot = MODE == kDown ? 1 : 0;
  launch_timed_part(slot, t.ks > 1 ? 1 : 3, kern, dim3(tile_blocks(t)), dim3(kTlNWV * 64), lds, s, p);
  if (int rc = check_launch("tiled32_kernel")) return rc;
  if (t.ks == 1) return 0;
  launch_timed_part(slot, 2, sum_kernel<WF, MODE>, dim3(t.ntail * (MODE == kPair ? 4 : 8) * MG), dim3(256), 0, s, p, MG);
  return check_launch("sum_kernel");
}

// Weights one token block reads pass the L2 by only where a load takes whole 16-byte pieces: bf4's
// 8-byte loads of two steps share their lines (64 tokens: 85.9 against 80.7 us).  Taller tiles are the
// one token block of few plans (27B: down at 129-160 tokens) and gain less there: bf16 layer 156.5 ->
// 155.4 us, bfp8 134.7 -> 134.1, bf4 level.
template <int WF, int MODE, int MG>
static int launch_height(const TlParams& p, const TilePlan& t, hipStream_t s) {
  if constexpr (WF != 2 && MG <= 3)
    if (t.nbm == 1) return launch_tiled32<WF, MODE, MG, true>(p, t, s);
  return launch_tiled32<WF, MODE, MG, false>(p, t, s);
}

template <int WF, int MODE>
static int launch_mode(const TlParams& p, const TilePlan& t, hipStream_t s) {
  if constexpr (MODE == kBoth) {
    return t.mg == 2 ? launch_height<WF, MODE, 2>(p, t, s) : launch_height<WF, MODE, 4>(p, t, s);
  } else {
    switch (t.mg) {
      case 2: return launch_height<WF, MODE, 2>(p, t, s);
      case 3: return launch_height<WF, MODE, 3>(p, t, s);
      case 4: return launch_height<WF, MODE, 4>(p, t, s);
      case 5: return launch_height<WF, MODE, 5>(p, t, s);
      case 6: return launch_height<WF, MODE, 6>(p, t, s);
      default: return launch_height<WF, MODE, 7>(p, t, s);
    }
  }
}

bool tiled_supported(int M, int H, int I) { return M >= 1 && I % 256 == 0 && H % 256 == 0; }

int launch_forward_tiled(const ForwardArgs& a, int num_cus, hipStream_t s) {
  if (!tiled_supported(a.M, a.H, a.I)) return set_error(-1, "tiled path: H=%d I=%d not multiples of 256", a.H, a.I);
  const WsLayout L = ws_layout(a.M, a.H, a.I, a.fmt);
  const int fmt = a.fmt;
  int* tx = (int*)(a.ws + L.tx);
  int* th = (int*)(a.ws + L.th);
  uint16_t* x16 = (uint16_t*)(a.ws + L.x16);
  uint16_t* h = (uint16_t*)(a.ws + L.h);
  if (fmt != 0) {
    int rc = launch_prep(a, s);
    if (rc) return rc;
  }
  TlParams g{};
  g.w0 = a.wg;
  g.w1 = a.wu;
  g.rowexp0 = (const int*)(a.wg + rowexp_offset(a.I, a.H, fmt));
  g.rowexp1 = (const int*)(a.wu + rowexp_offset(a.I, a.H, fmt));
  g.src = fmt != 0 ? x16 : (const uint16_t*)a.x;
  g.M = a.M;
  g.K = a.H;
  g.N = a.I;
  g.C = a.H / kSuperK;
  g.tsrc = tx;
  g.tout = th;
  g.out = h;
  g.part = (float*)(a.ws + L.split);
  g.part_bytes = (int)std::min<size_t>(L.split_bytes, (size_t)1 << 30);
  const TilePlan tg = plan_tiles(false, a.M, a.I, g.C, fmt, num_cus, (size_t)g.part_bytes);
  int rc;
  if (tg.mode == kBoth)
    rc = fmt == 2 ? launch_mode<2, kBoth>(g, tg, s) : launch_mode<1, kBoth>(g, tg, s);
  else
    rc = fmt == 2   ? launch_mode<2, kPair>(g, tg, s)
         : fmt == 1 ? launch_mode<1, kPair>(g, tg, s)
                    : launch_mode<0, kPair>(g, tg, s);
  if (rc) return rc;
  TlParams d{};
  d.w0 = a.wd;
  const int dfmt = down_format(fmt);
  d.rowexp0 = (const int*)(a.wd + rowexp_offset(a.H, a.I, dfmt));
  d.src = h;
  d.M = a.M;
  d.K = a.I;
  d.N = a.H;
  d.C = a.I / kSuperK;
  d.tsrc = th;
  d.out = a.out;
  d.residual = a.residual;
  d.out_f32 = a.out_f32;
  d.res_f32 = a.res_f32;
  d.part = g.part;
  d.part_bytes = g.part_bytes;
  const TilePlan td = plan_tiles(true, a.M, a.H, d.C, dfmt, num_cus, (size_t)d.part_bytes);
  return dfmt == 1 ? launch_mode<1, kDown>(d, td, s) : launch_mode<0, kDown>(d, td, s);
}

}  // namespace qmlp
