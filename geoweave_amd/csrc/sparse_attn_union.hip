// Sparse-index attention forward over per-block key unions on the matrix cores (gfx950, D = 64).
//
// The masked dense pass (sparse_attn_dense.hip) forms every (query, key) product although a
// query selects a few per cent of the keys. Here a wave owns 16 queries of one head and forms
// products only with the keys that at least one of its queries selected: with a share r of the
// keys selected per query that is 1 - (1 - r)^16 of them (31 % at 1,024 of 43,968 keys, 17 %
// at 1,024 of 87,936), so matrix work, exponentials and operand reads all shrink by that
// factor, while each K and V row is still read from memory once per workgroup (up to 512
// queries) and shared through LDS. With 16 heads and selections drawn independently the whole call
// takes 4.34 ms against the dense pass's 7.45 at 43,968 keys (K = 1,024) and 11.8 against 28.4 at
// 87,936; with an indexer's selections, which share more keys, 3.93 and 11.6.
//
// Pieces (all on the caller's stream):
//   union_lists_kernel  - the (block, tile) records of gw_union.h from the positions; a position
//                         listed twice for one query flags its 32-query block, which the gather
//                         kernel then computes (the reference counts a repeated position twice).
//   dense_vmax_kernel   - largest |v| per (head, d) column, and a flag per batch element whose K
//                         or V holds an inf or nan (computed by the gather kernel: a row that a
//                         query did not select must not reach it through 0 * inf).
//   union_tiles_kernel  - K rows and fp16 V rows (scaled per column by an exact power of two) in
//                         the LDS image of a tile, so that staging a tile is one contiguous copy.
//   union_attn_kernel   - the attention.
#include <math.h>

#include <algorithm>
#include <numeric>
#include <type_traits>

#include "gw_attn.h"
#include "gw_common.h"
#include "gw_dense.h"
#include "gw_union.h"
#include "gw_vscale.h"

namespace gw {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __fp16 fp16x4_t __attribute__((ext_vector_type(4)));

// D = A B + C for a 16x16 tile with a k-step of 32. Lane l supplies A[l % 16][8 (l / 16) + i]
// and B[8 (l / 16) + i][l % 16] (i < 8); accumulator entry r of lane l is D[4 (l / 16) + r][l % 16].
__device__ __forceinline__ f32x4 mma16(BF16, uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma16(FP16, uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                0, 0);
}

// ---------------------------------------------------------------------------------------
// Records of one 16-query block per workgroup: the block's positions set bits in an LDS array
// of 16-bit query sets (one per key of the chunk); then one wave per tile orders the tile's
// selected keys by (rank within the residue class mod 8, class) and writes the record. A chunk
// of tiles is as large as two workgroups per CU allow; each further chunk rereads the positions.
// ---------------------------------------------------------------------------------------
constexpr int kULThreads = 512;
constexpr int kULWaves = kULThreads / 64;
constexpr int kULMaxChunk = 136;  // tiles per chunk: 68 KB of query sets, two workgroups per CU

__global__ __launch_bounds__(kULThreads) void union_lists_kernel(
    const int32_t* __restrict__ pos, int64_t psb, int64_t pst, int T, int S, int K, int ntiles, int chunk, int vec,
    int vmax_words, int nqb, int blk0, uint8_t* __restrict__ rec, int* __restrict__ flags,
    uint32_t* __restrict__ vmax, int* __restrict__ bad) {
  extern __shared__ __align__(16) uint32_t qset[];  // key s of the chunk: 16 bits of word s / 2
  __shared__ __align__(16) uint32_t slots[kULWaves][kUTile];  // per wave: row offset | query set << 16
  __shared__ int dup_any;
  const int blk = blk0 + blockIdx.x, b = blockIdx.y, nblk = gridDim.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rows = min(kUQ, T - blk * kUQ);  // <= 0 for the padding blocks
  const int32_t* pblk = pos + b * psb + (int64_t)min(blk * kUQ, T - 1) * pst;
  if (blk == 0) {
    for (int i = threadIdx.x; i < vmax_words; i += kULThreads) vmax[(int64_t)b * vmax_words + i] = 0u;
    if (threadIdx.x == 0) bad[b] = 0;
  }
  if (threadIdx.x == 0) dup_any = 0;
  bool dup = false;
  uint8_t* brec = rec + ((int64_t)b * nblk + blockIdx.x) * ntiles * kURec;
  for (int t0 = 0; t0 < ntiles; t0 += chunk) {
    const int nt = min(chunk, ntiles - t0);
    const int k0 = t0 * kUTile;
    const uint32_t len = (uint32_t)min(nt * kUTile, S - k0);
    for (int i = threadIdx.x; i < nt * (kUTile / 8); i += kULThreads)
      reinterpret_cast<uint4*>(qset)[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    // Positions outside the chunk (other chunks, negative padding, >= S) wrap to large offsets.
    auto put = [&](int32_t sidx, int i) {
      const uint32_t sl = (uint32_t)sidx - (uint32_t)k0;
      if (sl < len) {
        const uint32_t bit = 1u << ((uint32_t)i + 16u * (sl & 1u));
        dup |= (atomicOr(&qset[sl >> 1], bit) & bit) != 0u;
      }
    };
    if (vec) {
      const int n4 = K >> 2;
      for (int j4 = threadIdx.x; j4 < n4; j4 += kULThreads) {
#pragma unroll 1
        for (int r0 = 0; r0 < rows; r0 += 8) {
          int4 v[8];
#pragma unroll
          for (int u = 0; u < 8; ++u)
            v[u] = r0 + u < rows ? reinterpret_cast<const int4*>(pblk + (int64_t)(r0 + u) * pst)[j4]
                                 : make_int4(-1, -1, -1, -1);
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            put(v[u].x, r0 + u);
            put(v[u].y, r0 + u);
            put(v[u].z, r0 + u);
            put(v[u].w, r0 + u);
          }
        }
      }
    } else {
#pragma unroll 1
      for (int i = 0; i < rows; ++i) {
        const int32_t* prow = pblk + (int64_t)i * pst;
        for (int j = threadIdx.x; j < K; j += kULThreads) put(prow[j], i);
      }
    }
    __syncthreads();
    for (int tl = wave; tl < nt; tl += kULWaves) {
      // Lane l holds keys 4 l + e (e < 4), of residue class 4 (l % 2) + e.
      const uint2 mk = *reinterpret_cast<const uint2*>(qset + tl * (kUTile / 2) + lane * 2);
      const uint32_t ms[4] = {mk.x & 0xFFFFu, mk.x >> 16, mk.y & 0xFFFFu, mk.y >> 16};
      uint32_t* sl = slots[wave];
      reinterpret_cast<uint4*>(sl)[lane] = make_uint4(0, 0, 0, 0);
      const uint64_t par = 0x5555555555555555ull;
      uint64_t bal[4];
      int n[8], tot = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bal[e] = __builtin_amdgcn_ballot_w64(ms[e] != 0u);
        n[e] = __popcll(bal[e] & par);
        n[4 + e] = __popcll(bal[e] & ~par);
        tot += n[e] + n[4 + e];
      }
      lds_fence();
      const uint64_t mine = ((lane & 1) ? ~par : par) & ((1ull << lane) - 1ull);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = __popcll(bal[e] & mine);
        const int c = 4 * (lane & 1) + e;
        int at = 0;
#pragma unroll
        for (int c2 = 0; c2 < 8; ++c2) at += min(n[c2], r + (c2 < c ? 1 : 0));
        if (ms[e] != 0u) sl[at] = union_row((uint32_t)(4 * lane + e)) | (ms[e] << 16);
      }
      lds_fence();
      const int un = (tot + 15) >> 4;
      uint8_t* r = brec + (int64_t)(t0 + tl) * kURec;
      for (int g = 0; g == 0 || 8 * g < un; ++g) {
        const int hi = lane >> 4, q = lane & 15;
        uint32_t w = 0xFFFFFFFFu;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            const uint4 v = *reinterpret_cast<const uint4*>(sl + 32 * (4 * g + s) + 16 * f + 4 * hi);
            const uint32_t vv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) w ^= ((vv[j] >> (16 + q)) & 1u) << (8 * j + 7 - 2 * s - f);
          }
        *reinterpret_cast<uint32_t*>(r + 256 * g + 4 * lane) = w;
        const int at = 32 * (4 * g + hi) + q;
        const uint32_t cnt = lane == 0 && g == 0 ? ((uint32_t)un & 15u) | (((uint32_t)un & 16u) << 12) : 0u;
        *reinterpret_cast<uint32_t*>(r + 512 + 256 * g + 4 * lane) = (sl[at] & 0xFFFFu) | (sl[at + 16] << 16) | cnt;
      }
      lds_fence();
    }
    __syncthreads();
  }
  if (dup) dup_any = 1;
  __syncthreads();
  if (threadIdx.x == 0 && (blk >> 1) < nqb) flags[((int64_t)b * nqb + (blk >> 1)) * 2 + (blk & 1)] = dup_any;
}

// ---------------------------------------------------------------------------------------
// The LDS image of a tile, [B][H][tile][64 KB]: planes K dims 0-31, K dims 32-63, V dims 0-31,
// V dims 32-63, each 256 rows of 64 bytes with the 16-byte chunks XOR-swizzled by (row / 2) % 4
// (union_row). Eight rows of distinct residues mod 8 read at one chunk, or at one 32-byte half,
// then touch distinct banks; the records order the slots by residue for that. Zero past S.
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void union_tiles_kernel(const uint16_t* __restrict__ k, int64_t ksb, int64_t kss,
                                                          int64_t ksh, const uint16_t* __restrict__ v, int64_t vsb,
                                                          int64_t vss, int64_t vsh, int S, int H, int ntiles,
                                                          int in_fp16, const uint32_t* __restrict__ vmax,
                                                          uint8_t* __restrict__ tiles) {
  __shared__ int es[64];
  const int h = blockIdx.y, b = blockIdx.z;
  const int tile = blockIdx.x >> 2, r0 = (blockIdx.x & 3) * 64;  // 64 rows of the tile
  if (threadIdx.x < 64) es[threadIdx.x] = vscale_exp(vmax[((int64_t)b * H + h) * 64 + threadIdx.x]);
  __syncthreads();
  uint8_t* out = tiles + (((int64_t)b * H + h) * ntiles + tile) * kUTileBytes;
#pragma unroll
  for (int pl = 0; pl < 2; ++pl) {
    const int r = r0 + (threadIdx.x >> 2), at = threadIdx.x & 3;
    const int c = pl * 4 + (at ^ ((r >> 1) & 3));
    const int s = tile * kUTile + r;
    uint4 kv = make_uint4(0, 0, 0, 0), vv = kv;
    if (s < S) {
      kv = *reinterpret_cast<const uint4*>(k + b * ksb + (int64_t)s * kss + h * ksh + c * 8);
      vv = *reinterpret_cast<const uint4*>(v + b * vsb + (int64_t)s * vss + h * vsh + c * 8);
    }
    const uint32_t w[4] = {vv.x, vv.y, vv.z, vv.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = pack_f16(ldexpf(in_to_float(in_fp16, w[i] & 0xFFFFu), es[c * 8 + 2 * i]),
                      ldexpf(in_to_float(in_fp16, w[i] >> 16), es[c * 8 + 2 * i + 1]));
    uint8_t* dst = out + pl * kUPlane + r * 64 + at * 16;
    *reinterpret_cast<uint4*>(dst) = kv;
    *reinterpret_cast<uint4*>(dst + 2 * kUPlane) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// ---------------------------------------------------------------------------------------
// The attention. A wave: 16 queries of one head; its lane (g, i) = (l / 16, l % 16) holds query
// i. Per step of 32 listed keys: S^T = K Q^T (two 16x16 tiles, two k-steps) from the selection
// as the initial accumulator (0, or -inf for a pair that is not selected); the weights
// p = exp2(s * scale log2 e - m), packed to fp16, are already the B operand of
// O^T += V^T P^T, whose A operand comes from the V rows by transposing LDS reads.
// The reference maximum is lazy, as in the masked dense pass: it moves only when a lane's
// weights of a step sum to more than kUSumCap.
//
// Bound (43,968 keys, 16 waves of one block each): VALU issue. A wave issues about 65 VALU and 8
// matrix instructions a step; by the counters a SIMD issues VALU 65 % of the cycles and its
// matrix core is busy 29 %, 38 % of that beside VALU. Part of the rest is the end of a tile, where
// the waves, of different step counts, meet at the barrier and queue for their first operands.
// Sixteen queries a block rather than 32: the union of 32 queries is 1.7 times as large at these
// sizes, so the exponentials grow by that while only the LDS reads shrink. Tiles of 256 keys: the
// largest that fit twice. Lists through buffer loads two tiles ahead (a flat load also counts as
// an LDS access, and every operand read waits for it). A tile's last step takes 16 slots when the
// rest are empty (4.6 -> 4.34 ms).
// Measured and not kept: the selection as a 4-bit-float matrix product instead of eight bit
// selects a step (4.52 ms: the product sits at the head of the step's dependent chain).
// ---------------------------------------------------------------------------------------
constexpr float kUSumCap = 32768.f;

// Lanes l and l ^ 16 exchange (v_permlane16_swap); both get op(own, partner).
__device__ __forceinline__ float row_max(float x) {
  const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
}
__device__ __forceinline__ float row_sum(float x) {
  const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
}

struct UnionParams {
  const uint16_t* q;
  const uint8_t* tiles;
  const uint8_t* rec;
  const uint32_t* vmax;
  const int* flags;
  const int* bad;
  uint16_t* o;
  float* lse;
  int64_t qsb, qst, qsh;
  int64_t osb, ost, osh;
  int T, H, nqb, ntiles;
  int blk0, nblk;  // the launch's 16-query blocks [blk0, blk0 + nblk), whose records rec holds
  float scale_log2;
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const u32x4 lds_u4;
typedef __attribute__((address_space(3))) fp16x4_t lds_h4;

__device__ __forceinline__ uint4 lds_read16(uint32_t a) {
  return __builtin_bit_cast(uint4, *reinterpret_cast<lds_u4*>((uintptr_t)a));
}
__device__ __forceinline__ uint32_t lds_read4(uint32_t a) {
  return *reinterpret_cast<__attribute__((address_space(3))) const uint32_t*>((uintptr_t)a);
}
__device__ __forceinline__ void lds_write4(uint32_t a, uint32_t x) {
  *reinterpret_cast<__attribute__((address_space(3))) uint32_t*>((uintptr_t)a) = x;
}
// 16 lanes read 4 rows of 32 bytes (lane i: 8 bytes of row i / 4); lane i receives column i of
// the four rows.
__device__ __forceinline__ uint2 lds_read_tr(uint32_t a) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4f16(reinterpret_cast<lds_h4*>((uintptr_t)a)));
}

// -inf where bit 7 of byte j of w is set, else 0 (one sign-extended byte select and mask).
__device__ __forceinline__ float select_bias16(uint32_t w, int j) {
  return __uint_as_float((uint32_t)(int32_t)(int8_t)(w >> (8 * j)) & 0xFF800000u);
}

template <typename E, int NB>
__global__ __launch_bounds__(1024) void union_attn_kernel(const UnionParams p) {
  // Two tiles of K and V rows, then two lists of row offsets (256 bytes) per wave and block.
  __shared__ __align__(16) uint8_t buf[2 * kUTileBytes + kUMaxWaves * NB * 512 + 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;
  const int h = blockIdx.x % p.H;  // consecutive workgroups (different XCDs) take different heads
  const int wg = blockIdx.x / p.H;
  const int b = blockIdx.y;
  const int g = lane >> 4, i16 = lane & 15;
  const float sl2 = p.scale_log2;
  const int ntiles = p.ntiles;

  int blk[NB];  // of the launch
  uint4 qb[NB][2];
  f32x4 acc[NB][4];
  float m[NB], l[NB];  // reference (exp2 domain; finite before the first selected key), row sum
  const char* rec[NB];
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    blk[a] = (wg * nw + wave) * NB + a;
    const int t = (p.blk0 + blk[a]) * kUQ + i16;
    const bool ok = blk[a] < p.nblk && t < p.T;
    const uint16_t* qr = p.q + b * p.qsb + (int64_t)(ok ? t : 0) * p.qst + h * p.qsh + g * 8;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      qb[a][ks] = ok ? *reinterpret_cast<const uint4*>(qr + ks * 32) : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int d = 0; d < 4; ++d) acc[a][d] = (f32x4){0.f, 0.f, 0.f, 0.f};
    m[a] = -3.4028234663852886e38f;
    l[a] = 0.f;
    rec[a] = uniform_ptr(
        reinterpret_cast<const char*>(p.rec + ((int64_t)b * p.nblk + min(blk[a], p.nblk - 1)) * ntiles * kURec));
  }

  const uint8_t* src = p.tiles + ((int64_t)b * p.H + h) * ntiles * kUTileBytes;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)buf;
  // The workgroups of a head copy the same tiles at about the same time: each starts at another
  // of the tile's 1 KB segments, so that they ask different cache channels.
  const int rot = wg * 5;
  auto stage = [&](int n, uint32_t to) __attribute__((always_inline)) {
    const uint8_t* tb = src + (int64_t)n * kUTileBytes;
    for (int s0 = wave; s0 < kUTileBytes / 1024; s0 += nw) {
      const uint32_t s = (uint32_t)(s0 + rot) & (kUTileBytes / 1024 - 1);
      lds_dma16_s(tb + s * 1024, (uint32_t)lane * 16u, to + s * 1024);
    }
  };
  const uint32_t kx = lds0 + ((uint32_t)g << 4);
  const uint32_t vx = lds0 + (((uint32_t)i16 >> 1 & 1u) << 4) + (((uint32_t)i16 & 1u) << 3) + 2 * kUPlane;
  const uint32_t ko = (uint32_t)i16 * 4u, vo = (uint32_t)(4 * g + (i16 >> 2)) * 4u;

  // One step of block a, its 32 slots or (half a step, F = 1) its first 16: w holds the step's
  // bits at bits 7 (slots 0-15) and 6 (slots 16-31) of its bytes.
  auto step = [&](auto fc, int a, uint32_t w, uint32_t kr, uint32_t vr, uint32_t kl, uint32_t vl) __attribute__((always_inline)) {
    constexpr int F = decltype(fc)::value;
    uint4 ka[F][2];
    uint2 va[4][F];
    const uint32_t wb[2] = {w, w << 1};
    const uint32_t kro[2] = {kr & 0xFFFFu, kr >> 16}, vro[2] = {vr & 0xFFFFu, vr >> 16};
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const uint32_t at = kro[f] ^ kl;
      ka[f][0] = lds_read16(at);
      ka[f][1] = lds_read16(at + kUPlane);
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const uint32_t at = vro[f] ^ vl, at2 = at ^ 32u;
      va[0][f] = lds_read_tr(at);
      va[1][f] = lds_read_tr(at2);
      va[2][f] = lds_read_tr(at + kUPlane);
      va[3][f] = lds_read_tr(at2 + kUPlane);
    }
    f32x4 s[F];
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
      for (int j = 0; j < 4; ++j) s[f][j] = select_bias16(wb[f], j);
#pragma unroll
    for (int f = 0; f < F; ++f) s[f] = mma16(E{}, ka[f][0], qb[a][0], s[f]);
#pragma unroll
    for (int f = 0; f < F; ++f) s[f] = mma16(E{}, ka[f][1], qb[a][1], s[f]);
    float pv[F][4];
    auto weights = [&](float nm) __attribute__((always_inline)) {
      float t[F];
#pragma unroll
      for (int f = 0; f < F; ++f) {
#pragma unroll
        for (int j = 0; j < 4; ++j) pv[f][j] = fexp2(fmaf(s[f][j], sl2, nm));
        t[f] = (pv[f][0] + pv[f][1]) + (pv[f][2] + pv[f][3]);
      }
      return F == 2 ? t[0] + t[F - 1] : t[0];
    };
    float ls = weights(-m[a]);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(ls <= kUSumCap)) != 0ull, 0)) {
      // Every query of the block moves its reference to its largest selected score of this step
      // if that is higher; O and the row sum are rescaled and the weights formed again.
      float mx = -INFINITY;
#pragma unroll
      for (int f = 0; f < F; ++f)
#pragma unroll
        for (int j = 0; j < 4; ++j) mx = fmaxf(mx, s[f][j]);
      mx = pair_max(row_max(mx));
      const float mn = fmaxf(m[a], mx * sl2);
      const float alpha = fexp2(m[a] - mn);
      m[a] = mn;
      l[a] *= alpha;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[a][d][r] *= alpha;
      ls = weights(-mn);
    }
    l[a] += ls;
    uint4 pb = make_uint4(pack_f16(pv[0][0], pv[0][1]), pack_f16(pv[0][2], pv[0][3]), 0u, 0u);
    if constexpr (F == 2) {
      pb.z = pack_f16(pv[1][0], pv[1][1]);
      pb.w = pack_f16(pv[1][2], pv[1][3]);
    }
#pragma unroll
    for (int d = 0; d < 4; ++d)
      acc[a][d] = mma16(FP16{}, make_uint4(va[d][0].x, va[d][0].y, va[d][F - 1].x, va[d][F - 1].y), pb, acc[a][d]);
  };

  // Tile n is in LDS buffer n % 2; while it is computed, tile n + 1's rows go to the other
  // buffer. The lists come through registers two tiles ahead (lane l: word l of the selection
  // bits and of the row offsets of the first four steps; the other four, where a tile has them,
  // are loaded at the tile's start); a wave writes the row offsets to its own LDS rows, those
  // of tile n + 1 while it computes tile n. One barrier per tile. The copies of tile n + 1 are
  // issued after a wave's first step, so that the first operand reads after the barrier do not
  // queue behind them.
  struct List {
    uint32_t w[NB], pr[NB];
  };
  const uint32_t pl = lds0 + 2 * kUTileBytes + (uint32_t)wave * (2 * NB * 256u);
  auto load_list = [&](int n, List& x) __attribute__((always_inline)) {
    const int64_t at = (int64_t)min(n, ntiles - 1) * kURec;
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      x.w[a] = buffer_load4(rec[a] + at, (uint32_t)lane * 4u);
      x.pr[a] = buffer_load4(rec[a] + at, (uint32_t)lane * 4u + 512u);
    }
  };
  // Row offsets of a tile's list to LDS (odd or even half of the wave's rows), its step counts,
  // and the rows of its first steps.
  auto put_rows = [&](const List& x, uint32_t half, int (&un)[NB], uint32_t (&kr)[NB], uint32_t (&vr)[NB]) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      const uint32_t c = (uint32_t)__builtin_amdgcn_readfirstlane(x.pr[a]);
      un[a] = blk[a] < p.nblk ? (int)((c & 15u) | ((c >> 12) & 16u)) : 0;
      const uint32_t at = pl + half + 256u * a;
      lds_write4(at + (uint32_t)lane * 4u, x.pr[a] & 0xFFF0FFF0u);
      kr[a] = lds_read4(at + ko);
      vr[a] = lds_read4(at + vo);
    }
  };
  List cur, nxt;
  int un[NB];  // units of 16 slots
  uint32_t kr0[NB], vr0[NB];
  load_list(0, cur);
  load_list(1, nxt);
  stage(0, lds0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
  put_rows(cur, 0u, un, kr0, vr0);
  __syncthreads();
#pragma unroll 1
  for (int n = 0; n < ntiles; ++n) {
    const uint32_t bo = (uint32_t)(n & 1) << 16;
    const uint32_t half = (uint32_t)(n & 1) * (NB * 256u);
    uint32_t w1[NB], pr1[NB];
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      w1[a] = pr1[a] = 0u;
      if (un[a] > 8) {
        const char* r = rec[a] + (int64_t)n * kURec;
        w1[a] = buffer_load4(r, (uint32_t)lane * 4u + 256u);
        pr1[a] = buffer_load4(r, (uint32_t)lane * 4u + 768u);
      }
    }
    List aft;
    int unn[NB];
    uint32_t krn[NB], vrn[NB];
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      uint32_t w = cur.w[a], kr = kr0[a], vr = vr0[a];
      const uint32_t pa = pl + half + 256u * a;
      uint32_t pk = pa + ko + 64u, pv = pa + vo + 64u;
      // A whole step and the next one's rows (past the last step: not used).
      auto next_step = [&](int s) __attribute__((always_inline)) {
        uint32_t kr2 = lds_read4(pk), vr2 = lds_read4(pv);
        step(std::integral_constant<int, 2>{}, a, w, kr, vr, kx + bo, vx + bo);
        pk += 64u;
        pv += 64u;
        w <<= 2;
        if (s == 3 && un[a] > 8) {
          w = w1[a];
          lds_write4(pa + (uint32_t)lane * 4u, pr1[a]);
          pk = pa + ko;
          pv = pa + vo;
          kr2 = lds_read4(pk);
          vr2 = lds_read4(pv);
          pk += 64u;
          pv += 64u;
        }
        kr = kr2;
        vr = vr2;
      };
      const int ns = un[a] >> 1;
      int s = 0;
      if (a == 0) {
        if (ns > 0) next_step(0);
        s = 1;
        // Past the end the last tile again, into the buffer no tile reads any more.
        stage(min(n + 1, ntiles - 1), lds0 + (bo ^ 65536u));
        load_list(n + 2, aft);
        put_rows(nxt, half ^ (NB * 256u), unn, krn, vrn);
      }
#pragma unroll 1
      for (; s < ns; ++s) next_step(s);
      if (un[a] & 1) step(std::integral_constant<int, 1>{}, a, w, kr, vr, kx + bo, vx + bo);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): this wave's copies of tile n + 1, its lists
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      un[a] = unn[a];
      kr0[a] = krn[a];
      vr0[a] = vrn[a];
    }
    cur = nxt;
    nxt = aft;
  }

  const uint32_t* vm = p.vmax + ((int64_t)b * p.H + h) * 64;
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    l[a] = pair_sum(row_sum(l[a]));
    const int qb32 = (p.blk0 + blk[a]) >> 1;
    const int t = (p.blk0 + blk[a]) * kUQ + i16;
    bool active = blk[a] < p.nblk && t < p.T && p.bad[b] == 0;
    if (qb32 < p.nqb) {
      const int* f = p.flags + ((int64_t)b * p.nqb + qb32) * 2;
      active &= (f[0] | f[1]) == 0;
    }
    if (active) {
      const float inv = l[a] > 0.f ? __frcp_rn(l[a]) : (l[a] == 0.f ? 0.f : l[a]);
      uint16_t* orow = p.o + b * p.osb + (int64_t)t * p.ost + h * p.osh;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        uint16_t hv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int dd = 16 * d + 4 * g + r;
          hv[r] = to_half_bits(E{}, acc[a][d][r] * inv * ldexpf(1.f, -vscale_exp(vm[dd])));
        }
        *reinterpret_cast<uint2*>(orow + 16 * d + 4 * g) =
            make_uint2((uint32_t)hv[0] | ((uint32_t)hv[1] << 16), (uint32_t)hv[2] | ((uint32_t)hv[3] << 16));
      }
      if (g == 0 && p.lse)
        p.lse[((int64_t)b * p.T + t) * p.H + h] =
            l[a] > 0.f ? (m[a] + flog2(l[a])) * kDLn2 : (l[a] == 0.f ? -INFINITY : l[a]);
    }
  }
}

struct UnionLayout {
  size_t rec, flags, bad, vmax, tiles, total;
  int nqb, ntiles;
  int64_t nblk, chunk;  // 16-query blocks in all, and per launch
};

// The records of a launch hold at most this much; a call with more takes its queries in several
// launches. They grow with T S: 1.94 GB at 87,936 queries and keys, where the dense pass's
// selection words take half of that, 4.8 GB at 137,400, which is three launches.
constexpr int64_t kURecBytes = 2ll << 30;
constexpr int64_t kUCus = 256;

UnionLayout union_layout(int64_t B, int64_t T, int64_t S, int64_t H) {
  UnionLayout L;
  const UnionListSizes u = union_list_sizes(T, S);
  L.ntiles = u.ntiles;
  L.nblk = u.nblk;
  // A launch is whole workgroups of the largest shape (also whole 32-query blocks), and where the
  // records of that many fit, as many as fill all CUs a whole number of times: each launch would
  // else end with CUs idle (137,400 queries, K = 1,500: 29.0 ms in three equal launches, 27.3 so,
  // 27.4 in one).
  const int64_t unit = 2 * kUMaxWaves, round = unit * (kUCus / std::gcd(B * H, kUCus));
  const int64_t fit = std::max<int64_t>(unit, kURecBytes / (B * L.ntiles * kURec) / unit * unit);
  L.chunk = L.nblk <= fit ? L.nblk : fit < round ? fit : fit / round * round;
  L.nqb = (int)((T + 31) / 32);
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  size_t o = 0;
  L.rec = o;
  o = up(o + (size_t)B * L.chunk * L.ntiles * kURec);
  L.flags = o;
  o = up(o + (size_t)B * L.nqb * 2 * 4);
  L.bad = o;
  o = up(o + (size_t)B * 4);
  L.vmax = o;
  o = up(o + (size_t)B * H * 64 * 4);
  L.tiles = o;
  o = up(o + (size_t)B * H * L.ntiles * kUTileBytes);
  L.total = o;
  return L;
}

// Waves per workgroup and 16-query blocks per wave. One workgroup fits a CU's LDS, so a launch
// takes rounds x a workgroup's time: the blocks per SIMD (between the fullest SIMD's and the
// mean; 15 % more each with three waves a SIMD to hide latency instead of four) plus about half a
// block for the copies and barriers, fitted at 8 to 64 views. The shape with the smallest product. Two blocks a wave halve the
// K and V traffic, which bounds long key ranges (87,936 keys: 11.8 ms, one block 14.5); at
// 43,968 one block fills the last round better (4.34 against 4.5 ms).
struct UnionShape {
  int waves, nb;
};
UnionShape union_shape(int64_t nblocks, int64_t heads, int cus) {
  UnionShape best = {16, 1};
  double best_t = 1e300;
  for (int nb = 1; nb <= 2; ++nb)
    for (int w = 16; w >= 9; --w) {
      const int64_t wgs = (nblocks + w * nb - 1) / (w * nb) * heads;
      const int per_simd = (w + 3) / 4;
      const double blocks = 0.5 * (per_simd + 0.25 * w) * nb * (per_simd == 4 ? 1.0 : 1.15);
      const double t = (double)((wgs + cus - 1) / cus) * (blocks + 0.5);
      if (t < best_t) {
        best_t = t;
        best = {w, nb};
      }
    }
  return best;
}

template <typename E>
void launch_union_attn(const UnionParams& p, UnionShape u, dim3 grid, hipStream_t st) {
  if (u.nb == 2)
    hipLaunchKernelGGL((union_attn_kernel<E, 2>), grid, dim3(u.waves * 64), 0, st, p);
  else
    hipLaunchKernelGGL((union_attn_kernel<E, 1>), grid, dim3(u.waves * 64), 0, st, p);
}

}  // namespace
}  // namespace gw

extern "C" size_t gw_sparse_attn_fwd_union_workspace_size(int64_t B, int64_t T, int64_t S, int64_t H, int64_t D,
                                                          int64_t K) {
  if (B <= 0 || T <= 0 || S <= 0 || H <= 0 || K <= 0 || D != 64) return 0;
  return gw::union_layout(B, T, S, H).total;
}

extern "C" int gw_sparse_attn_fwd_union(int dtype, const void* q, const int64_t* q_strides, const void* k,
                                        const int64_t* k_strides, const void* v, const int64_t* v_strides,
                                        const int32_t* kv_pos, int64_t pos_stride_b, int64_t pos_stride_t, void* o,
                                        const int64_t* o_strides, float* lse, int64_t B, int64_t T, int64_t S,
                                        int64_t H, int64_t D, int64_t K, float softmax_scale, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  using namespace gw;
  clear_error();
  GW_CHECK_ARG(dtype == GW_DTYPE_BF16 || dtype == GW_DTYPE_FP16, "unsupported dtype code %d", dtype);
  GW_CHECK_ARG(B >= 0 && T >= 0 && S >= 0 && H >= 1 && K >= 0, "invalid sizes B=%lld T=%lld S=%lld H=%lld K=%lld",
               (long long)B, (long long)T, (long long)S, (long long)H, (long long)K);
  if (D != 64) return set_error(GW_ERR_UNSUPPORTED, "the union forward needs head dim 64, got %lld", (long long)D);
  const float sl2 = softmax_scale * kDLog2e;
  if (!(sl2 >= 0x1p-60f) || !(sl2 <= 0x1p60f))
    return set_error(GW_ERR_UNSUPPORTED, "the union forward needs a softmax scale between 2^-60 and 2^60, got %g",
                     (double)softmax_scale);
  if (B == 0 || T == 0) return GW_OK;
  GW_CHECK_ARG(K >= 1 && S >= 1, "kv_positions must have at least one candidate and S >= 1");
  GW_CHECK_ARG(q && k && v && kv_pos && o, "null tensor pointer");
  GW_CHECK_ARG(q_strides && k_strides && v_strides && o_strides, "null stride array");
  GW_CHECK_ARG(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o), "q/k/v/o must be 16-byte aligned");
  for (int i = 0; i < 3; ++i)
    GW_CHECK_ARG(q_strides[i] % 8 == 0 && k_strides[i] % 8 == 0 && v_strides[i] % 8 == 0 && o_strides[i] % 8 == 0,
                 "b/t/h strides must be multiples of 8 elements");
  GW_CHECK_ARG(B <= 65535 && H <= 65535 && T < (1ll << 31) - 65536 && S < (1ll << 30) && K < (1ll << 31),
               "size exceeds the grid range");
  const UnionLayout L = union_layout(B, T, S, H);
  GW_CHECK_ARG(L.nblk * H < (1ll << 31), "size exceeds the grid range");
  GW_CHECK_ARG(workspace != nullptr && workspace_bytes >= L.total && aligned16(workspace),
               "the union forward needs a 16-byte aligned %zu-byte workspace, got %zu", L.total, workspace_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  uint8_t* rec = ws + L.rec;
  int* flags = reinterpret_cast<int*>(ws + L.flags);
  int* bad = reinterpret_cast<int*>(ws + L.bad);
  uint32_t* vmax = reinterpret_cast<uint32_t*>(ws + L.vmax);
  uint8_t* tiles = ws + L.tiles;
  const int in_fp16 = dtype == GW_DTYPE_FP16 ? 1 : 0;
  const int vec = (K % 4 == 0 && pos_stride_t % 4 == 0 && pos_stride_b % 4 == 0 &&
                   (reinterpret_cast<uintptr_t>(kv_pos) & 15) == 0)
                      ? 1
                      : 0;
  const int passes = (L.ntiles + kULMaxChunk - 1) / kULMaxChunk;
  const int tchunk = (L.ntiles + passes - 1) / passes;
  UnionParams p;
  p.q = static_cast<const uint16_t*>(q);
  p.tiles = tiles;
  p.rec = rec;
  p.vmax = vmax;
  p.flags = flags;
  p.bad = bad;
  p.o = static_cast<uint16_t*>(o);
  p.lse = lse;
  p.qsb = q_strides[0]; p.qst = q_strides[1]; p.qsh = q_strides[2];
  p.osb = o_strides[0]; p.ost = o_strides[1]; p.osh = o_strides[2];
  p.T = (int)T;
  p.H = (int)H;
  p.nqb = L.nqb;
  p.ntiles = L.ntiles;
  p.scale_log2 = sl2;
  for (int64_t blk0 = 0; blk0 < L.nblk; blk0 += L.chunk) {
    const int64_t nblk = std::min(L.chunk, L.nblk - blk0);
    p.blk0 = (int)blk0;
    p.nblk = (int)nblk;
    hipLaunchKernelGGL(union_lists_kernel, dim3((unsigned)nblk, (unsigned)B), dim3(kULThreads),
                       (size_t)tchunk * kUTile * 2, st, kv_pos, pos_stride_b, pos_stride_t, (int)T, (int)S, (int)K,
                       L.ntiles, tchunk, vec, (int)(H * 64), L.nqb, p.blk0, rec, flags, vmax, bad);
    GW_HIP_LAUNCH_CHECK("union_lists_kernel launch");
    if (blk0 == 0) {
      hipLaunchKernelGGL(dense_vmax_kernel, dim3((unsigned)((S + kVmaxKeys - 1) / kVmaxKeys), (unsigned)H, (unsigned)B),
                         dim3(256), 0, st, static_cast<const uint16_t*>(v), v_strides[0], v_strides[1], v_strides[2],
                         static_cast<const uint16_t*>(k), k_strides[0], k_strides[1], k_strides[2], (int)S, (int)H,
                         in_fp16, vmax, bad);
      GW_HIP_LAUNCH_CHECK("dense_vmax_kernel launch");
      hipLaunchKernelGGL(union_tiles_kernel, dim3((unsigned)(L.ntiles * 4), (unsigned)H, (unsigned)B), dim3(256), 0, st,
                         static_cast<const uint16_t*>(k), k_strides[0], k_strides[1], k_strides[2],
                         static_cast<const uint16_t*>(v), v_strides[0], v_strides[1], v_strides[2], (int)S, (int)H,
                         L.ntiles, in_fp16, vmax, tiles);
      GW_HIP_LAUNCH_CHECK("union_tiles_kernel launch");
    }
    // Blocks with queries: at least one (the padding is less than one chunk's granule).
    const int64_t nblocks = std::min(nblk, (T + kUQ - 1) / kUQ - blk0);
    if (nblocks <= 0) break;
    const UnionShape u = union_shape(nblocks, H * B, (int)kUCus);
    const dim3 grid((unsigned)((nblocks + u.waves * u.nb - 1) / (u.waves * u.nb) * H), (unsigned)B);
    if (dtype == GW_DTYPE_BF16)
      launch_union_attn<BF16>(p, u, grid, st);
    else
      launch_union_attn<FP16>(p, u, grid, st);
    GW_HIP_LAUNCH_CHECK("union_attn_kernel launch");
  }
  return attn_fwd_flagged_blocks(dtype, q, q_strides, k, k_strides, v, v_strides, kv_pos, pos_stride_b, pos_stride_t,
                                 o, o_strides, lse, nullptr, B, T, S, H, D, K, softmax_scale, nullptr, 0, 0, 0, 0.f,
                                 nullptr, nullptr, 0, flags, bad, L.nqb, 2, stream);
}
