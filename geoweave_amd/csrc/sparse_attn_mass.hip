// Attention mass of the selected keys, attn_sum[b, t, j] = sum_h exp(scale q.k - lse) at the
// key of position j (gfx950, D = 64), given the forward's lse (reference
// sparse_index_flash_attn.py:375-458). With logits, the row's indexer KL loss as well
// (indexer_kl_fused.py:8-155).
//
// The mass sums over heads what a forward pass holds one head at a time. Storing every selected
// score of every head for a later sum is 64 bytes a selected pair each way and, in the dense
// forward, doubles its instructions (5,496 keys, 16 heads, K = 1,024: 373 us against 190 us
// without, and 167 us for the sum). Here a second pass recomputes: a wave owns 32 queries x 128
// keys, keeps their sums over the heads in registers, and per head forms S^T = K Q^T on the
// matrix cores and adds exp2(s * scale log2 e - lse2) - no selection, no V, no row sums. The
// sums go to a score matrix of a chunk of queries, at most 256 MiB or one workgroup's queries,
// from which attn_mass_gather_kernel takes the selected ones. A value that is not selected is
// never read, so it needs no mask (also where it overflows or a key row is not finite).
//
// Sixteen waves share the head's K tile in LDS, four a SIMD at 120 registers. Bound: latency; the
// VALU, which a pair and head costs an FMA, an exponential and an add, is active 46 % of the
// cycles, the matrix cores 20 % (counters at 9,384 keys), and a timing copy without the copies to
// LDS, or without the exponentials, is 10-14 % faster. Eight waves of two
// 32-query blocks (232 registers) took 6.9 against 6.3 ms at 32,976 keys, their query operands
// read by the lanes instead of staged 7.6. At 5,496 keys this kernel takes 141 us and the gather 28;
// the whole forward with the mass 0.56 -> 0.37 ms against the stored scores, at 10,992 keys 1.31 -> 1.23.
#include <math.h>

#include "gw_common.h"
#include "gw_dense.h"

namespace gw {
namespace {

constexpr int kMWaves = 16;
constexpr int kMKeys = 128;                // keys per tile
constexpr int kMRows = kMWaves * 32;       // queries per workgroup
constexpr int64_t kMChunkBytes = 256ll << 20;  // score matrix of one chunk of query groups
constexpr int kMassMaxK = 1024;            // a row's values sit in registers in the gather

struct MassParams {
  const uint16_t* q;
  const uint16_t* k;
  const float* lse;  // natural log, [B, T, H]
  float* a;          // [rows of the chunk][Spad]
  int64_t qsb, qst, qsh;
  int64_t ksb, kss, ksh;
  int g0, ngroup;    // the chunk's groups of kMRows queries: [g0, g0 + ngroup)
  int gpb;           // groups per batch element: group g is queries [kMRows (g % gpb), ...) of element g / gpb
  int T, S, Spad, H;
  float scale_log2;
};

template <typename E>
__global__ __launch_bounds__(kMWaves * 64) void attn_mass_kernel(const MassParams p) {
  // Two K tiles (a head's and the next one's), then each wave's 32 query rows of one head.
  __shared__ __align__(16) uint8_t kt[2 * kMKeys * 128 + kMRows * 128];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int grp = blockIdx.x % p.ngroup, k0 = (blockIdx.x / p.ngroup) * kMKeys;
  const int b = (p.g0 + grp) / p.gpb, t0 = (p.g0 + grp) % p.gpb * kMRows;
  const int rows = min(kMRows, p.T - t0);
  const float sl2 = p.scale_log2;
  const int row0 = wave * 32;  // this wave's first row of the group
  const bool ok = row0 + col < rows;
  const float* lse = p.lse + ((int64_t)b * p.T + t0 + (ok ? row0 + col : 0)) * p.H;
  f32x16 acc[4];
#pragma unroll
  for (int st = 0; st < 4; ++st)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[st][i] = 0.f;

  // Rows reach LDS by direct copies, 8 rows of 128 bytes each: row R's 16-byte chunk c sits at
  // c ^ swz(R). A head's K tile is 16 of them, one per wave; a wave's own query rows four, which
  // it reads into registers before the next head's replace them (read from memory by their
  // lanes, 32 rows a load, they took as long as the products). Rows past the end read the last.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)kt;
  const uint32_t qs0 = lds0 + 2 * kMKeys * 128 + (uint32_t)wave * 4096u;
  const uint32_t kss_b = (uint32_t)p.kss * 2u, qst_b = (uint32_t)p.qst * 2u;
  const int qfirst = min(row0, rows - 1);
  const char* kbase = reinterpret_cast<const char*>(p.k + b * p.ksb + (int64_t)k0 * p.kss);
  const char* qbase = reinterpret_cast<const char*>(p.q + b * p.qsb + (int64_t)(t0 + qfirst) * p.qst);
  const int kR = wave * 8 + (lane >> 3);
  const uint32_t koff = __umul24((uint32_t)min(kR, p.S - 1 - k0), kss_b) + (uint32_t)(((lane & 7) ^ swz(kR)) << 4);
  uint32_t qoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int R = i * 8 + (lane >> 3);
    qoff[i] = __umul24((uint32_t)(min(row0 + R, rows - 1) - qfirst), qst_b) + (uint32_t)(((lane & 7) ^ swz(R)) << 4);
  }
  float l2n;
  auto stage = [&](int h, uint32_t kto) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_dma16_s(qbase + (int64_t)h * p.qsh * 2, qoff[i], qs0 + i * 1024);
    lds_dma16_s(kbase + (int64_t)h * p.ksh * 2, koff, kto + (uint32_t)wave * 1024u);
    l2n = lse[h];
  };
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  auto lds16 = [](uint32_t at) __attribute__((always_inline)) {
    return __builtin_bit_cast(uint4, *reinterpret_cast<__attribute__((address_space(3))) const u32x4*>((uintptr_t)at));
  };
  const int fc = swz(col);
  uint32_t rd[4];  // operand chunk 2 ks + half of row col
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) rd[ks] = (uint32_t)(col * 128 + (((2 * ks + half) ^ fc) << 4));
  // Workgroups start at different heads: a head's rows lie 2 KB apart (bthd), on few cache
  // channels, and all workgroups would ask those at once. The sums' order follows the grid.
  const int h0 = (int)(blockIdx.x % (uint32_t)p.H);
  auto head = [&](int i) { return h0 + i < p.H ? h0 + i : h0 + i - p.H; };
  stage(h0, lds0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
  __syncthreads();
#pragma unroll 1
  for (int h = 0; h < p.H; ++h) {
    const uint32_t bo = lds0 + (uint32_t)(h & 1) * (kMKeys * 128);
    const float nl2 = -l2n * kDLog2e;
    uint4 qa[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qa[ks] = lds16(qs0 + rd[ks]);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the query rows are in registers
    asm volatile("" ::: "memory");
    // Past the last head its rows again, where nothing is read any more.
    stage(head(min(h + 1, p.H - 1)), lds0 + (uint32_t)((h + 1) & 1) * (kMKeys * 128));
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      f32x16 s = f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) s = mma(E{}, lds16(bo + rd[ks] + st * 4096), qa[ks], s);
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[st][i] += fexp2(fmaf(s[i], sl2, nl2));
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): this wave's copies of the next rows
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  if (!ok) return;
  float* row = p.a + ((int64_t)grp * kMRows + row0 + col) * p.Spad + k0 + 4 * half;
#pragma unroll
  for (int st = 0; st < 4; ++st)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4*>(row + 32 * st + 8 * g) =
          make_float4(acc[st][4 * g], acc[st][4 * g + 1], acc[st][4 * g + 2], acc[st][4 * g + 3]);
}

struct MassGatherParams {
  const uint16_t* q;  // q, k and lse: for rows with an empty head
  const uint16_t* k;
  const float* lse;
  int64_t qsb, qst, qsh;
  int64_t ksb, kss, ksh;
  int in_fp16, H;
  float scale_log2;
  const int32_t* pos;
  int64_t psb, pst;
  float* a;
  float* attn_sum;  // [B, T, K]
  const void* logits;
  int logits_dt;
  int64_t lsb, lst;
  float kl_eps;
  float* row_loss;
  int g0, ngroup, gpb, T, S, Spad, K;
};

__device__ __forceinline__ float mass_load(int dt, const void* base, int64_t i) {
  if (dt == GW_DTYPE_FP32) return static_cast<const float*>(base)[i];
  const uint32_t u = static_cast<const uint16_t*>(base)[i];
  if (dt == GW_DTYPE_BF16) return __uint_as_float(u << 16);
  return (float)__builtin_bit_cast(_Float16, (uint16_t)u);
}
__device__ __forceinline__ float mass_wave_sum(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
  return x;
}
__device__ __forceinline__ float mass_wave_max(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off));
  return x;
}

// A head without weight in row t (lse = -inf: no score of a valid key above -inf) adds nothing to
// the row's sums, whatever its scores are; the matrix kernel has added exp2(score + inf). The
// wave sums the selected keys of such a row again over the other heads. Rare, and here because
// a test of each weight in the matrix kernel costs it the registers of its fourth wave (5,496
// keys: the forward with the mass 373 -> 642 us).
__device__ __forceinline__ void mass_empty_heads(const MassGatherParams& p, int b, int64_t t, const int32_t* prow,
                                                 float* arow, int lane) {
  const float* lse = p.lse + ((int64_t)b * p.T + t) * p.H;
  bool empty = false;
  for (int h = lane; h < p.H; h += 64) empty |= lse[h] == -INFINITY;
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(empty) == 0ull, 1)) return;
#pragma unroll 1
  for (int j = lane; j < p.K; j += 64) {
    const int s = prow[j];
    if ((uint32_t)s >= (uint32_t)p.S) continue;
    float sum = 0.f;
#pragma unroll 1
    for (int h = 0; h < p.H; ++h) {
      if (lse[h] == -INFINITY) continue;
      const uint16_t* qr = p.q + b * p.qsb + t * p.qst + h * p.qsh;
      const uint16_t* kr = p.k + b * p.ksb + (int64_t)s * p.kss + h * p.ksh;
      float d = 0.f;
#pragma unroll 1
      for (int i = 0; i < 64; ++i) d = fmaf(in_to_float(p.in_fp16, qr[i]), in_to_float(p.in_fp16, kr[i]), d);
      sum += fexp2(fmaf(d, p.scale_log2, -lse[h] * kDLog2e));
    }
    arow[s] = sum;
  }
  __threadfence_block();  // the stores before the wave's own loads of the row
}

// One wave per query row: the selected values of its matrix row (0 for positions outside [0, S)),
// and with KL the row's loss from them.
template <int R, bool KL>
__global__ __launch_bounds__(256) void attn_mass_gather_kernel(const MassGatherParams p) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  const int grp = p.g0 + (int)(row / kMRows);
  const int b = grp / p.gpb;
  const int64_t t = (int64_t)(grp % p.gpb) * kMRows + row % kMRows;
  if (t >= p.T) return;  // whole wave; no barriers below
  const int32_t* prow = p.pos + b * p.psb + t * p.pst;
  float* arow = p.a + row * p.Spad;
  mass_empty_heads(p, b, t, prow, arow, lane);
  float* out = p.attn_sum + ((int64_t)b * p.T + t) * p.K;
  float av[R], zv[R];
  float sa = 0.f, mz = -INFINITY;
  int ps[R];
#pragma unroll
  for (int i = 0; i < R; ++i) ps[i] = i * 64 + lane < p.K ? prow[i * 64 + lane] : -1;
#pragma unroll
  for (int i = 0; i < R; ++i) av[i] = (uint32_t)ps[i] < (uint32_t)p.S ? arow[ps[i]] : 0.f;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int j = i * 64 + lane;
    zv[i] = -INFINITY;
    if (j < p.K) {
      out[j] = av[i];
      if constexpr (KL) {
        zv[i] = mass_load(p.logits_dt, p.logits, b * p.lsb + t * p.lst + j);
        sa += av[i];
        mz = fmaxf(mz, zv[i]);
      }
    }
  }
  if constexpr (KL) {
    sa = mass_wave_sum(sa);
    mz = mass_wave_max(mz);
    float se = 0.f;
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (i * 64 + lane < p.K) se += expf(zv[i] - mz);
    se = mass_wave_sum(se);
    const float lse = mz + logf(se);
    const float denom = sa + p.kl_eps;
    float loss = 0.f;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i * 64 + lane < p.K) {
        const float pj = av[i] / denom;
        loss += pj * (logf(pj + p.kl_eps) - (zv[i] - lse));
      }
    }
    loss = mass_wave_sum(loss);
    if (lane == 0) p.row_loss[(int64_t)b * p.T + t] = loss;
  }
}

template <bool KL>
void launch_gather(const MassGatherParams& g, hipStream_t st) {
  const dim3 grid((unsigned)(g.ngroup * (kMRows / 4)));
  if (g.K <= 64)
    hipLaunchKernelGGL((attn_mass_gather_kernel<1, KL>), grid, dim3(256), 0, st, g);
  else if (g.K <= 256)
    hipLaunchKernelGGL((attn_mass_gather_kernel<4, KL>), grid, dim3(256), 0, st, g);
  else if (g.K <= 512)
    hipLaunchKernelGGL((attn_mass_gather_kernel<8, KL>), grid, dim3(256), 0, st, g);
  else
    hipLaunchKernelGGL((attn_mass_gather_kernel<16, KL>), grid, dim3(256), 0, st, g);
}

// Groups of kMRows queries per chunk: those of all batch elements in one order, so that a chunk of
// several small elements is one launch, their matrix within kMChunkBytes (one group at least).
struct MassChunks {
  int64_t gpb, groups, chunk;  // groups per batch element, in all, and per chunk
  int64_t spad;
};
MassChunks mass_chunks(int64_t B, int64_t T, int64_t S) {
  MassChunks c;
  c.spad = (S + kMKeys - 1) / kMKeys * kMKeys;
  c.gpb = (T + kMRows - 1) / kMRows;
  c.groups = B * c.gpb;
  const int64_t fit = kMChunkBytes / (c.spad * 4 * kMRows);
  c.chunk = fit < 1 ? 1 : fit < c.groups ? fit : c.groups;
  return c;
}

}  // namespace
}  // namespace gw

extern "C" size_t gw_sparse_attn_mass_workspace_size(int64_t B, int64_t T, int64_t S, int64_t H, int64_t D, int64_t K) {
  if (B <= 0 || T <= 0 || S <= 0 || H <= 0 || K <= 0 || D != 64) return 0;
  const gw::MassChunks c = gw::mass_chunks(B, T, S);
  return (size_t)(c.chunk * gw::kMRows * c.spad * 4);
}

extern "C" int gw_sparse_attn_mass(int dtype, const void* q, const int64_t* q_strides, const void* k,
                                   const int64_t* k_strides, const int32_t* kv_pos, int64_t pos_stride_b,
                                   int64_t pos_stride_t, const float* lse, float* attn_sum, int64_t B, int64_t T,
                                   int64_t S, int64_t H, int64_t D, int64_t K, float softmax_scale,
                                   const void* logits, int logits_dtype, int64_t logits_stride_b,
                                   int64_t logits_stride_t, float eps, float* row_loss, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  using namespace gw;
  clear_error();
  GW_CHECK_ARG(dtype == GW_DTYPE_BF16 || dtype == GW_DTYPE_FP16, "unsupported dtype code %d", dtype);
  GW_CHECK_ARG(B >= 0 && T >= 0 && S >= 0 && H >= 1 && K >= 0, "invalid sizes B=%lld T=%lld S=%lld H=%lld K=%lld",
               (long long)B, (long long)T, (long long)S, (long long)H, (long long)K);
  if (D != 64) return set_error(GW_ERR_UNSUPPORTED, "the mass pass needs head dim 64, got %lld", (long long)D);
  if (K > kMassMaxK)
    return set_error(GW_ERR_UNSUPPORTED, "the mass pass takes K <= %d, got %lld", kMassMaxK, (long long)K);
  if (B == 0 || T == 0) return GW_OK;
  GW_CHECK_ARG(K >= 1 && S >= 1, "kv_positions must have at least one candidate and S >= 1");
  GW_CHECK_ARG(q && k && kv_pos && lse && attn_sum && q_strides && k_strides, "null pointer");
  GW_CHECK_ARG(aligned16(q) && aligned16(k), "q and k must be 16-byte aligned");
  for (int i = 0; i < 3; ++i)
    GW_CHECK_ARG(q_strides[i] % 8 == 0 && k_strides[i] % 8 == 0, "b/t/h strides must be multiples of 8 elements");
  if (k_strides[1] < 0 || k_strides[1] >= (1ll << 23) || q_strides[1] < 0 || q_strides[1] >= (1ll << 23))
    return set_error(GW_ERR_UNSUPPORTED, "the mass pass needs Q and K token strides below 2^23 elements, got %lld, %lld",
                     (long long)q_strides[1], (long long)k_strides[1]);
  GW_CHECK_ARG(B <= 65535 && T < (1ll << 31) - 65536 && S < (1ll << 30) && B * ((T + kMRows - 1) / kMRows) < (1ll << 31),
               "size exceeds the grid range");
  const bool kl = logits != nullptr;
  if (kl) {
    GW_CHECK_ARG(row_loss != nullptr, "null row_loss pointer");
    GW_CHECK_ARG(logits_dtype == GW_DTYPE_BF16 || logits_dtype == GW_DTYPE_FP16 || logits_dtype == GW_DTYPE_FP32,
                 "unsupported logits dtype code %d", logits_dtype);
    GW_CHECK_ARG(eps >= 0.f, "eps must be non-negative, got %g", (double)eps);
  }
  const size_t need = gw_sparse_attn_mass_workspace_size(B, T, S, H, D, K);
  GW_CHECK_ARG(workspace != nullptr && workspace_bytes >= need && aligned16(workspace),
               "the mass pass needs a 16-byte aligned %zu-byte workspace, got %zu", need, workspace_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const MassChunks c = mass_chunks(B, T, S);
  MassParams p;
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k);
  p.lse = lse;
  p.a = static_cast<float*>(workspace);
  p.qsb = q_strides[0]; p.qst = q_strides[1]; p.qsh = q_strides[2];
  p.ksb = k_strides[0]; p.kss = k_strides[1]; p.ksh = k_strides[2];
  p.T = (int)T;
  p.S = (int)S;
  p.Spad = (int)c.spad;
  p.gpb = (int)c.gpb;
  p.H = (int)H;
  p.scale_log2 = softmax_scale * kDLog2e;
  MassGatherParams g;
  g.q = p.q;
  g.k = p.k;
  g.lse = lse;
  g.qsb = p.qsb; g.qst = p.qst; g.qsh = p.qsh;
  g.ksb = p.ksb; g.kss = p.kss; g.ksh = p.ksh;
  g.in_fp16 = dtype == GW_DTYPE_FP16 ? 1 : 0;
  g.H = p.H;
  g.scale_log2 = p.scale_log2;
  g.pos = kv_pos;
  g.psb = pos_stride_b;
  g.pst = pos_stride_t;
  g.a = p.a;
  g.attn_sum = attn_sum;
  g.logits = logits;
  g.logits_dt = logits_dtype;
  g.lsb = logits_stride_b;
  g.lst = logits_stride_t;
  g.kl_eps = eps;
  g.row_loss = row_loss;
  g.T = p.T;
  g.S = p.S;
  g.Spad = p.Spad;
  g.gpb = p.gpb;
  g.K = (int)K;
  for (int64_t g0 = 0; g0 < c.groups; g0 += c.chunk) {
    p.g0 = g.g0 = (int)g0;
    p.ngroup = g.ngroup = (int)(c.groups - g0 < c.chunk ? c.groups - g0 : c.chunk);
    const int64_t wgs = (int64_t)p.ngroup * (p.Spad / kMKeys);
    if (dtype == GW_DTYPE_BF16)
      hipLaunchKernelGGL((attn_mass_kernel<BF16>), dim3((unsigned)wgs), dim3(kMWaves * 64), 0, st, p);
    else
      hipLaunchKernelGGL((attn_mass_kernel<FP16>), dim3((unsigned)wgs), dim3(kMWaves * 64), 0, st, p);
    GW_HIP_LAUNCH_CHECK("attn_mass_kernel launch");
    if (kl)
      launch_gather<true>(g, st);
    else
      launch_gather<false>(g, st);
    GW_HIP_LAUNCH_CHECK("attn_mass_gather_kernel launch");
  }
  return GW_OK;
}
