// Kronecker gradient projection (GradProjLoRA), gfx950.
//
//   out[b] = scale * sum_t (L g_bt)(R a_bt)^T        L: [kL, n_g], R: [kR, n_a]
//
// Projections with more than 64 rows on a side run as several launches over 64-row slices of
// the projection matrices, each writing its block of the [kL, kR] partials.
//
// One workgroup takes one sample and a chunk of 32 tokens; its 8 waves take interleaved
// pieces of 128 bytes of every token row.  A wave streams its pieces of the G and A rows straight
// from HBM into MFMA operands (v_mfma_f32_16x16x32_bf16 / v_mfma_f32_16x16x4f32) against the
// projection rows (small, L2-resident), the next piece's rows in flight while the current one is
// multiplied, so G and A are read exactly once.  The wave shares (fp32) are summed in LDS, the
// chunk's outer-product sum is formed there with fp32 MFMAs, and the per-chunk partials are
// reduced per sample in a fixed order.  Bound by HBM: 32 x 1024 tokens of 1024 + 4096
// bf16 features at 16 x 16 projection rows take 67 us (5.0 TB/s, a 1 GiB copy 5.1; 75 us when
// all waves loaded, multiplied and waited in step), of 1024 + 3072 at 39 x 13 54 us (113 us with
// both sides padded to 64 rows and 133 KiB of LDS).  Rows off 16-byte boundaries are loaded 16
// bytes at a time too: of 1023 + 4095 features at 20 x 20 221 us (element by element 435, in
// chunks of 64 tokens 257), at 40 x 13 200 (452, 265).
//
// 16x16 MFMA layout: lane l supplies row (l % 16) of A and column (l % 16) of B with its
// k-slice chosen by l / 16; result element e of lane l is C[4*(l/16) + e][l % 16].

#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "gs_common.h"

namespace gs {

typedef __bf16 bf16x8p_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int PJ_TOK = 32;      // tokens per workgroup
constexpr int PJ_TG = PJ_TOK / 16;  // its 16-token MFMA row groups
constexpr int PJ_THREADS = 512;
constexpr int PJ_WAVES = PJ_THREADS / 64;
constexpr int PJ_KMAX = 64;     // projection rows per side of one launch

struct PjBF16 {
  using E = uint16_t;
  static constexpr int VEC = 8;    // elements per 16-byte lane load
  static constexpr int KSTEP = 32; // k covered by one MFMA across the 4 lane groups
  static constexpr int SUB = 1;    // MFMAs per lane load
  __device__ static __forceinline__ void mma(f32x4_t& c, const uint4& a, const uint4& b, int) {
    bf16x8p_t av, bv;
    __builtin_memcpy(&av, &a, 16);
    __builtin_memcpy(&bv, &b, 16);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, c, 0, 0, 0);
  }
};

struct PjF32 {
  using E = float;
  static constexpr int VEC = 4;
  static constexpr int KSTEP = 16;  // 4 MFMAs (k = 4 each) per 16-byte lane load
  static constexpr int SUB = 4;
  __device__ static __forceinline__ void mma(f32x4_t& c, const uint4& a, const uint4& b, int s) {
    const float* af = reinterpret_cast<const float*>(&a);
    const float* bf = reinterpret_cast<const float*>(&b);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[s], bf[s], c, 0, 0, 0);
  }
};

// One side's partial projections over this wave's share of the features of the chunk's
// PJ_TOK token rows: acc[tg][nb][e] = sum_f P[16 nb + l%16][f] * row(16 tg + 4 (l/16) + e)[f].
// A wave takes pieces of 2 KSTEP features (128 bytes of a row), lane group g the g-th 32 bytes
// of them, in two loads, so that a wave uses whole cache lines; every projection fragment
// serves the PJ_TG row groups.  `rows` point at valid rows (a token past the end reads another
// row and is dropped by the caller: an operand row reaches only its own result row), and rows of
// P past kP repeat its last row (columns nobody reads).  VEC false: rows or projections are
// not 16-byte aligned; they are loaded 16 bytes at a time all the same, a row's last partial 16
// element by element.
template <class Tr, int NB, bool VEC>
__device__ __forceinline__ void project_rows(const typename Tr::E* const (&rows)[PJ_TG],
                                             const typename Tr::E* P, int64_t n, int64_t kP,
                                             f32x4_t (&acc)[PJ_TG][NB]) {
  using E = typename Tr::E;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t koff = (lane >> 4) * 2 * Tr::VEC;  // this lane group's 32 bytes of a piece
  const E* prow[NB];  // this lane's projection row in each 16-row block
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int64_t r = 16 * nb + (lane & 15);
    prow[nb] = P + (r < kP ? r : kP - 1) * n;
  }
  constexpr int64_t PIECE = 2 * Tr::KSTEP, STEP = PJ_WAVES * PIECE;
  auto fetch = [&](const E* row, int64_t k, bool whole) -> uint4 {
    if constexpr (VEC) {
      // Past the end (VEC divides n, so a chunk is wholly inside or outside): a valid address,
      // then zeros.
      uint4 v = *reinterpret_cast<const uint4*>(row + (whole || k < n ? k : 0));
      if (!whole && k >= n) v = make_uint4(0u, 0u, 0u, 0u);
      return v;
    } else {
      union { uint4 v; E e[Tr::VEC]; } u;
      if (whole || k + Tr::VEC <= n) {
        __builtin_memcpy(&u.v, row + k, sizeof(u.v));
      } else {
#pragma unroll
        for (int i = 0; i < Tr::VEC; ++i) u.e[i] = k + i < n ? row[k + i] : E(0);
      }
      return u.v;
    }
  };
  auto load_rows = [&](uint4 (&a)[2][PJ_TG], int64_t f0, bool whole) {
#pragma unroll
    for (int tg = 0; tg < PJ_TG; ++tg)
#pragma unroll
      for (int u = 0; u < 2; ++u) a[u][tg] = fetch(rows[tg], f0 + koff + u * Tr::VEC, whole);
  };
  auto compute = [&](const uint4 (&a)[2][PJ_TG], int64_t f0, bool whole) {
    uint4 b[2][NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int u = 0; u < 2; ++u) b[u][nb] = fetch(prow[nb], f0 + koff + u * Tr::VEC, whole);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int tg = 0; tg < PJ_TG; ++tg)
#pragma unroll
          for (int s = 0; s < Tr::SUB; ++s) Tr::mma(acc[tg][nb], a[u][tg], b[u][nb], s);
  };
  // Whole steps first, then the wave's piece of the last, partial one; each piece is loaded
  // before its predecessor is used.  The whole steps start at a different one in every
  // workgroup: in step, all of them would read the same columns of rows a power of two apart,
  // which few HBM channels serve (1024 + 4096 features: 75 us
  // in step, 67 us so).
  const int64_t whole = n / STEP, f0 = wid * PIECE, tail = f0 + whole * STEP;
  const bool has_tail = tail < n;
  const int64_t rot = whole > 0 ? (blockIdx.x + blockIdx.y) % whole : 0;
  auto at = [&](int64_t i) {
    const int64_t j = i + rot;
    return f0 + (j < whole ? j : j - whole) * STEP;
  };
  uint4 a0[2][PJ_TG], a1[2][PJ_TG];
  auto advance = [&]() {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int tg = 0; tg < PJ_TG; ++tg) a0[u][tg] = a1[u][tg];
  };
  if (whole > 0)
    load_rows(a0, at(0), true);
  else if (has_tail)
    load_rows(a0, tail, false);
  int64_t i = 0;
  for (; i + 2 < whole; i += 2) {
    load_rows(a1, at(i + 1), true);
    compute(a0, at(i), true);
    load_rows(a0, at(i + 2), true);
    compute(a1, at(i + 1), true);
  }
  for (; i < whole; ++i) {  // the last one or two
    if (i + 1 < whole)
      load_rows(a1, at(i + 1), true);
    else if (has_tail)
      load_rows(a1, tail, false);
    compute(a0, at(i), true);
    advance();
  }
  if (has_tail) compute(a0, tail, false);
}

// Where a launch writes: its [kL, kR] block of the per-(sample, chunk) partials
// part[(b * chunks + c) * kl_tot * kr_tot + (l0 + p) * kr_tot + r0 + q].
struct PjSlice {
  int64_t kl_tot, kr_tot, l0, r0;
};

// GATHER: the input side is an embedding, whose "projected input" for token id x is column
// x of P_i, i.e. row x of R = P_i^T ([vocab, ldr], this launch's kR columns); `ids` replaces A.
// NL, NR: 16-row projection blocks of the two sides (kL <= 16 NL, kR <= 16 NR); VEC: 16-byte
// aligned rows and projections on both sides.
template <class Tr, bool GATHER, int NL, int NR, bool VEC>
__global__ void __launch_bounds__(PJ_THREADS, 4) kron_proj_kernel(
    const typename Tr::E* __restrict__ A, const int64_t* __restrict__ ids, int64_t vocab,
    const typename Tr::E* __restrict__ G, int64_t T, int64_t n_a, int64_t n_g,
    const typename Tr::E* __restrict__ R, const typename Tr::E* __restrict__ L, int64_t kR,
    int64_t kL, int64_t ldr, int64_t chunks, PjSlice sl, float* __restrict__ part) {
  using E = typename Tr::E;
  constexpr int TOK = PJ_TOK, TG = PJ_TG, LD = TOK + 4;  // LDS rows: one projection row, its tokens
  __shared__ __attribute__((aligned(16))) float slice[PJ_WAVES][16][LD];  // one 16-row block
  __shared__ float fin[(NL + NR) * 16][LD];   // the sums: L's projections, then R's
  const int64_t b = blockIdx.y, c = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t t0 = c * TOK;
  const int nvalid = static_cast<int>(T - t0 < TOK ? T - t0 : TOK);
  // Sums a block's wave shares in wave order into fin[row0 + 0..15]; tokens past the end get 0.
  auto combine = [&](const f32x4_t (&acc)[TG], int row0) {
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
      *reinterpret_cast<f32x4_t*>(&slice[wid][lane & 15][tg * 16 + 4 * (lane >> 4)]) = acc[tg];
    __syncthreads();
    for (int x = threadIdx.x; x < 16 * TOK; x += PJ_THREADS) {
      const int k = x / TOK, tok = x % TOK;
      float v = slice[0][k][tok];
#pragma unroll
      for (int w = 1; w < PJ_WAVES; ++w) v += slice[w][k][tok];
      fin[row0 + k][tok] = tok < nvalid ? v : 0.f;
    }
    __syncthreads();
  };
  auto side = [&](const E* X, int64_t n, const E* P, int64_t kP, int row0, auto nbc) {
    constexpr int NB = decltype(nbc)::value;
    const E* rows[TG];
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) {
      const int t = tg * 16 + (lane & 15);  // this lane's operand row
      rows[tg] = X + (b * T + t0 + (t < nvalid ? t : 0)) * n;
    }
    f32x4_t acc[TG][NB];
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[tg][nb][e] = 0.f;
    project_rows<Tr, NB, VEC>(rows, P, n, kP, acc);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      f32x4_t one[TG];
#pragma unroll
      for (int tg = 0; tg < TG; ++tg) one[tg] = acc[tg][nb];
      combine(one, row0 + 16 * nb);
    }
  };
  side(G, n_g, L, kL, 0, std::integral_constant<int, NL>{});
  if constexpr (GATHER) {
    for (int x = threadIdx.x; x < 16 * NR * TOK; x += PJ_THREADS) {
      const int q = x % (16 * NR), tok = x / (16 * NR);
      float v = 0.f;
      if (tok < nvalid && q < kR) {
        const int64_t id = ids[b * T + t0 + tok];
        if (id >= 0 && id < vocab) v = to_f32<E>(R[id * ldr + q]);
      }
      fin[16 * NL + q][tok] = v;
    }
    __syncthreads();
  } else {
    side(A, n_a, R, kR, 16 * NL, std::integral_constant<int, NR>{});
  }
  // part[p][q] = sum over the tokens of fin[p][tok] fin[16 NL + q][tok]: 16 x 16 blocks by fp32
  // MFMAs, four tokens each.
  float* dst = part + (b * chunks + c) * sl.kl_tot * sl.kr_tot + sl.l0 * sl.kr_tot + sl.r0;
  for (int blk = wid; blk < NL * NR; blk += PJ_WAVES) {
    const int p0 = blk / NR * 16, q0 = blk % NR * 16;
    const float* lp = &fin[p0 + (lane & 15)][lane >> 4];
    const float* rp = &fin[16 * NL + q0 + (lane & 15)][lane >> 4];
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < TOK; t += 4)
      o = __builtin_amdgcn_mfma_f32_16x16x4f32(lp[t], rp[t], o, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t p = p0 + 4 * (lane >> 4) + e, q = q0 + (lane & 15);
      if (p < kL && q < kR) dst[p * sl.kr_tot + q] = o[e];
    }
  }
}

template <class OE>
__global__ void kron_reduce_kernel(const float* __restrict__ part, int64_t chunks, int64_t nout,
                                   float scale, OE* __restrict__ out) {
  const int64_t b = blockIdx.y;
  const int64_t o = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (o >= nout) return;
  // Four running sums over whole groups of eight chunks keep the loads in flight together.
  const float* src = part + b * chunks * nout + o;
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
  int64_t c = 0;
  for (; c + 8 <= chunks; c += 8, src += 8 * nout) {
    a0 += src[0] + src[4 * nout];
    a1 += src[nout] + src[5 * nout];
    a2 += src[2 * nout] + src[6 * nout];
    a3 += src[3 * nout] + src[7 * nout];
  }
  for (; c < chunks; ++c, src += nout) a0 += *src;
  const float s = ((a0 + a1) + (a2 + a3)) * scale;
  if constexpr (std::is_same<OE, float>::value) {
    out[b * nout + o] = s;
  } else if constexpr (std::is_same<OE, __half>::value) {
    out[b * nout + o] = __float2half(s);
  } else {
    out[b * nout + o] = f32_to_bf16(s);
  }
}

namespace {
int64_t pj_cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// One launch over rows [l0, l0 + kl) of L and [r0, r0 + kr) of R (each at most PJ_KMAX).
template <class Tr, bool GATHER>
int launch_pj_slice(const typename Tr::E* A, const int64_t* ids, int64_t vocab,
                    const typename Tr::E* G, int64_t B, int64_t T, int64_t n_a, int64_t n_g,
                    const typename Tr::E* R, const typename Tr::E* L, int64_t kr, int64_t kl,
                    int64_t ldr, int va, int vg, int vr, int vl, int64_t chunks,
                    PjSlice sl, float* part, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(chunks), static_cast<unsigned>(B));
  const bool vec = vg && vl && (GATHER || (va && vr));
  auto go = [&](auto nl, auto nr, auto v) {
    auto k = kron_proj_kernel<Tr, GATHER, decltype(nl)::value, decltype(nr)::value,
                              decltype(v)::value>;
    hipLaunchKernelGGL(k, grid, dim3(PJ_THREADS), 0, s, A, ids, vocab, G, T, n_a, n_g, R, L, kr,
                       kl, ldr, chunks, sl, part);
  };
  auto blocks = [](int64_t k, auto f) {  // f(the number of 16-row blocks of k rows)
    if (k <= 16) return f(std::integral_constant<int, 1>{});
    if (k <= 32) return f(std::integral_constant<int, 2>{});
    if (k <= 48) return f(std::integral_constant<int, 3>{});
    return f(std::integral_constant<int, 4>{});
  };
  auto with = [&](auto v) {
    blocks(kl, [&](auto nl) { blocks(kr, [&](auto nr) { go(nl, nr, v); }); });
  };
  vec ? with(std::true_type{}) : with(std::false_type{});
  return check_launch(GATHER ? "kron_proj_kernel(gather)" : "kron_proj_kernel");
}

// All slices of a [kL_tot, kR_tot] projection: L rows and R rows (or, gathering, R columns)
// in pieces of PJ_KMAX.
template <class Tr, bool GATHER>
int launch_pj(const void* A, const int64_t* ids, int64_t vocab, const void* G, int64_t B,
              int64_t T, int64_t n_a, int64_t n_g, const void* R, const void* L, int64_t kR,
              int64_t kL, int va, int vg, int vr, int vl, int64_t chunks,
              float* part, hipStream_t s) {
  using E = typename Tr::E;
  for (int64_t l0 = 0; l0 < kL; l0 += PJ_KMAX) {
    for (int64_t r0 = 0; r0 < kR; r0 += PJ_KMAX) {
      const int64_t kl = std::min<int64_t>(PJ_KMAX, kL - l0);
      const int64_t kr = std::min<int64_t>(PJ_KMAX, kR - r0);
      const E* Ls = static_cast<const E*>(L) + l0 * n_g;
      const E* Rs = GATHER ? static_cast<const E*>(R) + r0 : static_cast<const E*>(R) + r0 * n_a;
      const PjSlice sl{kL, kR, l0, r0};
      const int rc = launch_pj_slice<Tr, GATHER>(
          static_cast<const E*>(A), ids, vocab, static_cast<const E*>(G), B, T, n_a, n_g, Rs, Ls,
          kr, kl, GATHER ? kR : n_a, va, vg, vr, vl, chunks, sl, part, s);
      if (rc) return rc;
    }
  }
  return GS_OK;
}

// Fixed-order per-sample sum of the chunk partials, scaled and converted to the output type.
int kron_finish(const float* part, int64_t B, int64_t chunks, int64_t nout, float scale,
                void* out, int out_dtype, hipStream_t s) {
  const dim3 rg(static_cast<unsigned>(pj_cdiv(nout, 256)), static_cast<unsigned>(B));
  if (out_dtype == GS_DTYPE_F32)
    hipLaunchKernelGGL(kron_reduce_kernel<float>, rg, dim3(256), 0, s, part, chunks, nout, scale,
                       static_cast<float*>(out));
  else if (out_dtype == GS_DTYPE_F16)
    hipLaunchKernelGGL(kron_reduce_kernel<__half>, rg, dim3(256), 0, s, part, chunks, nout, scale,
                       static_cast<__half*>(out));
  else
    hipLaunchKernelGGL(kron_reduce_kernel<uint16_t>, rg, dim3(256), 0, s, part, chunks, nout,
                       scale, static_cast<uint16_t*>(out));
  return check_launch("kron_reduce_kernel");
}
}  // namespace

}  // namespace gs

using namespace gs;

extern "C" size_t gs_kron_proj_workspace(int64_t B, int64_t T, int64_t k_i, int64_t k_o) {
  if (B <= 0 || T <= 0 || k_i <= 0 || k_o <= 0) return 0;
  Sizer sz;
  sz.take<float>(B * pj_cdiv(T, PJ_TOK) * k_i * k_o);
  return sz.used + 256;
}

extern "C" int gs_kron_proj(const void* A, const void* G, int dtype, int64_t B, int64_t T,
                            int64_t n_a, int64_t n_g, const void* P_i, const void* P_o,
                            int p_dtype, int64_t k_i, int64_t k_o, int layout, float scale,
                            void* out, int out_dtype, void* workspace, size_t workspace_bytes,
                            void* stream) {
  if (dtype != GS_DTYPE_BF16 && dtype != GS_DTYPE_F32)
    return fail(GS_ERR_DTYPE, "gs_kron_proj: dtype must be bf16 or fp32");
  if (p_dtype != dtype)
    return fail(GS_ERR_DTYPE, "gs_kron_proj: projection dtype must equal the operand dtype");
  if (out_dtype != GS_DTYPE_F32 && out_dtype != GS_DTYPE_BF16 && out_dtype != GS_DTYPE_F16)
    return fail(GS_ERR_DTYPE, "gs_kron_proj: out_dtype must be fp32, bf16 or fp16");
  if (B <= 0 || T <= 0 || n_a <= 0 || n_g <= 0 || k_i <= 0 || k_o <= 0 || A == nullptr ||
      G == nullptr || P_i == nullptr || P_o == nullptr || out == nullptr)
    return fail(GS_ERR_INVALID, "gs_kron_proj: invalid arguments");
  if (layout != GS_PROJ_KO_KI && layout != GS_PROJ_KI_KO)
    return fail(GS_ERR_INVALID, "gs_kron_proj: invalid layout");
  // KO_KI: L = P_o (applied to G), R = P_i (applied to A).  KI_KO swaps the matrices.
  const void* L = layout == GS_PROJ_KO_KI ? P_o : P_i;
  const void* R = layout == GS_PROJ_KO_KI ? P_i : P_o;
  const int64_t kL = layout == GS_PROJ_KO_KI ? k_o : k_i;
  const int64_t kR = layout == GS_PROJ_KO_KI ? k_i : k_o;
  const int64_t chunks = pj_cdiv(T, PJ_TOK);
  if (workspace == nullptr || workspace_bytes < gs_kron_proj_workspace(B, T, k_i, k_o) - 256)
    return fail(GS_ERR_WORKSPACE, "gs_kron_proj: workspace too small");
  if (chunks > 2 * 65535 || B > 65535) return fail(GS_ERR_UNSUPPORTED, "gs_kron_proj: grid too large");
  Carver cv(workspace, workspace_bytes);
  float* part = cv.take<float>(B * chunks * kL * kR);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t esz = elem_size(dtype);
  const int va = al16(A) && (n_a * static_cast<int64_t>(esz)) % 16 == 0;
  const int vg = al16(G) && (n_g * static_cast<int64_t>(esz)) % 16 == 0;
  const int vr = al16(R) && (n_a * static_cast<int64_t>(esz)) % 16 == 0;
  const int vl = al16(L) && (n_g * static_cast<int64_t>(esz)) % 16 == 0;
  int rc = dtype == GS_DTYPE_BF16
               ? launch_pj<PjBF16, false>(A, nullptr, 0, G, B, T, n_a, n_g, R, L, kR, kL, va, vg,
                                          vr, vl, chunks, part, s)
               : launch_pj<PjF32, false>(A, nullptr, 0, G, B, T, n_a, n_g, R, L, kR, kL, va, vg,
                                         vr, vl, chunks, part, s);
  if (rc) return rc;
  return kron_finish(part, B, chunks, kL * kR, scale, out, out_dtype, s);
}

extern "C" int gs_kron_embed_proj(const int64_t* ids, const void* G, int dtype, int64_t B,
                                  int64_t T, int64_t n_g, const void* P_iT, const void* P_o,
                                  int p_dtype, int64_t vocab, int64_t k_i, int64_t k_o,
                                  float scale, void* out, int out_dtype, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  if (dtype != GS_DTYPE_BF16 && dtype != GS_DTYPE_F32)
    return fail(GS_ERR_DTYPE, "gs_kron_embed_proj: dtype must be bf16 or fp32");
  if (p_dtype != dtype)
    return fail(GS_ERR_DTYPE, "gs_kron_embed_proj: projection dtype must equal the grad dtype");
  if (out_dtype != GS_DTYPE_F32 && out_dtype != GS_DTYPE_BF16 && out_dtype != GS_DTYPE_F16)
    return fail(GS_ERR_DTYPE, "gs_kron_embed_proj: out_dtype must be fp32, bf16 or fp16");
  if (B <= 0 || T <= 0 || n_g <= 0 || vocab <= 0 || k_i <= 0 || k_o <= 0 || ids == nullptr ||
      G == nullptr || P_iT == nullptr || P_o == nullptr || out == nullptr)
    return fail(GS_ERR_INVALID, "gs_kron_embed_proj: invalid arguments");
  const int64_t chunks = pj_cdiv(T, PJ_TOK);
  if (workspace == nullptr || workspace_bytes < gs_kron_proj_workspace(B, T, k_i, k_o) - 256)
    return fail(GS_ERR_WORKSPACE, "gs_kron_embed_proj: workspace too small");
  if (chunks > 2 * 65535 || B > 65535)
    return fail(GS_ERR_UNSUPPORTED, "gs_kron_embed_proj: grid too large");
  Carver cv(workspace, workspace_bytes);
  float* part = cv.take<float>(B * chunks * k_o * k_i);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t esz = elem_size(dtype);
  const int vg = al16(G) && (n_g * static_cast<int64_t>(esz)) % 16 == 0;
  const int vl = al16(P_o) && (n_g * static_cast<int64_t>(esz)) % 16 == 0;
  int rc = dtype == GS_DTYPE_BF16
               ? launch_pj<PjBF16, true>(nullptr, ids, vocab, G, B, T, 0, n_g, P_iT, P_o, k_i,
                                         k_o, 0, vg, 0, vl, chunks, part, s)
               : launch_pj<PjF32, true>(nullptr, ids, vocab, G, B, T, 0, n_g, P_iT, P_o, k_i,
                                        k_o, 0, vg, 0, vl, chunks, part, s);
  if (rc) return rc;
  return kron_finish(part, B, chunks, k_o * k_i, scale, out, out_dtype, s);
}
