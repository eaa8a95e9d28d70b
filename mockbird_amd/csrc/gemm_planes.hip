// Prefill-sized projections on operands that are already bf16 planes (gfx950):
//   C[M][N] (=, +=) epi(A[M][K] W[K][N] + bias[N])
// as bf16 products of A's and W's planes summed in fp32 (planes.h).  The
// kernels that produce A write its planes -- the LayerNorm (k_planes), the
// prompt attention, and this kernel's own GELU epilogue -- in the order the
// matrix unit takes them, so the k loop is loads to LDS, LDS reads and MFMAs
// alone: nothing is converted once per column tile.
//
// A planes operand of K columns (a multiple of 32) and M rows, rows in blocks
// of 16: per (row block, 32-deep k block, plane) 1 KB, lane l's 16 bytes
// holding A[16 rb + (l & 15)][32 kb + 8 (l >> 4) .. + 7] -- one MFMA operand.
// W planes likewise per 64-column strip and k block: [column block j][plane]
// [lane], lane l holding W[32 kb + 8 (l >> 4) ..][64 s + 4 (l & 15) + j]
// (launch_split_w / launch_split_w1).
#include <type_traits>
#include <utility>

#include "gemm_epi.h"
#include "kv_types.h"
#include "lds_dma.h"
#include "mb_internal.h"
#include "planes.h"

namespace mb {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// The planes of (x - mean) rstd [* gamma] of each 768-wide row: a workgroup
// takes 16 rows, thread (row, c) the 8-column chunks c, c + 16, ...  A wave's
// loads are whole 128-byte row pieces, its stores 1 KB blocks.  Bound: HBM (8
// or 10 bytes per element).
template <int P>
__global__ __launch_bounds__(256) void k_ln_planes(const float* __restrict__ x, int64_t ldx, int M,
                                                   const float* __restrict__ gamma,
                                                   uint4* __restrict__ out) {
  constexpr int CH = D / 128;
  __shared__ float red[2][4][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = threadIdx.x & 15, c0 = threadIdx.x >> 4;
  const int64_t grow = (int64_t)blockIdx.x * 16 + row;
  float v[CH][8];
  const float* src = x + min(grow, (int64_t)M - 1) * ldx + 8 * c0;  // rows past M repeat the last one
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const float4 a = *(const float4*)(src + 128 * i), b = *(const float4*)(src + 128 * i + 4);
    v[i][0] = a.x; v[i][1] = a.y; v[i][2] = a.z; v[i][3] = a.w;
    v[i][4] = b.x; v[i][5] = b.y; v[i][6] = b.z; v[i][7] = b.w;
  }
  // a row's 16 threads: 4 lanes of each wave (lanes row + 16 k), 4 waves
  auto row_sum = [&](int k, float s) {
    s = col_sum(s);
    if (lane < 16) red[k][wave][lane] = s;
    __syncthreads();
    return (red[k][0][row] + red[k][1][row]) + (red[k][2][row] + red[k][3][row]);
  };
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < CH; i++)
#pragma unroll
    for (int e = 0; e < 8; e++) s += v[i][e];
  const float mean = row_sum(0, s) * (1.f / D);
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < CH; i++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      v[i][e] -= mean;
      q = fmaf(v[i][e], v[i][e], q);
    }
  const float inv = 1.f / sqrtf(row_sum(1, q) * (1.f / D) + 1e-5f);
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const int c = c0 + 16 * i;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      v[i][e] *= inv;
      if (gamma) v[i][e] *= gamma[8 * c + e];
    }
    uint2 lo[P], hi[P];
    split4<P>(make_float4(v[i][0], v[i][1], v[i][2], v[i][3]), lo);
    split4<P>(make_float4(v[i][4], v[i][5], v[i][6], v[i][7]), hi);
#pragma unroll
    for (int p = 0; p < P; p++)
      out[plane_chunk(grow, c, D / 32, P, p)] = make_uint4(lo[p].x, lo[p].y, hi[p].x, hi[p].y);
  }
}

// A workgroup owns 16 MI WM rows x 64 WN columns over all of k: wave (wm, wn)
// MI row blocks and strip wn.  Per 32-deep k block the operands' 1 KB pieces
// reach LDS by the load unit, dealt evenly over the waves, D stages deep; one
// barrier per block publishes a stage and frees the one the next loads
// overwrite.  Every LDS read is 16 bytes per lane in lane order.  lnd (may be
// null): a folded LayerNorm's d, added before the bias.  PO > 0: the result's
// PO planes go to Op (the next projection's operand) instead of Cm.
template <int PA, int PW, int MI, int WM, int WN, int D, int EPI, int PO, int OCC>
__global__ __launch_bounds__(64 * WM * WN, OCC) void k_gemm_planes(
    const uint4* __restrict__ Ap, const uint4* __restrict__ Wx, int N, int nkb,
    const float* __restrict__ lnd, const float* __restrict__ bias, float* __restrict__ Cm,
    int64_t ldc, int M, uint4* __restrict__ Op) {
  constexpr int NW = WM * WN;
  constexpr int AP = MI * WM * PA, WP = WN * 4 * PW;  // 1 KB pieces per 32-deep block
  static_assert((AP + WP) % NW == 0, "the pieces divide over the waves");
  constexpr int PPW = (AP + WP) / NW;
  constexpr int STAGE = (AP + WP) * 1024;
  static_assert(D >= 2 && (D - 2) * PPW <= 63, "vmcnt holds at most 63 loads");
  __shared__ __align__(16) char lds[D * STAGE];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int l16 = lane & 15, r = lane >> 4;
  const int rb0 = blockIdx.y * (MI * WM), strip0 = blockIdx.x * WN;
  const int nrb = (M + 15) >> 4;

  // Three planes: the products of high planes are summed apart from the five
  // small ones, so the large sum is rounded once per block, not six times.
  constexpr bool APART = PA == 3 && PW == 3;
  f32x4_t acc[MI][4], low[APART ? MI : 1][4];
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (APART) low[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

  // this wave's pieces of block 0, and how far apart their blocks are
  const char* base[PPW];
  bool isa[PPW];
#pragma unroll
  for (int t = 0; t < PPW; t++) {
    const int pi = wave * PPW + t;
    isa[t] = pi < AP;
    if (pi < AP) {
      const int rb = min(rb0 + pi / PA, nrb - 1);  // past the last rows: its block again, never stored
      base[t] = (const char*)Ap + ((int64_t)rb * nkb * PA + pi % PA) * 1024;
    } else {
      const int q = pi - AP, s = q / (4 * PW), qq = q % (4 * PW);
      base[t] = (const char*)Wx + ((int64_t)(strip0 + s) * nkb * (4 * PW) + qq) * 1024;
    }
  }
  const uint32_t voff = lane * 16;
  auto issue = [&](int st, int kb) {
    char* const sp = lds + st * STAGE + wave * (PPW * 1024);
#pragma unroll
    for (int t = 0; t < PPW; t++)
      dma16(base[t] + (int64_t)kb * (isa[t] ? PA * 1024 : 4 * PW * 1024), voff, lds_addr(sp + t * 1024));
  };
  auto mma = [&](int st) {
    const char* const sp = lds + st * STAGE;
    bf16x8_t a[MI][PA], w[4][PW];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int p = 0; p < PW; p++)
        w[j][p] = *(const bf16x8_t*)(sp + (AP + wn * 4 * PW + PW * j + p) * 1024 + 16 * lane);
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int p = 0; p < PA; p++)
        a[i][p] = *(const bf16x8_t*)(sp + ((wm * MI + i) * PA + p) * 1024 + 16 * lane);
    plane_products<PA, PW>([&](auto pa, auto pw) {
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < MI; i++) {
          f32x4_t& c = APART && decltype(pa)::value + decltype(pw)::value > 0 ? low[i][j] : acc[i][j];
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][pa], w[j][pw], c, 0, 0, 0);
        }
    });
  };
#pragma unroll
  for (int s = 0; s < D - 1; s++) issue(s, min(s, nkb - 1));
  int st = 0, sn = D - 1;
  for (int c = 0; c < nkb; c++) {
    MB_WAIT_VMCNT64((D - 2) * PPW);
    __syncthreads();
    issue(sn, min(c + D - 1, nkb - 1));  // past the end: reloads, never read
    mma(st);
    st = st + 1 == D ? 0 : st + 1;
    sn = sn + 1 == D ? 0 : sn + 1;
  }
  MB_WAIT_VMCNT(0);

  if constexpr (APART) {
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] += low[i][j];
  }
  const int n = (strip0 + wn) * 64 + 4 * l16;
  const float4 dv = lnd ? *(const float4*)(lnd + n) : make_float4(0.f, 0.f, 0.f, 0.f);
  auto value = [&](int i, int e, const float* cp) {
    return epilogue4<EPI>(make_float4(acc[i][0][e] + dv.x, acc[i][1][e] + dv.y, acc[i][2][e] + dv.z,
                                      acc[i][3][e] + dv.w),
                          bias, n, cp);
  };
  if constexpr (PO == 0) {
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int row = (rb0 + wm * MI + i) * 16 + 4 * r + e;
        if (row >= M) continue;
        float* cp = Cm + (int64_t)row * ldc + n;
        *(float4*)cp = value(i, e, cp);
      }
  } else {
    // A lane holds rows 4r .. 4r + 3 of 4 columns, half a 16-byte chunk each;
    // the even lane of a pair takes the whole chunks of the first two rows,
    // the odd one those of the last two (8-byte stores took fc_in at 11.7k
    // rows 157 us, see launch_gemm_planes).
    const bool odd = l16 & 1;
#pragma unroll
    for (int i = 0; i < MI; i++) {
      const int rb = rb0 + wm * MI + i;
      if (rb >= nrb) break;  // uniform; rows past M in the last block are stored, never used
#pragma unroll
      for (int e = 0; e < 2; e++) {
        uint2 lo[PO], hi[PO];
        split4<PO>(value(i, e, nullptr), lo);
        split4<PO>(value(i, e + 2, nullptr), hi);
        uint4* op = Op + plane_chunk((int64_t)rb * 16 + 4 * r + e + (odd ? 2 : 0), n >> 3, N >> 5, PO, 0);
#pragma unroll
        for (int p = 0; p < PO; p++) {
          const uint2 mine = odd ? hi[p] : lo[p], send = odd ? lo[p] : hi[p];
          uint2 got;  // the neighbour lane's half (quad permute 1, 0, 3, 2)
          got.x = __builtin_amdgcn_mov_dpp(send.x, 0xB1, 0xF, 0xF, true);
          got.y = __builtin_amdgcn_mov_dpp(send.y, 0xB1, 0xF, 0xF, true);
          op[p * 64] = odd ? make_uint4(got.x, got.y, mine.x, mine.y) : make_uint4(mine.x, mine.y, got.x, got.y);
        }
      }
    }
  }
}

// The three planes of a column-block-major W [N / 64][K][64] (launch_tile_w,
// launch_fold_ln) in the operand order above: one thread per 16-byte piece of
// a plane triple (strip, k block, column block j, lane).
__global__ __launch_bounds__(256) void k_split_w3(const float* __restrict__ Wt, int K, int N,
                                                  uint4* __restrict__ Wx) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int nkb = K / 32;
  if (u >= (int64_t)(N / 64) * nkb * 256) return;
  const int lane = (int)(u & 63), j = (int)((u >> 6) & 3);
  const int64_t blk = u >> 8, strip = blk / nkb;
  const int64_t k = (blk % nkb) * 32 + 8 * (lane >> 4);
  const float* src = Wt + strip * K * 64 + k * 64 + 4 * (lane & 15) + j;
  float v[8];
#pragma unroll
  for (int t = 0; t < 8; t++) v[t] = src[t * 64];
  const Planes w = split3<true>(v);
#pragma unroll
  for (int p = 0; p < 3; p++) Wx[(blk * 4 + j) * 192 + p * 64 + lane] = __builtin_bit_cast(uint4, w.p[p]);
}

int launch_split_w3(mb_ctx* ctx, const float* Wt, int K, int N, void* Wx) {
  if (N % 64 || K % 32)
    return fail(ctx, MB_ERR_ARG, "weight planes need N %% 64 == 0 and K %% 32 == 0 (K %d N %d)", K, N);
  const int64_t n = (int64_t)(N / 64) * (K / 32) * 256;
  hipLaunchKernelGGL(k_split_w3, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, Wt, K, N,
                     (uint4*)Wx);
  MB_HIP(ctx, hipGetLastError());
  return MB_OK;
}

int launch_ln_planes(mb_ctx* ctx, int planes, const float* x, int64_t ldx, int M,
                     const float* gamma, void* out) {
  if (M <= 0) return MB_OK;
  hipLaunchKernelGGL(planes == 3 ? k_ln_planes<3> : k_ln_planes<2>, dim3((unsigned)((M + 15) / 16)),
                     dim3(256), 0, ctx->stream, x, ldx, M, gamma, (uint4*)out);
  MB_HIP(ctx, hipGetLastError());
  return MB_OK;
}

// 64 x 128 tiles, two stages, three workgroups per CU (two planes; two with
// three).  What bounds it is LDS traffic against the matrix unit: per k block
// a wave reads 12 KB (18) for 24 MFMAs (48), and the loads write 24 KB (36)
// per workgroup.  In a prompt pass of 11.7k rows c_attn / c_proj / fc_in /
// fc_out take 121 / 70 / 162 / 166 us with two planes (1.03 / 0.60 / 1.02 /
// 1.0 PFLOP/s of bf16 products; a library's 8192^3 product reaches 1.2), which
// k_gemm_xt, splitting A's rows again for every column tile, does in 154 / 69
// / 223 / 181; with three planes 214 / 105 / 303 / 312 us against the fp32 MFMA
// kernel's 435 / 209 / 555 / 684.  Other tiles, alone at that size (two planes,
// c_attn / c_proj; this one 114 / 50 us): 128 x 128 129 / 65, 256 x 128 on 8
// waves 122 / 73, 192 x 128 109 / 58, 256 x 256 on 16 waves 106 / 56 us but 98
// against 79 at 8192 rows (a part-full last round); three stages at two
// workgroups per CU 123 / 58.
int launch_gemm_planes(mb_ctx* ctx, int pa, int pw, int epi, const void* Ap, const void* Wx, int N,
                       int K, const float* lnd, const float* bias, float* Cm, int64_t ldc, int M,
                       void* out_planes) {
  if (M <= 0) return MB_OK;
  if (N % 128 || K % 32 || ldc % 4 || ((uintptr_t)Cm & 15) || ((uintptr_t)bias & 15) ||
      ((uintptr_t)lnd & 15))
    return fail(ctx, MB_ERR_ARG, "plane gemm shape/alignment unsupported (M %d N %d K %d)", M, N, K);
  if (out_planes ? epi != EPI_GELU : epi != EPI_STORE && epi != EPI_ADD)
    return fail(ctx, MB_ERR_ARG, "plane gemm has no such epilogue (%d)", epi);
  using std::integral_constant;
  auto go = [&](auto pa_, auto pw_, auto e_, auto po_) {
    constexpr int PA = decltype(pa_)::value, PW = decltype(pw_)::value;
    constexpr int MI = 2, WM = 2, WN = 2;
    hipLaunchKernelGGL((k_gemm_planes<PA, PW, MI, WM, WN, 2, decltype(e_)::value,
                                      decltype(po_)::value ? PA : 0, PA == 3 ? 2 : 3>),
                       dim3((unsigned)(N / (64 * WN)), (unsigned)((M + 16 * MI * WM - 1) / (16 * MI * WM))),
                       dim3(64 * WM * WN), 0, ctx->stream, (const uint4*)Ap, (const uint4*)Wx, N, K / 32,
                       lnd, bias, Cm, ldc, M, (uint4*)out_planes);
  };
  auto any = [&](auto pa_, auto pw_) {
    if (out_planes) go(pa_, pw_, integral_constant<int, EPI_GELU>{}, std::true_type{});
    else if (epi == EPI_ADD) go(pa_, pw_, integral_constant<int, EPI_ADD>{}, std::false_type{});
    else go(pa_, pw_, integral_constant<int, EPI_STORE>{}, std::false_type{});
  };
  if (pa == 2 && pw == 2) any(integral_constant<int, 2>{}, integral_constant<int, 2>{});
  else if (pa == 2 && pw == 1) any(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  else if (pa == 3 && pw == 3) any(integral_constant<int, 3>{}, integral_constant<int, 3>{});
  else return fail(ctx, MB_ERR_ARG, "plane gemm is not built for %d x %d planes", pa, pw);
  MB_HIP(ctx, hipGetLastError());
  return MB_OK;
}

}  // namespace mb
