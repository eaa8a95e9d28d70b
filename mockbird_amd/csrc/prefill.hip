// Causal prefill attention on MFMA (gfx950), flash-style: no S x S score
// matrix is ever materialised (the reference writes [12, S, S] scores and
// probabilities, kernels-batch.ts:246-350, and caps S at 256, prefill.ts:136).
//
// A wave owns 16 or 32 query columns of one (sequence, head).  The kernels
// compute S^T = K Q^T so that the accumulator tile (lane l holds rows
// (l/16)*4 + j, column l%16) is already half of the B operand of the next
// v_mfma_f32_16x16x32_bf16 (the order of its k values is free), so P^T goes
// from the softmax straight into O^T += V^T P^T without an LDS round trip.
//
// Queries: row r of sequence b sits at position cur = pos0[b] + r and sees
// the ring slots whose stored position p satisfies 0 <= cur - p < C (the
// window rule of kernels-decode.ts:608-611, which implies p <= cur: causal).
// Slots are visited in physical order, 64 at a time, up to
// min(last position in the tile + 1, C).
#include <type_traits>

#include "kv_types.h"
#include "lds_dma.h"
#include "mb_internal.h"
#include "planes.h"
#include "rope.h"

namespace mb {

typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int KT = 64;    // slots per K/V tile of the bf16 kernel
constexpr int QT = 64;    // query rows per workgroup of the fp32-query kernel

// Workgroup -> (sequence, head, query tile).  Query tile t of a causal
// prefill costs about t + 1 K/V tiles, so the work is numbered latest tile
// first, all (sequence, head) pairs of one tile before the next: every XCD
// gets an equal share of every tile length and the longest start first.
// (With the tile index as the fastest grid coordinate, an 8-tile grid would
// send all of tile t to one XCD.)
//
// The dispatcher deals consecutive workgroups round-robin to the nxcd XCDs
// (workgroup L to XCD L % nxcd, as that XCD's (L / nxcd)-th) and, within an
// XCD, round-robin to its cpx CUs: when a launch fits at once, a CU holds
// the XCD's workgroups c, c + cpx, c + 2 cpx, ...  Handing out the work in
// rounds of cpx, every second full round in reverse (a snake), pairs the
// long tiles with short ones on each CU.  Work item g = nxcd * j + x stays
// on XCD x, so a (sequence, head) pair's tiles share one L2 whenever the
// pair count is a multiple of nxcd.  cpx = 0 hands out the work in order.
// The launcher keeps the workgroup count below 2^31, so the numbering is
// done in 32-bit unsigned arithmetic (a 64-bit division by a run-time value
// is a long scalar and vector sequence, run by every wave before its first
// load).
__device__ __forceinline__ void work_item(int& b, int& h, int& qtile, int nxcd, int cpx) {
  const uint32_t L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const uint32_t pairs = gridDim.y * gridDim.z;
  uint32_t g = L;
  if (cpx > 0) {
    const uint32_t total = pairs * gridDim.x, ux = (uint32_t)nxcd, uc = (uint32_t)cpx;
    const uint32_t x = L % ux, i = L / ux, nx = (total - x + ux - 1) / ux;
    const uint32_t r = i / uc, c = i % uc;
    const uint32_t j = ((r & 1) && (r + 1) * uc <= nx) ? r * uc + (uc - 1 - c) : i;
    g = ux * j + x;
  }
  qtile = (int)(gridDim.x - 1 - g / pairs);
  const uint32_t hb = g % pairs;
  h = (int)(hb % gridDim.y);
  b = (int)(hb / gridDim.y);
}


// ---------------------------------------------------------------- bf16 MMA

// Q bf16 [B][rows_max][768] (roped), K/V bf16 ring, fp32 output.
//
// One workgroup = 128 query rows of one (sequence, head).  With 4 waves
// (the launch's choice) each wave owns 32 of them as two 16-query column
// blocks, so every K or V^T fragment read from LDS feeds two MFMAs; with 8,
// one block of 16.  Both products use v_mfma_f32_16x16x32_bf16:
//  - scores: S^T[16 slots][16 queries] += K[16 slots][32 dims] Q^T[32 dims][16 queries];
//  - P V:    O^T[16 dims][16 queries] += V^T[16 dims][32 slots] P^T[32 slots][16 queries].
// For P V, lane l (g = l/16) must hold P^T for 8 slots of one query; the score
// accumulators give it slots sb*16 + 4g + j (j < 4) of blocks sb = 2c and
// 2c + 1, and the MFMA's k order is free, so those 8 slots are its k range.
//
// K/V tiles of 64 slots reach LDS without passing through registers
// (global_load_lds_dwordx4: lane L of a load lands at the uniform LDS base +
// 16 L), three buffers deep, two tiles ahead of the one being computed.  Rows
// are stored in their natural [slot][dim] order with the 16-byte chunks of
// row s XOR-swizzled by s mod 8, so the 16 rows a fragment read touches
// spread over the banks.  V^T fragments come from the natural layout through
// ds_read_b64_tr_b16: within each 16-lane group, lane r points at 4
// consecutive dims of slot s0 + r/4, and lane i receives dim i of slots
// s0 .. s0 + 3 -- four k values of the A operand; two such reads make one.
//
// Every wave issues the same number of loads per tile (its 1 KB pieces of K
// and V, and the tile's 64 stored positions, which all waves write alike),
// with every lane active -- slots past the causal end are clamped to the last
// one and ignored by the compute -- so `vmcnt` counts tiles exactly.  Per tile
// each wave classifies the slots against its queries with two ballots: all in
// the future of every query (the causal upper triangle: skipped), all live
// for every query (no per-slot test), or mixed (the window rule per slot and
// query, against relative positions the wave reads back from its own LDS row).
//
// Where the time goes (16 sequences x 512 rows, 12 heads, ~16 us): the
// workgroups start over ~1.4 us, every one loads its q rows and first tile
// at once (~1.9 us with HBM near peak), and the longest query tiles then run
// ~10 us of tile loop on SIMDs that issue ~60 % of the time.  A wave's tile
// is a dependent chain (scores -> softmax -> P V); taken out of copies of an
// earlier form of the kernel, neither product's MFMAs cost time, the softmax
// did.  Software-pipelining the next tile's scores under this tile's softmax
// needs ~210 registers (2 waves per SIMD) and was slower, as were 8 waves of
// 16 queries, an order that keeps a sequence's query tiles on one XCD, and
// skipping the all-future half of a diagonal tile (its branches cost more
// than the work saved).
constexpr int BQ = 128;  // query rows per workgroup of the bf16 kernel
constexpr int kFlashWaves = 4;  // waves per workgroup of the bf16 kernel
constexpr int NBUF = 3;  // K/V tile buffers
constexpr float kScoreLog2 = 0.125f * 1.4426950408889634f;  // 1/sqrt(64) * log2(e)
constexpr int32_t kRelEmpty = INT32_MAX;  // relative position of an empty slot

typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x4_t lds_bf16x4_t;

// Maximum over the four lanes of a column, with plain v_max_f32: fmaxf
// wraps both values that come out of each cross-lane swap in a canonicalising
// max (four more instructions per column); the plain instruction returns the
// same maximum for every input but signalling NaNs, which no score is.
__device__ __forceinline__ float col_max_plain(float x) {
  return col_reduce(x, [](float u, float v) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(u), "v"(v));
    return r;
  });
}

// Element offset of (slot row, 8-dim chunk x) in a swizzled 64 x 64 tile.
__device__ __forceinline__ int swz(int row, int x) { return row * HD + ((x ^ (row & 7)) << 3); }

template <int NW>
__global__ __launch_bounds__(64 * NW, 3 * NW / 4) void k_flash_bf16(
    const uint16_t* __restrict__ q, Rows q_rows, const int32_t* __restrict__ pos0,
    const int32_t* __restrict__ n_rows, const uint16_t* __restrict__ ring_k,
    const uint16_t* __restrict__ ring_v, const int32_t* __restrict__ slot_pos,
    int64_t ring_seq_stride, int C, int W, float* __restrict__ out, Rows out_rows, int nxcd,
    int cpx) {
  constexpr int QB = BQ / (16 * NW);  // 16-query blocks per wave
  constexpr int WQ = 16 * QB;         // queries per wave
  constexpr int PIECES = KT / (8 * NW);  // 1 KB pieces of K (and of V) per wave per tile
  constexpr int LOADS = 2 * PIECES + 1;  // loads per wave per tile
  static_assert(QB >= 1 && PIECES >= 1, "wave count");
  __shared__ __align__(16) uint16_t Ks[NBUF][KT * HD];  // [slot][dim], chunks swizzled
  __shared__ __align__(16) uint16_t Vs[NBUF][KT * HD];  // [slot][dim], chunks swizzled
  __shared__ __align__(16) int32_t Ps[NBUF][KT];         // stored position per slot
  __shared__ __align__(16) int32_t Rl[NW][KT];           // per wave: relative positions
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qcol = lane & 15, grp = lane >> 4;
  int b, h, qtile;
  work_item(b, h, qtile, nxcd, cpx);
  const int n = n_rows[b];
  if (qtile * BQ >= n) return;  // uniform per workgroup, before any barrier
  const int64_t p0 = pos0[b];
  const int rw = qtile * BQ + wave * WQ;  // this wave's first query row
  const bool wave_rows = rw < n;
  const int rlast = min(qtile * BQ + BQ, n) - 1;
  const int64_t kv_end64 = p0 + rlast + 1;
  const int kv_end = kv_end64 < C ? (int)kv_end64 : C;
  if (kv_end <= 0) {  // every position negative: no slot to read, rows of zeros
    const int first = qtile * BQ;
    for (int i = tid; i < (rlast + 1 - first) * (HD / 4); i += 64 * NW)
      *(f32x4_t*)(out + row_at(out_rows, b, first + i / (HD / 4)) + h * HD + i % (HD / 4) * 4) =
          f32x4_t{0.f, 0.f, 0.f, 0.f};
    return;  // uniform per workgroup, before any barrier
  }

  // B operands of the score MFMA: Q[row][32*kc + 8*grp + 0..7] times
  // 1/sqrt(64) * log2(e), rounded to bf16 once here, so the MFMA yields the
  // scores in log2 units and the softmax needs no per-score scaling.  (The
  // extra rounding of q is a relative 2^-9 per element; the probabilities
  // are rounded to bf16 for P V anyway.)
  bf16x8_t qb[QB][2];
#pragma unroll
  for (int qi = 0; qi < QB; qi++) {
    const int r = rw + qi * 16 + qcol;
#pragma unroll
    for (int kc = 0; kc < 2; kc++) {
      uint4 raw = make_uint4(0, 0, 0, 0);
      if (r < n) raw = *(const uint4*)(q + row_at(q_rows, b, r) + h * HD + kc * 32 + grp * 8);
      const bf16x8_t v = __builtin_bit_cast(bf16x8_t, raw);
#pragma unroll
      for (int e = 0; e < 8; e++) qb[qi][kc][e] = (__bf16)((float)v[e] * kScoreLog2);
    }
  }
  // Window test in 32 bits.  Stored positions are at most INT32_MAX (the ring
  // write stores no larger one).  Relative to ref = min(p0 + qtile*BQ,
  // INT32_MAX), a slot at p has rel = p - ref (an int32) and the query at row
  // offset c within the workgroup has crel = c + ex, where ex = the part of
  // the first query's position above INT32_MAX (0 in practice; clamped at 2^30,
  // beyond every window).  crel - rel is then the true distance cur - p
  // whenever that is >= 0, exactly, as an unsigned 32-bit number, and a huge
  // one when p is in the future, so the window rule 0 <= cur - p < W is one
  // unsigned compare.  An empty slot (or one past the causal end) has rel =
  // INT32_MAX, which fails it for every query.
  const int64_t first = p0 + (int64_t)qtile * BQ;
  const int32_t ref = first < INT32_MAX ? (int32_t)first : INT32_MAX;
  const int32_t ex = (int32_t)min(first - ref, (int64_t)1 << 30);
  const int crel_lo = wave * WQ + ex, crel_hi = min(rw + WQ - 1, n - 1) - qtile * BQ + ex;
  const int lane_lim = kv_end - lane;  // t0 >= lane_lim: this lane's slot is past the end
  int crel[QB];
#pragma unroll
  for (int qi = 0; qi < QB; qi++) crel[qi] = crel_lo + qi * 16 + qcol;
  const uint16_t* kb = ring_k + (int64_t)b * ring_seq_stride + (int64_t)h * C * HD;
  const uint16_t* vb = ring_v + (int64_t)b * ring_seq_stride + (int64_t)h * C * HD;
  const int32_t* sp = slot_pos + (int64_t)b * C;

  // Tile t0 -> buffer bb: wave w loads its KT / NW rows of K and of V as
  // 1 KB pieces (lane L: row 8 (PIECES w + p) + L/8, LDS chunk L mod 8 =
  // global chunk (L mod 8) ^ (row mod 8)), and the 64 stored positions (every
  // wave writes them alike, so each issues the same count of loads).  A whole
  // tile is read from base + t0 * 64 at fixed per-lane offsets; the last,
  // partial tile clamps each lane's slot to the last one instead.
  int prow[PIECES], pchunk[PIECES];
  uint32_t poff[PIECES];
#pragma unroll
  for (int piece = 0; piece < PIECES; piece++) {
    prow[piece] = 8 * (PIECES * wave + piece) + (lane >> 3);
    pchunk[piece] = (lane & 7) ^ (prow[piece] & 7);
    poff[piece] = (uint32_t)(prow[piece] * HD + pchunk[piece] * 8) * 2u;
  }
  auto issue = [&](int t0, int bb) {
    if (t0 + KT <= kv_end) {  // uniform
#pragma unroll
      for (int piece = 0; piece < PIECES; piece++) {
        const int loff = 8 * (PIECES * wave + piece) * HD;
        dma16(kb + (int64_t)t0 * HD, poff[piece], lds_addr(&Ks[bb][loff]));
        dma16(vb + (int64_t)t0 * HD, poff[piece], lds_addr(&Vs[bb][loff]));
      }
      dma4(sp + t0, (uint32_t)lane * 4u, lds_addr(&Ps[bb][0]));
    } else {
#pragma unroll
      for (int piece = 0; piece < PIECES; piece++) {
        const int loff = 8 * (PIECES * wave + piece) * HD;
        const int slot = min(t0 + prow[piece], kv_end - 1);
        const uint32_t off = (uint32_t)(slot * HD + pchunk[piece] * 8) * 2u;
        dma16(kb, off, lds_addr(&Ks[bb][loff]));
        dma16(vb, off, lds_addr(&Vs[bb][loff]));
      }
      dma4(sp, (uint32_t)min(t0 + lane, kv_end - 1) * 4u, lds_addr(&Ps[bb][0]));
    }
  };

  f32x4_t acc[QB][4], lsum[QB];
  // Per query column: the running maximum m (log2 units) enters as the
  // score MFMA's accumulator input moff = -m (0 while m = -inf), so the
  // products come out as t = score - m, the exponent's argument.  lim is
  // the rescale threshold on t: -inf while m = -inf, then 8.
  f32x4_t moff[QB];
  float lim[QB];
#pragma unroll
  for (int qi = 0; qi < QB; qi++) {
#pragma unroll
    for (int d = 0; d < 4; d++) acc[qi][d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    lsum[qi] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    moff[qi] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    lim[qi] = -INFINITY;
  }
  bf16x8_t ones;
#pragma unroll
  for (int i = 0; i < 8; i++) ones[i] = (__bf16)1.f;
  // P V: lane r of each 16-lane group points at dims 16d + 4(r mod 4) .. + 3
  // of slot 32c + 4 grp + r/4 (and 16 slots later for the second half),
  // which the transposed read turns into V^T[16d + r][those 4 slots]
  const int trow = grp * 4 + (qcol >> 2), tdim = (qcol & 3) * 4;

  // One tile: wait for its loads, publish it, refill the buffer read two
  // tiles ago, then scores, softmax and P V.  FIRST = the wave's first tile
  // (tile 0), which needs no rescale: acc and the weight sum are still zero.
  auto step = [&](int t0, auto bufc, auto first) {
    constexpr int buf = decltype(bufc)::value;  // a constant: LDS offsets fold into the reads
    constexpr bool FIRST = decltype(first)::value;
    // this tile's loads are done once at most the next tile's are
    // outstanding (vmcnt counts in issue order)
    if (!FIRST) {
      if (t0 + KT < kv_end)
        MB_WAIT_VMCNT(LOADS);
      else
        MB_WAIT_VMCNT(0);
    }
    // every wave's part of this tile is in LDS, and every wave is done with
    // the buffer the next issue overwrites (read two tiles ago)
    __syncthreads();
    if (FIRST && KT < kv_end) issue(KT, 1);  // uniform per workgroup
    if (t0 + 2 * KT < kv_end) issue(t0 + 2 * KT, (buf + NBUF - 1) % NBUF);
    if (!wave_rows) return;
    // The slot positions, then (with registers to spare: two query blocks
    // per wave) the K fragments (A of the score MFMA = K[slot sb*16 +
    // qcol][dims 32 kc + 8 grp ..]), issued before the classification so
    // their LDS latency runs under it; the empty asm keeps the compiler from
    // sinking them below the skip branch.
    const int32_t praw = Ps[buf][lane];
    auto kfrag = [&](int sb, int kc) {
      return *(const bf16x8_t*)&Ks[buf][swz(sb * 16 + qcol, kc * 4 + grp)];
    };
    bf16x8_t ka[4][2];
    if constexpr (QB > 1) {
#pragma unroll
      for (int sb = 0; sb < 4; sb++)
#pragma unroll
        for (int kc = 0; kc < 2; kc++) ka[sb][kc] = kfrag(sb, kc);
      asm volatile("" ::: "memory");
    }
    // Per slot (lane): not after every query of this wave (else it is in
    // the causal upper triangle: a tile of such slots only is skipped), and
    // not live for every one of them (`partial`; rel <= crel_lo <= crel_hi
    // makes the unsigned difference exact).  Only the 16-slot blocks holding
    // a partial slot apply the per-slot window test.
    const int32_t rel_l = praw < 0 || t0 >= lane_lim ? kRelEmpty : praw - ref;
    if (__ballot(rel_l <= crel_hi) == 0) return;
    // (every lane is active here, so the complement of a ballot is the
    // ballot of the complement)
    const uint64_t partial =
        ~(__ballot(rel_l <= crel_lo) & __ballot((uint32_t)crel_hi - (uint32_t)rel_l < (uint32_t)W));

    // S^T blocks: rows = slots sb*16 + grp*4 + j, column = query qi*16 + qcol;
    // t = score - m in log2 units (the accumulator starts at -m)
    f32x4_t s[QB][4];
#pragma unroll
    for (int sb = 0; sb < 4; sb++)
#pragma unroll
      for (int qi = 0; qi < QB; qi++) {
        s[qi][sb] = moff[qi];
#pragma unroll
        for (int kc = 0; kc < 2; kc++)
          s[qi][sb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(QB > 1 ? ka[sb][kc] : kfrag(sb, kc),
                                                              qb[qi][kc], s[qi][sb], 0, 0, 0);
      }
    // The A operand of P V for 32-slot chunk c and dim block d; with
    // registers to spare they are read now, so their LDS latency runs under
    // the softmax.
    auto vfrag = [&](int c, int d) {
      const int dim = d * 16 + tdim;
      const int e0 = swz(c * 32 + trow, dim >> 3) + (dim & 7);
      const int e1 = swz(c * 32 + 16 + trow, dim >> 3) + (dim & 7);
      const bf16x4_t lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_t*)&Vs[buf][e0]);
      const bf16x4_t hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_t*)&Vs[buf][e1]);
      return bf16x8_t{lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
    };
    bf16x8_t va[2][4];
    if constexpr (QB > 1) {
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int d = 0; d < 4; d++) va[c][d] = vfrag(c, d);
    }
    if (partial) {  // uniform
      // the wave's own row of relative positions: lane l's four score
      // elements of block sb stand for slots sb*16 + 4*grp + j
      Rl[wave][lane] = rel_l;
#pragma unroll
      for (int sb = 0; sb < 4; sb++) {
        if ((partial >> (16 * sb)) & 0xFFFFu) {  // uniform
          const int4 pv = *(const int4*)&Rl[wave][sb * 16 + grp * 4];
          const int32_t pj[4] = {pv.x, pv.y, pv.z, pv.w};
#pragma unroll
          for (int j = 0; j < 4; j++)
#pragma unroll
            for (int qi = 0; qi < QB; qi++)
              if ((uint32_t)(crel[qi] - pj[j]) >= (uint32_t)W) s[qi][sb][j] = -INFINITY;
        }
      }
    }
    // Online softmax in log2 units.  The running maximum m only moves when a
    // tile's maximum exceeds it by more than 8 (the conditional rescaling of
    // FlashAttention-3): the weights 2^t then stay <= 256, and the rescale of
    // the accumulators, a wave-uniform branch taken for all query blocks at
    // once, is rare after the first tiles.  The test needs only each lane's
    // own maximum (a column moves iff one of its four lanes exceeds lim); the
    // column maximum is formed on the rare branch.  The result is the same
    // softmax: acc and the weight sum always share one m.
    float xm[QB];       // this lane's maximum of t
    uint64_t grow = 0;  // lanes whose maximum passes the threshold
#pragma unroll
    for (int qi = 0; qi < QB; qi++) {
      float x = -INFINITY;
#pragma unroll
      for (int sb = 0; sb < 4; sb++)
#pragma unroll
        for (int j = 0; j < 4; j++) x = fmaxf(x, s[qi][sb][j]);
      xm[qi] = x;
      grow |= __ballot(x > lim[qi]);
    }
    if (grow) {  // uniform
#pragma unroll
      for (int qi = 0; qi < QB; qi++) {
        const float xt = col_max_plain(xm[qi]);  // column maximum of t
        if (xt > lim[qi]) {  // uniform per column
          if constexpr (!FIRST) {
            // exp2(m_old - m_new); 0 while m_old = -inf (acc is still zero)
            const float scale = lim[qi] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(-xt);
#pragma unroll
            for (int d = 0; d < 4; d++) acc[qi][d] *= scale;
            lsum[qi] *= scale;
          }
#pragma unroll
          for (int sb = 0; sb < 4; sb++) s[qi][sb] -= xt;
          moff[qi] -= xt;
          lim[qi] = 8.f;
        }
      }
    }
    bf16x8_t pb[QB][2];
#pragma unroll
    for (int qi = 0; qi < QB; qi++)
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int e = 0; e < 8; e++)
          pb[qi][c][e] = (__bf16)__builtin_amdgcn_exp2f(s[qi][2 * c + (e >> 2)][e & 3]);
    // O^T[d-block] += V^T[d-block rows][32 slots of chunk c] P^T[those
    // slots][queries].  The weight sum is one more MFMA with an all-ones A,
    // so it adds the same rounded weights the products use.
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma unroll
      for (int d = 0; d < 4; d++) {
        const bf16x8_t a = QB > 1 ? va[c][d] : vfrag(c, d);
#pragma unroll
        for (int qi = 0; qi < QB; qi++)
          acc[qi][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[qi][c], acc[qi][d], 0, 0, 0);
      }
#pragma unroll
      for (int qi = 0; qi < QB; qi++)
        lsum[qi] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[qi][c], lsum[qi], 0, 0, 0);
    }
  };
  // the first tile and q, then every later tile two tiles ahead of its use
  // (kv_end >= 1 here)
  using std::integral_constant;
  issue(0, 0);
  MB_WAIT_VMCNT(0);
  step(0, integral_constant<int, 0>{}, std::true_type{});
  for (int t0 = KT; t0 < kv_end; t0 += NBUF * KT) {
    static_assert(NBUF == 3, "the loop is unrolled by the buffer count");
    step(t0, integral_constant<int, 1>{}, std::false_type{});
    if (t0 + KT >= kv_end) break;
    step(t0 + KT, integral_constant<int, 2>{}, std::false_type{});
    if (t0 + 2 * KT >= kv_end) break;
    step(t0 + 2 * KT, integral_constant<int, 0>{}, std::false_type{});
  }
  const int buf = ((kv_end + KT - 1) / KT) % NBUF;  // the buffer a next tile would fill
  // The output goes through LDS so that every store writes whole rows.
  // After the last tile's barrier no wave touches two of the three K/V
  // buffers again (the one before the last tile, and the one the next tile
  // would have filled: no load is in flight), so each wave stages its WQ x
  // 64 fp32 block in a quarter of their 32 KB without waiting for the
  // others, 16-byte chunks of row r XOR-swizzled by r mod 16 (conflict-free
  // both ways), and reads it back 16 lanes per row.  The stores are
  // non-temporal: this kernel never reads the rows again, and rows kept out
  // of the L2 leave nothing to write back when the kernel ends (16
  // sequences x 512 rows: 18.9 us with 64-byte pieces through the L2, 16.9
  // us whole rows non-temporal; non-temporal 64-byte pieces gain as much
  // there but lose 4 us at 64 sequences).
  static_assert(BQ * HD * 4 == 4 * KT * HD * 2 && NW % 4 == 0, "output stage");
  float* stage;
  {
    const int f = (wave / (NW / 4)) >> 1;            // which free buffer
    const int fb = f == 0 ? buf : (buf == NBUF - 1 ? 0 : buf + 1);
    uint16_t* region = (wave / (NW / 4)) & 1 ? &Vs[fb][0] : &Ks[fb][0];
    stage = (float*)region + (wave % (NW / 4)) * WQ * HD;
  }
#pragma unroll
  for (int qi = 0; qi < QB; qi++) {
    const float l = lsum[qi][0];
    const float inv = l > 0.f ? __builtin_amdgcn_rcpf(l) : 0.f;
#pragma unroll
    for (int d = 0; d < 4; d++)
      *(f32x4_t*)&stage[(qi * 16 + qcol) * HD + (((4 * d + grp) ^ qcol) << 2)] = acc[qi][d] * inv;
  }
  // Lane (grp, c = lane mod 16) stores chunk c of rows 4 i + grp.  The
  // swizzle (4 i + grp) mod 16 repeats every 4 rows-of-four, so four LDS
  // offsets serve all WQ / 4 reads.
  const int64_t rs = out_rows.row_stride;
  float* ob = out + row_at(out_rows, b, rw) + h * HD + grp * rs + qcol * 4;
  int soff[4];
#pragma unroll
  for (int i = 0; i < 4; i++) soff[i] = (i * 4 + grp) * HD + ((qcol ^ (i * 4 + grp)) << 2);
  auto row_out = [&](int i) {
    return *(const f32x4_t*)&stage[soff[i & 3] + (i >> 2) * 16 * HD];
  };
  if (rw + WQ <= n) {  // uniform: every row of the wave is a query row
#pragma unroll
    for (int i = 0; i < WQ / 4; i++) __builtin_nontemporal_store(row_out(i), (f32x4_t*)(ob + i * 4 * rs));
  } else {
#pragma unroll
    for (int i = 0; i < WQ / 4; i++)
      if (rw + i * 4 + grp < n) __builtin_nontemporal_store(row_out(i), (f32x4_t*)(ob + i * 4 * rs));
  }
}
#undef MB_WAIT_VMCNT

// ------------------------------------------------------------ fp32 queries

// Q fp32 [B][rows_max][768] (roped), K/V fp32 or bf16 ring, fp32 output: the
// model's prompt passes.  Tile classes and online softmax are k_flash_bf16's;
// every fp32 operand enters the bf16 matrix unit as three exact bf16 planes
// (split3), so a 32-deep product of an fp32 and a bf16 operand is three
// MFMAs of 16 cycles and one of two fp32 operands six, where
// v_mfma_f32_16x16x4f32 takes eight of 32.  The fp32 matrix rate bounded the
// kernel that used it.  The error against float64 is no larger than with fp32
// products (1 x 281 rows, fp32 ring 2.5e-7 -> 2.2e-7 relative; bf16 ring
// 3.3e-7 -> 2.8e-7): the sums are fp32 either way, in fewer roundings.  Rows
// whose sums are not finite are taken again with fp32 products.
//
// A workgroup is 64 query rows of one (sequence, head), 16 per wave.  K/V
// tiles of KS slots pass through registers into one of two LDS buffers (fp32
// ones split on the way, once per workgroup), the next tile's loads in flight
// under the current tile; one barrier per tile.  KS is 64 for bf16 rings and
// 32 for fp32 ones, whose three planes fill the same 48 KB twice over; 64
// fp32 slots (one workgroup per CU) took 98 us against 72 at 16 x 512 rows.
// Also slower: 32 rows per wave (1 x 281 / 16 x 512 / 48 x 64..400 rows with
// the ring write, fp32 ring 22.1 / 74.0 / 99.8 us against 17.4 / 71.1 / 91.2,
// bf16 15.8 / 51.0 / 70.4 against 12.8 / 47.9 / 62.9: fewer workgroups, more
// registers), two waves per workgroup (20.3 / 96.3 / 121.1 us, fp32), and
// k_flash_bf16's snake order (equal).  With the fp32 MFMA kernel the same
// calls took 28.3 / 109.3 / 130.6 us (fp32) and 29.1 / 106.2 / 121.7 (bf16).
// PO: the planes of the output (the O projection's operand) instead of fp32.
template <bool KV_BF16, int PO>
__global__ __launch_bounds__(256, 3) void k_flash_x(
    const float* __restrict__ q, Rows q_rows, const int32_t* __restrict__ pos0,
    const int32_t* __restrict__ n_rows, const void* __restrict__ ring_k,
    const void* __restrict__ ring_v, const int32_t* __restrict__ slot_pos,
    int64_t ring_seq_stride, int C, int W, float* __restrict__ out, Rows out_rows) {
  constexpr int KP = KV_BF16 ? 1 : 3;   // planes of K and V
  constexpr int KS = KV_BF16 ? 64 : 32;  // slots per tile
  constexpr int IT = KS * 8 / 256;       // 8-dim chunks of K (and of V) per thread per tile
  constexpr int U = KV_BF16 ? 1 : 2;     // 16-byte loads per chunk
  constexpr int SB = KS / 16, CH = KS / 32;
  __shared__ __align__(16) uint16_t Ks[2][KP][KS * HD];  // [slot][dim], chunks swizzled
  __shared__ __align__(16) uint16_t Vs[2][KP][KS * HD];
  __shared__ __align__(16) int32_t Ps[2][KS];            // stored position per slot
  __shared__ __align__(16) int32_t Rl[4][KS];           // per wave: relative positions
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qcol = lane & 15, grp = lane >> 4;
  int b, h, qtile;
  work_item(b, h, qtile, 8, 0);
  const int n = n_rows[b];
  if (qtile * QT >= n) return;  // uniform per workgroup, before any barrier
  const int64_t p0 = pos0[b];
  const int rw = qtile * QT + wave * 16;  // this wave's first query row
  const bool wave_rows = rw < n;
  const int rlast = min(qtile * QT + QT, n) - 1;
  const int64_t kv_end64 = p0 + rlast + 1;
  const int kv_end = kv_end64 < C ? (int)kv_end64 : C;

  constexpr int E = KV_BF16 ? 2 : 4;
  const char* kb = (const char*)ring_k + ((int64_t)b * ring_seq_stride + (int64_t)h * C * HD) * E;
  const char* vb = (const char*)ring_v + ((int64_t)b * ring_seq_stride + (int64_t)h * C * HD) * E;
  const int32_t* sp = slot_pos + (int64_t)b * C;
  // a tile in registers on its way to LDS
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  u32x4_t rk[IT][U], rv[IT][U];
  int32_t rp = -1;
  auto load = [&](int t0) {
#pragma unroll
    for (int i = 0; i < IT; i++) {
      const int it = tid + i * 256, slot = min(t0 + (it >> 3), kv_end - 1);
      const int64_t off = ((int64_t)slot * HD + (it & 7) * 8) * E;
#pragma unroll
      for (int u = 0; u < U; u++) {
        rk[i][u] = *(const u32x4_t*)(kb + off + 16 * u);
        rv[i][u] = *(const u32x4_t*)(vb + off + 16 * u);
      }
    }
    if (tid < KS) rp = t0 + tid < kv_end ? sp[t0 + tid] : -1;
  };
  auto stash = [&](int bb) {
#pragma unroll
    for (int i = 0; i < IT; i++) {
      const int it = tid + i * 256, e = swz(it >> 3, it & 7);
      if constexpr (KV_BF16) {
        *(u32x4_t*)&Ks[bb][0][e] = rk[i][0];
        *(u32x4_t*)&Vs[bb][0][e] = rv[i][0];
      } else {
        float kf[8], vf[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
          kf[j] = __uint_as_float(rk[i][j >> 2][j & 3]);
          vf[j] = __uint_as_float(rv[i][j >> 2][j & 3]);
        }
        const Planes kp = split3(kf), vp = split3(vf);
#pragma unroll
        for (int p = 0; p < 3; p++) {
          *(bf16x8_t*)&Ks[bb][p][e] = kp.p[p];
          *(bf16x8_t*)&Vs[bb][p][e] = vp.p[p];
        }
      }
    }
    if (tid < KS) Ps[bb][tid] = rp;
  };
  // every position of the tile's rows negative (kv_end <= 0): no slot is read,
  // and the rows are zero
  if (kv_end > 0) load(0);

  // B operands of the score MFMA: the planes of Q[row][32 kc + 8 grp + 0..7]
  // times 1/sqrt(64) * log2(e) (one fp32 rounding), so the MFMAs yield the
  // scores in log2 units
  const int r = rw + qcol;
  Planes qp[2];
  {
    const float* src = q + row_at(q_rows, b, min(r, n - 1)) + h * HD + grp * 8;
#pragma unroll
    for (int kc = 0; kc < 2; kc++) {
      const float4 x = *(const float4*)(src + kc * 32), y = *(const float4*)(src + kc * 32 + 4);
      const float v[8] = {x.x * kScoreLog2, x.y * kScoreLog2, x.z * kScoreLog2, x.w * kScoreLog2,
                          y.x * kScoreLog2, y.y * kScoreLog2, y.z * kScoreLog2, y.w * kScoreLog2};
      qp[kc] = split3(v);
    }
  }
  // the window test in 32 bits, relative to the workgroup's first query (see
  // k_flash_bf16)
  const int64_t first = p0 + (int64_t)qtile * QT;
  const int32_t ref = first < INT32_MAX ? (int32_t)first : INT32_MAX;
  const int32_t ex = (int32_t)min(first - ref, (int64_t)1 << 30);
  const int crel_lo = wave * 16 + ex, crel_hi = min(rw + 15, n - 1) - qtile * QT + ex;
  const int crel = crel_lo + qcol;

  f32x4_t acc[4];
#pragma unroll
  for (int d = 0; d < 4; d++) acc[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float lsum = 0.f;                         // this lane's share of the column's weight sum
  f32x4_t moff = f32x4_t{0.f, 0.f, 0.f, 0.f};  // -m (0 while m = -inf), where the scores start
  float lim = -INFINITY;                    // rescale threshold on t = score - m
  const int trow = grp * 4 + (qcol >> 2), tdim = (qcol & 3) * 4;

  auto compute = [&](int bb) {
    const int32_t praw = Ps[bb][lane & (KS - 1)];
    const int32_t rel_l = praw < 0 ? kRelEmpty : praw - ref;
    if (__ballot(rel_l <= crel_hi) == 0) return;
    const uint64_t partial =
        ~(__ballot(rel_l <= crel_lo) & __ballot((uint32_t)crel_hi - (uint32_t)rel_l < (uint32_t)W));
    f32x4_t s[SB];
#pragma unroll
    for (int sb = 0; sb < SB; sb++) s[sb] = moff;
#pragma unroll
    for (int kc = 0; kc < 2; kc++) {
      bf16x8_t ka[SB][KP];
#pragma unroll
      for (int sb = 0; sb < SB; sb++)
#pragma unroll
        for (int p = 0; p < KP; p++)
          ka[sb][p] = *(const bf16x8_t*)&Ks[bb][p][swz(sb * 16 + qcol, kc * 4 + grp)];
      plane_products<KP, 3>([&](auto i, auto j) {
#pragma unroll
        for (int sb = 0; sb < SB; sb++)
          s[sb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[sb][i], qp[kc].p[j], s[sb], 0, 0, 0);
      });
    }
    if (partial) {  // uniform
      Rl[wave][lane & (KS - 1)] = rel_l;
#pragma unroll
      for (int sb = 0; sb < SB; sb++) {
        if ((partial >> (16 * sb)) & 0xFFFFu) {  // uniform
          const int4 pv = *(const int4*)&Rl[wave][sb * 16 + grp * 4];
          const int32_t pj[4] = {pv.x, pv.y, pv.z, pv.w};
#pragma unroll
          for (int j = 0; j < 4; j++)
            if ((uint32_t)(crel - pj[j]) >= (uint32_t)W) s[sb][j] = -INFINITY;
        }
      }
    }
    float xm = -INFINITY;
#pragma unroll
    for (int sb = 0; sb < SB; sb++)
#pragma unroll
      for (int j = 0; j < 4; j++) xm = fmaxf(xm, s[sb][j]);
    if (__ballot(xm > lim)) {  // uniform
      const float xt = col_max(xm);
      if (xt > lim) {  // uniform per column
        const float scale = lim == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(-xt);
#pragma unroll
        for (int d = 0; d < 4; d++) acc[d] *= scale;
        lsum *= scale;
#pragma unroll
        for (int sb = 0; sb < SB; sb++) s[sb] -= xt;
        moff -= xt;
        lim = 8.f;
      }
    }
#pragma unroll
    for (int c = 0; c < CH; c++) {
      float w[8];
#pragma unroll
      for (int e = 0; e < 8; e++) w[e] = __builtin_amdgcn_exp2f(s[2 * c + (e >> 2)][e & 3]);
      lsum += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
      const Planes pp = split3(w);
      bf16x8_t va[4][KP];
#pragma unroll
      for (int d = 0; d < 4; d++)
#pragma unroll
        for (int p = 0; p < KP; p++) {
          const int dim = d * 16 + tdim;
          const int e0 = swz(c * 32 + trow, dim >> 3) + (dim & 7);
          const int e1 = swz(c * 32 + 16 + trow, dim >> 3) + (dim & 7);
          const bf16x4_t lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_t*)&Vs[bb][p][e0]);
          const bf16x4_t hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_t*)&Vs[bb][p][e1]);
          va[d][p] = bf16x8_t{lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
        }
      plane_products<KP, 3>([&](auto i, auto j) {
#pragma unroll
        for (int d = 0; d < 4; d++)
          acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[d][i], pp.p[j], acc[d], 0, 0, 0);
      });
    }
  };

  if (kv_end > 0) stash(0);
  if (KS < kv_end) load(KS);
  int bb = 0;
  for (int t0 = 0; t0 < kv_end; t0 += KS) {
    // tile t0 is in LDS, and every wave is done with the buffer the next one
    // goes to (read one tile ago)
    __syncthreads();
    if (wave_rows) compute(bb);
    bb ^= 1;
    if (t0 + KS < kv_end) {
      stash(bb);
      if (t0 + 2 * KS < kv_end) load(t0 + 2 * KS);
    }
  }
  float l = col_sum(lsum);
  // An infinity has no planes (inf - inf), and 0 times one in a plane is NaN.
  // A wave with a sum that is not finite takes its rows again, slot by slot
  // over the live slots with fp32 products: infinities and NaN reach the rows
  // that see them, as those products give them, and no others.
  float nf = lsum;
#pragma unroll
  for (int d = 0; d < 4; d++) nf += (acc[d][0] + acc[d][1]) + (acc[d][2] + acc[d][3]);
  if (wave_rows && __ballot(!(fabsf(nf) < INFINITY))) {  // uniform
    const float* src = q + row_at(q_rows, b, min(r, n - 1)) + h * HD + grp * 4;
    f32x4_t qf[4];
#pragma unroll
    for (int d = 0; d < 4; d++) {
      qf[d] = *(const f32x4_t*)(src + 16 * d) * kScoreLog2;
      acc[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    auto dims = [&](const char* base, int slot, int d) {  // dims 16d + 4 grp .. + 3
      const int64_t e = (int64_t)slot * HD + 16 * d + 4 * grp;
      if constexpr (KV_BF16) {
        const uint2 w = *(const uint2*)(base + e * 2);
        return f32x4_t{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
                       __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
      } else {
        return *(const f32x4_t*)(base + e * 4);
      }
    };
    float m = -INFINITY;
    l = 0.f;
    for (int slot = 0; slot < kv_end; slot++) {
      const int32_t ps = sp[slot];
      const bool live = ps >= 0 && (uint32_t)(crel - (ps - ref)) < (uint32_t)W;
      if (!__ballot(live)) continue;  // uniform
      float x = 0.f;
#pragma unroll
      for (int d = 0; d < 4; d++) {
        const f32x4_t k = dims(kb, slot, d);
        x += (qf[d][0] * k[0] + qf[d][1] * k[1]) + (qf[d][2] * k[2] + qf[d][3] * k[3]);
      }
      x = col_sum(x);
      if (live) {
        const float mn = fmaxf(m, x), mu = mn == -INFINITY ? 0.f : mn;
        const float scale = __builtin_amdgcn_exp2f(m - mu), p = __builtin_amdgcn_exp2f(x - mu);
        m = mn;
        l = l * scale + p;
#pragma unroll
        for (int d = 0; d < 4; d++) acc[d] = acc[d] * scale + dims(vb, slot, d) * p;
      }
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (r >= n) return;
  if constexpr (PO == 0) {
    float* op = out + row_at(out_rows, b, r) + h * HD;
#pragma unroll
    for (int d = 0; d < 4; d++) *(f32x4_t*)(op + d * 16 + grp * 4) = acc[d] * inv;
  } else {
    const int64_t row = (int64_t)out_rows.row_off[b] + r;
#pragma unroll
    for (int d = 0; d < 4; d++) {
      const f32x4_t v = acc[d] * inv;
      uint2 o[PO];
      split4<PO>(make_float4(v[0], v[1], v[2], v[3]), o);
#pragma unroll
      for (int p = 0; p < PO; p++)
        ((uint2*)out)[2 * plane_chunk(row, h * (HD / 8) + 2 * d + (grp >> 1), D / 32, PO, p) + (grp & 1)] =
            o[p];
    }
  }
}

// ------------------------------------------------ short chunks, long windows

// Attention of a short chunk of consecutive queries (up to 16 * QB rows per
// sequence, fp32) against a long window: the codec's stages append 4..32
// positions per frame and attend over windows of 500..3248.  A workgroup is
// one (sequence, head); its NW waves take the slot range's 16-slot groups in
// turn (wave w: groups w, w + NW, ...), so the workgroup reads its
// (sequence, head) run front to back as one stream (against each wave
// streaming a contiguous run: 64 voices 1.214 -> 1.198 ms, 256 voices 2.266
// -> 2.248 ms per codec frame, same GPU, alternating), and each wave computes
// every query of the chunk against its groups, reading K and V straight from
// HBM into MFMA operands (no LDS staging).  A wave's first group is issued
// before the chunk's rows are written when it holds none of their slots
// (else after), and is in flight while the rows are written
// (64 voices 1.158 -> 1.150 ms per codec frame, 256 voices level).  Scores
// are S^T[16 slots][16 queries]; the P V output block
// d holds dims 4i + d in row i, so in the step for slot 4g + j (g = lane/16)
// a lane feeds 4 contiguous dims of that V row and its own score element j.
//  - fp32 rings: v_mfma_f32_16x16x4f32; lane l feeds K[slot l%16][16g + kc]
//    and Q[query l%16][16g + kc] in step kc (16 contiguous K dims per lane).
//  - bf16 rings: v_mfma_f32_16x16x32_bf16 for the scores (lane l feeds 8
//    contiguous K dims 32c + 8g.. of its slot) and v_mfma_f32_16x16x16bf16_1k
//    for P V (lane l feeds 4 slots 4g..4g+3 of dim 4(l%16) + d, packed from
//    its four 8-byte V loads).  K and V are exact in bf16; q and P are split
//    into a bf16 high part and a bf16 remainder, two MFMAs each, so the
//    products keep about 16 bits (the scores and weights agree with the fp32
//    path to ~1e-5 relative) at an eighth of the fp32 MFMA time.
//    q's parts are read from LDS at each group: held in registers (136 for
//    32 queries) they left one workgroup per CU, now two run (119).  The fp32
//    form keeps q in registers: from LDS it gains no workgroup and 256 voices
//    took 14.84 against 14.75 ms per four frames.
// Partials (max, sum, 64 dims per query) fold across the waves through LDS.
// SPLIT: gridDim.z workgroups share one window, and each leaves its folded
// state in `part` (k_window_merge adds them up).  Where a launch has few
// units, the bound is one workgroup's chain of dependent groups, not the
// memory: a voice's stage-4 layer (3280 slots, fp32) took 77.8 us on 4
// workgroups, 12.7 + 4.9 us on 64 and the merge.
// Liveness is the window rule: slot position p (empty slots never live) is
// visible to a query at cur iff 0 <= cur - p < W.
constexpr int kWindowWaves = 8;          // waves per workgroup
constexpr int kWindowSplitBlocks = 256;  // workgroups of a split launch at most (one per CU)
constexpr int WPART = HD + 4;  // floats of a SPLIT state: 64 sums, max (log2 units), denominator
static_assert((size_t)kWindowSplitBlocks * 32 * WPART <= kWindowPartFloats, "split states");

// K and V loads, with the streaming hint if ST.  An fp32 ring's K keeps plain
// loads: a lane reads its 64 bytes of a row in four instructions, and with the
// hint the lines do not stay for the later ones (200 voices, four frames 13.50
// -> 14.91 ms; V alone, whole lines per instruction, 13.15).
template <bool ST, class T>
__device__ __forceinline__ T load_kv(const char* p) {
  typedef uint32_t Vec __attribute__((ext_vector_type(sizeof(T) / 4)));
  if constexpr (ST) return __builtin_bit_cast(T, __builtin_nontemporal_load((const Vec*)p));
  else return *(const T*)p;
}

template <bool KV_BF16, int QB, int NW, bool SPLIT, bool ST>
__global__ __launch_bounds__(64 * NW) void k_attn_window(
    const float* __restrict__ qkv, Rows qkv_rows, const int32_t* __restrict__ pos0,
    const int32_t* __restrict__ n_rows, void* __restrict__ ring_k, void* __restrict__ ring_v,
    int32_t* __restrict__ slot_pos, int64_t ring_seq_stride, int C, int W, int wrap,
    const float2* __restrict__ rope_tab, float* __restrict__ out, Rows out_rows,
    float* __restrict__ part) {
  constexpr int NQ = 16 * QB;
  __shared__ float red_ml[NW][2][NQ];        // per wave: max (log2 units), sum
  __shared__ float red_acc[NW][NQ][HD + 1];  // per wave: unnormalised output
  // the chunk's roped q rows (this head): fp32, or for bf16 rings their bf16
  // high parts and remainders, 8-dim chunks swizzled
  __shared__ __align__(16) float q_l[KV_BF16 ? 1 : NQ][HD];
  __shared__ __align__(16) uint16_t q_p[KV_BF16 ? 2 : 1][KV_BF16 ? NQ * HD : 8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int qc = lane & 15, g = lane >> 4;
  const int h = blockIdx.x, b = blockIdx.y;
  // SPLIT: workgroup z of gridDim.z takes the groups g0, g0 + step, ... of
  // its waves (the unsplit workgroup's numbering with gridDim.z * NW waves)
  const int g0 = SPLIT ? (int)blockIdx.z * NW + wave : wave;
  const int step = SPLIT ? (int)gridDim.z * NW : NW;
  const int n = n_rows[b];
  const int64_t p0 = pos0[b];
  const int64_t end64 = p0 + n;
  const int kv_end = end64 < C ? (int)end64 : C;
  const int groups = (kv_end + 15) >> 4;

  constexpr int E = KV_BF16 ? 2 : 4;
  const char* kb = (const char*)ring_k + ((int64_t)b * ring_seq_stride + (int64_t)h * C * HD) * E;
  const char* vb = (const char*)ring_v + ((int64_t)b * ring_seq_stride + (int64_t)h * C * HD) * E;
  const int32_t* sp = slot_pos + (int64_t)b * C;

  // One 16-slot group's loads, as raw registers: K of the lane's slot
  // s0 + qc, V (4 dims) and the stored positions of slots s0 + 4g + j.  Every
  // index is clamped into the window so the loads carry no branch, and the
  // loop issues group gi + 1's loads before computing group gi: the loads of
  // one group stay in flight under the MFMAs of the one before.
  struct Raw {
    uint4 k[KV_BF16 ? 2 : 4];
    uint4 v[KV_BF16 ? 2 : 4];  // bf16: slots j = 0..3 as 2 x uint2 per uint4
    int32_t p[4];
  };
  auto load_group = [&](int gi, Raw& r) {
    const int s0 = gi * 16;
    const int ks = min(s0 + qc, kv_end - 1);
    if constexpr (KV_BF16) {
#pragma unroll
      for (int c = 0; c < 2; c++) r.k[c] = load_kv<ST, uint4>(kb + ((int64_t)ks * HD + c * 32 + g * 8) * 2);
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) r.k[i] = *(const uint4*)(kb + ((int64_t)ks * HD + g * 16 + 4 * i) * 4);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int sl = s0 + 4 * g + j;
      const int vs = min(sl, kv_end - 1);
      if constexpr (KV_BF16) {
        const uint2 w = load_kv<ST, uint2>(vb + ((int64_t)vs * HD + 4 * qc) * 2);
        if (j & 1) { r.v[j >> 1].z = w.x; r.v[j >> 1].w = w.y; }
        else { r.v[j >> 1].x = w.x; r.v[j >> 1].y = w.y; }
      } else {
        r.v[j] = load_kv<ST, uint4>(vb + ((int64_t)vs * HD + 4 * qc) * 4);
      }
      r.p[j] = sp[vs];
    }
  };

  // The wave's first group is issued before the chunk's rows are written
  // when it holds none of the slots they go to (the slots of rows
  // max(0, n - C) .. n - 1, at p0 + r mod C): the other slots' K, V and
  // positions are not written by this launch, so the loads see what they
  // would see after the barrier.  A group that may hold a written slot loads
  // after the barrier.
  Raw cur, nxt;
  bool early = false;
  if (g0 < groups && p0 >= 0) {
    const int lo = g0 * 16, hi = min(lo + 16, kv_end);
    const int wr0 = n > C ? n - C : 0;
    const int len = n - wr0;
    bool hit = true;
    if (len <= 0) {
      hit = false;
    } else if (len < C) {
      const int64_t first = p0 + wr0;
      const int start = wrap ? (int)(first % C) : (int)min(first, (int64_t)C);
      const int end = start + len;  // the range [start, end) taken mod C
      hit = end <= C ? (start < hi && lo < end) : (start < hi || lo < end - C);
    }
    early = !hit;
    if (early) load_group(g0, cur);
  }

  // The chunk's rows enter the ring first, as k_ring_write writes them but
  // for this head only: thread (r, d0) ropes q and k of row r's dims d0 ..
  // d0 + 7 at position p0 + r, stores K and V at slot pos mod C (only the
  // last C rows of a call longer than C) and keeps q in LDS; every head's
  // workgroup records the slots' positions (the same values), so each reads
  // only what it wrote itself once the barrier below has passed.
  {
    const int Dw = (int)gridDim.x * HD;  // width of each of q, k, v in a fused row
    for (int t = threadIdx.x; t < NQ * 8; t += 64 * NW) {
      const int r = t >> 3, d0 = (t & 7) * 8;
      const int64_t p64 = p0 + r;
      const bool ok = r < n && p64 >= 0 && p64 <= INT32_MAX && (wrap || p64 < C);
      float qo[8], ko[8], vv[8];
      if (ok) {
        const int32_t pos = (int32_t)p64;
        float qi[8], ki[8];
        const int64_t roff = row_at(qkv_rows, b, r) + h * HD + d0;
        load8<false>(qkv, roff, qi);
        load8<false>(qkv, roff + Dw, ki);
        load8<false>(qkv, roff + 2 * Dw, vv);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          float c, sn;
          rope_cs(rope_tab, pos, (d0 >> 1) + j, c, sn);
          rope_pair(qi[2 * j], qi[2 * j + 1], c, sn, qo[2 * j], qo[2 * j + 1]);
          rope_pair(ki[2 * j], ki[2 * j + 1], c, sn, ko[2 * j], ko[2 * j + 1]);
        }
        if (!(n > C && r < n - C)) {
          const int slot = wrap ? (int)(p64 % C) : (int)p64;
          // SPLIT: a row is written by the workgroup that reads its slot
          // (slots of live rows are below kv_end), so no workgroup waits for
          // another's stores
          if (!SPLIT || (slot >> 4) % step / NW == (int)blockIdx.z) {
            const int64_t koff = (int64_t)b * ring_seq_stride + ((int64_t)h * C + slot) * HD + d0;
            store8<KV_BF16>(ring_k, koff, ko);
            store8<KV_BF16>(ring_v, koff, vv);
            if (d0 == 0) slot_pos[(int64_t)b * C + slot] = pos;
          }
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++) qo[e] = 0.f;
      }
      if constexpr (KV_BF16) {
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; j++) split2_pair(qo[2 * j], qo[2 * j + 1], hi[j], lo[j]);
        *(uint4*)&q_p[0][swz(r, d0 >> 3)] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        *(uint4*)&q_p[1][swz(r, d0 >> 3)] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      } else {
        *(float4*)&q_l[r][d0] = make_float4(qo[0], qo[1], qo[2], qo[3]);
        *(float4*)&q_l[r][d0 + 4] = make_float4(qo[4], qo[5], qo[6], qo[7]);
      }
    }
  }
  __threadfence_block();
  __syncthreads();  // the rows are in the ring and q in LDS for every wave

  // the wave's first group is in flight while its state is set up
  if (g0 < groups && !early) load_group(g0, cur);
  // Positions relative to the sequence's first query, clamped so the window
  // test is one unsigned compare; an empty slot and a query past n are
  // outside every window.
  constexpr int32_t kFar = 1 << 30;
  int32_t crel[QB];
#pragma unroll
  for (int qb = 0; qb < QB; qb++) crel[qb] = qb * 16 + qc < n ? qb * 16 + qc : -kFar;
  float qv[QB][16];  // fp32 rings: dims 16g .. 16g + 15 of query qb * 16 + qc
  if constexpr (!KV_BF16) {
#pragma unroll
    for (int qb = 0; qb < QB; qb++)
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        const float4 t = *(const float4*)&q_l[qb * 16 + qc][g * 16 + i];
        qv[qb][i] = t.x; qv[qb][i + 1] = t.y; qv[qb][i + 2] = t.z; qv[qb][i + 3] = t.w;
      }
  }
  f32x4_t acc[QB][4];
#pragma unroll
  for (int qb = 0; qb < QB; qb++)
#pragma unroll
    for (int d = 0; d < 4; d++) acc[qb][d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m[QB], l[QB];
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    m[qb] = -INFINITY;
    l[qb] = 0.f;
  }

  auto compute = [&](int gi) {
    const int s0 = gi * 16;
    float kf[16];
    bf16x8_t kh[2];
    float vf[4][4];
    uint2 vw[4];
    if constexpr (KV_BF16) {
#pragma unroll
      for (int c = 0; c < 2; c++) kh[c] = __builtin_bit_cast(bf16x8_t, cur.k[c]);
#pragma unroll
      for (int j = 0; j < 4; j++)
        vw[j] = (j & 1) ? make_uint2(cur.v[j >> 1].z, cur.v[j >> 1].w)
                        : make_uint2(cur.v[j >> 1].x, cur.v[j >> 1].y);
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        kf[4 * i] = __uint_as_float(cur.k[i].x); kf[4 * i + 1] = __uint_as_float(cur.k[i].y);
        kf[4 * i + 2] = __uint_as_float(cur.k[i].z); kf[4 * i + 3] = __uint_as_float(cur.k[i].w);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        vf[j][0] = __uint_as_float(cur.v[j].x); vf[j][1] = __uint_as_float(cur.v[j].y);
        vf[j][2] = __uint_as_float(cur.v[j].z); vf[j][3] = __uint_as_float(cur.v[j].w);
      }
    }
    int32_t pj[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int sl = s0 + 4 * g + j;
      const int32_t p = sl < kv_end ? cur.p[j] : -1;
      const int64_t d = (int64_t)p - p0;
      pj[j] = p < 0 ? kFar : (int32_t)(d < -kFar ? -kFar : d > kFar ? kFar : d);
    }
    // bf16 P V operands: for block d, slots 4g..4g+3 of dim 4qc + d
    i16x4_t va[4];
    if constexpr (KV_BF16) {
#pragma unroll
      for (int d = 0; d < 4; d++) {
        const uint32_t sel = (d & 1) ? 0x07060302u : 0x05040100u;
        const int w = d >> 1;
        const uint32_t lo = __builtin_amdgcn_perm(w ? vw[1].y : vw[1].x, w ? vw[0].y : vw[0].x, sel);
        const uint32_t hi = __builtin_amdgcn_perm(w ? vw[3].y : vw[3].x, w ? vw[2].y : vw[2].x, sel);
        va[d] = __builtin_bit_cast(i16x4_t, make_uint2(lo, hi));
      }
    }
#pragma unroll
    for (int qb = 0; qb < QB; qb++) {
      f32x4_t sc = {0.f, 0.f, 0.f, 0.f};
      if constexpr (KV_BF16) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
          const int e = swz(qb * 16 + qc, c * 4 + g);  // dims 32c + 8g .. + 7
          sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh[c], *(const bf16x8_t*)&q_p[0][e], sc, 0, 0, 0);
          sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh[c], *(const bf16x8_t*)&q_p[1][e], sc, 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int kc = 0; kc < 16; kc++)
          sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kc], qv[qb][kc], sc, 0, 0, 0);
      }
      float t[4];
      float mt = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        t[j] = (unsigned)(crel[qb] - pj[j]) < (unsigned)W ? sc[j] * kScoreLog2 : -INFINITY;
        mt = fmaxf(mt, t[j]);
      }
      mt = col_max(mt);
      // conditional rescale (the running max moves only by more than 8)
      const bool grow = mt > m[qb] + 8.f;
      if (__ballot(grow)) {
        const float mn = grow ? mt : m[qb];
        const float scale = grow ? __builtin_amdgcn_exp2f(m[qb] - mn) : 1.f;
        m[qb] = mn;
        l[qb] *= scale;
#pragma unroll
        for (int d = 0; d < 4; d++) acc[qb][d] *= scale;
      }
      const float mu = m[qb] == -INFINITY ? 0.f : m[qb];
      float pw[4], ls = 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        pw[j] = __builtin_amdgcn_exp2f(t[j] - mu);
        ls += pw[j];
      }
      l[qb] += col_sum(ls);
      if constexpr (KV_BF16) {
        i16x4_t ph, pl;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const __bf16 hi = (__bf16)pw[j];
          ph[j] = __builtin_bit_cast(short, hi);
          pl[j] = __builtin_bit_cast(short, (__bf16)(pw[j] - (float)hi));
        }
#pragma unroll
        for (int d = 0; d < 4; d++) {
          acc[qb][d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va[d], ph, acc[qb][d], 0, 0, 0);
          acc[qb][d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va[d], pl, acc[qb][d], 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int d = 0; d < 4; d++)
            acc[qb][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[j][d], pw[j], acc[qb][d], 0, 0, 0);
      }
    }
  };
  // The last group has no load after it: reloading a group there to keep one
  // loop body was 1 load in 5 at a window of 500 slots.  With q's parts in
  // LDS, four frames, bf16 rings: 32 / 100 / 256 voices 2443 -> 2430, 4605 ->
  // 4513, 8749 -> 8560 us; fp32 rings 32 / 256 voices 3287 -> 3267, 14702 ->
  // 14638.
  if (g0 < groups) {
    int gi = g0;
    for (; gi + step < groups; gi += step) {
      load_group(gi + step, nxt);
      if constexpr (KV_BF16)
        asm volatile("" ::: "memory");  // q's parts are read again below, not kept in registers
      compute(gi);
      cur = nxt;
    }
    compute(gi);
  }

  // fold the waves: lane (qc, g) holds dims 4((g*4) + r) + d of query qb*16 + qc
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    if (g == 0) {
      red_ml[wave][0][qb * 16 + qc] = m[qb];
      red_ml[wave][1][qb * 16 + qc] = l[qb];
    }
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
      for (int r = 0; r < 4; r++) red_acc[wave][qb * 16 + qc][4 * (4 * g + r) + d] = acc[qb][d][r];
  }
  __syncthreads();
  for (int t = threadIdx.x; t < NQ * HD; t += 64 * NW) {
    const int qi = t / HD, dim = t % HD;
    if (qi >= n) continue;
    float M = -INFINITY;
    for (int w = 0; w < NW; w++) M = fmaxf(M, red_ml[w][0][qi]);
    float L = 0.f, o = 0.f;
    if (M != -INFINITY) {
      for (int w = 0; w < NW; w++) {
        const float mw = red_ml[w][0][qi];
        const float wt = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
        L += wt * red_ml[w][1][qi];
        o += wt * red_acc[w][qi][dim];
      }
    }
    if constexpr (SPLIT) {
      float* pp = part + (((int64_t)b * gridDim.x + h) * gridDim.z + blockIdx.z) * (NQ * WPART) +
                  qi * WPART;
      pp[dim] = o;
      if (dim == 0) {
        pp[HD] = M;
        pp[HD + 1] = L;
      }
    } else {
      out[row_at(out_rows, b, qi) + h * HD + dim] = L > 0.f ? o / L : 0.f;
    }
  }
}

// Merges the SPLIT form's states: workgroup (head, sequence), thread (query,
// 4 dims).  Every split's maximum and sum are loaded before the first use,
// then the weighted rows.
template <int QB, int S>
__global__ __launch_bounds__(256 * QB) void k_window_merge(const float* __restrict__ part,
                                                           const int32_t* __restrict__ n_rows,
                                                           float* __restrict__ out, Rows out_rows) {
  constexpr int NQ = 16 * QB;
  const int h = blockIdx.x, b = blockIdx.y;
  const int qi = threadIdx.x >> 4, dim = (threadIdx.x & 15) * 4;
  const float* pp = part + ((int64_t)b * gridDim.x + h) * S * (NQ * WPART) + qi * WPART;
  const int n = n_rows[b];  // rows past it have no state: what is loaded for them is not stored
  float2 ml[S];
  float4 o[S];
#pragma unroll
  for (int s = 0; s < S; s++) {
    ml[s] = *(const float2*)(pp + s * (NQ * WPART) + HD);
    o[s] = *(const float4*)(pp + s * (NQ * WPART) + dim);
  }
  float M = -INFINITY;
#pragma unroll
  for (int s = 0; s < S; s++) M = fmaxf(M, ml[s].x);
  float L = 0.f;
  float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int s = 0; s < S; s++) {
    const float wt = ml[s].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[s].x - M);
    L += wt * ml[s].y;
    r.x += wt * o[s].x; r.y += wt * o[s].y; r.z += wt * o[s].z; r.w += wt * o[s].w;
  }
  if (L > 0.f) {
    r.x /= L; r.y /= L; r.z /= L; r.w /= L;
  } else {
    r = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (qi < n) *(float4*)(out + row_at(out_rows, b, qi) + h * HD + dim) = r;
}

// How many workgroups share a (sequence, head) window of `slots`: a power of
// two up to 16 that keeps the launch within one workgroup per CU and leaves
// every wave a 16-slot group.  With one workgroup per unit a voice's 4 heads
// are 4 workgroups, each a chain of ~26 dependent groups per wave at 3280
// slots.  Per 4-frame codec call on full windows, one workgroup -> this rule:
// fp32 rings 1 / 8 / 32 voices 3213 -> 1884 / 3460 -> 2223 / 3791 -> 3251 us,
// bf16 2222 -> 1735 / 2092 -> 1631 / 2591 -> 2444 us.  Two workgroups per CU
// lost from 8 voices up (fp32 2362 / 3390 us at 8 / 32), as did splitting the
// 64 voices that already fill the chip (4623 -> 4923 us); two groups per wave
// cost a single voice 6 % (2002 us).
int window_splits(int units, int slots) {
  const int groups = (slots + 15) / 16;
  int s = 1;
  while (s < 16 && 2 * s * units <= kWindowSplitBlocks && groups >= 2 * s * kWindowWaves) s *= 2;
  return s;
}

// Chunks of up to 32 consecutive rows per sequence (the codec's stages):
// each row's K/V enters the ring and its query attends the window in one
// launch; rows_max bounds n_rows.  `part` (kWindowPartFloats floats, or null)
// lets a launch with few (sequence, head) units share each window between
// workgroups, whose states a second launch merges.
int launch_window_attention(mb_ctx* ctx, const RingView& ring, int B, int rows_max,
                            const float* qkv, const Rows& qkv_rows, const int32_t* pos0,
                            const int32_t* n_rows, float* out, const Rows& out_rows, float* part,
                            bool stream) {
  if (rows_max < 1 || rows_max > 32)
    return fail(ctx, MB_ERR_ARG, "window attention takes 1..32 rows per sequence, not %d", rows_max);
  if (B > 65535) return fail(ctx, MB_ERR_ARG, "at most 65535 sequences per call");
  if (B == 0) return MB_OK;
  constexpr int NW = kWindowWaves;
  const int S = part ? window_splits(ring.heads * B, ring.C) : 1;
  const dim3 grid((unsigned)ring.heads, (unsigned)B, (unsigned)S);
  auto go = [&](auto bf_, auto qb_, auto split_, auto st_) {
    constexpr bool BF = decltype(bf_)::value, SP = decltype(split_)::value, ST = decltype(st_)::value;
    constexpr int QB = decltype(qb_)::value;
    hipLaunchKernelGGL((k_attn_window<BF, QB, NW, SP, ST>), grid, dim3(64 * NW), 0, ctx->stream, qkv,
                       qkv_rows, pos0, n_rows, ring.k, ring.v, ring.sp, ring.seq_stride, ring.C,
                       ring.window, ring.wrap, ctx->rope_tab, out, out_rows, part);
  };
  auto merge = [&](auto qb_, auto s_) {
    constexpr int QB = decltype(qb_)::value;
    hipLaunchKernelGGL((k_window_merge<QB, decltype(s_)::value>),
                       dim3((unsigned)ring.heads, (unsigned)B), dim3(256 * QB), 0, ctx->stream,
                       part, n_rows, out, out_rows);
  };
  using std::integral_constant;
  auto all = [&](auto qb_) {
    auto by_type = [&](auto split_) {
      auto by_hint = [&](auto bf_) {
        if (stream) go(bf_, qb_, split_, std::true_type{});
        else go(bf_, qb_, split_, std::false_type{});
      };
      if (ring.bf16) by_hint(std::true_type{});
      else by_hint(std::false_type{});
    };
    if (S == 1) return by_type(std::false_type{});
    by_type(std::true_type{});
    if (S == 2) merge(qb_, integral_constant<int, 2>{});
    else if (S == 4) merge(qb_, integral_constant<int, 4>{});
    else if (S == 8) merge(qb_, integral_constant<int, 8>{});
    else merge(qb_, integral_constant<int, 16>{});
  };
  if (rows_max <= 16) all(integral_constant<int, 1>{});
  else all(integral_constant<int, 2>{});
  MB_HIP(ctx, hipGetLastError());
  return MB_OK;
}

int launch_prefill_attention(mb_ctx* ctx, const RingView& ring, int B, int rows_max,
                             const void* q, int q_dtype, const Rows& q_rows, const int32_t* pos0,
                             const int32_t* n_rows, float* out, const Rows& out_rows,
                             int out_planes) {
  if (out_planes && (q_dtype != MB_DT_F32 || !out_rows.row_off || ring.heads != H || out_planes != (ring.bf16 ? 2 : 3)))
    return fail(ctx, MB_ERR_ARG, "attention planes: packed fp32 rows of the model's ring");
  if (q_dtype == MB_DT_BF16 && !ring.bf16)
    return fail(ctx, MB_ERR_ARG, "bf16 queries need a bf16 ring (the bf16 MFMA path)");
  if (B > 65535) return fail(ctx, MB_ERR_ARG, "at most 65535 sequences per prefill call");
  if (B == 0 || rows_max == 0) return MB_OK;
  if ((int64_t)((rows_max + QT - 1) / QT) * ring.heads * B >= INT32_MAX)
    return fail(ctx, MB_ERR_ARG, "too many query tiles in one prefill call");
  const unsigned nh = (unsigned)ring.heads;
  if (q_dtype == MB_DT_BF16)
    hipLaunchKernelGGL(k_flash_bf16<kFlashWaves>,
                       dim3((unsigned)((rows_max + BQ - 1) / BQ), nh, (unsigned)B),
                       dim3(64 * kFlashWaves), 0, ctx->stream, (const uint16_t*)q, q_rows,
                       pos0, n_rows, (const uint16_t*)ring.k, (const uint16_t*)ring.v, ring.sp,
                       ring.seq_stride, ring.C, ring.window, out, out_rows, ctx->xcds,
                       ctx->cus_per_xcd);
  else
    hipLaunchKernelGGL(ring.bf16 ? (out_planes ? k_flash_x<true, 2> : k_flash_x<true, 0>)
                                 : (out_planes ? k_flash_x<false, 3> : k_flash_x<false, 0>),
                       dim3((unsigned)((rows_max + QT - 1) / QT), nh, (unsigned)B), dim3(256), 0,
                       ctx->stream, (const float*)q, q_rows, pos0, n_rows, ring.k, ring.v, ring.sp,
                       ring.seq_stride, ring.C, ring.window, out, out_rows);
  MB_HIP(ctx, hipGetLastError());
  return MB_OK;
}

}  // namespace mb
