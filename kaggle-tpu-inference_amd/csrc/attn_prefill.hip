// Causal prefill attention on MFMA (model.py:195-215 at T > 1).
//
// The prompt's query rows attend the paged K/V cache (written beforehand by
// kv_append): query row t sits at position p0 + t and attends keys
// [lo, p0 + t], lo = max(0, p0 + t + 1 - W) on sliding layers, else 0.
// The reference's rounding points are kept: s = f32(bf16(q . k)) with scale
// 1.0, optional softcap, an f32 softmax over the row, probabilities rounded to
// bf16 after normalisation, ctx = bf16(sum_j p_j v_j) with f32 accumulation
// (model.py:207-213).  So the kernel makes two passes over the keys of a query
// block: pass 1 computes each row's max m and sum l of exp(s - m) (online
// over key blocks); pass 2 recomputes the scores, forms p = bf16(exp(s - m) /
// l) -- exactly the bf16 operand the reference's PV product takes -- and
// accumulates P . V on MFMA.
//
// Block: 128 query rows = 128 / G positions x the G query heads of one KV head
// (the K/V tiles are shared by the group), 4 waves.  The products are taken
// transposed, S^T = K . Q^T and O^T = V^T . P^T, on v_mfma_f32_32x32x16_bf16:
// lane l then holds scores of one query row (column l % 32), so the row max and
// sum are lane-local until the end of pass 1, and the probabilities are already
// in the B operand's order (below).
//
// Operand layout (32x32x16): lane l, half h = l / 32, holds A[l%32][8h..+7]
// and B[8h..+7][l%32] and receives C[8(i/4) + 4h + i%4][l%32], i < 16.  So the
// lane's scores i = 8s .. 8s+7 of a 32-key tile are keys 16s + 8((i%8)/4) + 4h
// + i%4: taken as the B operand of k-step s they stand for those keys in that
// order, and the A operand reads V in the same order: two transposing LDS
// reads (ds_read_b64_tr_b16: each 16 lanes read 4 keys x 16 dims and lane j
// receives dim j of the 4 keys), keys 16s + 4h .. +3 and 16s + 8 + 4h .. +3.
//
// K and V key blocks are staged row-major in a ring of four LDS tiles by direct
// global->LDS loads, requested three tiles ahead.  16-byte slot p of K row r
// holds chunk p ^ (r % 16), 64-byte chunk c of V row r holds chunk c ^ (r % 8),
// so the fragment reads spread over all banks (no conflicts counted).
//
// Who reads what from LDS: scores of 64 rows x 32 keys per wave (at head_dim
// 512 in pass 2 of 32 rows: the 128 x 512 outputs take 256 of a lane's 512
// registers and a second row tile's Q fragments would not fit), so a K fragment
// feeds two MFMAs; P goes through LDS, so that a wave can hold all 128 rows x
// D / 4 dims of O and a V fragment feeds four.  One wave per SIMD: the softmax
// arithmetic and the tile requests are written between the MFMAs of the next
// product (a wave issues an instruction every 4-6 cycles, an MFMA takes 32; 44
// measured on random operands).
//
// Measured (26B-A4B layers, us, before = 16 rows per wave on 16x16x32 with V
// transposed by 2-byte LDS stores): full layer, 4,096 rows: 1,268 -> 414;
// sliding layer, 2,000 rows: 125 -> 63.  At 4,096 rows a 32-key block costs a
// wave 6.9 kcycles of which its 96 MFMAs are 4.3; what bounds the rest is the
// issue of the other instructions of a wave that is alone on its SIMD.
#include <math.h>

#include "capi_util.h"
#include "common.h"

namespace g4mi {

struct PfAttnArgs {
  const uint16_t* q;        // [T, NH, D] normalised + rotated
  const uint16_t* k_pages;  // [num_pages, KV, PAGE, D]
  const uint16_t* v_pages;
  const int32_t* pt;        // page table row [max_pages]
  uint16_t* ctx;            // [T, NH, D]
  int T, NH, KV, G, page, num_pages, max_pages, p0, window;
  float softcap, cap_k;     // cap_k = -2 log2(e) / softcap
  int nqb;   // query blocks per KV head
  int xmap;  // block order: 0 plain, 1 KV divides 8, 2 KV a multiple of 8
};

// Block order.  The launch is a 1-D grid whose blocks the dispatcher hands to
// the 8 XCDs in turn (block b to the XCD of b % 8), and each XCD has its own
// L2.  The query blocks of one KV head read the same K/V rows, so they are
// kept on the XCDs of that head: with KV dividing 8, XCD x serves head
// x % KV and every (8 / KV)-th query block of it (long and short blocks
// alike, so the XCDs finish together); with KV a multiple of 8, XCD x serves
// heads x, x + 8, ...; other head counts take the plain order (block b: head
// b / nqb).  Within a head the query blocks go longest first.  Returns false
// for the padding blocks of the first order.
__device__ __forceinline__ bool pf_block(const PfAttnArgs& a, int& kv, int& qb) {
  const int b = (int)blockIdx.x, x = b & 7, slot = b >> 3;
  int j;
  if (a.xmap == 1) {
    kv = x % a.KV;
    j = x / a.KV + (8 / a.KV) * slot;
  } else if (a.xmap == 2) {
    const int per = a.KV / 8;
    kv = x + 8 * (slot % per);
    j = slot / per;
  } else {
    kv = b / a.nqb;
    j = b % a.nqb;
  }
  qb = a.nqb - 1 - j;
  return j < a.nqb;
}

// ---------------------------------------------------------------- q norm + RoPE
// q = rope(rms_norm(q_raw, q_norm)) in place for T rows of NH heads at
// positions p0 + t (model.py:198-199); grid (T, ceil(NH/4)), wave per head.
// Lane l owns the D/64 consecutive values at l*D/64; the RoPE partner
// (d +- D/2) sits in lane l^32.
template <int D>
__global__ __launch_bounds__(256) void q_norm_rope_kernel(uint16_t* __restrict__ q, const uint16_t* __restrict__ w,
                                                          const uint16_t* __restrict__ cs_tab,
                                                          const uint16_t* __restrict__ sn_tab, int NH, int p0,
                                                          float eps) {
  constexpr int PL = D / 64;
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  const int h = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (h >= NH) return;
  const int so = lane * PL, jo = so % (D / 2);
  const int pos = p0 + t;
  uint16_t* row = q + ((size_t)t * NH + h) * D + so;
  float x[PL], ww[PL], cs[PL], sn[PL];
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    x[i] = bf2f(row[i]);
    ww[i] = bf2f(w[so + i]);
    cs[i] = bf2f(cs_tab[(size_t)pos * (D / 2) + jo + i]);
    sn[i] = bf2f(sn_tab[(size_t)pos * (D / 2) + jo + i]);
  }
  double ss = 0.0;
#pragma unroll
  for (int i = 0; i < PL; ++i) ss = fma((double)x[i], (double)x[i], ss);
  const float r = rms_scale(group_sum_f64<64>(ss), D, eps);
#pragma unroll
  for (int i = 0; i < PL; ++i) x[i] = rbf(x[i] * r * ww[i]);
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const float partner = __shfl_xor(x[i], 32, kWave);
    const float rot = (so + i < D / 2) ? -partner : partner;
    row[i] = f2bf(rbf(rbf(x[i] * cs[i]) + rbf(rot * sn[i])));
  }
}

// ---------------------------------------------------------------- attention
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr int kPfRing = 4;    // K/V tiles in LDS
constexpr int kPfRows = 128;  // query rows per block
// what a tile of an invalid page reads (no tile is larger)
__device__ __align__(16) uint8_t pf_zeros[32768];

constexpr float kLog2e = 0x1.715476p+0f;

// XOR of a K row's 16-byte slots (8 per row at head_dim 64).
template <int D>
__device__ constexpr int pf_kswz(int row) {
  return D >= 128 ? (row & 15) : ((row & 7) ^ ((row >> 3) & 1));
}

// XOR of a V row's 16-byte slots: its 64-byte chunks (D / 32 per row) by row.
template <int D>
__device__ constexpr int pf_vswz(int row) {
  return (row & (D >= 256 ? 7 : D / 32 - 1)) << 2;
}
// Hides a value's origin from the compiler.
__device__ __forceinline__ void opaque(uint32_t& x) { asm volatile("" : "+v"(x)); }
// Pins the computation of a value to this point of the instruction stream
// (volatile asm keeps its order; plain arithmetic may sink to its use).
__device__ __forceinline__ void pinned(float& x) { asm volatile("" : "+v"(x)); }
// pack2 whose halves are unpacked again: left to itself the compiler converts
// each value on its own, with two shifts per value.
__device__ __forceinline__ uint32_t pf_pack(float lo, float hi) {
  uint32_t r = pack2(lo, hi);
  asm("" : "+v"(r));
  return r;
}

// How the four waves of a block (128 query rows) share the work.
//   scores: a wave takes RT row tiles of 32 and one tile of 32 keys.  A staged
//     tile holds SK keys: 64 up to head_dim 256, the two halves of the waves
//     (wave % 2) taking a half each; 32 at 512, where in pass 1 the halves take
//     a tile each (GT tiles per step) and in pass 2 wave w takes row tile w.
//   P . V: a wave takes RTO row tiles x DTO dim tiles, over all SK keys.
template <int D>
struct PfShape {
  static constexpr int SK = (D >= 512) ? 32 : 64;
  static constexpr int TB = SK * D * 2;          // bytes of a staged K or V tile
  static constexpr int CPW = TB / 1024 / 4;      // 1 KB loads per wave and tile
  static constexpr int GT = (D >= 512) ? 2 : 1;  // tiles per pass 1 step
  static constexpr int RT2 = (D >= 512) ? 1 : 2; // row tiles per wave in pass 2's scores
  static constexpr int DW = D / 32 < 4 ? D / 32 : 4;  // dim groups
  static constexpr int DTO = D / 32 / DW;        // dim tiles per wave
  static constexpr int RTO = DW;                 // row tiles per wave: 4 / (4 / DW)
  static constexpr int NKS = SK / 16;            // k-steps of P . V
};

template <int D, bool CAP>
__global__ __launch_bounds__(256) void attn_prefill_kernel(PfAttnArgs a) {
  using P = PfShape<D>;
  constexpr int SK = P::SK, TB = P::TB, CPW = P::CPW, GT = P::GT, RT2 = P::RT2;
  constexpr int DTO = P::DTO, RTO = P::RTO, NKS = P::NKS;
  constexpr int RB = D * 2;      // bytes of a K/V row
  constexpr int KS = D / 16;     // MFMA k-steps over D (scores)
  static_assert(CPW >= 1 && CPW * 4096 == TB && TB <= (int)sizeof(pf_zeros), "tile loads");
  __shared__ __align__(1024) uint8_t tiles[kPfRing][TB];
  __shared__ __align__(16) u32x4 pl[4][NKS][64];  // P^T of a key block: [row tile][k-step][lane], B operands
  __shared__ float stm[2][128], stl[2][128];      // a row's max and sum over each half of the keys
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int h = lane >> 5, col = lane & 31, half = wave & 1;
  int kv, qb;
  if (!pf_block(a, kv, qb)) return;
  const int G = a.G, t0 = qb * (kPfRows / G);

  // row tile rt of the block: the lane's query row is 32 rt + col (rows past T
  // repeat the last position and are not stored)
  auto row_t = [&](int rt) { return min(t0 + (32 * rt + col) / G, a.T - 1); };
  auto row_lo = [&](int pos) { return (a.window > 0) ? max(0, pos + 1 - a.window) : 0; };
  // key range of the block
  const int pos_last = a.p0 + min(t0 + kPfRows / G, a.T) - 1;
  const int kb0 = row_lo(a.p0 + t0) / SK, n = pos_last / SK - kb0 + 1;
  const int n1 = (n + GT - 1) / GT * GT;  // pass 1 tiles (a tile past the last key is all masked)

  // The block's tiles form one stream, used in this order: tile i < n1 is K
  // block kb0 + i (pass 1); then K 0, K 1, V 0, K 2, V 1, ..., K n, V n-1 (pass
  // 2, whose P . V runs one block behind its scores; K n is not used): K g is
  // tile n1 + 2g - 1 (K 0: n1), V g is n1 + 2g + 2.  Tile i lives in ring slot
  // i % 4, requested once tile i - 4 has been used.
  //
  // A walk hands out the addresses of consecutive blocks of K or of V.  The
  // page-table entries of 64 pages sit in a register, one per lane (reloaded
  // when the walk leaves them): no memory access, and no division by the page
  // size, between the tiles.  Blocks past the last page read a page of the row's
  // last entry, an invalid page an array of zeros.
  struct Walk {
    int idx, base;  // page index of the next block, of lane 0's entry
    uint64_t off;   // its byte offset in the page
    int win;        // entry of page base + lane
  };
  const uint64_t page_bytes = (uint64_t)a.page * RB, pool_bytes = page_bytes * a.KV;  // of one head, of a page
  const uint8_t* const kbase = (const uint8_t*)a.k_pages + kv * page_bytes;
  const uint8_t* const vbase = (const uint8_t*)a.v_pages + kv * page_bytes;
  auto window = [&](Walk& w) __attribute__((always_inline)) {
    w.base = w.idx;
    w.win = a.pt[min(w.idx + lane, a.max_pages - 1)];
    asm volatile("" : "+v"(w.win));  // waited for here
  };
  Walk start;
  start.idx = kb0 * SK / a.page;
  start.off = (uint64_t)(kb0 * SK % a.page) * RB;
  window(start);
  auto step = [&](Walk& w, const uint8_t* base) __attribute__((always_inline)) {
    const int pg = __builtin_amdgcn_readlane(w.win, w.idx - w.base);
    const uint8_t* src = base + (uint64_t)(uint32_t)pg * pool_bytes + w.off;
    if ((uint32_t)pg >= (uint32_t)a.num_pages) src = pf_zeros;
    w.off += TB;
    if (w.off == page_bytes) {
      w.off = 0;
      if (++w.idx == w.base + 64) window(w);
    }
    return src;
  };
  // A tile's request: CPW direct global->LDS loads of 1 KB per wave, in LDS
  // order (M0 = LDS address; the instruction's offset moves both addresses).
  // The lane's 16 bytes of load j are LDS bytes (wave * CPW + j) * 1024 + lane *
  // 16, that is slot p0 of row r0 + j * 1024 / RB; the swizzle of that row is
  // r0's XOR a constant of j.  Inline asm: the compiler sees no LDS writer; the
  // waits are explicit (`landed`).
  struct Request {
    const uint8_t* src;
    uint32_t lds;
  };
  const int o0 = wave * CPW * 1024 + lane * 16, r0 = o0 / RB, p0 = (o0 % RB) / 16;
  const uint32_t xk = (uint32_t)(p0 ^ pf_kswz<D>(r0)) * 16u + (uint32_t)(r0 * RB);
  const uint32_t xv = (uint32_t)(p0 ^ pf_vswz<D>(r0)) * 16u + (uint32_t)(r0 * RB);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)tiles[0] + wave * CPW * 1024);
  auto load = [&](auto is_v, const Request& q, auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value, dr = j * 1024 / RB;
    constexpr uint32_t dx = (uint32_t)(decltype(is_v)::value ? pf_vswz<D>(dr) : pf_kswz<D>(dr)) * 16u;
    const uint32_t x = decltype(is_v)::value ? xv : xk, l = q.lds + j / 4 * 4096;
    const uint8_t* sp = q.src + j / 4 * 4096;
    uint32_t vo;
    asm volatile("s_mov_b32 m0, %2\n\tv_xor_b32 %0, %4, %1\n\tglobal_load_lds_dwordx4 %0, %3 offset:%5"
                 : "=&v"(vo)
                 : "v"(x), "s"(l), "s"(sp), "n"(dx), "n"(j % 4 * 1024)
                 : "memory", "m0");
  };
  uint32_t ntile = 0;  // tiles requested
  Walk wk = start, wv = start;
  auto next_k = [&]() __attribute__((always_inline)) {
    if (ntile == (uint32_t)n1) wk = start;  // pass 2 starts over
    Request q;
    q.src = step(wk, kbase);
    q.lds = lds0 + (ntile++ & (kPfRing - 1)) * TB;
    return q;
  };
  auto next_v = [&]() __attribute__((always_inline)) {
    Request q;
    q.src = step(wv, vbase);
    q.lds = lds0 + (ntile++ & (kPfRing - 1)) * TB;
    return q;
  };
  auto loads = [&](auto is_v, const Request& q) __attribute__((always_inline)) {
    static_for<CPW>([&](auto jc) __attribute__((always_inline)) { load(is_v, q, jc); });
  };
  using IsK = std::false_type;
  using IsV = std::true_type;
  // This wave's loads landed except those of the latest AHEAD tiles, and its
  // LDS accesses are done; then the barrier.
  auto landed = [&](auto ahead) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(decltype(ahead)::value* CPW) : "memory");
  };
  using Two = std::integral_constant<int, 2>;
  using None = std::integral_constant<int, 0>;

  // S^T of 32 keys (rows krow0 .. of the tile at kt) x R row tiles (fragments
  // q), with side(MFMA index) after each MFMA: independent work that runs while
  // the MFMA does (a wave alone on its SIMD issues an instruction every 4-6
  // cycles, an MFMA takes 32).  K chunk 2 st + h of row krow sits in slot (2 st
  // + h) ^ ksw: at the row's first slot's address XOR 32 (st % 8), plus 256 (st /
  // 8).  A ring of RQ fragments keeps RQ - 1 LDS reads ahead of the MFMAs.
  constexpr int RQ = 4;
  auto scores = [&](const uint8_t* kt, int krow0, auto& q, auto& acc, auto side) __attribute__((always_inline)) {
    constexpr int R = sizeof(acc) / sizeof(acc[0]);
#pragma unroll
    for (int rt = 0; rt < R; ++rt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[rt][i] = 0.0f;
    const int krow = krow0 + col;
    uint32_t ka = (uint32_t)(krow * RB + ((h ^ pf_kswz<D>(krow)) * 16));
    opaque(ka);
    u32x4 kf[RQ];
    auto read = [&](auto sc) __attribute__((always_inline)) {
      constexpr int st = decltype(sc)::value;
      kf[st % RQ] = *(const u32x4*)(kt + (ka ^ (32u * (st % 8))) + 256 * (st / 8));
    };
    static_for<RQ - 1>([&](auto sc) __attribute__((always_inline)) { read(sc); });
    static_for<KS>([&](auto sc) __attribute__((always_inline)) {
      constexpr int st = decltype(sc)::value;
      if constexpr (st + RQ - 1 < KS) read(std::integral_constant<int, st + RQ - 1>{});
      static_for<R>([&](auto rc) __attribute__((always_inline)) {
        constexpr int rt = decltype(rc)::value;
        __builtin_amdgcn_sched_barrier(0);
        acc[rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[st % RQ]),
                                                          __builtin_bit_cast(bf16x8, q[rt][st]), acc[rt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        side(std::integral_constant<int, st * R + rt>{});
      });
    });
  };
  // runs units [i * NU / NM, (i + 1) * NU / NM) of NU after MFMA i of NM
  auto spread = [&](auto nu, auto nm, auto ic, auto unit) __attribute__((always_inline)) {
    constexpr int NU = decltype(nu)::value, NM = decltype(nm)::value, i = decltype(ic)::value;
    constexpr int u0 = i * NU / NM, u1 = (i + 1) * NU / NM;
    static_for<u1 - u0>([&](auto uc) __attribute__((always_inline)) {
      unit(std::integral_constant<int, u0 + decltype(uc)::value>{});
    });
  };
  auto nothing = [](auto) __attribute__((always_inline)) {};
  // s = f32(bf16(q . k)) of a pair of scores (with CAP this is done by `edge`)
  auto rounded = [&](float s0, float s1, float& r0, float& r1) __attribute__((always_inline)) {
    if constexpr (CAP) {
      r0 = s0;
      r1 = s1;
    } else {
      const uint32_t w = pf_pack(s0, s1);
      r0 = bf_lo(w);
      r1 = bf_hi(w);
    }
  };
  // softcap (cap * tanh(s / cap), tanh |y| = (1 - e) / (1 + e), e = exp(-2 |y|)),
  // and -inf for the keys of the 32 from kb outside [lo, pos] of the lane's row;
  // pos0 and lo1 are the first position and the last lo of the row tile
  auto edge = [&](f32x16& s, int kb, int pos, int pos0, int lo1) __attribute__((always_inline)) {
    if constexpr (CAP) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float x = rbf(s[i]), e = __builtin_amdgcn_exp2f(fabsf(x) * a.cap_k);
        s[i] = copysignf(a.softcap * ((1.0f - e) * __builtin_amdgcn_rcpf(1.0f + e)), x);
      }
    }
    if (kb < lo1 || kb + 31 > pos0) {  // wave-uniform: some row of the tile does not attend all 32
      const int lo = row_lo(pos);
#pragma unroll
      for (int i = 0; i < 16; ++i)  // key kb + 4h + 8(i/4) + i%4
        s[i] = ((uint32_t)(kb + 4 * h - lo + 8 * (i >> 2) + (i & 3)) <= (uint32_t)(pos - lo)) ? s[i] : -INFINITY;
    }
  };

  // ---- pass 1: the lane's max m and sum l of exp(s - m) over its keys, for the
  // two row tiles 2 (wave / 2) + rt.  A block's statistics are taken while the
  // next block's scores are computed, in 17 parts per tile: 8 pairs rounded into
  // the max, the rescale, 8 pairs of exps.
  const int rt0 = wave & 2;
  // Q goes through LDS too (whole rows per load; a fragment load from memory
  // touches 32 rows): up to head_dim 256 beside K tiles 0 and 1, in the place of
  // tiles 2 and 3; at 512 its 128 KB come first.
  constexpr int QB = kPfRows * RB;  // bytes of the block's query rows
  constexpr bool kFirst = QB <= 2 * TB;
  static_assert(QB == (kFirst ? 2 : kPfRing) * TB, "query rows in the ring");
  uint8_t* const qs = kFirst ? tiles[2] : tiles[0];
  if constexpr (kFirst) {
    loads(IsK{}, next_k());
    loads(IsK{}, next_k());
  }
  static_for<QB / 4096>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    const int o = (wave * (QB / 4096) + j) * 1024 + lane * 16, r = o / RB, ch = (o % RB / 16) ^ pf_kswz<D>(r);
    const int tc = min(t0 + r / G, a.T - 1);
    const uint16_t* src = a.q + ((size_t)tc * a.NH + kv * G + r % G) * D + 8 * ch;
    const uint32_t l = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)qs) + (wave * (QB / 4096) + j) * 1024;
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(l) : "memory", "m0");
  });
  landed(None{});
  u32x4 qf[2][KS];  // B fragments of Q^T: k-step st holds dims 16 st + 8h .. +7
  int pos1[2], first1[2], lo1[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int r = 32 * (rt0 + rt) + col;
    const uint8_t* qrow = qs + r * RB;
#pragma unroll
    for (int st = 0; st < KS; ++st) qf[rt][st] = *(const u32x4*)(qrow + ((2 * st + h) ^ pf_kswz<D>(r)) * 16);
    pos1[rt] = a.p0 + row_t(rt0 + rt);
    first1[rt] = a.p0 + min(t0 + 32 * (rt0 + rt) / G, a.T - 1);
    lo1[rt] = row_lo(a.p0 + min(t0 + (32 * (rt0 + rt) + 31) / G, a.T - 1));
  }
  lds_barrier();  // every wave has its fragments
  if constexpr (!kFirst) {
    loads(IsK{}, next_k());
    loads(IsK{}, next_k());
  }
  float m[2], l[2], mm[2], mx[2];
  f32x16 s[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    m[rt] = -INFINITY;
    l[rt] = mm[rt] = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[rt][i] = -INFINITY;
  }
  auto stats = [&](auto uc) __attribute__((always_inline)) {
    constexpr int rt = decltype(uc)::value / 17, u = decltype(uc)::value % 17;
    if constexpr (u < 8) {
      float r0, r1;
      rounded(s[rt][2 * u], s[rt][2 * u + 1], r0, r1);
      s[rt][2 * u] = r0;
      s[rt][2 * u + 1] = r1;
      mx[rt] = fmaxf(fmaxf(u == 0 ? m[rt] : mx[rt], r0), r1);
      pinned(mx[rt]);
    } else if constexpr (u == 8) {
      mm[rt] = (mx[rt] == -INFINITY) ? 0.0f : mx[rt];  // no key yet: every exp2 below is exp2(-inf) = 0
      l[rt] *= __builtin_amdgcn_exp2f((m[rt] - mm[rt]) * kLog2e);
      m[rt] = mx[rt];
      pinned(l[rt]);
    } else {
      l[rt] += __builtin_amdgcn_exp2f((s[rt][2 * (u - 9)] - mm[rt]) * kLog2e);
      l[rt] += __builtin_amdgcn_exp2f((s[rt][2 * (u - 9) + 1] - mm[rt]) * kLog2e);
      pinned(l[rt]);
    }
  };
  using NStats = std::integral_constant<int, 34>;
  using NScores1 = std::integral_constant<int, 2 * KS>;
  // after the scores of pass 1 step g: the masked scores become the next step's s
  auto keep = [&](f32x16 (&acc)[2], int g) __attribute__((always_inline)) {
    const int kb = GT == 2 ? (kb0 + 2 * g + half) * SK : (kb0 + g) * SK + 32 * half;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      edge(acc[rt], kb, pos1[rt], first1[rt], lo1[rt]);
      s[rt] = acc[rt];
    }
  };
  // loads of tiles q[0] .. spread over the first MFMAs, the statistics over all
  auto side1 = [&](auto is_v, const auto& q, auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value, nt = sizeof(q) / sizeof(q[0]);
    if constexpr (i < nt * CPW) load(is_v, q[i / CPW], std::integral_constant<int, i % CPW>{});
    spread(NStats{}, NScores1{}, ic, stats);
  };
  if constexpr (GT == 1) {
    loads(IsK{}, next_k());
    f32x16 acc[2];
    for (int g = 0; g + 1 < n; ++g) {
      landed(Two{});
      const Request q[1] = {next_k()};
      scores(tiles[g & (kPfRing - 1)], 32 * half, qf, acc,
             [&](auto ic) __attribute__((always_inline)) { side1(IsK{}, q, ic); });
      keep(acc, g);
    }
    landed(Two{});
    const Request q[1] = {next_v()};  // V 0
    scores(tiles[(n - 1) & (kPfRing - 1)], 32 * half, qf, acc,
           [&](auto ic) __attribute__((always_inline)) { side1(IsV{}, q, ic); });
    keep(acc, n - 1);
  } else {
    for (int g = 0; g < n1 / 2; ++g) {
      landed(None{});
      Request q[2];
      q[0] = next_k();
      q[1] = next_k();
      f32x16 acc[2];
      scores(tiles[(2 * g + half) & (kPfRing - 1)], 0, qf, acc,
             [&](auto ic) __attribute__((always_inline)) { side1(IsK{}, q, ic); });
      keep(acc, g);
    }
  }
  static_for<34>(stats);
  // the row's max and sum: the lane halves, then the key halves through LDS
  auto merge = [](float& m, float& l, float m2, float l2) {
    const float mn = fmaxf(m, m2), mm = (mn == -INFINITY) ? 0.0f : mn;
    l = l * __builtin_amdgcn_exp2f((m - mm) * kLog2e) + l2 * __builtin_amdgcn_exp2f((m2 - mm) * kLog2e);
    m = mn;
  };
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    merge(m[rt], l[rt], __shfl_xor(m[rt], 32, kWave), __shfl_xor(l[rt], 32, kWave));
    if (h == 0) {
      stm[half][32 * (rt0 + rt) + col] = m[rt];
      stl[half][32 * (rt0 + rt) + col] = l[rt];
    }
  }
  lds_barrier();  // (every wave is past its pass 1 tiles)
  if constexpr (GT == 2) loads(IsV{}, next_v());  // V 0

  // ---- pass 2: p = bf16(exp(s - m) / l) = bf16(2^((s - m) log2 e - log2 l)), O^T += V^T . P^T.
  // Scores of row tiles r2 + rt; P of a key block goes through LDS.
  const int r2 = RT2 == 2 ? rt0 : wave;
  float mrow[RT2], lg[RT2];
  int pos2[RT2], first2[RT2], lo2[RT2];
#pragma unroll
  for (int rt = 0; rt < RT2; ++rt) {
    const int r = 32 * (r2 + rt) + col;
    float mr = stm[0][r], lr = stl[0][r];
    merge(mr, lr, stm[1][r], stl[1][r]);
    mrow[rt] = (mr == -INFINITY) ? 0.0f : mr;
    lg[rt] = (lr == 0.0f) ? INFINITY : __builtin_amdgcn_logf(lr);  // log2; a row without keys: p = 0
    if constexpr (RT2 == 2) {
      pos2[rt] = pos1[rt];
      first2[rt] = first1[rt];
      lo2[rt] = lo1[rt];
    } else {  // row tile `wave` is this wave's pass 1 tile `half`
      pos2[rt] = half ? pos1[1] : pos1[0];
      first2[rt] = half ? first1[1] : first1[0];
      lo2[rt] = half ? lo1[1] : lo1[0];
#pragma unroll
      for (int st = 0; st < KS; ++st) qf[0][st] = half ? qf[1][st] : qf[0][st];
    }
  }
  const int key2 = RT2 == 2 ? 32 * half : 0;  // this wave's keys of a tile
  const int dg = wave % P::DW, rw = wave / P::DW * RTO;  // dim group, first row tile of P . V
  f32x16 o[RTO][DTO];
#pragma unroll
  for (int rt = 0; rt < RTO; ++rt)
#pragma unroll
    for (int dt = 0; dt < DTO; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[rt][dt][i] = 0.0f;
  // transposed reads: lane (group q = lane / 16, j = lane % 16) reads 4 dims
  // from 32 dt + 16 (q & 1) + 4 (j & 3) of key 16 ks + 8 x + 4 (q >> 1) + j / 4
  const int vkey = 4 * (lane >> 5) + ((lane & 15) >> 2);  // key % 8
  const uint32_t voff = (uint32_t)(vkey * RB + 16 * pf_vswz<D>(vkey) + 32 * ((lane >> 4) & 1) + 8 * (lane & 3)) ^
                        (uint32_t)(64 * DTO * dg % 512);
  // P . V of the block in pl and vt: per (k-step, dim tile) one V fragment and
  // RTO MFMAs, the next fragments' LDS reads one such group ahead; side after
  // each MFMA
  constexpr int NPV = NKS * DTO * RTO;
  auto accumulate = [&](const uint8_t* vt, auto side) __attribute__((always_inline)) {
    uint32_t va = voff;
    opaque(va);
    const uint8_t* vb = vt + 64 * DTO * dg / 512 * 512;
    s16x8 vf[2];
    u32x4 pf[2][RTO];
    auto read_v = [&](auto uc) __attribute__((always_inline)) {  // group u = ks * DTO + dt
      constexpr int u = decltype(uc)::value, ks = u / DTO, dt = u % DTO;
      const uint8_t* p = vb + (va ^ (64u * (dt % 8))) + 16 * ks * RB;
      const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
      const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 8 * RB));
      vf[u % 2] = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto read_p = [&](auto kc) __attribute__((always_inline)) {
      constexpr int ks = decltype(kc)::value;
#pragma unroll
      for (int rt = 0; rt < RTO; ++rt) pf[ks % 2][rt] = pl[rw + rt][ks][lane];
    };
    read_p(std::integral_constant<int, 0>{});
    read_v(std::integral_constant<int, 0>{});
    static_for<NKS * DTO>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value, ks = u / DTO, dt = u % DTO;
      if constexpr (u + 1 < NKS * DTO) read_v(std::integral_constant<int, u + 1>{});
      if constexpr (dt == DTO - 1 && ks + 1 < NKS) read_p(std::integral_constant<int, ks + 1>{});
      static_for<RTO>([&](auto rc) __attribute__((always_inline)) {
        constexpr int rt = decltype(rc)::value;
        __builtin_amdgcn_sched_barrier(0);
        o[rt][dt] =
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf[u % 2]),
                                                    __builtin_bit_cast(bf16x8, pf[ks % 2][rt]), o[rt][dt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        side(std::integral_constant<int, u * RTO + rt>{});
      });
    });
  };
  // unit 8 rt + u: the probabilities of scores 2u, 2u + 1 of row tile rt as word
  // u of its B operands
  f32x16 acc[RT2];
  u32x4 pb[RT2][2];
  auto prob = [&](auto uc) __attribute__((always_inline)) {
    constexpr int rt = decltype(uc)::value / 8, u = decltype(uc)::value % 8;
    float r0, r1;
    rounded(acc[rt][2 * u], acc[rt][2 * u + 1], r0, r1);
    uint32_t w = pack2(__builtin_amdgcn_exp2f(__builtin_fmaf(r0 - mrow[rt], kLog2e, -lg[rt])),
                       __builtin_amdgcn_exp2f(__builtin_fmaf(r1 - mrow[rt], kLog2e, -lg[rt])));
    opaque(w);  // pinned here
    pb[rt][u / 4][u % 4] = w;
  };
  using NProb = std::integral_constant<int, 8 * RT2>;
  auto block_scores = [&](uint32_t tile, int g, auto side) __attribute__((always_inline)) {
    scores(tiles[tile & (kPfRing - 1)], key2, qf, acc, side);
#pragma unroll
    for (int rt = 0; rt < RT2; ++rt) edge(acc[rt], (kb0 + g) * SK + key2, pos2[rt], first2[rt], lo2[rt]);
  };
  // (k-step 2 * (key2 / 32) + x of the tile)
  auto put_p = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < RT2; ++rt)
#pragma unroll
      for (int x = 0; x < 2; ++x) pl[r2 + rt][(RT2 == 2 ? 2 * half : 0) + x][lane] = pb[rt][x];
  };
  // block 0's scores (tile n1); tile n1 + 3 is K 2
  landed(Two{});
  {
    const Request q = next_k();
    block_scores(n1, 0, [&](auto ic) __attribute__((always_inline)) {
      if constexpr (decltype(ic)::value < CPW) load(IsK{}, q, ic);
    });
  }
  static_for<8 * RT2>(prob);
  for (int g = 1; g < n; ++g) {
    const uint32_t i = n1 + 2 * g - 1;  // K g; V g - 1 is tile i + 1
    landed(Two{});                      // (and every wave is done with block g - 2's P)
    put_p();
    const Request qv = next_v();        // V g, tile i + 3
    block_scores(i, g, [&](auto ic) __attribute__((always_inline)) {
      if constexpr (decltype(ic)::value < CPW) load(IsV{}, qv, ic);
    });
    landed(Two{});
    const Request qk = next_k();        // K g + 2, tile i + 4
    accumulate(tiles[(i + 1) & (kPfRing - 1)], [&](auto ic) __attribute__((always_inline)) {
      if constexpr (decltype(ic)::value < CPW) load(IsK{}, qk, ic);
      spread(NProb{}, std::integral_constant<int, NPV>{}, ic, prob);
    });
  }
  lds_barrier();  // every wave is done with the last P but one
  put_p();
  landed(None{});  // V n - 1, tile n1 + 2n (and what was requested after it)
  accumulate(tiles[(n1 + 2 * n) & (kPfRing - 1)], nothing);

  // ---- ctx = bf16(O), through LDS (rows of 16-byte slots, slot p of row r holds
  // chunk p ^ ksw(r)): whole rows per store
  lds_barrier();  // every wave is done with the tiles
  uint8_t* const os = tiles[0];
#pragma unroll
  for (int rt = 0; rt < RTO; ++rt) {
    const int r = 32 * (rw + rt) + col;
#pragma unroll
    for (int dt = 0; dt < DTO; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint2 w;
        w.x = pack2(o[rt][dt][4 * q], o[rt][dt][4 * q + 1]);
        w.y = pack2(o[rt][dt][4 * q + 2], o[rt][dt][4 * q + 3]);
        *(uint2*)(os + r * RB + ((4 * (DTO * dg + dt) + q) ^ pf_kswz<D>(r)) * 16 + 8 * h) = w;
      }
  }
  lds_barrier();
#pragma unroll 4
  for (int j = 0; j < QB / 4096; ++j) {
    const int b = (wave * (QB / 4096) + j) * 1024 + lane * 16, r = b / RB, ch = (b % RB / 16) ^ pf_kswz<D>(r);
    const int t = t0 + r / G;
    if (t >= a.T) continue;
    uint16_t* dst = a.ctx + ((size_t)t * a.NH + kv * G + r % G) * D + 8 * ch;
    const u32x4 v = *(const u32x4*)(os + b);
    if (((uintptr_t)a.ctx & 15u) == 0) {
      *(u32x4*)dst = v;
    } else {  // (ctx need not be aligned)
#pragma unroll
      for (int i = 0; i < 8; ++i) dst[i] = (uint16_t)(v[i / 2] >> (16 * (i & 1)));
    }
  }
}

// ---------------------------------------------------------------- few keys
// head_dim 512 while no row attends more than kPfFewKeys keys: 64 rows per block,
// 16 per wave on v_mfma_f32_16x16x32_bf16 with plain fragment loads of Q.  A
// block then has at most three key steps and its time is its chain of memory
// round trips, of which the kernel above has more (Q through LDS, then the tile
// ring): 17 rows 12.2 against 18.4 us, 54 rows 16.9 against 20.2, 96 rows 21.7
// against 23.8, 112 rows 26.3 against 25.7.  K is staged as [key][D], V
// transposed to [D][key].
constexpr int kPfFewKeys = 96;

// max / sum over the 16 lanes of a DPP row (the 16 key columns of a tile row).
// The max is one v_max_f32 with a DPP operand per round (fmaxf on a DPP move
// would add a move and two canonicalising maxes; the scores hold no NaN); the
// s_nop gives the two wait states a DPP read of a just-written VGPR needs.
template <int CTRL>
__device__ __forceinline__ float dpp_max_f(float v) {
  float r;
  if constexpr (CTRL == kDppXor1)
    asm("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(v));
  else if constexpr (CTRL == kDppXor2)
    asm("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(v));
  else if constexpr (CTRL == kDppHalfMirror)
    asm("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(v));
  else
    asm("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 row_mirror row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(v));
  return r;
}
__device__ __forceinline__ float row16_max(float v) {
  v = dpp_max_f<kDppXor1>(v);
  v = dpp_max_f<kDppXor2>(v);
  v = dpp_max_f<kDppHalfMirror>(v);
  v = dpp_max_f<kDppMirror>(v);
  return v;
}
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_f<kDppXor1>(v);
  v += dpp_f<kDppXor2>(v);
  v += dpp_f<kDppHalfMirror>(v);
  v += dpp_f<kDppMirror>(v);
  return v;
}

// p = bf16(e / l) from the reciprocal rl = rcp(l): e * rl lies within 3.5 f32
// ulps of the rounded quotient (rcp within 1 ulp, the product's rounding), so
// it rounds to the same bf16 unless it sits within 8 ulps of a bf16 rounding
// midpoint (low 16 bits 0x7ff8..0x8008); those take the IEEE division.
__device__ __forceinline__ bool near_bf16_midpoint(float x) {
  return ((__float_as_uint(x) - 0x7ff8u) & 0xffffu) <= 16u;
}

template <int G, bool CAP>
__global__ __launch_bounds__(256) void attn_prefill_few_kernel(PfAttnArgs a) {
  constexpr int D = 512;
  constexpr int NW = 4;                     // waves
  constexpr int NTH = 64 * NW;              // threads
  constexpr int ROWS = 16 * NW;             // query rows per block
  constexpr int KB = 32;                    // keys per block step (divides the page)
  constexpr int QP = ROWS / G;              // positions per block
  constexpr int KS = D / 32;                // MFMA k-steps over D (scores)
  constexpr int NT = KB / 16;               // key tiles per step
  constexpr int DT = D / 16;                // output d tiles
  constexpr int LDK = D + 8;                // K row stride in LDS (elements)
  constexpr int LDV = KB + 8;               // V^T row stride
  constexpr int LDP = KB + 8;               // P row stride
  // the K/V tiles are double-buffered: the next step's rows go to the other
  // buffer while this one is read (151 KB of LDS)
  constexpr int NBUF = 2;
  constexpr int kPtl = kPfFewKeys / 64 + 1;  // pages the keys span at most
  __shared__ __align__(16) uint16_t kt[NBUF][KB * LDK];
  __shared__ __align__(16) uint16_t vt[NBUF][D * LDV];
  __shared__ __align__(16) uint16_t pt[ROWS * LDP];
  __shared__ int ptl[kPtl];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  int kv, qb;
  if (!pf_block(a, kv, qb)) return;
  const int t0 = qb * QP;
  const int fr = lane & 15, fk = (lane >> 4) * 8;

  // this lane's rows in the C layout: r = 16*wave + 4*(lane/16) + i
  int rpos[4];
  bool rvalid[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * wave + 4 * (lane >> 4) + i;
    const int t = t0 + r / G;
    rvalid[i] = t < a.T;
    rpos[i] = a.p0 + min(t, a.T - 1);
  }
  // A fragments of Q: row 16*wave + fr (position t0 + row/G, head kv*G + row%G)
  u32x4 qf[KS];
  {
    const int r = 16 * wave + fr;
    const int t = min(t0 + r / G, a.T - 1);
    const uint16_t* qrow = a.q + ((size_t)t * a.NH + kv * G + r % G) * D + fk;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = ld16((const u32x4*)(qrow + 32 * s));
  }
  // key range of the block
  const int pos_first = a.p0 + t0, pos_last = a.p0 + min(t0 + QP, a.T) - 1;
  const int k_lo = (a.window > 0) ? max(0, pos_first + 1 - a.window) : 0;
  const int kb0 = k_lo / KB, kb1 = pos_last / KB;
  const float cap = a.softcap;
  // key block kb is interior when every row of the block attends all its keys
  // (no mask, no -inf score); the others (the diagonal, the window's start)
  // take the masked steps
  const int lo_max = (a.window > 0) ? max(0, pos_last + 1 - a.window) : 0;
  auto interior = [&](int kb) { return kb * KB >= lo_max && kb * KB + KB - 1 <= pos_first; };
  using Edge = std::true_type;
  using Inner = std::false_type;

  // the block's page-table entries, staged once (a barrier follows before use)
  const int first_pg = (kb0 * KB) / a.page;
  for (int i = tid; i < kPtl; i += NTH) ptl[i] = a.pt[min(first_pg + i, a.max_pages - 1)];
  auto page_of = [&](int kb) { return ptl[(kb * KB) / a.page - first_pg]; };
  // K (and V) rows of key block kb into registers (fetch), then into LDS
  // (put); invalid pages read as zero.  The loads are unconditional (page 0
  // stands in for an invalid entry) and the zero is selected afterwards.
  constexpr int CPT = KB * D / 8 / NTH;  // 16-byte chunks per thread and tile
  static_assert(CPT >= 1 && CPT * NTH * 8 == KB * D, "tile chunks");
  struct Tile {
    u32x4 k[CPT], v[CPT];
    bool ok;
  };
  auto fetch = [&](int kb, bool with_v, Tile& T) {
    const int k0 = kb * KB;
    const int pg = page_of(kb);
    T.ok = pg >= 0 && pg < a.num_pages;
    const size_t base = (((size_t)(T.ok ? pg : 0) * a.KV + kv) * a.page + (k0 % a.page)) * D;
#pragma unroll
    for (int i = 0; i < CPT; ++i) T.k[i] = ld16((const u32x4*)(a.k_pages + base) + tid + NTH * i);
    if (with_v) {
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int c = tid + NTH * i, j = c % KB, d0 = (c / KB) * 8;
        T.v[i] = ld16((const u32x4*)(a.v_pages + base + (size_t)j * D + d0));
      }
    }
  };
  auto put = [&](const Tile& T, bool with_v, int buf) {
    uint16_t* kw = kt[buf];
    uint16_t* vw = vt[buf];
    const u32x4 z = {0u, 0u, 0u, 0u};
    // K: lanes walk a key row (conflict-free 16-byte stores)
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + NTH * i, j = c / (D / 8), d0 = (c % (D / 8)) * 8;
      *(u32x4*)(kw + j * LDK + d0) = T.ok ? T.k[i] : z;
    }
    // V transposed: lanes walk the keys of one 8-value column group, so the
    // 2-byte LDS stores of a wave land in consecutive halfwords
    if (with_v) {
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int c = tid + NTH * i, j = c % KB, d0 = (c / KB) * 8;
        const u32x4 v4 = T.ok ? T.v[i] : z;
        const uint32_t w[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vw[(d0 + 2 * e) * LDV + j] = (uint16_t)(w[e] & 0xffffu);
          vw[(d0 + 2 * e + 1) * LDV + j] = (uint16_t)(w[e] >> 16);
        }
      }
    }
  };
  // scores of this wave's 16 rows x KB keys: s[n][i] = row 4(l/16)+i, key k0 + 16n + l%16
  auto scores = [&](int kb, float (*s)[4], auto edge, int buf) {
    const int k0 = kb * KB;
    const uint16_t* kr = kt[buf];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int st = 0; st < KS; ++st) {
        const u32x4 b = *(const u32x4*)(kr + (16 * n + fr) * LDK + 32 * st + fk);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, qf[st]),
                                                      __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
      }
      const int j = k0 + 16 * n + fr;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float sv = rbf(acc[i]);
        if constexpr (CAP) sv = tanhf(sv / cap) * cap;
        if constexpr (decltype(edge)::value) {
          const int lo = (a.window > 0) ? max(0, rpos[i] + 1 - a.window) : 0;
          s[n][i] = (j >= lo && j <= rpos[i]) ? sv : -INFINITY;
        } else {
          s[n][i] = sv;
        }
      }
    }
  };

  // Pass 1 (row max and sum of exp), then pass 2 (p = bf16(exp(s - m) / l),
  // O += P . V), each step's K/V rows requested one step ahead (pass 2's
  // first tile during pass 1's last step).  Step q < n is pass 1 over key
  // block kb0 + q, step n + q pass 2 over the same block. 
  const int n = kb1 - kb0 + 1;
  auto target = [&](int q, Tile& T) {  // request step q's rows (no-op past the last step)
    if (q < 2 * n) fetch(kb0 + (q < n ? q : q - n), q >= n, T);
  };
  float m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m[i] = -INFINITY;
    l[i] = 0.0f;
  }
  // Step g (pass 1: g = q, pass 2: g = n + q) reads buffer g % 2, stores step g +
  // 1's rows (requested one step earlier) into the other buffer, requests step g
  // + 2's, and ends at the barrier that makes them visible (and frees buffer g %
  // 2 for step g + 2).
  auto stage = [&](int g, Tile& T) {
    if (g + 1 < 2 * n) put(T, g + 1 >= n, (g + 1) & 1);
    target(g + 2, T);
  };
  auto step1 = [&](int q, Tile& T, auto edge) {
    stage(q, T);
    float s[NT][4];
    scores(kb0 + q, s, edge, q % NBUF);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float bm = s[0][i];
#pragma unroll
      for (int n = 1; n < NT; ++n) bm = fmaxf(bm, s[n][i]);
      bm = row16_max(bm);
      const float mn = fmaxf(m[i], bm);
      float e = 0.0f;
      if constexpr (decltype(edge)::value) {
        if (mn != -INFINITY) {
#pragma unroll
          for (int n = 0; n < NT; ++n) e += (s[n][i] == -INFINITY) ? 0.0f : exp_nonpos(s[n][i] - mn);
        }
      } else {
#pragma unroll
        for (int n = 0; n < NT; ++n) e += exp_nonpos(s[n][i] - mn);
      }
      e = row16_sum(e);
      // rescale the sum when the max moved (exp(0) = 1 leaves it as it is)
      if (m[i] == -INFINITY)
        l[i] = e;
      else if (m[i] != mn)
        l[i] = l[i] * exp_nonpos(m[i] - mn) + e;
      else
        l[i] += e;
      m[i] = mn;
    }
    lds_barrier();
  };
  Tile tile;
  lds_barrier();  // ptl
  target(0, tile);
  put(tile, false, 0);  // step 0 is a pass-1 step (n >= 1)
  target(1, tile);
  lds_barrier();
  {
    int q = 0;
    for (; q < n && !interior(kb0 + q); ++q) step1(q, tile, Edge{});
    for (; q < n && interior(kb0 + q); ++q) step1(q, tile, Inner{});
    for (; q < n; ++q) step1(q, tile, Edge{});
  }

  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  uint16_t* pw = pt + 16 * wave * LDP;  // this wave's 16 rows of P
  float rl[4];                          // 1 / l (0 for a row without keys)
#pragma unroll
  for (int i = 0; i < 4; ++i) rl[i] = (l[i] > 0.0f) ? __builtin_amdgcn_rcpf(l[i]) : 0.0f;
  auto step2 = [&](int q, Tile& T, auto edge) {
    const int g = n + q, buf = g % NBUF;
    stage(g, T);
    float s[NT][4];
    scores(kb0 + q, s, edge, buf);
    // p = bf16(exp(s - m) / l), 0 for a masked key or a row without keys
#pragma unroll
    for (int nn = 0; nn < NT; ++nn)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float e;
        if constexpr (decltype(edge)::value)
          e = (s[nn][i] == -INFINITY) ? 0.0f : exp_nonpos(s[nn][i] - m[i]);
        else
          e = exp_nonpos(s[nn][i] - m[i]);
        float p = e * rl[i];
        if (near_bf16_midpoint(p)) p = e / l[i];
        pw[(4 * (lane >> 4) + i) * LDP + 16 * nn + fr] = f2bf(p);
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int st = 0; st < KB / 32; ++st) {
      const u32x4 pa = *(const u32x4*)(pw + fr * LDP + 32 * st + fk);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const u32x4 vb = *(const u32x4*)(vt[buf] + (16 * dt + fr) * LDV + 32 * st + fk);
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pa),
                                                        __builtin_bit_cast(bf16x8, vb), o[dt], 0, 0, 0);
      }
    }
    lds_barrier();
  };
  {
    int q = 0;
    for (; q < n && !interior(kb0 + q); ++q) step2(q, tile, Edge{});
    for (; q < n && interior(kb0 + q); ++q) step2(q, tile, Inner{});
    for (; q < n; ++q) step2(q, tile, Edge{});
  }

  // ---- ctx = bf16(O): row 4(l/16)+i of the wave, d = 16*dt + l%16
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (!rvalid[i]) continue;
    const int r = 16 * wave + 4 * (lane >> 4) + i;
    uint16_t* out = a.ctx + ((size_t)(t0 + r / G) * a.NH + kv * G + r % G) * D + fr;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) out[16 * dt] = f2bf(o[dt][i]);
  }
}

}  // namespace g4mi

using namespace g4mi;

extern "C" {

int g4mi_q_norm_rope(uint16_t* q, const uint16_t* q_norm, const uint16_t* rope_cos, const uint16_t* rope_sin,
                     int64_t T, int64_t NH, int64_t D, int64_t p0, int64_t rope_len, float eps, void* stream) {
  G4MI_REQUIRE(q && q_norm && rope_cos && rope_sin, G4MI_EINVAL, "q_norm_rope: missing argument");
  G4MI_REQUIRE(T >= 1 && T <= 2147483647 && NH >= 1 && NH <= 65535 * 4 && p0 >= 0 && p0 + T <= rope_len, G4MI_EINVAL,
               "q_norm_rope: T=%lld NH=%lld p0=%lld outside the rope table (%lld positions)", (long long)T,
               (long long)NH, (long long)p0, (long long)rope_len);
  dim3 grid((unsigned)T, (unsigned)((NH + 3) / 4));
  hipStream_t st = as_stream(stream);
  switch (D) {
    case 64: hipLaunchKernelGGL(q_norm_rope_kernel<64>, grid, dim3(256), 0, st, q, q_norm, rope_cos, rope_sin, (int)NH, (int)p0, eps); break;
    case 128: hipLaunchKernelGGL(q_norm_rope_kernel<128>, grid, dim3(256), 0, st, q, q_norm, rope_cos, rope_sin, (int)NH, (int)p0, eps); break;
    case 256: hipLaunchKernelGGL(q_norm_rope_kernel<256>, grid, dim3(256), 0, st, q, q_norm, rope_cos, rope_sin, (int)NH, (int)p0, eps); break;
    case 512: hipLaunchKernelGGL(q_norm_rope_kernel<512>, grid, dim3(256), 0, st, q, q_norm, rope_cos, rope_sin, (int)NH, (int)p0, eps); break;
    default: G4MI_REQUIRE(false, G4MI_EUNSUPPORTED, "q_norm_rope: head_dim %lld not in {64,128,256,512}", (long long)D);
  }
  return check_launch("q_norm_rope");
}

int g4mi_prefill_attention(const uint16_t* q, const uint16_t* k_pages, const uint16_t* v_pages, int64_t num_pages,
                           const int32_t* page_table, int64_t max_pages, int64_t page_size, int64_t T, int64_t p0,
                           int64_t NH, int64_t KV, int64_t D, int64_t window, float softcap, uint16_t* ctx,
                           void* stream) {
  G4MI_REQUIRE(q && k_pages && v_pages && page_table && ctx, G4MI_EINVAL, "prefill_attention: missing argument");
  G4MI_REQUIRE(KV >= 1 && KV <= 65535 && NH >= KV && NH % KV == 0, G4MI_EINVAL,
               "prefill_attention: bad NH=%lld KV=%lld", (long long)NH, (long long)KV);
  const int64_t G = NH / KV;
  G4MI_REQUIRE(D == 64 || D == 128 || D == 256 || D == 512, G4MI_EUNSUPPORTED,
               "prefill_attention: head_dim %lld not in {64,128,256,512}", (long long)D);
  G4MI_REQUIRE(G == 1 || G == 2 || G == 4 || G == 8, G4MI_EUNSUPPORTED,
               "prefill_attention: %lld query heads per KV head not in {1,2,4,8}", (long long)G);
  G4MI_REQUIRE(page_size % 64 == 0 && page_size >= 64, G4MI_EUNSUPPORTED,
               "prefill_attention: page size %lld must be a multiple of 64", (long long)page_size);
  G4MI_REQUIRE(T >= 1 && p0 >= 0 && p0 + T <= max_pages * page_size, G4MI_EINVAL,
               "prefill_attention: positions [%lld, %lld) beyond the page table", (long long)p0, (long long)(p0 + T));
  G4MI_REQUIRE(((uintptr_t)q & 15u) == 0 && ((uintptr_t)k_pages & 15u) == 0 && ((uintptr_t)v_pages & 15u) == 0,
               G4MI_EALIGN, "prefill_attention: q and the pages must be 16-byte aligned");
  PfAttnArgs a;
  a.q = q; a.k_pages = k_pages; a.v_pages = v_pages; a.pt = page_table; a.ctx = ctx;
  a.T = (int)T; a.NH = (int)NH; a.KV = (int)KV; a.page = (int)page_size; a.num_pages = (int)num_pages;
  a.max_pages = (int)max_pages; a.p0 = (int)p0; a.window = (int)window; a.softcap = softcap; a.G = (int)G;
  a.cap_k = softcap > 0.0f ? -2.0f * kLog2e / softcap : 0.0f;
  hipStream_t st = as_stream(stream);
  // 1-D grid in the order of pf_block
  auto grid_of = [&](int64_t qp) -> int64_t {
    const int64_t nqb = (T + qp - 1) / qp;
    a.nqb = (int)nqb;
    if (8 % KV == 0) {
      a.xmap = 1;
      const int64_t per = 8 / KV;
      return KV * ((nqb + per - 1) / per * per);
    }
    a.xmap = (KV % 8 == 0) ? 2 : 0;
    return KV * nqb;
  };
  if (D == 512 && p0 + T <= kPfFewKeys) {
    const int64_t nb = grid_of(64 / G);
#define G4MI_PF(GG)                                                                                              \
  case GG:                                                                                                       \
    if (softcap > 0.0f)                                                                                          \
      hipLaunchKernelGGL((attn_prefill_few_kernel<GG, true>), dim3((unsigned)nb), dim3(256), 0, st, a);          \
    else                                                                                                         \
      hipLaunchKernelGGL((attn_prefill_few_kernel<GG, false>), dim3((unsigned)nb), dim3(256), 0, st, a);         \
    break;
    switch (G) { G4MI_PF(1) G4MI_PF(2) G4MI_PF(4) G4MI_PF(8) }
#undef G4MI_PF
    return check_launch("prefill_attention");
  }
  const int64_t nb = grid_of(kPfRows / G);
  G4MI_REQUIRE(nb <= 2147483647, G4MI_EINVAL, "prefill_attention: %lld blocks", (long long)nb);
#define G4MI_PF(DD)                                                                                              \
  case DD:                                                                                                       \
    if (softcap > 0.0f)                                                                                          \
      hipLaunchKernelGGL((attn_prefill_kernel<DD, true>), dim3((unsigned)nb), dim3(256), 0, st, a);              \
    else                                                                                                         \
      hipLaunchKernelGGL((attn_prefill_kernel<DD, false>), dim3((unsigned)nb), dim3(256), 0, st, a);             \
    break;
  switch (D) { G4MI_PF(64) G4MI_PF(128) G4MI_PF(256) G4MI_PF(512) }
#undef G4MI_PF
  return check_launch("prefill_attention");
}

}  // extern "C"
