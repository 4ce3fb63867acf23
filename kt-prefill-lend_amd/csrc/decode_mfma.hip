// Decode-sized hot-expert layer on the matrix cores (KTMI_MODE_DECODE, and the shortest chunks
// of KTMI_MODE_GROUPED): three launches, the weights decoded from their GGUF blocks straight
// into v_mfma_f32_16x16x32_bf16 operands (bpiece.h: the exact dequantised values, one bf16
// rounding, the values the grouped prefill kernels and the dequant entry point use), the routes
// of one slot as the MFMA's 16 columns.
//
//   dm_gate_up      block (k-th slot with routes, 16 intermediate rows): the 4 waves split the
//                   hidden dimension; each moves its columns of the 16 gate and 16 up rows
//                   through a ring in LDS, decodes them and multiplies them against the bf16 x
//                   rows of the slot's routes; the partial sums meet in LDS,
//                   h = bf16(silu(g) * u) (the grouped epilogue's) goes to h [R, N].
//   dm_down         block (k-th slot with routes, 64 or 128 hidden rows): each wave runs its 16
//                   or 32 down rows of the slot through a ring of its own against the h rows of
//                   the slot's routes and writes each route's outputs, rounded to bf16 (the
//                   reference's per-route bf16 output), to yv [R, K].
//   dm_combine      the weighted top-k sum in k order (hot/kt_gguf_hot.py:43-71).
//
// What bounds them: the touched weights' bytes (up to 5 TB/s on large experts) and, close
// behind, the decode (2.5 to 4 VALU a value); on small layers the three launches. The weights
// pass through LDS one super-block column at a time, so any row length runs at the same
// occupancy: the 7168 x 2048 Q4_K/Q6_K layer with 24 slots at 5 tokens takes 92 us (stage-by-
// stage GEMV 206), the 2048 x 768 Q8_0 layer with 16 slots at 24 tokens 35 us (170).
//
// Lane map (16x16x32 operands): row or column l % 16, k-chunk g = l / 16 (8 values). Lane
// group g holds the piece of BPiece step SUB = 2 s + (g & 1), half g >> 1 of each 128-value
// double step s of a super-block column; MFMA j of the double step takes the piece's values
// 8j..8j+7. The activation operand of column c reads the same K positions of its row, so
// every lane pair of A and B refers to the same k. The K order inside a super-block is a
// permutation, which leaves every dot product unchanged.
//
// Against the GEMV mode (decode_layer.hip, the reference's int8 numerics): no q8_1
// quantisation of x or h, fp32 sums of bf16 products; the outputs stay within the layer's
// relative-L2 bar against the fp64 FFN. Per route the work is a fixed number of MFMAs, so
// a slot with 12 routes costs what a slot with one does.
//
// Membership (the k-th slot with routes, a slot's routes) is computed by every wave on its
// own from the slot ids (ballots, and a 16-word slot bitmap ORed over the wave by DPP into
// scalar registers): no block barrier before the weight loads are issued.
#include <type_traits>

#include "bpiece.h"
#include "kernels.h"

namespace ktmi {

namespace {

constexpr int DM_WAVES = 4;                   // waves of a block
constexpr int DM_THREADS = DM_WAVES * 64;
constexpr int DM_RT = 16;                     // rows of a row tile (the MFMA's rows)
constexpr int DM_ROUTES = 1024;               // routes of a call these kernels take

__device__ __forceinline__ f32x4_t mfma16(const bf16x8_t& a, const bf16x8_t& b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8_t words8(const uint32_t* w) {
  const u32x4_t v = {w[0], w[1], w[2], w[3]};
  return __builtin_bit_cast(bf16x8_t, v);
}

// silu(g) * u as the grouped gate/up epilogue computes it
__device__ __forceinline__ float dm_silu_mul(float g, float u) {
  return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
}

__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The call's routes, NR a lane: route 64 i + lane has slot sid[i] (-1: no slot here).
template <int NR>
struct WaveRoutes {
  int sid[NR];
  __device__ __forceinline__ void load(const int32_t* __restrict__ slot_ids, int R, int S) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = 64 * i + lane;
      const int s = r < R ? slot_ids[r] : -1;
      sid[i] = s >= 0 && s < S ? s : -1;
    }
  }
};

// OR of a 32-bit value over the wave, in scalar registers: DPP inside each row of 16 lanes
// (quad swaps, then the half-row and row mirrors), then the four rows' values read out
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_or(uint32_t v) {
  return v | (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
  asm volatile("" : "+v"(v));  // a vector register: the compiler may otherwise feed DPP a scalar one
  v = dpp_or<0xB1>(v);   // quad_perm [1,0,3,2]
  v = dpp_or<0x4E>(v);   // quad_perm [2,3,0,1]
  v = dpp_or<0x141>(v);  // row_half_mirror
  v = dpp_or<0x140>(v);  // row_mirror
  return (uint32_t)(__builtin_amdgcn_readlane((int)v, 0) | __builtin_amdgcn_readlane((int)v, 16) |
                    __builtin_amdgcn_readlane((int)v, 32) | __builtin_amdgcn_readlane((int)v, 48));
}

// The slots with routes as 8 words of 64 slots (S <= 512), the same in every lane (scalar
// registers): each word is the OR over the wave of the lanes' own route bits.
struct SlotSet {
  static constexpr int NW = 8;
  uint32_t word[2 * NW];
  template <int NR>
  __device__ __forceinline__ void build(const WaveRoutes<NR>& wr, int S) {
    const int nw = (S + 31) >> 5;
#pragma unroll
    for (int c = 0; c < 2 * NW; ++c) {
      word[c] = 0u;
      if (c < nw) {  // uniform
        uint32_t m = 0u;
#pragma unroll
        for (int i = 0; i < NR; ++i) m |= (wr.sid[i] >> 5) == c ? 1u << (wr.sid[i] & 31) : 0u;  // -1 >> 5 is -1
        word[c] = wave_or(m);
      }
    }
  }
  // the k-th slot with routes in ascending order, -1 past the last (uniform over the wave): in
  // the word that holds it, the lane whose bit is set with k set bits below it
  __device__ __forceinline__ int kth(int k) const {
    int e = -1;
#pragma unroll
    for (int c = 0; c < NW; ++c) {
      const uint32_t lo = word[2 * c], hi = word[2 * c + 1];
      const int n = __popc(lo) + __popc(hi);
      if (e < 0 && k >= 0 && k < n) {  // uniform
        const int lane = threadIdx.x & 63;
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
        const uint32_t bit = ((lane < 32 ? lo : hi) >> (lane & 31)) & 1u;
        e = 64 * c + (int)__builtin_ctzll(__ballot(bit && (int)below == k));
      }
      k -= n;
    }
    return e;
  }
};

// The routes of slot e in ascending order at mem[0 .. m) (LDS; every wave of the block writes
// the same list and reads what it wrote itself, so the block needs no barrier); returns m.
// m <= tokens unless a token lists a slot twice; either way every route of the slot is listed.
template <int NR>
__device__ __forceinline__ int slot_routes(const WaveRoutes<NR>& wr, int e, uint16_t* mem) {
  const int lane = threadIdx.x & 63;
  const uint64_t below = (1ull << lane) - 1ull;
  int base = 0;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const bool hit = wr.sid[i] == e;
    const uint64_t b = __ballot(hit);
    const int at = base + __popcll(b & below);
    if (hit) mem[at] = (uint16_t)(64 * i + lane);
    base += __popcll(b);
  }
  wave_fence();
  return base;
}

// s_waitcnt operand: at most n vector memory operations outstanding (expcnt and lgkmcnt free)
constexpr int dm_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// K offset inside a super-block column of the 8 values lane group (p, h) holds for MFMA j of
// double step S2 (the piece's values 8j..8j+7)
template <class BP, int S2>
__device__ __forceinline__ int kpos(int p, int h, int j) {
  const int q = j < 2 ? BP::off0(h) / 8 + j : BP::off1(h) / 8 + j - 2;
  return BP::template ksub_hp<S2>(p) + BP::coff(q);
}

// A wave's weights on their way to the matrix cores: NT tiles of 16 rows, one super-block
// column (256 values of every row) at a time, moved into the wave's own LDS ring of NB columns
// by direct loads. A staged row keeps its bytes from the 16-byte boundary below them, CH chunks
// of 16 bytes a row: an odd number, so the 16 rows of a tile fall into different banks.
template <int TYPE, int NT, int NB>
struct ColRing {
  static constexpr int QB = TYPE == GGML_Q8_0 ? 8 * QB8_0 : (int)Fmt<TYPE>::QB;  // a row's bytes of a column
  // 16-byte aligned columns (QB and row_bytes multiples of 16) or 2-byte aligned ones
  static constexpr bool ALIGNED = QB % 16 == 0;
  static constexpr int USED = (QB + (ALIGNED ? 0 : 14) + 15) / 16;  // chunks that hold the row's bytes
  static constexpr int CH = USED | 1;
  static constexpr int ROW = 16 * CH;
  static constexpr int BUF = NT * DM_RT * ROW;
  static constexpr int BYTES = NB * BUF;  // a wave's ring
  static constexpr int NI = (NT * DM_RT * CH + 63) / 64;  // direct loads a column
  uint8_t* lds;
  const uint8_t* base;  // the slot's matrix from the 16-byte boundary below it
  uint32_t bytes;
  uint32_t off[NI];    // the lane's chunk of load i: its row's offset (+ 16 chunk where ALIGNED)
  uint32_t roff[NT];   // offset of this lane's own row (lane % 16) of tile t
  // row0[t]: first row of tile t in the slot's matrix at wexp (rb bytes a row, rows of them)
  __device__ __forceinline__ void init(uint8_t* region, const uint8_t* wexp, int rows, int64_t rb,
                                       const int (&row0)[NT]) {
    const int lane = threadIdx.x & 63;
    lds = region;
    const uint32_t mis = (uint32_t)(uintptr_t)wexp & 15u;
    base = wexp - mis;
    bytes = ((uint32_t)(rows * rb) + mis + 15u) & ~15u;  // whole chunks: each holds a byte of the matrix
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int q = 64 * i + lane, row = q / CH;
      const int t = min(row / DM_RT, NT - 1);
      off[i] = mis + (uint32_t)((row0[t] + row % DM_RT) * rb) + (ALIGNED ? 16u * (uint32_t)(q % CH) : 0u);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) roff[t] = mis + (uint32_t)((row0[t] + (lane & 15)) * rb);
  }
  // column sb into buffer buf; where more is false the same loads go past the end of a buffer
  // of no bytes (zeros, no memory access), so that the count of operations in flight does not
  // depend on the column. The scalar offset is 0 there too: a range check of the lane's offset
  // against the bytes less the scalar offset would wrap with any other
  __device__ __forceinline__ void issue(int sb, int buf, bool more) const {
    const int lane = threadIdx.x & 63;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, more ? bytes : 0u, 0x00020000);
    const int soff = ALIGNED && more ? sb * QB : 0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int q = 64 * i + lane;
      const uint32_t o = ALIGNED ? off[i] : ((off[i] + (uint32_t)(sb * QB)) & ~15u) + 16u * (uint32_t)(q % CH);
      if ((i < NI - 1 || q < NT * DM_RT * CH) && (USED == CH || q % CH < USED))
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsrc, (__attribute__((address_space(3))) void*)(lds + buf * BUF + 1024 * i), 16, (int)o, soff, 0, 0);
    }
  }
  // the lane's row of tile t in buffer buf, as a row that starts at column sb
  __device__ __forceinline__ const uint8_t* row(int sb, int buf, int t) const {
    return lds + buf * BUF + (16 * t + (threadIdx.x & 15)) * ROW + (ALIGNED ? 0 : (roff[t] + (uint32_t)(sb * QB)) & 15u);
  }
};

// Columns [sb0, sb1) of the ring's NT tiles against the activation rows of ng <= G groups of 16
// routes (a row per lane % 16 and group, at byte xoff[cg] of act; past the routes an offset past
// the buffer, whose loads return zeros): acc[t][cg] += tile t x group cg.
//
// Order of a column's memory operations: the activation loads of its first half (at G = 1 of
// both halves), its weight bytes out of LDS into registers, the direct loads of column
// sb + NB into the buffer just read, then (G > 1) the activation loads of the second half; the
// decode of a half (about 450 VALU cycles a tile) runs while its activation loads are in flight.
// PLAIN: the decoders' plain products; without it, whether a scale is infinite or NaN, so that the
// wave has to run the columns again with it.
// Loads return in order, so at G > 1 the wait for the second half's activations also completes
// the direct loads before them: the ring then covers a half of a column's work, not a column. At
// G = 1 the next columns' loads stay in flight for Q4_K and Q8_0; the direct loads of Q6_K and
// IQ3_S are under lane masks (padding chunks), where the compiler counts none of them and its
// waits for the activations drain the ring too.
template <int TYPE, int NT, int NB, int G, bool PLAIN>
__device__ __forceinline__ bool window_pass(const ColRing<TYPE, NT, NB>& ring, const __amdgpu_buffer_rsrc_t& act,
                                               const uint32_t (&xoff)[G], int ng, int sb0, int sb1,
                                               const uint32_t* grid, f32x4_t (&acc)[NT][G]) {
  using BP = BPiece<TYPE>;
  const int lane = threadIdx.x & 63;
  const int p = (lane >> 4) & 1, h = (lane >> 5) & 1;
  bf16x8_t xv[G == 1 ? 2 : 1][G][4];
  auto xissue = [&](int sb, auto s2c) {
    constexpr int S2 = decltype(s2c)::value;
#pragma unroll
    for (int cg = 0; cg < G; ++cg)
      if (cg < ng)  // uniform
#pragma unroll
        for (int j = 0; j < 4; ++j)
          xv[G == 1 ? S2 : 0][cg][j] = __builtin_bit_cast(
              bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(
                            act, (int)(xoff[cg] + 2u * (uint32_t)(kpos<BP, S2>(p, h, j))), 512 * sb, 0));
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  int buf = 0;
  bool rare = false;
  for (int sb = sb0; sb < sb1; ++sb) {
    xissue(sb, H0{});
    if constexpr (G == 1) xissue(sb, H1{});
    __builtin_amdgcn_sched_barrier(0);  // the activation loads stay ahead of the wait that counts them
    // the column's direct loads have landed once at most the younger operations are in flight:
    // the next column's (NB = 2) and this column's activation loads (at least 4, 8 at G = 1); the
    // numbers are checked against the compiled code by a test
    constexpr int NX = G == 1 ? 8 : 4;
    __builtin_amdgcn_s_waitcnt(dm_vmcnt((NB - 1) * ColRing<TYPE, NT, NB>::NI + NX));
    wave_fence();
    typename BP::Head hd[NT];
    typename BP::Raw raw[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint8_t* row = ring.row(sb, buf, t);
      BP::template load_head<LMem>(row, 0, h, hd[t]);
      BP::template load_hp<0, LMem>(row, 0, h, p, grid, raw[t][0]);
      BP::template load_hp<1, LMem>(row, 0, h, p, grid, raw[t][1]);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the buffer has been read
    wave_fence();
    ring.issue(sb + NB, buf, sb + NB < sb1);
    auto half = [&](auto s2c) {
      constexpr int S2 = decltype(s2c)::value;
      uint32_t a[NT][16];
#pragma unroll
      for (int t = 0; t < NT; ++t) BP::template decode_hp<S2, PLAIN>(hd[t], raw[t][S2], grid, p, a[t]);
#pragma unroll
      for (int cg = 0; cg < G; ++cg)
        if (cg < ng)  // uniform
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              acc[t][cg] = mfma16(words8(&a[t][4 * j]), xv[G == 1 ? S2 : 0][cg][j], acc[t][cg]);
    };
    if constexpr (!PLAIN)
#pragma unroll
      for (int t = 0; t < NT; ++t) rare |= BP::unbounded(hd[t], raw[t][0]) | BP::unbounded(hd[t], raw[t][1]);
    half(H0{});
    if constexpr (G > 1) xissue(sb, H1{});
    half(H1{});
    buf = NB == 2 ? buf ^ 1 : 0;
  }
  __builtin_amdgcn_s_waitcnt(dm_vmcnt(0));  // the loads past the last column have written their zeros
  return rare;
}

// The ring's first columns issued, the columns run (acc from zero), and run again with plain
// products where a scale is infinite: in the loop those cost Q8_0 windows 3 to 4 % (2048 x 512, 16
// tokens 34.3 us, so 33.1; 7168 x 2048, 5 tokens 152 and 148), and only infinities need them.
template <int TYPE, int NT, int NB, int G>
__device__ __forceinline__ void window_columns(const ColRing<TYPE, NT, NB>& ring, const __amdgpu_buffer_rsrc_t& act,
                                               const uint32_t (&xoff)[G], int ng, int sb0, int sb1,
                                               const uint32_t* grid, f32x4_t (&acc)[NT][G]) {
  auto start = [&]() {
    ring.issue(sb0, 0, sb0 < sb1);
    if (NB == 2) ring.issue(sb0 + 1, 1, sb0 + 1 < sb1);
#pragma unroll
    for (int cg = 0; cg < G; ++cg)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t][cg] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  };
  start();
  const bool rare = window_pass<TYPE, NT, NB, G, false>(ring, act, xoff, ng, sb0, sb1, grid, acc);
  if constexpr (TYPE == GGML_Q8_0 || TYPE == GGML_Q6_K)
    if (__builtin_expect(__any(rare), 0)) {
      start();
      window_pass<TYPE, NT, NB, G, true>(ring, act, xoff, ng, sb0, sb1, grid, acc);
    }
}

// The k-th slot with routes of this block, its routes listed in mem: (slot, route count), slot
// -1 past the slots with routes (the same in every wave)
template <int NR>
__device__ __forceinline__ int2 block_slot(const int32_t* __restrict__ slot_ids, int R, int S, int kslot,
                                           uint16_t* mem) {
  WaveRoutes<NR> wr;
  wr.load(slot_ids, R, S);
  SlotSet ss;
  ss.build(wr, S);
  const int e = ss.kth(kslot);
  if (e < 0) return make_int2(-1, 0);
  return make_int2(e, slot_routes(wr, e, mem));
}

// waves a SIMD that the registers are held to, without spilling but for Q6_K at G = 4 (12). For
// Q8_0 at G = 1 the rings (70 KB a block) leave two blocks a CU whatever it says
template <int TYPE, int G>
constexpr int dm_waves() {
  return G == 4 ? 2 : G == 1 ? (TYPE == GGML_Q4_K ? 4 : 3) : TYPE == GGML_Q4_K || TYPE == GGML_Q8_0 ? 3 : 2;
}

// One block per (k-th slot with routes, 16 intermediate rows): each wave takes a quarter of the
// hidden dimension of the block's 16 gate and 16 up rows, the partial sums meet in LDS and
// h = bf16(silu(g) * u) goes to h [R, N] of the routes. G groups of 16 routes share a pass over
// the weights.
template <int TYPE, int G, int NR, int NB>
__global__ __launch_bounds__(DM_THREADS, (dm_waves<TYPE, G>())) void dm_gate_up(const uint16_t* __restrict__ x, int K, int N,
                                                         const int32_t* __restrict__ slot_ids, int R, int S,
                                                         int top_k, const uint8_t* __restrict__ W13, int w_is_table,
                                                         int64_t w_stride, uint16_t* __restrict__ hbuf) {
  using Ring = ColRing<TYPE, 2, NB>;
  // one LDS object (a second one makes the compiler wait for every direct load before each LDS
  // read): the IQ3_S codebook, the route list, the waves' rings, over them the partial sums
  constexpr int GRID = TYPE == GGML_IQ3_S ? 2048 : 0;
  constexpr int RING_OFF = GRID + NR * 64 * 2;
  constexpr int PART = DM_WAVES * 2 * G * 4 * 64 * 4;
  constexpr int RINGS = DM_WAVES * Ring::BYTES;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[RING_OFF + (RINGS > PART ? RINGS : PART)];
  uint32_t* grid = (uint32_t*)smem;
  uint16_t* mem = (uint16_t*)(smem + GRID);
  float (*part)[2][G][4][64] = (float(*)[2][G][4][64])(smem + RING_OFF);  // [wave][tile: gate, up]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int NG = N / DM_RT;
  const int kslot = blockIdx.x / NG, rg = blockIdx.x - kslot * NG;
  if constexpr (TYPE == GGML_IQ3_S) stage_iq3s_sel(grid);
  const int2 em = block_slot<NR>(slot_ids, R, S, kslot, mem);
  const int e = em.x, m = em.y;
  if (e < 0) return;
  if constexpr (TYPE == GGML_IQ3_S) __syncthreads();  // the codebook
  const int r = lane & 15;
  const uint32_t x_bytes = (uint32_t)(R / top_k) * (uint32_t)K * 2u;
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, x_bytes, 0x00020000);
  const uint8_t* wexp = w_is_table ? (const uint8_t*)((const int64_t*)W13)[e] : W13 + (int64_t)e * w_stride;
  Ring ring;
  ring.init(smem + RING_OFF + wave * Ring::BYTES, wexp, 2 * N, row_bytes(K, TYPE), {DM_RT * rg, N + DM_RT * rg});
  const int nsb = K / 256;
  const int per = (nsb + DM_WAVES - 1) / DM_WAVES;
  const int sb0 = wave * per, sb1 = min(nsb, sb0 + per);
  const int c = threadIdx.x >> 4, rr = threadIdx.x & 15;
  const int ln = 16 * (rr >> 2) + c, i = rr & 3;
  const int ncg = (m + 15) >> 4;
  for (int cg0 = 0; cg0 < ncg; cg0 += G) {
    const int ng = min(G, ncg - cg0);
    uint32_t xoff[G];
#pragma unroll
    for (int cg = 0; cg < G; ++cg) {
      const int col = 16 * (cg0 + cg) + r;
      xoff[cg] = col < m ? (uint32_t)(mem[col] / top_k) * (uint32_t)K * 2u : x_bytes;
    }
    if (cg0 > 0) __syncthreads();  // the previous pass has read the partial sums
    f32x4_t acc[2][G];
    window_columns<TYPE, 2, NB, G>(ring, x_rsrc, xoff, ng, sb0, sb1, grid, acc);
    __syncthreads();  // every wave has read its ring
#pragma unroll
    for (int cg = 0; cg < G; ++cg)
      if (cg < ng)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q) part[wave][t][cg][q][lane] = acc[t][cg][q];
    __syncthreads();
    // output (row rr, column c): lane 16 (rr / 4) + c of each wave holds it as element rr % 4;
    // 16 consecutive threads write one route's 16 values of h (32 bytes)
#pragma unroll
    for (int cg = 0; cg < G; ++cg) {
      const int col = 16 * (cg0 + cg) + c;
      if (col < m) {
        float g = 0.0f, u = 0.0f;
#pragma unroll
        for (int w = 0; w < DM_WAVES; ++w) {
          g += part[w][0][cg][i][ln];
          u += part[w][1][cg][i][ln];
        }
        hbuf[(int64_t)mem[col] * N + DM_RT * rg + rr] = f2bf(dm_silu_mul(g, u));
      }
    }
  }
}

// One block per (k-th slot with routes, 64 NT hidden rows); wave w takes the tile's rows
// 16 NT w .. over the whole intermediate dimension against the h rows of the slot's routes (L2
// hits: every block of the slot reads the same rows) and writes each route's outputs, rounded
// to bf16 (the reference's per-route bf16 output), to yv [R, K]. The weighted top-k sum is a
// launch of its own (dm_combine): inside this one, the blocks of a tile would have to order
// themselves through device-scope fences, which write back and invalidate the whole L2 of
// their XCD. The registers are held to 4, 3 and 2 waves a SIMD; Q6_K at NT = 2, G = 4 spills 11
// of them for it and IQ3_S at NT = 2, G = 2 four.
template <int TYPE, int NT, int G, int NR, int NB>
__global__ __launch_bounds__(DM_THREADS, (G == 1 ? 4 : G == 2 ? 3 : 2)) void dm_down(const uint16_t* __restrict__ hbuf, int K, int N,
                                                      const int32_t* __restrict__ slot_ids, int R, int S,
                                                      const uint8_t* __restrict__ W2, int w_is_table, int64_t w_stride,
                                                      uint16_t* __restrict__ yv) {
  using Ring = ColRing<TYPE, NT, NB>;
  constexpr int GRID = TYPE == GGML_IQ3_S ? 2048 : 0;
  constexpr int RING_OFF = GRID + NR * 64 * 2;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[RING_OFF + DM_WAVES * Ring::BYTES];
  uint32_t* grid = (uint32_t*)smem;
  uint16_t* mem = (uint16_t*)(smem + GRID);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int TILE = DM_WAVES * NT * DM_RT;
  const int ntile = K / TILE;
  const int kslot = blockIdx.x / ntile, tile = blockIdx.x - kslot * ntile;
  if constexpr (TYPE == GGML_IQ3_S) stage_iq3s_sel(grid);
  const int2 em = block_slot<NR>(slot_ids, R, S, kslot, mem);
  const int e = em.x, m = em.y;
  if (e < 0) return;
  if constexpr (TYPE == GGML_IQ3_S) __syncthreads();  // the codebook
  const int r = lane & 15;
  const uint32_t hrow = 2u * (uint32_t)N;
  const uint32_t h_bytes = (uint32_t)R * hrow;
  const __amdgpu_buffer_rsrc_t h_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)hbuf, (short)0, h_bytes, 0x00020000);
  const uint8_t* wexp = w_is_table ? (const uint8_t*)((const int64_t*)W2)[e] : W2 + (int64_t)e * w_stride;
  const int rw0 = tile * TILE + wave * NT * DM_RT;
  int row0[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) row0[t] = rw0 + DM_RT * t;
  Ring ring;
  ring.init(smem + RING_OFF + wave * Ring::BYTES, wexp, K, row_bytes(N, TYPE), row0);
  const int nsb = N / 256;
  const int ncg = (m + 15) >> 4;
  for (int cg0 = 0; cg0 < ncg; cg0 += G) {
    const int ng = min(G, ncg - cg0);
    uint32_t hoff[G];
#pragma unroll
    for (int cg = 0; cg < G; ++cg) {
      const int col = 16 * (cg0 + cg) + r;
      hoff[cg] = col < m ? (uint32_t)mem[col] * hrow : h_bytes;
    }
    f32x4_t acc[NT][G];
    window_columns<TYPE, NT, NB, G>(ring, h_rsrc, hoff, ng, 0, nsb, grid, acc);
    // lane l holds rows 4 (l / 16) + i of column l % 16: four consecutive bf16 of yv
#pragma unroll
    for (int cg = 0; cg < G; ++cg) {
      const int col = 16 * (cg0 + cg) + r;
      if (col < m) {
        const int rt = mem[col];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const f32x4_t& v = acc[t][cg];
          *(uint2*)(yv + (int64_t)rt * K + row0[t] + 4 * (lane >> 4)) = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
        }
      }
    }
  }
}

// y[t, c] = bf16( sum over k ascending, hot routes only, of bf16(Y * bf16(w)) ): a thread per
// (token, eight hidden columns); the loads of eight routes are issued before their sums
__global__ __launch_bounds__(256) void dm_combine(const uint16_t* __restrict__ yv, const int32_t* __restrict__ slot_ids,
                                                  const float* __restrict__ topk_w, int T, int top_k, int S, int K,
                                                  uint16_t* __restrict__ y) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  const int G = K / 8;
  if (q >= T * G) return;
  const int t = q / G, c = 8 * (q - t * G);
  float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  for (int k0 = 0; k0 < top_k; k0 += 8) {
    int sl[8];
    float w[8];
    uint4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int rt = t * top_k + min(k0 + u, top_k - 1);  // past top_k: a repeat, not summed
      sl[u] = slot_ids[rt];
      w[u] = topk_w[rt];
      v[u] = *(const uint4*)(yv + (int64_t)rt * K + c);  // every route's row lies in yv
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (k0 + u >= top_k || sl[u] < 0 || sl[u] >= S) continue;  // cold or past top_k: its yv row is stale
      const float wb = bf2f(f2bf(w[u]));
      const uint32_t wd[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] += bf2f(f2bf(bf2f((uint16_t)(wd[i] & 0xFFFFu)) * wb));
        acc[2 * i + 1] += bf2f(f2bf(bf2f((uint16_t)(wd[i] >> 16)) * wb));
      }
    }
  }
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = (uint32_t)f2bf(acc[2 * i]) | ((uint32_t)f2bf(acc[2 * i + 1]) << 16);
  *(uint4*)(y + (int64_t)t * K + c) = make_uint4(o[0], o[1], o[2], o[3]);
}

// The routes a pass over a slot's weights has room for: those that the popular slots may have, at
// most the tokens (unless a token lists a slot twice) and hardly more than eight times the mean.
// G, the groups of 16 routes of a pass, goes by it (more groups are more registers: by the tokens
// alone, 40 tokens x top-2 on 80 slots of the 2048 x 1024 Q6_K layer took 113 us, so 74), NR, the
// ids a lane of the membership, by the routes
int64_t pass_routes(int64_t tokens, int64_t R, int64_t S) {
  const int64_t m = (8 * R + S - 1) / S;
  return m < tokens ? m : tokens;
}

template <int TYPE>
int launch_dm_gate_up(const ktmi_layer* L, const uint16_t* x, const int32_t* slot_ids, int64_t tokens, int64_t top_k,
                      uint16_t* hbuf, hipStream_t stream) {
  const int64_t K = L->hidden, N = L->inter, S = L->n_slots, R = tokens * top_k;
  const int64_t st13 = 2 * N * row_bytes(K, TYPE);
  // blocks numbered (k-th slot with routes, row group), row group fastest; the blocks past
  // the slots with routes exit at once
  const unsigned nb = (unsigned)(S < R ? S : R) * (unsigned)(N / DM_RT);
#define KTMI_GU(G, NR)                                                                                        \
  dm_gate_up<TYPE, G, NR, 2><<<nb, DM_THREADS, 0, stream>>>(x, (int)K, (int)N, slot_ids, (int)R, (int)S, (int)top_k, \
                                                            (const uint8_t*)L->w13, L->w_is_table, st13, hbuf)
  const int64_t m = pass_routes(tokens, R, S);
  if (R <= 256) {
    if (m <= 16) KTMI_GU(1, 4); else if (m <= 32) KTMI_GU(2, 4); else KTMI_GU(4, 4);
  } else if constexpr (TYPE == GGML_Q6_K) {
    set_error("window gate/up: %lld routes of Q6_K (window_fits leaves them to the GEMMs)", (long long)R);
    return KTMI_EINVAL;
  } else {
    if (m <= 32) KTMI_GU(2, 16); else KTMI_GU(4, 16);
  }
#undef KTMI_GU
  KTMI_HIP_TRY(hipGetLastError());
  return KTMI_OK;
}

template <int TYPE>
int launch_dm_down(const ktmi_layer* L, const uint16_t* hbuf, const int32_t* slot_ids, const float* topk_w,
                   int64_t tokens, int64_t top_k, uint16_t* yv, uint16_t* y, hipStream_t stream) {
  const int64_t K = L->hidden, N = L->inter, S = L->n_slots, R = tokens * top_k;
  const int64_t st2 = K * row_bytes(N, TYPE);
  // blocks numbered (k-th slot with routes, hidden tile), tile fastest; the blocks past the
  // slots with routes exit at once
#define KTMI_DN(NT, G, NR)                                                                                     \
  dm_down<TYPE, NT, G, NR, 2><<<(unsigned)(S < R ? S : R) * (unsigned)(K / (64 * NT)), DM_THREADS, 0, stream>>>( \
      hbuf, (int)K, (int)N, slot_ids, (int)R, (int)S, (const uint8_t*)L->w2, L->w_is_table, st2, yv)
  const int64_t m = pass_routes(tokens, R, S);
  if (R <= 256) {
    if (m <= 16) KTMI_DN(1, 1, 4); else if (m <= 32) KTMI_DN(1, 2, 4); else KTMI_DN(1, 4, 4);
  } else {
    if (m <= 32) KTMI_DN(2, 2, 16); else KTMI_DN(2, 4, 16);
  }
#undef KTMI_DN
  KTMI_HIP_TRY(hipGetLastError());
  const unsigned nc = (unsigned)((tokens * (K / 8) + 255) / 256);
  dm_combine<<<nc, 256, 0, stream>>>(yv, slot_ids, topk_w, (int)tokens, (int)top_k, (int)S, (int)K, y);
  KTMI_HIP_TRY(hipGetLastError());
  return KTMI_OK;
}

}  // namespace

// what the kernels take, whatever the mode; a slot's matrix, x, h and yv are addressed by buffer
// instructions with 32-bit offsets
static bool window_shape(const ktmi_layer* L) {
  const int64_t K = L->hidden, N = L->inter, limit = 0xFFFF0000ll;
  if (!blck_size(L->type13) || !blck_size(L->type2)) return false;
  return K % 256 == 0 && N % 256 == 0 && L->n_slots <= 512 && 2 * DM_ROUTES * (K > N ? K : N) <= limit &&
         2 * N * row_bytes(K, L->type13) <= limit && K * row_bytes(N, L->type2) <= limit;
}

bool decode_mfma_fits(const ktmi_layer* L, int64_t tokens, int64_t top_k) {
  return window_shape(L) && tokens * top_k <= DM_MAX_ROUTES && tokens <= DM_MAX_TOKENS;
}

// The chunks the grouped mode gives to these kernels instead of the GEMMs, whose blocks pay for
// 128 routes a slot however few it has. These pay for their weights once a pass of 64 routes, and
// their x and h rows, one 16-byte piece a lane from 16 rows at a time, grow with the routes. The
// lines lie where they were not slower on some 900 layers drawn over types, sizes, 6 to 128 slots,
// top-1 to top-10 and popularities, all experts in slots among them (us, these kernels against the
// GEMMs):
//   Q8_0 and IQ3_S in both projections (the GEMMs gather these rows a lane each): up to 64 tokens
//     30-158 / 57-215; up to 128 with at most 18 routes a slot (counting cold ones) 110-291 /
//     143-493, on short rows up to 640 routes (past them up to 96 / 85)
//   with Q4_K or Q6_K: up to 40 tokens 27-109 / 49-153. Past them the GEMMs gain with every chip
//     round (one gate/up block a CU) that their blocks fill: at most 0.7 full 57 / 64 (2048 x 512,
//     40 slots, 77 tokens) and 205 / 304 (7168 x 2048, 20, 66); fuller, only few routes a slot
//     (2048 x 512, 52 slots, 96 tokens 82 / 67; 7168 x 2048, 14 of 24 experts, 64 tokens 232 / 175)
//   Q6_K gate/up: the GEMMs (2048 x 1024, 64 slots, 55 tokens 205 / 155)
bool window_fits(const ktmi_layer* L, int64_t tokens, int64_t top_k) {
  const int64_t R = tokens * top_k, S = L->n_slots;
  if (!window_shape(L) || R > DM_ROUTES || tokens > 128 || L->type13 == GGML_Q6_K) return false;
  if (tokens > 64 && R > 18 * S) return false;
  const bool long_rows = L->hidden >= 4096;
  const auto gathered = [](int t) { return t == GGML_Q8_0 || t == GGML_IQ3_S; };
  if (gathered(L->type13) && gathered(L->type2)) return tokens <= 64 || long_rows || R <= 640;
  const int64_t blocks = S * (L->inter / 128), rounds = (blocks + 255) / 256;
  const int64_t most = 10 * blocks <= 7 * 256 * rounds ? (long_rows ? 40 : 64) : (long_rows ? 15 : 8);
  return tokens <= 40 || (R <= 640 && R <= most * S);
}

namespace {
int64_t up256(int64_t v) { return (v + 255) & ~(int64_t)255; }
}  // namespace

// h [R, N] bf16, then yv [R, K] bf16 (the routes' down outputs)
int64_t decode_mfma_workspace(const ktmi_layer* L, int64_t tokens, int64_t top_k) {
  const int64_t R = tokens * top_k;
  return up256(R * L->inter * 2) + up256(R * L->hidden * 2);
}

int launch_decode_mfma(const ktmi_layer* L, const uint16_t* x, const float* topk_w, const int32_t* slot_ids,
                       int64_t tokens, int64_t top_k, uint16_t* y, uint8_t* ws, hipStream_t stream) {
  return launch_window(L, x, topk_w, slot_ids, tokens, top_k, y, (uint16_t*)ws,
                       (uint16_t*)(ws + up256(tokens * top_k * L->inter * 2)), stream);
}

int launch_window(const ktmi_layer* L, const uint16_t* x, const float* topk_w, const int32_t* slot_ids, int64_t tokens,
                  int64_t top_k, uint16_t* y, uint16_t* hbuf, uint16_t* yv, hipStream_t stream) {
  record_stage(0, stream);
  record_stage(1, stream);
  int rc;
  switch (L->type13) {
    case GGML_Q8_0: rc = launch_dm_gate_up<GGML_Q8_0>(L, x, slot_ids, tokens, top_k, hbuf, stream); break;
    case GGML_Q4_K: rc = launch_dm_gate_up<GGML_Q4_K>(L, x, slot_ids, tokens, top_k, hbuf, stream); break;
    case GGML_Q6_K: rc = launch_dm_gate_up<GGML_Q6_K>(L, x, slot_ids, tokens, top_k, hbuf, stream); break;
    case GGML_IQ3_S: rc = launch_dm_gate_up<GGML_IQ3_S>(L, x, slot_ids, tokens, top_k, hbuf, stream); break;
    default: set_error("decode layer: ggml type %d has no kernel", L->type13); return KTMI_ETYPE;
  }
  if (rc) return rc;
  record_stage(2, stream);
  record_stage(3, stream);
  switch (L->type2) {
    case GGML_Q8_0: rc = launch_dm_down<GGML_Q8_0>(L, hbuf, slot_ids, topk_w, tokens, top_k, yv, y, stream); break;
    case GGML_Q4_K: rc = launch_dm_down<GGML_Q4_K>(L, hbuf, slot_ids, topk_w, tokens, top_k, yv, y, stream); break;
    case GGML_Q6_K: rc = launch_dm_down<GGML_Q6_K>(L, hbuf, slot_ids, topk_w, tokens, top_k, yv, y, stream); break;
    case GGML_IQ3_S: rc = launch_dm_down<GGML_IQ3_S>(L, hbuf, slot_ids, topk_w, tokens, top_k, yv, y, stream); break;
    default: set_error("decode layer: ggml type %d has no kernel", L->type2); return KTMI_ETYPE;
  }
  record_stage(4, stream);
  record_stage(5, stream);
  return rc;
}

}  // namespace ktmi
