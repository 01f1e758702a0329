// FP8 GEMM of the FP8 linear layers (gfx950): out[m][n] = bf16(sum_k x8[m][k] w8[n][k], scaled, + bias[n]), x8 and w8
// e4m3 with K contiguous, fp32 accumulation on v_mfma_scale_f32_32x32x64_f8f6f4. Two scalings: rowwise (one fp32
// scale per token and per output channel, applied to the finished sum) and MX (one E8M0 scale per 32 values along K
// of each operand, applied by the MFMA itself).
//
// Tile: TM tokens x TN channels per workgroup, WGM x WGN waves (times KS shares of K). The W rows are the MFMA's A
// operand and the X rows its B operand, so a lane holds one token and runs of four consecutive channels of the result.
// K is walked in stages of 128 bytes per row (whole cache lines), streamed into NST LDS stages by direct global -> LDS loads; a
// wave reads the fragments of the next 64-deep half while its matrix products run on the current one, so one barrier
// per stage is all the synchronisation there is, and the products after it start from registers. The loads of a stage
// are issued between the products, one after each (all at once after the barrier: 96 instead of 85 us for the 256 x
// 256 tile at 6032 x 8960 x 1536). The result goes out through LDS, 16 bytes a lane.
//
// What bounds it: at 6032 x 8960 x 1536 the 192 x 192 tile takes 67-71 us (2.35-2.48 PFLOP/s); timing copies without
// the loads ran 58 us, without the products 51 us, without the fragment reads 61 us, so L2 -> LDS traffic (17 TB/s
// alone) and the matrix core (power-limited near 1.9 GHz) overlap but for ~10 us. Touching later stages in the L2
// first and 64-byte stages in a deeper ring were measured and brought nothing.
#include <type_traits>

#include "../../include/lbw_gemm.h"
#include "lbw_common.h"

#pragma clang fp contract(off)   // the epilogue's roundings are defined (without it even __fmul_rn + __fadd_rn fuse)

namespace lbw {

constexpr int GK = 128;             // bytes of K per stage
constexpr int G_ONE = 0x7F7F7F7F;   // E8M0 scale 1 in every byte

struct GemmArgs {
  const uint8_t* x;
  const uint8_t* w;
  const float* xs;       // rowwise: [m]
  const float* ws;       // rowwise: [n]
  const uint8_t* xe;     // MX: [k / 128][m][4]
  const uint8_t* we;     // MX: [k / 128][n][4]
  const uint16_t* bias;  // bf16 [n] or null
  uint16_t* out;         // bf16 [m][n]
  int m, n, k, mt, nt;   // mt x nt tiles
  int first, tiles;      // the tiles of this launch: first .. first + tiles of the tile order
};

// The last stage of a K that is not a multiple of 128 reads its missing 16-byte chunks from here.
__device__ __attribute__((aligned(16))) uint32_t gemm_zeros[4] = {0, 0, 0, 0};

__device__ __forceinline__ uint32_t lds_off(const uint8_t* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p;
}

// Direct global -> LDS loads of 16 bytes a lane (lane i to lds + 16 i), as inline asm like the attention kernel's: the
// compiler would otherwise wait for every one of them before each LDS read. dma_rows: the wave's N pieces of one operand
// from a uniform base plus a 32-bit byte offset per lane and piece, STEP bytes of LDS apart, M0 saved and restored once
// around them (the additions to M0 write SCC). dma16_at: one piece from a 64-bit address per lane. dma4: a dword a lane.
template <int N, int STEP>
__device__ __forceinline__ void dma_rows(const void* base, const uint32_t* off, uint32_t lds) {
  static_assert(N >= 1 && N <= 4, "pieces");
  uint32_t keep;
#define LBW_GEMM_NEXT "s_add_u32 m0, m0, %4\n\ts_nop 0\n\t"
#define LBW_GEMM_HEAD "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %1\n\t"
  if constexpr (N == 1)
    asm volatile(LBW_GEMM_HEAD "s_mov_b32 m0, %0" : "=&s"(keep) : "s"(base), "s"(lds), "v"(off[0]) : "memory");
  else if constexpr (N == 2)
    asm volatile(LBW_GEMM_HEAD LBW_GEMM_NEXT "global_load_lds_dwordx4 %5, %1\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(base), "s"(lds), "v"(off[0]), "i"(STEP), "v"(off[1]) : "memory", "scc");
  else if constexpr (N == 3)
    asm volatile(LBW_GEMM_HEAD LBW_GEMM_NEXT "global_load_lds_dwordx4 %5, %1\n\t" LBW_GEMM_NEXT
                 "global_load_lds_dwordx4 %6, %1\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(base), "s"(lds), "v"(off[0]), "i"(STEP), "v"(off[1]), "v"(off[2])
                 : "memory", "scc");
  else
    asm volatile(LBW_GEMM_HEAD LBW_GEMM_NEXT "global_load_lds_dwordx4 %5, %1\n\t" LBW_GEMM_NEXT
                 "global_load_lds_dwordx4 %6, %1\n\t" LBW_GEMM_NEXT "global_load_lds_dwordx4 %7, %1\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(base), "s"(lds), "v"(off[0]), "i"(STEP), "v"(off[1]), "v"(off[2]), "v"(off[3])
                 : "memory", "scc");
#undef LBW_GEMM_NEXT
#undef LBW_GEMM_HEAD
}
__device__ __forceinline__ void dma16_at(const void* p, uint32_t lds) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"((uint64_t)(uintptr_t)p), "s"(lds) : "memory");
}
__device__ __forceinline__ void dma4(const void* base, uint32_t off, uint32_t lds) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(off), "s"(base), "s"(lds) : "memory");
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Workgroup barrier: this wave's LDS reads are done (their stage may be refilled), and no access moves across.
__device__ __forceinline__ void stage_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

template <int TM, int TN, int WGM, int WGN, int NST, int KS, bool AHEAD, bool MX>
struct Gemm {
  static constexpr int NW = WGM * WGN, THREADS = 64 * NW * KS;   // NW waves for each of KS shares of K
  static constexpr int WM = TM / WGM, WN = TN / WGN, MT = WM / 32, NT = WN / 32;   // wave tile, in 32 x 32 products
  static constexpr int RP = 1024 / GK, CPR = GK / 16;   // rows of a 1 KB piece, 16-byte chunks of a row
  static constexpr int PX = TM / RP / NW, P = PX + TN / RP / NW;                   // 1 KB pieces per wave: of X, all
  static constexpr int TILE = (TM + TN) * GK;
  static constexpr int SCALES = MX ? (TM + TN) * 4 : 0;                            // one dword per row and stage
  static constexpr int PS = MX ? ((TM + TN) / 64 + NW - 1) / NW : 0;               // scale loads per wave and stage
  static constexpr int NPB = P + PS;
  static constexpr int STAGE = TILE + SCALES;
  // a tile's parameters: token scales, channel scales (rowwise), bias; two sets, the next tile's arriving while the
  // current one is in use
  static constexpr int PJ = (TM + TN) / 64 + (TN + 127) / 128, PP = (PJ + NW - 1) / NW;    // parameter loads, per wave
  static constexpr int PAR = 256 * PJ;
  static constexpr int OFF_PAR = KS * NST * STAGE, OFF_OUT = AHEAD ? OFF_PAR + 2 * PAR : 0;
  static constexpr int OUT_W = 2048;                                               // a 32 x 32 result tile per wave
  static constexpr int LDS = OFF_PAR + 2 * PAR + (AHEAD ? NW * OUT_W : 0);
  static constexpr int STORES = MT * NT * 2;                                       // result stores per wave and tile
  // waves per SIMD the registers are sized for: at least two, so that the accumulators stay in plain registers (with
  // one, the compiler moves them to the accumulation registers and copies them around the barriers)
  static constexpr int WAVES = 163840 / LDS * NW / 4 > 2 ? 163840 / LDS * NW / 4 : 2;
  static_assert(TM % (RP * NW) == 0 && TN % (RP * NW) == 0 && WM % 32 == 0 && WN % 32 == 0, "tile");
  static_assert(TM % 64 == 0 && TN % 64 == 0 && PAR % 16 == 0, "scale loads");
  static_assert(LDS <= 163840, "LDS");
  static_assert(NPB * (NST - 1) + PP + STORES <= 63, "vmcnt");

  const GemmArgs& a;
  uint8_t* lds;
  uint8_t* ring;     // this share's stages
  int lane, w, wm, wn, ks;
  uint32_t lbase;
  int m0, n0;
  uint32_t off[P];   // this lane's place in each of the wave's pieces, from the tile's first row

  __device__ __forceinline__ Gemm(const GemmArgs& a_, uint8_t* lds_) : a(a_), lds(lds_) {
    lane = threadIdx.x & 63;
    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    ks = KS > 1 ? w / NW : 0;
    w -= ks * NW;
    wm = w % WGM;
    wn = w / WGM;
    ring = lds + ks * NST * STAGE;
    lbase = lds_off(ring);
  }

  // The lane number, opaque to the compiler: what a phase derives from it is formed in that phase. Kept over the
  // products instead, those values do not fit the registers beside the accumulators.
  __device__ __forceinline__ int own_lane() const {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  }

  // Share ks of K takes stages ks, ks + KS, ...; every share the same count (a stage past K is all zeros).
  __device__ __forceinline__ int share_stages() const { return (a.k + KS * GK - 1) / (KS * GK); }
  __device__ __forceinline__ int stage_k(int s) const { return (KS * s + ks) * GK; }

  // Loads of a tile: its parameters (set `par`) and its first stages. Piece p = i NW + w holds rows 8 p .. 8 p + 7 of
  // the stage (X rows, then W rows), 8 lanes a row; LDS chunk c of a row holds its global chunk c ^ ((row >> 1) & 7),
  // so the fragment reads have no bank conflicts. Rows past the matrix read its last row (their results are not
  // stored).
  __device__ __forceinline__ void begin(int tm, int tn, int par) {
    m0 = tm * TM;
    n0 = tn * TN;
    const int lane = own_lane();
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const bool isx = i < PX;
      const int row = RP * ((isx ? i : i - PX) * NW + w) + lane / CPR, last = isx ? a.m - 1 - m0 : a.n - 1 - n0;
      off[i] = (uint32_t)(row < last ? row : last) * (uint32_t)a.k + 16 * ((lane % CPR) ^ swz(row));
    }
#pragma unroll
    for (int i = 0; i < PP; ++i) {   // parameter job: 64 dwords
      int j = i * NW + w;
      if (j >= PJ) j = 0;
      const uint32_t dst = lds_off(lds) + OFF_PAR + par * PAR + 256 * j;   // (every share writes the same)
      const void* p = gemm_zeros;
      uint32_t o = 0;
      if (j < TM / 64) {
        const int row = 64 * j + lane, last = a.m - 1 - m0;
        if (!MX) { p = a.xs + m0; o = 4 * (row < last ? row : last); }
      } else if (j < (TM + TN) / 64) {
        const int row = 64 * j - TM + lane, last = a.n - 1 - n0;
        if (!MX) { p = a.ws + n0; o = 4 * (row < last ? row : last); }
      } else if (a.bias) {   // pairs of channels; n is even
        const int pr = 64 * j - TM - TN + lane, last = (a.n - n0) / 2 - 1;
        p = a.bias + n0;
        o = 4 * (pr < last ? pr : last);
      }
      dma4(p, o, dst);
    }
    const int ns = share_stages();
#pragma unroll
    for (int s = 0; s < NST; ++s)
      if (s < ns) issue(s, s);
  }

  static __device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }
  __device__ __forceinline__ void issue(int s, int st) {
    const uint32_t lb = lbase + st * STAGE;
    const int k0 = stage_k(s);
    const uint8_t* xb = a.x + (int64_t)m0 * a.k + k0;
    const uint8_t* wb = a.w + (int64_t)n0 * a.k + k0;
    if (k0 + GK <= a.k) {
      dma_rows<PX, NW * 1024>(xb, off, lb + w * 1024);
      dma_rows<P - PX, NW * 1024>(wb, off + PX, lb + TM * GK + w * 1024);
    } else {
      const int l = own_lane(), lr = l / CPR, lc = l % CPR;
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const int row = RP * ((i < PX ? i : i - PX) * NW + w) + lr;
        const uint8_t* g = (i < PX ? xb : wb) + off[i];
        dma16_at(k0 + 16 * (lc ^ swz(row)) < a.k ? (const void*)g : (const void*)gemm_zeros,
                 lb + (i * NW + w) * 1024);
      }
    }
    issue_scales(s, st);
  }
  __device__ __forceinline__ void issue_scales(int s, int st) const {
    if constexpr (MX) {
      // scale loads: 64 rows each, one dword (a stage's four E8M0 scales) a row; the waves left over repeat the first
      // 64 rows, so every wave counts the same loads
      const int lane = own_lane(), k0 = stage_k(s), sk = k0 < a.k ? k0 / GK : 0;   // a stage past K: any finite scales
#pragma unroll
      for (int i = 0; i < PS; ++i) {
        int b = 64 * (i * NW + w);
        if (b >= TM + TN) b = 0;
        const bool isx = b < TM;
        const int row = b + lane - (isx ? 0 : TM), last = isx ? a.m - 1 - m0 : a.n - 1 - n0;
        dma4(isx ? a.xe + ((int64_t)sk * a.m + m0) * 4 : a.we + ((int64_t)sk * a.n + n0) * 4,
             4 * (uint32_t)(row < last ? row : last), lbase + st * STAGE + TILE + 4 * b);
      }
    }
  }

  struct Set {
    v8i x[MT], w[NT];
    int xe[MT], we[NT];
  };
  // Fragment reads: row r of each 32-row tile, half j of the stage: chunks 4 j + h and 4 j + 2 + h, i.e. K-block 2 j
  // in the operand's first 16 bytes and 2 j + 1 in its last (the MX scales' blocks).
  struct Place {
    int r, h, fo[2][2];
  };
  __device__ __forceinline__ Place place() const {
    Place p;
    const int l = own_lane();
    p.r = l & 31;
    p.h = l >> 5;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int c = 0; c < 2; ++c) p.fo[j][c] = p.r * GK + (((4 * j + 2 * c + p.h) ^ swz(p.r)) << 4);
    return p;
  }
  __device__ __forceinline__ v8i frag(const Place& pl, const uint8_t* p, int j) const {
    const v4i lo = *(const v4i*)(p + pl.fo[j][0]), hi = *(const v4i*)(p + pl.fo[j][1]);
    const v8i f = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return f;
  }
  __device__ __forceinline__ void read(const Place& pl, Set& f, int st, int j, int q) const {   // fragment q
    if (q < MT) f.x[q] = frag(pl, ring + st * STAGE + (wm * WM + 32 * q) * GK, j);
    else if (q < MT + NT) f.w[q - MT] = frag(pl, ring + st * STAGE + TM * GK + (wn * WN + 32 * (q - MT)) * GK, j);
  }
  __device__ __forceinline__ void read_scales(const Place& pl, Set& f, int st) const {
    if constexpr (MX) {
      const uint8_t* sc = ring + st * STAGE + TILE;
#pragma unroll
      for (int i = 0; i < MT; ++i) f.xe[i] = *(const int*)(sc + 4 * (wm * WM + 32 * i + pl.r)) >> (8 * pl.h);
#pragma unroll
      for (int i = 0; i < NT; ++i) f.we[i] = *(const int*)(sc + 4 * (TM + wn * WN + 32 * i + pl.r)) >> (8 * pl.h);
    }
  }

  // The products of `cur` (half JC of its stage), the reads of `nxt` (half 1 - JC, of stage st) between them.
  // DMA: also the loads of stage s (a whole one) into stage buffer sd, spread over the products.
  template <int JC, bool DMA>
  __device__ __forceinline__ void half(const Place& pl, v16f (&acc)[MT][NT], const Set& cur, Set& nxt, int st, int s,
                                       int sd) const {
    constexpr int PER = (MT + NT + MT * NT - 1) / (MT * NT), DPER = (P + MT * NT - 1) / (MT * NT);
    const uint8_t* xb = a.x + (int64_t)m0 * a.k + stage_k(s);
    const uint8_t* wb = a.w + (int64_t)n0 * a.k + stage_k(s);
    const uint32_t lb = lbase + sd * STAGE + w * 1024;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if constexpr (MX)   // byte 2 JC of the scale dword, shifted by the lane half: K-block 2 JC + h
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(cur.w[j], cur.x[i], acc[i][j], 0, 0, 2 * JC,
                                                                      cur.we[j], 2 * JC, cur.xe[i]);
        else
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(cur.w[j], cur.x[i], acc[i][j], 0, 0, 0, G_ONE,
                                                                      0, G_ONE);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < PER; ++q) read(pl, nxt, st, 1 - JC, PER * (i * NT + j) + q);
        if constexpr (DMA) {
#pragma unroll
          for (int q = 0; q < DPER; ++q) {
            const int p = DPER * (i * NT + j) + q;
            if (p < P) dma_rows<1, 0>(p < PX ? xb : wb, off + p, lb + p * NW * 1024);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    // products are pure register operations: without this the compiler moves them past the barrier
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) asm volatile("" : "+v"(acc[i][j]));
  }

  // The whole of K for the tile whose loads begin() issued; `pend`: STORES result stores of the tile before were
  // issued after them (retired in order behind them).
  __device__ __forceinline__ void sum(v16f (&acc)[MT][NT], bool pend) {
    const int ns = share_stages();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    if (ns < NST) wait_vmcnt<0>();
    else if (pend) wait_vmcnt<NPB * (NST - 1) + STORES>();
    else wait_vmcnt<NPB * (NST - 1)>();
    stage_barrier();
    const Place pl = place();
    Set fa, fb;
#pragma unroll
    for (int q = 0; q < MT + NT; ++q) read(pl, fa, 0, 0, q);
    read_scales(pl, fa, 0);
    int st = 0, behind = pend;
    auto pass = [&](auto steady, int s) {   // steady: stage s + NST exists and is a whole one
      constexpr bool STEADY = decltype(steady)::value;
      if constexpr (MX) {   // the stage's scales serve both halves
#pragma unroll
        for (int i = 0; i < MT; ++i) fb.xe[i] = fa.xe[i];
#pragma unroll
        for (int i = 0; i < NT; ++i) fb.we[i] = fa.we[i];
      }
      half<0, false>(pl, acc, fa, fb, st, 0, 0);
      // this wave's loads of stage s + 1 have landed (NST - 2 newer stages may be in flight)
      if (!STEADY && s + NST > ns) wait_vmcnt<0>();
      else if (behind) wait_vmcnt<NPB * (NST - 2) + STORES>();
      else wait_vmcnt<NPB * (NST - 2)>();
      behind = 0;
      asm volatile("" : "+s"(behind));   // opaque: the first pass is not peeled off the loop
      stage_barrier();   // every wave has read stage s and has its part of stage s + 1 in LDS
      const int sd = st;
      st = st + 1 == NST ? 0 : st + 1;
      if (!STEADY && s + NST < ns) issue(s + NST, sd);
      half<1, STEADY>(pl, acc, fb, fa, st, s + NST, sd);   // past the last stage it reads bytes that nothing uses
      if (STEADY) issue_scales(s + NST, sd);
      read_scales(pl, fa, st);
    };
    int s = 0;
    for (; (KS * (s + NST) + KS) * GK <= a.k; ++s) pass(std::true_type{}, s);
    for (; s < ns; ++s) pass(std::false_type{}, s);
  }

  // The shares' sums added into share 0's, through the (drained) stages; false in the other shares.
  __device__ __forceinline__ bool gather(v16f (&acc)[MT][NT]) const {
    if constexpr (KS > 1) {
      static_assert(KS == 2 && NW * MT * NT * 4096 <= OFF_PAR, "shares");
      stage_barrier();   // every wave has read its last fragments
      float* p = (float*)lds + (w * MT * NT) * 1024 + 4 * own_lane();
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float4* d = (float4*)(p + (i * NT + j) * 1024 + q * 256);
            if (ks) *d = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
          }
      stage_barrier();
      if (ks) return false;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float4 f = *(const float4*)(p + (i * NT + j) * 1024 + q * 256);
            acc[i][j][4 * q] += f.x; acc[i][j][4 * q + 1] += f.y; acc[i][j][4 * q + 2] += f.z; acc[i][j][4 * q + 3] += f.w;
          }
    }
    return true;
  }

  // The tile (m0_, n0_) from parameter set `par`: scales and bias in fp32, rounded to bf16, out through LDS a
  // 32 x 32 tile at a time (a wave's LDS accesses execute in order, so its 2 KB is reused without a wait), 16-byte
  // chunks XOR-swizzled by row.
  template <bool FULL>
  __device__ __forceinline__ void finish(const v16f (&acc)[MT][NT], int m0_, int n0_, int par) const {
    const uint8_t* pp = lds + OFF_PAR + par * PAR;
    uint8_t* ob = lds + OFF_OUT + w * OUT_W;
    const int lane = own_lane(), r = lane & 31, h = lane >> 5;
    const int row = lane >> 2, c = lane & 3;   // the 16 bytes this lane stores of rows row, row + 16
    uint8_t* op = (uint8_t*)(a.out + (int64_t)(m0_ + wm * WM) * a.n + n0_ + wn * WN);   // uniform
    const uint32_t o0 = (uint32_t)(2 * (row * a.n + 8 * c)), o1 = o0 + 32 * (uint32_t)a.n;
    const int rows = a.m - m0_ - wm * WM - row, cols = a.n - n0_ - wn * WN - 8 * c;   // left from this lane's place on
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      float sw[16], bi[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ch = wn * WN + 32 * j + 8 * q + 4 * h;   // this lane's four channels
        const uint2 b = *(const uint2*)(pp + (TM + TN) * 4 + 2 * ch);
        bi[4 * q] = __uint_as_float(b.x << 16);
        bi[4 * q + 1] = __uint_as_float(b.x & 0xFFFF0000u);
        bi[4 * q + 2] = __uint_as_float(b.y << 16);
        bi[4 * q + 3] = __uint_as_float(b.y & 0xFFFF0000u);
        if constexpr (!MX) {
          const float4 f = *(const float4*)(pp + TM * 4 + 4 * ch);
          sw[4 * q] = f.x; sw[4 * q + 1] = f.y; sw[4 * q + 2] = f.z; sw[4 * q + 3] = f.w;
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const float sx = MX ? 1.f : *(const float*)(pp + 4 * (wm * WM + 32 * i + r));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = acc[i][j][4 * q + e];
            // Results stay what callers had from the library GEMM that ran here before. Rowwise: the channel's scale,
            // the token's, the bias, each operation rounded (with exact sums the same bits as hipBLASLt at every shape
            // tried; other orders or an FMA differ in a few of 1e5 values, which FP8 layers after it amplify). MX: the
            // sum is cut to bf16 (toward zero), then the bias added, as the separate addition did.
            if constexpr (MX) y[e] = __uint_as_float(__float_as_uint(v) & 0xFFFF0000u) + bi[4 * q + e];
            else y[e] = (v * sw[4 * q + e]) * sx + bi[4 * q + e];
          }
          typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
          const bf2 lo = {(__bf16)y[0], (__bf16)y[1]}, hi = {(__bf16)y[2], (__bf16)y[3]};
          *(uint2*)(ob + r * 64 + ((q ^ ((r >> 2) & 3)) << 4) + 8 * h) =
              make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
        }
        const uint8_t* rp = ob + row * 64 + ((c ^ ((row >> 2) & 3)) << 4);
        const v4i v0 = *(const v4i*)rp, v1 = *(const v4i*)(rp + 1024);
        uint8_t* dst = op + (int64_t)(64 * i) * a.n + 64 * j;
        if (FULL) {
          *(v4i*)(dst + o0) = v0;
          *(v4i*)(dst + o1) = v1;
        } else if (32 * j < cols) {
          if (32 * i < rows) *(v4i*)(dst + o0) = v0;
          if (32 * i + 16 < rows) *(v4i*)(dst + o1) = v1;
        }
      }
    }
  }
};

// Tile order: 4 token tiles for each channel tile, so the tiles an XCD works on at a time share few operand rows.
// HALF: mt x nt are tiles twice as wide, each two tiles in a row of this order.
template <bool HALF>
__device__ __forceinline__ void tile_at(const GemmArgs& a, int id, int& tm, int& tn) {
  const int sub = HALF ? id & 1 : 0;
  if (HALF) id >>= 1;
  constexpr int GM = 4;
  const int grp = id / (GM * a.nt), first = grp * GM, gm = a.mt - first < GM ? a.mt - first : GM;
  const int in = id - grp * GM * a.nt;
  tm = first + in % gm;
  tn = HALF ? 2 * (in / gm) + sub : in / gm;
}

// Persistent: workgroup g runs on XCD g % 8, each XCD takes a contiguous range of the tiles, dealt round-robin among
// its workgroups. AHEAD: the next tile's parameters and first stages are loaded while this one is finished and stored.
template <int TM, int TN, int WGM, int WGN, int NST, int KS, bool AHEAD, bool HALF, bool MX>
__global__ __launch_bounds__(64 * WGM * WGN * KS, (Gemm<TM, TN, WGM, WGN, NST, KS, AHEAD, MX>::WAVES))
void gemm_kernel(GemmArgs a) {
  using G = Gemm<TM, TN, WGM, WGN, NST, KS, AHEAD, MX>;
  static_assert(KS == 1 || !AHEAD, "the shares are added in the stages");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[G::LDS];
  const int x = blockIdx.x & 7, gx = gridDim.x >> 3;
  const int lo = a.first + (int)((int64_t)x * a.tiles / 8), hi = a.first + (int)((int64_t)(x + 1) * a.tiles / 8);
  int id = lo + (blockIdx.x >> 3), tm, tn;
  const auto seek = [&]() {   // the tile of id, passing over halves past the last channel; false at the range's end
    for (; id < hi; id += gx) {
      tile_at<HALF>(a, id, tm, tn);
      if (!HALF || tn * TN < a.n) return true;
    }
    return false;
  };
  if (!seek()) return;
  G g(a, lds);
  int par = 0;
  g.begin(tm, tn, 0);
  bool pend = false;
  for (;;) {
    v16f acc[G::MT][G::NT];
    g.sum(acc, pend);
    const int m0 = g.m0, n0 = g.n0;
    id += gx;
    const bool more = seek(), mine = g.gather(acc);
    stage_barrier();   // every wave has read its last fragments (or the other share's sums)
    if (AHEAD && more) g.begin(tm, tn, par ^ 1);
    const bool full = m0 + TM <= a.m && n0 + TN <= a.n;
    if (mine) {
      if (full) g.template finish<true>(acc, m0, n0, par);
      else g.template finish<false>(acc, m0, n0, par);
    }
    if (!more) return;
    if (AHEAD) {
      pend = full;
      if (!full) wait_vmcnt<0>();
      par ^= 1;
    } else {
      stage_barrier();   // every wave has read its results back
      g.begin(tm, tn, 0);
    }
  }
}

// Tiles [first, first + tiles) of a's order (all of them when tiles is 0). HALF: a.mt, a.nt are set by the caller.
template <int TM, int TN, int WGM, int WGN, int NST, int KS, bool AHEAD, bool HALF, bool MX>
static void gemm_launch(GemmArgs& a, hipStream_t stream, int64_t first = 0, int64_t tiles = 0) {
  using G = Gemm<TM, TN, WGM, WGN, NST, KS, AHEAD, MX>;
  if (!HALF) {
    a.mt = (a.m + TM - 1) / TM;
    a.nt = (a.n + TN - 1) / TN;
  }
  a.first = (int)first;
  a.tiles = (int)(tiles ? tiles : (int64_t)a.mt * a.nt);
  const int64_t per = ((int64_t)a.tiles + 7) / 8, cap = 32 * (163840 / G::LDS);
  hipLaunchKernelGGL((gemm_kernel<TM, TN, WGM, WGN, NST, KS, AHEAD, HALF, MX>),
                     dim3((unsigned)(8 * (per < cap ? per : cap))), dim3(G::THREADS), 0, stream, a);
}

// The tile for a shape, by tile counts (one workgroup per CU but for the 64 x 64 form: 256 CUs). Measured in us at
// (tokens x K x channels), graph replays of 20 calls, rowwise:
//                        64 x 64  its K split  128 x 128  192 x 192  256 x 256   library GEMM it replaced
//   512 x 1536 x 1536        5.8          6.2        8.1       11.1       16.8      6.6
//   64 x 8960 x 1536        17.4         14.3       26.4       41.2       68.6     13.4
//   1508 x 1536 x 1536      10.8         13.9        8.9       11.9       17.7     11.7
//   1508 x 8960 x 1536      43.5         43.9       29.7       44.0       75.8     40.6
//   700 x 1536 x 8960       21.0         31.0       17.4       14.3       19.6     16.9
//   6032 x 8960 x 1536       133          138         96         67         81       90
//   1508 x 1536 x 8960      42.4         59.9       31.3       28.3       23.0     27.2
//   3016 x 1536 x 8960      80.4          112       54.2       48.9       42.4     48.6
// So: the smallest tile that gives every CU at most one tile, as a round's time falls with the tile; K in two shares
// once it is long (3.1 us less at K = 8960, 0.4 us more at 1536). Past one round of 256 x 256 tiles, the smaller of
// rounds x (stages x time of a stage + fixed part) as fitted to these figures. The MX form of 256 x 256 does not fit
// the registers beside its scales (29.3 us against 29.3 for 192 x 192 at 1508 x 1536 x 8960, 114 against 102 at 6032
// tokens), so MX stops at 192 x 192.
// Behind the library GEMM by itself where tiles are few: 8960 x 1536 takes 14.3-14.8 against 10.4-10.8 us at 16 to 128
// tokens (14.6 against 13.5 at 64), 16.1 against 15.3 at 257, 27.5 against 26.1-26.7 at 700 and 1024; 1536 x 1536 and
// 2048 x 1024 are 0.5-0.9 us behind at up to 128 (24 tiles of long K on 256 CUs: K is not split over workgroups). A call
// from Python is shorter all the same, 20 us of host work against 40; in a captured graph these shapes lose.
// A last round of at most 128 such tiles goes out as half tiles in a launch of its own, which takes about half a
// round (a half past the last channel is passed over): feed-forward at 6032 tokens 197.8 -> 192.0 us. (In the same launch,
// after the whole tiles, the second tile body cost 28 spilled registers and 7 us.)
template <bool MX>
static int gemm_dispatch(GemmArgs& a, hipStream_t stream) {
  const auto tiles = [&](int64_t t) { return ((a.m + t - 1) / t) * ((a.n + t - 1) / t); };
  const auto rounds = [&](int64_t t) { return (tiles(t) + 255) / 256; };
  const int64_t ns = (a.k + GK - 1) / GK, all = tiles(256), rest = all % 256;
  const bool halves = all > 256 && rest > 0 && rest <= 128;
  const int64_t half_rounds = all / 256 * 2 + (rest == 0 ? 0 : halves ? 1 : 2);
  if (tiles(64) <= 256) {
    if (a.k >= 4096) gemm_launch<64, 64, 2, 2, 4, 2, false, false, MX>(a, stream);
    else gemm_launch<64, 64, 2, 2, 4, 1, false, false, MX>(a, stream);
  } else if (tiles(128) <= 256) {
    gemm_launch<128, 128, 4, 2, 4, 1, false, false, MX>(a, stream);
  } else if (MX || rounds(192) == 1 || rounds(192) * (82 * ns + 700) <= half_rounds * (50 * ns + 550)) {
    gemm_launch<192, 192, 2, 6, 3, 1, false, false, MX>(a, stream);
  } else {
    if constexpr (!MX) {
      if (halves) {
        gemm_launch<256, 256, 4, 2, 2, 1, true, false, false>(a, stream, 0, all - rest);
        gemm_launch<256, 128, 4, 2, 3, 1, false, true, false>(a, stream, 2 * (all - rest), 2 * rest);
      } else {
        gemm_launch<256, 256, 4, 2, 2, 1, true, false, false>(a, stream);
      }
    }
  }
  if (hipGetLastError() != hipSuccess) return LBW_E_LAUNCH;
  return LBW_OK;
}

// 32-bit row offsets inside a tile (256 rows), 31-bit tile counts
static int gemm_check(const void* x, const void* xs, const void* w, const void* ws, const uint16_t* bias, int64_t m,
                      int64_t n, int64_t k, const uint16_t* out) {
  if (!x || !xs || !w || !ws || !out) return LBW_E_NULL;
  if (m <= 0 || n <= 0 || k <= 0 || n % 16 != 0 || k % 16 != 0) return LBW_E_SHAPE;
  if (m > (1 << 30) || n > (1 << 22) || k > (1 << 22) || ((m + 63) / 64) * ((n + 63) / 64) > (1 << 30)) return LBW_E_SHAPE;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15 || ((uintptr_t)xs | (uintptr_t)ws | (uintptr_t)bias) & 3)
    return LBW_E_ALIGN;
  return check_device();
}

}  // namespace lbw

using namespace lbw;

extern "C" int lbw_gemm_fp8_rows(const uint8_t* x8, const float* x_scale, const uint8_t* w8, const float* w_scale,
                                 const uint16_t* bias, int64_t m, int64_t n, int64_t k, uint16_t* out, void* stream) {
  if (const int st = gemm_check(x8, x_scale, w8, w_scale, bias, m, n, k, out)) return st;
  GemmArgs a{};
  a.x = x8; a.w = w8; a.xs = x_scale; a.ws = w_scale; a.bias = bias; a.out = out;
  a.m = (int)m; a.n = (int)n; a.k = (int)k;
  return gemm_dispatch<false>(a, (hipStream_t)stream);
}

extern "C" int lbw_gemm_fp8_mx(const uint8_t* x8, const uint8_t* x_scale_t, const uint8_t* w8, const uint8_t* w_scale_t,
                               const uint16_t* bias, int64_t m, int64_t n, int64_t k, uint16_t* out, void* stream) {
  if (const int st = gemm_check(x8, x_scale_t, w8, w_scale_t, bias, m, n, k, out)) return st;
  if (k % GK != 0) return LBW_E_SHAPE;
  GemmArgs a{};
  a.x = x8; a.w = w8; a.xe = x_scale_t; a.we = w_scale_t; a.bias = bias; a.out = out;
  a.m = (int)m; a.n = (int)n; a.k = (int)k;
  return gemm_dispatch<true>(a, (hipStream_t)stream);
}
