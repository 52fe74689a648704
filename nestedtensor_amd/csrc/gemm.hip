// Packed projection GEMM for nested multi-head attention (gfx950 MFMA).
//
//   C[M, N] = A[M, K] * W[N, K]^T + bias[N]
//
// A is the packed token buffer viewed as [T, E] (no padded rows exist), W is a
// torch Linear weight, so both operands are K-contiguous: every MFMA operand
// fragment is one 16-byte run of a row.  A workgroup owns a BM x BN tile of C,
// its wavefronts a WAVES_M x WAVES_N grid of (WM*32) x (WN*32) sub-tiles made of
// 32x32 MFMA blocks (fp32 accumulate; f16 / bf16: v_mfma_f32_32x32x16_*, fp32:
// v_mfma_f32_32x32x2_f32).  K is walked in tiles of 128 bytes per row.  When K
// is a whole number of tiles the K tiles go from global memory straight into LDS
// (global_load_lds_dwordx4: no staging registers, no ds_write), two to three
// tiles resident, in an unpadded layout whose 16-byte pieces are XOR-swizzled so
// that the 128-bit fragment reads of 16 consecutive lanes fall into distinct
// banks; any other K takes a register-staged loop with padded LDS rows and
// element-wise tails.
//
// Three kernels.  split_kernel, fp32 of at least 192 k: operands split into three bf16 parts
// for the bf16 instruction.  phased_kernel, for problems that fill the chip and K of at least two whole
// K tiles: eight wavefronts in two groups half a phase apart, tile shapes of 128 to 320 rows
// by 128 or 256 columns.  linear_kernel, whose wavefronts all do the same thing at the same
// time: a problem with fewer 256x128 tiles than half the CUs (the query and output
// projections of cross-attention, a few thousand rows) gets 128x64 tiles of four wavefronts,
// or 128x128 when those would not fit in one round (its duration is one tile's life, and a
// quarter of a tile on four times as many CUs ends sooner: 3200 x 512 x 512 10.6 -> 6.3 us;
// the fused in-projection of a layer of a few hundred tokens 16.0 -> 11.6 us), at most 64
// columns 128x64 tiles, ragged K tiles of 256 rows by 128, 192 or 256 columns, and those
// also where few K tiles or rows that end inside a 16-byte piece leave phased_kernel
// nothing to gain (choose_tile).
//
// Epilogues:
//   plain  - C row-major + bias;
//   QKV    - the fused in-projection of self-attention: columns [0, n_split)
//            (Q and K) go row-major into C, columns [n_split, N) (V) are written
//            TRANSPOSED into Vt[n - n_split][m] so that the attention kernel
//            finds V^T tiles key-contiguous.
#include "nt_common.h"

#include <type_traits>

namespace nt {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float acc16 __attribute__((ext_vector_type(16)));

template <typename T> struct Mma;

template <> struct Mma<_Float16> {
  typedef half8 Frag;
  static constexpr int kK = 16;  // K per MFMA
  static __device__ __forceinline__ acc16 run(Frag a, Frag b, acc16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

template <> struct Mma<__bf16> {
  typedef bf16x8 Frag;
  static constexpr int kK = 16;
  static __device__ __forceinline__ acc16 run(Frag a, Frag b, acc16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

// fp32: v_mfma_f32_32x32x2_f32 contracts two k values per instruction, one per
// lane half.  Which two is free as long as both operands agree, so a fragment is
// the same 16-byte piece of a row as for the 16-bit types (lane half g holds
// k = 8 s + 4 g .. + 3 of step s) and is spent over four instructions: the LDS
// reads are the conflict-free 128-bit ones of the swizzled layout instead of
// 4-byte column reads (which collide four to eight ways in it).
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <> struct Mma<float> {
  typedef f32x4 Frag;
  static constexpr int kK = 8;
  static __device__ __forceinline__ acc16 run(Frag a, Frag b, acc16 c) {
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[0], b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[1], b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[2], b[2], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a[3], b[3], c, 0, 0, 0);
  }
};

template <int WAVES_M_, int WAVES_N_, int WM_, int WN_, int BKB_>
struct GemmCfg {
  static constexpr int kWavesM = WAVES_M_, kWavesN = WAVES_N_, kWM = WM_, kWN = WN_;
  static constexpr int kThreads = 64 * WAVES_M_ * WAVES_N_;
  static constexpr int kWavesPerSimd = kThreads >= 512 ? 2 : 1;   // the kernel is compiled for this occupancy
  static constexpr int kBM = WAVES_M_ * WM_ * 32;
  static constexpr int kBN = WAVES_N_ * WN_ * 32;
  static constexpr int kRowBytes = BKB_;              // K-tile bytes per row
  static constexpr int kLdsRow = BKB_ + 16;           // padded LDS row
  static constexpr int kChunksPerRow = BKB_ / 16;
  static constexpr int kChunks = (kBM + kBN) * kChunksPerRow;
  static constexpr int kPerA = kBM * kChunksPerRow / kThreads;   // A pieces per thread
  static constexpr int kPerB = kBN * kChunksPerRow / kThreads;   // W pieces per thread
  static constexpr int kPerThread = kPerA + kPerB;
  static constexpr int kBufBytes = (kBM + kBN) * kLdsRow;
  // direct global -> LDS loads: unpadded rows, the K tiles of A and of W in a ring
  // each, three tiles deep
  static constexpr int kATileBytes = kBM * BKB_;
  static constexpr int kBTileBytes = kBN * BKB_;
  static constexpr int kLdsBudget = 160 * 1024 - 2048;
  static constexpr bool kThreeOfBoth = 3 * (kATileBytes + kBTileBytes) <= kLdsBudget;
  static constexpr int kBufsB = kThreeOfBoth ? 3 : 2;
  static constexpr int kBufsA = kThreeOfBoth ? 3 : 2;
  static constexpr int kRingBytes = kBufsA * kATileBytes + kBufsB * kBTileBytes;
  // tile buffers (kernels for a ragged K use two padded, register-staged buffers)
  static constexpr int kLdsBytes = kRingBytes > 2 * kBufBytes ? kRingBytes : 2 * kBufBytes;
  static_assert((kBM * kChunksPerRow) % kThreads == 0 && (kBN * kChunksPerRow) % kThreads == 0,
                "tile pieces must divide among the threads");
};

template <typename T>
struct GemmArgs {
  const T* A;
  int64_t lda;
  const T* W;
  const T* bias;
  T* C;
  int64_t ldc;
  int64_t M, N, K;
  T* Vt;            // QKV epilogue: transposed destination of columns >= n_split
  int64_t ldvt;
  int64_t n_split;
  int act;          // row-major tiles: 0 none, 1 relu, 2 gelu (erf) applied to A W^T + bias
};

// 16-byte piece of a row at element k.
// ALIGNED_K (K is a multiple of the K tile): branch-free and mask-free.
// Out-of-range rows are clamped to the last row -- they only feed accumulators
// that are never stored -- and the caller clamps the K tile index, so every
// address is valid and nothing has to be zeroed.  This matters: control flow
// around the loads, or a mask applied to the loaded value, makes the wavefront
// wait for the load right away and serialises the global-load / MFMA pipeline.
// Otherwise (any K): element-wise tail handling.
template <typename T, bool ALIGNED_K>
__device__ __forceinline__ u32x4 load_chunk(const T* base, int64_t ld, int64_t row, int64_t nrows,
                                            int64_t k, int64_t K) {
  constexpr int kPer = 16 / sizeof(T);
  if (ALIGNED_K) {
    const int64_t r = row < nrows ? row : nrows - 1;
    return load16_unaligned(reinterpret_cast<const char*>(base + r * ld + k));
  }
  u32x4 v = {0, 0, 0, 0};
  if (row < nrows) {
    const T* p = base + row * ld + k;
    if (k + kPer <= K) {
      v = load16_unaligned(reinterpret_cast<const char*>(p));
    } else {
      T tmp[kPer];
#pragma unroll
      for (int j = 0; j < kPer; ++j) tmp[j] = (k + j < K) ? p[j] : (T)0.0f;
      __builtin_memcpy(&v, tmp, 16);
    }
  }
  return v;
}

// kEpiAct: the plain epilogue with the activation of GemmArgs::act; a kernel of
// its own, because even a never-taken activation branch in the plain epilogue
// costs the projection GEMMs 10 % (measured)
enum { kEpiPlain = 0, kEpiQkv = 1, kEpiAct = 2 };

// LDS a wavefront needs to store its accumulators: one 32-row strip.
template <typename T, int WM, int WN, bool VT_OUT>
constexpr int strip_bytes() {
  return 32 * ((VT_OUT ? WM : WN) * 32 * (int)sizeof(T) + 16);
}

// Epilogue of one wavefront: its (WM * 32) x (WN * 32) accumulators, whose first row
// is m_wave and whose first column is n0 + n_wave, go to C (or, VT_OUT, transposed to
// Vt) with the bias added.
//
// The accumulators of a 32x32 MFMA block hold, per lane, four runs of four
// consecutive rows of one column of D.  Both operand fragments have the same
// register layout, so exchanging them transposes D for free: a tile that goes
// row-major into C is computed as C^T (a lane then holds runs of four
// consecutive COLUMNS of one row of C), a V tile as C (runs of four consecutive
// tokens of one feature = consecutive elements of a Vt row).  The epilogue
// moves each 32-row strip through a private LDS region of the wavefront, 8 or
// 16 bytes per lane in, and back out as 16-byte pieces of whole rows, so the
// global stores are row-contiguous instead of 2 bytes per lane.
template <typename T, int WM, int WN, bool VT_OUT, bool ACT>
__device__ __forceinline__ void store_tile(const GemmArgs<T>& a, const acc16 (&acc)[WM][WN], int64_t m_wave,
                                           int64_t n0, int n_wave, char* strip, const float* lds_bias) {
  constexpr int kPer = 16 / sizeof(T);
  const int lane = threadIdx.x & 63;
  const int l32 = lane & 31;
  const int g = lane >> 5;
  constexpr int kStripW = VT_OUT ? WM : WN;                    // 32-wide blocks per strip row
  constexpr int kStripRow = kStripW * 32 * (int)sizeof(T) + 16;
  constexpr int kCpr = kStripW * 32 * (int)sizeof(T) / 16;    // 16-byte pieces per strip row
  typedef T Quad __attribute__((ext_vector_type(4)));

  if (!VT_OUT) {
    // acc[i][j][e] = C[row, col], row = .. + i*32 + l32, col = .. + j*32 + 8*(e/4) + 4*g + e%4
    const bool row_vec_ok = (a.ldc * (int64_t)sizeof(T)) % 16 == 0 &&
                            reinterpret_cast<uintptr_t>(a.C) % 16 == 0;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        auto block = [&](auto act) __attribute__((always_inline)) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int c0 = j * 32 + 8 * r + 4 * g;
            const float4 bv = *reinterpret_cast<const float4*>(lds_bias + n_wave + c0);
            Quad q;
            q[0] = (T)act(acc[i][j][4 * r + 0] + bv.x);
            q[1] = (T)act(acc[i][j][4 * r + 1] + bv.y);
            q[2] = (T)act(acc[i][j][4 * r + 2] + bv.z);
            q[3] = (T)act(acc[i][j][4 * r + 3] + bv.w);
            *reinterpret_cast<Quad*>(strip + l32 * kStripRow + c0 * (int)sizeof(T)) = q;
          }
        };
        // The activation of a feed-forward layer, in fp32 before the one rounding.  The
        // choice (a kernel argument) is made once per 32 x 32 block: made per element it
        // kept the sixteen chains of a lane apart, and nothing else runs beside them.
        if (ACT && a.act == 2) {
          block([](float v) { return gelu_erf(v); });
        } else if (ACT && a.act == 1) {
          block([](float v) { return fmaxf(v, 0.0f); });
        } else {
          block([](float v) { return v; });
        }
      }
      __builtin_amdgcn_wave_barrier();   // LDS serves a wavefront's accesses in order
#pragma unroll
      for (int it = 0; it < 32 * kCpr / 64; ++it) {
        const int idx = it * 64 + lane;
        const int r = idx / kCpr, c = idx % kCpr;
        const int64_t row = m_wave + i * 32 + r;
        const int64_t col = n0 + n_wave + c * kPer;
        const u32x4 v = *reinterpret_cast<const u32x4*>(strip + r * kStripRow + c * 16);
        if (row < a.M && col < a.N) {
          T* dst = a.C + row * a.ldc + col;
          if (row_vec_ok && col + kPer <= a.N) {
            store16(reinterpret_cast<char*>(dst), v);
          } else {
            T tmp[kPer];
            __builtin_memcpy(tmp, &v, 16);
#pragma unroll
            for (int e = 0; e < kPer; ++e)
              if (col + e < a.N) dst[e] = tmp[e];
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  } else {
    // acc[i][j][e] = C[row, col], row = .. + i*32 + 8*(e/4) + 4*g + e%4, col = .. + j*32 + l32
    const bool row_vec_ok = (a.ldvt * (int64_t)sizeof(T)) % 16 == 0 &&
                            reinterpret_cast<uintptr_t>(a.Vt) % 16 == 0;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const float bv = lds_bias[n_wave + j * 32 + l32];
#pragma unroll
      for (int i = 0; i < WM; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          Quad q;
#pragma unroll
          for (int e = 0; e < 4; ++e) q[e] = (T)(acc[i][j][4 * r + e] + bv);
          *reinterpret_cast<Quad*>(strip + l32 * kStripRow +
                                   (i * 32 + 8 * r + 4 * g) * (int)sizeof(T)) = q;
        }
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int it = 0; it < 32 * kCpr / 64; ++it) {
        const int idx = it * 64 + lane;
        const int r = idx / kCpr, c = idx % kCpr;
        const int64_t col = n0 + n_wave + j * 32 + r;           // feature
        const int64_t row = m_wave + c * kPer;          // first token of the piece
        const u32x4 v = *reinterpret_cast<const u32x4*>(strip + r * kStripRow + c * 16);
        if (col < a.N && row < a.M) {
          T* dst = a.Vt + (col - a.n_split) * a.ldvt + row;
          if (row_vec_ok && row + kPer <= a.M) {
            store16(reinterpret_cast<char*>(dst), v);
          } else {
            T tmp[kPer];
            __builtin_memcpy(tmp, &v, 16);
#pragma unroll
            for (int e = 0; e < kPer; ++e)
              if (row + e < a.M) dst[e] = tmp[e];
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// One BM x BN tile.  VT_OUT marks a V tile of the fused QKV projection, whose
// result goes transposed into Vt.
template <typename T, class Cfg, bool VT_OUT, bool ALIGNED_K, bool ACT = false>
__device__ __forceinline__ void gemm_tile(const GemmArgs<T>& a, int64_t m0, int64_t n0, char* lds) {
  typedef Mma<T> MM;
  typedef typename MM::Frag Frag;
  constexpr int kPer = 16 / sizeof(T);
  constexpr int kBK = Cfg::kRowBytes / sizeof(T);
  constexpr int kSteps = kBK / MM::kK;
  constexpr int kFragBytes = (MM::kK / 2) * sizeof(T);
  constexpr int WM = Cfg::kWM, WN = Cfg::kWN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / Cfg::kWavesN;
  const int wn = wave % Cfg::kWavesN;
  const int l32 = lane & 31;
  const int g = lane >> 5;

  acc16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int64_t nk = (a.K + kBK - 1) / kBK;

  // bias of the tile's columns as fp32, behind the tile buffers (visible after
  // the first barrier below)
  if (tid < Cfg::kBN) {
    const int64_t col = n0 + tid;
    reinterpret_cast<float*>(lds + Cfg::kLdsBytes)[tid] =
        (a.bias && col < a.N) ? (float)a.bias[col] : 0.0f;
  }

  if (ALIGNED_K) {
    // K tiles travel global -> LDS directly (global_load_lds_dwordx4): no staging
    // registers, no ds_write instructions.  A wavefront-level load writes its 64
    // 16-byte pieces to 1 KiB of consecutive LDS, i.e. eight unpadded 128-byte rows,
    // so bank conflicts of the fragment reads are avoided by WHICH piece of the row a
    // lane fetches: slot p of row r holds piece p ^ ((r >> 1) & 7).  The compiler
    // does not see these loads (inline asm), so their completion is awaited by hand
    // before the barrier that publishes the tile.  The asm writes M0 (the LDS
    // destination).  M0 cannot be declared as a clobber: the compiler treats it as a
    // reserved register, warns and ignores the entry.  The s_mov and the load that
    // reads M0 sit in one asm statement, so the compiler cannot put anything
    // between them; in the other direction the rule for this file is that nothing
    // makes the compiler keep a value of its own in M0 across these statements (no
    // LDS-direct builtin, no dynamic register indexing, no sendmsg).
    static_assert(Cfg::kRowBytes == 128 && Cfg::kBM % 64 == 0 && Cfg::kBN % 64 == 0,
                  "1 KiB blocks of eight rows, a whole number of them per wavefront");
    constexpr int kWaves = Cfg::kThreads / 64;
    constexpr int kNA = Cfg::kBM / 8 / kWaves;      // 1 KiB blocks of an A tile per wavefront
    constexpr int kNW = Cfg::kBN / 8 / kWaves;      // ... of a W tile
    constexpr int kRA = Cfg::kBufsA, kRW = Cfg::kBufsB;
    static_assert(kRA >= 2 && kRW >= 2 && kRA - kRW <= 1 && kRW - kRA <= 1, "the wait below counts on the issue order");
    constexpr bool kWLast = kRW > kRA;              // the deeper ring is issued last in an iteration
    constexpr int kInFlight = (kRA - 2) * kNA + (kRW - 2) * kNW;   // loads that may be outstanding at a barrier
    static_assert(kInFlight <= 63, "vmcnt is a 6-bit counter");
    const char* aptr[kNA];
    const char* wptr[kNW];
#pragma unroll
    for (int i = 0; i < kNA; ++i) {
      const int r = (i * kWaves + wave) * 8 + (lane >> 3);
      const int c = (lane & 7) ^ ((r >> 1) & 7);
      int64_t row = m0 + r;
      row = row < a.M ? row : a.M - 1;
      aptr[i] = reinterpret_cast<const char*>(a.A + row * a.lda + c * kPer);
    }
#pragma unroll
    for (int i = 0; i < kNW; ++i) {
      const int r = (i * kWaves + wave) * 8 + (lane >> 3);
      const int c = (lane & 7) ^ ((r >> 1) & 7);
      int64_t row = n0 + r;
      row = row < a.N ? row : a.N - 1;
      wptr[i] = reinterpret_cast<const char*>(a.W + row * a.K + c * kPer);
    }
    const unsigned lds_base = (unsigned)reinterpret_cast<uintptr_t>(lds);
    constexpr int kWRing = kRA * Cfg::kATileBytes;          // the W ring lies behind the A ring
    auto dma_a = [&](int buf, int64_t kt_in) {
      const int64_t kt = kt_in >= nk ? nk - 1 : kt_in;    // past the end: re-read, never used
#pragma unroll
      for (int i = 0; i < kNA; ++i) {
        const unsigned dst = __builtin_amdgcn_readfirstlane(
            lds_base + (unsigned)(buf * Cfg::kATileBytes + (i * kWaves + wave) * 1024));
        const char* src = aptr[i] + kt * Cfg::kRowBytes;
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     :: "v"(src), "s"(dst) : "memory");
      }
    };
    auto dma_w = [&](int buf, int64_t kt_in) {
      const int64_t kt = kt_in >= nk ? nk - 1 : kt_in;
#pragma unroll
      for (int i = 0; i < kNW; ++i) {
        const unsigned dst = __builtin_amdgcn_readfirstlane(
            lds_base + (unsigned)(kWRing + buf * Cfg::kBTileBytes + (i * kWaves + wave) * 1024));
        const char* src = wptr[i] + kt * Cfg::kRowBytes;
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     :: "v"(src), "s"(dst) : "memory");
      }
    };
    const int sw = (l32 >> 1) & 7;
    auto read_frags = [&](Frag* fa, Frag* fb, int abuf, int wbuf, int s) {
      const char* a_base = lds + abuf * Cfg::kATileBytes + (wm * WM * 32 + l32) * 128;
      const char* b_base = lds + kWRing + wbuf * Cfg::kBTileBytes + (wn * WN * 32 + l32) * 128;
      const int off = s * MM::kK * (int)sizeof(T) + g * kFragBytes;   // byte offset in the row
      const int koff = ((((off >> 4) ^ sw)) << 4) | (off & 15);
#pragma unroll
      for (int i = 0; i < WM; ++i)
        fa[i] = *reinterpret_cast<const Frag*>(a_base + i * 32 * 128 + koff);
#pragma unroll
      for (int j = 0; j < WN; ++j)
        fb[j] = *reinterpret_cast<const Frag*>(b_base + j * 32 * 128 + koff);
    };
    // While K tile kt is multiplied, the tiles kt + 1 .. kt + kRA - 1 of A and
    // kt + 1 .. kt + kRW - 1 of W are resident or in flight.  Loads complete in the
    // order of issue and every iteration issues the tile of the deeper ring last,
    // so when at most kInFlight loads are outstanding, tile kt + 1 of both has landed.
    // Prologue: tiles in the order the loop would have issued them.
#pragma unroll
    for (int j = 0; j < (kRA > kRW ? kRA : kRW) - 1; ++j) {
      if (!kWLast && j < kRW - 1) dma_w(j, j);
      if (j < kRA - 1) dma_a(j, j);
      if (kWLast && j < kRW - 1) dma_w(j, j);
    }
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kInFlight) : "memory");
    __syncthreads();
    int abuf = 0, wbuf = 0;
    Frag fa[2][WM], fb[2][WN];
    for (int64_t kt = 0; kt < nk; ++kt) {
      // (kt + kR - 1) % kR: free since the last barrier
      // This iteration's loads (the tile of the shallower ring first) are not issued
      // in one burst: a DMA load occupies the issuing wavefront until the memory
      // path has taken its 64 addresses, so a burst keeps every wavefront of the
      // workgroup from its matrix instructions at the same time.  They are dealt out
      // behind the k-steps instead.
      const int a_new = abuf == 0 ? kRA - 1 : abuf - 1;     // (kt + kR - 1) % kR: free since the last barrier
      const int w_new = wbuf == 0 ? kRW - 1 : wbuf - 1;
      const int64_t a_kt = kt + kRA - 1 >= nk ? nk - 1 : kt + kRA - 1;   // past the end: re-read, never used
      const int64_t w_kt = kt + kRW - 1 >= nk ? nk - 1 : kt + kRW - 1;
      auto dma_one = [&](int idx) {
        const bool is_w = kWLast ? idx >= kNA : idx < kNW;
        const int i = kWLast ? (is_w ? idx - kNA : idx) : (is_w ? idx : idx - kNW);
        const unsigned off = is_w ? (unsigned)(kWRing + w_new * Cfg::kBTileBytes) : (unsigned)(a_new * Cfg::kATileBytes);
        const unsigned dst = __builtin_amdgcn_readfirstlane(lds_base + off + (unsigned)((i * kWaves + wave) * 1024));
        const char* src = is_w ? wptr[i] + w_kt * Cfg::kRowBytes : aptr[i] + a_kt * Cfg::kRowBytes;
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     :: "v"(src), "s"(dst) : "memory");
      };
      constexpr int kLoads = kNA + kNW;
      read_frags(fa[0], fb[0], abuf, wbuf, 0);
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        if (s + 1 < kSteps) read_frags(fa[(s + 1) & 1], fb[(s + 1) & 1], abuf, wbuf, s + 1);
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int jj = 0; jj < WN; ++jj) {
            if (VT_OUT) {
              acc[i][jj] = MM::run(fa[s & 1][i], fb[s & 1][jj], acc[i][jj]);
            } else {
              acc[i][jj] = MM::run(fb[s & 1][jj], fa[s & 1][i], acc[i][jj]);
            }
          }
#pragma unroll
        for (int idx = s * kLoads / kSteps; idx < (s + 1) * kLoads / kSteps; ++idx) dma_one(idx);
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kInFlight) : "memory");
      __syncthreads();
      abuf = abuf + 1 == kRA ? 0 : abuf + 1;
      wbuf = wbuf + 1 == kRW ? 0 : wbuf + 1;
    }
    // The last iterations issued clamped re-reads of the last K tile; up to
    // kInFlight of them per lane may still be in flight, and their LDS destinations
    // overlap the strips of the epilogue.  Drain them, workgroup-wide.
    if (kInFlight > 0) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
  } else {
    // Any K: element-wise tails, one K tile in registers ahead of the MFMAs, two
    // padded LDS buffers.
    u32x4 stage[1][Cfg::kPerThread];
    auto gload = [&](int64_t kt) {
#pragma unroll
      for (int i = 0; i < Cfg::kPerA; ++i) {
        const int c = tid + i * Cfg::kThreads;
        stage[0][i] = load_chunk<T, false>(a.A, a.lda, m0 + c / Cfg::kChunksPerRow, a.M,
                                           kt * kBK + (c % Cfg::kChunksPerRow) * kPer, a.K);
      }
#pragma unroll
      for (int i = 0; i < Cfg::kPerB; ++i) {
        const int c = tid + i * Cfg::kThreads;
        stage[0][Cfg::kPerA + i] =
            load_chunk<T, false>(a.W, a.K, n0 + c / Cfg::kChunksPerRow, a.N,
                                 kt * kBK + (c % Cfg::kChunksPerRow) * kPer, a.K);
      }
    };
    auto lstore = [&](int buf) {
      char* base = lds + buf * Cfg::kBufBytes;
#pragma unroll
      for (int i = 0; i < Cfg::kPerThread; ++i) {
        const bool is_a = i < Cfg::kPerA;
        const int c = tid + (is_a ? i : i - Cfg::kPerA) * Cfg::kThreads;
        const int row = (is_a ? 0 : Cfg::kBM) + c / Cfg::kChunksPerRow;
        store16(base + row * Cfg::kLdsRow + (c % Cfg::kChunksPerRow) * 16, stage[0][i]);
      }
    };
    gload(0);
    lstore(0);
    __syncthreads();
    for (int64_t kt = 0; kt < nk; ++kt) {
      const int buf = (int)(kt & 1);
      if (kt + 1 < nk) gload(kt + 1);
      const char* a_base = lds + buf * Cfg::kBufBytes + (wm * WM * 32 + l32) * Cfg::kLdsRow;
      const char* b_base =
          lds + buf * Cfg::kBufBytes + (Cfg::kBM + wn * WN * 32 + l32) * Cfg::kLdsRow;
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const int koff = s * MM::kK * (int)sizeof(T) + g * kFragBytes;
        Frag fa[WM], fb[WN];
#pragma unroll
        for (int i = 0; i < WM; ++i)
          fa[i] = *reinterpret_cast<const Frag*>(a_base + i * 32 * Cfg::kLdsRow + koff);
#pragma unroll
        for (int j = 0; j < WN; ++j)
          fb[j] = *reinterpret_cast<const Frag*>(b_base + j * 32 * Cfg::kLdsRow + koff);
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j) {
            if (VT_OUT) {
              acc[i][j] = MM::run(fa[i], fb[j], acc[i][j]);
            } else {
              acc[i][j] = MM::run(fb[j], fa[i], acc[i][j]);
            }
          }
      }
      if (kt + 1 < nk) lstore(buf ^ 1);
      __syncthreads();
    }
  }

  // the K loop ended with a barrier and no load into LDS is outstanding: the tile
  // buffers are free
  static_assert((Cfg::kThreads / 64) * strip_bytes<T, WM, WN, VT_OUT>() <= Cfg::kLdsBytes, "strips must fit");
  store_tile<T, WM, WN, VT_OUT, ACT>(a, acc, m0 + wm * WM * 32, n0, wn * WN * 32,
                                     lds + wave * strip_bytes<T, WM, WN, VT_OUT>(),
                                     reinterpret_cast<const float*>(lds + Cfg::kLdsBytes));
}

// Workgroup i runs on XCD i % 8 and every XCD has its own L2.  The tile order
// gives XCD x the row tiles x, x + 8, x + 16, ... for every column panel, one
// column panel after the other: its share of A (an eighth of the rows) stays
// L2-resident while the W panels stream through, so A leaves HBM once instead
// of once per column panel.
// The second launch bound (wavefronts per SIMD the kernel is compiled for) is
// what lets the compiler keep a whole K tile of fragments in registers: left at
// its default it schedules for maximum occupancy, keeps three fragments live
// and waits for LDS in front of every MFMA.
template <typename T, class Cfg, int EPI, bool ALIGNED_K>
__global__ __launch_bounds__(Cfg::kThreads, Cfg::kWavesPerSimd) void linear_kernel(GemmArgs<T> a) {
  extern __shared__ __align__(16) char lds[];
  const int64_t tiles_m = (a.M + Cfg::kBM - 1) / Cfg::kBM;
  const int64_t per_xcd = (tiles_m + 7) / 8;
  const int64_t xcd = blockIdx.x & 7;
  const int64_t local = blockIdx.x >> 3;
  const int64_t tn = local / per_xcd;
  const int64_t tm = (local - tn * per_xcd) * 8 + xcd;
  if (tm >= tiles_m) return;
  const int64_t m0 = tm * Cfg::kBM;
  const int64_t n0 = tn * Cfg::kBN;
  if (EPI == kEpiQkv && n0 >= a.n_split) {
    gemm_tile<T, Cfg, true, ALIGNED_K>(a, m0, n0, lds);    // V tile: transposed into Vt
  } else {
    gemm_tile<T, Cfg, false, ALIGNED_K, EPI == kEpiAct>(a, m0, n0, lds);
  }
}

template <typename T, class Cfg, int EPI, bool ALIGNED_K>
static int launch_kernel(const GemmArgs<T>& a, hipStream_t stream) {
  const int64_t tiles_m = (a.M + Cfg::kBM - 1) / Cfg::kBM;
  const int64_t tiles_n = (a.N + Cfg::kBN - 1) / Cfg::kBN;
  const int64_t wgs = ((tiles_m + 7) / 8) * 8 * tiles_n;
  if (wgs > 0x7fffffffLL) return fail(NT_ERR_UNSUPPORTED, "linear: too many tiles");
  const int lds_bytes = Cfg::kLdsBytes + Cfg::kBN * (int)sizeof(float);
  const int rc = allow_lds<linear_kernel<T, Cfg, EPI, ALIGNED_K>>(lds_bytes, "linear");
  if (rc != NT_OK) return rc;
  hipLaunchKernelGGL((linear_kernel<T, Cfg, EPI, ALIGNED_K>), dim3((unsigned)wgs),
                     dim3(Cfg::kThreads), lds_bytes, stream, a);
  return check_launch("linear_kernel");
}

template <typename T, class Cfg, int EPI>
static int launch_cfg(const GemmArgs<T>& a, hipStream_t stream) {
  // the branch-free loads need whole K tiles
  const bool aligned = a.K > 0 && a.K % (Cfg::kRowBytes / (int64_t)sizeof(T)) == 0;
  if (aligned) return launch_kernel<T, Cfg, EPI, true>(a, stream);
  return launch_kernel<T, Cfg, EPI, false>(a, stream);
}

// ---- the pipelined tile ---------------------------------------------------------
//
// A (64 NI) x (128 NJ) tile of eight wavefronts for problems that fill the chip.  What
// bounds a tile whose wavefronts all do the same thing at the same time (linear_kernel)
// is not the matrix pipe: after every barrier all wavefronts first wait for fragments
// from LDS and only then multiply, and a K tile's loads are waited for in the iteration
// that issued them.  Here
//  * the wavefronts form two groups of four, one wavefront of each group per SIMD,
//    half a phase apart: while one group reads fragments and issues loads (stage M),
//    the other multiplies (stage C), so a SIMD's matrix pipe always has work;
//  * a phase is one 64-row block of A (32 rows per group, consecutive from phase to
//    phase so that a wavefront's rows are one run) against all columns: 4 fragment
//    reads and 4 NJ matrix instructions per wavefront; the W fragments of a K tile stay
//    in registers over its NI phases;
//  * an LDS slot is refilled as soon as its last reader is two phases past it: the load
//    of a block is issued NI * kBufs - 2 phases before the block is read (2500 to 5000
//    cycles), and the wait for it counts exactly the loads issued since.
// Measured (fp16): on operands of zeros a 320 x 256 tile takes 1.12 us per K tile of 64,
// its 80 matrix instructions per SIMD back to back at 2.3 GHz; on N(0, 1) operands
// 1.85 us with all CUs at work, where the chip lowers its clock (1.28 PFLOP/s over
// all CUs; the vendor's 8192^3 product reaches 1.16 to 1.2).  Outside the K loop a launch
// costs about 3.5 us and 0.9 us per NI * NJ, the burst of stores at 4.7 TB/s.
// Against linear_kernel: 8040 x 2304 x 768 46.0 -> 32.9 us, 12900 x 3072 x 1024
// 99.6 -> 80.3, 20000 x 6144 x 2048 501 -> 408, 20500 x 1024 x 512 43.3 -> 30.5,
// 8040 x 768 x 768 16.5 -> 13.5.  (Whether the four to two loads of a W tile go out one,
// two or four per phase makes no difference, nor does writing C through or around the
// L2.)
template <typename T, int NI_, int NJ_, int BUFS_>
struct PhasedCfg {
  static constexpr int kNI = NI_, kNJ = NJ_, kBufs = BUFS_;
  static constexpr int kThreads = 512;
  static constexpr int kBM = 64 * NI_, kBN = 128 * NJ_;
  static constexpr int kABytes = kBM * 128, kBBytes = kBN * 128;   // one K tile: 128 bytes per row
  static constexpr int kLdsBytes = BUFS_ * (kABytes + kBBytes);
  static_assert(kLdsBytes + kBN * 4 <= 160 * 1024, "tile buffers must fit the LDS");
};

// Schedule of the loads.  In phase i of K tile t a wavefront issues one load of A (its
// eight rows of the block NI * kBufs - 2 phases on) and then some of the Q 64-row parts
// ("quarters") of a W tile: those of tile T go out in the first phases after the last
// read of its slot, from phase 2 of tile T - kBufs on.
template <int NI, int Q>
struct PhasedSchedule {
  static constexpr int kPerPhase = (Q + NI - 1) / NI > 2 ? (Q + NI - 1) / NI : 2;
  static constexpr int window(int i) { return (i + NI - 2) % NI; }       // place of phase i among those NI
  static constexpr int at_window(int w) {
    return Q <= kPerPhase * w ? 0 : Q - kPerPhase * w < kPerPhase ? Q - kPerPhase * w : kPerPhase;
  }
  static constexpr int quarters(int i) { return at_window(window(i)); }
  static constexpr int first_quarter(int i) {
    int q = 0;
    for (int w = 0; w < window(i); ++w) q += at_window(w);
    return q;
  }
  static constexpr int last_window() { return (Q + kPerPhase - 1) / kPerPhase - 1; }
  // loads issued before phase i of K tile t (any origin)
  static constexpr int issued_before(int t, int i) {
    int n = t * (NI + Q);
    for (int k = 0; k < i; ++k) n += 1 + quarters(k);
    return n;
  }
  static constexpr int issued_before_phase(int p) {   // p may be negative
    const int t = (p + 64 * NI) / NI - 64;
    return issued_before(t, p - t * NI);
  }
  // Loads that may be outstanding at the end of stage M of phase i of a K tile with
  // `left` tiles to go (this one included; the last kBufs tiles issue fewer loads)
  // such that everything the next phase reads has landed.
  static constexpr int may_be_outstanding(int bufs, int i, int left) {
    const int next = i + 1;                           // phase, relative to the tile
    const int ahead = NI * bufs - 2;
    int needed = issued_before_phase(next - ahead) + 1;          // A is the first load of its phase
    if (next == NI) {                                            // a new K tile: its last W quarter
      const int w = issued_before_phase(NI - NI * bufs + 2 + last_window() + 1);
      if (w > needed) needed = w;
    }
    int issued = issued_before_phase(next);
    const int final = issued_before_phase((left - bufs) * NI + 2);
    if (final < issued) issued = final;
    return issued > needed ? issued - needed : 0;
  }
};

template <typename T, class Cfg, bool VT_OUT, bool ACT>
__device__ __forceinline__ void phased_tile(const GemmArgs<T>& a, int64_t m0, int64_t n0, char* lds) {
  typedef Mma<T> MM;
  typedef typename MM::Frag Frag;
  constexpr int NI = Cfg::kNI, NJ = Cfg::kNJ, kBufs = Cfg::kBufs, kQ = Cfg::kBN / 64;
  typedef PhasedSchedule<NI, kQ> S;
  constexpr int kSteps = 128 / (MM::kK * (int)sizeof(T));
  static_assert(kSteps == 4 && MM::kK * (int)sizeof(T) == 32, "a step is two 16-byte pieces of a row");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave >> 2;      // rows group * 32 NI .. of the tile
  const int wn = wave & 3;          // columns wn * 32 NJ ..
  const int l32 = lane & 31;
  const int g = lane >> 5;

  acc16 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int nk = (int)(a.K * (int64_t)sizeof(T) / 128);
  if (tid < Cfg::kBN) {
    const int64_t col = n0 + tid;
    reinterpret_cast<float*>(lds + Cfg::kLdsBytes)[tid] = (a.bias && col < a.N) ? (float)a.bias[col] : 0.0f;
  }

  // Global addresses: a wavefront loads 8 rows of 128 bytes per instruction, slot p of
  // row r holding piece p ^ ((r >> 1) & 7) so that fragment reads are conflict-free.
  // Per-lane 32-bit offsets (rows past the end clamped to the last one: they only feed
  // accumulators that are not stored) from a scalar base that moves with the K tile.
  const int r8 = wave * 8 + (lane >> 3);                       // row of the 64-row block
  const int piece = ((lane & 7) ^ ((r8 >> 1) & 7)) * 16;
  unsigned a_off[NI], w_off[kQ];
  const int64_t rows_left = a.M - m0, cols_left = a.N - n0;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    int64_t row = (r8 >> 5) * (32 * NI) + i * 32 + (r8 & 31);
    row = row < rows_left ? row : rows_left - 1;
    a_off[i] = (unsigned)(row * a.lda * (int64_t)sizeof(T) + piece);
  }
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    int64_t row = q * 64 + r8;
    row = row < cols_left ? row : cols_left - 1;
    w_off[q] = (unsigned)(row * a.K * (int64_t)sizeof(T) + piece);
  }
  const char* a_base = reinterpret_cast<const char*>(a.A + m0 * a.lda);
  const char* w_base = reinterpret_cast<const char*>(a.W + n0 * a.K);
  const unsigned lds_base = (unsigned)reinterpret_cast<uintptr_t>(lds);
  constexpr unsigned kWRing = kBufs * Cfg::kABytes;
  const unsigned my_kib = (unsigned)wave * 1024;
  auto load_lds = [&](const char* base, unsigned off, unsigned dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst)
                 : "memory");
  };
  // the loads of phase i of a K tile: block (i - 2 mod NI) of A and the quarters of W
  // of K tile `tile`, into its slot
  auto issue = [&](int i, int tile, int slot) {
    const int64_t koff = (int64_t)tile * 128;
    const int blk = (i + NI - 2) % NI;
    load_lds(a_base + koff, a_off[blk], lds_base + slot * Cfg::kABytes + blk * 8192 + my_kib);
    const int q0 = S::first_quarter(i);
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      if (q < q0 || q >= q0 + S::quarters(i)) continue;
      load_lds(w_base + koff, w_off[q], lds_base + kWRing + slot * Cfg::kBBytes + q * 8192 + my_kib);
    }
  };

  // fragment addresses: piece 2 s + g of row l32 of a 32-row block
  const int sw = (l32 >> 1) & 7;
  int koff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) koff[s] = ((2 * s + g) ^ sw) * 16;
  const int a_row = (group * 32 + l32) * 128;
  const int w_row = (wn * (32 * NJ) + l32) * 128;

  Frag fa[4], fb[NJ][4];

  // Prologue: what the kBufs virtual K tiles before the first would have issued.
#pragma unroll
  for (int v = 0; v < kBufs; ++v) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (v == 0 && i < 2) continue;
      const int tile = i < 2 ? v - 1 : v;
      issue(i, tile, tile);
    }
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::may_be_outstanding(kBufs, NI - 1, 64)) : "memory");
  __syncthreads();
  if (group == 1) {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }

  int slot = 0, prev = kBufs - 1;
  // one K tile; LEFT: tiles to go including this one (any number above kBufs: steady state)
  auto k_tile = [&](int t, auto left_c) __attribute__((always_inline)) {
    constexpr int LEFT = decltype(left_c)::value;
    const char* at = lds + slot * Cfg::kABytes + a_row;
    const char* wt = lds + kWRing + slot * Cfg::kBBytes + w_row;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      // stage M
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        fa[s] = *reinterpret_cast<const Frag*>(at + i * 8192 + koff[s]);
        if (i == 0) {
#pragma unroll
          for (int j = 0; j < NJ; ++j) fb[j][s] = *reinterpret_cast<const Frag*>(wt + j * (32 * 128) + koff[s]);
        }
      }
      if (i < 2 ? LEFT >= kBufs : LEFT > kBufs) {
        if (i < 2) issue(i, t + kBufs - 1, prev);
        else issue(i, t + kBufs, slot);
      }
      if (!(LEFT == 1 && i == NI - 1)) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::may_be_outstanding(kBufs, i, LEFT)) : "memory");
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      // stage C
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          if (VT_OUT) {
            acc[i][j] = MM::run(fa[s], fb[j][s], acc[i][j]);
          } else {
            acc[i][j] = MM::run(fb[j][s], fa[s], acc[i][j]);
          }
        }
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    prev = slot;
    slot = slot + 1 == kBufs ? 0 : slot + 1;
  };
  int t = 0;
  for (; t < nk - kBufs; ++t) k_tile(t, std::integral_constant<int, 64>());
  if constexpr (kBufs >= 4) k_tile(t++, std::integral_constant<int, 4>());
  if constexpr (kBufs >= 3) k_tile(t++, std::integral_constant<int, 3>());
  k_tile(t++, std::integral_constant<int, 2>());
  k_tile(t, std::integral_constant<int, 1>());
  if (group == 0) __builtin_amdgcn_s_barrier();
  __syncthreads();

  static_assert(8 * strip_bytes<T, NI, NJ, VT_OUT>() <= Cfg::kLdsBytes, "strips must fit");
  store_tile<T, NI, NJ, VT_OUT, ACT>(a, acc, m0 + group * (32 * NI), n0, wn * (32 * NJ),
                                    lds + wave * strip_bytes<T, NI, NJ, VT_OUT>(),
                                    reinterpret_cast<const float*>(lds + Cfg::kLdsBytes));
}

// Tile order: workgroup i runs on XCD i % 8, and every XCD gets one contiguous run of
// the tile list (equal lengths up to one tile, so no XCD runs a round more than the
// others).  The list walks bands of four row tiles, column panel by column panel: the
// tiles an XCD runs at a time share few rows of A and few panels of W, which its L2
// serves.  False: the workgroup has no tile.
template <int BM, int BN>
__device__ __forceinline__ bool tile_of_workgroup(int64_t M, int64_t N, int64_t* m0, int64_t* n0) {
  const int tiles_m = (int)((M + BM - 1) / BM);
  const int tiles_n = (int)((N + BN - 1) / BN);
  const int total = tiles_m * tiles_n;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int share = total >> 3, more = total & 7;
  if (local >= share + (xcd < more ? 1 : 0)) return false;
  const int id = xcd * share + (xcd < more ? xcd : more) + local;
  constexpr int kBand = 4;
  const int band = id / (kBand * tiles_n);
  const int in_band = id - band * (kBand * tiles_n);
  const int rows = tiles_m - band * kBand < kBand ? tiles_m - band * kBand : kBand;
  const int tn = in_band / rows;
  const int tm = band * kBand + in_band - tn * rows;
  *m0 = (int64_t)tm * BM;
  *n0 = (int64_t)tn * BN;
  return true;
}

template <typename T, class Cfg, int EPI>
__global__ __launch_bounds__(512, 2) void phased_kernel(GemmArgs<T> a) {
  extern __shared__ __align__(16) char lds[];
  int64_t m0, n0;
  if (!tile_of_workgroup<Cfg::kBM, Cfg::kBN>(a.M, a.N, &m0, &n0)) return;
  if constexpr (EPI == kEpiQkv) {
    if (n0 >= a.n_split) {
      phased_tile<T, Cfg, true, false>(a, m0, n0, lds);
      return;
    }
  }
  phased_tile<T, Cfg, false, EPI == kEpiAct>(a, m0, n0, lds);
}

template <typename T, class Cfg, int EPI>
static int launch_phased(const GemmArgs<T>& a, hipStream_t stream) {
  const int64_t tiles = ((a.M + Cfg::kBM - 1) / Cfg::kBM) * ((a.N + Cfg::kBN - 1) / Cfg::kBN);
  const int lds_bytes = Cfg::kLdsBytes + Cfg::kBN * (int)sizeof(float);
  const int rc = allow_lds<phased_kernel<T, Cfg, EPI>>(lds_bytes, "linear");
  if (rc != NT_OK) return rc;
  hipLaunchKernelGGL((phased_kernel<T, Cfg, EPI>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(512), lds_bytes, stream,
                     a);
  return check_launch("phased_kernel");
}

// ---- fp32 products on the bf16 matrix instruction ---------------------------------
//
// The fp32 matrix instruction does a sixteenth of the bf16 one's work per cycle, and a
// product of fp32 operands is bound by it (phased_kernel reached 0.8 of its rate).  An fp32
// number is the sum of three bf16 ones (24 significant bits in three of 8, each the rounded
// rest of the one before: exact), so a product of two is nine bf16 products, each exact in the
// fp32 accumulators.  Eight are kept; that of the two third parts, below 2^-34 of |x| |w|, is
// left out.  (Splitting by rounding and rest is Dekker's.)  The product of the first parts is
// summed in accumulators of its own and the seven others, below 2^-7 of it, in a second set,
// added once at the end: so a partial sum is rounded no oftener than by the fp32 instruction,
// however few of the products are other than zero.  All in one set, a row with one product per
// 16 k was rounded up to eight times per product.  Error against 64 bits, 2-norm, fp32
// instruction / here: N(0, 1) operands of K 256 2.9e-7 / 0.9e-7, 768 5.0e-7 / 1.6e-7, 2048
// 8.1e-7 / 2.7e-7; one product per 16 k, over 1, 4, 48 steps 2.53e-8 / 2.53e-8, 4.0e-8 / 2.6e-8, 1.25e-7 /
// 0.51e-7; rows behind a relu, K 768 3.5e-7 / 1.2e-7.  (Of six products, without the two next
// smallest, a single one has 1.03 times the error of the fp32 instruction, up to a whole
// rounding more; they would take 0.85 of the time.)
//
// The operands are split on the way from global memory to LDS, once per tile: a step of 16
// k of all its rows is fetched into registers kDepth steps ahead, split between the matrix
// instructions of the step before its own and written to the other of two tile buffers.
// Two sets of accumulators leave room for tiles of up to 320 x 128 at two wavefronts per SIMD.
// Bound by the matrix pipe at the clock that random operands leave.  Fp32 instruction / here, us:
// 8040 x 2304 x 768 216 / 185, 8040 x 768 x 768 76 / 63, 20000 x 3072 x 1024 894 / 744, 2000 x 1536 x 512 36 / 26,
// 300 x 768 x 256 19.1 / 8.9; 0.55 of the time over 174 products of K 192 to 2048 (0.86 at most).
template <int GM_, int GN_, int NI_, int NJ_, int DEPTH_>
struct SplitCfg {
  static constexpr int kGM = GM_, kGN = GN_, kNI = NI_, kNJ = NJ_;   // wavefronts, 32 x 32 blocks of each
  static constexpr int kDepth = DEPTH_;                              // steps fetched ahead of the one written to LDS
  static_assert(GM_ * GN_ == 8, "eight wavefronts");
  static constexpr int kBM = GM_ * NI_ * 32, kBN = GN_ * NJ_ * 32;
  static constexpr int kBlocks = (kBM + kBN) / 32;
  static constexpr int kBufBytes = kBlocks * 3 * 1024;               // 16 k of all rows, three parts
  static constexpr int kLdsBytes = 2 * kBufBytes;
  static_assert(8 * strip_bytes<float, NI_, NJ_, false>() <= kLdsBytes, "strips must fit");
  static_assert(kLdsBytes + kBN * 4 <= 160 * 1024, "tile buffers must fit the LDS");
};

// 32-row blocks of A and W lie in LDS as three parts of 1 KiB, a part as the 16-byte pieces
// (k 0..3 and 8..11, or, half 1, the others) of the 32 rows one after the other.  In the
// second half rows trade places by eights, so that sixteen consecutive lanes fall into
// distinct banks both as a fragment's rows (reads) and as two pieces of eight rows (writes).
// The order of the 16 k is the same for A and W, which is all that the product asks for.
__device__ __forceinline__ int split_slot(int half, int row) { return half * 512 + ((row ^ (half << 3)) << 4); }

// One thread's part of a K step: FLOATS (8, 4 or 2) consecutive values of a row of A or W,
// or with 8 two runs of four eight apart, their three parts written to LDS FLOATS * 2 bytes
// each.
template <int FLOATS, int DEPTH>
struct SplitPiece {
  const char* base;      // of A or W at the first row of the tile, the same in a wavefront
  unsigned off;          // of the row and the thread's place in it, in bytes
  unsigned dst;          // in a tile buffer
  uint32_t raw[DEPTH][FLOATS];

  __device__ __forceinline__ void place(const GemmArgs<float>& a, int64_t m0, int64_t n0, int a_blocks, int block,
                                        int row_in_block, int piece) {
    const bool is_a = block < a_blocks;
    int64_t row = (is_a ? block : block - a_blocks) * 32 + row_in_block;
    const int64_t left = is_a ? a.M - m0 : a.N - n0;
    row = row < left ? row : left - 1;               // only feeds accumulators that are not stored
    base = reinterpret_cast<const char*>(is_a ? a.A + m0 * a.lda : a.W + n0 * a.K);
    off = (unsigned)(row * (is_a ? a.lda : a.K) * 4) + piece * (FLOATS == 8 ? 16 : FLOATS * 4);
    // the four k that the piece begins with or lies in, for 8 floats: 0..3 or 4..7
    const int four = FLOATS == 2 ? piece >> 1 : piece;
    dst = block * 3072 + split_slot(four & 1, row_in_block) + (four >> 1) * 8 + (FLOATS == 2 ? (piece & 1) * 4 : 0);
  }
  __device__ __forceinline__ void fetch(int step, int slot) {
    const char* src = base + (int64_t)step * 64;
    __builtin_memcpy(raw[slot], src + off, FLOATS < 8 ? FLOATS * 4 : 16);
    if constexpr (FLOATS == 8) __builtin_memcpy(raw[slot] + 4, src + off + 32, 16);
  }
  __device__ __forceinline__ void put(char* buf, int slot) const {
    uint32_t part[3][FLOATS / 2];
#pragma unroll
    for (int e = 0; e < FLOATS / 2; ++e) {
      split_bf16_pair(__builtin_bit_cast(float, raw[slot][2 * e]) * kSplitScale,
                      __builtin_bit_cast(float, raw[slot][2 * e + 1]) * kSplitScale, part[0][e], part[1][e], part[2][e]);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
      __builtin_memcpy(__builtin_assume_aligned(buf + dst + p * 1024, FLOATS * 2), part[p], FLOATS * 2);
  }
};

template <class Cfg, bool ACT>
__device__ __forceinline__ void split_tile(const GemmArgs<float>& a, int64_t m0, int64_t n0, char* lds) {
  constexpr int NI = Cfg::kNI, NJ = Cfg::kNJ, kDepth = Cfg::kDepth;
  constexpr int kUnits = Cfg::kBlocks / 8, kTail4 = Cfg::kBlocks & 4, kTail2 = Cfg::kBlocks & 2;
  static_assert(Cfg::kBlocks % 2 == 0, "blocks are dealt to the wavefronts whole, by halves and by quarters");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::kGN, wn = wave % Cfg::kGN;
  const int l32 = lane & 31;
  const int g = lane >> 5;

  acc16 acc[NI][NJ], low[NI][NJ];        // products of the first parts; the seven others
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = low[i][j][e] = 0.0f;

  float* lds_bias = reinterpret_cast<float*>(lds + Cfg::kLdsBytes);
  if (tid < Cfg::kBN) {
    const int64_t col = n0 + tid;
    lds_bias[tid] = (a.bias && col < a.N) ? a.bias[col] : 0.0f;
  }

  const int n_steps = (int)(a.K / 16);
  constexpr int kABlocks = Cfg::kBM / 32;
  SplitPiece<8, kDepth> unit[kUnits > 0 ? kUnits : 1];
  SplitPiece<4, kDepth> half;
  SplitPiece<2, kDepth> quarter;
#pragma unroll
  for (int u = 0; u < kUnits; ++u)
    unit[u].place(a, m0, n0, kABlocks, wave + 8 * u, lane >> 1, lane & 1);
  if (kTail4)
    half.place(a, m0, n0, kABlocks, 8 * kUnits + (wave >> 1), (wave & 1) * 16 + (lane >> 2), lane & 3);
  if (kTail2)
    quarter.place(a, m0, n0, kABlocks, 8 * kUnits + kTail4 + (wave >> 2), (wave & 3) * 8 + (lane >> 3), lane & 7);

  constexpr int kPuts = kUnits + (kTail4 ? 1 : 0) + (kTail2 ? 1 : 0);
  auto fetch = [&](int u, int step, int slot) __attribute__((always_inline)) {
    step = step < n_steps ? step : n_steps - 1;          // past the end: not used
    if (u < kUnits) unit[u < kUnits ? u : 0].fetch(step, slot);
    else if (u == kUnits && kTail4) half.fetch(step, slot);
    else quarter.fetch(step, slot);
  };
  auto put = [&](int u, char* buf, int slot) __attribute__((always_inline)) {
    if (u < kUnits) unit[u < kUnits ? u : 0].put(buf, slot);
    else if (u == kUnits && kTail4) half.put(buf, slot);
    else quarter.put(buf, slot);
  };
  auto publish = [] __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // the pieces of step s wait in slot s % kDepth
#pragma unroll
  for (int d = 0; d < kDepth; ++d)
#pragma unroll
    for (int u = 0; u < kPuts; ++u) fetch(u, d, d);
#pragma unroll
  for (int u = 0; u < kPuts; ++u) {
    put(u, lds, 0);
    fetch(u, kDepth, 0);
  }
  publish();

  const char* a_lds = lds + wm * NI * 3072 + split_slot(g, l32);
  const char* w_lds = lds + (kABlocks + wn * NJ) * 3072 + split_slot(g, l32);
  bf16x8 fa[2][3], fb[NJ][3];
  auto read_a = [&](bf16x8 (&f)[3], int buf, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 3; ++p) f[p] = *reinterpret_cast<const bf16x8*>(a_lds + buf + i * 3072 + p * 1024);
  };
  read_a(fa[0], 0, 0);
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int p = 0; p < 3; ++p) fb[j][p] = *reinterpret_cast<const bf16x8*>(w_lds + j * 3072 + p * 1024);

  int cur = 0;
  auto one_step = [&](int step, int slot) __attribute__((always_inline)) {   // slot: that of the next step
    const int other = Cfg::kBufBytes - cur;
    bf16x8 fb_next[NJ][3];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      // the splits of the next step, dealt out over the blocks in front of the last
      constexpr int kSlots = NI > 1 ? NI - 1 : 1;
#pragma unroll
      for (int u = 0; u < kPuts; ++u)
        if (u * kSlots / kPuts == i) {
          put(u, lds + other, slot);
          fetch(u, step + 1 + kDepth, slot);
        }
      if (i + 1 < NI) {
        read_a(fa[(i + 1) & 1], cur, i + 1);
      } else {
        // Every fragment of this step is read and every piece of the next written: the one
        // barrier of a step, with a block's products left to cover the first reads behind it.
        publish();
        read_a(fa[(i + 1) & 1], other, 0);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int p = 0; p < 3; ++p)
            fb_next[j][p] = *reinterpret_cast<const bf16x8*>(w_lds + other + j * 3072 + p * 1024);
      }
      // smallest products first; the first parts' among them, for a break in the chain of sums
      constexpr int kPa[7] = {1, 2, 0, 1, 2, 0, 1}, kPw[7] = {2, 1, 2, 1, 0, 1, 0};
#pragma unroll
      for (int p = 0; p < 7; ++p) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          low[i][j] = Mma<__bf16>::run(fb[j][kPw[p]], fa[i & 1][kPa[p]], low[i][j]);
          if (p == 4) acc[i][j] = Mma<__bf16>::run(fb[j][0], fa[i & 1][0], acc[i][j]);
        }
      }
      if (i + 1 < NI) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);   // the next block's reads first
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p) fb[j][p] = fb_next[j][p];
    if (NI & 1) {
#pragma unroll
      for (int p = 0; p < 3; ++p) fa[0][p] = fa[1][p];
    }
    cur = other;
  };
  int step = 0;
  for (; step + kDepth <= n_steps; step += kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) one_step(step + d, (d + 1) % kDepth);
  }
#pragma unroll
  for (int d = 0; d + 1 < kDepth; ++d)
    if (step + d < n_steps) one_step(step + d, (d + 1) % kDepth);

  // A result that is no finite number: an infinity, a NaN or a magnitude from 2^111 on went in,
  // or a sum, 2^32 times the result's, overflowed.
  unsigned redo = 0;                            // a bit per block of 32 rows, the same in a wavefront
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    float probe = 0.0f;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[i][j][e] += low[i][j][e];
        probe = fmaf(acc[i][j][e], 0.0f, probe);
        acc[i][j][e] *= kSplitUnscale;
      }
    if (__ballot(probe != probe) != 0) redo |= 1u << i;
  }
  __syncthreads();
  char* strip = lds + wave * strip_bytes<float, NI, NJ, false>();
  store_tile<float, NI, NJ, false, ACT>(a, acc, m0 + wm * (32 * NI), n0, wn * (32 * NJ), strip, lds_bias);
  if (redo == 0) return;
  // Those blocks once more by the fp32 instruction, operands straight from global memory, and over
  // what has been stored.  Seldom worth more: one row of 8040 x 2304 x 768 not finite costs 35 us more (190 with
  // all rows of the wavefront done again), all of them take 590 us (the fp32 instruction alone 215).
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll 1
  for (int i = 0; i < NI; ++i) {
    if (!(redo >> i & 1)) continue;
    acc16 row[1][NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) row[0][j][e] = 0.0f;
    const int64_t m = m0 + (wm * NI + i) * 32 + l32;
    const float* ap = a.A + (m < a.M ? m : a.M - 1) * a.lda + g * 4;
    const float* wp[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int64_t n = n0 + (wn * NJ + j) * 32 + l32;
      wp[j] = a.W + (n < a.N ? n : a.N - 1) * a.K + g * 4;
    }
    f32x4 xa[2], xw[NJ][2];
    auto load = [&](int64_t k) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        xa[h] = __builtin_bit_cast(f32x4, load16_unaligned(reinterpret_cast<const char*>(ap + k + 8 * h)));
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          xw[j][h] = __builtin_bit_cast(f32x4, load16_unaligned(reinterpret_cast<const char*>(wp[j] + k + 8 * h)));
      }
    };
    load(0);
#pragma unroll 1
    for (int64_t k = 0; k < a.K; k += 16) {
      f32x4 ya[2], yw[NJ][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        ya[h] = xa[h];
#pragma unroll
        for (int j = 0; j < NJ; ++j) yw[j][h] = xw[j][h];
      }
      load(k + 16 < a.K ? k + 16 : 0);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < NJ; ++j) row[0][j] = Mma<float>::run(yw[j][h], ya[h], row[0][j]);
    }
    store_tile<float, 1, NJ, false, ACT>(a, row, m0 + (wm * NI + i) * 32, n0, wn * (32 * NJ), strip, lds_bias);
  }
}

template <class Cfg, int EPI>
__global__ __launch_bounds__(512, 2) void split_kernel(GemmArgs<float> a) {
  extern __shared__ __align__(16) char lds[];
  int64_t m0, n0;
  if (!tile_of_workgroup<Cfg::kBM, Cfg::kBN>(a.M, a.N, &m0, &n0)) return;
  split_tile<Cfg, EPI == kEpiAct>(a, m0, n0, lds);
}

template <class Cfg, int EPI>
static int launch_split(const GemmArgs<float>& a, hipStream_t stream) {
  const int64_t tiles = ((a.M + Cfg::kBM - 1) / Cfg::kBM) * ((a.N + Cfg::kBN - 1) / Cfg::kBN);
  const int lds_bytes = Cfg::kLdsBytes + Cfg::kBN * (int)sizeof(float);
  const int rc = allow_lds<split_kernel<Cfg, EPI>>(lds_bytes, "linear");
  if (rc != NT_OK) return rc;
  hipLaunchKernelGGL((split_kernel<Cfg, EPI>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(512), lds_bytes, stream, a);
  return check_launch("split_kernel");
}

// WAVES_M, WAVES_N, WM, WN, K-tile bytes per row
typedef GemmCfg<4, 2, 2, 2, 128> Cfg128;   // 256 x 128: whatever the pipelined tile does not take,
typedef GemmCfg<4, 2, 2, 3, 128> Cfg192;   // and in 16 bit 256 x 192
typedef GemmCfg<4, 2, 2, 4, 128> Cfg256;   // and 256 x 256
typedef GemmCfg<2, 2, 2, 1, 128> CfgSmall; // 128 x 64, four wavefronts: problems of fewer 256-row tiles than CUs
typedef GemmCfg<2, 2, 2, 2, 128> CfgMid;   // 128 x 128, four wavefronts

static int compute_units(int* n) {
  static int num_cus = 0;
  if (num_cus == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess ||
        prop.multiProcessorCount < 1) {
      return fail(NT_ERR_HIP, "linear: cannot query the device");
    }
    num_cus = prop.multiProcessorCount;
  }
  *n = num_cus;
  return NT_OK;
}

// What a problem of 16-bit operands takes on a tile shape, in microseconds: `alone` and
// `full` per K tile (128 bytes of a row) of a workgroup when few CUs and when all CUs are at
// work (the difference is the clock the chip holds on random operands), `first` for the fill
// and the burst of stores of one round over the CUs and `round` for those of a further one,
// `pieces` for a round of stores to rows that are no whole 16-byte pieces.  Fitted on the
// shape that is fastest of all in 903 problems (72 to 8192 columns, K 128 to 4096, 2500 to
// 200000 rows) and not on single times: what it picks takes 1.010 times the fastest shape's
// time on average, 1.06 at the 95th percentile.  Without the shapes of linear_kernel, with 4 us
// for any further round and whole pieces throughout it was 1.031 and 1.16, and one problem in five
// (two to six K tiles, or rows that end inside a piece) lost 3 to 40 % against linear_kernel.
struct TileCost {
  double alone, full, first, round, pieces;
};
struct PhasedShape {
  int ni, nj, bufs;
  TileCost cost;
};
static const PhasedShape kPhasedShapes[] = {
    {2, 2, 3, {0.602, 0.956, 3.46, 3.89, 2.47}},
    {3, 2, 2, {1.1, 1.23, 4.06, 7.84, 3.37}},
    {4, 2, 2, {1.1, 1.63, 5.17, 8.88, 11.8}},
    {5, 2, 2, {1.6, 1.95, 9.4, 9.5, 7.15}},
    {2, 1, 4, {0.25, 0.522, 1, 2.87, 8.7}},
    {3, 1, 3, {0.35, 0.756, 2.01, 5.04, 4.29}},
    {4, 1, 3, {0.735, 0.987, 3.51, 4.38, 6.58}},
    {5, 1, 2, {0.9, 1.17, 3.94, 5.97, 8.67}}};
constexpr int kPhasedCount = (int)(sizeof(kPhasedShapes) / sizeof(kPhasedShapes[0]));
// linear_kernel's tiles of 256 rows by 128, 192 and 256 columns
static const TileCost kLinearCosts[] = {
    {0.406, 1.1, 0.741, 6.47, 3.54},
    {0.669, 1.9, 2, 6.09, 7.69},
    {1.83, 2, 2, 9.84, 13.3}};

static double tile_time(const TileCost& c, double launch, int64_t tiles, int64_t nk, bool pieces, int num_cus) {
  const int64_t whole = tiles / num_cus, rest = tiles % num_cus;
  double last = c.full * (double)rest / num_cus;
  if (rest > 0 && last < c.alone) last = c.alone;
  const double us = launch + nk * (whole * c.full + last) + c.first + c.round * (double)(whole + (rest > 0) - 1);
  return us + (pieces ? c.pieces * (whole > 0 ? (double)tiles / num_cus : 1.0) : 0.0);
}

// Pipelined shape with the least estimated time for M x N with nk K tiles of fp32: 64
// cycles of matrix pipe per instruction, no lowered clock.
static int pick_phased_f32(int64_t M, int64_t N, int64_t nk, int num_cus) {
  int best = -1;
  double best_us = 0.0;
  for (int c = 0; c < kPhasedCount; ++c) {
    const PhasedShape& s = kPhasedShapes[c];
    if (nk < s.bufs) continue;                       // the prologue fills the whole ring
    const int64_t tiles = ((M + 64 * s.ni - 1) / (64 * s.ni)) * ((N + 128 * s.nj - 1) / (128 * s.nj));
    const double area = s.ni * s.nj;
    const TileCost cost = {0.853 * area, 0.853 * area, 1.8 * area, 4.0, 0.0};
    const double us = tile_time(cost, 3.5, tiles, nk, false, num_cus);
    if (best < 0 || us < best_us) {
      best = c;
      best_us = us;
    }
  }
  return best;
}

// Tiles of split_kernel and what one takes, in microseconds per 16 k; fitted like the above on
// 174 products (16 to 60000 rows, K 192 to 2048): what it picks takes 1.002 times the fastest
// shape's time on average, 1.02 at most.
struct SplitShape {
  int bm, bn;
  TileCost cost;
};
static const SplitShape kSplitShapes[] = {
    {320, 128, {1.471, 1.85, 13.606, 1.721, 0.0}},
    {256, 128, {1.317, 1.519, 7.484, 1.847, 0.0}},
    {192, 128, {1.105, 1.207, 3.214, 6.064, 0.0}},
    {128, 128, {0.664, 0.835, 3.496, 6.615, 0.0}},
    {64, 128, {0.402, 0.481, 2.089, 1.249, 0.0}},
    {128, 64, {0.31, 0.476, 3.686, 0.603, 0.0}}};
constexpr int kSplitCount = (int)(sizeof(kSplitShapes) / sizeof(kSplitShapes[0]));

static int pick_split(int64_t M, int64_t N, int64_t K, int num_cus) {
  int best = 0;
  double best_us = 0.0;
  for (int c = 0; c < kSplitCount; ++c) {
    const SplitShape& s = kSplitShapes[c];
    const int64_t tiles = ((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
    const double us = tile_time(s.cost, 0.0, tiles, K / 16, false, num_cus);
    if (c == 0 || us < best_us) {
      best = c;
      best_us = us;
    }
  }
  return best;
}

// What a problem runs on: a shape of linear_kernel or, kTilePhased + c, kPhasedShapes[c] or,
// kTileSplit + c, kSplitShapes[c].
enum { kTile256x128, kTile256x192, kTile256x256, kTile128x64, kTile128x128, kTilePhased,
       kTileSplit = kTilePhased + kPhasedCount };

// The tile of M x N x K; row-major A has lda elements per row, columns from n_split on go
// transposed into Vt (n_split = 0: to either side of no boundary).  qkv: there are such
// columns.  pieces: the rows of the result end inside a 16-byte piece.  -1: a tile would
// straddle the boundary.
static int choose_tile(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t n_split, bool qkv, bool pieces,
                       int elem_bytes, int num_cus) {
  const bool half = elem_bytes == 2;
  // Fewer 256 x 128 tiles than half the CUs: the launch is one tile's life on a fraction
  // of the chip, and a quarter-size tile on four times as many CUs is shorter
  // (3200 x 512 x 512: 6.2 us, against 6.8 with the smallest pipelined tile).
  if (half && ((M + 255) / 256) * ((N + 127) / 128) * 2 <= num_cus) {
    const bool small = ((M + 127) / 128) * ((N + 63) / 64) <= num_cus;
    if (small && n_split % CfgSmall::kBN == 0) return kTile128x64;
    if (!small && n_split % CfgMid::kBN == 0) return kTile128x128;
  }
  // At most 64 columns: such a product reads A once and is bound by that, half of a
  // 128-column tile would be padding, and three workgroups of this tile share a CU where the
  // larger ones have it to themselves while they fill and drain (589481 x 64 x 256
  // 95.8 -> 77.5 us = 4.9 TB/s, 300000 x 32 x 64 33.2 -> 22.6, 100000 x 32 x 256 18.1 -> 13.4;
  // with 128 columns it loses: 300000 x 128 x 128 32.4 -> 49.2).
  // Deep whole K tiles keep the CU busy by themselves (70000 x 64 x 3072: 97 us, 84 with 320 x 128;
  // 40000 x 64 x 8192: 173, 142 with 192 x 128; 33000 x 64 x 2048: 27.7, 28.6 with 256 x 128).
  if (half && N <= CfgSmall::kBN && n_split % CfgSmall::kBN == 0 && (K <= 2048 || K % 64 != 0)) return kTile128x64;
  // The pipelined tile needs whole K tiles, at least two of them, and 32-bit offsets
  // inside a tile.  (fp32: row-major results only, the transposed strips
  // would not fit its LDS.)
  constexpr int64_t kMaxSpan = (int64_t(1) << 32) - 1;
  const int64_t row_bytes = K * elem_bytes;
  // fp32 goes to the bf16 instruction in whole steps of 16 k.  The line at 192 k is not where the
  // two meet: split_kernel takes 0.23 to 0.88 of the time of what runs below it, too (eleven
  // shapes each of K 16 to 176; 8040 x 512 x 128 14.1 us against 12.3, x 176 32.9 against 14.7).  Below it the
  // shapes of phased_kernel for fp32 are held by test_gpu_linear_pipelined.py (K 64, 128 and 160).
  if (!half && !qkv && K % 16 == 0 && K >= 192 && lda * elem_bytes * 320 < kMaxSpan && row_bytes * 256 < kMaxSpan &&
      (M / 64 + 1) * (N / 64 + 1) < (int64_t(1) << 30)) {
    return kTileSplit + pick_split(M, N, K, num_cus);
  }
  if ((half || !qkv) && row_bytes % 128 == 0 && row_bytes >= 2 * 128 && lda * elem_bytes * 320 < kMaxSpan &&
      row_bytes * 256 < kMaxSpan && (M / 64 + 1) * (N / 64 + 1) < (int64_t(1) << 30)) {
    const int64_t nk = row_bytes / 128;
    if (!half) {
      // Two K tiles and one round of 256 x 128 tiles: linear_kernel fills sooner (9000 x 128 x 64
      // 13.5 us against 15.5, 53000 x 64 x 64 14.3 against 16.6; in two rounds it loses, 20000 x
      // 512 x 64 28.7 against 19.6).
      if (nk == 2 && ((M + 255) / 256) * ((N + 127) / 128) <= num_cus) return kTile256x128;
      const int c = pick_phased_f32(M, N, nk, num_cus);
      if (c >= 0) return kTilePhased + c;
    } else {
      int best = -1;
      double best_us = 0.0;
      for (int c = 0; c < 3 + kPhasedCount; ++c) {
        const bool phased = c >= 3;
        const PhasedShape& s = kPhasedShapes[phased ? c - 3 : 0];
        const int64_t bm = phased ? 64 * s.ni : 256, bn = phased ? 128 * s.nj : 128 + 64 * c;
        // a tile must not straddle the K | V boundary, and the prologue fills the whole ring
        if (n_split % bn != 0 || (phased && nk < s.bufs)) continue;
        const int64_t tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
        const double us = phased ? tile_time(s.cost, 2.59, tiles, nk, pieces, num_cus)
                                 : tile_time(kLinearCosts[c], 4.7, tiles, nk, pieces, num_cus);
        if (best < 0 || us < best_us) {
          best = phased ? kTilePhased + c - 3 : kTile256x128 + c;
          best_us = us;
        }
      }
      if (best >= 0) return best;
    }
  }
  if (half) {
    // What is left: K of no whole number of K tiles or of one, rows of A or W too long for
    // 32-bit offsets.  Estimated time: tile area over the measured rate of
    // its shape (wider tiles read less LDS and L2 per product), times the mean of the whole
    // rounds and of tiles / CUs.  Never the 256 x 128 tile alone: an attention layer of 15 heads
    // of 32 on 35548 tokens (its projections have K = 480) took 285 us with it, 262 like this.
    const int bn[3] = {Cfg128::kBN, Cfg192::kBN, Cfg256::kBN};
    const double rate[3] = {1.0, 1.08, 1.17};
    int best = -1;
    double best_cost = 0.0;
    for (int c = 0; c < 3; ++c) {
      if (n_split % bn[c] != 0) continue;          // a tile must not straddle the K | V boundary
      const int64_t tiles = ((M + 255) / 256) * ((N + bn[c] - 1) / bn[c]);
      const double rounds = 0.5 * ((double)((tiles + num_cus - 1) / num_cus) + (double)tiles / num_cus);
      const double cost = rounds * bn[c] / rate[c];
      if (best < 0 || cost < best_cost) {
        best = c;
        best_cost = cost;
      }
    }
    if (best >= 0) return kTile256x128 + best;
    if (n_split % CfgSmall::kBN == 0) return kTile128x64;
  }
  return n_split % Cfg128::kBN == 0 ? kTile256x128 : -1;
}

template <typename T, int EPI>
static int launch_epi(const GemmArgs<T>& a, hipStream_t stream) {
  const int64_t n_split = EPI == kEpiQkv ? a.n_split : 0;
  int num_cus = 0;
  const int rc = compute_units(&num_cus);
  if (rc != NT_OK) return rc;
  const bool pieces = ((EPI == kEpiQkv && n_split == 0 ? a.ldvt : a.ldc) * (int64_t)sizeof(T)) % 16 != 0;
  const int tile = choose_tile(a.M, a.N, a.K, a.lda, n_split, EPI == kEpiQkv, pieces, (int)sizeof(T), num_cus);
  if constexpr (sizeof(T) == 2 || EPI != kEpiQkv) {
    switch (tile) {
      case kTilePhased + 0: return launch_phased<T, PhasedCfg<T, 2, 2, 3>, EPI>(a, stream);
      case kTilePhased + 1: return launch_phased<T, PhasedCfg<T, 3, 2, 2>, EPI>(a, stream);
      case kTilePhased + 2: return launch_phased<T, PhasedCfg<T, 4, 2, 2>, EPI>(a, stream);
      case kTilePhased + 3: return launch_phased<T, PhasedCfg<T, 5, 2, 2>, EPI>(a, stream);
      case kTilePhased + 4: return launch_phased<T, PhasedCfg<T, 2, 1, 4>, EPI>(a, stream);
      case kTilePhased + 5: return launch_phased<T, PhasedCfg<T, 3, 1, 3>, EPI>(a, stream);
      case kTilePhased + 6: return launch_phased<T, PhasedCfg<T, 4, 1, 3>, EPI>(a, stream);
      case kTilePhased + 7: return launch_phased<T, PhasedCfg<T, 5, 1, 2>, EPI>(a, stream);
    }
  }
  if constexpr (sizeof(T) == 4 && EPI != kEpiQkv) {
    switch (tile) {
      case kTileSplit + 0: return launch_split<SplitCfg<2, 4, 5, 1, 1>, EPI>(a, stream);
      case kTileSplit + 1: return launch_split<SplitCfg<2, 4, 4, 1, 1>, EPI>(a, stream);
      case kTileSplit + 2: return launch_split<SplitCfg<2, 4, 3, 1, 1>, EPI>(a, stream);
      case kTileSplit + 3: return launch_split<SplitCfg<2, 4, 2, 1, 4>, EPI>(a, stream);
      case kTileSplit + 4: return launch_split<SplitCfg<2, 4, 1, 1, 2>, EPI>(a, stream);
      case kTileSplit + 5: return launch_split<SplitCfg<4, 2, 1, 1, 2>, EPI>(a, stream);
    }
  }
  if constexpr (sizeof(T) == 2) {
    switch (tile) {
      case kTile256x192: return launch_cfg<T, Cfg192, EPI>(a, stream);
      case kTile256x256: return launch_cfg<T, Cfg256, EPI>(a, stream);
      case kTile128x64: return launch_cfg<T, CfgSmall, EPI>(a, stream);
      case kTile128x128: return launch_cfg<T, CfgMid, EPI>(a, stream);
    }
  }
  if (tile != kTile256x128) {
    return fail(NT_ERR_UNSUPPORTED, "linear: QKV split %lld is not a multiple of a column tile", (long long)n_split);
  }
  return launch_cfg<T, Cfg128, EPI>(a, stream);
}

template <typename T>
static int launch_linear(GemmArgs<T> a, bool qkv, hipStream_t stream) {
  if (qkv) return launch_epi<T, kEpiQkv>(a, stream);
  if (a.act != 0) return launch_epi<T, kEpiAct>(a, stream);
  return launch_epi<T, kEpiPlain>(a, stream);
}

static int check_linear(const void* A, int64_t lda, const void* W, const void* C, int64_t ldc,
                        int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K < 0 || lda < K || ldc < 0) {
    return fail(NT_ERR_INVALID_ARGUMENT, "linear: bad shape M=%lld N=%lld K=%lld lda=%lld ldc=%lld",
                (long long)M, (long long)N, (long long)K, (long long)lda, (long long)ldc);
  }
  if (M > 0 && N > 0 && (!A || !W || !C)) return fail(NT_ERR_INVALID_ARGUMENT, "linear: NULL pointer");
  return NT_OK;
}

template <typename T>
static GemmArgs<T> make_args(const void* A, int64_t lda, const void* W, const void* bias, void* C,
                             int64_t ldc, int64_t M, int64_t N, int64_t K) {
  GemmArgs<T> a;
  a.A = static_cast<const T*>(A);
  a.lda = lda;
  a.W = static_cast<const T*>(W);
  a.bias = static_cast<const T*>(bias);
  a.C = static_cast<T*>(C);
  a.ldc = ldc;
  a.M = M;
  a.N = N;
  a.K = K;
  a.Vt = nullptr;
  a.ldvt = 0;
  a.n_split = N;
  a.act = 0;
  return a;
}

}  // namespace nt

using namespace nt;

extern "C" int nt_linear_act(const void* A, int64_t lda, const void* W, const void* bias, void* C,
                             int64_t ldc, int64_t M, int64_t N, int64_t K, int act, int dtype,
                             void* stream) {
  int rc = check_linear(A, lda, W, C, ldc, M, N, K);
  if (rc != NT_OK) return rc;
  if (ldc < N) return fail(NT_ERR_INVALID_ARGUMENT, "linear: ldc %lld < N %lld", (long long)ldc, (long long)N);
  if (act < 0 || act > 2) return fail(NT_ERR_INVALID_ARGUMENT, "linear: activation %d is not 0, 1 or 2", act);
  if (M == 0 || N == 0) return NT_OK;
  hipStream_t s = (hipStream_t)stream;
#define NT_LIN_CASE(TYPE)                                                   \
  {                                                                         \
    GemmArgs<TYPE> a = make_args<TYPE>(A, lda, W, bias, C, ldc, M, N, K);   \
    a.act = act;                                                            \
    return launch_linear<TYPE>(a, false, s);                                \
  }
  switch (dtype) {
    case NT_F32: NT_LIN_CASE(float)
    case NT_F16: NT_LIN_CASE(_Float16)
    case NT_BF16: NT_LIN_CASE(__bf16)
    default: return fail(NT_ERR_INVALID_ARGUMENT, "linear: unknown dtype %d", dtype);
  }
#undef NT_LIN_CASE
}

extern "C" int nt_linear_tile(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldc, int64_t n_split, int dtype,
                              int num_cus, int* tile) {
  if (M < 1 || N < 1 || K < 0 || lda < K || ldc < 1 || n_split > N || num_cus < 0 || !tile ||
      (dtype != NT_F32 && dtype != NT_F16 && dtype != NT_BF16)) {
    return fail(NT_ERR_INVALID_ARGUMENT, "linear_tile: bad arguments");
  }
  if (num_cus == 0) {
    const int rc = compute_units(&num_cus);
    if (rc != NT_OK) return rc;
  }
  const bool qkv = n_split >= 0;
  const int elem_bytes = dtype == NT_F32 ? 4 : 2;
  const int c = choose_tile(M, N, K, lda, qkv ? n_split : 0, qkv, ldc * elem_bytes % 16 != 0, elem_bytes, num_cus);
  if (c < 0) return fail(NT_ERR_UNSUPPORTED, "linear: QKV split %lld is not a multiple of a column tile", (long long)n_split);
  if (c >= kTileSplit) {
    tile[0] = kSplitShapes[c - kTileSplit].bm;
    tile[1] = kSplitShapes[c - kTileSplit].bn;
    tile[2] = -1;
    return NT_OK;
  }
  static const int kShapes[kTilePhased][2] = {{256, 128}, {256, 192}, {256, 256}, {128, 64}, {128, 128}};
  tile[0] = c >= kTilePhased ? 64 * kPhasedShapes[c - kTilePhased].ni : kShapes[c][0];
  tile[1] = c >= kTilePhased ? 128 * kPhasedShapes[c - kTilePhased].nj : kShapes[c][1];
  tile[2] = c >= kTilePhased ? kPhasedShapes[c - kTilePhased].bufs : 0;
  return NT_OK;
}

extern "C" int nt_linear(const void* A, int64_t lda, const void* W, const void* bias, void* C,
                         int64_t ldc, int64_t M, int64_t N, int64_t K, int dtype, void* stream) {
  return nt_linear_act(A, lda, W, bias, C, ldc, M, N, K, 0, dtype, stream);
}

extern "C" int nt_linear_qkv(const void* A, int64_t lda, const void* W, const void* bias, void* QK,
                             int64_t ldqk, void* Vt, int64_t ldvt, int64_t M, int64_t E, int64_t K,
                             int dtype, void* stream) {
  int rc = check_linear(A, lda, W, QK, ldqk, M, 3 * E, K);
  if (rc != NT_OK) return rc;
  if (ldqk < 2 * E || ldvt < M) {
    return fail(NT_ERR_INVALID_ARGUMENT, "linear_qkv: ldqk %lld < 2E or ldvt %lld < M",
                (long long)ldqk, (long long)ldvt);
  }
  if (M == 0 || E == 0) return NT_OK;
  if (!Vt) return fail(NT_ERR_INVALID_ARGUMENT, "linear_qkv: Vt is NULL");
  hipStream_t s = (hipStream_t)stream;
#define NT_QKV_CASE(TYPE)                                                       \
  {                                                                             \
    GemmArgs<TYPE> a = make_args<TYPE>(A, lda, W, bias, QK, ldqk, M, 3 * E, K); \
    a.Vt = static_cast<TYPE*>(Vt);                                              \
    a.ldvt = ldvt;                                                              \
    a.n_split = 2 * E;                                                          \
    return launch_linear<TYPE>(a, true, s);                                     \
  }
  switch (dtype) {
    case NT_F32: NT_QKV_CASE(float)
    case NT_F16: NT_QKV_CASE(_Float16)
    case NT_BF16: NT_QKV_CASE(__bf16)
    default: return fail(NT_ERR_INVALID_ARGUMENT, "linear_qkv: unknown dtype %d", dtype);
  }
#undef NT_QKV_CASE
}

extern "C" int nt_linear_kv(const void* A, int64_t lda, const void* W, const void* bias, void* Kout,
                            int64_t ldk, void* Vt, int64_t ldvt, int64_t M, int64_t E, int64_t K, int dtype,
                            void* stream) {
  int rc = check_linear(A, lda, W, Kout, ldk, M, 2 * E, K);
  if (rc != NT_OK) return rc;
  if (ldk < E || ldvt < M) {
    return fail(NT_ERR_INVALID_ARGUMENT, "linear_kv: ldk %lld < E or ldvt %lld < M", (long long)ldk, (long long)ldvt);
  }
  if (M == 0 || E == 0) return NT_OK;
  if (!Vt) return fail(NT_ERR_INVALID_ARGUMENT, "linear_kv: Vt is NULL");
  hipStream_t s = (hipStream_t)stream;
  // the fused in-projection's kernel with the row-major | transposed boundary at column E
#define NT_KV_CASE(TYPE)                                                        \
  {                                                                             \
    GemmArgs<TYPE> a = make_args<TYPE>(A, lda, W, bias, Kout, ldk, M, 2 * E, K); \
    a.Vt = static_cast<TYPE*>(Vt);                                              \
    a.ldvt = ldvt;                                                              \
    a.n_split = E;                                                              \
    return launch_linear<TYPE>(a, true, s);                                     \
  }
  switch (dtype) {
    case NT_F32: NT_KV_CASE(float)
    case NT_F16: NT_KV_CASE(_Float16)
    case NT_BF16: NT_KV_CASE(__bf16)
    default: return fail(NT_ERR_INVALID_ARGUMENT, "linear_kv: unknown dtype %d", dtype);
  }
#undef NT_KV_CASE
}

extern "C" int nt_linear_transposed(const void* A, int64_t lda, const void* W, const void* bias,
                                    void* Ct, int64_t ldct, int64_t M, int64_t N, int64_t K, int dtype,
                                    void* stream) {
  int rc = check_linear(A, lda, W, Ct, ldct, M, N, K);
  if (rc != NT_OK) return rc;
  if (ldct < M) {
    return fail(NT_ERR_INVALID_ARGUMENT, "linear_transposed: ldct %lld < M %lld", (long long)ldct,
                (long long)M);
  }
  if (M == 0 || N == 0) return NT_OK;
  hipStream_t s = (hipStream_t)stream;
  // every tile is a transposed-output tile of the fused QKV kernel: split at column 0
#define NT_LT_CASE(TYPE)                                                     \
  {                                                                          \
    GemmArgs<TYPE> a = make_args<TYPE>(A, lda, W, bias, Ct, ldct, M, N, K);  \
    a.C = nullptr;                                                           \
    a.Vt = static_cast<TYPE*>(Ct);                                           \
    a.ldvt = ldct;                                                           \
    a.n_split = 0;                                                           \
    return launch_linear<TYPE>(a, true, s);                                  \
  }
  switch (dtype) {
    case NT_F32: NT_LT_CASE(float)
    case NT_F16: NT_LT_CASE(_Float16)
    case NT_BF16: NT_LT_CASE(__bf16)
    default: return fail(NT_ERR_INVALID_ARGUMENT, "linear_transposed: unknown dtype %d", dtype);
  }
#undef NT_LT_CASE
}
