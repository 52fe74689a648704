// Bias-free 1x1 convolution on the row-major (NCHW) packed buffer, without the two
// layout changes around the GEMM (gfx950, f16 / bf16).
//
// The reference turns a 1x1 convolution of a nested tensor of images into one
// matrix product over all pixels: transpose_nchw_nhwc, matmul with the [C_out,
// C_in] weight, transpose_nhwc_nchw (nestedtensor/csrc/conv2d.cpp:33-75).  The
// product itself is memory-bound at these depths (C_in = 64 -> C_out = 256: 128
// bytes in, 512 bytes out per pixel), so the two transposes triple its traffic.
// Here the product reads and writes the images as they lie: per image b,
//   Y_b[C_out, P_b] = W[C_out, C_in] X_b[C_in, P_b],
// with the pixels P_b = H_b W_b contiguous in both X_b and Y_b.
//
// Two things shape the kernel.
// (1) The matrix instruction wants eight consecutive K (input channels) of one
// pixel in a lane, while memory has consecutive pixels of one channel.  That
// transposition happens in LDS the way transpose_u16_kernel does it: a tile of X
// (C_in rows of 128 pixels) is stored as dwords (two neighbouring pixels) with an
// odd row stride, a lane reads the dword of its pixel pair in eight consecutive
// channel rows (conflict-free) and v_perm picks its pixel's half of each.  The
// pixels are the A operand (rows of the accumulator block) and the weight the B
// operand (lanes = output channels), so that a lane holds runs of four consecutive
// pixels of ONE output channel and the accumulators reach the output strip in LDS
// (rows = channels, elements = pixels) with 8-byte writes.
// (2) Output rows are P_b elements apart, so a 64-pixel piece of every row starts
// somewhere inside a 128-byte line, differently for every row, and a piece that
// covers two half lines is written at about half the rate of whole lines (measured:
// 2.5 TB/s of stores, which made a first version with plain 64-pixel tiles slower
// than the transposes it replaced).  So a tile is not a rectangle: tile k of an
// image is, for every output row, the 64 pixels of that row's k-th 128-byte LINE.
// The rows' lines begin up to 63 pixels before pixel 64 k, so the wavefront
// multiplies the 128 pixels [64 k - 64, 64 k + 64) (twice the matrix work, which
// is not what bounds the kernel) and every row then takes its own aligned
// 64-pixel window out of the strip: five dword reads and four v_alignbit per
// 16-byte piece when the window starts on an odd pixel.  Every store instruction
// of the wavefront then writes eight whole lines; only a row's first and last
// line are partial.
//
// (3) With two wavefronts per SIMD the instructions of a tile count.  Nearly all tiles lie
// inside their image with their whole window, and those load and store without a look at
// the bounds; an output row's position moves on by one addition, and the half-dword
// shift of a window is the variable count of v_alignbit.  Stores go past the L2, which
// a result of this size does not fit.  On input that no cache holds 64 -> 256 channels on
// 591 264 pixels (378 MB) 129.9 -> 111.0 us = 3.4 TB/s, 32 -> 128 on 1.4 M (448 MB) 118.5 -> 101.7,
// 128 -> 64 on 128 437 (49 MB) 45.8 -> 40.7; on input that lies in the memory-side cache 128.5 ->
// 102.2, 119.4 -> 81.9 and 42.8 -> 38.6.
//
// Large results only; the others take conv1x1_direct_kernel.
//
// Persistent workgroups (the weight is loaded into LDS once each) of WAVES
// wavefronts, and every wavefront works on tiles of its own with its own X tile
// and strip: no workgroup barrier after the weight is in place, the next tile's
// pixels are in flight in registers while the current tile is multiplied and
// stored, and the wavefronts of a compute unit drift apart so that their loads,
// products and stores overlap.
#include "attn_common.h"
#include <type_traits>

namespace nt {

constexpr int kConvTile = 64;                 // pixels of a row that one tile writes
constexpr int kConvMaxIn = 128, kConvMaxOut = 512;

// The weight into LDS, rows of `ld` elements.
template <typename T, int THREADS>
__device__ __forceinline__ void load_weight(const T* __restrict__ w, T* lds, int ld, int c_in, int c_out) {
  const int per_row = c_in / 8;
  for (int i = threadIdx.x; i < c_out * per_row; i += THREADS) {
    const int row = i / per_row, ch = i - row * per_row;
    const u32x4 v = *reinterpret_cast<const u32x4*>(w + (size_t)row * c_in + ch * 8);
    *reinterpret_cast<u32x4*>(lds + (size_t)row * ld + ch * 8) = v;
  }
}

template <typename T, int WAVES, int LOADS>
__global__ __launch_bounds__(64 * WAVES) void conv1x1_nchw_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                                  T* __restrict__ y,
                                                                  const int64_t* __restrict__ pix_offsets,
                                                                  const int64_t* __restrict__ tile_offsets, int64_t B,
                                                                  int64_t total_tiles, int c_in, int c_out) {
  typedef AttnT<T> AT;
  typedef typename AT::Frag Frag;
  constexpr int TW = 2 * kConvTile;             // pixels multiplied per tile
  constexpr int kPB = TW / 32;                  // 32-pixel blocks of those
  // LOADS: load instructions per tile and lane, each covering 4 channel rows of 128
  // pixels (a compile-time bound keeps the staged pieces in registers)
  constexpr int KS = LOADS / 4;                 // 16-channel steps of the product, at most
  constexpr int S = TW / 2 + 1;                 // dwords per row of the X tile (odd)
  constexpr int SSD = TW / 2 + 4;               // dwords per row of the output strip (8-byte aligned rows)
  extern __shared__ __align__(16) char lds[];
  const int SW = c_in + 8;                      // elements per row of the weight in LDS
  const int t = threadIdx.x, l = t & 63, wave = t >> 6;
  T* Wl = reinterpret_cast<T*>(lds);
  // The strip takes the place of the X tile: the tile is read into registers (pf) in full
  // before the first channel block is stored, and LDS operations of one wavefront
  // execute in order.
  const size_t x_bytes = (size_t)c_in * S * 4, strip_bytes = (size_t)32 * SSD * 4;
  char* mine = lds + (size_t)c_out * SW * sizeof(T) + (size_t)wave * (x_bytes > strip_bytes ? x_bytes : strip_bytes);
  uint32_t* Xl = reinterpret_cast<uint32_t*>(mine);
  uint32_t* strip = reinterpret_cast<uint32_t*>(mine);

  load_weight<T, 64 * WAVES>(w, Wl, SW, c_in, c_out);     // once
  __syncthreads();
  // tiles of this wavefront: first, first + G * WAVES, ... with G workgroups; the
  // workgroups of one XCD (ids congruent modulo 8) take a contiguous run
  const int64_t G = gridDim.x;
  int64_t wg = blockIdx.x;
  if (G % 8 == 0) wg = (int64_t)(blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
  const int64_t stride = G * WAVES;
  int64_t tile = wg * WAVES + wave;

  const int chunk = l & 15, row0 = l >> 4;      // this lane's 16-byte piece: 8 pixels of row row0 + 4 i
  u32x4 stage[LOADS];
  // pixels of the image, 64 k of the tile, image, its first pixel, and its tile range
  // (a wavefront's tiles are G * WAVES apart and an image has thousands: the range is
  // kept in registers and the search runs only when a tile leaves it)
  int64_t P = 0, k64 = 0, img = 0, pix0 = 0, t_lo = 0, t_hi = 0;
  auto locate = [&](int64_t id) {
    if (id >= t_hi) {
      img = find_segment_uniform(tile_offsets, B, id);
      t_lo = tile_offsets[img];
      t_hi = tile_offsets[img + 1];
      pix0 = pix_offsets[img];
      P = pix_offsets[img + 1] - pix0;
    }
    k64 = (id - t_lo) * kConvTile;
  };
  // all 128 pixels of the tile's window lie inside the image
  auto interior = [&](int64_t k, int64_t pixels) { return k >= kConvTile && k + kConvTile <= pixels; };
  auto fetch = [&]() {
    const int64_t first = k64 - kConvTile + chunk * 8;      // first pixel of this piece, may lie outside [0, P)
    const char* p = reinterpret_cast<const char*>(x + pix0 * c_in + first + row0 * P);
    const int64_t step = 8 * P;                             // bytes from one row of four to the next
    if (interior(k64, P)) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        if (4 * i < c_in) stage[i] = load16_unaligned(p);
        p += step;
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (4 * i >= c_in) {
      } else if (first >= 0 && first + 8 <= P) {
        v = load16_unaligned(p);
      } else if (first + 8 > 0 && first < P) {
        T e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          e[j] = (first + j >= 0 && first + j < P) ? reinterpret_cast<const T*>(p)[j] : (T)0.0f;
        }
        __builtin_memcpy(&v, e, 16);
      }
      stage[i] = v;
      p += step;
    }
  };
  if (tile < total_tiles) {
    locate(tile);
    fetch();
  }
  const int n = l & 31, g = l >> 5;
  const uint32_t sel = (n & 1) ? 0x07060302u : 0x05040100u;
  const int nob = c_out / 32;
  while (tile < total_tiles) {
    const int64_t cur_P = P, cur_k64 = k64, cur_pix0 = pix0;
    // registers -> this wavefront's X tile
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      if (4 * i < c_in) {
        uint32_t* d = Xl + (row0 + 4 * i) * S + chunk * 4;
        d[0] = stage[i].x;
        d[1] = stage[i].y;
        d[2] = stage[i].z;
        d[3] = stage[i].w;
      }
    }
    __builtin_amdgcn_wave_barrier();
    const int64_t next = tile + stride;
    if (next < total_tiles) {
      locate(next);
      fetch();                                   // in flight during the products and stores below
    }
    // the pixel operands of the whole tile, once: pixel n of block pb, channels 16 ks + 8 g .. + 7
    Frag pf[KS][kPB];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (16 * ks < c_in) {
#pragma unroll
        for (int pb = 0; pb < kPB; ++pb) {
          const uint32_t* col = Xl + (16 * ks + 8 * g) * S + ((32 * pb + n) >> 1);
          uint32_t xv[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) xv[j] = col[j * S];
          u32x4 f;
          f.x = __builtin_amdgcn_perm(xv[1], xv[0], sel);
          f.y = __builtin_amdgcn_perm(xv[3], xv[2], sel);
          f.z = __builtin_amdgcn_perm(xv[5], xv[4], sel);
          f.w = __builtin_amdgcn_perm(xv[7], xv[6], sel);
          __builtin_memcpy(&pf[ks][pb], &f, 16);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();                          // the X tile is dead from here on
    const int64_t y_img = cur_pix0 * c_out;                  // first element of the image in y
    const bool whole = interior(cur_k64, cur_P);
    // first element of the output row a lane is at: r0, then every eighth row
    const int r0 = l >> 3, j8 = 8 * (l & 7);
    int64_t row_start = y_img + r0 * cur_P;
    T* const y_tile = y + cur_k64 + j8;
    for (int ob = 0; ob < nob; ++ob) {
      acc16 acc[kPB];
#pragma unroll
      for (int pb = 0; pb < kPB; ++pb)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[pb][e] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (16 * ks < c_in) {
          const Frag wf = *reinterpret_cast<const Frag*>(Wl + (size_t)(ob * 32 + n) * SW + 16 * ks + 8 * g);
#pragma unroll
          for (int pb = 0; pb < kPB; ++pb) acc[pb] = AT::mma(pf[ks][pb], wf, acc[pb]);
        }
      }
      // accumulators (rows = pixels 8 q + 4 g + 0..3 of block pb, lane = channel n of the
      // block) -> strip row n, 8 bytes per run of four pixels
#pragma unroll
      for (int pb = 0; pb < kPB; ++pb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t two[2];
          two[0] = AT::cvt2(acc[pb][4 * q], acc[pb][4 * q + 1]);
          two[1] = AT::cvt2(acc[pb][4 * q + 2], acc[pb][4 * q + 3]);
          uint64_t v;
          __builtin_memcpy(&v, two, 8);
          *reinterpret_cast<uint64_t*>(strip + n * SSD + ((32 * pb + 8 * q + 4 * g) >> 1)) = v;
        }
      __builtin_amdgcn_wave_barrier();
      // every row takes the 64 pixels of its own line k out of the strip
      auto rows = [&](auto whole_c) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole_c)::value;
#pragma unroll
        for (int ps = 0; ps < 4; ++ps) {
          const int ph = (int)row_start & 63;
          const int col = kConvTile - ph + j8;                                 // first strip element of the piece
          const uint32_t* src = strip + (r0 + 8 * ps) * SSD + (col >> 1);
          uint32_t d[5];
#pragma unroll
          for (int i = 0; i < 5; ++i) d[i] = src[i];
          const uint32_t odd = (uint32_t)(col & 1) * 16;
          u32x4 v;
          v.x = __builtin_amdgcn_alignbit(d[1], d[0], odd);
          v.y = __builtin_amdgcn_alignbit(d[2], d[1], odd);
          v.z = __builtin_amdgcn_alignbit(d[3], d[2], odd);
          v.w = __builtin_amdgcn_alignbit(d[4], d[3], odd);
          T* qd = y_tile + (row_start - ph);                                 // 16-byte aligned by construction
          const int64_t pixel = cur_k64 - ph + j8;                             // first pixel of the piece
          if (WHOLE || (pixel >= 0 && pixel + 8 <= cur_P)) {
            store16_stream(reinterpret_cast<char*>(qd), v);
          } else if (pixel + 8 > 0 && pixel < cur_P) {
            T e[8];
            __builtin_memcpy(e, &v, 16);
#pragma unroll
            for (int i = 0; i < 8; ++i)
              if (pixel + i >= 0 && pixel + i < cur_P) qd[i] = e[i];
          }
          row_start += 8 * cur_P;
        }
      };
      if (whole) {
        rows(std::true_type());
      } else {
        rows(std::false_type());
      }
      __builtin_amdgcn_wave_barrier();
    }
    tile = next;
  }
}

// The same product without LDS for pixels and results.  A wavefront takes a window of 64
// pixels; lane n holds pixels 2 n and 2 n + 1, one dword of every channel row straight from
// global memory, and v_perm makes an operand of the even and one of the odd pixels of it.  With
// the weight as the A operand a lane ends up with runs of four output channels of its pixels,
// so the even and the odd accumulator of a channel are one dword of the result: 128 contiguous
// bytes of a row per store and lane half.  Nothing is transposed, no window is
// multiplied twice, and CG wavefronts share a window, a CG-th of the output channels each, so
// that a small batch still spreads over the chip (us, in the cache / not, whole-line kernel -> here):
//   64 -> 256 on 2 600, 29 000, 127 000 pixels    28 / 31 -> 8 / 10, 28 / 33 -> 10 / 14, 36 / 44 -> 20 / 28
//   64 -> 64  on 2 800, 32 000, 128 000           15 / 18 -> 6 / 7, 15 / 17 -> 6 / 8, 17 / 22 -> 10 / 15
//   32 -> 128 on 3 400, 31 000, 122 000           14 / 16 -> 5 / 6, 14 / 16 -> 6 / 9, 15 / 19 -> 11 / 15
//   128 -> 256 on 35 000, 110 000, 517 000        54 / 67 -> 17 / 21, 93 / 103 -> 25 / 32, 249 / 260 -> 141 / 148
//   128 -> 64  on 95 000, 549 000                 37 / 43 -> 12 / 18, 92 / 113 -> 53 / 89
// A row's 128 bytes are no whole line, and the parts of a line come from two wavefronts: they
// meet in the L2 as long as the result is not much larger than that.  Beyond 64 MiB the
// whole lines of conv1x1_nchw_kernel win (64 -> 256 on 552 000 pixels 84 / 93 against 127 / 168,
// 64 -> 64 on 559 000 43 / 49 against 39 / 57, 96 -> 256 on 443 000 121 / 127 against 130 / 142), but not
// where its tiles leave the LDS no room for enough wavefronts (96 -> 64 on 524 000 137 / 227
// against 40 / 63, 128 channels above).
template <typename T, int KS, int CG>
__global__ __launch_bounds__(512, 2) void conv1x1_direct_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                                T* __restrict__ y, const int64_t* __restrict__ pix_offsets,
                                                                const int64_t* __restrict__ tile_offsets, int64_t B,
                                                                int64_t total_tiles, int c_in, int c_out) {
  typedef AttnT<T> AT;
  typedef typename AT::Frag Frag;
  typedef uint32_t Pair __attribute__((aligned(2)));       // two pixels of a row, wherever it begins
  constexpr int WAVES = 8;
  extern __shared__ __align__(16) char lds[];
  const int SW = c_in + 8;                      // elements per row of the weight in LDS
  const int t = threadIdx.x, l = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n = l & 31, g = l >> 5;
  T* Wl = reinterpret_cast<T*>(lds);
  load_weight<T, 64 * WAVES>(w, Wl, SW, c_in, c_out);
  __syncthreads();

  const int nob = c_out / 32, cg = wave % CG;
  const int ob_lo = cg * nob / CG, ob_hi = (cg + 1) * nob / CG;
  // tiles of this wavefront; the workgroups of one XCD take a contiguous run of each round
  const int64_t G = gridDim.x;
  int64_t wg = blockIdx.x;
  if (G % 8 == 0) wg = (int64_t)(blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
  int64_t tile = (wg * WAVES + wave) / CG;
  const int64_t stride = G * WAVES / CG;
  int64_t P = 0, k64 = 0, pix0 = 0, t_lo = 0, t_hi = 0;
  // goes to the next tile with pixels (the last of an image has none); false: there is none
  auto locate = [&]() {
    for (; tile < total_tiles; tile += stride) {
      if (tile >= t_hi) {
        const int64_t img = find_segment_uniform(tile_offsets, B, tile);
        t_lo = tile_offsets[img];
        t_hi = tile_offsets[img + 1];
        pix0 = pix_offsets[img];
        P = pix_offsets[img + 1] - pix0;
      }
      k64 = (tile - t_lo) * kConvTile;
      if (k64 < P) return true;
    }
    return false;
  };
  uint32_t stage[KS][8];                        // channels 16 ks + 8 g + j
  auto fetch = [&]() {
    const T* p = x + pix0 * c_in + k64 + 8 * g * P + 2 * n;
    const int64_t left = P - k64 - 2 * n;       // pixels from this lane's first on
    const bool whole = k64 + kConvTile <= P;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (16 * ks >= c_in) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const T* q = p + (16 * ks + j) * P;
        if (whole || left >= 2) {
          stage[ks][j] = *reinterpret_cast<const Pair*>(q);
        } else {
          stage[ks][j] = left == 1 ? *reinterpret_cast<const uint16_t*>(q) : 0u;
        }
      }
    }
  };
  bool have = locate();
  if (have) fetch();
  while (have) {
    const int64_t cur_P = P, cur_k64 = k64, cur_pix0 = pix0;
    Frag xf[KS][2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (16 * ks >= c_in) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        u32x4 f;
#pragma unroll
        for (int d = 0; d < 4; ++d)
          f[d] = __builtin_amdgcn_perm(stage[ks][2 * d + 1], stage[ks][2 * d], i ? 0x07060302u : 0x05040100u);
        __builtin_memcpy(&xf[ks][i], &f, 16);
      }
    }
    tile += stride;
    have = locate();
    if (have) fetch();                          // in flight during the products and stores below
    T* out = y + cur_pix0 * c_out + cur_k64 + (32 * ob_lo + 4 * g) * cur_P + 2 * n;
    const int64_t left = cur_P - cur_k64 - 2 * n;
    const bool whole = cur_k64 + kConvTile <= cur_P;
    for (int ob = ob_lo; ob < ob_hi; ++ob) {
      acc16 acc[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (16 * ks >= c_in) continue;
        const Frag wf = *reinterpret_cast<const Frag*>(Wl + (size_t)(ob * 32 + n) * SW + 16 * ks + 8 * g);
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i] = AT::mma(wf, xf[ks][i], acc[i]);
      }
      // accumulator e: channel 32 ob + 8 (e / 4) + 4 g + e % 4
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t two = AT::cvt2(acc[0][e], acc[1][e]);
        T* q = out + (8 * (e / 4) + e % 4) * cur_P;
        if (whole || left >= 2) {
          *reinterpret_cast<Pair*>(q) = two;
        } else if (left == 1) {
          *reinterpret_cast<uint16_t*>(q) = (uint16_t)two;
        }
      }
      out += 32 * cur_P;
    }
  }
}

static size_t conv_lds_bytes(int c_in, int c_out, int waves, size_t elem) {
  const size_t x_bytes = (size_t)c_in * (kConvTile + 1) * 4, strip_bytes = (size_t)32 * (kConvTile + 4) * 4;
  return (size_t)c_out * (c_in + 8) * elem + (size_t)waves * (x_bytes > strip_bytes ? x_bytes : strip_bytes);
}

template <typename T, int WAVES, int LOADS>
static int launch_conv(const void* x, const void* w, void* y, const int64_t* pix_offsets, const int64_t* tile_offsets,
                       int64_t B, int64_t total_tiles, int c_in, int c_out, int cus, hipStream_t stream) {
  const size_t lds = conv_lds_bytes(c_in, c_out, WAVES, sizeof(T));
  auto kernel = conv1x1_nchw_kernel<T, WAVES, LOADS>;
  const int rc = allow_lds<conv1x1_nchw_kernel<T, WAVES, LOADS>>(160 * 1024, "conv1x1");
  if (rc != NT_OK) return rc;
  int64_t grid = cus;
  const int64_t needed = (total_tiles + WAVES - 1) / WAVES;
  if (grid > needed) grid = needed;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * WAVES), lds, stream, static_cast<const T*>(x),
                     static_cast<const T*>(w), static_cast<T*>(y), pix_offsets, tile_offsets, B, total_tiles, c_in,
                     c_out);
  return check_launch("conv1x1_nchw_kernel");
}

template <typename T, int WAVES>
static int launch_conv_w(const void* x, const void* w, void* y, const int64_t* pix_offsets,
                         const int64_t* tile_offsets, int64_t B, int64_t total_tiles, int c_in, int c_out, int cus,
                         hipStream_t stream) {
#define NT_CONV_ARGS x, w, y, pix_offsets, tile_offsets, B, total_tiles, c_in, c_out, cus, stream
  if (c_in <= 16) return launch_conv<T, WAVES, 4>(NT_CONV_ARGS);
  if (c_in <= 32) return launch_conv<T, WAVES, 8>(NT_CONV_ARGS);
  if (c_in <= 64) return launch_conv<T, WAVES, 16>(NT_CONV_ARGS);
  return launch_conv<T, WAVES, 32>(NT_CONV_ARGS);
#undef NT_CONV_ARGS
}

template <typename T, int KS, int CG>
static int launch_direct(const void* x, const void* w, void* y, const int64_t* pix_offsets, const int64_t* tile_offsets,
                         int64_t B, int64_t total_tiles, int c_in, int c_out, int cus, hipStream_t stream) {
  auto kernel = conv1x1_direct_kernel<T, KS, CG>;
  const int rc = allow_lds<conv1x1_direct_kernel<T, KS, CG>>(160 * 1024, "conv1x1");
  if (rc != NT_OK) return rc;
  int64_t grid = cus;
  const int64_t needed = (total_tiles * CG + 7) / 8;
  if (grid > needed) grid = needed;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(512), (size_t)c_out * (c_in + 8) * sizeof(T), stream,
                     static_cast<const T*>(x), static_cast<const T*>(w), static_cast<T*>(y), pix_offsets, tile_offsets, B,
                     total_tiles, c_in, c_out);
  return check_launch("conv1x1_direct_kernel");
}

template <typename T, int CG>
static int launch_direct_ks(const void* x, const void* w, void* y, const int64_t* pix_offsets, const int64_t* tile_offsets,
                            int64_t B, int64_t total_tiles, int c_in, int c_out, int cus, hipStream_t stream) {
#define NT_CONV_ARGS x, w, y, pix_offsets, tile_offsets, B, total_tiles, c_in, c_out, cus, stream
  if (c_in <= 16) return launch_direct<T, 1, CG>(NT_CONV_ARGS);
  if (c_in <= 32) return launch_direct<T, 2, CG>(NT_CONV_ARGS);
  if (c_in <= 64) return launch_direct<T, 4, CG>(NT_CONV_ARGS);
  return launch_direct<T, 8, CG>(NT_CONV_ARGS);
#undef NT_CONV_ARGS
}

// The most wavefronts per workgroup (8, 7, 6, 4 or 2) whose tiles fit the LDS beside the weight; 0: none.
static int conv_waves(int c_in, int c_out, size_t elem) {
  const int choices[] = {8, 7, 6, 4, 2};
  for (int waves : choices) {
    if (conv_lds_bytes(c_in, c_out, waves, elem) <= 160 * 1024) return waves;
  }
  return 0;
}

// What a convolution runs on: `waves` wavefronts per workgroup of conv1x1_nchw_kernel, or `parts`
// wavefronts per window of conv1x1_direct_kernel.  Both 0: it does not fit the LDS.
struct ConvRoute {
  int waves, parts;
};

static ConvRoute choose_conv(int64_t B, int64_t total_tiles, int c_in, int c_out, int cus, size_t elem) {
  // Which kernel: see conv1x1_direct_kernel.  (total_tiles counts one tile too many per image.)
  const int64_t windows = total_tiles - B > 0 ? total_tiles - B : 0;
  const bool small = windows <= (int64_t(64) << 20) / (kConvTile * (int64_t)elem) / c_out;
  const int64_t round = 8 * (int64_t)cus;         // wavefronts in flight
  // Few channels leave little to save: whole lines win from two or three rounds of windows on (16 -> 64 on
  // 300 000 pixels 17.1 against 17.8, on 400 000 19.6 against 23.0, 32 -> 96 on 300 000 25.5 against 27.5, 16 -> 32 on
  // 400 000 15.3 against 15.4, on 900 000 22.7 against 25.8; but 32 -> 32 34.8 against 34.2).
  const bool few_channels = c_out == 32 ? c_in == 16 && windows > 3 * round : c_in <= 32 && c_out <= 96 && windows > 2 * round;
  if ((small && !few_channels) || c_in > 96 || (c_in > 64 && c_out <= 2 * c_in)) {
    if ((size_t)c_out * (c_in + 8) * elem > 160 * 1024) return {0, 0};
    // As many wavefronts per window as one round of them can take (4 / 2 / 1, us: 64 -> 256 on 24 000
    // pixels 9.5 / 11.6 / 16.0, on 40 000 18.4 / 12.4 / 16.7, on 75 000 28.9 / 27.0 / 20.0).
    if (c_out % 128 == 0 && 4 * windows <= round) return {0, 4};
    if (2 * windows <= round) return {0, 2};
    if (windows <= round) return {0, 1};
    // Beyond one round two to a window while three half rounds do for two whole ones (2 / 1: 64 -> 96 on
    // 150 000 24.7 / 27.5, on 200 000 31.0 / 27.9), and for many input channels, whose windows take longest
    // to fetch (128 -> 64 on 200 000 31.1 / 39.2, on 700 000 82.5 / 89.7).
    // With 32 output channels the second wavefront only fetches the same pixels: worth it where the
    // windows are few (32 -> 32 on 30 000 5.4 / 6.0, 96 -> 32 on 150 000 18.8 / 27.9), but not for few channels
    // beyond a round (32 -> 32 on 900 000 44.8 / 34.2) or beyond four rounds (96 -> 32 on 900 000 77.6 / 67.5).
    const bool two = 2 * windows <= 3 * round ? c_out > 32 || c_in > 32 : c_in > 64 && (c_out > 32 || windows <= 4 * round);
    return {0, two ? 2 : 1};
  }
  return {conv_waves(c_in, c_out, elem), 0};
}

template <typename T>
static int launch_conv_t(const void* x, const void* w, void* y, const int64_t* pix_offsets, const int64_t* tile_offsets,
                         int64_t B, int64_t total_tiles, int c_in, int c_out, int cus, hipStream_t stream) {
#define NT_CONV_ARGS x, w, y, pix_offsets, tile_offsets, B, total_tiles, c_in, c_out, cus, stream
  const ConvRoute route = choose_conv(B, total_tiles, c_in, c_out, cus, sizeof(T));
  switch (route.parts) {
    case 4: return launch_direct_ks<T, 4>(NT_CONV_ARGS);
    case 2: return launch_direct_ks<T, 2>(NT_CONV_ARGS);
    case 1: return launch_direct_ks<T, 1>(NT_CONV_ARGS);
    default: break;
  }
  switch (route.waves) {
    case 8: return launch_conv_w<T, 8>(NT_CONV_ARGS);
    case 7: return launch_conv_w<T, 7>(NT_CONV_ARGS);
    case 6: return launch_conv_w<T, 6>(NT_CONV_ARGS);
    case 4: return launch_conv_w<T, 4>(NT_CONV_ARGS);
    case 2: return launch_conv_w<T, 2>(NT_CONV_ARGS);
    default: break;
  }
#undef NT_CONV_ARGS
  return fail(NT_ERR_UNSUPPORTED, "conv1x1: %d -> %d channels do not fit the LDS", c_in, c_out);
}

}  // namespace nt

using namespace nt;

static int compute_units(int* cus) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || *cus < 1) {
    (void)hipGetLastError();
    return fail(NT_ERR_HIP, "conv1x1: cannot query the device");
  }
  return NT_OK;
}

extern "C" int64_t nt_conv1x1_tile_pixels(void) { return kConvTile; }

extern "C" int nt_conv1x1_supported(int64_t c_in, int64_t c_out, int dtype) {
  if (dtype != NT_F16 && dtype != NT_BF16) return 0;
  if (c_in < 16 || c_in % 16 != 0 || c_in > kConvMaxIn || c_out < 32 || c_out % 32 != 0 || c_out > kConvMaxOut) return 0;
  // of a small batch and of a large one
  for (int64_t tiles : {int64_t(1), int64_t(0x7fffffff)}) {
    const ConvRoute route = choose_conv(0, tiles, (int)c_in, (int)c_out, 256, 2);
    if (route.waves == 0 && route.parts == 0) return 0;
  }
  return 1;
}

extern "C" int nt_conv1x1_route(int64_t B, int64_t total_tiles, int64_t c_in, int64_t c_out, int dtype, int num_cus,
                                int* route) {
  if (B < 0 || total_tiles < 0 || num_cus < 0 || !route) return fail(NT_ERR_INVALID_ARGUMENT, "conv1x1_route: bad arguments");
  if (!nt_conv1x1_supported(c_in, c_out, dtype)) {
    return fail(NT_ERR_UNSUPPORTED, "conv1x1: %lld -> %lld channels", (long long)c_in, (long long)c_out);
  }
  if (num_cus == 0) {
    const int rc = compute_units(&num_cus);
    if (rc != NT_OK) return rc;
  }
  const ConvRoute r = choose_conv(B, total_tiles, (int)c_in, (int)c_out, num_cus, 2);
  route[0] = r.waves;
  route[1] = r.parts;
  return NT_OK;
}

extern "C" int nt_conv1x1_nchw(const void* x, const void* weight, void* y, const int64_t* pix_offsets,
                               const int64_t* tile_offsets, int64_t B, int64_t total_tiles, int64_t c_in,
                               int64_t c_out, int dtype, void* stream) {
  if (B < 0 || total_tiles < 0 || c_in < 1 || c_out < 1) {
    return fail(NT_ERR_INVALID_ARGUMENT, "conv1x1: bad shape");
  }
  if (c_in % 16 != 0 || c_in > kConvMaxIn || c_out % 32 != 0 || c_out > kConvMaxOut) {
    return fail(NT_ERR_UNSUPPORTED,
                "conv1x1: %lld -> %lld channels (input channels: a multiple of 16 up to %d; output channels: a "
                "multiple of 32 up to %d)", (long long)c_in, (long long)c_out, kConvMaxIn, kConvMaxOut);
  }
  if (dtype != NT_F16 && dtype != NT_BF16) return fail(NT_ERR_UNSUPPORTED, "conv1x1: dtype must be f16 or bf16");
  if (B == 0 || total_tiles == 0) return NT_OK;
  if (!x || !weight || !y || !pix_offsets || !tile_offsets) return fail(NT_ERR_INVALID_ARGUMENT, "conv1x1: NULL pointer");
  if ((reinterpret_cast<uintptr_t>(weight) & 15) != 0 || (reinterpret_cast<uintptr_t>(y) & 127) != 0) {
    return fail(NT_ERR_INVALID_ARGUMENT, "conv1x1: the weight must be 16-byte and the output 128-byte aligned");
  }
  if (total_tiles > 0x7fffffffLL) return fail(NT_ERR_UNSUPPORTED, "conv1x1: too many tiles");
  int cus = 0;
  const int rc = compute_units(&cus);
  if (rc != NT_OK) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == NT_F16) {
    return launch_conv_t<_Float16>(x, weight, y, pix_offsets, tile_offsets, B, total_tiles, (int)c_in, (int)c_out, cus, s);
  }
  return launch_conv_t<__bf16>(x, weight, y, pix_offsets, tile_offsets, B, total_tiles, (int)c_in, (int)c_out, cus, s);
}
