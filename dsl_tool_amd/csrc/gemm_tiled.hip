// Dense quantized GEMM: C[M,N] = A[M,K] . W[N,K]^T on gfx950 MFMA.
// Variant selection (tile shape, split-K) lives in launch_gemm below.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "gemm_core.h"

namespace dsl {

// Floats between consecutive split-K partial slices in the workspace: M*N
// rounded up to whole float4s, so that every slice starts 16-byte aligned.
__host__ __device__ inline int64_t splitk_slice(int64_t M, int64_t N) {
  return (M * N + 3) / 4 * 4;
}

template <int MODE, class Cfg>
__global__ __launch_bounds__(Cfg::NT) void gemm_tiled_kernel(const GemmArgs p) {
  __shared__ __align__(16) uint8_t smem[Cfg::LDS];
  const int nbm = (p.M + Cfg::BM - 1) / Cfg::BM, nbn = (p.N + Cfg::BN - 1) / Cfg::BN;
  int tmi, tni;
  tile_coords(blockIdx.x, nbm, nbn, tmi, tni);
  const int m0 = tmi * Cfg::BM, n0 = tni * Cfg::BN;

  TileView tv;
  tv.a = p.a + (int64_t)m0 * p.Kb;
  tv.b = p.b + (int64_t)n0 * p.Kb;
  tv.a_rows = min(Cfg::BM, p.M - m0);
  tv.b_rows = min(Cfg::BN, p.N - n0);
  tv.Kb = p.Kb;
  tv.K = p.K;
  tv.sa = tv.sb = nullptr;
  tv.sa_ld = tv.sb_ld = 0;
  if constexpr (MODE == MODE_MXFP4 || MODE == MODE_NVFP4) {
    const int64_t ld = MODE == MODE_MXFP4 ? p.K / 32 : p.K / 16;
    tv.sa = static_cast<const uint8_t *>(p.sa) + (int64_t)m0 * ld;
    tv.sb = static_cast<const uint8_t *>(p.sb) + (int64_t)n0 * ld;
    tv.sa_ld = tv.sb_ld = ld;
  } else if constexpr (MODE == MODE_FP8_BLOCK) {
    const int64_t nkg = (p.K + 127) / 128;
    tv.sa = static_cast<const float *>(p.sa) + (int64_t)m0 * nkg;
    tv.sb = static_cast<const float *>(p.sb) + (int64_t)(n0 / 128) * nkg;
    tv.sa_ld = tv.sb_ld = nkg;
  } else if constexpr (MODE == MODE_FP8_GCOL) {
    const int64_t nkg = (p.K + 127) / 128;
    tv.sa = static_cast<const float *>(p.sa) + (int64_t)m0 * nkg;
    tv.sb = static_cast<const float *>(p.sb) + n0;
    tv.sa_ld = nkg;
    tv.sb_ld = p.N;
  }

  const int nks = (p.Kb + 127) / 128;
  int ks0 = 0, ks1 = nks;
  if (p.ksplit > 1) {
    const int per = (nks + p.ksplit - 1) / p.ksplit;
    ks0 = blockIdx.y * per;
    ks1 = min(nks, ks0 + per);
  }

  v4f acc[Cfg::TM][Cfg::TN];
  tile_mainloop<MODE, Cfg>(tv, ks0, ks1, smem, acc);

  float s1 = 1.f, s2 = 1.f;
  if constexpr (MODE == MODE_FP8_TENSOR || MODE == MODE_NVFP4) {
    s1 = *p.ga;
    s2 = *p.gb;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / Cfg::WGN, wn = wave % Cfg::WGN;
  const int r16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int tm = 0; tm < Cfg::TM; ++tm)
#pragma unroll
    for (int tn = 0; tn < Cfg::TN; ++tn) {
      const int col = n0 + wn * Cfg::WN + tn * 16 + r16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + wm * Cfg::WM + tm * 16 + 4 * g + i;
        if (row < p.M && col < p.N) {
          float v = acc[tm][tn][i];
          if constexpr (MODE == MODE_FP8_TENSOR || MODE == MODE_NVFP4) v = (v * s1) * s2;
          if (p.ksplit > 1) {
            // this K split's own slice of the workspace: the finalize pass
            // adds the slices in split order, so every run sums alike
            p.ws[(int64_t)blockIdx.y * splitk_slice(p.M, p.N) + (int64_t)row * p.N + col] = v;
          } else if (p.out_f32) {
            float *d = static_cast<float *>(p.c) + (int64_t)row * p.ldc + col;
            *d = p.accumulate ? *d + v : v;
          }
          else
            static_cast<uint16_t *>(p.c)[(int64_t)row * p.ldc + col] = f32_to_bf16(v);
        }
      }
    }
}

// Split-K finalize: C (bf16, fp32, or fp32 += for accumulate) from the
// ksplit fp32 partial slices in ws ([ksplit][M][N], slice stride
// splitk_slice(M, N)), added in split order.  Rows over blockIdx.y
// (grid-stride), four columns per thread; `vec`: N % 4 == 0 and C rows
// aligned for 16-byte (fp32) / 8-byte (bf16) stores, so a thread moves its
// four columns with one load per slice and one store (no per-element index
// division).
__global__ void splitk_finalize_kernel(const float *__restrict__ ws, int ksplit,
                                       void *__restrict__ c, int M, int N, int64_t ldc,
                                       int out_f32, int accumulate, int vec) {
  const int col = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (col >= N) return;
  const int64_t slice = splitk_slice(M, N);
  for (int r = blockIdx.y; r < M; r += gridDim.y) {
    const float *src = ws + (int64_t)r * N + col;
    if (vec) {
      float4 v = *reinterpret_cast<const float4 *>(src);
      for (int s = 1; s < ksplit; ++s) {
        const float4 u = *reinterpret_cast<const float4 *>(src + s * slice);
        v = make_float4(v.x + u.x, v.y + u.y, v.z + u.z, v.w + u.w);
      }
      if (out_f32) {
        float4 *d = reinterpret_cast<float4 *>(static_cast<float *>(c) + r * ldc + col);
        if (accumulate) {
          const float4 o = *d;
          v = make_float4(o.x + v.x, o.y + v.y, o.z + v.z, o.w + v.w);
        }
        *d = v;
      } else {
        *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(c) + r * ldc + col) =
            make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
      }
    } else {
      for (int t = 0; t < 4 && col + t < N; ++t) {
        float v = src[t];
        for (int s = 1; s < ksplit; ++s) v += src[s * slice + t];
        if (out_f32) {
          float *d = static_cast<float *>(c) + r * ldc + col + t;
          *d = accumulate ? *d + v : v;
        } else {
          static_cast<uint16_t *>(c)[r * ldc + col + t] = f32_to_bf16(v);
        }
      }
    }
  }
}

// ----------------------------------------------------------------------------
// Variant selection.
// ----------------------------------------------------------------------------
namespace {

struct Plan {
  int variant;   // 0: 256x256 (8 waves)  1: 128x128 (4 waves)  2: 64x128  3: 16x256
  int bm, bn;
  int ksplit;
};

Plan plan_for(int M, int N, int Kb) {
  Plan pl;
  if (M <= 16) { pl.variant = 3; pl.bm = 16; pl.bn = 256; }
  else if (M <= 64) { pl.variant = 2; pl.bm = 64; pl.bn = 128; }
  else if (M <= 128 || N <= 128) { pl.variant = 1; pl.bm = 128; pl.bn = 128; }
  else { pl.variant = 0; pl.bm = 256; pl.bn = 256; }
  const int tiles = ((M + pl.bm - 1) / pl.bm) * ((N + pl.bn - 1) / pl.bn);
  const int nks = (Kb + 127) / 128;
  int ks = 1;
  if (tiles < 256) {
    ks = (256 + tiles - 1) / tiles;
    const int maxk = nks / 4 > 0 ? nks / 4 : 1;    // keep >= 4 stages per split
    if (ks > maxk) ks = maxk;
    if (ks > 16) ks = 16;
    if (ks < 1) ks = 1;
  }
  pl.ksplit = ks;
  return pl;
}

template <int MODE, class Cfg>
void launch_variant(const GemmArgs &p, hipStream_t st) {
  const int tiles = ((p.M + Cfg::BM - 1) / Cfg::BM) * ((p.N + Cfg::BN - 1) / Cfg::BN);
  dim3 grid(tiles, p.ksplit, 1);
  gemm_tiled_kernel<MODE, Cfg><<<grid, Cfg::NT, 0, st>>>(p);
}

template <int MODE>
void launch_mode(const Plan &pl, const GemmArgs &p, hipStream_t st) {
  switch (pl.variant) {
    case 0: launch_variant<MODE, TileCfg<MODE, 256, 256, 2, 4>>(p, st); break;
    case 1: launch_variant<MODE, TileCfg<MODE, 128, 128, 2, 2>>(p, st); break;
    case 2: launch_variant<MODE, TileCfg<MODE, 64, 128, 1, 4>>(p, st); break;
    default: launch_variant<MODE, TileCfg<MODE, 16, 256, 1, 4>>(p, st); break;
  }
}

}  // namespace

// True when environment variable `name` is "0", "off" or "false" (any case).
static bool env_off(const char *name) {
  const char *e = getenv(name);
  if (!e) return false;
  char buf[8] = {0};
  for (int i = 0; i < 7 && e[i]; ++i) buf[i] = (char)((e[i] >= 'A' && e[i] <= 'Z') ? e[i] + 32 : e[i]);
  return strcmp(buf, "0") == 0 || strcmp(buf, "off") == 0 || strcmp(buf, "false") == 0;
}

// Kernel path for a problem.  The choice depends on the shape and on the
// alignment of the scale pointers only, so the workspace query (which sees
// no pointers and assumes aligned scales) and the launch agree whenever the
// scales are aligned; with misaligned scales the launch may fall back to
// the register-staged kernels, split-K only if a workspace was passed.
//   DSL_GEMM_DECODE = 0/off    never use the skinny-M kernel
//   DSL_GEMM_STREAM = 0/off    never use the streaming kernel
//   DSL_GEMM_SKINNY = stream   2 <= M <= 16 on the streaming kernel too
//                              (default: the skinny-M decode kernel there)
//   DSL_GEMM_PIPE   = 0/off    never use the LDS-DMA pipelined kernels
//   DSL_GEMM_PIPE   = 1..9     force that pipelined variant for large problems
//                              (and no 64x128, deep 128x128 or 256x128 tiles)
//   DSL_GEMM_PERSIST = 0/off   use the per-tile pipelined kernels instead of
//                              the persistent one for large problems
enum { PATH_DECODE = 0, PATH_PIPE = 1, PATH_TILED = 2, PATH_PERSIST = 3, PATH_STREAM = 4 };
struct Route {
  int path;
  int variant;    // PATH_PIPE variant
  Plan tiled;     // PATH_TILED plan
  bool narrow = false;       // PATH_PERSIST: 256x128 tiles
  bool pad_scales = false;   // PATH_PERSIST / PATH_PIPE: E8M0 / E4M3 rows first copied to a padded pitch
};

// E8M0 / E4M3 scale rows that are no whole 16-byte quads (persistent kernel)
// or 4-byte words per stage (pipelined tiles): [rows][len] bytes -> [rows][pitch], `fill` past len (one launch for
// both operands; 4 bytes per thread).
__global__ void pad_scales_kernel(const uint8_t *__restrict__ a, int rows_a,
                                  const uint8_t *__restrict__ b, int rows_b, int len, int pitch,
                                  uint32_t fill, uint32_t *__restrict__ out) {
  const int wpr = pitch / 4;
  const int64_t total = ((int64_t)rows_a + rows_b) * wpr;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = i / wpr;
    const int c = (int)(i - row * wpr) * 4;
    const uint8_t *src = row < rows_a ? a + row * len : b + (row - rows_a) * len;
    uint32_t v = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) v |= (c + k < len ? (uint32_t)src[c + k] : fill) << (8 * k);
    out[i] = v;
  }
}

static int scale_row_len(int mode, int K) { return mode == MODE_MXFP4 ? K / 32 : K / 16; }
static int padded_pitch(int mode, int K) { return (scale_row_len(mode, K) + 15) / 16 * 16; }

constexpr int kAccShortK = 512;   // C += result with K up to this streams where it can

static bool stream_enabled() {
  static const bool on = !env_off("DSL_GEMM_STREAM");
  return on;
}

// DSL_GEMM_PIPE: -1 unset, -2 off, else the forced variant.
static int pipe_switch() {
  static const int forced = [] {
    if (env_off("DSL_GEMM_PIPE")) return -2;
    const char *e = getenv("DSL_GEMM_PIPE");
    return (e && e[0] >= '1' && e[0] <= '9' && !e[1]) ? e[0] - '0' : -1;
  }();
  return forced;
}

// The deep rings (variants 6, 7) advance the prefetching modes by pairs of
// 128-byte stages: an odd or partial last pair takes the ragged form, whose padding
// stage costs as much as a whole one.  Short K pays for it, and for filling the
// ring, against variant 1: per-tensor 724x3200x640 8.2 us / 6.3, 410x7680x1664
// 12.1 / 10.3, level from about 2560; whole pairs to K=1536 6.5 / 6.0.
static bool prefetches(int mode) { return mode == MODE_FP8_TENSOR || mode == MODE_BF16; }
static bool deep_pays(int mode, int Kb) { return !prefetches(mode) || Kb >= (Kb % 256 == 0 ? 1536 : 2560); }

// `padded`: a workspace for padded scale rows is there.  `ragged` false: the
// kernel that serves the shape without the ragged forms and the one-round tiles
// (rows and scale rows of whole steps only); the workspace contract is that
// route's.
static Route pick_route(int mode, int M, int N, int K, int Kb, bool sc4, bool sc16, bool padded, bool f32,
                        bool ragged) {
  static const bool decode_on = !env_off("DSL_GEMM_DECODE");
  const bool stream_on = stream_enabled();
  const char *skinny = getenv("DSL_GEMM_SKINNY");      // read per launch (tests switch it)
  const bool skinny_stream = skinny && strcmp(skinny, "stream") == 0;
  const bool skinny_decode = skinny && strcmp(skinny, "decode") == 0;
  static const bool persist_on = !env_off("DSL_GEMM_PERSIST");
  const int pipe_forced = pipe_switch();
  Route r{PATH_TILED, -1, plan_for(M, N, Kb)};
  bool streamable = stream_on && stream_supported(mode, M, N, K, Kb, sc4) &&
                    (ragged || stream_whole(mode, K, Kb, sc16));
  // The streaming kernel's time grows with the number of 64-row activation
  // blocks times N (each block streams all of W, and each W slice re-reads
  // its activation rows), while the 128x128 / persistent tiles stay at about
  // one round up to a few thousand rows.  The edge is a span of
  // 2 * ceil(M/64) * N (thr2 below, in units of 4096), measured for each
  // mode (the crossover moves little with K: both sides scale with it).
  // NVFP4 (dequantized to fp16 in the tiles) streams up to 256 rows whatever
  // N, and above that below span 30 (M=768 N=4096: 61.8 against 76.5 us;
  // M=320 N=14336: 91.4 against 88.1).  Rows of an odd number of 256-byte
  // chunks stream in 32-row blocks: twice the blocks.
  const int64_t t128 = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
  // (ragged K: from half the CUs; 768x1640x4168, 78 tiles, 58 us on them
  // against about 40 streamed)
  const bool bf16_pipe_round = mode == MODE_BF16 && pipe_forced != -2 && M > 64 &&
                               (Kb % 128 == 0 || (ragged && 2 * t128 >= device_cu_count())) &&
                               N > 64 && t128 >= 40 && t128 <= device_cu_count();
  // 64x128 pipelined tiles where one round of them holds the problem (not
  // NVFP4, which streams): 1.3-1.5 times faster than the 128x128 tiles they
  // replace there, and than the streaming kernel from a span of about 5
  // (M=192 N=K=4096, streamed / tiles: per-tensor 11.5 / 10.8 us, block 17.6 /
  // 16.1, groupwise 18.4 / 16.7; M=128 8.7 / 10.5, 10.0 / 15.9, 10.4 / 16.4);
  // MXFP4 and bf16 keep their edge of 9 (M=256: 9.0 / 10.5, 18.8 / 19.6).  At
  // least 24 tiles: fewer leave most CUs without one, and the register-staged
  // tiles split K over them.
  const int64_t t64 = (int64_t)((M + 63) / 64) * ((N + 127) / 128);
  const bool small = ragged && pipe_forced == -1 && mode != MODE_NVFP4 && M > 64 && N > 64 && t64 >= 24 &&
                     t64 <= device_cu_count() && (mode == MODE_FP8_TENSOR || mode == MODE_BF16 || sc4) &&
                     (mode != MODE_MXFP4 || Kb % 128 == 0 || padded);
  if (streamable && !skinny_stream && M > 32 && (mode != MODE_NVFP4 || M > 256)) {
    const int bm = stream_blocks64(mode, M, K, Kb, sc16) ? 64 : 32;
    const int64_t span2 = 2 * (int64_t)((M + bm - 1) / bm) * N;   // twice the span
    // crossovers re-measured against the prefetching / eight-wave 128x128
    // tiles (same-box sweep, M = 256..1024, N = 2048..14336, K = 2048 and
    // 4096; streamed against the tiles at the first span past the edge):
    // per-tensor and MXFP4 stream up to span 8 x 4096 (10: 12.5 against
    // 9.5 us, MXFP4 13.2 against 8.8), FP8 block up to 10 (14: 20.6 against
    // 14.7), groupwise per-column up to 12 (14: 21.4 against 15.8), bf16
    // where one round of tiles holds it up to 8 (10: 20.8 against 18.0),
    // other bf16 below 30 (35: 53.5 against 45.4 on the persistent tiles).
    // (whole lines of 128 bytes that are no whole 512 stream slower: 6 there;
    // bf16 700x1500x1472 20.4 / 14.2; other rows slow the tiles too, K=4160
    // M=256 N=4096 bf16 22.8 / 26.2, MXFP4 12.8 / 15.8)
    const bool plain = (stream_whole(mode, K, Kb, sc16) && Kb % 512 == 0) || Kb % 128 != 0;
    const int64_t thr2 = small ? (mode == MODE_MXFP4 || mode == MODE_BF16 ? (plain ? 9 : 6) : 5)
                         : mode == MODE_FP8_GCOL ? 13
                         : mode_grouped_k(mode) ? 11
                         : (mode == MODE_BF16 ? (bf16_pipe_round ? 9 : 30)
                                              : (mode == MODE_NVFP4 ? 30 : 9));
    if (span2 >= thr2 * 4096) streamable = false;
  }
  // Skinny M (measured, graph timing over rotating weights): the streaming
  // kernel is the faster one for M <= 8 (FP8, MXFP4: 4-25%), for bf16 at
  // every M <= 16 (5-26%), and at M = 9..16 wherever the decode kernel's
  // 32-row grid leaves CUs idle or needs a second round (N = 4096: 5.3
  // against 6.1 us, N = 14336: 11.4 against 13.1).  The decode kernel keeps
  // 9 <= M <= 16 when that grid fills 7/8 of the CUs or more in one round
  // (N = 7168: 7.1 against 7.4 us, N = 8192).  NVFP4: the GEMV for M = 1,
  // the streaming kernel above that (N=14336 K=4096: M=1 8.4 against 9.4 us;
  // M=2 10.0 against 14.4; M=4 10.0 against 22.5: the GEMV's time grows with
  // M).  DSL_GEMM_SKINNY=stream|decode forces one of them (tests).
  bool prefer_stream;
  if (skinny_stream) {
    prefer_stream = true;
  } else if (skinny_decode) {
    prefer_stream = false;
  } else if (mode == MODE_NVFP4) {
    prefer_stream = M > 1;
  } else if (M <= 8 || M > 16 || mode == MODE_BF16) {
    prefer_stream = true;
  } else {
    const int64_t g = (N + 31) / 32, cus = device_cu_count();
    prefer_stream = !(8 * g >= 7 * cus && g <= cus);
  }
  if (decode_on && !(prefer_stream && streamable) && decode_supported(mode, M, K, Kb, sc4, sc16)) {
    r.path = PATH_DECODE;
    return r;
  }
  if (streamable) {
    r.path = PATH_STREAM;
    return r;
  }
  const int one_round = ragged && mode != MODE_NVFP4 && t128 <= device_cu_count() && pipe_forced < 0 &&
                                deep_pays(mode, Kb) ? 7 : 1;
  if (small) {
    r.path = PATH_PIPE;
    // (an odd pair count at short K: 7.0 us, 6.4 in variant 1, per-tensor K=896)
    r.variant = prefetches(mode) && Kb % 256 == 128 && Kb < 1536 && t128 >= 40 ? 1 : 6;
    r.pad_scales = mode == MODE_MXFP4 && Kb % 128 != 0;
    return r;
  }
  // 256x128 persistent tiles where one round of them holds a problem that
  // takes the 128x128 tiles more than one round (and the 256x256 ones half a
  // round at most).  One full round costs about 0.65 of a full 256x256 round,
  // one of 128x128 tiles 0.41, two 0.72 (per-tensor K=4096: 37.3, 57.8, 23.5,
  // 41.9 us).  us before -> after, per-tensor / block / MXFP4 / NVFP4 / bf16:
  // 1500x4096x11008 109 -> 83, 109 -> 98, 71 -> 60, 222 -> 159, 188 -> 160;
  // 2048x4096x4096 42 -> 37, 45 -> 42, 31 -> 28, 90 -> 70, 80 -> 70.  NVFP4,
  // whose 128x128 tiles spend most of a stage dequantizing, from 0.6 rounds of
  // those (1024x4096x4096 74 -> 60; 512x4096x4096, half a round, 40 -> 44).
  const int64_t tn = (int64_t)((M + 255) / 256) * ((N + 127) / 128), cu = device_cu_count();
  const bool narrow = ragged && persist_on && pipe_forced < 0 && M > 128 && N > 128 && tn <= cu &&
                      (mode == MODE_NVFP4 ? 10 * t128 > 6 * cu : t128 > cu) &&
                      persist_supported(mode, M, N, K, Kb, sc4);
  // The persistent kernel's last column of tiles stores element by element where
  // its columns do not all exist (every tile where N % 8 != 0): up to 11 us per
  // 128 columns of it.  Against variant 1 the 256x128 tiles gain this much per
  // 1024 bytes of K, so short ragged problems stay there: per-tensor
  // 583x9952x512 18.5 us / 11.0, block 6720x752x1024 25.3 / 13.5.  (fp32
  // results: variant 1 stores those element by element too.)
  static constexpr float narrow_gain[] = {2.0f, 1.2f, 7.2f, 38.f, 2.0f, 0.f};   // by mode; NVFP4: two rounds
  auto last_tile = [&](int bn) { return N % 8 ? 1.f : (float)(N % bn) / bn; };
  const float gain = (mode == MODE_NVFP4 && t128 <= cu ? 8.f : narrow_gain[mode]) * Kb / 1024 -
                     (mode == MODE_MXFP4 ? 2.f : (mode == MODE_NVFP4 ? 1.f : 0.f));
  const bool narrow_wins = f32 || Kb % 128 != 0 || gain >= 11 * last_tile(128);
  if (mode == MODE_BF16) {   // pipelined, persistent or register-staged tiles
    const int64_t t256 = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
    // one round of 128x128 pipelined tiles (40 to one per CU) beats a
    // partial round of 256x256 persistent tiles, which leaves 3/4 of the
    // CUs idle (M=1536 N=2048 K=4096: 44.2 against 84.0 us; M=1024 N=4096:
    // 54.7 against 73.9); past one round the persistent kernel (M=1536
    // N=4096: 95.4 against 100.4).  Then one partial round of the persistent
    // kernel beats the register-staged tiles from about a sixth of the CUs'
    // worth of 256x256 tiles (M=768 N=4096 K=4096: 77 against 102 us;
    // M=2048 N=7168: 104 against 220) and about 2.4M outputs (M=288 N=7168,
    // 56 tiles of which 28 hold 32 rows: 77 against 70 us; M=384: 78 against
    // 89)
    if (bf16_pipe_round) {
      r.path = PATH_PIPE;
      r.variant = one_round;
    } else if (persist_on && 6 * t256 >= device_cu_count() && (int64_t)M * N >= 2400000 &&
               persist_supported(mode, M, N, K, Kb, sc4) && (ragged || Kb % 128 == 0)) {
      r.path = PATH_PERSIST;
    }
    if (narrow) {
      r.path = PATH_PERSIST;
      r.narrow = true;
    }
    return r;
  }
  // K of no whole 128 bytes: the ragged forms of both kernels, MXFP4 and NVFP4
  // with their scale rows at a padded pitch (the persistent kernel also where
  // only the scale rows are ragged)
  const bool fp4 = mode == MODE_MXFP4 || mode == MODE_NVFP4;
  const bool rag = Kb % 128 != 0, pad = fp4 && !persist_whole(mode, K, Kb, sc16);
  const bool pipe_ok = pipe_forced != -2 && (mode == MODE_FP8_TENSOR || sc4) &&
                       (!rag || (ragged && (!fp4 || padded)));
  const bool persist_ok = persist_on && pipe_forced < 0 &&
                          persist_supported(mode, M, N, K, Kb, sc4) && (!pad || padded) &&
                          (ragged || persist_whole(mode, K, Kb, sc16));
  if (pipe_ok) {
    const int64_t t256 = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
    // Rounds of tiles per CU: a round of 256x256 persistent tiles costs
    // about as much as 1.6 rounds of the 128x128 pipelined tiles (1.5-2 with
    // block scales), so the persistent kernel takes over once the 128x128
    // grid needs twice its rounds (three times with block scales); below
    // that the 128x128 tiles, down to 40 of them: one round of those beats
    // the register-staged split-K tiles by 1.3-4.6x (M=300 N=5000 K=4096:
    // 24 against 67 us; block 31 against 149).  Measured at N = 512..14336,
    // K = 4096 and 8192, M = 288..3072.  With the prefetching 128x128 tiles
    // FP8 per-tensor keeps two rounds of them too (same-box, M = 1536..4096,
    // N = 2048 and 4096, K = 2048 and 4096: 7-12% ahead of the persistent
    // kernel at six of seven shapes, 2048x4096x4096 41.1 against 42.2 us);
    // MXFP4 does not (two rounds: 33.9 against 28.1 us at 1536x4096x4096).
    const int64_t cus = device_cu_count();
    const int64_t r128 = (t128 + cus - 1) / cus, r256 = (t256 + cus - 1) / cus;
    const int rounds128 = (mode_grouped_k(mode) || mode == MODE_FP8_TENSOR) ? 3 : 2;
    const bool persist_wins = t256 >= 240 || r128 >= rounds128 * r256;
    if (persist_wins) {
      r.path = PATH_PIPE;
      r.variant = pipe_forced >= 0 ? pipe_forced : (t256 >= 240 ? 0 : one_round);
      // Rows of whole 128 bytes whose scale rows are no whole quads: the tiles
      // above serve them too, and win on short K (the scales' copy, and up to 24
      // us for a last column of tiles that is nearly full; block 6569x1520x768
      // 43.5 us / 16.9, MXFP4 1319x8624x768 33.4 / 15.4; whole columns: block
      // 4128x7680x768 36.1 / 38.1, MXFP4 7231x4608x1280 45.7 / 50.9).
      const bool short_k = !f32 && !rag && !persist_whole(mode, K, Kb, sc16) &&
                           Kb < (mode == MODE_FP8_BLOCK ? 1024 + 6144 * last_tile(256)
                                                        : 512 + 2560 * last_tile(256));
      if (persist_ok && !short_k) r.path = PATH_PERSIST;
    } else if (M > 64 && N > 64 && t128 >= 40) {
      r.path = PATH_PIPE;
      r.variant = one_round;
    }
  }
  if (narrow && persist_ok && (r.path == PATH_PERSIST || narrow_wins)) {
    r.path = PATH_PERSIST;
    r.narrow = true;
  }
  r.pad_scales = (r.path == PATH_PERSIST && pad) || (r.path == PATH_PIPE && fp4 && rag);
  return r;
}

// Predicted times in us of the pipelined tiles (one stage of 128 bytes by mode
// and form; `fill` workgroups per CU, two of variant 1 share one) and of the
// register-staged tiles split over K (64-byte steps of the longest split, the
// partial sums written and read, the operands).  Fitted to 10800 sampled sizes,
// M to 8192 and K to 32768: 4 in 5 within 15%.
static float pipe_estimate(int mode, const Route &r, int M, int N, int Kb) {
  static constexpr float deep64[6][2] = {   // whole, ragged
      {.23f, .36f}, {.42f, .49f}, {.52f, .65f}, {0, 0}, {.25f, .40f}, {.43f, .55f}};
  static constexpr float deep128[6][2] = {
      {.40f, .50f}, {.66f, .80f}, {.85f, .98f}, {0, 0}, {.43f, .55f}, {.73f, .86f}};
  static constexpr float two[6][2] = {
      {.37f, .46f}, {.67f, .82f}, {.70f, .88f}, {3.9f, 4.0f}, {.42f, .57f}, {.73f, .90f}};
  const int rag = Kb % (prefetches(mode) && r.variant != 1 ? 256 : 128) != 0, bm = r.variant == 6 ? 64 : 128;
  const int64_t tiles = (int64_t)((M + bm - 1) / bm) * ((N + 127) / 128), cu = device_cu_count();
  const float fill = (float)tiles / cu, stages = (float)((Kb + 127) / 128), pad = r.pad_scales ? 4.5f : 0.f;
  if (r.variant == 6) return 3.3f + .7f * rag + pad + stages * deep64[mode][rag] * (.8f + .2f * fill);
  if (r.variant == 7) return 4.f + pad + stages * deep128[mode][rag] * (.75f + .25f * fill);
  if (r.variant != 1) return 0;
  const float again = (float)((tiles + cu - 1) / cu - 1);
  return 3.2f + pad + stages * two[mode][rag] * (1.f + .4f * fill + .6f * again) + 2.f * again;
}

static float split_estimate(int mode, const Plan &pl, int M, int N, int Kb) {
  static constexpr float step[6] = {.5f, .63f, .80f, 2.6f, .5f, .65f};
  static constexpr float step256[6] = {1.4f, 6.2f, 6.6f, 10.9f, 1.4f, 6.2f};
  const float steps = (float)Kb / pl.ksplit / 64, mb = (float)(M + N) * Kb * 1e-6f;
  const float part = (float)pl.ksplit * M * (float)N * 4e-6f;
  if (pl.variant == 0) {   // 256x256: few spills per-tensor and bf16, many in the others
    if (mode != MODE_FP8_TENSOR && mode != MODE_BF16) return steps * step256[mode] + 1.4f * part + 1.2f * mb;
    if (Kb % 128 == 0) return 13.f + steps * (mode == MODE_BF16 ? .95f : .68f) + .35f * part;
    return 8.5f + steps * step256[mode] + .35f * part;
  }
  static constexpr float fixed[] = {0, 7.3f, 5.2f, 3.9f}, per_part[] = {0, .5f, .65f, .5f},
                         per_mb[] = {0, .1f, .03f, .12f};
  return fixed[pl.variant] + steps * step[mode] + per_part[pl.variant] * part + per_mb[pl.variant] * mb;
}

// 0: not predicted
static float route_estimate(int mode, const Route &r, int M, int N, int K, int Kb, bool sc16) {
  if (r.path == PATH_STREAM) return stream_estimate(mode, M, N, K, Kb, sc16);
  if (r.path == PATH_PIPE) return pipe_estimate(mode, r, M, N, Kb);
  if (r.path == PATH_TILED && r.tiled.ksplit > 1) return split_estimate(mode, r.tiled, M, N, Kb);
  return 0;
}

// A shape takes the ragged forms and the one-round tiles unless the kernel that
// serves it without them is predicted faster.  Those walk K in one chain per
// workgroup: where few workgroups and a long K leave CUs idle, the split-K tiles
// (or, NVFP4 and rows of an odd number of chunks, the other of the two) win:
// bf16 129x3840x10528 streamed 80 us, split 41; per-tensor 2253x128x29776 on
// 64x128 tiles 102, split 36; NVFP4 218x13312x256 streamed 45, 128x128 tiles 8.
// Over 10800 sampled sizes the choice by size alone made 4% slower than the
// kernels served before it, by up to 5.9 times; this leaves 1%, by 1.7 at most.
// `ws`: bytes for the split's partial sums (their room is in the contract).
static Route route_for(int mode, int M, int N, int K, int Kb, bool sc4, bool sc16, bool padded, bool f32,
                       size_t ws) {
  const Route r = pick_route(mode, M, N, K, Kb, sc4, sc16, padded, f32, true);
  if (r.path != PATH_STREAM && r.path != PATH_PIPE) return r;
  // The second pick and the estimates cost host time (0.13 us of a 5.4 us call of
  // 3 rows): not for up to 16 rows, which stream at least as fast as either of the
  // others (groupwise 5x45352x1184 14.0 us, split 16.0; MXFP4 3x36464x256 10.1 /
  // 10.1 on tiles), nor for a whole K, which streams either way.
  if (r.path == PATH_STREAM && (M <= 16 || stream_whole(mode, K, Kb, sc16))) return r;
  const Route w = pick_route(mode, M, N, K, Kb, sc4, sc16, padded, f32, false);
  if (r.path == w.path) return r;
  if (w.path == PATH_TILED && (w.tiled.ksplit < 2 || ws / sizeof(float) / w.tiled.ksplit < (size_t)splitk_slice(M, N)))
    return r;
  const float tr = route_estimate(mode, r, M, N, K, Kb, sc16), tw = route_estimate(mode, w, M, N, K, Kb, sc16);
  return tr > 0 && tw > 0 && tr > tw ? w : r;
}

// C += result streams where the router picks a skinny kernel, and for short K (a
// LoRA adapter add: W is then small enough to stream once per activation block).
// K of no whole chunk streams in the TAIL form, one chunk that three of a
// workgroup's four waves wait for: past about 15K columns over the 64-row blocks
// the pipelined tiles win where the router picks those (rank 8 to 32, the whole
// layer, us streamed / tiles: 541x1024x1024 18.1 / 24.2, 300x2992x2624 37.4 /
// 40.3, 276x3216x576 28.0 / 25.8, 773x3496x896 41.4 / 30.6).
static bool acc_streams(int mode, int path, int M, int N, int K, int Kb, bool sc4, bool sc16) {
  if (!stream_enabled() || !stream_supported(mode, M, N, K, Kb, sc4)) return false;
  if (path == PATH_STREAM || path == PATH_DECODE) return true;
  return K <= kAccShortK && (path != PATH_PIPE || stream_whole(mode, K, Kb, sc16) ||
                             (int64_t)((M + 63) / 64) * N <= 15 * 1024);
}

// C += result (fp32 out, one writer per element): the streaming kernel, the
// pipelined tiles where the router picks those (not block-scaled), else the
// register-staged kernels.
static void accumulate_route(int mode, Route *r, int M, int N, int K, int Kb, bool sc4, bool sc16) {
  if (acc_streams(mode, r->path, M, N, K, Kb, sc4, sc16)) r->path = PATH_STREAM;
  else if (r->path != PATH_PIPE || mode_grouped_k(mode)) r->path = PATH_TILED;
}

bool gemm_routes_to_stream(int mode, int64_t M, int64_t N, int64_t K, bool or_pipe, bool accumulate) {
  const int Kb = (mode == MODE_MXFP4 || mode == MODE_NVFP4) ? (int)(K / 2)
                                                            : (mode == MODE_BF16 ? (int)(2 * K) : (int)K);
  int path = route_for(mode, (int)M, (int)N, (int)K, Kb, true, true, true, true, SIZE_MAX).path;
  if (accumulate && acc_streams(mode, path, (int)M, (int)N, (int)K, Kb, true, true))
    path = PATH_STREAM;   // as launch_gemm routes C += result
  return path == PATH_STREAM || (or_pipe && path == PATH_PIPE && (!accumulate || !mode_grouped_k(mode)));
}

size_t gemm_workspace_required(int mode, int64_t M, int64_t N, int64_t K, bool accumulate) {
  const int Kb = (mode == MODE_MXFP4 || mode == MODE_NVFP4) ? (int)(K / 2)
                                                            : (mode == MODE_BF16 ? (int)(2 * K) : (int)K);
  Route r = pick_route(mode, (int)M, (int)N, (int)K, Kb, true, true, false, true, false);
  if (accumulate) r.path = PATH_TILED;
  return (r.path == PATH_TILED && r.tiled.ksplit > 1)
             ? (size_t)r.tiled.ksplit * (size_t)splitk_slice(M, N) * sizeof(float)
             : 0;
}

size_t gemm_workspace_bytes(int mode, int64_t M, int64_t N, int64_t K, bool accumulate) {
  const size_t need = gemm_workspace_required(mode, M, N, K, accumulate);
  if (accumulate || (mode != MODE_MXFP4 && mode != MODE_NVFP4) || persist_whole(mode, (int)K, (int)(K / 2), true))
    return need;                     // no scale rows to pad
  const Route r = route_for(mode, (int)M, (int)N, (int)K, (int)(K / 2), true, true, true, true, SIZE_MAX);
  return r.pad_scales ? std::max(need, (size_t)(M + N) * (size_t)padded_pitch(mode, (int)K)) : need;
}

// The columns [n1, N) of a problem (n1 a multiple of 256).
static GemmArgs columns_from(int mode, GemmArgs p, int n1) {
  p.b += (int64_t)n1 * p.Kb;
  p.c = static_cast<uint8_t *>(p.c) + (int64_t)n1 * (p.out_f32 ? 4 : 2);
  if (p.sb) {
    const int64_t off = mode == MODE_FP8_BLOCK ? (int64_t)(n1 / 128) * ((p.K + 127) / 128) * 4
                                               : (int64_t)n1 * scale_row_len(mode, p.K);
    p.sb = static_cast<const uint8_t *>(p.sb) + off;
  }
  p.N -= n1;
  p.ws = nullptr;
  p.ws_bytes = 0;
  return p;
}

// Columns to take off a persistent launch so that its 256x256 tiles fill whole
// rounds, the rest going to a second launch of smaller tiles: a last round of
// a few tiles costs most of a full one (K=4096: 64 tiles 0.73 of it), the same
// columns in 128x128 tiles 0.41 at most.  0: leave it whole.  Taken where the
// columns are at most a quarter of the CUs' worth of tiles, which one round of
// 128x128 tiles (or the streaming kernel) holds.  us before -> after,
// per-tensor / block / MXFP4 / NVFP4 / bf16: 2304x7680x4096 (270 tiles) 90 ->
// 75, 106 -> 93, 63 -> 58, 190 -> 178, 177 -> 145; 4300x4300x4096 (289 tiles)
// 141 -> 116, 158 -> 132, 113 -> 101, 241 -> 218, 230 -> 185.  Not under
// DSL_GEMM_PIPE, which names the tiles or forbids them.
static int strip_columns(const GemmArgs &p) {
  const int cu = device_cu_count();
  const int nbm = (p.M + 255) / 256, nbn = (p.N + 255) / 256;
  const int64_t tiles = (int64_t)nbm * nbn, full = tiles / cu * cu;
  if (p.accumulate || pipe_switch() != -1 || full == 0 || tiles == full || nbm > cu / 4) return 0;
  const int keep = (int)(full / nbm);                // whole columns of tiles in whole rounds
  if ((int64_t)nbm * (nbn - keep) > cu / 4 || keep < 1) return 0;
  return p.N - keep * 256;
}

// Pipelined tiles for those columns: 64x128 or deep 128x128 ones where one round
// holds them, as pick_route has it.
static int pipe_variant(int mode, int M, int N, int Kb) {
  const int64_t cu = device_cu_count();
  if (mode == MODE_NVFP4) return 1;
  if ((int64_t)((M + 63) / 64) * ((N + 127) / 128) <= cu) return 6;
  return (int64_t)((M + 127) / 128) * ((N + 127) / 128) <= cu && deep_pays(mode, Kb) ? 7 : 1;
}

void describe_gemm(int mode, int64_t M, int64_t N, int64_t K, bool f32, bool accumulate, char *buf,
                   size_t len) {
  const int Kb = (mode == MODE_MXFP4 || mode == MODE_NVFP4) ? (int)(K / 2)
                                                            : (mode == MODE_BF16 ? (int)(2 * K) : (int)K);
  auto name = [&](const Route &r, int m, int n, char *to, size_t room) {
    static const char *const tiles[] = {"256x256", "128x128", "", "", "", "", "64x128 deep", "128x128 deep"};
    int tma = 0, tn = 0;
    if (r.path == PATH_STREAM) {
      const bool tail = stream_plan(mode, m, n, (int)K, Kb, true, &tma, &tn);
      snprintf(to, room, "stream%s %dx%d", tail ? " tail" : "", 16 * tma, 16 * tn);
    } else if (r.path == PATH_PIPE) {
      snprintf(to, room, "pipe %s", r.variant >= 0 && r.variant < 8 ? tiles[r.variant] : "forced");
    } else if (r.path == PATH_PERSIST) {
      snprintf(to, room, "persist 256x%d", r.narrow ? 128 : 256);
    } else if (r.path == PATH_TILED) {
      snprintf(to, room, "split %dx%d/%d", r.tiled.bm, r.tiled.bn, r.tiled.ksplit);
    } else {
      snprintf(to, room, "decode");
    }
  };
  Route r = route_for(mode, (int)M, (int)N, (int)K, Kb, true, true, true, f32, SIZE_MAX);
  if (accumulate && f32) accumulate_route(mode, &r, (int)M, (int)N, (int)K, Kb, true, true);
  name(r, (int)M, (int)N, buf, len);
  GemmArgs p{};
  p.M = (int)M;
  p.N = (int)N;
  p.accumulate = accumulate;
  const int strip = r.path != PATH_PERSIST || r.narrow || r.pad_scales ? 0 : strip_columns(p);
  if (strip == 0) return;
  Route rest = route_for(mode, (int)M, strip, (int)K, Kb, true, true, false, f32, 0);
  if (rest.path != PATH_STREAM) {
    rest.path = PATH_PIPE;
    rest.variant = pipe_variant(mode, (int)M, strip, Kb);
  }
  const size_t used = strlen(buf);
  snprintf(buf + used, len - used, " + ");
  name(rest, (int)M, strip, buf + strlen(buf), len - strlen(buf));
}

hipError_t launch_gemm(int mode, GemmArgs p, hipStream_t st) {
  const uintptr_t sc = reinterpret_cast<uintptr_t>(p.sa) | reinterpret_cast<uintptr_t>(p.sb);
  if (p.Kb2 > 0) {   // a second K segment: the persistent BF16 kernel only
    if (mode != MODE_BF16 || p.accumulate || p.lora_scales || p.Kb % 128 != 0 ||
        p.Kb2 % 128 != 0 || !persist_supported(mode, p.M, p.N, p.K, p.Kb + p.Kb2, true))
      return hipErrorInvalidValue;
    // W2 read from a narrower B whose pairs repeat: whole pairs, a power of
    // two of them per row
    if (p.rep2 != 0 && ((p.rep2 & (p.rep2 - 1)) != 0 || p.ldb2 % 16 != 0 ||
                        p.ldb2 < p.rep2 * 128 || p.Kb2 % (p.rep2 * 128) != 0))
      return hipErrorInvalidValue;
    return launch_gemm_persist(mode, p, st);
  }
  if (p.rep2 != 0 || p.ldb2 != 0) return hipErrorInvalidValue;
  // scale rows are padded only into a workspace that holds them
  const bool padded = (mode == MODE_MXFP4 || mode == MODE_NVFP4) && p.ws &&
                      (reinterpret_cast<uintptr_t>(p.ws) & 15) == 0 &&
                      p.ws_bytes >= (size_t)((int64_t)p.M + p.N) * (size_t)padded_pitch(mode, p.K);
  Route r = route_for(mode, p.M, p.N, p.K, p.Kb, (sc & 3) == 0, (sc & 15) == 0, padded, p.out_f32 != 0,
                      p.ws ? p.ws_bytes : 0);
  if (p.lora_scales) {   // the LoRA epilogue: the streaming kernel only
    if (mode != MODE_BF16 || !stream_supported(mode, p.M, p.N, p.K, p.Kb, true) || p.accumulate)
      return hipErrorInvalidValue;
    return launch_gemm_stream(mode, p, st);
  }
  if (p.accumulate) {
    if (p.out_f32) accumulate_route(mode, &r, p.M, p.N, p.K, p.Kb, (sc & 3) == 0, (sc & 15) == 0);
    else r.path = PATH_TILED;
  }
  p.ksplit = 1;
  if (r.path == PATH_DECODE) return launch_gemm_decode(mode, p, st);
  if (r.path == PATH_STREAM) return launch_gemm_stream(mode, p, st);
  if (r.path == PATH_PERSIST || r.path == PATH_PIPE) {
    if (r.pad_scales) {
      const int pitch = padded_pitch(mode, p.K);
      const int64_t words = ((int64_t)p.M + p.N) * (pitch / 4);
      const unsigned g = (unsigned)std::min<int64_t>((words + 255) / 256, 4096);
      uint8_t *out = reinterpret_cast<uint8_t *>(p.ws);
      pad_scales_kernel<<<g, 256, 0, st>>>(static_cast<const uint8_t *>(p.sa), p.M,
                                           static_cast<const uint8_t *>(p.sb), p.N,
                                           scale_row_len(mode, p.K), pitch,
                                           mode == MODE_MXFP4 ? 0x7fu : 0u,
                                           reinterpret_cast<uint32_t *>(out));
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      p.sa = out;
      p.sb = out + (int64_t)p.M * pitch;
      p.sld = pitch;
    }
    if (r.path == PATH_PIPE) return launch_gemm_pipe(mode, p, r.variant, st);
    const int strip = r.narrow || r.pad_scales ? 0 : strip_columns(p);
    if (strip > 0) {
      GemmArgs main = p;
      main.N = p.N - strip;
      const hipError_t e = launch_gemm_persist(mode, main, st, false);
      if (e != hipSuccess) return e;
      const GemmArgs rest = columns_from(mode, p, main.N);
      return route_for(mode, rest.M, rest.N, rest.K, rest.Kb, (sc & 3) == 0, (sc & 15) == 0, false, p.out_f32 != 0, 0).path ==
                     PATH_STREAM
                 ? launch_gemm_stream(mode, rest, st)
                 : launch_gemm_pipe(mode, rest, pipe_variant(mode, rest.M, rest.N, rest.Kb), st);
    }
    return launch_gemm_persist(mode, p, st, r.narrow);
  }
  const Plan pl = r.tiled;
  // split-K into as many [M][N] fp32 slices as the workspace holds (at most
  // the plan's split count; fewer than two: one pass over K)
  const size_t slice_bytes = (size_t)splitk_slice(p.M, p.N) * sizeof(float);
  const size_t fit = p.ws ? p.ws_bytes / slice_bytes : 0;
  p.ksplit = fit >= 2 ? (int)std::min<size_t>((size_t)pl.ksplit, fit) : 1;
  switch (mode) {
    case MODE_FP8_TENSOR: launch_mode<MODE_FP8_TENSOR>(pl, p, st); break;
    case MODE_FP8_BLOCK: launch_mode<MODE_FP8_BLOCK>(pl, p, st); break;
    case MODE_FP8_GCOL: launch_mode<MODE_FP8_GCOL>(pl, p, st); break;
    case MODE_MXFP4: launch_mode<MODE_MXFP4>(pl, p, st); break;
    case MODE_NVFP4: launch_mode<MODE_NVFP4>(pl, p, st); break;
    case MODE_BF16: launch_mode<MODE_BF16>(pl, p, st); break;
    default: return hipErrorInvalidValue;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (p.ksplit > 1) {
    const int esz = p.out_f32 ? 4 : 2;
    const int vec = p.N % 4 == 0 && p.ldc % 4 == 0 &&
                    (reinterpret_cast<uintptr_t>(p.c) % (4 * esz)) == 0;
    const dim3 fgrid((unsigned)((p.N + 1023) / 1024), (unsigned)std::min(p.M, 4096));
    splitk_finalize_kernel<<<fgrid, 256, 0, st>>>(p.ws, p.ksplit, p.c, p.M, p.N, p.ldc,
                                                  p.out_f32, p.accumulate, vec);
    e = hipGetLastError();
  }
  return e;
}

}  // namespace dsl
