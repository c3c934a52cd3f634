// Gather convolution over 64-row tiles whose offsets can be split over groups of waves
// (gfx950): fp32 sets of any size, each fp32 operand as the sum of three bf16 values, and
// 16-bit sets of few tiles.
//
//   out[o] = act(bias + sum_k in[gidx[o, k]] . W[:, k, :]^T) (+ residual[o])
//
// fp32: 2^16 x = x1 + x2 + x3 with x1 = bf16(2^16 x), x2 = bf16(2^16 x - x1) and x3 the rest,
// each rounded to nearest. They hold every bit of an fp32 value: 24, and with the scale bf16's
// smallest step, 2^-133, is the last bit of a subnormal x (without it values below 2^-110 lost
// bits: at 2^-120 the result had an error of 3.5e-5). Of the nine products the kernel keeps
// w1 x1, w1 x2, w2 x1, w1 x3, w3 x1 and w2 x2; the other three are together at most about
// 2^-24 of the product. Products of two bf16 values are exact in fp32 and the MFMA adds them
// to fp32 accumulators, as the fp32 MFMA does: fp32 accuracy at six 32x32x16 bf16 MFMAs in the
// place of eight 32x32x2 fp32 ones, 192 cycles against 512. Relative error against 64-bit
// sums, normal random values: C128, 327,581 voxels 2.3e-7 (fp32 MFMA 6.8e-7), C64, 45,128
// voxels 1.6e-7 (5.1e-7), C256, 100,000 voxels 3.4e-7 (9.9e-7): one MFMA sums 16 products, and
// the products of each size (w1 x1, 2^-8 and 2^-16 of it) have a sum of their own (in one sum
// for all, without the scale, the three errors were 5.9e-7, 4.3e-7, 8.6e-7 and the times about
// 3 % less). What bounds it: the bf16 matrix rate, at C64 as much the vector operations of the
// split.
//
// Infinities, NaN, values from 2^112 and sums from 2^96 on, whose scaled forms overflow,
// leave a sum that is not finite (a part x2 or x3 of an infinity is NaN). A workgroup with
// such outputs walks its stages once more with the fp32 MFMA, which takes the weights from
// their parts, and replaces those outputs; a row sums the offsets that it has (C128 on
// 100,000 voxels, every row NaN: 1.15 ms, fp32 MFMA 0.67, the plain sum of one output after
// another 40 ms).
//
// Reference semantics: subm_conv (src/hi3d_mac/torch_backend/sparse_conv.py:152-195).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "conv_group.h"
#include "conv_tile.h"
#include "rownorm.h"

namespace hi3d {
namespace {

constexpr int kGroupMaxKvol = 27;
constexpr int kGroupMaxRowBytes = 2048;
constexpr int kSplitMaxCin = kGroupMaxRowBytes / 4;
constexpr int kGroupThreads = 256;
// Tables of few offsets (the strided pair, the child projection) are bound by their rows'
// traffic until the products per row are many: the fp32 MFMA kernels ran the 64 -> 64
// pair on 100k voxels in 52 us and the 128-channel child step on 200k parents in 897 us
// against 56 and 934 us here; the 128 <-> 256 pair on 400k voxels took 653 us there and
// 471 us here, the 256-channel child step 1790 and 1699 us.
constexpr int kFewOffsets = 8;
constexpr int64_t kFewOffsetsWork = 128 * 256;

constexpr float kPartScale = 65536.0f;
constexpr float kPartMax = 0x1p111f;  // no scaled value below it rounds to infinity

// row that absent neighbours read
__device__ __attribute__((aligned(16))) const uint32_t g_group_zero_row[kGroupMaxRowBytes / 4] = {};

// The three bf16 parts of 8 fp32 values.
__device__ __forceinline__ void split8(const f32x4 lo, const f32x4 hi, bf16x8 (&p)[3]) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = kPartScale * (j < 2 ? lo[2 * j] : hi[2 * j - 4]), b = kPartScale * (j < 2 ? lo[2 * j + 1] : hi[2 * j - 3]);
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const bf16x2 v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
      uint32_t u = __builtin_bit_cast(uint32_t, v);
      asm("" : "+v"(u));  // one packed conversion, not another of each value alone
      p[t][2 * j] = __builtin_bit_cast(bf16x2, u)[0];
      p[t][2 * j + 1] = __builtin_bit_cast(bf16x2, u)[1];
      if (t < 2) {
        a -= __builtin_bit_cast(float, u << 16);
        b -= __builtin_bit_cast(float, u & 0xffff0000u);
      }
    }
  }
}

// Value e of 8 from their parts as split_weight_kernel stores them.
__device__ __forceinline__ float joined(const u32x4 (&p)[3], int e) {
  uint32_t u[3];  // the parts as fp32 bits
#pragma unroll
  for (int i = 0; i < 3; ++i) u[i] = e % 2 ? p[i][e / 2] & 0xffff0000u : p[i][e / 2] << 16;
  const float first = __builtin_bit_cast(float, u[0]);
  const float sum = first + (__builtin_bit_cast(float, u[1]) + __builtin_bit_cast(float, u[2]));  // exact
  return first == first ? sum * (1.0f / kPartScale) : __builtin_bit_cast(float, u[1] | u[2] >> 16);
}

// One thread per 16-byte piece of a part: channel 32 nb + lane % 32, inputs
// 16 ks + 8 (lane / 32) .. + 7, all three parts. Channels past cout are zero. vec: the
// inputs of a channel lie next to each other and every 8 of them are 16-byte aligned.
__global__ __launch_bounds__(256) void split_weight_kernel(const float* __restrict__ w, int64_t wn, int64_t wk,
                                                           int64_t wc, bool vec, int cout, int cin, int col_blocks,
                                                           int64_t total, char* __restrict__ packed) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (t >= total) return;
  const int lane = static_cast<int>(t & 63);
  const int64_t block = t >> 6;  // (k, ks, nb)
  const int nb = static_cast<int>(block % col_blocks);
  const int64_t kks = block / col_blocks;
  const int ksteps = cin / 16;
  const int ks = static_cast<int>(kks % ksteps);
  const int64_t k = kks / ksteps;
  const int n = nb * 32 + (lane & 31);
  f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
  if (n < cout) {
    const float* src = w + n * wn + k * wk + (ks * 16 + 8 * (lane >> 5)) * wc;
    if (vec) {
      lo = *reinterpret_cast<const f32x4*>(src);
      hi = *reinterpret_cast<const f32x4*>(src + 4);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo[i] = src[i * wc];
        hi[i] = src[(i + 4) * wc];
      }
    }
  }
  bf16x8 p[3];
  split8(lo, hi, p);
  // a weight whose scaled form overflows: NaN and the two halves of its bits
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float v = e < 4 ? lo[e] : hi[e - 4];
    if (fabsf(v) < kPartMax) continue;
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    p[0][e] = __builtin_bit_cast(__bf16, static_cast<uint16_t>(0x7fc0));
    p[1][e] = __builtin_bit_cast(__bf16, static_cast<uint16_t>(u >> 16));
    p[2][e] = __builtin_bit_cast(__bf16, static_cast<uint16_t>(u));
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(packed + block * 3072 + i * 1024 + lane * 16) = p[i];
}

// A workgroup owns BM = 64 plan rows and BN channels; its 4 G waves form G groups, each a
// 2 x 2 grid of waves over the whole tile that takes every G-th offset, so that a set of
// few tiles spreads its chain of offsets over a CU's four SIMDs' worth of waves. The
// groups' sums are added in order in the epilogue.
//  * Stages (per group): (present offset, 64 KS bytes of the input rows): BM gathered rows
//    and the weights (fp32: BN / 32 x KS x 3 KB of parts, laid out as the fragments are
//    read; 16-bit: BN rows), by direct-to-LDS 16-byte loads NS - 1 stages ahead into a
//    ring of NS slots, one barrier a stage. The next loads go out first, then a stage's
//    fragments are all read before its first product (fp32 C256 on 100,000 voxels 1.23 ms,
//    with the loads after the fragments 1.29; C128 on 3,000 voxels 51 against 53 us).
//  * fp32 rows stay fp32 in LDS and each wave splits its fragments in registers (13 vector
//    ops per pair of values).
//  * The gather indices of all offsets reach LDS once, and with them the offsets that each
//    32-row block has; a wave skips its block's products of the others.
//  * The MFMAs take the weights as their first operand: a lane ends with four consecutive
//    channels of one row. The output leaves through LDS as whole row pieces.
template <typename T, int BN, int KS, int NS, int G, bool kLN = false>
__global__ __launch_bounds__(kGroupThreads * G, 2) void conv_group_kernel(GroupConv a) {
  constexpr bool kSplit = sizeof(T) == 4;
  constexpr int BM = 64, KV = kGroupMaxKvol, THREADS = kGroupThreads * G, NWG = kGroupThreads / 64, NW = NWG * G;
  constexpr int WN = BN / 2, NB = WN / 32;
  constexpr int ES = static_cast<int>(sizeof(T));
  constexpr int ROWB = 64 * KS, LPR = 4 * KS;  // staged row: bytes, 16-byte chunks
  constexpr int A_BYTES = BM * ROWB, B_BYTES = kSplit ? (BN / 32) * KS * 3072 : BN * ROWB, STAGE = A_BYTES + B_BYTES;
  constexpr int LA = A_BYTES / (1024 * NWG), BKB = B_BYTES / 1024;
  constexpr int LB = (BKB + NWG - 1) / NWG, LBMIN = BKB / NWG;  // loads of the waves below BKB % NWG, of the others
  static_assert(LA * 1024 * NWG == A_BYTES && (KS == 1 || KS == 2) && NS >= 2 && NS <= 4, "stage shape");
  static_assert(kTileRows % BM == 0, "a workgroup's rows lie in one plan tile");
  constexpr int RING = G * NS * STAGE;
  constexpr int SROW = BN * 4;  // staged sums: bytes of a row
  static_assert(G * BM * SROW <= RING, "staged sums");
  __shared__ __attribute__((aligned(16))) char smem[RING + (KV + 1) * BM * 4 + NW * 12];
  int32_t* const gl = reinterpret_cast<int32_t*>(smem + RING);
  int32_t* const srow = gl + KV * BM;
  uint32_t* const smask = reinterpret_cast<uint32_t*>(srow + BM);  // [wave][32-row block]
  uint32_t* const sbad = smask + 2 * NW;  // [wave]: sums that are not finite

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave_all / NWG, wave = wave_all % NWG;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t item = xcd_remap(blockIdx.x, static_cast<int64_t>(gridDim.x));
  const int64_t tile = item / a.ny;
  const int ct = static_cast<int>(item - tile * a.ny);
  const int n0 = ct * BN;
  const int kvol = a.kvol;
  const uint64_t n_in = static_cast<uint64_t>(a.n_in);
  const int64_t p0 = tile * BM;  // < ntiles * kTileRows
  const int32_t* const gsrc = a.gidx + (p0 / kTileRows) * kvol * kTileRows + (p0 % kTileRows);

  // gather indices of all offsets (-1: absent), this wave's offsets wave_all, + NW, ...
  {
    constexpr int PER = (KV + NW - 1) / NW;
    int32_t g[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int k = wave_all + NW * j;
      g[j] = gsrc[(k < kvol ? k : 0) * kTileRows + lane];
    }
    if (tid < BM) srow[tid] = a.rows[p0 + tid];
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int k = wave_all + NW * j;
      if (k >= kvol) continue;
      const bool ok = static_cast<uint64_t>(static_cast<uint32_t>(g[j])) < n_in;
      const uint64_t b = __builtin_amdgcn_ballot_w64(ok);
      if (static_cast<uint32_t>(b) != 0) lo |= 1u << k;
      if (static_cast<uint32_t>(b >> 32) != 0) hi |= 1u << k;
      gl[k * BM + lane] = ok ? g[j] : -1;
    }
    if (lane == 0) {
      smask[wave_all * 2] = lo;
      smask[wave_all * 2 + 1] = hi;
    }
  }
  __syncthreads();
  uint32_t mask = 0, bmask = 0;  // offsets of the tile, of this wave's row block
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    mask |= smask[w * 2] | smask[w * 2 + 1];
    bmask |= smask[w * 2 + wm];
  }
  mask = __builtin_amdgcn_readfirstlane(mask);
  bmask = __builtin_amdgcn_readfirstlane(bmask);

  // this group's offsets k = group mod G, whatever the tile: a row's sum does not depend on
  // the rows it shares a tile with (absent neighbours add zeros)
  constexpr uint32_t EVERY = G == 4 ? 0x11111111u : 0xffffffffu;
  static_assert(G == 1 || G == 4, "offset groups");
  const uint32_t mine = mask & (EVERY << group);
  int most = 0;
#pragma unroll
  for (int g = 0; g < G; ++g) most = max(most, __popc(mask & (EVERY << g)));
  const int row_bytes = a.cin * ES;
  const int ksteps = row_bytes / ROWB;  // stages per offset
  const int S = __popc(mine) * ksteps;
  const int SMAX = most * ksteps;  // barriers are the workgroup's
  char* const ring = smem + group * (NS * STAGE);

  // load u of this wave fills 1 KB of the stage's rows: 16 / KS rows, 4 KS lanes a row
  auto row_off = [](int row, int chunk) {
    return KS == 1 ? row * 64 + ((chunk ^ ((row >> 2) & 3)) << 4) : lds_offset(row, chunk);
  };
  auto load_row = [&](int u) { return (wave + NWG * u) * (64 / LPR) + lane / LPR; };
  auto load_byte = [&](int u) {  // of the row, at this lane's place
    const int r = load_row(u), c = lane % LPR;
    return (KS == 1 ? (c ^ ((r >> 2) & 3)) : (c ^ ((r >> 1) & 7))) * 16;
  };
  uint32_t rest = 0;
  int lks = 0, lslot = 0;
  const char* src[LA];
  const char* wsrc = nullptr;
  const int wstep = kSplit ? KS * a.col_blocks * 3072 : ROWB;  // to the weights of the next stage
  int64_t woff[LB];  // KB wave + 4 u of a stage's weights
#pragma unroll
  for (int u = 0; u < LB; ++u) {
    if constexpr (kSplit) {
      const int i = wave + NWG * u, s = i / (3 * (BN / 32));
      woff[u] = s * (a.col_blocks * 3072) + (i - s * (3 * (BN / 32))) * 1024 + lane * 16;
    } else {
      const int n = n0 + load_row(u);  // channels past cout re-read the last (never stored)
      woff[u] = static_cast<int64_t>(n < a.cout ? n : a.cout - 1) * kvol * row_bytes + load_byte(u);
    }
  }
  auto issue = [&]() __attribute__((always_inline)) {
    if (lks == 0) {
      const int k = rest ? __builtin_ctz(rest) : 0;
      rest &= rest - 1u;
#pragma unroll
      for (int u = 0; u < LA; ++u) {
        const int32_t g = gl[k * BM + load_row(u)];
        uint64_t pin = reinterpret_cast<uint64_t>(a.in) + static_cast<uint64_t>(static_cast<int64_t>(g) * row_bytes);
        asm volatile("" : "+v"(pin));  // a select of addresses, not a branch
        src[u] = (g >= 0 ? reinterpret_cast<const char*>(pin) : reinterpret_cast<const char*>(g_group_zero_row)) + load_byte(u);
      }
      wsrc = kSplit ? a.packed + (static_cast<int64_t>(k) * ksteps * KS * a.col_blocks + ct * (BN / 32)) * 3072
                    : a.weight + static_cast<int64_t>(k) * row_bytes;
    }
    char* st = ring + lslot * STAGE;
#pragma unroll
    for (int u = 0; u < LA; ++u) lds_dma16(src[u] + lks * ROWB, st + (wave + NWG * u) * 1024);
#pragma unroll
    for (int u = 0; u < LB; ++u)
      if (u < LBMIN || wave < BKB % NWG) lds_dma16(wsrc + woff[u], st + A_BYTES + (wave + NWG * u) * 1024);
    wsrc += wstep;
    lslot = lslot == NS - 1 ? 0 : lslot + 1;
    if (++lks == ksteps) lks = 0;
  };

  constexpr int NA = kSplit ? 3 : 1;  // fp32: sums of the products by their size
  f32x16 acc[NA][NB];

  // a stage's fragments: rows x, weights w (fp32: KS steps of 16 inputs, a step's row
  // fragment as two 16-byte chunks and its weights as three parts; 16-bit: 2 KS groups)
  constexpr int XF = 2 * KS, WF = kSplit ? 3 * KS : 2 * KS;
  u32x4 x[XF], w[NB][WF];
  auto frags = [&](int slot) __attribute__((always_inline)) {
    const char* st = ring + slot * STAGE;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int f = 0; f < WF; ++f) {
        if constexpr (kSplit)
          w[nb][f] = *reinterpret_cast<const u32x4*>(
              st + A_BYTES + (((f / 3) * (BN / 32) + wn * NB + nb) * 3 + f % 3) * 1024 + lane * 16);
        else
          w[nb][f] = *reinterpret_cast<const u32x4*>(
              st + A_BYTES + row_off((wn * NB + nb) * 32 + (lane & 31), 2 * f + (lane >> 5)));
      }
#pragma unroll
    for (int f = 0; f < XF; ++f) {
      const int c = kSplit ? 4 * (f / 2) + 2 * (lane >> 5) + f % 2 : 2 * f + (lane >> 5);
      x[f] = *reinterpret_cast<const u32x4*>(st + row_off(wm * 32 + (lane & 31), c));
    }
  };
  auto products = [&](auto plain) __attribute__((always_inline)) {
    if constexpr (plain) {
      // input j of 16 and input 8 + j in one MFMA
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float xj = __builtin_bit_cast(f32x4, x[2 * s + j / 4])[j % 4];
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const u32x4 p[3] = {w[nb][3 * s], w[nb][3 * s + 1], w[nb][3 * s + 2]};
            acc[1][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(joined(p, j), xj, acc[1][nb], 0, 0, 0);
          }
        }
    } else if constexpr (kSplit) {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8 xp[3];
        split8(__builtin_bit_cast(f32x4, x[2 * s]), __builtin_bit_cast(f32x4, x[2 * s + 1]), xp);
        // those of x1 first where one group works (C128 on 30,000 voxels 156 -> 152 us; with
        // four groups a C64 tile's time went 29.4 -> 30.1 us)
        constexpr int WP[6] = {0, G == 1 ? 1 : 0, G == 1 ? 2 : 1, 0, 1, G == 1 ? 0 : 2};
        constexpr int XP[6] = {0, G == 1 ? 0 : 1, 0, G == 1 ? 1 : 2, 1, G == 1 ? 2 : 0};
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            f32x16& sum = acc[WP[t] + XP[t]][nb];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w[nb][3 * s + WP[t]]), xp[XP[t]], sum,
                                                          0, 0, 0);
          }
      }
    } else {
#pragma unroll
      for (int f = 0; f < XF; ++f)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) Mfma<T>::run(w[nb][f], x[f], acc[0][nb]);
    }
  };

  // The stages, and the sums to LDS: [group][64 rows][BN] fp32, 16-byte chunk c of row r at
  // c ^ (r % 16). plain: in acc[0], each offset's products in acc[1] first, which only rows
  // that have the offset take.
  auto walk = [&](auto plain) __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < NA; ++l)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[l][nb][v] = 0.0f;
    rest = mine;
    lks = lslot = 0;
    // At the barrier of stage s every wave has its share of stage s in LDS and has read
    // the fragments of stage s - 1, whose slot stage s + NS - 1 takes.
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
      if (s < S) issue();
    uint32_t crest = mine;
    int cks = 0, slot = 0;
    for (int s = 0; s < SMAX; ++s) {
      constexpr int AHEAD = NS - 2;  // stages that may stay in flight
      if (s + AHEAD < S) {
        if (wave < BKB % NWG) wait_vmcnt<AHEAD * (LA + LB)>();
        else wait_vmcnt<AHEAD * (LA + LBMIN)>();
      } else {
        wait_vmcnt<0>();
      }
      wait_lgkm0();
      raw_barrier();
      // this block has the offset (none left: false)
      const bool have = s < S && (bmask & (crest & (0u - crest))) != 0;
      if (s + NS - 1 < S) issue();
      __builtin_amdgcn_sched_barrier(0);
      if (have) {
        frags(slot);
        __builtin_amdgcn_sched_barrier(0);
        products(plain);
      }
      slot = slot == NS - 1 ? 0 : slot + 1;
      if (++cks == ksteps) {
        if constexpr (plain) {
          if (have) {
            const bool row_has = gl[__builtin_ctz(crest) * BM + wm * 32 + (lane & 31)] >= 0;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
              for (int v = 0; v < 16; ++v) {
                acc[0][nb][v] += row_has ? acc[1][nb][v] : 0.0f;
                acc[1][nb][v] = 0.0f;
              }
          }
        }
        cks = 0;
        crest &= crest - 1u;
      }
    }
    if constexpr (kSplit && !plain) {
      float bad = 0.0f;  // NaN if a sum is not finite
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          acc[0][nb][v] = (acc[0][nb][v] + (acc[1][nb][v] + acc[2][nb][v])) * (1.0f / (kPartScale * kPartScale));
          bad = fmaf(acc[0][nb][v], 0.0f, bad);
        }
      const uint64_t b = __builtin_amdgcn_ballot_w64(!(bad == 0.0f));
      if (lane == 0) sbad[wave_all] = b != 0 ? 1 : 0;
    }
    wait_lgkm0();
    raw_barrier();
    char* const stg = smem + (group * BM + wm * 32 + (lane & 31)) * SROW;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int chunk = (wn * WN + nb * 32 + 8 * q + 4 * (lane >> 5)) >> 2;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[0][nb][4 * q + e];
        *reinterpret_cast<f32x4*>(stg + ((chunk ^ (lane & 15)) << 4)) = v;
      }
    }
    wait_lgkm0();
    raw_barrier();
  };
  walk(std::false_type{});
  constexpr int E = 16 / ES, CPR = BN / E;                 // 16-byte output pieces of a row
  constexpr int TPR = kLN ? 8 : CPR;                       // threads of a row
  constexpr int PASS = (BM * TPR + THREADS - 1) / THREADS;
  static_assert(!kLN || (ES == 2 && BN == 128), "the row norm takes whole 128-channel rows");
  // the four sums of chunk c of row r
  auto sums = [&](int r, int c) {
    f32x4 v = *reinterpret_cast<const f32x4*>(smem + r * SROW + ((c ^ (r & 15)) << 4));
#pragma unroll
    for (int g = 1; g < G; ++g) v += *reinterpret_cast<const f32x4*>(smem + (g * BM + r) * SROW + ((c ^ (r & 15)) << 4));
    return v;
  };
  auto biased = [&](float y, int n) {
    if (a.bias != nullptr) y += static_cast<float>(reinterpret_cast<const T*>(a.bias)[n]);
    return a.act == HI3D_ACT_SILU ? silu_f32(y) : y;
  };
  if constexpr (kSplit) {
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(sbad[lane % NW] != 0) != 0, 0)) {
      // finite sums first, an output at a time, then the others from the plain walk
      static_assert(PASS * E <= 32, "a bit for each of a thread's outputs");
      uint32_t later = 0;
      auto finish = [&](bool second) {
        for (int i = 0; i < PASS; ++i) {
          const int r = tid / TPR + (THREADS / TPR) * i, n = n0 + tid % CPR * E;
          const int32_t orow = r < BM ? srow[r] : -1;
          if (orow < 0 || orow >= a.n_out || n >= a.cout) continue;
          const f32x4 v = sums(r, tid % CPR);
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const uint32_t bit = 1u << (i * E + e);
            if (!second && !(fabsf(v[e]) < INFINITY)) later |= bit;
            if (second != ((later & bit) != 0)) continue;
            const int64_t at = static_cast<int64_t>(orow) * a.cout + n + e;
            float y = biased(v[e], n + e);
            if (a.residual != nullptr) y += reinterpret_cast<const float*>(a.residual)[at];
            reinterpret_cast<float*>(a.out)[at] = y;
          }
        }
      };
      finish(false);
      wait_vmcnt<0>();
      wait_lgkm0();
      raw_barrier();
      walk(std::true_type{});
      finish(true);
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < PASS; ++i) {
    // (with the norm eight lanes share a row, lane g its pieces g and g + 8)
    const int r = tid / TPR + (THREADS / TPR) * i;
    if (r >= BM) break;
    const int32_t orow = srow[r];
    const bool live = orow >= 0 && orow < a.n_out;
    T h[kLN ? 2 : 1][E];
#pragma unroll
    for (int j = 0; j < (kLN ? 2 : 1); ++j) {
      const int piece = kLN ? tid % 8 + 8 * j : tid % CPR;
      const int n = n0 + piece * E;
      if (!kLN && (!live || n >= a.cout)) continue;  // cout is a multiple of E
#pragma unroll
      for (int p = 0; p < E / 4; ++p) {
        const f32x4 v = sums(r, piece * (E / 4) + p);
#pragma unroll
        for (int e = 0; e < 4; ++e) h[j][4 * p + e] = static_cast<T>(biased(v[e], n + 4 * p + e));
      }
    }
    if constexpr (kLN) {
      f16x8 o[2];
      __builtin_memcpy(o, h, sizeof(o));
      int b = live ? a.ln_coords[static_cast<int64_t>(orow) * 4] : 0;
      b = b < 0 ? 0 : (b >= a.ln_batches ? a.ln_batches - 1 : b);
      const int g = tid % 8;
      ln_modulate_silu_row128(o, a.ln_eps, static_cast<const _Float16*>(a.ln_scale) + b * BN,
                              static_cast<const _Float16*>(a.ln_shift) + b * BN, g);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (live) *reinterpret_cast<f16x8*>(a.out + (static_cast<int64_t>(orow) * BN + (g + 8 * j) * 8) * 2) = o[j];
    } else {
      const int n = n0 + tid % CPR * E;
      if (!live || n >= a.cout) continue;
      const int64_t off = (static_cast<int64_t>(orow) * a.cout + n) * ES;
      u32x4 v;
      __builtin_memcpy(&v, h, sizeof(v));
      if (a.residual != nullptr) v = add_chunk<T>(v, *reinterpret_cast<const u32x4*>(a.residual + off));
      *reinterpret_cast<u32x4*>(a.out + off) = v;
    }
  }
}

template <typename T, int BN, int KS, int NS, int G, bool kLN = false>
int launch_group(const GroupConv& base, hipStream_t stream) {
  GroupConv a = base;
  a.ny = static_cast<int32_t>(ceil_div(a.cout, BN));
  const int64_t blocks = ceil_div(a.n_out, 64) * a.ny;
  HI3D_REQUIRE(blocks < (int64_t(1) << 31), "too many tiles");
  hipLaunchKernelGGL((conv_group_kernel<T, BN, KS, NS, G, kLN>), dim3(static_cast<unsigned>(blocks)),
                     dim3(kGroupThreads * G), 0, stream, a);
  HI3D_LAUNCH_CHECK();
  return HI3D_OK;
}

// 32-channel blocks of the packed weights: whole column tiles.
int col_blocks(int cout) { return cout % 128 == 0 ? cout / 32 : static_cast<int>(ceil_div(cout, 64)) * 2; }

}  // namespace

namespace {

// Which 16-bit convolutions run here, from 9 offsets on (one GPU, fp16, microseconds there
// -> here):
//  * Few 64 x 64 tiles: four offset groups a workgroup, one round of workgroups over the
//    CUs, or two where a tile is worth 128 x 64 products an offset (1,531 voxels C128
//    40 -> 16, 16,000 voxels 42 -> 32; C256 4,000 voxels 130 -> 32; three rounds lose:
//    24,000 voxels C128 41.5 against 48; C64, two rounds, 19.9 against 20.2).
//  * From 256 x 256 channels on, two rounds of 64 x 128 tiles (16,000 voxels C256
//    129 -> 73; three rounds 131 against 131).
//  * Channel counts that the ring and wide kernels do not take, where 64 x 64 tiles cost less
//    than the pipelined kernel's, whose tiles are 256 x 64, 256 x 128 or 128 x 256
//    (any_pays).
enum class Group16 { kNone, kFew, kWide, kAny };

// The pipelined kernel pads to its larger tiles and to whole rounds over the CUs (long rows:
// to one; 1024 -> 128 on 66,001 voxels, two tiles more than a round, 869 us, 947 here); here an
// input row is read again for every 64 channels. Against its 64-channel tiles these are
// always faster (two-voxel shells of 240k and 300k voxels: 32 -> 40 1.9 times, 256 -> 40
// 1.4, 1024 -> 64 1.1). Against the others `per` is the measured time here for an equal
// area of output there, on two-voxel shells of 240k to 300k voxels, where rows have the most
// neighbours: it grows with the row length (64 -> 512 1.17, 256 -> 224 1.37, 512 -> 224 1.61,
// 1024 -> 512 1.69), and rows that are no multiple of 128 bytes, which the pipelined kernel
// reads in halves, do better here (32 -> 224 0.72, 96 -> 224 0.93, 480 -> 224 1.51). 5 % for
// what the measurements spread. Of 891 shapes and sizes timed both ways five of those that the
// rule sends here lose more than 3 %, 6 % at most (64 -> 192 on 30,011 voxels 45 -> 48 us);
// the gains are 96 -> 160 on 120,007 voxels 283 -> 148 us, 128 -> 320 on 300,007 1253 -> 997.
// Kept there: 1024 -> 1024 on 30,011 voxels 2.44 ms against 4.31 here, 576 -> 256 on 300,007
// 3.1 against 4.5, 64 -> 256 on 30,011 47 us against 57.
bool any_pays(int64_t n_out, int cin, int cout, int64_t cus) {
  if (cout <= 64) return true;
  if (cus <= 0) return false;
  const double per = cin % 64 == 0 ? std::min(1.1 + cin / 900.0, 1.7) : std::min(0.7 + cin / 450.0, 1.5);
  const int64_t tiles = cout <= 128 ? ceil_div(n_out, 256) : ceil_div(n_out, 128) * ceil_div(cout, 256);
  const int64_t there = (cin <= 512 ? ceil_div(tiles, cus) * cus : std::max(tiles, cus)) * (128 * 256);
  const int64_t here = ceil_div(n_out, 64) * 64 * ceil_div(cout, 64) * 64;
  return per * static_cast<double>(here) <= 0.95 * static_cast<double>(there);
}

Group16 group16(int64_t n_out, int cin, int cout, int kvol) {
  const int rb = cin * 2;
  if (kvol <= kFewOffsets || kvol > kGroupMaxKvol || cin % 32 != 0 || rb > kGroupMaxRowBytes || cout % 8 != 0)
    return Group16::kNone;
  const int64_t cus = compute_units(), row_tiles = ceil_div(n_out, 64);
  if (row_tiles * ceil_div(cout, 64) <= (static_cast<int64_t>(cin) * cout >= 128 * 64 ? 2 : 1) * cus)
    return Group16::kFew;
  if (cin % 64 == 0 && cin >= 256 && cout % 256 == 0 && row_tiles * (cout / 128) <= 2 * cus) return Group16::kWide;
  const bool ring = (rb % 64 == 0 && rb >= 256 && rb <= 1024 && cout % 128 == 0) ||
                    ((rb == 128 || rb == 256) && (cout == 64 || cout == 128));
  return !ring && any_pays(n_out, cin, cout, cus) ? Group16::kAny : Group16::kNone;
}

template <typename T>
int group16_run(const GroupConv& c, hipStream_t stream) {
  switch (group16(c.n_out, c.cin, c.cout, c.kvol)) {
    case Group16::kFew:
      return c.cin % 64 == 0 ? launch_group<T, 64, 2, 2, 4>(c, stream) : launch_group<T, 64, 1, 2, 4>(c, stream);
    case Group16::kWide: return launch_group<T, 128, 2, 2, 1>(c, stream);
    default: return launch_group<T, 64, 1, 3, 1>(c, stream);
  }
}

}  // namespace

bool group_conv16_takes(int64_t n_out, int cin, int cout, int kvol) {
  return group16(n_out, cin, cout, kvol) != Group16::kNone;
}

int group_conv16(const GroupConv& c, bool bf16, hipStream_t stream) {
  // the row norm (fp16, 128 channels) takes few tiles: 128-channel ones, the same sums
  if (c.ln_coords != nullptr) return launch_group<_Float16, 128, 1, 3, 4, true>(c, stream);
  return bf16 ? group16_run<__bf16>(c, stream) : group16_run<_Float16>(c, stream);
}

}  // namespace hi3d

using namespace hi3d;

extern "C" {

int32_t hi3d_gather_conv_group16(int64_t n_out, int32_t cin, int32_t cout, int32_t kvol) {
  return n_out > 0 && cin > 0 && cout > 0 ? static_cast<int32_t>(group16(n_out, cin, cout, kvol)) : 0;
}

int hi3d_gather_conv_f32_workspace(int32_t cin, int32_t cout, int32_t kvol, int64_t* bytes_host) {
  HI3D_REQUIRE(bytes_host != nullptr, "null pointer argument");
  HI3D_REQUIRE(cin > 0 && cout > 0 && kvol > 0, "channels and kvol must be positive");
  const bool taken = kvol <= kGroupMaxKvol && cin <= kSplitMaxCin && cin % 32 == 0 && cout % 4 == 0 &&
                     (kvol > kFewOffsets || static_cast<int64_t>(cin) * cout >= kFewOffsetsWork);
  *bytes_host = taken ? static_cast<int64_t>(kvol) * (cin / 16) * col_blocks(cout) * 3072 : 0;
  return HI3D_OK;
}

int hi3d_gather_conv_f32(const float* in, int64_t n_in, int32_t cin, const float* weight, int64_t stride_out,
                         int64_t stride_offset, int64_t stride_in, const float* bias, int32_t cout, int32_t kvol,
                         const int32_t* rows, const int32_t* gidx, int64_t n_out, const float* residual, int32_t act,
                         float* out, void* workspace, int64_t workspace_bytes, void* stream) {
  int64_t need = 0;
  if (const int e = hi3d_gather_conv_f32_workspace(cin, cout, kvol, &need)) return e;
  HI3D_REQUIRE(need > 0, "gather conv f32 takes Cin a multiple of 32 up to %d, Cout a multiple of 4 and at most %d offsets",
               kSplitMaxCin, kGroupMaxKvol);
  HI3D_REQUIRE(n_in >= 0 && n_out >= 0, "sizes must be non-negative");
  HI3D_REQUIRE(act == HI3D_ACT_NONE || act == HI3D_ACT_SILU, "unknown activation %d", act);
  if (n_out == 0) return HI3D_OK;
  HI3D_REQUIRE(in && weight && rows && gidx && out, "null pointer argument");
  HI3D_REQUIRE(workspace != nullptr && workspace_bytes >= need, "workspace of %lld bytes needed", static_cast<long long>(need));
  const uintptr_t align = reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out) |
                          reinterpret_cast<uintptr_t>(residual) | reinterpret_cast<uintptr_t>(workspace);
  HI3D_REQUIRE((align & 15) == 0, "feature, residual, output and workspace pointers must be 16-byte aligned");
  HI3D_REQUIRE(stride_out >= 0 && stride_offset >= 0 && stride_in >= 0, "weight strides must be non-negative");
  const bool dense = stride_in == 1 && stride_offset == cin && stride_out == static_cast<int64_t>(cin) * kvol;
  HI3D_REQUIRE((reinterpret_cast<uintptr_t>(weight) & (dense ? 15 : 3)) == 0, "the weight must be 16-byte aligned");
  const bool vec = stride_in == 1 && stride_offset % 4 == 0 && stride_out % 4 == 0 &&
                   (reinterpret_cast<uintptr_t>(weight) & 15) == 0;
  HI3D_REQUIRE((reinterpret_cast<uintptr_t>(bias) & 3) == 0, "the bias must be 4-byte aligned");
  hipStream_t s = as_stream(stream);
  GroupConv a{};
  a.in = reinterpret_cast<const char*>(in);
  a.n_in = n_in;
  a.cin = cin;
  a.packed = static_cast<const char*>(workspace);
  a.col_blocks = col_blocks(cout);
  a.bias = reinterpret_cast<const char*>(bias);
  a.cout = cout;
  a.kvol = kvol;
  a.rows = rows;
  a.gidx = gidx;
  a.n_out = n_out;
  a.residual = reinterpret_cast<const char*>(residual);
  a.act = act;
  a.out = reinterpret_cast<char*>(out);
  const int64_t total = need / 3 / 16;
  hipLaunchKernelGGL(split_weight_kernel, dim3(static_cast<unsigned>(ceil_div(total, 256))), dim3(256), 0, s, weight, stride_out,
                     stride_offset, stride_in, vec, cout, cin, a.col_blocks, total, static_cast<char*>(workspace));
  HI3D_LAUNCH_CHECK();
  // Shapes, against the fp32 MFMA kernels (one box, 3^3 maps, with the weight's split): at
  // most one 64 x 64 tile a CU runs four offset groups a workgroup (3,000 voxels C256: 463 ->
  // 102 us, 8,000 voxels C64: 41 -> 31). Whole 128-channel tiles read each gathered row once
  // per 128 channels (327,581 voxels C128: 1362 -> 814 us; 20,000 voxels 236 -> 131); the
  // others two stages in 48 KB, so that three workgroups share a CU (45,128 voxels C64: 87 ->
  // 71 us). The alternatives, timed before the parts were scaled and summed by size: one
  // group for the two small sets 141 and 43 us for 93 and 30 with four, four groups for 20,000
  // voxels 120 for 107 (a CU with two or three tiles); 64-channel tiles for C128 870 us for
  // 805, 128-row tiles with half the weight reads 808; three slots and two workgroups for
  // C64 84 us for 61.
  if (ceil_div(n_out, 64) * ceil_div(cout, 64) <= compute_units()) return launch_group<float, 64, 1, 2, 4>(a, s);
  if (cout % 128 == 0) return launch_group<float, 128, 2, 2, 1>(a, s);
  return launch_group<float, 64, 2, 2, 1>(a, s);
}

}  // extern "C"
