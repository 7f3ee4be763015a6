// CacheGen codec kernels for MI355X (gfx950): calculate_cdf, encode and
// decode of per-(layer, channel) prefix-code bitstreams.
//
// Replaces calculate_cdf / encode_fast_new / decode_fast_prefsum
// (csrc/cachegen_kernels.cpp:17-155).  The code is the one the reference's
// tests pin (tests/v1/test_cachegen_kernels.py:31-239;
// docs/cachegen/Cachegen.md:30-39): each symbol owns a power-of-two aligned
// interval of the 16-bit CDF range and is always written as the same bit
// string (the top l bits of its interval base), MSB first, each stream
// zero-padded to a byte.  The open points of that format are fixed as
// follows (the CPU oracle states the same rules):
//   L1  low 4 bits of a CDF entry = code length (0 = absent); bases are the
//       entry with those bits cleared; calculate_cdf emits lengths 1..12;
//   L2  bases never decrease: an entry below its predecessor stands for
//       0x10000, and entry n_bins is the end of the range (0x10000);
//   L3  length = low bits, or 16 - floor(log2(width)) when they are 0;
//   L4  calculate_cdf: the lengths of an optimal alphabetic code, the leaf
//       depths of the Garsia-Wachs tree over the present symbols' counts
//       (one present symbol: length 1), when the longest fits 8 bits (at
//       most 256 counted symbols) or 12 (more); otherwise Shannon lengths
//       ceil(log2(n / count)) clamped to [1, 12], Kraft-repaired by
//       lengthening the rarest present symbol; intervals assigned in symbol
//       order with widths halved until aligned (only ever needed for the
//       Shannon lengths), absent symbols at the next present base;
//   L5  encode writes at most `chunk` bytes per stream and reports the full
//       byte length;
//   L6  decode takes the largest symbol whose base is <= the next 16 bits.
//
// Work mapping: nothing here is a dense contraction, so there is no MFMA
// work.  A block takes 64 consecutive (layer, channel) streams, channels
// fastest, and may span layers; lane i of each of its waves works on stream
// i, so a token's symbols are a coalesced 64-byte row.  Per-stream tables
// (histogram, code table, decode tables) live in LDS as [symbol][lane], so
// every lane works in its own column without bank conflicts.
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>
#include "common.h"
#include "cachegen_decode.h"
#include "cachegen_gw.h"
#include "gmem.h"

// Output words (CDF rows, bitstream words, decoded symbols) are stored with
// the streaming hint: nothing in the kernel reads them back.  Measured on
// MI355X (32 layers x 256 tokens x 1024 channels, K and V, three runs each,
// event times): decode 27.3-27.5 -> 25.2-25.3 us, encode 19.9-20.0 ->
// 19.2-19.5 us.
template <typename T> __device__ __forceinline__ void cg_st(T *p, T v) { gstore_nt(p, v); }
// The split encoder stages its CDF rows and symbols with the streaming hint
// (19.4-19.5 -> 18.9-19.1 us by events); calculate_cdf's and decode's
// staging loads stay plain (13.1 -> 14.0 and 25.6 -> 26.5 us with it).

namespace lmc {

namespace {

constexpr int kMaxBins = 64;
constexpr int kPrec = 16;
constexpr int kMaxLen = 12;
constexpr int kBatch = 32;  // symbol loads in flight per lane

// Inclusive prefix sum over the 64 lanes of a wave with DPP moves: shifts
// by 1, 2, 4 and 8 within each row of 16 lanes, then the last lane of row
// 0 (row_bcast:15) and of row 1 (row_bcast:31) added to the rows after it.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  int x = static_cast<int>(v);
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, true);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, true);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false); // row_bcast:15 to rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false); // row_bcast:31 to rows 2, 3
  return static_cast<uint32_t>(x);
}

// Address of stream s's symbol of token 0 (streams are numbered over the
// layers, channels fastest; a layer's symbols are [T, C]).
__device__ __forceinline__ const uint8_t *stream_column(const uint8_t *in, int64_t s, int T, int C) {
  // (a 64-bit division is about 150 instructions)
  const int64_t l = s < (int64_t(1) << 32) ? static_cast<uint32_t>(s) / static_cast<uint32_t>(C) : s / C;
  return in + l * T * C + (s - l * C);
}

// calculate_cdf: 64 streams per block, four waves.  The block's symbols are
// staged into LDS 256 tokens at a time ([tokens][64] u8, 16-byte loads); wave
// q counts the q-th quarter of each staged piece into per-stream LDS
// histogram columns (no-return adds, one column per lane).  Wave q then
// takes symbols [j0, j1) of every stream (lane = stream) for the count sums
// and present-symbol counts.  The Garsia-Wachs steps (cachegen_gw.h) run
// next: one lane per stream in one wave (rotating with the block index, so
// that the blocks of a CU use different SIMDs) when no stream of the block
// has more than 16 present symbols, a quad of lanes per stream in all four
// waves otherwise; a stream whose tree fits the length limit leaves its
// depth counters in LDS and a flag.  The waves again take a quarter of the
// symbols each for the lengths (the tree's depths, or the Shannon lengths,
// the smallest l with count << l >= n from two leading-zero counts) and the
// partial sums of the interval widths, from which every wave writes the
// intervals of its symbols of the Garsia-Wachs streams; the rotating wave
// makes the serial aligned assignment of the other streams (the width of
// each interval capped by the lowest set bit of the running base, after the
// Kraft repair).  The block's 64 rows, contiguous in the output, leave as
// coalesced dword stores.  Blocks take 64 consecutive streams whatever their
// layer, so no block is partly filled but the last.  With `lens` the streams'
// lengths in bytes under these rows are written too (the sum of count times
// code length, from the counts already in registers), and per block the sum
// of the lengths cut to `cap`, so a caller knows every stream's place before
// anything has been encoded.
constexpr int kCdfWaves = 4;
constexpr int kCdfThreads = 64 * kCdfWaves;
constexpr int kCdfPiece = 256;  // tokens staged at a time
// Histogram entries after the derivation: (length << kLenShift) | count.
constexpr int kLenShift = 27;
constexpr uint32_t kCountMask = (1u << kLenShift) - 1u;

// Orders a wave's LDS writes before its later reads of other lanes' words
// (a wave's LDS accesses are performed in order).
__device__ __forceinline__ void wave_sync_cdf() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of cdf_tile_kernel: [staged symbols, later the compacted count lists]
// [histogram [nb][64] u32] [partial interval sums [4][64]] [count sums]
// [Garsia-Wachs flags] [present symbols] [rows [64][nb + 1] int16].  The
// partial sums' first row doubles as histogram row nb while the symbols are
// counted: symbols >= nb are counted there, and the row is written before
// it is read as partial sums.
// The first area holds a staged piece (at most 256 x 64 bytes), the count
// lists (nb <= 64 rows of 64 words) and the node-id mode's leaf sets (63
// rows): 64 rows of 64 words whatever T and nb.
__host__ __device__ constexpr int cdf_stage_words(int, int) { return 64 * 64; }
__host__ __device__ constexpr int cdf_lds_bytes(int T, int nb) {
  return 4 * (cdf_stage_words(T, nb) + nb * 64 + 3 * 64 + kCdfWaves * 64) + 64 * (nb + 1) * 2;
}

// Garsia-Wachs lengths for the streams of this lane's group (Q = 1: lane =
// stream, one wave; Q = 4: four lanes per stream, 16 streams per wave).
// When the longest depth fits the limit (8 bits for at most 256 counted
// symbols, else 12), stores the leaf depths' bit-sliced counters and the
// presence mask in the stream's list column and sets its flag in `gwok`.
template <int Q, int CAP, class It, int kBins>
__device__ __forceinline__ void gw_lengths(uint32_t *hist, uint32_t *lists, uint32_t *gwok, const uint32_t *nsum,
                                           int nb, int stream, int g, int m_max) {
  uint32_t *col = hist + stream;
  uint32_t *lst = lists + stream;
  // Compaction: the counts of the present symbols in symbol order.  Every
  // symbol's count is written at the next free position (m <= s < nb), so
  // an absent one is overwritten by the next present one or lies past the
  // list; the lanes of a group write the same words.  No branches.
  // The histogram holds plain counts here (lengths are stored later).
  using PM = typename std::conditional<(kBins <= 32), uint32_t, uint64_t>::type;
  PM pres = 0;
  int m = 0;
  uint32_t cs[kBins];
#pragma unroll
  for (int s = 0; s < kBins; ++s) cs[s] = s < nb ? col[s * 64] : 0u;
#pragma unroll
  for (int s = 0; s < kBins; ++s) {
    if (s < nb) lst[m * 64] = cs[s];
    const uint32_t here = min(cs[s], 1u);  // present: no compare, no SGPR mask
    pres |= static_cast<PM>(here) << s;
    m += static_cast<int>(here);
  }
  wave_sync_cdf();
  typename It::V a[CAP];
  uint32_t lw[CAP];
  // List position of slot i: lane-major (g CAP + i) for the node-id quads,
  // interleaved (Q i + g) otherwise.
  constexpr bool kLaneMajor = std::is_same<It, cggw::ItemId>::value && Q == 4;
  auto position = [g](int i) { return kLaneMajor ? g * CAP + i : Q * i + g; };
#pragma unroll
  for (int i = 0; i < CAP; ++i) {
    const int pos = position(i);
    lw[i] = lst[(pos < nb ? pos : nb - 1) * 64];
  }
#pragma unroll
  for (int i = 0; i < CAP; ++i) {
    // The empty asm takes the loaded word as an operand, so the loads stay
    // unconditional and back to back: otherwise the compiler moves each
    // load into a branch on `pos < m` and waits for it there (16 serial
    // LDS round trips in the one-lane mode).
    asm volatile("" : "+v"(lw[i]));
    const int pos = position(i);
    a[i] = pos < m ? It::leaf(lw[i], pos) : It::inf();
  }
  if constexpr (std::is_same<It, cggw::ItemId>::value) {
    // Leaf sets by id over the dead list: leaf j's at word j.
#pragma unroll
    for (int i = 0; i < CAP; ++i) lst[position(i) * 64] = 1u << position(i);
  }
  cggw::Depths<typename It::L> dep;
  cggw::run<Q, CAP, It>(a, g, m, m_max, dep, lst);
  const bool ok = m >= 2 && dep.over(nsum[stream] > 256u) == 0;
  if (!ok) return;
  // The lengths phase reads the depths by leaf from the stream's (dead)
  // list column: rows 0-3 the counters' low words, 4-7 their high words,
  // 8-9 the presence mask (the lanes of a group hold the same values).
  using L = typename It::L;
  const L d[4] = {dep.d0, dep.d1, dep.d2, dep.d3};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    lst[k * 64] = static_cast<uint32_t>(d[k]);
    lst[(4 + k) * 64] = static_cast<uint32_t>(static_cast<uint64_t>(d[k]) >> 32);
  }
  lst[8 * 64] = static_cast<uint32_t>(pres);
  lst[9 * 64] = static_cast<uint32_t>(static_cast<uint64_t>(pres) >> 32);
  gwok[stream] = 1u;
}

// kBins: register capacity for per-symbol values (nb <= kBins); kExact: nb
// == kBins, so every per-symbol bound is a constant.
// The code (55 KB for 32 bins) starts on a 64 KB page, so that where it and
// the encoder behind it lie does not follow from the size of the code before
// them: encode_chunk, which runs both back to back, takes 43.4 to 44.9 us at
// this place and at most others, but 46.5 at some (64 x 256 x 1024 symbols;
// this kernel by itself takes the same time anywhere).
template <int kBins, bool kExact>
__attribute__((aligned(65536))) __global__ void __launch_bounds__(kCdfThreads)
    cdf_tile_kernel(const uint8_t *__restrict__ in, int T, int C, int nb,
                    int16_t *__restrict__ out, int64_t n_streams, int vec_tile,
                    int32_t *__restrict__ lens, int64_t *__restrict__ sums, int64_t cap) {
  // Wave priority: 1, and 0 for a wave making the one-lane Garsia-Wachs
  // steps.  A step wave issues VALU almost every cycle and the SIMD arbiter
  // prefers the oldest wave among equals: with every wave at one priority,
  // the steps of an earlier block kept the later blocks' waves on the same
  // SIMD from counting their symbols (that phase took up to 2x longer).  The
  // one-lane steps (at most 16 present symbols) are the shortest chain of
  // the kernel, so they yield; the quad steps of the blocks with up to 32
  // present symbols, the longest chain, keep priority 1.  Measured on a
  // 32 x 256 x 1024 K+V chunk in a standalone build of this kernel: one
  // priority for every wave 26.1 us; priority 0 for both kinds of steps
  // 23.6 (23.3 once the lengths phase lost its branches); this 22.6.
  __builtin_amdgcn_s_setprio(1);
  if (kExact) nb = kBins;
  extern __shared__ uint32_t lds[];
  const int tid = static_cast<int>(threadIdx.x);
  // The wave index, read as a scalar: every per-wave bound below (a wave's
  // symbol share, the wave that runs the one-lane steps) is then uniform.
  const int q = __builtin_amdgcn_readfirstlane(tid / 64);
  const int lane = tid % 64;
  const int64_t s0 = static_cast<int64_t>(blockIdx.x) * 64;
  const int cnt = n_streams - s0 < 64 ? static_cast<int>(n_streams - s0) : 64;
  // The stream column this thread stages: its 16-byte piece of every token
  // row (vec_tile), or its lane's byte.  A piece lies in one layer (C % 16
  // == 0 with vec_tile).
  const int col = vec_tile ? 16 * (tid & 3) : lane;
  const bool col_on = col < cnt;
  const uint8_t *col_src = stream_column(in, s0 + (col_on ? col : 0), T, C);
  uint8_t *tile = reinterpret_cast<uint8_t *>(lds);
  uint32_t *hist = lds + cdf_stage_words(T, nb);
  uint32_t *psum = hist + nb * 64;          // [wave][stream]: partial interval sums
  uint32_t *nsum = psum + kCdfWaves * 64;   // per stream: symbol count
  uint32_t *gwok = nsum + 64;               // per stream: Garsia-Wachs lengths taken
  uint32_t *msum = gwok + 64;               // per stream: present symbols
  int16_t *rows = reinterpret_cast<int16_t *>(msum + 64);
  typedef unsigned int w4 __attribute__((ext_vector_type(4)));
  // The thread's share of a piece: four tokens' 16 bytes (tokens past T
  // repeat the last one, which is stored again).
  w4 v[4];
  auto load_piece = [&](int t0) {
    const uint8_t *src = col_src + static_cast<int64_t>(t0) * C;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int t = k * (kCdfThreads / 4) + (tid >> 2);
      v[k] = gload(reinterpret_cast<const w4 *>(src + static_cast<int64_t>(t < T - t0 ? t : T - t0 - 1) * C));
    }
  };
  if (vec_tile && T > 0) load_piece(0);
  for (int i = tid; i < nb * 64; i += kCdfThreads) hist[i] = 0;
  if (tid < 192) nsum[tid] = 0;
  for (int t0 = 0; t0 < T; t0 += kCdfPiece) {
    const int tc = T - t0 < kCdfPiece ? T - t0 : kCdfPiece;
    if (t0 > 0) __syncthreads();  // the previous piece has been counted
    if (vec_tile) {
      if (col_on) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int t = k * (kCdfThreads / 4) + (tid >> 2);
          reinterpret_cast<w4 *>(tile)[(t < tc ? t : tc - 1) * 4 + (tid & 3)] = v[k];
        }
      }
      // The next piece's loads are under this one's counting (56 planes x
      // 1000 tokens x 256 channels 22.6 -> 21.0 us).
      if (t0 + kCdfPiece < T) load_piece(t0 + kCdfPiece);
    } else if (col_on) {
      const uint8_t *src = col_src + static_cast<int64_t>(t0) * C;
      for (int t = q; t < tc; t += kCdfWaves) tile[t * 64 + lane] = src[static_cast<int64_t>(t) * C];
    }
    __syncthreads();
    const int Tq = (tc + kCdfWaves - 1) / kCdfWaves;
    const int tb = q * Tq < tc ? q * Tq : tc;
    const int te = tb + Tq < tc ? tb + Tq : tc;
    if (lane < cnt && tb < te) {
      // Symbols >= nb (and the padding of a partial batch) are counted in
      // row nb, the partial sums' first row, which no count read sees: two
      // VALU operations per symbol (the row, then the address) and no branch.
      const int tq = te - tb;
      const uint8_t *scol = tile + tb * 64 + lane;
      for (int u0 = 0; u0 < tq; u0 += kBatch) {
        uint32_t sym[kBatch];
        if (u0 + kBatch <= tq) {
#pragma unroll
          for (int i = 0; i < kBatch; ++i) sym[i] = scol[(u0 + i) * 64];
        } else {
#pragma unroll
          for (int i = 0; i < kBatch; ++i) sym[i] = u0 + i < tq ? scol[(u0 + i) * 64] : 0xFFu;
        }
#pragma unroll
        for (int i = 0; i < kBatch; ++i)
          atomicAdd(&hist[min(sym[i], static_cast<uint32_t>(nb)) * 64 + lane], 1u);
      }
    }
  }
  __syncthreads();
  // Count sums and present-symbol counts, spread over the waves: wave q
  // takes symbols [j0, j1) of every stream (lane = stream).
  constexpr int kS = kBins / kCdfWaves;
  const int share = (nb + kCdfWaves - 1) / kCdfWaves;
  const int j0 = q * share;
  const int j1 = j0 + share < nb ? j0 + share : nb;
  {
    uint32_t part = 0, present = 0;
#pragma unroll
    for (int k = 0; k < kS; ++k) {
      const uint32_t c = (k < share && j0 + k < j1) ? hist[(j0 + k) * 64 + lane] : 0u;
      part += c;
      present += min(c, 1u);
    }
    if (lane < cnt && part) {
      atomicAdd(nsum + lane, part);
      atomicAdd(msum + lane, present);
    }
  }
  __syncthreads();
  // Garsia-Wachs lengths; the mode depends on the block's largest number of
  // present symbols, the same in every wave.
  {
    // The wave's maximum by DPP within each 16-lane row (quad, half-row
    // mirror, row mirror), then the four rows' lane 0 by readlane.
    uint32_t m_max = msum[lane];
    m_max = max(m_max, cggw::qp<cggw::kSwap>(m_max));
    m_max = max(m_max, cggw::qp<cggw::kRot2>(m_max));
    m_max = max(m_max, cggw::qp<0x141>(m_max));  // row_half_mirror
    m_max = max(m_max, cggw::qp<0x140>(m_max));  // row_mirror
    const uint32_t r0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m_max), 0));
    const uint32_t r1 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m_max), 16));
    const uint32_t r2 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m_max), 32));
    const uint32_t r3 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m_max), 48));
    const int mm = static_cast<int>(max(max(r0, r1), max(r2, r3)));
    uint32_t *lists = lds;  // the staged symbols are dead
    if (mm >= 2) {
      if (mm <= 16 && T < 65536) {
        __builtin_amdgcn_s_setprio(0);
        if (q == static_cast<int>(blockIdx.x % kCdfWaves))
          gw_lengths<1, 16, cggw::Item16, kBins>(hist, lists, gwok, nsum, nb, lane, 0, mm);
      } else if (mm <= 32 && T < 65536) {
        gw_lengths<4, 8, cggw::ItemId, kBins>(hist, lists, gwok, nsum, nb, q * 16 + lane / 4, lane & 3, mm);
      } else if (mm <= 32) {
        gw_lengths<4, 8, cggw::Item32, kBins>(hist, lists, gwok, nsum, nb, q * 16 + lane / 4, lane & 3, mm);
      } else if constexpr (kBins > 32) {
        gw_lengths<4, 16, cggw::Item64, kBins>(hist, lists, gwok, nsum, nb, q * 16 + lane / 4, lane & 3, mm);
      }
    }
  }
  __syncthreads();
  __builtin_amdgcn_s_setprio(1);
  // Lengths and interval assignment, spread over the waves: wave q takes
  // symbols [j0, j1) of every stream (lane = stream).  A Garsia-Wachs stream
  // keeps its tree's depths; the others (one present symbol, no counted
  // symbol, or a tree deeper than the limit) take the Shannon lengths
  // ceil(log2(n / count)) clamped to [1, 12].  Each wave sums its symbols'
  // widths 2^(16 - length) into LDS: for a Garsia-Wachs stream the lengths
  // form a complete alphabetic code, so each symbol's interval starts at the
  // sum of the widths before it, already aligned to its own width, and every
  // wave writes its own symbols' entries; an absent symbol (length 0) takes
  // the base of the next present one (or the end).
  const bool gw = gwok[lane] != 0;
  {
    const uint32_t n = nsum[lane];
    const int ln31 = -__builtin_clz(n | 1u);  // floor(log2 n) - 31
    // A Garsia-Wachs stream's depths by leaf (the leaf of symbol s is the
    // number of present symbols below it).
    const uint32_t *dcol = lds + lane;
    uint64_t dsl[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      dsl[k] = static_cast<uint64_t>(dcol[k * 64]) | (static_cast<uint64_t>(dcol[(4 + k) * 64]) << 32);
    const uint64_t pres = static_cast<uint64_t>(dcol[8 * 64]) | (static_cast<uint64_t>(dcol[9 * 64]) << 32);
    // The wave's counts (plain counts: no length is stored yet), all read
    // before the first is used; the empty asm keeps each read unconditional
    // (the compiler would otherwise move it into a branch and wait there).
    uint32_t cv[kS];
#pragma unroll
    for (int k = 0; k < kS; ++k) cv[k] = hist[min(j0 + k, nb - 1) * 64 + lane];
#pragma unroll
    for (int k = 0; k < kS; ++k) asm volatile("" : "+v"(cv[k]));
    uint32_t len[kS];
    uint32_t own = 0;
#pragma unroll
    for (int k = 0; k < kS; ++k) {
      const bool in_range = kExact || (k < share && j0 + k < j1);  // uniform
      const int s = in_range ? j0 + k : 0;
      const uint32_t cs = in_range ? cv[k] : 0u;
      // The Shannon length: the smallest x with cs << x >= n, which is
      // x0 = floor(log2 n) - floor(log2 cs) or x0 + 1.  For cs >= 1,
      // cs << x0 < 2^(floor(log2 n) + 1) <= 2^26, so the test is a 32-bit
      // subtraction's sign.
      int x = ln31 + static_cast<int>(__builtin_clz(cs | 1u));  // x0
      x += static_cast<int>(((cs << x) - n) >> 31);
      x = min(max(x, 1), kMaxLen);
      const int j = kBins <= 32 ? __builtin_popcount(static_cast<uint32_t>(pres) & ((1u << s) - 1u))
                                : __builtin_popcountll(pres & ((1ull << s) - 1ull));
      uint32_t depth;
      if constexpr (kBins <= 32) {
        const uint32_t jj = static_cast<uint32_t>(j) & 31u;
        depth = __builtin_amdgcn_ubfe(static_cast<uint32_t>(dsl[0]), jj, 1u) |
                (__builtin_amdgcn_ubfe(static_cast<uint32_t>(dsl[1]), jj, 1u) << 1) |
                (__builtin_amdgcn_ubfe(static_cast<uint32_t>(dsl[2]), jj, 1u) << 2) |
                (__builtin_amdgcn_ubfe(static_cast<uint32_t>(dsl[3]), jj, 1u) << 3);
      } else {
        const int jj = j & 63;
        depth = static_cast<uint32_t>(((dsl[0] >> jj) & 1u) | (((dsl[1] >> jj) & 1u) << 1) |
                                      (((dsl[2] >> jj) & 1u) << 2) | (((dsl[3] >> jj) & 1u) << 3));
      }
      // Both lengths are computed for every symbol (no branch on cs).
      uint32_t xs = static_cast<uint32_t>(x);
      asm volatile("" : "+v"(xs), "+v"(depth));
      const uint32_t xl = cs ? (gw ? depth : xs) : 0u;
      len[k] = xl;
      own += 0x8000u >> ((xl - 1u) & 31u);  // 2^(16 - xl), 0 for xl = 0
      // Every lane stores; only the Shannon streams' words are read again.
      if (in_range) hist[s * 64 + lane] = (xl << kLenShift) | cs;
    }
    psum[q * 64 + lane] = own;
    // The wave's share of the stream's length in bits, in list rows that
    // hold no depths (16 on): the lists are dead.
    if (lens != nullptr) {
      uint32_t nbits = 0;
#pragma unroll
      for (int k = 0; k < kS; ++k)
        if (kExact || (k < share && j0 + k < j1)) nbits += len[k] * cv[k];
      lds[(16 + q) * 64 + lane] = nbits;
    }
    __syncthreads();
    int16_t *row = rows + lane * (nb + 1);
    if (gw) {
      uint32_t pos = 0;
#pragma unroll
      for (int w = 0; w < kCdfWaves - 1; ++w) pos += w < q ? psum[w * 64 + lane] : 0u;
#pragma unroll
      for (int k = 0; k < kS; ++k) {
        if (kExact || (k < share && j0 + k < j1)) {
          row[j0 + k] = static_cast<int16_t>(static_cast<uint16_t>((pos | len[k]) & 0xFFFFu));
          pos += 0x8000u >> ((len[k] - 1u) & 31u);  // 2^(16 - len), 0 for len 0
        }
      }
    }
    if (q == 0) row[nb] = 0;
  }
  // The Shannon streams, in one wave: the Kraft repair (lengthen the rarest
  // present symbol below the cap, the last one among equals, until the code
  // fits; only a length capped at 12 bits, more than 4096 counted symbols,
  // can need it, so it runs out of line on the LDS column), then the aligned
  // in-order assignment: a symbol's base is the running position `pos`, its
  // width 2^(16 - length) capped by the lowest set bit of `pos` (the code
  // lengthened to match).
  if (q == static_cast<int>(blockIdx.x % kCdfWaves) && lane < cnt && !gw) {
    uint32_t *wcol = hist + lane;  // (length << kLenShift) | count
    uint32_t kraft = 0;            // units of 2^-16
#pragma unroll
    for (int w = 0; w < kCdfWaves; ++w) kraft += psum[w * 64 + lane];
    while (kraft > (1u << kPrec)) {
      int pick = -1;
      uint32_t best = 0;
#pragma unroll 1
      for (int s = 0; s < nb; ++s) {
        const uint32_t v = wcol[s * 64], ls = v >> kLenShift, cs = v & kCountMask;
        if (ls != 0 && ls < kMaxLen && (pick < 0 || cs <= best)) {
          pick = s;
          best = cs;
        }
      }
      if (pick < 0) break;
      const uint32_t lp = wcol[pick * 64] >> kLenShift;
      kraft -= 1u << (kPrec - lp - 1);
      wcol[pick * 64] += 1u << kLenShift;
    }
    uint32_t len[kBins];
#pragma unroll
    for (int s = 0; s < kBins; ++s) {
      const uint32_t v = wcol[(s < nb ? s : 0) * 64];  // every read issued before the first use
      len[s] = s < nb ? v >> kLenShift : 0u;
    }
    int16_t *row = rows + lane * (nb + 1);
    // r is the running base with bit 16 set, so its lowest set bit is the
    // base's alignment (0x10000 for base 0, above every width); the width
    // taken is min(2^(16 - length), that bit), and the length follows from
    // it.  The chain from one symbol to the next is four operations.
    uint32_t r = 1u << kPrec;
    uint32_t nbits = 0;
#pragma unroll
    for (int s = 0; s < kBins; ++s) {
      if (s < nb) {
        const uint32_t x0 = len[s];
        const uint32_t w0 = x0 ? 1u << (kPrec - x0) : 0u;
        const uint32_t w = min(w0, r & (0u - r));
        const uint32_t x = x0 ? static_cast<uint32_t>(__builtin_clz(w)) - (31u - kPrec) : 0u;
        row[s] = static_cast<int16_t>(static_cast<uint16_t>((r | x) & 0xFFFFu));
        r += w;
        if (lens != nullptr) nbits += x * (wcol[s * 64] & kCountMask);
      }
    }
    // In place of the waves' shares.
    if (lens != nullptr) {
#pragma unroll
      for (int w = 0; w < kCdfWaves; ++w) lds[(16 + w) * 64 + lane] = w == 0 ? nbits : 0u;
    }
  }
  __syncthreads();
  // Stream lengths in bytes, and the block's bytes once every stream is cut
  // to cap.
  if (lens != nullptr && q == 0) {
    uint32_t nbits = 0;
#pragma unroll
    for (int w = 0; w < kCdfWaves; ++w) nbits += lds[(16 + w) * 64 + lane];
    const uint32_t nbytes = lane < cnt ? (nbits + 7) >> 3 : 0u;
    if (lane < cnt) lens[s0 + lane] = static_cast<int32_t>(nbytes);
    const uint32_t kept = static_cast<int64_t>(nbytes) < cap ? nbytes : static_cast<uint32_t>(cap);
    // A stream has at most 2^26 codes of 12 bits, so the sum of 64 fits only
    // 64 bits: two scans, of the low and high halves.
    const uint32_t lo = wave_incl_scan(kept & 0xFFFFu), hi = wave_incl_scan(kept >> 16);
    if (lane == 63) sums[blockIdx.x] = (static_cast<int64_t>(hi) << 16) + lo;
  }
  // The block's rows are contiguous in the output.
  int16_t *dst = out + s0 * (nb + 1);
  const int total = cnt * (nb + 1);
  if ((reinterpret_cast<uintptr_t>(dst) & 3) == 0) {
    for (int i = tid; i < total / 2; i += kCdfThreads)
      cg_st(reinterpret_cast<uint32_t *>(dst) + i, reinterpret_cast<const uint32_t *>(rows)[i]);
    if ((total & 1) && tid == 0) dst[total - 1] = rows[total - 1];
  } else {
    for (int i = tid; i < total; i += kCdfThreads) dst[i] = rows[i];
  }
}

// Encode: 64 streams per block (consecutive ones, whatever their layer) and
// PIECES waves, kEncTokens tokens at a time, wave w taking tokens
// [w * Q, (w + 1) * Q) of every stream (Q = kEncTokens / PIECES), lane s
// stream s.  Each lane walks a serial chain of only Q codes, and every wave
// instruction works for 64 streams.
//   1. The block's CDF rows (contiguous in memory) are staged with dword
//      loads; its symbols are staged untransposed, [token][64 channels]
//      bytes, with 16-byte stores (tokens past T read as 0xFF, not
//      coded).  Lane s then reads token t's symbol at t * 64 + s: the 64
//      lanes read 16 consecutive words.
//   2. Code table in LDS, [symbol][stream] words of (code << 11) | length
//      (rules L1-L3), built with lane = stream, so its stores and the
//      lookups of step 3 each hit 64 distinct banks; row nb is all zeros
//      and takes every symbol >= nb.  Wave w writes the w-th share of the
//      symbols, after finding from the row whether the wrap of rule L2
//      (an entry below its predecessor) lies before its share.  The block
//      notes whether any code is longer than 8 bits.
//   3. Each lane looks up its Q codes into registers and sums their
//      lengths (the sum of the entries' low 11 bits: at most 64 x 15 bits,
//      so no carry reaches the code field).  The piece lengths of a stream
//      give each piece its bit offset.
//   4. The staged symbols are dead; the same LDS holds the zeroed bits, and
//      each lane ORs its codes in as runs of at most 32 bits: four codes per
//      run when no code of the block is longer than 8 bits, else two.
//   5. The bits leave as dwords, and the last bytes of a stream one by one.
//
// The streams' places: rows of `chunk` bytes (place 0), or one after the
// other from the block's first row on, each cut to `chunk` bytes (place 1; a
// later copy then moves whole blocks).  Three forms:
//   kRows   place 0, at most kEncTokens tokens.
//   kImage  place 1, at most kEncTokens tokens, no stream cut: the streams'
//           bits lie one after the other in LDS as well, so only the bytes
//           in use are cleared and they leave as 16-byte stores.
//   kLong   the rest.  Steps 1, 3, 4 and 5 once per kEncTokens, the last
//           dword of a stream carried over, the next symbols loaded under
//           the present ones' coding.  A stream's bits are laid out in LDS
//           from its address modulo 4, so LDS dwords are memory dwords
//           wherever it starts; with place 1 its length is read from `lens`.
//           It takes 94 registers, which leaves two blocks on a CU where the
//           other forms have four (kRows' work in it: 22.2 us against 16.6).
//
// Measured on MI355X, 64 planes x 256 tokens x 1024 channels (32 bins in the
// first 10 planes, 16 in the others): kRows 16.9 us, kImage 12.3 to 13.0; 56
// planes x 1000 tokens x 256 channels, kLong 22 us, against 128 us for a lane
// per stream walking all its tokens.
enum class EncMode { kRows, kImage, kLong };
constexpr int kEncLanes = 64;
#ifndef LMC_ENC_PIECES
#define LMC_ENC_PIECES 8    // waves (token pieces) per block of the encoder
#endif
constexpr int kEncPieces = LMC_ENC_PIECES;
constexpr int kEncTokens = 256;

__device__ __forceinline__ void enc_append(uint32_t *brow, uint32_t &pos, uint32_t run, uint32_t n) {
  // `run` holds n <= 32 bits (0 when n is 0); its top-aligned form is ORed
  // into the one or two words it touches.
  const uint32_t top = run << ((32u - n) & 31u);
  const uint32_t wi = pos >> 5, sh = pos & 31u;
  atomicOr(brow + wi, top >> sh);  // a no-op when n is 0
  if (sh + n > 32u) atomicOr(brow + wi + 1, top << (32u - sh));
  pos += n;
}

// LDS of the encoder, in words: [64][nb + 1] int16 rows and [256][64] u8
// symbols, and over them the bits (64 rows of row_words, or the block's bits
// one stream after the other); [nb + 1][64] u32 codes, inside the bits' area
// when the whole chunk is coded at once and after it otherwise; then
// [PIECES][64] piece lengths, the long-code flag and [64] u64 decrease masks.
struct EncLds {
  int rows_words, tab_at, row_words, plen_at, bytes;
};
inline EncLds enc_lds(int64_t T, int nb) {
  EncLds e;
  const int tokens = static_cast<int>(std::min<int64_t>(T, kEncTokens));
  e.rows_words = ((nb + 1) * kEncLanes * 2 + 15) / 16 * 4;
  // Codes are at most 15 bits; a carried dword or a lead of 3 bytes before
  // them, and a partial dword after.  An odd number of words, so that the
  // streams' rows start in different banks.
  e.row_words = ((tokens * 15 + 31) / 32 + 2) | 1;
  const int staged = e.rows_words + kEncTokens * kEncLanes / 4;
  const int bits = kEncLanes * e.row_words;
  const int codes = (nb + 1) * kEncLanes;
  e.tab_at = T > kEncTokens ? std::max(staged, bits) : staged;
  e.plen_at = std::max(e.tab_at + codes, bits);
  e.bytes = 4 * (((e.plen_at + kEncPieces * kEncLanes + 2) & ~1) + 2 * kEncLanes);
  return e;
}

// Exclusive prefix sums of n block byte counts by one workgroup of NT
// threads: off[b] for block b, off[n] and *total the sum.  `total` is host
// memory a thread may be watching: it is written last, at system scope.
// `wave_sum` is scratch in LDS.
struct BlockOffsets {
  const int64_t *sums;  // null: no offsets to make
  int64_t n;
  int64_t *off;
  int64_t *total;
};
template <int NT> __device__ __forceinline__ void block_offsets(const BlockOffsets &b, int64_t *wave_sum) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int wave = static_cast<int>(threadIdx.x) >> 6;
  int64_t carry = 0;
  for (int64_t i0 = 0; i0 < b.n; i0 += NT) {
    const int64_t i = i0 + threadIdx.x;
    const int64_t own = i < b.n ? b.sums[i] : 0;
    int64_t incl = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t v = __shfl_up(incl, d, 64);
      incl += lane >= d ? v : 0;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    int64_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
      before += w < wave ? wave_sum[w] : 0;
      all += wave_sum[w];
    }
    if (i < b.n) b.off[i] = carry + before + incl - own;
    carry += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    b.off[b.n] = carry;
    __hip_atomic_store(b.total, carry, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// With `offsets` the launch has one block more, the first: it makes the
// blocks' offsets while the others encode (as a kernel of its own before them
// it took 4.1 us of the chunk's time).
template <int PIECES, EncMode MODE>
__global__ void __launch_bounds__(64 * PIECES)
    encode_split_kernel(const int16_t *__restrict__ cdf, const uint8_t *__restrict__ in, int T, int C, int nb,
                        int64_t n_streams, uint8_t *__restrict__ out, int64_t chunk, int32_t *__restrict__ lens,
                        int place, int vec_tile, int rows_dw, const EncLds at, const BlockOffsets offsets) {
  constexpr int NT = 64 * PIECES;
  constexpr int Q = kEncTokens / PIECES;  // tokens per piece
  constexpr bool IMAGE = MODE == EncMode::kImage, LONG = MODE == EncMode::kLong;
  extern __shared__ uint32_t lds[];
  typedef unsigned int w4 __attribute__((ext_vector_type(4)));
  const int tid = static_cast<int>(threadIdx.x);
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  int64_t block = blockIdx.x;
  if (offsets.sums != nullptr) {
    if (block == 0) {
      block_offsets<NT>(offsets, reinterpret_cast<int64_t *>(lds));
      return;
    }
    --block;
  }
  const int64_t s0 = block * kEncLanes;
  const int cnt = n_streams - s0 < kEncLanes ? static_cast<int>(n_streams - s0) : kEncLanes;
  int16_t *stage = reinterpret_cast<int16_t *>(lds);
  uint8_t *tile = reinterpret_cast<uint8_t *>(lds + at.rows_words);
  uint32_t *tab = lds + at.tab_at;
  uint32_t *bits = lds;
  uint32_t *plen = lds + at.plen_at;
  uint32_t *long_flag = plen + PIECES * kEncLanes;
  uint64_t *dmask = reinterpret_cast<uint64_t *>(lds + ((at.plen_at + PIECES * kEncLanes + 2) & ~1));

  // 1. Staging: every global load of the thread, then its LDS stores.  The
  //    thread stages one 16-byte piece of a token (vec_tile; it lies in one
  //    layer, C % 16 == 0) or one byte.
  const int col = vec_tile ? 16 * (tid & 3) : lane;
  const bool col_on = col < cnt;
  const uint8_t *src = stream_column(in, s0 + (col_on ? col : 0), T, C);
  constexpr int kV = (4 * kEncTokens + NT - 1) / NT;  // 16-byte pieces per thread
  const w4 none = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};
  w4 v[kV];
  auto load_symbols = [&](int t0) {
#pragma unroll
    for (int k = 0; k < kV; ++k) {
      const int t = t0 + k * (NT / 4) + (tid >> 2);
      v[k] = gload_nt(reinterpret_cast<const w4 *>(src + static_cast<int64_t>(t < T ? t : T - 1) * C));
    }
  };
  auto store_symbols = [&](int t0) {
    if (vec_tile) {
#pragma unroll
      for (int k = 0; k < kV; ++k)  // every piece of the 256 x 64 tile, in or past T
        reinterpret_cast<w4 *>(tile)[k * NT + tid] =
            col_on && t0 + k * (NT / 4) + (tid >> 2) < T ? v[k] : none;
    } else {
      for (int t = wv; t < kEncTokens; t += PIECES)
        tile[t * kEncLanes + lane] =
            col_on && t0 + t < T ? src[static_cast<int64_t>(t0 + t) * C] : static_cast<uint8_t>(0xFF);
    }
  };
  {
    const int rcount = cnt * (nb + 1);
    if (rows_dw && cnt == kEncLanes) {
      const uint32_t *rsrc = reinterpret_cast<const uint32_t *>(cdf + s0 * (nb + 1));
      constexpr int kR = (kEncLanes * 33 / 2 + NT - 1) / NT;  // row dwords per thread for nb <= 32
      uint32_t rv[kR];
      int ri[kR];
#pragma unroll
      for (int k = 0; k < kR; ++k) {
        const int i = k * NT + tid;
        ri[k] = i < rcount / 2 ? i : rcount / 2 - 1;
        rv[k] = gload_nt(rsrc + ri[k]);
      }
      if (vec_tile && T > 0) load_symbols(0);
      store_symbols(0);
      uint32_t *rdst = reinterpret_cast<uint32_t *>(stage);
#pragma unroll
      for (int k = 0; k < kR; ++k) rdst[ri[k]] = rv[k];
      for (int i = kR * NT + tid; i < rcount / 2; i += NT) rdst[i] = rsrc[i];
    } else {
      if (vec_tile && T > 0) load_symbols(0);
      store_symbols(0);
      for (int i = tid; i < kEncLanes * (nb + 1); i += NT)
        stage[i] = i < rcount ? cdf[s0 * (nb + 1) + i] : static_cast<int16_t>(0);
    }
    if (tid == 0) *long_flag = 0u;
    if (tid < kEncLanes) dmask[tid] = 0u;
  }
  __syncthreads();

  // 2. Code table, lane = stream; wave w writes symbols [j0, j1).  First
  //    each wave marks the decreases of rule L2 in its range (entry j below
  //    entry j - 1) in the stream's 64-bit mask, so that afterwards symbol j
  //    is wrapped exactly when the mask has a bit at or below j.
  {
    constexpr int kShare = (kMaxBins + PIECES - 1) / PIECES;
    const int16_t *row = stage + lane * (nb + 1);
    const int share = (nb + PIECES - 1) / PIECES;
    const int j0 = wv * share;
    const int j1 = j0 + share < nb ? j0 + share : nb;
    uint32_t m[kShare + 1];  // masked entries j0 .. j0 + kShare (0 past nb - 1)
#pragma unroll
    for (int k = 0; k <= kShare; ++k)
      m[k] = (k <= share && j0 + k < nb) ? (static_cast<uint16_t>(row[j0 + k]) & 0xFFF0u) : 0u;
    const uint32_t m_before = j0 > 0 && j0 < nb ? (static_cast<uint16_t>(row[j0 - 1]) & 0xFFF0u) : 0u;
    uint64_t dec = 0;
#pragma unroll
    for (int k = 0; k < kShare; ++k) {
      const int jj = j0 + k;
      const uint32_t prev = k == 0 ? m_before : m[k - 1];
      if (k < share && jj < j1 && jj >= 1 && m[k] < prev) dec |= uint64_t(1) << jj;
    }
    if (dec) atomicOr(dmask + lane, static_cast<unsigned long long>(dec));
    __syncthreads();
    const uint64_t D = dmask[lane];
    uint32_t longest = 0;
#pragma unroll
    for (int k = 0; k < kShare; ++k) {
      const int jj = j0 + k;
      if (k < share && jj < j1) {
        const uint32_t raw = static_cast<uint16_t>(row[jj]);
        const bool wrapped = (D & (~uint64_t(0) >> (63 - jj))) != 0;
        const bool has_n = jj + 1 < nb;
        const bool wrapped_n = has_n && (D & (~uint64_t(0) >> (62 - jj))) != 0;
        const uint32_t base = wrapped ? 0x10000u : m[k];
        const uint32_t next = (has_n && !wrapped_n) ? m[k + 1] : 0x10000u;
        const uint32_t width = next - base;
        // Rule L3: the low bits, else 16 - floor(log2(width)) (0 for an empty interval).
        const uint32_t wlen = width ? static_cast<uint32_t>(__builtin_clz(width)) - 15u : 0u;
        const uint32_t len = (raw & 0xFu) ? (raw & 0xFu) : wlen;
        const uint32_t code = __builtin_amdgcn_ubfe(base, kPrec - len, len);  // 0 when len is 0
        tab[jj * kEncLanes + lane] = (code << 11) | len;
        longest = len > longest ? len : longest;
      }
    }
    if (wv == 0) tab[nb * kEncLanes + lane] = 0u;
    if (__ballot(longest > 8u) && lane == 0) *long_flag = 1u;
  }
  __syncthreads();
  const bool long_codes = *long_flag != 0u;

  // Where the lane's stream goes: its bytes start `dst`, the LDS bits at
  // bit 8 * (dst % 4); `bit` is the bits of the present dword already taken
  // (the lead, then the carry), `carry` their value, `first` the index of
  // that dword from dst - dst % 4.
  uint8_t *block_out = out + s0 * chunk;
  int64_t off = static_cast<int64_t>(lane) * chunk;
  if (LONG && place == 1) {
    const int64_t len = lane < cnt ? lens[s0 + lane] : 0;
    const uint32_t kept = static_cast<uint32_t>(len < chunk ? len : chunk);
    const uint32_t lo = wave_incl_scan(kept & 0xFFFFu), hi = wave_incl_scan(kept >> 16);
    off = (static_cast<int64_t>(hi) << 16) + lo - kept;
  }
  const uint32_t lead = LONG ? static_cast<uint32_t>(reinterpret_cast<uintptr_t>(block_out + off) & 3) : 0u;
  uint32_t bit = 8u * lead, carry = 0, first = 0;

  int t0 = 0;
  do {
    const bool more = LONG && t0 + kEncTokens < T;
    // 3. Lookups into registers, and the piece's length.
    uint32_t e[Q];
    uint32_t sum = 0;
    {
      const uint8_t *scol = tile + wv * Q * kEncLanes + lane;
      const uint32_t *tcol = tab + lane;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const uint32_t x = scol[i * kEncLanes];
        e[i] = tcol[(x < static_cast<uint32_t>(nb) ? x : static_cast<uint32_t>(nb)) * kEncLanes];
      }
#pragma unroll
      for (int i = 0; i < Q; i += 2) sum += e[i] + e[i + 1];
    }
    plen[wv * kEncLanes + lane] = sum & 0x7FFu;
    if (more && vec_tile) load_symbols(t0 + kEncTokens);
    __syncthreads();

    // 4. The bits: cleared, then each piece ORed in at its offset.
    uint32_t pos = bit, total = bit;
#pragma unroll
    for (int w = 0; w < PIECES; ++w) {
      const uint32_t n = plen[w * kEncLanes + lane];
      pos += w < wv ? n : 0u;
      total += n;
    }
    uint32_t *brow = bits + lane * at.row_words;
    uint32_t words = static_cast<uint32_t>(kEncLanes * at.row_words);
    uint32_t image_bytes = 0;
    if (IMAGE) {
      const uint32_t nbytes = (total + 7) >> 3;
      const uint32_t incl = wave_incl_scan(nbytes);
      pos += 8u * (incl - nbytes);
      brow = bits;
      image_bytes = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), kEncLanes - 1));
      words = (image_bytes + 15) / 16 * 4;
    }
    {
      w4 *b4 = reinterpret_cast<w4 *>(bits);
      const w4 z = {0u, 0u, 0u, 0u};
      for (uint32_t i = tid; i < words / 4; i += NT) b4[i] = z;
      for (uint32_t i = words / 4 * 4 + tid; i < words; i += NT) bits[i] = 0u;
    }
    __syncthreads();
    if (LONG && wv == 0 && carry != 0) atomicOr(brow, carry);
    if (!long_codes) {
      // Codes of at most 8 bits: four to a run.
#pragma unroll
      for (int i = 0; i < Q; i += 4) {
        uint32_t run = e[i] >> 11;
        run = (run << (e[i + 1] & 31u)) | (e[i + 1] >> 11);
        run = (run << (e[i + 2] & 31u)) | (e[i + 2] >> 11);
        run = (run << (e[i + 3] & 31u)) | (e[i + 3] >> 11);
        const uint32_t n = (e[i] + e[i + 1] + e[i + 2] + e[i + 3]) & 0x7FFu;
        enc_append(brow, pos, run, n);
      }
    } else {
#pragma unroll
      for (int i = 0; i < Q; i += 2) {
        const uint32_t run = ((e[i] >> 11) << (e[i + 1] & 31u)) | (e[i + 1] >> 11);
        const uint32_t n = (e[i] + e[i + 1]) & 0x7FFu;  // <= 30
        enc_append(brow, pos, run, n);
      }
    }
    if (IMAGE) {
      if (wv == 0 && lane < cnt) lens[s0 + lane] = static_cast<int32_t>((total + 7) >> 3);
      __syncthreads();
      // 5. The block's bytes: whole 16-byte vectors as far as they lie in the
      //    block's place, cnt * chunk bytes.  A last block of few streams and
      //    tokens may end inside a vector of its place; those bytes leave one
      //    by one.
      const int64_t room = cnt * chunk / 16;
      const uint32_t vecs = room < words / 4 ? static_cast<uint32_t>(room) : words / 4;
      for (uint32_t i = tid; i < vecs; i += NT) {
        w4 x = reinterpret_cast<const w4 *>(bits)[i];
        x.x = __builtin_bswap32(x.x);
        x.y = __builtin_bswap32(x.y);
        x.z = __builtin_bswap32(x.z);
        x.w = __builtin_bswap32(x.w);
        cg_st(reinterpret_cast<w4 *>(block_out) + i, x);
      }
      for (uint32_t b = 16 * vecs + tid; b < image_bytes; b += NT)
        block_out[b] = static_cast<uint8_t>(bits[b >> 2] >> (24 - 8 * (b & 3u)));
      return;
    }
    if (!LONG) {
      if (wv == 0 && lane < cnt) lens[s0 + lane] = static_cast<int32_t>((total + 7) >> 3);
      __syncthreads();
      // 5. A wave per stream: full words as dword stores where the rows start
      //    on dwords, the bytes of a last partial word by one lane each.
      const bool word_stores = chunk % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 3) == 0;
      for (int st = wv; st < cnt; st += PIECES) {
        const uint32_t tb = __builtin_amdgcn_readlane(static_cast<int>(total), st);  // wave-uniform
        const uint32_t tbytes = (tb + 7) >> 3;
        const uint32_t nbytes = chunk < static_cast<int64_t>(tbytes) ? static_cast<uint32_t>(chunk) : tbytes;
        uint8_t *orow = block_out + st * chunk;
        const uint32_t *sb = bits + st * at.row_words;
        const uint32_t nw = word_stores ? nbytes >> 2 : 0u;
        for (uint32_t k = lane; k < nw; k += kEncLanes)
          cg_st(reinterpret_cast<uint32_t *>(orow) + k, __builtin_bswap32(sb[k]));
        for (uint32_t b = 4 * nw + lane; b < nbytes; b += kEncLanes)
          orow[b] = static_cast<uint8_t>(sb[b >> 2] >> (24 - 8 * (b & 3u)));
      }
      return;
    }
    // Bytes of the stream from dst - lead: [lead, end) may be stored.
    const int64_t bytes = static_cast<int64_t>(first) * 4 + ((total + 7) >> 3);
    const int64_t room = lead + chunk;
    const int64_t end = more || bytes > room ? room : bytes;
    if (wv == 0 && lane < cnt && !more) lens[s0 + lane] = static_cast<int32_t>(bytes - lead);
    __syncthreads();

    // 5. Half a wave per stream, its dwords [first, first + nw).
    const uint32_t nw = more ? total >> 5 : (total + 31) >> 5;
    const int half = lane >> 5;
#pragma unroll 2
    for (int p = wv; 2 * p < cnt; p += PIECES) {
      const int st = 2 * p + half;
      const uint32_t st_nw = __shfl(nw, st, 64), st_first = __shfl(first, st, 64), st_lead = __shfl(lead, st, 64);
      const int64_t st_end = __shfl(end, st, 64);
      uint8_t *row = block_out + __shfl(off, st, 64) - st_lead;
      const uint32_t *sb = bits + st * at.row_words;
      if (st < cnt) {
        for (uint32_t k = lane & 31; k < st_nw; k += 32) {
          const int64_t b0 = 4 * (static_cast<int64_t>(st_first) + k);
          const uint32_t x = __builtin_bswap32(sb[k]);
          if (b0 >= st_lead && b0 + 4 <= st_end) {
            cg_st(reinterpret_cast<uint32_t *>(row + b0), x);
          } else {
#pragma unroll
            for (int b = 0; b < 4; ++b)
              if (b0 + b >= st_lead && b0 + b < st_end) row[b0 + b] = static_cast<uint8_t>(x >> (8 * b));
          }
        }
      }
    }
    if (!more) return;
    carry = (total & 31u) ? brow[total >> 5] : 0u;
    first += total >> 5;
    bit = total & 31u;
    __syncthreads();  // the bits are dead
    t0 += kEncTokens;
    store_symbols(t0);
    __syncthreads();
  } while (true);
}

// Decode: 64 streams per block (one wave) and 40 KiB of LDS per block, so
// the four blocks of a CU's four SIMDs fit its 160 KiB.  The block's 64
// streams are adjacent in the byte buffer; their CDF rows and (up to the
// window size) their bytes are staged into LDS with coalesced 16-byte
// loads, so the per-symbol loop touches no global memory except for
// streams that do not fit the window.
//
// Symbol lookup (rule L6) is table driven, with per-stream tables built in
// LDS from the staged rows.  n_bins <= 32 takes cgdec::ByteTables: one byte
// per 8-bit window prefix, so every code of at most 8 bits (all of them for
// chunks of up to 256 tokens) is one LDS read, and the table is built
// without data-dependent loops.  Larger n_bins take DecTables below.  Bases
// are multiples of 16, so the top 12 bits of the 16-bit window decide the
// symbol.  DecTables' L1 has one entry per 7-bit prefix: symbol | length <<
// 8 when one symbol owns the prefix's whole range; 0x8000 | k << 8 |
// s_first when symbol boundaries fall inside it, k naming one of the
// stream's kSubTables L2 tables whose 32 one-byte entries (next 5 bits)
// hold (s - s_first) << 4 | length; and kOverflow when the stream ran out
// of L2 tables (or a prefix spans more than 16 symbols), which falls back
// to a binary search over the bases.
constexpr int kDecLanes = cgdec::kLanes;
#ifndef LMC_DEC_LANES
#define LMC_DEC_LANES 1  // per-lane stream regions for n_bins <= 32
#endif
constexpr int kDirectBits = 7;
constexpr int kSubBits = 5;
constexpr int kSubTables = 4;
constexpr uint32_t kOverflow = 0xFFFFu;
constexpr int kDecLds = 40 * 1024;
constexpr int kL1Bytes = (1 << kDirectBits) * kDecLanes * 2;
constexpr int kL2Bytes = kSubTables * (1 << kSubBits) * kDecLanes;
constexpr int kObufBytes = 4 * kDecLanes;
static_assert(kObufBytes >= 256, "the byte table build writes past the table into the 256 bytes after it");
constexpr int kRowChunks = 5;   // 16-byte row chunks per lane and load batch (33 x 64 x 2 B)
constexpr int kWinChunks = 12;  // 16-byte window chunks per lane and load batch (12 KiB)

// Loads up to kDecLanes * N 16-byte chunks [j0, j0 + 64 N) of a run of n
// chunks at the 16-byte aligned global address src into registers, one
// chunk per lane and slot; indexes past the run are clamped to its last
// chunk (n >= 1).
// Global (not flat) loads: they are counted by vmcnt alone and return in
// order, so a store of an early chunk waits only for the loads before it.
typedef uint32_t chunk16 __attribute__((ext_vector_type(4)));
using global_chunk16 = const __attribute__((address_space(1))) chunk16;

template <int N>
__device__ __forceinline__ void load_chunks(uintptr_t src, int n, int j0, int lane, chunk16 (&v)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int j = j0 + k * kDecLanes + lane;
    v[k] = reinterpret_cast<global_chunk16 *>(src)[j < n ? j : n - 1];
  }
}

// Stores the chunks of load_chunks to LDS at dst (several lanes may store
// the same clamped last chunk, with the same bytes); kSwap byte-reverses
// each dword (the big-endian order of the stream bits).
template <bool kSwap, int N>
__device__ __forceinline__ void store_chunks(uint8_t *dst, int n, int j0, int lane, const chunk16 (&v)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int j = j0 + k * kDecLanes + lane;
    chunk16 w = v[k];
    if (kSwap) {
      w.x = __builtin_bswap32(w.x);
      w.y = __builtin_bswap32(w.y);
      w.z = __builtin_bswap32(w.z);
      w.w = __builtin_bswap32(w.w);
    }
    reinterpret_cast<chunk16 *>(dst)[j < n ? j : n - 1] = w;
  }
}

using cgdec::StagedRow;

// Per-lane decode tables: L1 and L2 columns of stride kDecLanes.
struct DecTables {
  static constexpr int kBytes = kL1Bytes + kL2Bytes;
  uint16_t *l1;
  uint8_t *l2;
  StagedRow row;
  int nb;
  int top;  // largest power of two below nb (1 if nb <= 2)

  __device__ __forceinline__ void bind(uint8_t *lds, int lane) {
    l1 = reinterpret_cast<uint16_t *>(lds) + lane;
    l2 = lds + kL1Bytes + lane;
  }

  // Builds L1/L2 from the staged row in one pass over the symbols (a loop
  // every lane runs in step).  Symbol s owns the windows [lo, hi): lo is
  // its base (0 for s = 0, which also takes windows below the first base),
  // hi the next base.  Prefixes entirely inside [lo, hi) get a direct
  // entry; a prefix holding a boundary is opened by the symbol covering its
  // start and filled by that symbol and the following ones.  Also finds
  // row.wrap.
  __device__ __forceinline__ void clear() {}   // build() writes every entry
  __device__ __forceinline__ void finish() {}  // build() sets row.wrap and top

  __device__ __forceinline__ void build(uint8_t *) {
    constexpr uint32_t span = 1u << (kPrec - kDirectBits);
    constexpr uint32_t sub = 1u << (kPrec - kDirectBits - kSubBits);
    row.wrap = nb;
    uint32_t raw = static_cast<uint16_t>(row.r[0]);
    uint32_t base = raw & 0xFFF0u;
    uint32_t last = base;  // last base before any wrap
    int open_k = -1, open_first = 0, nsub = 0;
    for (int s = 0; s < nb; ++s) {
      uint32_t next = 0x10000u, next_raw = 0;
      if (s + 1 < nb) {
        next_raw = static_cast<uint16_t>(row.r[s + 1]);
        const uint32_t nbase = next_raw & 0xFFF0u;
        if (row.wrap == nb && nbase >= last) {
          next = nbase;
          last = nbase;
        } else if (row.wrap == nb) {
          row.wrap = s + 1;
        }
      }
      int len = static_cast<int>(raw & 0xFu);
      if (len == 0) {
        const uint32_t w = next - base;
        if (w != 0) len = kPrec - (31 - __builtin_clz(w));
      }
      const uint32_t lo = s == 0 ? 0u : base, hi = next;
      if (hi > lo) {
        const uint32_t ent = static_cast<uint32_t>(s) | (static_cast<uint32_t>(len) << 8);
        uint32_t e = lo / span;
        if (lo % span) {  // inside a prefix opened by an earlier symbol
          if (open_k >= 0) {
            const int ds = s - open_first;
            if (ds > 15) {
              l1[e * kDecLanes] = static_cast<uint16_t>(kOverflow);
              open_k = -1;
            } else {
              const uint32_t j1 = hi - e * span < span ? (hi - e * span) / sub : span / sub;
              for (uint32_t j = (lo % span) / sub; j < j1; ++j)
                l2[(open_k * (1 << kSubBits) + j) * kDecLanes] =
                    static_cast<uint8_t>((ds << 4) | len);
            }
          }
          ++e;
        }
        for (; e < hi / span; ++e) l1[e * kDecLanes] = static_cast<uint16_t>(ent);
        if ((hi % span) && lo <= hi - hi % span) {  // opens the prefix holding hi
          e = hi / span;
          if (nsub < kSubTables) {
            open_k = nsub++;
            open_first = s;
            l1[e * kDecLanes] = static_cast<uint16_t>(0x8000u | (open_k << 8) | s);
            for (uint32_t j = 0; j < (hi % span) / sub; ++j)
              l2[(open_k * (1 << kSubBits) + j) * kDecLanes] = static_cast<uint8_t>(len);
          } else {
            open_k = -1;
            l1[e * kDecLanes] = static_cast<uint16_t>(kOverflow);
          }
        }
      }
      raw = next_raw;
      base = next;
    }
    top = 1;
    while (top * 2 < nb) top *= 2;
  }

  // Symbol and code length for the 16-bit window v.
  __device__ __forceinline__ void lookup(uint32_t v, int &s, int &len) const {
    const uint32_t d = l1[(v >> (kPrec - kDirectBits)) * kDecLanes];
    if (d < 0x8000u) {
      s = static_cast<int>(d & 0xFFu);
      len = static_cast<int>(d >> 8);
    } else if (d != kOverflow) {
      const uint32_t j = (v >> (kPrec - kDirectBits - kSubBits)) & ((1u << kSubBits) - 1);
      const uint32_t x = l2[(((d >> 8) & 0x7Fu) * (1 << kSubBits) + j) * kDecLanes];
      s = static_cast<int>((d & 0xFFu) + (x >> 4));
      len = static_cast<int>(x & 0xFu);
    } else {
      s = 0;
      for (int step = top; step > 0; step >>= 1)
        if (s + step < nb && row.base(s + step) <= v) s += step;
      len = row.len(s);
    }
  }
};

// Bytes of the aligned dword at address `a` that lie in [lo, hi), as a mask
// over the dword's little-endian value.
__device__ __forceinline__ uint32_t live_mask(uintptr_t a, uintptr_t lo, uintptr_t hi) {
  const int64_t from = static_cast<int64_t>(lo) - static_cast<int64_t>(a);
  const int64_t to = static_cast<int64_t>(hi) - static_cast<int64_t>(a);
  const int f = from < 0 ? 0 : (from > 4 ? 4 : static_cast<int>(from));
  const int t = to < 0 ? 0 : (to > 4 ? 4 : static_cast<int>(to));
  const uint32_t below_t = t >= 4 ? ~0u : ((1u << (8 * t)) - 1u);
  const uint32_t below_f = f >= 4 ? ~0u : ((1u << (8 * f)) - 1u);
  return below_t & ~below_f;
}

// Big-endian dword of the staged window at byte offset q (a multiple of 4),
// with the bytes at or past `hi` (an offset too) zeroed.  The read is
// clamped to the window's last dword; whatever it returns past hi is
// masked off.
__device__ __forceinline__ uint32_t win_word(const uint32_t *win, uint32_t last, uint32_t q,
                                             uint32_t hi) {
  const uint32_t w = win[(q < last ? q : last) >> 2];
  const int t = static_cast<int>(hi) - static_cast<int>(q);
  const int k = t < 0 ? 0 : (t > 4 ? 4 : t);
  return k >= 4 ? w : (w & ~(~0u >> (8 * k)));
}

// Keeps the bytes of a big-endian dword at stream offset q that lie before
// the stream end `hi` (bytes at or past hi read as zero).
__device__ __forceinline__ uint32_t clip_word(uint32_t w, uint32_t q, uint32_t hi) {
  const int t = static_cast<int>(hi) - static_cast<int>(q);
  const int k = t < 0 ? 0 : (t > 4 ? 4 : t);
  return k >= 4 ? w : (w & ~(~0u >> (8 * k)));
}

// Orders a wave's LDS writes before its later reads of other lanes' words.
// Decode blocks are one wave, and a wave's LDS accesses are performed in
// order, so no block barrier is needed.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// All 64 streams of the block lie in the window: L1/L2 lookups and symbols
// transposed through LDS so each lane stores one dword (4 channels of one
// token) per 4 tokens.  The bit window is refilled without branches: every
// symbol reads the window dword at q (the next one to append) alongside its
// L1 read, and the following symbol appends it when 32 bits or fewer are
// left, so no LDS latency beyond the table lookup sits on the chain.
template <class Tab>
__device__ __forceinline__ void decode_block_fast(const Tab &tb, int T, int C,
                                                  const uint32_t *win, uint32_t win_last,
                                                  uint32_t lo, uint32_t hi, uint8_t *obuf,
                                                  uint32_t *__restrict__ odst) {
  const int lane = static_cast<int>(threadIdx.x);
  uint32_t q = lo & ~3u;
  uint64_t buf = static_cast<uint64_t>(clip_word(win[q >> 2], q, hi)) << 32;
  buf <<= 8 * (lo & 3u);
  int have = 32 - 8 * static_cast<int>(lo & 3u);
  q += 4;
  uint32_t nraw = win[(q < win_last ? q : win_last) >> 2];
  auto step = [&]() -> int {
    const bool refill = have <= 32;  // leaves more than 32 bits; codes are <= 15
    const uint32_t w = refill ? clip_word(nraw, q, hi) : 0u;
    buf |= static_cast<uint64_t>(w) << (refill ? 32 - have : 0);
    have += refill ? 32 : 0;
    q += refill ? 4u : 0u;
    int s, len;
    const uint32_t v = static_cast<uint32_t>(buf >> 48);
    nraw = win[(q < win_last ? q : win_last) >> 2];
    tb.lookup(v, s, len);
    buf <<= len;
    have -= len;
    return s;
  };
  // odst: DecBlock::quad, a full block.
  const int64_t step4 = static_cast<int64_t>(C);  // in dwords: 4 tokens of C bytes
  int t = 0;
  for (; t + 4 <= T; t += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) obuf[i * kDecLanes + lane] = static_cast<uint8_t>(step());
    wave_sync();
    cg_st(odst, reinterpret_cast<const uint32_t *>(obuf)[lane]);
    odst += step4;
    wave_sync();
  }
  if (t < T) {
    for (int i = 0; t + i < T; ++i) obuf[i * kDecLanes + lane] = static_cast<uint8_t>(step());
    wave_sync();
    if ((lane >> 4) < T - t) cg_st(odst, reinterpret_cast<const uint32_t *>(obuf)[lane]);
  }
}


// Fast path of the byte tables: every stream of the block lies in the window
// and no table entry is an escape, so each symbol is one LDS read and the
// loop has no branches (cgdec::BitCursor, cgdec::ByteTables::step).
// Symbols go through the 4-token LDS transpose as in decode_block_fast.
__device__ __forceinline__ void decode_block_bytes(const cgdec::ByteTables &tb, int T, int C,
                                                   const uint32_t *win, uint32_t win_last,
                                                   uint32_t lo, uint32_t hi, uint8_t *obuf,
                                                   uint32_t *__restrict__ odst) {
  const int lane = static_cast<int>(threadIdx.x);
  cgdec::BitCursor cur;
  cur.start(win, win_last, 8 * lo, hi);
  auto step = [&]() -> uint32_t { return tb.step(cur) >> 3; };
  // odst: DecBlock::quad, a full block.
  const int64_t step4 = static_cast<int64_t>(C);  // in dwords: 4 tokens of C bytes
  int t = 0;
  for (; t + 4 <= T; t += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) obuf[i * kDecLanes + lane] = static_cast<uint8_t>(step());
    wave_sync();
    cg_st(odst, reinterpret_cast<const uint32_t *>(obuf)[lane]);
    odst += step4;
    wave_sync();
  }
  if (t < T) {
    for (int i = 0; t + i < T; ++i) obuf[i * kDecLanes + lane] = static_cast<uint8_t>(step());
    wave_sync();
    if ((lane >> 4) < T - t) cg_st(odst, reinterpret_cast<const uint32_t *>(obuf)[lane]);
  }
}

// Blocks whose streams all fit the window: byte tables without an escape
// entry in any lane take the branch-free loop, every other block the loop
// with the escape branch.
__device__ __forceinline__ void decode_fast(const cgdec::ByteTables &tb, int T, int C,
                                            const uint32_t *win, uint32_t win_last, uint32_t lo,
                                            uint32_t hi, uint8_t *obuf, uint32_t *__restrict__ odst) {
  if (__any(tb.escapes)) {
    cgdec::ByteTables t = tb;
    t.finish();
    decode_block_fast(t, T, C, win, win_last, lo, hi, obuf, odst);
  } else {
    decode_block_bytes(tb, T, C, win, win_last, lo, hi, obuf, odst);
  }
}

__device__ __forceinline__ void decode_fast(const DecTables &tb, int T, int C, const uint32_t *win,
                                            uint32_t win_last, uint32_t lo, uint32_t hi, uint8_t *obuf,
                                            uint32_t *__restrict__ odst) {
  decode_block_fast(tb, T, C, win, win_last, lo, hi, obuf, odst);
}

// One stream occupying [lo, hi) (addresses), symbols to o[0], o[C], ...
// kWin: every dword the stream needs is in the LDS window holding the bytes
// from a_lo to a_hi, read with the index clamped into the window.
// Otherwise dwords come from global memory, and only those holding a byte
// of [lo, hi) are read.
template <bool kWin, class Tab>
__device__ __forceinline__ void decode_stream(const Tab &tb, int T, int C,
                                              const uint8_t *__restrict__ bytes, const uint32_t *win,
                                              uintptr_t a_lo, uintptr_t a_hi, uintptr_t lo,
                                              uintptr_t hi, uint8_t *__restrict__ o) {
  const uintptr_t base0 = reinterpret_cast<uintptr_t>(bytes);
  auto word_at = [&](uintptr_t q) -> uint32_t {
    if (kWin) {
      const uint32_t last = static_cast<uint32_t>(a_hi - a_lo) - 4;
      return win_word(win, last, static_cast<uint32_t>(q - a_lo), static_cast<uint32_t>(hi - a_lo));
    }
    uint32_t raw = 0;
    if (q < hi) raw = *reinterpret_cast<const uint32_t *>(bytes + (q - base0));
    return __builtin_bswap32(raw & live_mask(q, lo, hi));
  };
  uintptr_t q = lo & ~uintptr_t(3);
  uint64_t buf = static_cast<uint64_t>(word_at(q)) << 32;
  q += 4;
  buf <<= 8 * (lo & 3);
  int have = 32 - 8 * static_cast<int>(lo & 3);
  for (int t = 0; t < T; ++t) {
    if (have <= 32) {
      buf |= static_cast<uint64_t>(word_at(q)) << (32 - have);
      have += 32;
      q += 4;
    }
    int s, len;
    tb.lookup(static_cast<uint32_t>(buf >> 48), s, len);
    o[static_cast<int64_t>(t) * C] = static_cast<uint8_t>(s);
    buf <<= len;
    have -= len;
  }
}

// The channels of a layer, and division by them with a multiplication (Granlund
// and Montgomery, "Division by invariant integers using multiplication",
// figure 4.1): a decode block finds its first stream's layer before its first
// load, and the compiler's division is about 40 dependent instructions there
// (64 planes x 256 tokens x 512 channels 18.2 -> 17.7 us; the encoder and
// calculate_cdf gain nothing from it).
struct Channels {
  int n;
  uint32_t mul, sh1, sh2;
  explicit Channels(int64_t c) : n(static_cast<int>(c)) {
    int l = 0;
    while ((int64_t(1) << l) < c) ++l;
    mul = static_cast<uint32_t>(((uint64_t((int64_t(1) << l) - c) << 32) / static_cast<uint64_t>(c)) + 1);
    sh1 = l < 1 ? l : 1;
    sh2 = l > 1 ? l - 1 : 0;
  }
  __device__ __forceinline__ uint32_t divide(uint32_t x) const {
    const uint32_t t = __umulhi(x, mul);
    return (t + ((x - t) >> sh1)) >> sh2;
  }
  __device__ __forceinline__ int64_t layer_of(int64_t s) const {
    return s < (int64_t(1) << 32) ? divide(static_cast<uint32_t>(s)) : s / n;
  }
};

// Layer and channel of a stream `k` streams after (l, c); streams are
// numbered over the layers, channels fastest.
struct StreamAt {
  int64_t l;
  int c;
};
__device__ __forceinline__ StreamAt stream_at(int64_t l, int c, uint32_t k, const Channels &chans) {
  const uint32_t x = static_cast<uint32_t>(c) + k;
  const uint32_t up = chans.divide(x);
  return {l + up, static_cast<int>(x - up * static_cast<uint32_t>(chans.n))};
}

// Inclusive prefix sum of 32-bit values over the 64 lanes of a wave, in 64
// bits (the sums of their halves fit 32).
__device__ __forceinline__ int64_t wave_incl_scan_wide(uint32_t v) {
  return (static_cast<int64_t>(wave_incl_scan(v >> 16)) << 16) + wave_incl_scan(v & 0xFFFFu);
}

// Where the streams lie in the byte buffer: inclusive prefix sums of their
// lengths, or (prefix null) the lengths with the sums length_sums_kernel
// makes of them.  Prefix sums and 32-bit sums give a stream's end as the same
// int32, the sum of the lengths up to it modulo 2^32; buffers of 2 GiB and
// more take 64-bit sums.
struct StreamEnds {
  const int32_t *prefix;
  const int32_t *lens;
  const uint32_t *sums;    // [64-stream blocks]: lengths before the block in its group of 64 blocks
  const uint32_t *groups;  // [groups]: lengths of a group
  const int64_t *wide_sums, *wide_groups;  // the same in 64 bits, in place of the 32-bit ones
};
constexpr int kSumThreads = 1024;
constexpr int kGroupBlocks = 64;  // 64-stream blocks per group

// Stream geometry of one decode block: lane i of a wave owns stream
// s0 + i; bytes of the block's streams are [B0, B1) of the byte buffer.
struct DecBlock {
  int cnt;  // streams of the block: 64 but for the last
  int64_t s0, start, end, B0, B1;
  int64_t l0;  // layer and channel of stream s0
  int c0;
  uintptr_t R0, R1, r_lo;

  __device__ __forceinline__ void init(const int16_t *cdf, int64_t nbytes, const StreamEnds &ends,
                                       int64_t n_streams, const Channels &chans, int nb, int lane) {
    s0 = static_cast<int64_t>(blockIdx.x) * kDecLanes;
    l0 = chans.layer_of(s0);
    c0 = static_cast<int>(s0 - l0 * chans.n);
    cnt = n_streams - s0 < kDecLanes ? static_cast<int>(n_streams - s0) : kDecLanes;
    const int64_t stream = s0 + (lane < cnt ? lane : 0);
    auto clampb = [&](int64_t x) { return x < 0 ? 0 : (x > nbytes ? nbytes : x); };
    if (ends.prefix != nullptr) {
      start = clampb(stream == 0 ? 0 : ends.prefix[stream - 1]);
      end = clampb(ends.prefix[stream]);
      B0 = clampb(s0 == 0 ? 0 : ends.prefix[s0 - 1]);
      B1 = clampb(ends.prefix[s0 + cnt - 1]);
    } else if (ends.wide_sums != nullptr) {
      const int32_t len = lane < cnt ? max(ends.lens[stream], 0) : 0;
      int64_t part = 0;
      for (int64_t g = lane; g < static_cast<int64_t>(blockIdx.x) / kGroupBlocks; g += kDecLanes)
        part += ends.wide_groups[g];
#pragma unroll
      for (int d = 1; d < kDecLanes; d <<= 1) part += __shfl_xor(part, d, kDecLanes);
      const int64_t base = ends.wide_sums[blockIdx.x] + part;
      const int64_t incl = wave_incl_scan_wide(static_cast<uint32_t>(len));
      start = clampb(base + incl - len);
      end = clampb(base + incl);
      B0 = clampb(base);
      B1 = clampb(base + __shfl(incl, kDecLanes - 1, kDecLanes));
    } else {
      const uint32_t len = lane < cnt ? static_cast<uint32_t>(ends.lens[stream]) : 0u;
      uint32_t base = ends.sums[blockIdx.x];
      const int group = static_cast<int>(blockIdx.x) / kGroupBlocks;
      uint32_t part = 0;
      for (int g = lane; g < group; g += kDecLanes) part += ends.groups[g];
      const uint32_t incl = wave_incl_scan(len);
      base += static_cast<uint32_t>(
          __builtin_amdgcn_readlane(static_cast<int>(wave_incl_scan(part)), kDecLanes - 1));
      const uint32_t all = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), kDecLanes - 1));
      auto at = [&](uint32_t x) { return clampb(static_cast<int32_t>(base + x)); };
      start = at(incl - len);
      end = at(incl);
      B0 = at(0);
      B1 = at(all);
    }
    end = end < start || lane >= cnt ? start : end;
    // Rows: bytes [R0, R1) from the 16-byte aligned address at or below R0.
    R0 = reinterpret_cast<uintptr_t>(cdf + s0 * (nb + 1));
    R1 = R0 + static_cast<uintptr_t>(cnt) * (nb + 1) * 2;
    r_lo = R0 & ~uintptr_t(15);
  }

  // The transposed symbols of four tokens are stored as dwords: lane j's is
  // dword `at` of the transpose (token at / 16 of the four, streams
  // 4 * (at % 16) .. + 3, of one layer: C % 4 == 0), stored at `dst` for the
  // first four tokens.  `at` is j in a full block; in a block of 32 streams
  // (C % 32 == 0, so there is no other) the upper eight dwords of a token
  // repeat the lower eight, so that no store is predicated.
  struct Quad {
    int at;
    uint32_t *dst;
  };
  __device__ __forceinline__ Quad quad(uint8_t *out, int T, const Channels &chans, int lane) const {
    const int at = cnt == kDecLanes ? lane : lane & 0x37;
    const StreamAt a = stream_at(l0, c0, 4u * static_cast<uint32_t>(at & 15), chans);
    return {at, reinterpret_cast<uint32_t *>(out + (a.l * T + (at >> 4)) * chans.n + a.c)};
  }

  // 16-byte chunks of the window staged from a_lo: the block's bytes from
  // the 16-byte aligned address at or below B0, at most cap bytes.  Every
  // chunk staged (rows or window) holds a byte of its range, so no load
  // leaves the buffers' pages.
  __device__ __forceinline__ int win_chunks(uintptr_t base0, uintptr_t a_lo, int cap) const {
    if (B1 <= B0) return 0;
    const uintptr_t want = base0 + B1 - a_lo;
    const uintptr_t c = static_cast<uintptr_t>(cap);
    return static_cast<int>(((want < c ? want : c) + 15) >> 4);
  }
};

// One wave decodes the block's 64 streams, one lane per stream.
// LDS: [tables][obuf: 4 tokens x 64 lanes][staged rows][byte window].
template <class Tab>
__device__ __forceinline__ void decode_one_wave(uint8_t *lds, const int16_t *__restrict__ cdf,
                                                const uint8_t *__restrict__ bytes, int64_t nbytes,
                                                const StreamEnds ends, int T, const Channels &chans,
                                                int nb, uint8_t *__restrict__ out, int64_t n_streams,
                                                int lane) {
  const int C = chans.n;
  constexpr int kRowsOff = Tab::kBytes + kObufBytes;
  const int rows_cap = ((nb + 1) * kDecLanes * 2 + 32 + 15) & ~15;
  const int win_off = kRowsOff + rows_cap;
  const int win_cap = (kDecLds - win_off) & ~15;
  DecBlock bk;
  bk.init(cdf, nbytes, ends, n_streams, chans, nb, lane);
  const int live = lane < bk.cnt;
  const uintptr_t base0 = reinterpret_cast<uintptr_t>(bytes);
  const uintptr_t a_lo = (base0 + bk.B0) & ~uintptr_t(15);
  const int n16 = bk.win_chunks(base0, a_lo, win_cap);
  const int nrow = static_cast<int>((bk.R1 - bk.r_lo + 15) >> 4);
  // The rows' loads are issued first and the window's behind them; the
  // table is built from the stored rows while the window is in flight.
  chunk16 rv[kRowChunks], wv[kWinChunks];
  load_chunks(bk.r_lo, nrow, 0, lane, rv);
  // Without a window the rows' first chunk is loaded and dropped, so no
  // branch separates these loads from the row stores that wait for rv only.
  load_chunks(n16 > 0 ? a_lo : bk.r_lo, n16 > 0 ? n16 : 1, 0, lane, wv);
  Tab tb;
  tb.bind(lds, lane);
  tb.clear();
  store_chunks<false>(lds + kRowsOff, nrow, 0, lane, rv);
  for (int j0 = kDecLanes * kRowChunks; j0 < nrow; j0 += kDecLanes * kRowChunks) {
    load_chunks(bk.r_lo, nrow, j0, lane, rv);
    store_chunks<false>(lds + kRowsOff, nrow, j0, lane, rv);
  }
  wave_sync();
  tb.row.r = reinterpret_cast<const int16_t *>(lds + kRowsOff + (bk.R0 - bk.r_lo)) + lane * (nb + 1);
  tb.nb = nb;
  if (live) tb.build(lds + Tab::kBytes + lane);  // obuf byte: scratch for skipped writes
  if (n16 > 0) {
    store_chunks<true>(lds + win_off, n16, 0, lane, wv);
    for (int j0 = kDecLanes * kWinChunks; j0 < n16; j0 += kDecLanes * kWinChunks) {
      load_chunks(a_lo, n16, j0, lane, wv);
      store_chunks<true>(lds + win_off, n16, j0, lane, wv);
    }
  }
  wave_sync();
  const uintptr_t lo = base0 + static_cast<uintptr_t>(bk.start);
  const uintptr_t hi = base0 + static_cast<uintptr_t>(bk.end);
  const uintptr_t a_hi = a_lo + 16 * static_cast<uintptr_t>(n16);
  const bool in_win = hi > lo && (lo & ~uintptr_t(3)) >= a_lo && ((hi + 3) & ~uintptr_t(3)) <= a_hi;
  const bool fast = bk.cnt == kDecLanes && (reinterpret_cast<uintptr_t>(out) & 3) == 0 && (C & 3) == 0 &&
                    __all(in_win);
  if (!live) return;
  const uint32_t *win = reinterpret_cast<const uint32_t *>(lds + win_off);
  if (fast) {
    uint32_t *odst = bk.quad(out, T, chans, lane).dst;  // a full block
    decode_fast(tb, T, C, win, static_cast<uint32_t>(a_hi - a_lo) - 4,
                static_cast<uint32_t>(lo - a_lo), static_cast<uint32_t>(hi - a_lo),
                lds + Tab::kBytes, odst);
  } else {
    tb.finish();
    const StreamAt at = stream_at(bk.l0, bk.c0, static_cast<uint32_t>(lane), chans);
    uint8_t *o = out + at.l * T * C + at.c;
    if (in_win)
      decode_stream<true>(tb, T, C, bytes, win, a_lo, a_hi, lo, hi, o);
    else
      decode_stream<false>(tb, T, C, bytes, win, a_lo, a_hi, lo, hi, o);
  }
}

// The streams of a block from their regions, for tables without escapes.
// Four tokens per group (cgdec::GroupCursor): the four table entries go
// through the LDS transpose and the symbols of the resulting word are
// extracted at once, (word >> 3) & 0x1F1F1F1F; each word is stored one
// group late, so no group waits for its own transpose read.  The
// transpose writes, that store and the transposing read sit between the
// group's codes, each under a table read (the cursor's scheduling
// barriers keep them there).  Measured on MI355X (symbol loop, shader
// cycles per symbol, s_memtime stamps): 128-133 with the refilled lane
// cursor (its chain four VALU instructions and the table read, the
// refill on it every fourth code) -> 112 with this cursor -> 102 with
// the transpose spread between the codes -> 100 with the window's
// permutations one code later.  The chain alone, timed in isolation,
// takes 72 cycles; the rest is issue of the other instructions under
// it and LDS traffic.
__device__ __forceinline__ void decode_groups(const cgdec::ByteTables &tb, const uint32_t *region, uint32_t region_at,
                                              uint32_t off, uint32_t len, uint8_t *obuf, const DecBlock::Quad &quad,
                                              int T, int C, int lane) {
  uint32_t *odst = quad.dst;
  const int64_t step4 = static_cast<int64_t>(C);  // in dwords: 4 tokens of C bytes
  cgdec::GroupCursor gc;
  gc.start(tb, region, region_at, off, len);
  int t = 0;
  uint32_t word = 0;
  for (; t + 4 <= T; t += 4) {
    const uint32_t e0 = gc.step0(tb);
    const uint32_t e1 = gc.step1(tb);
    obuf[lane] = static_cast<uint8_t>(e0);
    if (t > 0) {
      cg_st(odst, (word >> 3) & 0x1F1F1F1Fu);
      odst += step4;
    }
    const uint32_t e2 = gc.step2(tb);
    obuf[kDecLanes + lane] = static_cast<uint8_t>(e1);
    const uint32_t e3 = gc.step3(tb);
    obuf[2 * kDecLanes + lane] = static_cast<uint8_t>(e2);
    obuf[3 * kDecLanes + lane] = static_cast<uint8_t>(e3);
    wave_sync();
    word = reinterpret_cast<const uint32_t *>(obuf)[quad.at];
    wave_sync();
  }
  if (t > 0) {
    cg_st(odst, (word >> 3) & 0x1F1F1F1Fu);
    odst += step4;
  }
  if (t < T) {
    for (int i = 0; t + i < T; ++i) obuf[i * kDecLanes + lane] = static_cast<uint8_t>(gc.single(tb));
    wave_sync();
    if ((quad.at >> 4) < T - t) cg_st(odst, reinterpret_cast<const uint32_t *>(obuf)[quad.at]);
  }
}

// Byte tables with per-lane stream regions (cgdec::LaneRegion): each lane
// stages the 16-byte aligned chunks holding its own stream into its own LDS
// region and zeroes what lies past the stream's end, so the cursors read
// the region without masking the stream's end: cgdec::GroupCursor for
// tables without escapes (four codes per group, windows re-read from the
// region on a fixed schedule), cgdec::LaneCursor for the others.  The 256
// bytes after the table (obuf) are scratch while the table is built.
// Serves full 64-stream blocks with dword-aligned output rows whose regions
// fit the LDS left after the tables and rows; returns false, having written
// nothing, for any other block, which then takes decode_one_wave.
__device__ __forceinline__ bool decode_one_wave_lanes(uint8_t *lds, const int16_t *__restrict__ cdf,
                                                      const uint8_t *__restrict__ bytes, int64_t nbytes,
                                                      const StreamEnds ends, int T, const Channels &chans, int nb,
                                                      uint8_t *__restrict__ out, int64_t n_streams,
                                                      int lane) {
  using Tab = cgdec::ByteTables;
  const int C = chans.n;
  constexpr int kRowsOff = Tab::kBytes + kObufBytes;
  constexpr int kLaneBatch = 8;  // 16-byte chunks per lane and load batch
  const int rows_cap = ((nb + 1) * kDecLanes * 2 + 32 + 15) & ~15;
  const int reg_off = kRowsOff + rows_cap;
  const uint32_t reg_cap = static_cast<uint32_t>((kDecLds - reg_off) & ~15);
  // LDS address of the block's table (the start of the kernel's dynamic
  // LDS); the table step ORs a dword offset into it.
  const uint32_t lds_at =
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t *)lds));
  DecBlock bk;
  bk.init(cdf, nbytes, ends, n_streams, chans, nb, lane);
  if ((reinterpret_cast<uintptr_t>(out) & 3) != 0 || (C & 3) != 0 || (lds_at & (Tab::kBytes - 1)) != 0)
    return false;
  // The rows' loads depend on the block alone: issued before the stream
  // lengths (prefix loads) are waited for.
  const int nrow = static_cast<int>((bk.R1 - bk.r_lo + 15) >> 4);
  chunk16 rv[kRowChunks], cv[kLaneBatch];
  load_chunks(bk.r_lo, nrow, 0, lane, rv);
  const uintptr_t base0 = reinterpret_cast<uintptr_t>(bytes);
  const uintptr_t s_lo = base0 + static_cast<uintptr_t>(bk.start);
  const uintptr_t s_hi = base0 + static_cast<uintptr_t>(bk.end);
  const uint32_t len = static_cast<uint32_t>(bk.end - bk.start);
  const uintptr_t a0 = s_lo & ~uintptr_t(15);
  // Chunks [a0, a0 + 16 n_ch) each hold a byte of the stream, so no load
  // leaves the buffer's pages.
  const uint32_t n_ch = len ? static_cast<uint32_t>(((s_hi - 1) >> 4) - (s_lo >> 4) + 1) : 0u;
  // Chunks plus the sealed room; at most one byte more than there is, so that
  // the sum of the lanes' cannot wrap.
  const uint32_t rbytes = min(16u * n_ch + cgdec::LaneRegion::kRoom, reg_cap + 1u);
  uint32_t incl = rbytes, n_max = n_ch;
#pragma unroll
  for (int d = 1; d < kDecLanes; d <<= 1) {
    const uint32_t v = __shfl_up(incl, d, kDecLanes);
    incl += lane >= d ? v : 0u;
    const uint32_t m = __shfl_xor(n_max, d, kDecLanes);
    n_max = m > n_max ? m : n_max;
  }
  const uint32_t total = __shfl(incl, kDecLanes - 1, kDecLanes);
  if (total > reg_cap) return false;
  uint8_t *region = lds + reg_off + (incl - rbytes);
  Tab tb;
  tb.bind(lds, lane, lds_at);
  tb.clear();
  store_chunks<false>(lds + kRowsOff, nrow, 0, lane, rv);
  for (int j0 = kDecLanes * kRowChunks; j0 < nrow; j0 += kDecLanes * kRowChunks) {
    load_chunks(bk.r_lo, nrow, j0, lane, rv);
    store_chunks<false>(lds + kRowsOff, nrow, j0, lane, rv);
  }
  // The first batch of the lane's chunks, issued once the rows have landed
  // (every wave of the launch loads its rows and streams at its start, so
  // the rows, which the table build needs first, do not share the memory
  // system with the larger streams); the table is built while the chunks
  // are in flight.
#pragma unroll
  for (int u = 0; u < kLaneBatch; ++u)
    if (static_cast<uint32_t>(u) < n_ch) cv[u] = reinterpret_cast<global_chunk16 *>(a0)[u];
  wave_sync();
  // A lane without a stream (the last block) decodes stream s0's row over an
  // empty region and stores nothing.
  tb.row.r = reinterpret_cast<const int16_t *>(lds + kRowsOff + (bk.R0 - bk.r_lo)) +
             (lane < bk.cnt ? lane : 0) * (nb + 1);
  tb.nb = nb;
  tb.build(lds + Tab::kBytes + lane);  // obuf byte: scratch for skipped writes
#pragma unroll
  for (int u = 0; u < kLaneBatch; ++u)
    if (static_cast<uint32_t>(u) < n_ch) reinterpret_cast<chunk16 *>(region)[u] = cv[u];
  for (uint32_t k0 = kLaneBatch; k0 < n_max; k0 += kLaneBatch) {
#pragma unroll
    for (int u = 0; u < kLaneBatch; ++u)
      if (k0 + u < n_ch) cv[u] = reinterpret_cast<global_chunk16 *>(a0)[k0 + u];
#pragma unroll
    for (int u = 0; u < kLaneBatch; ++u)
      if (k0 + u < n_ch) reinterpret_cast<chunk16 *>(region)[k0 + u] = cv[u];
  }
  uint32_t *reg32 = reinterpret_cast<uint32_t *>(region);
  cgdec::LaneRegion::seal(reg32, static_cast<uint32_t>(s_lo - a0), len);
  uint8_t *obuf = lds + Tab::kBytes;
  const DecBlock::Quad quad = bk.quad(out, T, chans, lane);
  uint32_t *odst = quad.dst;
  const int64_t step4 = static_cast<int64_t>(C);  // in dwords: 4 tokens of C bytes
  if (!__any(tb.escapes)) {
    decode_groups(tb, reg32, lds_at + static_cast<uint32_t>(region - lds), static_cast<uint32_t>(s_lo - a0), len, obuf, quad,
                  T, C, lane);
  } else {
    tb.finish();
    cgdec::LaneCursor cur;
    cur.start(reg32, static_cast<uint32_t>(s_lo - a0), len);
    auto step = [&]() -> uint8_t {
      int s, l;
      tb.lookup(cur.top16(), s, l);
      cur.consume(l);
      cur.refill();
      return static_cast<uint8_t>(s);
    };
    int t = 0;
    for (; t + 4 <= T; t += 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) obuf[i * kDecLanes + lane] = step();
      wave_sync();
      cg_st(odst, reinterpret_cast<const uint32_t *>(obuf)[quad.at]);
      odst += step4;
      wave_sync();
    }
    if (t < T) {
      for (int i = 0; t + i < T; ++i) obuf[i * kDecLanes + lane] = step();
      wave_sync();
      if ((quad.at >> 4) < T - t) cg_st(odst, reinterpret_cast<const uint32_t *>(obuf)[quad.at]);
    }
  }
  return true;
}

template <class Tab>
__global__ void __launch_bounds__(kDecLanes)
    decode_kernel(const int16_t *__restrict__ cdf,
                  const uint8_t *__restrict__ bytes, int64_t nbytes,
                  const StreamEnds ends, int T, const Channels chans, int nb,
                  uint8_t *__restrict__ out, int64_t n_streams) {
  extern __shared__ uint32_t lds_words[];
  uint8_t *lds = reinterpret_cast<uint8_t *>(lds_words);
  const int lane = static_cast<int>(threadIdx.x);
  if constexpr (std::is_same<Tab, cgdec::ByteTables>::value) {
    if (LMC_DEC_LANES && decode_one_wave_lanes(lds, cdf, bytes, nbytes, ends, T, chans, nb, out, n_streams, lane))
      return;
  }
  decode_one_wave<Tab>(lds, cdf, bytes, nbytes, ends, T, chans, nb, out, n_streams, lane);
}

// Decode of chunks of more than kLaneMaxT tokens (n_bins <= 32).  Codes are
// looked up in cgdec::LongTables (chunks of more than 256 tokens have codes
// of up to 12 bits) and the streams are read through per-lane rings
// (cgdec::RingCursorT), so the LDS this takes does not grow with the streams.
// The line is at 256 tokens because calculate_cdf's codes are at most 8 bits
// long up to there, which the byte tables and lane regions of decode_kernel
// hold whole.
constexpr int kLaneMaxT = 256;
constexpr int kLongRing = cgdec::LongTables::kBytes;

// A lane's stream in 16-byte aligned chunks from a0; `end` is the stream's
// end from a0 in bytes.  Chunks 0 .. n_ch - 1 each hold a byte of the stream,
// so no load leaves the buffer's pages.  Of a longer stream kMost bytes count,
// so that positions fit an int; a chunk's codes (calculate_cdf takes fewer
// than 2^26 tokens) end below 2^27 bytes.
struct LaneChunks {
  static constexpr uint32_t kMost = 0x7FFFFFE0u;
  uintptr_t a0;
  uint32_t off, end, n_ch;

  __device__ __forceinline__ LaneChunks(const uint8_t *bytes, const DecBlock &bk) {
    const uintptr_t s_lo = reinterpret_cast<uintptr_t>(bytes) + static_cast<uintptr_t>(bk.start);
    const uint32_t len = min(static_cast<uint32_t>(bk.end - bk.start), kMost);
    a0 = s_lo & ~uintptr_t(15);
    off = static_cast<uint32_t>(s_lo - a0);
    end = off + len;
    n_ch = len ? (end + 15u) >> 4 : 0u;
  }
  __device__ __forceinline__ uint32_t len() const { return end - off; }
  __device__ __forceinline__ chunk16 load(uint32_t k) const {
    chunk16 v = {0u, 0u, 0u, 0u};
    if (k < n_ch) v = reinterpret_cast<global_chunk16 *>(a0)[k];
    return v;
  }
  // Chunk k, its bytes past the stream's end zero, to slot `slot` of a ring
  // of `dwords` dwords.
  __device__ __forceinline__ void put(uint32_t *ring, uint32_t dwords, uint32_t slot, uint32_t k,
                                      const chunk16 &v) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int left = static_cast<int>(end) - static_cast<int>(16u * k) - 4 * i;
      const uint32_t x = i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
      const uint32_t keep = left >= 4 ? ~0u : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
      ring[((4u * slot + static_cast<uint32_t>(i)) & (dwords - 1u)) * kDecLanes] = x & keep;
    }
  }
};

// The 4 x 64 transpose in registers: each lane holds the low bytes of its
// stream's four tokens; dword `at` of the transpose (DecBlock::Quad) is byte
// at / 16 of the lanes 4 * (at % 16) .. + 3.  send() issues the exchanges,
// take() puts the dword together.
struct LaneTranspose {
  int from;            // 4 x the first of the four lanes
  uint32_t sel;        // byte permutation: a byte of either operand
  uint32_t r0, r1, r2, r3;
  __device__ __forceinline__ explicit LaneTranspose(int at)
      : from(16 * (at & 15)), sel(0x0C0C0400u + 0x0101u * static_cast<uint32_t>(at >> 4)), r0(0), r1(0), r2(0), r3(0) {}
  __device__ __forceinline__ void send(uint32_t e0, uint32_t e1, uint32_t e2, uint32_t e3) {
    const uint32_t lo = cgdec::byte_perm(e1, e0, 0x0C0C0400u), hi = cgdec::byte_perm(e3, e2, 0x0C0C0400u);
    const int four = static_cast<int>(lo | (hi << 16));
    r0 = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from, four));
    r1 = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from + 4, four));
    r2 = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from + 8, four));
    r3 = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from + 12, four));
  }
  __device__ __forceinline__ uint32_t take() const {
    return cgdec::byte_perm(r1, r0, sel) | (cgdec::byte_perm(r3, r2, sel) << 16);
  }
};

// One wave decodes a block's streams, one lane per stream.  It takes kEpoch
// tokens at a time: the chunks that refill the ring over an epoch are loaded
// at its start and stored at its end, so nothing waits for them.  A ring
// holds 128 bytes; kEpoch codes of at most 16 bits take 32 of them, and an
// epoch loads as many chunks as there is room for, up to 32 bytes, so at
// least 80 bytes lie ahead of the cursor at the start of every epoch.
// `irregular`: some row of the block takes the binary search.
// Bound by the serial chain of each stream, about 210 cycles a code.
constexpr int kEpoch = 16;
constexpr int kEpochChunks = 2;  // 16-byte chunks per lane and epoch
constexpr int kFirstChunks = 8;

__device__ __forceinline__ void decode_serial(cgdec::LongTables &tb, bool irregular, const DecBlock &bk,
                                              const LaneChunks &ch, uint8_t *lds, uint32_t lds_at, int ring_off,
                                              int T, const Channels &chans, int lane, uint8_t *__restrict__ out) {
  const int C = chans.n;
  uint32_t *ring = reinterpret_cast<uint32_t *>(lds + ring_off) + lane;
  constexpr uint32_t kRingDw = cgdec::RingCursor::kBytes / 4;
  {
    chunk16 cv[kFirstChunks];
#pragma unroll
    for (uint32_t u = 0; u < kFirstChunks; ++u) cv[u] = ch.load(u);
#pragma unroll
    for (uint32_t u = 0; u < kFirstChunks; ++u) ch.put(ring, kRingDw, u, u, cv[u]);
  }
  uint32_t filled = kFirstChunks;  // chunks in the ring or before it
  wave_sync();
  const DecBlock::Quad quad = bk.quad(out, T, chans, lane);
  uint32_t *odst = quad.dst;
  const int64_t step4 = static_cast<int64_t>(C);  // in dwords: 4 tokens of C bytes
  const int groups = (T + 3) / 4;
  const uint32_t column = lds_at + static_cast<uint32_t>(ring_off) + 4u * static_cast<uint32_t>(lane);
  chunk16 nv[kEpochChunks];
  uint32_t room = 0;
  auto load_epoch = [&](uint32_t q) {
    room = (cgdec::RingCursor::kBytes - (16u * filled - q)) >> 4;
    room = room < kEpochChunks ? room : kEpochChunks;
#pragma unroll
    for (uint32_t u = 0; u < kEpochChunks; ++u) nv[u] = ch.load(u < room ? filled + u : ~0u);
  };
  auto store_epoch = [&]() {
#pragma unroll
    for (uint32_t u = 0; u < kEpochChunks; ++u)
      if (u < room) ch.put(ring, kRingDw, filled + u, filled + u, nv[u]);
    filled += room;
    wave_sync();
  };
  if (!irregular) {
    cgdec::PairCursor cur;
    cur.start(tb, column, 8u * ch.off);
    LaneTranspose tr(quad.at);
    // Four tokens; each transposed word is stored one group late, as in
    // decode_groups.
    auto group = [&](bool store_prev) {
      uint32_t e0, e1, e2, e3;
      cur.pair(tb, e0, e1);
      if (store_prev) {
        cg_st(odst, (tr.take() >> 3) & 0x1F1F1F1Fu);
        odst += step4;
      }
      cur.pair(tb, e2, e3);
      tr.send(e0, e1, e2, e3);
    };
    constexpr int kGroups = kEpoch / 4;
    int g = 0;
    for (; g + kGroups <= groups; g += kGroups) {
      load_epoch(cur.ring.q);
#pragma unroll
      for (int i = 0; i < kGroups; ++i) group(i > 0 || g > 0);
      store_epoch();
    }
    for (; g < groups; ++g) group(g > 0);
    if ((quad.at >> 4) < T - 4 * (groups - 1)) cg_st(odst, (tr.take() >> 3) & 0x1F1F1F1Fu);
  } else {
    tb.one.finish();
    LaneTranspose tr(quad.at);
    cgdec::RingCursor cur;
    cur.start(column, 8u * ch.off);
    for (int g = 0; g < groups; ++g) {
      if (g % (kEpoch / 4) == 0) load_epoch(cur.q);
      uint32_t sym[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int x, n;
        tb.search(cur.hi() >> 16, x, n);
        sym[i] = static_cast<uint32_t>(x);
        cur.advance(static_cast<uint32_t>(n));
      }
      tr.send(sym[0], sym[1], sym[2], sym[3]);
      if ((quad.at >> 4) < T - 4 * g) cg_st(odst, tr.take());
      odst += step4;
      if (g % (kEpoch / 4) == kEpoch / 4 - 1) store_epoch();
    }
  }
}

// The lanes' regions (cgdec::LaneRegion), one after the other in `room` bytes
// of LDS: the lane's chunks and the sealed room behind them.  `at` is where
// the lane's starts, `most` the largest number of chunks of a lane.
struct Regions {
  uint32_t at, total, most, room;
  __device__ __forceinline__ Regions(const LaneChunks &ch, uint32_t lds_room, int lane) : room(lds_room) {
    // At most one byte more than there is, so that the sum cannot wrap.
    const uint32_t own = min(16u * ch.n_ch + cgdec::LaneRegion::kRoom, room + 1u);
    uint32_t incl = own;
    most = ch.n_ch;
#pragma unroll
    for (int d = 1; d < kDecLanes; d <<= 1) {
      const uint32_t v = __shfl_up(incl, d, kDecLanes);
      incl += lane >= d ? v : 0u;
      const uint32_t m = __shfl_xor(most, d, kDecLanes);
      most = m > most ? m : most;
    }
    total = __shfl(incl, kDecLanes - 1, kDecLanes);
    at = incl - own;
  }
  __device__ __forceinline__ bool fit() const { return total <= room; }
};

// A lane's chunks into its region: the first N (cv) are in registers, the
// others are loaded N at a time.  Seals the region.
template <int N>
__device__ __forceinline__ void fill_region(const LaneChunks &ch, uint32_t most, chunk16 (&cv)[N], uint8_t *region) {
#pragma unroll
  for (int u = 0; u < N; ++u)
    if (static_cast<uint32_t>(u) < ch.n_ch) reinterpret_cast<chunk16 *>(region)[u] = cv[u];
  for (uint32_t k0 = N; k0 < most; k0 += N) {
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (k0 + u < ch.n_ch) cv[u] = reinterpret_cast<global_chunk16 *>(ch.a0)[k0 + u];
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (k0 + u < ch.n_ch) reinterpret_cast<chunk16 *>(region)[k0 + u] = cv[u];
  }
  cgdec::LaneRegion::seal(reinterpret_cast<uint32_t *>(region), ch.off, ch.len());
}

// Whether the staged rows (16-byte chunks) may be of short codes only: bases
// at multiples of 256 and lengths of at most 8.
__device__ __forceinline__ bool short_rows(const uint8_t *rows, int nrow, int lane) {
  uint32_t off = 0;
#pragma unroll
  for (int k = 0; k < kRowChunks; ++k) {
    const int j = k * kDecLanes + lane;
    const chunk16 v = reinterpret_cast<const chunk16 *>(rows)[j < nrow ? j : nrow - 1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t x = i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;  // two entries
      off |= (x & 0x00F000F0u) | (((x & 0x000F000Fu) + 0x00070007u) & 0x00100010u);
    }
  }
  return !__any(off != 0);
}

// A block of short codes: the byte table holds them all and the streams lie in
// regions behind it (from kShortRegions on, over the second table and the
// rings), so that a code takes the group cursor's 100 cycles in place of the
// two tables' 210 (decode_fast_prefsum of 512 blocks of 300 tokens over four
// symbols 39 -> 22 us, of 224 blocks of 700 over 16 56 -> 37).  short_table builds the table (false if it has escapes
// after all), decode_short decodes; cv holds the lanes' first chunks.
constexpr int kShortRegions = cgdec::ByteTables::kBytes;
__device__ __forceinline__ bool short_table(cgdec::ByteTables &tb, uint8_t *obuf, int lane) {
  tb.build(obuf + lane);
  return !__any(tb.escapes);
}
__device__ __forceinline__ void decode_short(const cgdec::ByteTables &tb, const DecBlock &bk, const LaneChunks &ch,
                                             chunk16 (&cv)[kFirstChunks], const Regions &regions, uint8_t *lds,
                                             uint32_t lds_at, uint8_t *obuf, int T, const Channels &chans, int lane,
                                             uint8_t *__restrict__ out) {
  const uint32_t at = kShortRegions + regions.at;
  fill_region(ch, regions.most, cv, lds + at);
  decode_groups(tb, reinterpret_cast<const uint32_t *>(lds + at), lds_at + at, ch.off, ch.len(), obuf,
                bk.quad(out, T, chans, lane), T, chans.n, lane);
}

// The staged rows, at up to 15 bytes past a 16-byte boundary; a table build
// reads kMaxBins entries of a row whatever nb is.
constexpr int rows_lds_bytes(int nb) { return ((nb + 1) * kDecLanes * 2 + 32 + 2 * cgdec::ByteTables::kMaxBins + 15) & ~15; }

// LDS of decode_long_kernel: the two tables and the rings, 40 KiB, so that
// four blocks fit a CU (1024 blocks of 300 tokens: 41 us, and 77 with the three
// that 53 KiB left; fewer than 769 the same).  The staged rows lie in the rings' place until the
// tables are built (an irregular block's then move to the tables' place), and
// scratch for skipped writes, or the transpose of short codes, at its end.
constexpr int kLongObuf = kDecLds - kObufBytes;
static_assert(kLongRing + static_cast<int>(cgdec::RingCursor::kBytes) * kDecLanes == kDecLds, "rings end the LDS");
static_assert(kLongRing + rows_lds_bytes(cgdec::ByteTables::kMaxBins) <= kLongObuf, "rows lie before the scratch");

// Any length, one wave per block (56 planes x 1000 tokens x 256 channels: 100
// us, where the shared-window kernel took 1307 us: the streams of a block
// outgrow its LDS window and were read a dword at a time from memory, with a
// binary search per symbol after the table's first long code).
__global__ void __launch_bounds__(kDecLanes)
    decode_long_kernel(const int16_t *__restrict__ cdf, const uint8_t *__restrict__ bytes, int64_t nbytes,
                       const StreamEnds ends, int T, const Channels chans, int nb, uint8_t *__restrict__ out,
                       int64_t n_streams) {
  extern __shared__ uint32_t lds_words[];
  uint8_t *lds = reinterpret_cast<uint8_t *>(lds_words);
  const uint32_t lds_at =
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t *)lds));
  const int lane = static_cast<int>(threadIdx.x);
  DecBlock bk;
  bk.init(cdf, nbytes, ends, n_streams, chans, nb, lane);
  const int nrow = static_cast<int>((bk.R1 - bk.r_lo + 15) >> 4);
  chunk16 rv[kRowChunks];
  load_chunks(bk.r_lo, nrow, 0, lane, rv);
  const LaneChunks ch(bytes, bk);
  cgdec::LongTables tb;
  tb.bind(lds, lane, lds_at);
  tb.clear();
  store_chunks<false>(lds + kLongRing, nrow, 0, lane, rv);  // (all of them: n_bins <= 32)
  wave_sync();
  const int row_at = static_cast<int>(bk.R0 - bk.r_lo) + (lane < bk.cnt ? lane : 0) * (nb + 1) * 2;
  tb.one.row.r = reinterpret_cast<const int16_t *>(lds + kLongRing + row_at);
  tb.one.nb = nb;
  uint8_t *obuf = lds + kLongObuf;
  if (short_rows(lds + kLongRing, nrow, lane)) {
    const Regions regions(ch, kLongObuf - kShortRegions, lane);
    chunk16 cv[kFirstChunks];
#pragma unroll
    for (uint32_t u = 0; u < kFirstChunks; ++u) cv[u] = ch.load(u);
    if (regions.fit()) {
      if (short_table(tb.one, obuf, lane)) {
        decode_short(tb.one, bk, ch, cv, regions, lds, lds_at, obuf, T, chans, lane, out);
        return;
      }
      tb.clear();
    }
  }
  tb.build(lds_at + static_cast<uint32_t>(kLongObuf + lane));
  const bool irregular = __any(tb.irregular) != 0;
  if (irregular) {  // the search reads the rows, not the tables
#pragma unroll
    for (int k = 0; k < kRowChunks; ++k) {
      const int j = k * kDecLanes + lane;
      if (j < nrow) reinterpret_cast<chunk16 *>(lds)[j] = reinterpret_cast<const chunk16 *>(lds + kLongRing)[j];
    }
    tb.one.row.r = reinterpret_cast<const int16_t *>(lds + row_at);
    wave_sync();
  }
  decode_serial(tb, irregular, bk, ch, lds, lds_at, kLongRing, T, chans, lane, out);
}

// Split decode: four waves per block of 64 streams, each taking a quarter of
// every stream (lane = stream).  Where a quarter's codes start is not stored,
// so waves 1 to 3 begin at the bit where it should lie, less `warm` codes,
// and decode those without keeping them: prefix codes resynchronise (Gaussian
// data at 16 / 32 bins: 99.9% of decoders started anywhere are on the true
// boundaries after 12 / 28 codes).  Each wave then keeps its symbols, in LDS
// and in a column of the lane's, until it passes the bit the next wave began
// keeping at.  If it stopped on that bit in every lane, the next wave was on
// the boundaries; otherwise that wave decodes again from where it did stop,
// so after at most three more rounds every quarter follows from the one
// before, whatever the streams hold.  The symbols' counts then place the
// quarters, and the waves write the block's tokens, each gathering four
// streams' symbols per dword.
//   A lane takes a long code in two table lookups (cgdec::StepCursor), so the
// lanes are not on the same symbol, which the columns do not need.
//   Bound by the steps' dependent instructions, about 213 cycles a step with
// one wave per SIMD.  56 planes x 1000 tokens x 256 channels on MI355X: 58 us,
// 100 us with one wave per block; of its 128k cycles 24k build the tables,
// 71k decode and 25k write the tokens out.  Writing the symbols in rows of 64
// bytes ([n][lane], up to four lanes on a bank) and gathering each dword of
// the output from four streams byte by byte took 62 us.
//   Blocks with an irregular row, with a stream that ends before its T
// symbols, or with a quarter that outgrows its rows of the buffer (codes
// bunched at one end) are decoded by one wave (decode_serial).
struct SplitPlan {
  int first, rest;          // tokens wave 0 and each other wave are meant to take
  int warm;                 // codes decoded before a later wave's own, a multiple of 16
  int cap0, cap;            // rows of the buffers of wave 0 and of each other wave
  int meta_off, rows_off, lds;
};
constexpr int kSplit = 4;
constexpr int kSplitThreads = kSplit * kDecLanes;
constexpr int kSplitSteps = 16;  // steps per epoch: at most 16 bytes of the ring
constexpr int kSplitRing = static_cast<int>(cgdec::StepCursor::Ring::kBytes) * kDecLanes;
constexpr int kSplitBuf = kLongRing + kSplit * kSplitRing;
constexpr int kSplitFlags = 16;
constexpr int kSplitShort = 15;
// Its LDS holds chunks of up to kSplitMaxT tokens, and leaves one block on a
// CU where decode_long_kernel has four, so it takes launches that leave it a
// CU per block, and chunks long enough for the codes decoded before each
// quarter's own not to matter (300 tokens, 96 blocks: 42 us against 39 for one
// wave per block; 512 tokens, 512 blocks: 90 against 60; 1000 tokens, 224
// blocks: 58 against 100).
constexpr int kSplitMaxT = 1024;
constexpr int kSplitMinT = 385;
constexpr int kSplitMaxBlocks = 256;
inline SplitPlan split_plan(int T, int nb) {
  SplitPlan p;
  p.warm = T <= 400 ? 32 : T <= 700 ? 48 : 64;
  // Every wave decodes about as much: wave 0 has no codes before its own.
  p.first = (T + 3 * p.warm + 3) / 4;
  p.rest = std::max(p.first - p.warm, 0);
  const auto cap = [](int n) { return (n + n / 8 + 32 + kSplitSteps - 1) / kSplitSteps * kSplitSteps; };
  p.cap0 = cap(p.first);
  p.cap = cap(p.rest);
  p.meta_off = kSplitBuf + (p.cap0 + 3 * p.cap) * kDecLanes;
  p.rows_off = p.meta_off + 4 * (3 * kSplit * kDecLanes + kSplitFlags);
  p.lds = p.rows_off + rows_lds_bytes(nb);
  return p;
}

// First row of wave w's buffer (rows of 64 bytes).
__device__ __forceinline__ int split_base(const SplitPlan &p, int w) {
  return w == 0 ? 0 : p.cap0 + (w - 1) * p.cap;
}

__global__ void __launch_bounds__(kSplitThreads)
    decode_split_kernel(const int16_t *__restrict__ cdf, const uint8_t *__restrict__ bytes, int64_t nbytes,
                        const StreamEnds ends, int T, const Channels chans, int nb, uint8_t *__restrict__ out,
                        int64_t n_streams,
                        const SplitPlan plan) {
  const int C = chans.n;
  extern __shared__ uint32_t lds_words[];
  uint8_t *lds = reinterpret_cast<uint8_t *>(lds_words);
  const uint32_t lds_at =
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t *)lds));
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  uint32_t *starts = reinterpret_cast<uint32_t *>(lds + plan.meta_off);  // [wave][lane]: where its symbols start
  uint32_t *stops = starts + kSplit * kDecLanes;                         // first boundary past its end
  uint32_t *counts = stops + kSplit * kDecLanes;
  // [0]: an irregular row; [1 + 2 r], [2 + 2 r]: round r left a wave off its
  // boundaries, a wave out of room (each written in its own round, so that
  // every wave reads the same); [kSplitShort]: decode_short takes the block.
  uint32_t *flags = counts + kSplit * kDecLanes;
  DecBlock bk;
  bk.init(cdf, nbytes, ends, n_streams, chans, nb, lane);
  const bool live = lane < bk.cnt;
  const LaneChunks ch(bytes, bk);
  // T codes of at most 12 bits end before 2 T bytes: longer streams are of no
  // use, and their bits would not fit 32 bits.
  const uint32_t len = ch.n_ch ? ch.end - ch.off : 0u;
  const uint32_t most = 2u * static_cast<uint32_t>(T) + 8u;
  const uint32_t stream_bits = 8u * (len < most ? len : most);

  // The segment's ring: local chunk 0 is the chunk of its first bit.
  uint32_t *ring = reinterpret_cast<uint32_t *>(lds + kLongRing + wave * kSplitRing) + lane;
  constexpr uint32_t kRingDw = cgdec::StepCursor::Ring::kBytes / 4;
  const uint32_t column = lds_at + static_cast<uint32_t>(kLongRing + wave * kSplitRing) + 4u * static_cast<uint32_t>(lane);
  uint32_t guess = static_cast<uint32_t>(static_cast<float>(stream_bits) * static_cast<float>(wave * plan.rest) /
                                         static_cast<float>(T));
  guess = guess < stream_bits ? guess : stream_bits;
  uint32_t chunk0 = (8u * ch.off + guess) >> 7, filled = 0;
  chunk16 cv[kFirstChunks];
  auto load_first = [&]() {
#pragma unroll
    for (uint32_t u = 0; u < kFirstChunks; ++u) cv[u] = ch.load(chunk0 + u);
  };
  auto put_first = [&]() {
#pragma unroll
    for (uint32_t u = 0; u < kFirstChunks; ++u) ch.put(ring, kRingDw, u, chunk0 + u, cv[u]);
    filled = kFirstChunks;
    wave_sync();
  };
  load_first();

  // Tables: cleared by every wave, marked by wave 0, scanned by all, the
  // markers put in by wave 0.
  cgdec::LongTables tb;
  tb.bind(lds, lane, lds_at);
  const int nrow = static_cast<int>((bk.R1 - bk.r_lo + 15) >> 4);
  {
    uint32_t *t32 = reinterpret_cast<uint32_t *>(tb.one.tab);
    for (int d = wave * (128 / kSplit); d < (wave + 1) * (128 / kSplit); ++d) t32[d * kDecLanes] = 0;
    for (int j = static_cast<int>(threadIdx.x); j < nrow; j += kSplitThreads)
      reinterpret_cast<chunk16 *>(lds + plan.rows_off)[j] = reinterpret_cast<global_chunk16 *>(bk.r_lo)[j];
    if (threadIdx.x < kSplitFlags) flags[threadIdx.x] = 0;
  }
  __syncthreads();
  tb.one.row.r = reinterpret_cast<const int16_t *>(lds + plan.rows_off + (bk.R0 - bk.r_lo)) +
                 (live ? lane : 0) * (nb + 1);
  tb.one.nb = nb;
  const uint32_t dummy = lds_at + static_cast<uint32_t>(kSplitBuf + lane);  // scratch for skipped writes
  // Short codes: one wave takes the block (every wave finds the same).  The
  // regions reach up to the transpose, at the end of the buffers; wave 0's
  // first chunks are the streams'.
  if (short_rows(lds + plan.rows_off, nrow, lane)) {
    const int obuf_off = plan.meta_off - kObufBytes;
    const Regions regions(ch, static_cast<uint32_t>(obuf_off - kShortRegions), lane);
    if (regions.fit()) {
      if (wave == 0 && short_table(tb.one, lds + obuf_off, lane) && lane == 0) flags[kSplitShort] = 1;
      __syncthreads();
      if (flags[kSplitShort] != 0) {
        if (wave == 0) decode_short(tb.one, bk, ch, cv, regions, lds, lds_at, lds + obuf_off, T, chans, lane, out);
        return;
      }
      if (wave == 0) tb.clear();
    }
  }
  if (wave == 0) {
    tb.mark(dummy);
    if (__any(tb.irregular) && lane == 0) flags[0] = 1;
  } else {
    put_first();
  }
  __syncthreads();
  if (wave == 0) tb.one.scan(0, 64, 0);
  else tb.scan_second(wave - 1, kSplit - 1);
  __syncthreads();
  if (wave == 0) {
    tb.escapes(dummy);
    put_first();
  }
  __syncthreads();

  bool one_wave = flags[0] != 0;  // the same in every wave, here and below
  if (!one_wave) {
    cgdec::StepCursor cur;
    cur.start(tb, column, (8u * ch.off + guess) & 127u, guess);
    auto epoch = [&](uint32_t to, auto &&each) {
      // One chunk of room or more: the chunk read ahead over the epoch.
      const bool room = 16u * filled - cur.ring.q <= cgdec::StepCursor::Ring::kBytes - 16u;
      const chunk16 nv = ch.load(room ? chunk0 + filled : ~0u);
#pragma unroll
      for (int i = 0; i < kSplitSteps / 2; ++i) cur.pair(tb, to, each);
      if (room) {
        ch.put(ring, kRingDw, filled, chunk0 + filled, nv);
        ++filled;
      }
      wave_sync();
    };
    if (wave > 0)
      for (int w = 0; w < plan.warm; w += kSplitSteps) epoch(~0u, [](uint32_t, bool) {});
    uint32_t start = cur.bd;
    starts[wave * kDecLanes + lane] = start;
    __syncthreads();
    const uint32_t hi = wave + 1 < kSplit ? starts[(wave + 1) * kDecLanes + lane] : stream_bits;
    const int cap = wave == 0 ? plan.cap0 : plan.cap;
    const uint32_t buf = lds_at + static_cast<uint32_t>(kSplitBuf + split_base(plan, wave) * kDecLanes + 4 * lane);
    bool run = true;
    for (int round = 0;; ++round) {
      if (run) {
        // Symbol n of the lane is byte n % 4 of dword n / 4 of its column
        // (dwords [n / 4][lane]: every lane in its own bank).
        uint32_t n = 0;
        for (int steps = 0; steps < cap && __any(cur.bd < hi); steps += kSplitSteps)
          epoch(hi, [&](uint32_t e, bool counts) {
            cgdec::lds_set_byte(buf + (n << 6) - 63u * (n & 3u), e >> 3);
            n += counts ? 1u : 0u;
          });
        if (__any(live && cur.bd < hi) && lane == 0) flags[2 + 2 * round] = 1;
        stops[wave * kDecLanes + lane] = cur.bd;
        counts[wave * kDecLanes + lane] = n;
      }
      __syncthreads();
      const uint32_t before = wave > 0 ? stops[(wave - 1) * kDecLanes + lane] : 0u;
      const bool off_bound = wave > 0 && live && before != start;
      run = __any(off_bound) != 0;
      if (run && lane == 0) flags[1 + 2 * round] = 1;
      __syncthreads();
      const bool again = flags[1 + 2 * round] != 0;
      one_wave = flags[2 + 2 * round] != 0 || (again && round + 1 == kSplit);
      if (one_wave || !again) break;
      if (run) {
        start = off_bound ? before : start;
        chunk0 = (8u * ch.off + start) >> 7;
        load_first();
        put_first();
        cur.start(tb, column, (8u * ch.off + start) & 127u, start);
      }
    }
    uint32_t symbols = 0;
#pragma unroll
    for (int w = 0; w < kSplit; ++w) symbols += counts[w * kDecLanes + lane];
    one_wave = one_wave || __any(live && symbols < static_cast<uint32_t>(T)) != 0;
  }
  if (one_wave) {
    __syncthreads();
    if (wave == 0)
      decode_serial(tb, flags[0] != 0, bk, ch, lds, lds_at, kLongRing, T, chans, lane, out);
    return;
  }
  // The tokens, four at a time, a quarter of them per wave; lane = stream.  A
  // lane's four symbols are four bytes of its column, two dwords shifted
  // together, unless its tokens lie in two quarters; the dwords go through
  // the transpose in the wave's (dead) ring and are stored one group late.
  uint32_t until[kSplit];  // tokens up to the end of quarter k
  uint32_t t0 = 0;
#pragma unroll
  for (int k = 0; k < kSplit; ++k) {
    t0 += counts[k * kDecLanes + lane];
    // (a lane without a stream: rows inside the buffers)
    until[k] = live ? t0 : static_cast<uint32_t>(T);
  }
  // LDS byte of the lane's symbol of token t.
  const uint32_t column0 = lds_at + static_cast<uint32_t>(kSplitBuf + 4 * lane);
  auto place = [&](uint32_t t, uint32_t &row) {  // returns the quarter's first row in the buffers
    uint32_t base = 0, before = 0;
#pragma unroll
    for (int k = 0; k + 1 < kSplit; ++k) {
      const bool past = t >= until[k];
      base = past ? static_cast<uint32_t>(split_base(plan, k + 1)) : base;
      before = past ? until[k] : before;
    }
    row = t - before;
    return base;
  };
  auto end_of = [&](uint32_t t) {
    uint32_t e = until[0];
#pragma unroll
    for (int k = 0; k + 1 < kSplit; ++k) e = t >= until[k] ? until[k + 1] : e;
    return e;
  };
  const DecBlock::Quad quad = bk.quad(out, T, chans, lane);
  uint8_t *obuf = lds + kLongRing + wave * kSplitRing;
  const int groups = (T + 3) / 4, share = (groups + kSplit - 1) / kSplit;
  const int g1 = (wave + 1) * share < groups ? (wave + 1) * share : groups;
  uint32_t word = 0;
  int stored = wave * share;  // groups stored
  for (int g = wave * share; g < g1; ++g) {
    const uint32_t t = 4u * static_cast<uint32_t>(g);
    uint32_t row;
    const uint32_t base = place(t, row);
    const uint32_t at = column0 + (base + (row & ~3u)) * kDecLanes;
    uint32_t four = __builtin_amdgcn_alignbyte(cgdec::lds_dword(at + 4u * kDecLanes), cgdec::lds_dword(at), row & 3u);
    if (__any(live && end_of(t) < t + 4u)) {
      four = 0;
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        uint32_t r;
        // Tokens past T: any byte of the column.
        const uint32_t b = place(t + i < static_cast<uint32_t>(T) ? t + i : t, r);
        const uint32_t d = cgdec::lds_dword(column0 + (b + (r & ~3u)) * kDecLanes);
        four |= ((d >> (8u * (r & 3u))) & 0xFFu) << (8u * i);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) obuf[i * kDecLanes + lane] = static_cast<uint8_t>(four >> (8 * i));
    if (g > stored) {
      cg_st(quad.dst + static_cast<int64_t>(stored) * C, word);
      ++stored;
    }
    wave_sync();
    word = reinterpret_cast<const uint32_t *>(obuf)[quad.at];
    wave_sync();
  }
  if (stored < g1 && 4 * stored + (quad.at >> 4) < T) cg_st(quad.dst + static_cast<int64_t>(stored) * C, word);
}

// Moves the blocks' bytes together: block b's off[b + 1] - off[b] bytes, from
// b * stride of `blocks`, to off[b] of `out`.  A thread takes 16-byte aligned
// pieces of the destination, each from five source dwords shifted together;
// the bytes of the pieces shared with the blocks before and after are stored
// one by one.  Every source dword read holds a byte of the block.  A block is
// shared by kPackParts workgroups: medians of the kernel behind the encoder
// (MI355X, traced), one workgroup a block -> two -> four: 64 planes x 256
// tokens x 1024 channels (1024 blocks, 6.9 MB) 6.6 -> 5.4 -> 5.4 us, 128
// planes 9.4 -> 8.2 -> 8.5, 56 x 256 x 256 (224 blocks, 1.5 MB) 4.8 -> 3.8 ->
// 3.7, 56 x 1000 x 256 (224 blocks, 5.7 MB) 9.0 -> 6.2 -> 5.0, 64 x 1000 x
// 1024 (26 MB) 13.2 -> 12.6 -> 10.8.  (A copy stream by stream from rows of
// their own, each with such edges, took twice as long, and a boolean mask over
// the rows with a masked select about 330 us.)
constexpr int kPackThreads = 256;
constexpr unsigned kPackParts = 4;
__global__ void __launch_bounds__(kPackThreads)
    pack_blocks_kernel(const uint8_t *__restrict__ blocks, int64_t stride, const int64_t *__restrict__ off,
                       uint8_t *__restrict__ out, int64_t size) {
  typedef unsigned int w4 __attribute__((ext_vector_type(4)));
  typedef unsigned int w4u __attribute__((ext_vector_type(4), aligned(4)));
  const int64_t begin = off[blockIdx.x];
  const int64_t end = off[blockIdx.x + 1];
  const int64_t n = (end < size ? end : size) - begin;  // `out` holds `size` bytes
  const uint8_t *src = blocks + static_cast<int64_t>(blockIdx.x) * stride;
  uint8_t *dst = out + begin;
  const int64_t lead = static_cast<int64_t>(reinterpret_cast<uintptr_t>(dst) & 15);
  // Piece i of the destination holds the block's bytes 16 i - lead .. + 15.
  const int64_t step = 16 * static_cast<int64_t>(kPackThreads) * gridDim.y;
  for (int64_t at = 16 * static_cast<int64_t>(blockIdx.y * kPackThreads + threadIdx.x) - lead; at < n; at += step) {
    if (at >= 0 && at + 16 <= n) {
      const uint8_t *p = src + at;
      const uint32_t sh = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 3);
      const w4u x = *reinterpret_cast<const __attribute__((address_space(1))) w4u *>(
          reinterpret_cast<uintptr_t>(p - sh));
      const uint32_t y = sh ? gload(reinterpret_cast<const uint32_t *>(p - sh) + 4) : 0u;
      w4 r;
      r.x = __builtin_amdgcn_alignbyte(x.y, x.x, sh);
      r.y = __builtin_amdgcn_alignbyte(x.z, x.y, sh);
      r.z = __builtin_amdgcn_alignbyte(x.w, x.z, sh);
      r.w = __builtin_amdgcn_alignbyte(y, x.w, sh);
      gstore(reinterpret_cast<w4 *>(dst + at), r);
    } else {
      for (int64_t b = at < 0 ? 0 : at; b < at + 16 && b < n; ++b) dst[b] = src[b];
    }
  }
}

// What a call that waits for a device value needs: a word of pinned host
// memory, which the kernel writes and the host watches, and an event behind
// the kernel, which bounds the watch.  Taken from a pool per call and given
// back once the word has been written; the pool keeps at most kKept of them.
class HostWord {
public:
  explicit HostWord(int device) {
    {
      std::lock_guard<std::mutex> g(mu());
      auto &p = pool();
      for (size_t i = 0; i < p.size(); ++i)
        if (p[i].device == device) {
          s_ = p[i];
          p.erase(p.begin() + static_cast<std::ptrdiff_t>(i));
          return;
        }
    }
    s_.device = device;
    hip_check(hipEventCreateWithFlags(&s_.event, hipEventDisableTiming), "hipEventCreate");
    const hipError_t e = hipHostMalloc(reinterpret_cast<void **>(&s_.word), sizeof(int64_t),
                                       hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent);
    if (e != hipSuccess) {
      (void)hipEventDestroy(s_.event);
      hip_check(e, "hipHostMalloc");
    }
  }
  HostWord(const HostWord &) = delete;
  HostWord &operator=(const HostWord &) = delete;
  // A word is given back only when no kernel may still write it: wait() has
  // seen it written, and a call that fails after its launch waits for the
  // stream here.
  ~HostWord() {
    if (pending_) (void)hipStreamSynchronize(stream_);
    {
      std::lock_guard<std::mutex> g(mu());
      if (pool().size() < kKept) {
        pool().push_back(s_);
        return;
      }
    }
    (void)hipEventDestroy(s_.event);
    (void)hipHostFree(s_.word);
  }
  // Call before the launch of the kernel that writes the word (a value of 0
  // or more), then record() after it.
  int64_t *launching(hipStream_t stream) {
    stream_ = stream;
    pending_ = true;
    __atomic_store_n(s_.word, int64_t(-1), __ATOMIC_RELEASE);
    return s_.word;
  }
  void record() { hip_check(hipEventRecord(s_.event, stream_), "hipEventRecord"); }
  int64_t wait() {
    for (;;) {
      for (int i = 0; i < 256; ++i) {
        const int64_t v = __atomic_load_n(s_.word, __ATOMIC_ACQUIRE);
        if (v >= 0) {
          pending_ = false;
          return v;
        }
        __builtin_ia32_pause();
      }
      const hipError_t e = hipEventQuery(s_.event);
      if (e == hipErrorNotReady) continue;
      hip_check(e, "hipEventQuery");
      // The kernel is over: its word is there.
      const int64_t v = __atomic_load_n(s_.word, __ATOMIC_ACQUIRE);
      pending_ = false;
      check(v >= 0, "the kernel left no value");
      return v;
    }
  }

private:
  struct Slot {
    int device = 0;
    hipEvent_t event = nullptr;
    int64_t *word = nullptr;
  };
  static constexpr size_t kKept = 16;
  static std::mutex &mu() {
    static std::mutex m;
    return m;
  }
  static std::vector<Slot> &pool() {
    static std::vector<Slot> *p = new std::vector<Slot>();  // outlives the runtime's own teardown
    return *p;
  }
  Slot s_;
  hipStream_t stream_ = nullptr;
  bool pending_ = false;
};

// The sums of StreamEnds: a workgroup takes a group of 64 blocks of 64
// streams, four lengths per thread.  A decode block adds the groups before
// its own to its block's sum, which for 65536 streams is one load per lane
// and one wave sum, so the prefix sums of the streams are never written.
// Traced on MI355X (65536 streams): 3.9 to 4.7 us and the decode kernel behind
// it 20.3 us, against four launches of about 17 us for prefix sums in 64 bits
// (widening, scan, narrowing) and 24.4 us for the decode kernel reading them;
// decode_chunk 35.9 -> 22.4 us.
// S: uint32_t, or int64_t for buffers of 2 GiB and more (negative lengths
// count as 0 there).
template <typename S>
__global__ void __launch_bounds__(kSumThreads)
    length_sums_kernel(const int32_t *__restrict__ lens, int64_t n_streams, int64_t n_blocks,
                       S *__restrict__ sums, S *__restrict__ groups) {
  constexpr bool WIDE = sizeof(S) == 8;
  __shared__ S block_sum[kGroupBlocks];
  const int tid = static_cast<int>(threadIdx.x);
  const int64_t s = (static_cast<int64_t>(blockIdx.x) * kSumThreads + tid) * 4;
  S own = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int32_t n = s + k < n_streams ? lens[s + k] : 0;
    own += static_cast<S>(WIDE ? max(n, 0) : n);
  }
  // 16 threads hold a block's lengths.
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) own += __shfl_xor(own, d, 64);
  if ((tid & 15) == 0) block_sum[tid >> 4] = own;
  __syncthreads();
  if (tid < kGroupBlocks) {
    const S b = block_sum[tid];
    S incl = b;
    if constexpr (WIDE) {
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const S v = __shfl_up(incl, d, 64);
        incl += tid >= d ? v : 0;
      }
    } else {
      incl = wave_incl_scan(b);
    }
    const int64_t block = static_cast<int64_t>(blockIdx.x) * kGroupBlocks + tid;
    if (block < n_blocks) sums[block] = incl - b;
    if (tid == kGroupBlocks - 1) groups[blockIdx.x] = incl;
  }
}

// Row-major contiguity; a tensor without elements has no layout to check.
bool contiguous(const lmc_tensor &t) {
  if (numel(t) == 0) return true;
  int64_t expect = 1;
  for (int i = t.ndim - 1; i >= 0; --i) {
    if (t.sizes[i] != 1 && t.strides[i] != expect) return false;
    expect *= t.sizes[i];
  }
  return true;
}

void need_device(const lmc_tensor &t, const char *what) {
  check(t.device >= 0, std::string(what) + " is not a GPU tensor");
  check(contiguous(t), std::string(what) + " must be contiguous");
}

// calculate_cdf (csrc/cachegen_kernels.cpp:119-155), with the streams'
// lengths and the 64-stream blocks' bytes when `lens` is given (see
// cdf_tile_kernel).
void make_cdf(const lmc_tensor &in, int32_t n_bins, const lmc_tensor &o, int32_t *lens, int64_t *sums, int64_t cap,
              hipStream_t stream) {
  need_device(in, "input");
  need_device(o, "output");
  check(in.ndim == 3, "input must be [layers, tokens, channels]");
  check(in.dtype == LMC_U8 || in.dtype == LMC_I8, "input must be uint8/int8");
  check(o.dtype == LMC_I16, "output must be int16");
  check(n_bins >= 1 && n_bins <= kMaxBins,
        "n_bins must be in [1, " + std::to_string(kMaxBins) + "]");
  const int64_t L = in.sizes[0], T = in.sizes[1], C = in.sizes[2];
  check(o.ndim == 3 && o.sizes[0] == L && o.sizes[1] == C &&
            o.sizes[2] == n_bins + 1,
        "output must be [layers, channels, n_bins + 1]");
  check(T < (int64_t(1) << 26) && C < (int64_t(1) << 30), "input too large");
  if (L == 0 || C == 0) return;
  DeviceGuard guard(in.device);
  const int64_t n_streams = L * C;
  const int64_t blocks = (n_streams + 63) / 64;
  check(blocks < (int64_t(1) << 31), "too many streams");
  const size_t lds = static_cast<size_t>(cdf_lds_bytes(static_cast<int>(T), n_bins));
  const int vec_tile = (C % 16 == 0 && (reinterpret_cast<uintptr_t>(in.data) & 15) == 0) ? 1 : 0;
  const auto kern = n_bins == 32         ? cdf_tile_kernel<32, true>
                    : n_bins < 32        ? cdf_tile_kernel<32, false>
                    : n_bins == kMaxBins ? cdf_tile_kernel<kMaxBins, true>
                                         : cdf_tile_kernel<kMaxBins, false>;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(kCdfThreads), lds, stream,
                     static_cast<const uint8_t *>(in.data), (int)T, (int)C, n_bins,
                     static_cast<int16_t *>(o.data), n_streams, vec_tile, lens, sums, cap);
  hip_check(hipGetLastError(), "cdf_tile_kernel launch");
}

// encode_fast_new (csrc/cachegen_kernels.cpp:17-58) with place 0; with place
// 1 the streams of each block of 64 one after the other (encode_split_kernel;
// `ol` then holds their lengths already, and cdf is calculate_cdf's).
void encode_rows(const lmc_tensor &cdf, const lmc_tensor &in, const lmc_tensor &ob, const lmc_tensor &ol, int place,
                 const BlockOffsets &offsets, hipStream_t stream) {
  need_device(cdf, "cdf");
  need_device(in, "input_sym");
  need_device(ob, "output_buffer");
  need_device(ol, "output_lengths");
  check(in.ndim == 3 && cdf.ndim == 3 && ob.ndim == 3,
        "cdf, input_sym and output_buffer must be 3-D");
  const int64_t L = in.sizes[0], T = in.sizes[1], C = in.sizes[2];
  const int64_t nb = cdf.sizes[2] - 1;
  const int64_t chunk = ob.sizes[2];
  // csrc/cachegen_kernels.cpp:33-35
  check(C <= (1 << 15),
        "encode takes at most 32768 channels per layer");
  check(in.dtype == LMC_U8 || in.dtype == LMC_I8, "input_sym must be int8/uint8");
  check(cdf.dtype == LMC_I16, "cdf must be int16");
  check(ob.dtype == LMC_U8 || ob.dtype == LMC_I8, "output_buffer must be uint8");
  check(ol.dtype == LMC_I32 && numel(ol) == L * C, "output_lengths must be int32 [L, C]");
  check(nb >= 1 && nb <= kMaxBins, "number of bins must be in [1, 64]");
  check(cdf.sizes[0] == L && cdf.sizes[1] == C, "cdf must be [L, C, nbins + 1]");
  check(ob.sizes[0] == L && ob.sizes[1] == C, "output_buffer must be [L, C, chunk]");
  if (L == 0 || C == 0) return;
  DeviceGuard guard(in.device);
  const int64_t n_streams = L * C;
  const int64_t blocks = (n_streams + kEncLanes - 1) / kEncLanes;
  check(blocks < (int64_t(1) << 31) && T < (int64_t(1) << 31), "input too large");
  const int vec_in = (C % 16 == 0 && (reinterpret_cast<uintptr_t>(in.data) & 15) == 0) ? 1 : 0;
  const int rows_dw = (reinterpret_cast<uintptr_t>(cdf.data) & 3) == 0 ? 1 : 0;
  const EncLds at = enc_lds(T, static_cast<int>(nb));
  // calculate_cdf's codes are at most 12 bits, so rows of 2 bytes a symbol
  // cut no stream.
  const bool image = place == 1 && T <= kEncTokens && chunk >= 2 * T &&
                     (reinterpret_cast<uintptr_t>(ob.data) & 15) == 0;
  const auto kern = image                                ? encode_split_kernel<kEncPieces, EncMode::kImage>
                    : place == 0 && T <= kEncTokens ? encode_split_kernel<kEncPieces, EncMode::kRows>
                                                         : encode_split_kernel<kEncPieces, EncMode::kLong>;
  check(at.bytes <= 65536, "encode: LDS budget exceeded");
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks + (offsets.sums != nullptr ? 1 : 0))),
                     dim3(64 * kEncPieces), at.bytes, stream,
                     static_cast<const int16_t *>(cdf.data), static_cast<const uint8_t *>(in.data), (int)T, (int)C,
                     (int)nb, n_streams, static_cast<uint8_t *>(ob.data), chunk, static_cast<int32_t *>(ol.data),
                     place, vec_in, rows_dw, at, offsets);
  hip_check(hipGetLastError(), "encode_split_kernel launch");
}

// decode_fast_prefsum (csrc/cachegen_kernels.cpp:67-112); with `sums`,
// scratch for StreamEnds, `ln` holds the streams' lengths in place of their
// prefix sums.
void decode_streams(const lmc_tensor &cdf, const lmc_tensor &bs, const lmc_tensor &ln, const lmc_tensor &o,
                    const lmc_tensor *sums, hipStream_t stream) {
  // csrc/cachegen_kernels.cpp:78-88
  check(cdf.device >= 0, "cdf is not a GPU tensor");
  check(bs.device >= 0, "bytestreams is not a GPU tensor");
  check(ln.device >= 0, "lengths is not a GPU tensor");
  check(o.device >= 0, "output is not a GPU tensor");
  need_device(cdf, "cdf");
  need_device(bs, "bytestreams");
  need_device(ln, "lengths");
  need_device(o, "output");
  check(cdf.ndim == 3, "cdf must be [L, C, nbins + 1]");
  const int64_t L = cdf.sizes[0], C = cdf.sizes[1], nb = cdf.sizes[2] - 1;
  check(C % 32 == 0, "decode takes a channel count that is a multiple of 32");
  check(nb < 64, "decode takes fewer than 64 bins per stream");
  check(nb >= 1, "cdf needs at least one bin");
  check(cdf.dtype == LMC_I16, "cdf must be int16");
  check(bs.dtype == LMC_U8 || bs.dtype == LMC_I8, "bytestreams must be uint8");
  check(ln.dtype == LMC_I32 && numel(ln) == L * C, "lengths must be int32 [L, C]");
  check(o.dtype == LMC_U8 || o.dtype == LMC_I8, "output must be uint8");
  check(o.ndim >= 2, "output must be [L, T, C]");
  const int64_t T = o.sizes[1];
  check(numel(o) == L * T * C, "output must hold L * T * C symbols");
  if (L == 0 || C == 0 || T == 0) return;
  DeviceGuard guard(bs.device);
  const int64_t n_streams = L * C;
  const int64_t blocks = (n_streams + kDecLanes - 1) / kDecLanes;
  check(blocks < (int64_t(1) << 31), "too many streams");
  StreamEnds ends = {};
  if (sums == nullptr) {
    ends.prefix = static_cast<const int32_t *>(ln.data);
  } else {
    const int64_t groups = (blocks + kGroupBlocks - 1) / kGroupBlocks;
    need_device(*sums, "sums");
    check((sums->dtype == LMC_I32 || sums->dtype == LMC_I64) && numel(*sums) >= blocks + groups,
          "sums must be int32 or int64 with an entry per block of 64 streams and per 64 blocks");
    const dim3 sum_grid(static_cast<unsigned>(groups));
    ends.lens = static_cast<const int32_t *>(ln.data);
    if (sums->dtype == LMC_I64) {
      int64_t *b = static_cast<int64_t *>(sums->data);
      ends.wide_sums = b;
      ends.wide_groups = b + blocks;
      hipLaunchKernelGGL(length_sums_kernel<int64_t>, sum_grid, dim3(kSumThreads), 0, stream, ends.lens, n_streams,
                         blocks, b, b + blocks);
    } else {
      uint32_t *b = static_cast<uint32_t *>(sums->data);
      ends.sums = b;
      ends.groups = b + blocks;
      hipLaunchKernelGGL(length_sums_kernel<uint32_t>, sum_grid, dim3(kSumThreads), 0, stream, ends.lens, n_streams,
                         blocks, b, b + blocks);
    }
    hip_check(hipGetLastError(), "length_sums_kernel launch");
  }
  const int16_t *rows = static_cast<const int16_t *>(cdf.data);
  const uint8_t *bytes = static_cast<const uint8_t *>(bs.data);
  uint8_t *out = static_cast<uint8_t *>(o.data);
  const dim3 grid(static_cast<unsigned>(blocks));
  if (nb <= cgdec::ByteTables::kMaxBins && T > kLaneMaxT && (reinterpret_cast<uintptr_t>(out) & 3) == 0) {
    if (T >= kSplitMinT && T <= kSplitMaxT && blocks <= kSplitMaxBlocks) {
      const SplitPlan plan = split_plan(static_cast<int>(T), static_cast<int>(nb));
      hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(decode_split_kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, plan.lds),
                "decode LDS size");
      hipLaunchKernelGGL(decode_split_kernel, grid, dim3(kSplitThreads), plan.lds, stream, rows, bytes, numel(bs), ends,
                         (int)T, Channels(C), (int)nb, out, n_streams, plan);
    } else {
      hipLaunchKernelGGL(decode_long_kernel, grid, dim3(kDecLanes), kDecLds, stream, rows, bytes, numel(bs), ends,
                         (int)T, Channels(C), (int)nb, out, n_streams);
    }
  } else {
    hipLaunchKernelGGL(nb <= cgdec::ByteTables::kMaxBins ? decode_kernel<cgdec::ByteTables> : decode_kernel<DecTables>,
                       grid, dim3(kDecLanes), kDecLds, stream, rows, bytes, numel(bs), ends, (int)T, Channels(C), (int)nb,
                       out, n_streams);
  }
  hip_check(hipGetLastError(), "decode_kernel launch");
}

} // namespace

} // namespace lmc

using namespace lmc;

extern "C" {

int lmc_calculate_cdf(const lmc_tensor *input, int32_t n_bins,
                      const lmc_tensor *output, void *stream) {
  return guarded([&] {
    make_cdf(deref(input, "input"), n_bins, deref(output, "output"), nullptr, nullptr, 0,
             static_cast<hipStream_t>(stream));
  });
}

int lmc_encode_fast_new(const lmc_tensor *cdf_t, const lmc_tensor *input_sym,
                        const lmc_tensor *output_buffer,
                        const lmc_tensor *output_lengths, void *stream) {
  return guarded([&] {
    encode_rows(deref(cdf_t, "cdf"), deref(input_sym, "input_sym"), deref(output_buffer, "output_buffer"),
                deref(output_lengths, "output_lengths"), 0, BlockOffsets{nullptr, 0, nullptr, nullptr},
                static_cast<hipStream_t>(stream));
  });
}

int lmc_cachegen_encode_rows(const lmc_tensor *input, int32_t n_bins, const lmc_tensor *cdf_t,
                             const lmc_tensor *rows_t, const lmc_tensor *lengths_t,
                             const lmc_tensor *offsets_t, int64_t *total, void *stream_p) {
  return guarded([&] {
    const lmc_tensor &in = deref(input, "input");
    const lmc_tensor &cdf = deref(cdf_t, "cdf");
    const lmc_tensor &rows = deref(rows_t, "rows");
    const lmc_tensor &lens = deref(lengths_t, "lengths");
    const lmc_tensor &off = deref(offsets_t, "offsets");
    check_value(total != nullptr, "total is null");
    need_device(in, "input");
    need_device(rows, "rows");
    need_device(lens, "lengths");
    need_device(off, "offsets");
    check(in.ndim == 3 && rows.ndim == 3, "input and rows must be 3-D");
    check(lens.dtype == LMC_I32 && numel(lens) == in.sizes[0] * in.sizes[2], "lengths must be int32 [L, C]");
    const int64_t n_streams = in.sizes[0] * in.sizes[2];
    const int64_t blocks = (n_streams + 63) / 64;
    check(off.dtype == LMC_I64 && numel(off) == 2 * blocks + 1,
          "offsets must be int64 with one entry per block of 64 streams, one more, and one per block of scratch");
    *total = 0;
    hipStream_t stream = static_cast<hipStream_t>(stream_p);
    if (n_streams == 0) {
      make_cdf(in, n_bins, cdf, nullptr, nullptr, 0, stream);
      return;
    }
    DeviceGuard guard(in.device);
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    hip_check(hipStreamIsCapturing(stream, &cap), "hipStreamIsCapturing");
    check(cap == hipStreamCaptureStatusNone,
          "a chunk's size is read on the host: its encoding cannot be captured into a graph");
    int64_t *offsets = static_cast<int64_t *>(off.data);
    int64_t *sums = offsets + blocks + 1;
    make_cdf(in, n_bins, cdf, static_cast<int32_t *>(lens.data), sums, rows.sizes[2], stream);
    // The sizes follow from the histograms, so the host learns the total
    // while the streams are still being encoded.
    HostWord word(in.device);
    encode_rows(cdf, in, rows, lens, 1, BlockOffsets{sums, blocks, offsets, word.launching(stream)}, stream);
    word.record();
    *total = word.wait();
  });
}

int lmc_cachegen_pack_rows(const lmc_tensor *rows_t, const lmc_tensor *offsets_t, const lmc_tensor *streams_t,
                           void *stream) {
  return guarded([&] {
    const lmc_tensor &rows = deref(rows_t, "rows");
    const lmc_tensor &off = deref(offsets_t, "offsets");
    const lmc_tensor &o = deref(streams_t, "streams");
    need_device(rows, "rows");
    need_device(off, "offsets");
    need_device(o, "streams");
    check(rows.ndim == 3 && rows.dtype == LMC_U8 && o.dtype == LMC_U8, "rows and streams must be uint8");
    const int64_t n_streams = rows.sizes[0] * rows.sizes[1];
    const int64_t blocks = (n_streams + 63) / 64;
    check(off.dtype == LMC_I64 && numel(off) == 2 * blocks + 1, "offsets do not match the rows");
    if (n_streams == 0 || numel(o) == 0) return;
    check(blocks < (int64_t(1) << 31), "too many streams");
    DeviceGuard guard(rows.device);
    hipLaunchKernelGGL(pack_blocks_kernel, dim3(static_cast<unsigned>(blocks), kPackParts), dim3(kPackThreads), 0,
                       static_cast<hipStream_t>(stream), static_cast<const uint8_t *>(rows.data),
                       kEncLanes * rows.sizes[2], static_cast<const int64_t *>(off.data),
                       static_cast<uint8_t *>(o.data), numel(o));
    hip_check(hipGetLastError(), "pack_blocks_kernel launch");
  });
}

int lmc_decode_fast_new(const lmc_tensor *, const lmc_tensor *,
                        const lmc_tensor *, const lmc_tensor *, void *) {
  // csrc/cachegen_kernels.cpp:60-65
  set_last_error("decode_fast_new is not implemented; use decode_fast_prefsum");
  return LMC_ERR_NOT_IMPLEMENTED;
}

int lmc_decode_fast_prefsum(const lmc_tensor *cdf_t,
                            const lmc_tensor *bytestreams,
                            const lmc_tensor *lengths,
                            const lmc_tensor *output, void *stream) {
  return guarded([&] {
    decode_streams(deref(cdf_t, "cdf"), deref(bytestreams, "bytestreams"), deref(lengths, "lengths"),
                   deref(output, "output"), nullptr, static_cast<hipStream_t>(stream));
  });
}

int lmc_cachegen_decode(const lmc_tensor *cdf_t, const lmc_tensor *bytestreams, const lmc_tensor *lengths,
                        const lmc_tensor *sums, const lmc_tensor *output, void *stream) {
  return guarded([&] {
    decode_streams(deref(cdf_t, "cdf"), deref(bytestreams, "bytestreams"), deref(lengths, "lengths"),
                   deref(output, "output"), &deref(sums, "sums"), static_cast<hipStream_t>(stream));
  });
}

} // extern "C"
