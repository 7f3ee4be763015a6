// Host build of the decoder for long chunks (LongTables, RingCursor,
// PairCursor and StepCursor of lmcache-ascend_amd/csrc/cachegen_decode.h), checked against
// the CPU oracle's decoder (oracle/cachegen.c, oc_decode) on random CDF rows
// and byte streams.  Built and run by
// tests/test_decode_long_cpu.py.
//
// Every row's tables are built as the kernel builds them and its streams are
// decoded as the kernel decodes them: pairs of codes from the tables, or the
// binary search where the row is irregular, the ring refilled every 16 codes
// with chunks whose bytes past the stream's end are zero.  LDS is one buffer
// of the kernel's size (built with AddressSanitizer).
//
// Usage: decode_long_check <rows> <seed>; prints "ok ..." or the first
// mismatch and exits 1.
#define __device__
#define __forceinline__ inline
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>
using std::max;
using std::min;
#include "../lmcache-ascend_amd/csrc/cachegen_decode.h"

extern "C" void oc_decode(const int16_t *cdf, const uint8_t *bytes, int64_t nbytes,
                          const int32_t *prefix, int L, int T, int C, int nb, uint8_t *out);

using lmc::cgdec::kLanes;
using lmc::cgdec::LongTables;
using lmc::cgdec::PairCursor;
using lmc::cgdec::RingCursor;

namespace {

// Kind 0: a complete alphabetic code of nb symbols with lengths up to 12
// (random splits), some symbols absent; kind 1: aligned intervals of lengths
// 1..12 with gaps; kind 2: sorted bases in steps of 16 with random nibbles;
// kind 3: random entries.  Any of them may hold a decreasing entry.
void split(std::mt19937_64 &rng, int n, int depth, std::vector<int> &len) {
  if (n == 1) {
    len.push_back(depth);
    return;
  }
  const int cap = depth + 1 >= 12 ? 1 : 1 << std::min(12 - depth - 1, 20);
  int left = 1 + static_cast<int>(rng() % (n - 1));
  if (rng() % 2) left = rng() % 2 ? 1 : n - 1;  // deep at one end
  left = std::max(left, n - cap);
  left = std::min(left, cap);
  split(rng, left, depth + 1, len);
  split(rng, n - left, depth + 1, len);
}

void make_row(std::mt19937_64 &rng, int nb, int kind, int16_t *row) {
  auto put = [&](int s, uint32_t v) { row[s] = static_cast<int16_t>(static_cast<uint16_t>(v)); };
  if (kind == 0) {
    std::vector<char> on(nb, 1);
    for (auto &x : on) x = rng() % 5 != 0;
    int m = static_cast<int>(std::count(on.begin(), on.end(), 1));
    if (m == 0) on[0] = 1, m = 1;
    std::vector<int> len;
    if (m == 1) len.push_back(1);
    else split(rng, m, 0, len);
    uint32_t pos = 0;
    int k = 0;
    for (int s = 0; s < nb; ++s) {
      if (!on[s]) {
        put(s, pos & 0xFFF0u);
        continue;
      }
      put(s, (pos & 0xFFF0u) | static_cast<uint32_t>(len[k]));
      pos += 0x10000u >> len[k++];
    }
  } else if (kind == 1) {
    uint32_t pos = 0;
    for (int s = 0; s < nb; ++s) {
      const int l = 1 + static_cast<int>(rng() % 12);
      const uint32_t w = 1u << (16 - l);
      pos = (pos + w - 1) & ~(w - 1);
      if (rng() % 5 == 0 || pos + w > 0x10000u) {
        put(s, pos >= 0x10000u ? 0u : pos & 0xFFF0u);
        continue;
      }
      put(s, pos | static_cast<uint32_t>(l));
      pos += w;
      if (rng() % 6 == 0) pos = std::min(0x10000u, pos + (16u << (rng() % 10)));
    }
  } else if (kind == 2) {
    std::vector<uint32_t> b(nb);
    for (auto &x : b) x = static_cast<uint32_t>(rng() % 4096) * 16;
    std::sort(b.begin(), b.end());
    for (int s = 0; s < nb; ++s) put(s, b[s] | (rng() % 2 ? 0u : static_cast<uint32_t>(rng() % 16)));
  } else {
    for (int s = 0; s < nb; ++s) put(s, static_cast<uint32_t>(rng() & 0xFFFF));
  }
  if (nb > 2 && kind != 0 && rng() % 4 == 0) row[1 + rng() % (nb - 1)] = 0;
  row[nb] = static_cast<int16_t>(rng() & 0xFFFF);  // entry n_bins: ignored by the rules
}

}  // namespace

int main(int argc, char **argv) {
  const int rows = argc > 1 ? atoi(argv[1]) : 2000;
  std::mt19937_64 rng(argc > 2 ? strtoull(argv[2], nullptr, 10) : 1);
  constexpr uint32_t kRingAt = LongTables::kBytes;
  // The tables, the rings and a scratch byte for skipped writes.
  std::vector<uint8_t> lds(kRingAt + RingCursor::kBytes * kLanes + 1);
  const uint32_t dummy = static_cast<uint32_t>(lds.size()) - 1;
  long long symbols = 0, regular = 0, with_long = 0, irregular = 0;
  for (int it = 0; it < rows; ++it) {
    const int nb = it % 3 == 1 ? LongTables::kMaxBins : 1 + static_cast<int>(rng() % LongTables::kMaxBins);
    const int kind = it % 5 == 4 ? 0 : it % 4;
    std::vector<int16_t> buf(LongTables::kMaxBins + 8);
    for (auto &x : buf) x = static_cast<int16_t>(rng() & 0xFFFF);
    make_row(rng, nb, kind, buf.data());
    memset(lds.data(), 0xA5, lds.size());
    lmc::cgdec::host_lds_base() = lds.data();
    const int lane = static_cast<int>(rng() % kLanes);
    LongTables tb;
    tb.bind(lds.data(), lane, 0);
    tb.one.row.r = buf.data();
    tb.one.nb = nb;
    tb.clear();
    tb.build(dummy);
    tb.one.finish();
    (tb.irregular ? irregular : tb.longs ? with_long : regular) += 1;
    uint32_t *ring = reinterpret_cast<uint32_t *>(lds.data() + kRingAt) + lane;
    for (int k = 0; k < 4; ++k) {
      const int T = 1 + static_cast<int>(rng() % 700);
      const uint32_t len = static_cast<uint32_t>(rng() % 1200);
      const uint32_t off = static_cast<uint32_t>(rng() % 16);
      std::vector<uint8_t> bytes(16 * ((off + len + 15) / 16) + 16);
      for (auto &x : bytes) x = static_cast<uint8_t>(rng());
      std::vector<uint8_t> want(T), got(T + 4);
      const int32_t prefix = static_cast<int32_t>(len);
      oc_decode(buf.data(), bytes.data() + off, len, &prefix, 1, T, 1, nb, want.data());
      const uint32_t end = off + len;
      auto put = [&](uint32_t chunk) {
        for (uint32_t d = 4 * chunk; d < 4 * chunk + 4; ++d) {
          uint32_t v = 0;
          for (uint32_t b = 0; b < 4; ++b)
            if (4 * d + b < end && len) v |= static_cast<uint32_t>(bytes[4 * d + b]) << (8 * b);
          ring[(d & (RingCursor::kBytes / 4 - 1)) * kLanes] = v;
        }
      };
      uint32_t filled = 8;
      for (uint32_t c = 0; c < filled; ++c) put(c);
      const uint32_t column = kRingAt + 4u * static_cast<uint32_t>(lane);
      auto refill = [&](uint32_t q_before) {
        uint32_t room = (RingCursor::kBytes - (16 * filled - q_before)) >> 4;
        room = room < 2 ? room : 2;
        for (uint32_t u = 0; u < room; ++u) put(filled + u);
        filled += room;
      };
      if (!tb.irregular) {
        PairCursor cur;
        cur.start(tb, column, 8 * off);
        for (int t0 = 0; t0 < T; t0 += 16) {
          const uint32_t q0 = cur.ring.q;
          for (int t = t0; t < t0 + 16 && t < T; t += 2) {
            uint32_t e0, e1;
            cur.pair(tb, e0, e1);
            got[t] = static_cast<uint8_t>((e0 >> 3) & 31u);
            got[t + 1] = static_cast<uint8_t>((e1 >> 3) & 31u);
          }
          refill(q0);
        }
      } else {
        RingCursor cur;
        cur.start(column, 8 * off);
        for (int t = 0; t < T; t += 16) {
          const uint32_t q0 = cur.q;
          for (int i = t; i < t + 16 && i < T; ++i) {
            int s, n;
            tb.search(cur.hi() >> 16, s, n);
            got[i] = static_cast<uint8_t>(s);
            cur.advance(static_cast<uint32_t>(n));
          }
          refill(q0);
        }
      }
      for (int t = 0; t < T; ++t)
        if (got[t] != want[t]) {
          printf("MISMATCH row %d (nb %d, kind %d, irregular %d) stream %d token %d of %d: got %d want %d\n", it, nb,
                 kind, tb.irregular ? 1 : 0, k, t, T, got[t], want[t]);
          return 1;
        }
      // The step cursor over its own smaller ring, refilled every 16 steps.
      if (!tb.irregular) {
        using lmc::cgdec::StepCursor;
        constexpr uint32_t kDw = StepCursor::Ring::kBytes / 4;
        auto put_small = [&](uint32_t chunk) {
          for (uint32_t d = 4 * chunk; d < 4 * chunk + 4; ++d) {
            uint32_t v = 0;
            for (uint32_t b = 0; b < 4; ++b)
              if (4 * d + b < end && len) v |= static_cast<uint32_t>(bytes[4 * d + b]) << (8 * b);
            ring[(d & (kDw - 1)) * kLanes] = v;
          }
        };
        uint32_t have = 8;
        for (uint32_t c = 0; c < have; ++c) put_small(c);
        StepCursor sc;
        sc.start(tb, column, 8 * off, 0);
        int t = 0;
        while (t < T) {
          const uint32_t q0 = sc.ring.q;
          for (int i = 0; i < 8; ++i)
            sc.pair(tb, ~0u, [&](uint32_t e, bool counts) {
              if (counts && t < T) got[t] = static_cast<uint8_t>(e >> 3);
              t += counts ? 1 : 0;
            });
          if (16 * have - q0 <= StepCursor::Ring::kBytes - 16) put_small(have++);
        }
        for (int u = 0; u < T; ++u)
          if (got[u] != want[u]) {
            printf("STEP MISMATCH row %d (nb %d, kind %d) stream %d token %d of %d: got %d want %d\n", it, nb, kind, k,
                   u, T, got[u], want[u]);
            return 1;
          }
      }
      symbols += T;
    }
  }
  printf("ok rows=%d (short codes %lld, long codes %lld, irregular %lld) symbols=%lld\n", rows, regular, with_long,
         irregular, symbols);
  return regular > 0 && with_long > 0 && irregular > 0 ? 0 : 1;
}
