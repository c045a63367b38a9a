// Checks of the bit-plane core on the host: the boolean rule against the block
// rule table for every state and variant, the wall slots against two half
// blocks, the one-pair shift, and the packing of rows.  Reads the table
// (4 x 65536 u16, lut[v * 65536 + s]) from argv[1].
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../fallingsand3d_amd/csrc/plane_core.h"

using namespace fs3d::plane;

static const int kRing[4] = {0, 1, 3, 2};

// 32 block states and variants through the planes
template <bool WALL>
static u32 run32(const unsigned (&s)[32], const unsigned (&v)[32], u32 w, unsigned (&out)[32]) {
  u32 lo[2][4] = {}, hi[2][4] = {}, v0 = 0, v1 = 0;
  for (int b = 0; b < 32; b++) {
    for (int l = 0; l < 2; l++)
      for (int k = 0; k < 4; k++) {
        const unsigned c = (s[b] >> (2 * (kRing[k] + 4 * l))) & 3u;
        lo[l][k] |= (~c & 1u) << b;
        hi[l][k] |= (c >> 1) << b;
      }
    v0 |= (v[b] & 1u) << b;
    v1 |= (v[b] >> 1) << b;
  }
  const u32 chg = block_rule<WALL>(lo, hi, v0, v1, w);
  for (int b = 0; b < 32; b++) {
    out[b] = 0;
    for (int l = 0; l < 2; l++)
      for (int k = 0; k < 4; k++)
        out[b] |= ((((lo[l][k] >> b) & 1u) ^ 1u) | (((hi[l][k] >> b) & 1u) << 1)) << (2 * (kRing[k] + 4 * l));
  }
  return chg;
}

#define CHECK(c)                                            \
  do {                                                      \
    if (!(c)) {                                             \
      std::printf("FAILED line %d: %s\n", __LINE__, #c);    \
      return 1;                                             \
    }                                                       \
  } while (0)

int main(int argc, char **argv) {
  if (argc < 2) return 2;
  std::vector<uint16_t> lut(4 * 65536);
  FILE *f = std::fopen(argv[1], "rb");
  if (!f || std::fread(lut.data(), 2, lut.size(), f) != lut.size()) return 2;
  std::fclose(f);

  // every state and variant, with and without the wall code (empty wall)
  for (unsigned base = 0; base < 65536; base += 32)
    for (unsigned v = 0; v < 4; v++) {
      unsigned s[32], vv[32], o[32], o2[32];
      for (int b = 0; b < 32; b++) {
        s[b] = base + b;
        vv[b] = (v + b) & 3;
      }
      const u32 c = run32<false>(s, vv, 0, o), c2 = run32<true>(s, vv, 0, o2);
      for (int b = 0; b < 32; b++) {
        const unsigned want = lut[vv[b] * 65536 + s[b]];
        CHECK(o[b] == want && o2[b] == want);
        CHECK(((c >> b) & 1u) == (want != s[b] ? 1u : 0u) && c2 == c);
      }
    }
  // wall slots: the x = 0 and the x = 1 columns of a block, each beside STATIC,
  // whatever the variants of the two half blocks
  for (unsigned base = 0; base < 65536; base += 32)
    for (unsigned v = 0; v < 4; v++) {
      unsigned s[32], vv[32], o[32];
      for (int b = 0; b < 32; b++) {
        s[b] = base + b;
        vv[b] = (v + b) & 3;
      }
      const u32 w = 0xFFFF0FF1u;
      run32<true>(s, vv, w, o);
      for (int b = 0; b < 32; b++) {
        unsigned want = lut[vv[b] * 65536 + s[b]];
        if ((w >> b) & 1u) {
          const unsigned m0 = 0x3333u, m1 = 0xCCCCu, st = 0x5555u;
          for (unsigned q = 0; q < 4; q++) {
            const unsigned l = lut[q * 65536 + ((s[b] & m0) | (st & m1))] & m0;
            const unsigned r = lut[((q + v) & 3) * 65536 + ((s[b] & m1) | (st & m0))] & m1;
            CHECK(o[b] == (l | r));
          }
        } else {
          CHECK(o[b] == want);
        }
      }
    }
  std::mt19937 rng(7);
  for (int n = 0; n < 2000; n++) {
    // shifts: three words of odd cells, the middle one shifted and back
    u32 wds[3];
    for (u32 &x : wds) x = rng();
    const u32 l = shift_in(wds[1], wds[0]), ln = shift_in(wds[2], wds[1]);
    for (int j = 0; j < 32; j++) {
      const u32 want = j ? (wds[1] >> pair_bit(j - 1)) & 1u : (wds[0] >> pair_bit(31)) & 1u;
      CHECK(((l >> pair_bit(j)) & 1u) == want);
    }
    CHECK(shift_back(l, ln) == wds[1]);
    // rows: 64 cells packed, bit by bit, and unpacked
    u32 d[16], w[4], back[16];
    for (u32 &x : d) x = rng() & 0x03030303u;
    pack_word(d, w);
    for (int x = 0; x < 64; x++) {
      const u32 c = (d[x >> 2] >> (8 * (x & 3))) & 3u;
      const int b = pair_bit(x >> 1);
      CHECK(((w[x & 1] >> b) & 1u) == (c & 1u) && ((w[2 + (x & 1)] >> b) & 1u) == (c >> 1));
    }
    unpack_word(w, back);
    for (int k = 0; k < 16; k++) CHECK(back[k] == d[k]);
    // variants: 2 bits per block of each group's word
    const u32 seg = rng() & 63u, vb = rng();
    u32 v0, v1;
    variant_planes(seg, vb, v0, v1);
    for (int j = 0; j < 32; j++) {
      const u32 bx = 32 * seg + j, word = mix32((bx >> 4) * 0x9E3779B1u + vb);
      const u32 v = (word >> (2 * (bx & 15))) & 3u;
      CHECK(((v0 >> pair_bit(j)) & 1u) == (v & 1u) && ((v1 >> pair_bit(j)) & 1u) == (v >> 1));
    }
  }
  std::printf("plane checks passed\n");
  return 0;
}
