// The device's lookup of sinf / cosf exceptions (rl_trig.h), on the host: for tables
// of no exception, of one per function, and of the largest covered input, every byte
// looked at is in the bitmap and the results are those of the bucketed table.
#include "rl_trig.h"

#include <stdio.h>

#include <vector>

using namespace rltrig;

struct Exceptions {
  std::vector<uint32_t> off;
  std::vector<uint16_t> keys;
  int e_min = 0;
  std::vector<uint8_t> bits;
  explicit Exceptions(uint32_t xb) : off(RLT_NBUCKETS + 1, 0) {  // the one input xb, none if 0
    const uint32_t ab = xb & 0x7fffffffu, b = (ab >> RLT_BUCKET_SHIFT) | (xb >> 31 << RLT_SIGN_SHIFT);
    if (xb) keys.push_back((uint16_t)(ab & 0xfffu));
    for (uint32_t i = 0; i <= RLT_NBUCKETS; ++i) off[i] = xb && i > b ? 1 : 0;
    e_min = table_min_exponent(off.data(), keys.data());
    bits.assign(bitmap_bytes(e_min), 0);
    table_to_bitmap(off.data(), keys.data(), e_min, bits.data());
  }
};

int main() {
  const uint32_t cases[][2] = {{0, 0}, {0, 0x3f800000u}, {0xbf800001u, 0}, {0x42800000u, 0xc2800000u}, {0x38000000u, 0x42800000u}};
  // zeros, subnormals, both ends of each case's bitmap, 64 and just past it, the largest, infinity, NaN
  const uint32_t xs[] = {0u, 1u, 0x7fffffu, 0x37ffffffu, 0x38000000u, 0x3f7fffffu, 0x3f800000u, 0x3f800001u, 0x427fffffu,
                         0x42800000u, 0x42800001u, 0x42800007u, 0x42800008u, 0x42ffffffu, 0x43000000u, 0x7f7fffffu,
                         0x7f800000u, 0x7fc00000u};
  for (const auto& c : cases) {
    Exceptions s(c[0]), k(c[1]);
    const double delta = 0.4999;  // nearly every input is looked up
    const Table ts{s.off.data(), s.keys.data(), delta}, tc{k.off.data(), k.keys.data(), delta};
    for (uint32_t x : xs)
      for (uint32_t sign : {0u, 0x80000000u}) {
        const uint32_t xb = x | sign;
        for (const Exceptions* e : {&s, &k}) {
          bool look = true;
          const uint32_t at = bitmap_byte(e->e_min, xb, &look);
          if (at >= e->bits.size()) {
            printf("table %08x %08x, input %08x: byte %u of %zu\n", c[0], c[1], xb, at, e->bits.size());
            return 1;
          }
        }
        const Bitmap bs{s.bits.data(), s.e_min, delta}, bc{k.bits.data(), k.e_min, delta};
        float a, b, want_a, want_b;
        sincosf_libc_bm(u2f(xb), bs, bc, &a, &b);
        sincosf_libc(u2f(xb), ts, tc, &want_a, &want_b);
        if (((xb & 0x7fffffffu) < 0x43000000u && (f2u(a) != f2u(want_a) || f2u(b) != f2u(want_b))) ||
            (a != a) != (want_a != want_a)) {
          printf("table %08x %08x, input %08x: %a %a instead of %a %a\n", c[0], c[1], xb, a, b, want_a, want_b);
          return 1;
        }
      }
  }
  printf("ok\n");
  return 0;
}
