// Host driver for tests/test_fr29_cpu.py: runs Fr29 (the transforms' signed
// 29-bit limbs) on the CPU.  Built with hipcc as host code.
//
// Input:
// "inv A" prints the inverse of the element A (x 2^256 -> x^-1 2^256) by both of
// inverse()'s constants, plain and up.
// "chain A B N" and N lines "W" (canonical x 2^256 mod r, 64 hex digits).
// Step i takes the butterfly (a, b) -> (a + b W_i, a - b W_i) with the factor b
// as the step before left it and a normalised every second step only, as a quad
// of a pass does, and swaps the two on odd i.  Output per step: both values
// after reduce(), as words, and whether their limbs were within the bounds.
#include <cstdio>
#include <cstring>

#include "../zkpoly-compiler_amd/csrc/field/fr29.hpp"

using namespace zkp;

static bool read_hex(const char* s, u32 (&w)[8]) {
  if (strlen(s) != 64) return false;
  for (int k = 0; k < 8; k++) {
    unsigned v = 0;
    if (sscanf(s + 8 * (7 - k), "%8x", &v) != 1) return false;
    w[k] = v;
  }
  return true;
}

static void print_reduced(const Fr29& a) {
  u32 w[8];
  a.reduce().to_words(w);
  for (int k = 7; k >= 0; k--) printf("%08x", w[k]);
}

// limbs 0..7 strictly inside (-3 2^29, 3 2^29), limb 8 inside (-2^28, 2^28)
static bool in_bounds(const Fr29& a) {
  for (int i = 0; i < 8; i++)
    if ((int64_t)a.l[i] <= -3ll << 29 || (int64_t)a.l[i] >= 3ll << 29) return false;
  return a.l[8] > -(1 << 28) && a.l[8] < 1 << 28;
}

int main() {
  char sa[128], sb[128];
  int n;
  char op[16];
  while (scanf(" %15s", op) == 1) {
    u32 w[8];
    if (strcmp(op, "inv") == 0) {
      if (scanf(" %127s", sa) != 1 || !read_hex(sa, w)) return 2;
      print_reduced(Fr29Inverse::inverse(Fr29::from_words<0>(w), Fr29Inverse::INV_PLAIN));
      printf(" ");
      print_reduced(Fr29Inverse::inverse(Fr29::from_words<5>(w).reduce(), Fr29Inverse::INV_UP));
      printf("\n");
      continue;
    }
    if (scanf(" %127s %127s %d", sa, sb, &n) != 3) return 2;
    if (!read_hex(sa, w)) return 2;
    Fr29 a = Fr29::from_words<0>(w);
    if (!read_hex(sb, w)) return 2;
    Fr29 b = Fr29::from_words<0>(w);
    for (int i = 0; i < n; i++) {
      if (scanf(" %127s", sa) != 1 || !read_hex(sa, w)) return 2;
      const Fr29 t = Fr29::mul(b, Fr29::from_words<5>(w));
      if (i % 2 == 0) a = a.norm();
      const Fr29 s = a + t, d = a - t;
      a = i & 1 ? d : s;
      b = i & 1 ? s : d;
      print_reduced(a);
      printf(" ");
      print_reduced(b);
      printf(" %d\n", in_bounds(a) && in_bounds(b));
    }
  }
  return 0;
}
