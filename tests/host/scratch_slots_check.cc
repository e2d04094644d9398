// Scratch slots of streams (csrc/scratch_slots.h): one a stream, free again when a stream whose work is done goes away,
// and nobody's where that is not known.
#include <cstdio>

#include "../../mshadow_amd/csrc/scratch_slots.h"

static int g_wrong = 0;
static void Is(const char *what, int got, int want) {
  if (got == want) return;
  ++g_wrong;
  printf("%s: %d, not %d\n", what, got, want);
}

int main() {
  static mshadow_abi::ScratchSlots<3> t = {};
  char handle[6];
  const char *a = handle, *b = handle + 1, *c = handle + 2, *d = handle + 3;
  Is("none yet", t.Has(a), 0);
  Is("first", t.Take(0, a), 0);
  Is("second", t.Take(0, b), 1);
  Is("again", t.Take(0, a), 0);
  Is("default stream", t.Take(0, nullptr), 2);
  Is("all taken", t.Take(0, c), -1);
  Is("another device", t.Take(1, c), 0);
  Is("of any device", t.Has(c), 1);
  t.Release(b, true);
  Is("gone", t.Has(b), 0);
  Is("freed", t.Take(0, c), 1);
  Is("new stream of the same handle", t.Take(0, b), -1);
  // work that may still be running: the slot goes to no one else, nor to a new stream of that handle
  t.Release(a, false);
  Is("not known to be done", t.Has(a), 0);
  Is("kept from others", t.Take(0, d), -1);
  Is("kept from its handle", t.Take(0, a), -1);
  Is("the others' stay", t.Take(0, c), 1);
  t.Release(c, true);
  Is("on this device", t.Take(0, d), 1);
  Is("and on the other", t.Take(1, d), 0);
  if (g_wrong == 0) printf("OK\n");
  return g_wrong != 0;
}
