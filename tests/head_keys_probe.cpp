// The head's keys of the persistent decode kernel, as host arithmetic: the
// two sets of keys as memory, every workgroup's alike, under schedules of
// launches that turn a 16-bit tag around (ana_feed's launches, which run no
// head; loops; loops stopped by a NaN; loops that time out). Before a head
// writes its set, the set must not carry its tag: a poll would take the old
// keys for this head's.
//
// Launches that start from the epoch as it is must find a stale key in the
// schedules marked so: they reach what they are for.
//
// Prints one line per case, "ok <name>" or "FAIL <name> ...", and exits 0
// when every case holds.
#include <cstdint>
#include <cstdio>

#include "ana_internal.h"

using namespace ana;

static int fails = 0;

struct Host {
  bool plain;                  // launches start from the epoch as it is
  uint32_t epoch = 0;
  uint32_t keys[2] = {0, 0};   // the tags in the two sets; zeroed at open
  HeadKeys hk;
  uint64_t stale = 0;

  void feed() { epoch += 3; }
  // a launch of `steps` that picks `ran` of them; short of that it stops on
  // a head of its own (a NaN), or on a time-out
  void loop(uint32_t steps, uint32_t ran, bool timeout = false) {
    const uint32_t ctl[4] = {timeout, timeout, ran, ran < steps && !timeout};
    const uint32_t was = epoch;
    if (!plain) epoch = hk.start(epoch);
    if (epoch - was > 4) stale++;   // (a few epochs skipped at most)
    for (uint32_t k = 0; k < ctl[2] + ctl[3]; k++) {
      const uint32_t ep = epoch + k + 1;
      if (keys[ep & 1] == (ep & 0xFFFFu)) stale++;
      keys[ep & 1] = ep & 0xFFFFu;
    }
    if (timeout) {
      if (!plain) keys[0] = keys[1] = 0;
      hk.cleared();
    } else {
      hk.ran(epoch, ctl);
    }
    epoch += steps + 2;
  }
};

template <typename F>
static void run(const char* name, bool plain_stale, F&& schedule) {
  Host a{false}, b{true};
  schedule(a);
  schedule(b);
  const bool ok = a.stale == 0 && (b.stale != 0) == plain_stale;
  if (!ok) fails++;
  printf("%s %s (stale %llu, plain %llu)\n", ok ? "ok" : "FAIL", name, (unsigned long long)a.stale,
         (unsigned long long)b.stale);
}

int main() {
  run("loops alone, four turns", false, [](Host& h) {
    for (int i = 0; i < 300; i++) h.loop(1024, 1024);
  });
  run("feeds, then the context's first loop", true, [](Host& h) {
    for (int i = 0; i < 21845; i++) h.feed();
    h.loop(3, 3);
  });
  for (uint32_t between : {21844u, 43689u, 65535u})
    run("feeds between two loops", true, [&](Host& h) {
      h.loop(5, 5);
      for (uint32_t i = 0; i < between; i++) h.feed();
      h.loop(5, 5);
    });
  run("a step and feeds in turn", false, [](Host& h) {
    for (uint32_t i = 0; i < 70000; i++) {
      h.loop(1, 1);
      for (uint32_t j = 0; j < i % 4; j++) h.feed();
      if (i % 30000 == 29999)
        for (uint32_t j = 0; j < 21844; j++) h.feed();
    }
  });
  run("loops stopped at their first step", false, [](Host& h) {
    for (uint32_t i = 0; i < 70000; i++) h.loop(2, 0);
    h.loop(64, 64);
  });
  run("loops that time out", true, [](Host& h) {
    for (uint32_t i = 0; i < 70000; i++) {
      h.loop(7, i % 3, true);
      h.loop(3, 3);
      if (i % 20000 == 19999)
        for (uint32_t j = 0; j < 21844; j++) h.feed();
    }
  });
  Host h{false};
  h.epoch = 0xFFFFFFFFu - 30;
  for (int i = 0; i < 9; i++) h.loop(1 + i, 1 + i);
  if (h.stale) fails++;
  printf("%s the epoch's own turn\n", h.stale ? "FAIL" : "ok");
  printf("%d failed\n", fails);
  return fails ? 1 : 0;
}
