// Host checks of the step's continuation and of the features' quotients.  Built and run by
// tests/test_cpu_engine_step.py (host code only; no GPU):
//  1. continue_postchance (apply in place, probe only where a failure needs it, the state
//     put back by reload()) == the reference's order (postchance50.h:509-539: probe, then
//     apply on a copy) on the rows of random games and on rows with random fields changed,
//     pending choices and pi selections among them: same status, commit and row;
//  2. quotient<S>(v) == v / S in float, bit for bit, for every v below 65,536 and every
//     scale of the encoder.
// Prints one line per check and exits non-zero on the first mismatch.
#include "engine.h"

#include <cstdio>
#include <cstring>
#include <random>

using namespace cugo_amd;

// postchance50.h:509-539 as it stands: the probe, then the apply on a copy that is kept only
// on success.
static u8 continue_plain(Env& e, bool& committed) {
  committed = false;
  Pending p = pending_of(e);
  Action a = p.action;
  if (p.sel_pi != 0) a.pisel = p.sel_pi;
  Env staged;
  const Probe probe = probe_postchance_per_kind(e, p, staged);
  if (probe.status != kOk) return probe.status;
  if (probe.decision != kDecNone) return kOk;
  Env applied = e;
  const u8 s = apply_action(applied, a);
  if (s != kOk) return s;
  e = applied;
  p.action = a;
  p.active = 0;
  set_pending(e, p);
  committed = true;
  return kOk;
}

static u16 random_legal(const Mask3& m, std::mt19937_64& g) {
  const u64 w[3] = {m.w0, m.w1, m.w2};
  const u32 c = popc(w[0]) + popc(w[1]) + popc(w[2]);
  if (c == 0) return kInvalidAction16;
  u32 r = (u32)(g() % c);
  for (u32 i = 0; i < 3; ++i) {
    if (r < popc(w[i])) return (u16)(64 * i + select_rank_in(w[i], r));
    r -= popc(w[i]);
  }
  return kInvalidAction16;
}

static int check_continue(std::mt19937_64& g) {
  long cases = 0, commits = 0, waiting = 0, selected = 0, failed = 0;
  for (int game = 0; game < 6000; ++game) {
    u64 row[kRowWords];
    pack_row(create_env(g(), (u32)(g() & 1)), row);
    for (int t = 0; t < 60; ++t) {
      for (int k = 0; k < 4; ++k) {
        u64 r[kRowWords];
        std::memcpy(r, row, sizeof r);
        if (k > 0) {  // wild rows: some fields changed, some with a pi selection
          for (int q = (int)(g() % 3); q >= 0; --q) r[g() % kRowWords] ^= 1ull << (g() % 64);
          if (g() % 4 == 0) r[26] = g() & g() & kDeckMask;
        }
        Env e = unpack_row(r);
        const PacketHead h = packet_head(e);
        const u16 act = random_legal(h.legal, g);
        if (act == kInvalidAction16) continue;
        if (e.pactive != 0) record_postchance_choice(e, h.decision_kind, (u8)(act - kActChoice));
        else if (stage_postchance(e, act, h.legal) != kOk) continue;
        ++e.n_choice;  // a counter the step raises before it continues
        Env a = e, b = e;
        bool ca = false, cb = false;
        const u8 sa = continue_postchance(a, ca, [&] { return unpack_row(r); });
        const u8 sb = continue_plain(b, cb);
        u64 ra[kRowWords], rb[kRowWords];
        pack_row(a, ra);
        pack_row(b, rb);
        ++cases;
        commits += ca;
        selected += e.sel_pi != 0;
        waiting += sa == kOk && !ca;
        failed += sa != kOk;
        if (sa != sb || ca != cb || std::memcmp(ra, rb, sizeof ra) != 0) {
          std::printf("continue: game %d turn %d action %u: status %u/%u commit %d/%d\n", game, t,
                      act, sa, sb, ca, cb);
          return 1;
        }
      }
      Env e = unpack_row(row);
      if (e.done) break;
      const u16 act = random_legal(packet_head(e).legal, g);
      if (act == kInvalidAction16) break;
      torch_step(e, act);
      pack_row(e, row);
    }
  }
  std::printf("continue: %ld cases (%ld committed, %ld left pending, %ld failed, %ld with a pi "
              "selection) equal\n", cases, commits, waiting, failed, selected);
  return commits > 1000 && waiting > 1000 && failed > 1000 && selected > 1000 ? 0 : 1;
}

template <u32 kScale>
static int check_quotient() {
  for (u32 v = 0; v < 65536; ++v) {
    volatile float x = (float)v, y = (float)kScale;
    const float want = x / y, got = quotient<kScale>(v);
    if (std::memcmp(&want, &got, 4) != 0) {
      std::printf("quotient: %u / %u\n", v, kScale);
      return 1;
    }
  }
  return 0;
}

int main() {
  std::mt19937_64 g(20261204);
  if (check_continue(g)) return 1;
  if (check_quotient<3>() || check_quotient<4>() || check_quotient<5>() || check_quotient<8>() ||
      check_quotient<10>() || check_quotient<20>() || check_quotient<30>() ||
      check_quotient<32>() || check_quotient<50>() || check_quotient<64>() ||
      check_quotient<kActPrimaryCount>())
    return 1;
  std::printf("quotients: 11 scales x 65536 values equal\n");
  return 0;
}
