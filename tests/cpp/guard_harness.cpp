// Drives csrc/ring_guard.hpp over a made-up runtime: streams are numbers, an event remembers its stream and how much was
// queued there, and every call is noted.  Exits with the number of the first expectation that does not hold.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <string>
#include <thread>
#include <utility>

#include "ring_guard.hpp"

struct Ev { int st = 0, at = 0; };

struct Fake {
  using Stream = int;              // 0: none, -1: the calling thread's own
  using Event = Ev;
  static thread_local int thread;
  static std::map<int, int> queued, finished;      // launches per stream (per-thread streams: -1 - thread)
  static std::set<int> capture, gone;
  static std::set<std::pair<int, int>> order;      // (stream, stream it waits for)
  static int records, quiet;

  struct Quiet {
    Quiet() { ++quiet; }
    ~Quiet() { --quiet; }
  };
  static int real(Stream st) { return st == -1 ? -1 - thread : st; }
  static unsigned long owner(Stream st) { return st == -1 ? (unsigned long)thread : 0; }
  static bool capturing(Stream st) { return capture.count(real(st)) != 0; }
  static bool record(Event& ev, Stream st) {
    ++records;
    if (quiet == 0) std::exit(2);
    if (gone.count(st)) return false;
    ev = Ev{real(st), queued[real(st)]};
    return true;
  }
  static bool wait(Stream st, Event ev) {
    order.insert({real(st), ev.st});
    return true;
  }
  static bool done(Event ev) { return quiet > 0 && finished[ev.st] >= ev.at; }
};
thread_local int Fake::thread = 1;
std::map<int, int> Fake::queued, Fake::finished;
std::set<int> Fake::capture, Fake::gone;
std::set<std::pair<int, int>> Fake::order;
int Fake::records = 0, Fake::quiet = 0;

using Guard = ResidencyGuard<Fake>;

static int checks = 0;
static void expect(bool ok, const char* what) {
  ++checks;
  if (ok) return;
  std::printf("not so: %s\n", what);
  std::exit(1);
}
static void launch(Guard& g, int st, int held) {
  Guard::Launch l(g, st, held);
  ++Fake::queued[Fake::real(st)];
}
static bool waits(int st, int behind) {
  const bool w = Fake::order.count({st, behind}) != 0;
  Fake::order.clear();
  return w;
}
static void reset() {
  Fake::queued.clear();
  Fake::finished.clear();
  Fake::capture.clear();
  Fake::gone.clear();
  Fake::order.clear();
  Fake::records = 0;
}

int main() {
  {
    Guard g(32);
    for (int i = 0; i < 5; ++i) launch(g, 1, 31);
    expect(Fake::records == 0 && Fake::order.empty(), "one stream records nothing and waits for nothing");
    launch(g, 2, 31);
    expect(waits(2, 1), "two launches that can fill an XCD between them are ordered");
    launch(g, 1, 31);
    expect(waits(1, 2), "and back");
  }
  reset();
  {
    Guard g(32);
    launch(g, 1, 3);
    launch(g, 2, 3);
    launch(g, 3, 15);
    expect(Fake::order.empty(), "launches that fit an XCD between them run side by side");
    launch(g, 4, 15);
    expect(Fake::order.size() == 3, "the one that does not fit any more waits for all");
  }
  reset();
  {
    Guard g(32);
    launch(g, 1, 31);                     // teams of 32
    launch(g, 2, 3);                      // a cluster launch
    expect(waits(2, 1), "clusters and full-width teams are ordered");
    launch(g, 3, 15);
    expect(waits(3, 1), "a launch is still counted when another one waits for it");
  }
  reset();
  {
    Guard g(32);
    launch(g, 1, 31);
    Fake::finished[1] = 1;
    launch(g, 2, 31);
    expect(Fake::order.empty(), "finished launches are not waited for");
    launch(g, 2, 31);
    const int n = Fake::records;
    launch(g, 2, 31);
    expect(Fake::records == n, "and a program back on one stream records nothing again");
  }
  reset();
  {
    Guard g(32);
    launch(g, 1, 31);
    launch(g, 2, 31);                     // from here on every launch is marked as it is made
    Fake::order.clear();
    launch(g, 1, 31);
    Fake::order.clear();
    Fake::capture.insert(1);
    launch(g, 2, 31);
    expect(waits(2, 1), "an earlier launch of a stream that is capturing now is waited for");
    launch(g, 1, 31);
    expect(Fake::order.empty(), "nothing is waited for under capture");
  }
  reset();
  {
    Guard g(32);
    launch(g, -1, 31);
    expect(Fake::records == 1, "a per-thread stream is marked at once: no other thread could");
    std::thread([&] {
      Fake::thread = 2;
      launch(g, -1, 31);
    }).join();
    expect(waits(-3, -2), "the same per-thread handle in two threads is two streams");
  }
  reset();
  {
    Guard g(32);
    launch(g, 1, 31);
    Fake::gone.insert(1);
    launch(g, 2, 31);
    expect(Fake::order.empty(), "a stream that is gone is forgotten");
  }
  reset();
  {
    Guard g(32);
    expect(g.beside(1) == 0, "nobody is beside the first launch");
    launch(g, 1, 15);
    expect(g.beside(1) == 0 && Fake::records == 0, "a stream is not beside itself");
    expect(g.beside(2) == 1, "an unfinished launch of another stream is");
    launch(g, 2, 7);
    expect(g.beside(1) == 1 && g.beside(3) == 2, "streams are counted, not launches");
    launch(g, 2, 15);
    expect(g.beside(1) == 1 && g.beside(3) == 2, "however many units their launches hold");
    Fake::finished[1] = 1;
    expect(g.beside(3) == 1 && g.beside(2) == 0, "finished launches are not");
    Fake::capture.insert(3);
    const int n = Fake::records;
    expect(g.beside(3) == -1 && Fake::records == n, "a capturing stream does not know");
  }
  reset();
  {
    Guard g(32);
    launch(g, 1, 15);
    launch(g, 1, 7);
    launch(g, 1, 15);
    expect(Fake::records == 0, "one stream records nothing, whatever its launches hold");
  }
  reset();
  {
    Guard g(32);
    launch(g, 1, 15);
    launch(g, 2, 15);
    Fake::order.clear();
    for (int i = 0; i < 3; ++i) launch(g, 1, 7), launch(g, 2, 7);
    expect(Fake::order.empty(), "a narrow launch runs beside a wide one");
    launch(g, 3, 7);
    expect(waits(3, 1), "what is queued holds what its widest launch does");
    Fake::finished[1] = Fake::finished[2] = 1;
    launch(g, 4, 7);
    expect(Fake::order.empty(), "until that one has finished");
  }
  std::printf("guard ok: %d\n", checks);
  return 0;
}
