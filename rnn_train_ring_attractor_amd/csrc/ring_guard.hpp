// Order between streams of launches whose workgroups wait for each other (team and cluster kernels).
//
// Workgroups of one launch become resident in order on every XCD, so of the groups of G workgroups that wait for each
// other at most one per XCD is incomplete and holds up to G - 1 compute units for nothing.  Launches that could hold all
// compute units of an XCD between them in this way would starve each other: those run one after the other.  All others
// run side by side.  This spares time; that a starved launch still ends with its result is the kernels' part (a team that
// does not gather gives up, see ring_team.hpp), and it is all there is for launches this guard cannot order: of other
// processes, in replayed graphs (nothing is recorded or waited for under capture), and a stream's earlier ones when that
// stream is capturing by the time the first event is due.
//
// A program with one stream pays nothing: the first event of a stream is recorded when a second stream comes along (so it
// stands for all that was queued until then), and behind every launch from then on.
//
// A stream's launches run one after the other, so it holds what the widest of its unfinished ones does: launches that hold
// different numbers of units are kept apart, each number with the event behind the last launch of it, so that one wide launch
// at the head of a long queue does not count for all that is queued behind it.
#pragma once
#include <mutex>
#include <vector>

// Rt: Stream, Event, and
//   unsigned long owner(Stream)        which thread's stream the handle means (0: the same for all threads)
//   bool capturing(Stream)
//   bool record(Event&, Stream)        makes the event if there is none yet
//   bool wait(Stream, Event)
//   bool done(Event)
//   Rt::Quiet                          held around calls that another thread's capture must not notice
template <typename Rt>
class ResidencyGuard {
 public:
  using Stream = typename Rt::Stream;

  explicit ResidencyGuard(int units) : units_(units) {}

  // Held around one launch on `st` that can hold `held` units of an XCD while it waits for the rest.
  class Launch {
   public:
    Launch(ResidencyGuard& g, Stream st, int held) : g_(g), lock_(g.mu_), st_(st), held_(held), plain_(!Rt::capturing(st)) {
      if (plain_) g_.enter(st, held);
    }
    ~Launch() {
      if (plain_) g_.leave(st_, held_);
    }
    Launch(const Launch&) = delete;
    Launch& operator=(const Launch&) = delete;

   private:
    ResidencyGuard& g_;
    std::lock_guard<std::mutex> lock_;
    Stream st_;
    int held_;
    bool plain_;
  };

  // How many streams other than `st` have launches that have not finished; -1: `st` is capturing, and what its graph will be
  // replayed beside nobody knows.
  int beside(Stream st) {
    std::lock_guard<std::mutex> lock(mu_);
    if (Rt::capturing(st)) return -1;
    int n = 0;
    if (settle(st))
      for (size_t i = 0; i < entries_.size(); ++i) n += !mine(entries_[i], st) && widest(i);
    return n;
  }

 private:
  struct Entry {          // the unfinished launches of a stream that hold so many units, as far as known
    Stream st{};
    unsigned long owner = 0;
    int held = 0;
    typename Rt::Event ev{};
    bool marked = false;  // the event stands behind the last launch
  };

  bool mine(const Entry& e, Stream st) const { return e.st == st && e.owner == Rt::owner(st); }

  // Of a stream's entries the first of those that hold most.
  bool widest(size_t i) const {
    const Entry& e = entries_[i];
    for (size_t j = 0; j < entries_.size(); ++j)
      if (j != i && entries_[j].st == e.st && entries_[j].owner == e.owner && (entries_[j].held > e.held || (entries_[j].held == e.held && j < i)))
        return false;
    return true;
  }

  bool others(Stream st) const {
    for (const Entry& e : entries_)
      if (!mine(e, st)) return true;
    return false;
  }

  // Marks what other streams have queued and forgets what of it has finished.  Whether any is left.
  bool settle(Stream st) {
    if (!others(st)) return false;
    typename Rt::Quiet quiet;
    bool left = false;
    for (size_t i = 0; i < entries_.size();) {
      Entry& e = entries_[i];
      if (!mine(e, st)) {
        if (!e.marked && (e.owner == 0 || e.owner == Rt::owner(e.st)) && !Rt::capturing(e.st)) {
          e.marked = Rt::record(e.ev, e.st);
          if (!e.marked) {                        // no such stream any more
            drop(i);
            continue;
          }
        }
        if (e.marked && Rt::done(e.ev)) {
          drop(i);
          continue;
        }
        left = true;
      }
      ++i;
    }
    return left;
  }

  void enter(Stream st, int held) {
    if (settle(st)) {
      typename Rt::Quiet quiet;
      int sum = held;
      for (size_t i = 0; i < entries_.size(); ++i)
        if (!mine(entries_[i], st) && widest(i)) sum += entries_[i].held;
      if (sum >= units_)
        for (const Entry& e : entries_)
          if (!mine(e, st) && e.marked) Rt::wait(st, e.ev);
    }
    for (Entry& e : entries_)
      if (mine(e, st) && e.held == held) {
        e.marked = false;
        return;
      }
    Entry e;
    e.st = st;
    e.owner = Rt::owner(st);
    e.held = held;
    if (!spare_.empty()) {
      e.ev = spare_.back();
      spare_.pop_back();
    }
    entries_.push_back(e);
  }

  void leave(Stream st, int held) {
    if (!others(st) && Rt::owner(st) == 0) return;
    typename Rt::Quiet quiet;
    for (Entry& e : entries_)
      if (mine(e, st) && e.held == held) e.marked = Rt::record(e.ev, st);
  }

  void drop(size_t i) {
    spare_.push_back(entries_[i].ev);
    entries_.erase(entries_.begin() + (long)i);
  }

  const int units_;
  std::mutex mu_;
  std::vector<Entry> entries_;
  std::vector<typename Rt::Event> spare_;
};
