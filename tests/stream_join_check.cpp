// Checks the order that StreamJoin (powersparse_amd/host/stream_join.h) gives a
// dispatcher's launch, over every mix of three streams: null, blocking or
// non-blocking, with or without work left, and the null stream likewise. The
// runtime's calls are replaced by ones that record what waits for what; a launch
// is ordered behind a stream's work when it goes to that stream, when an event
// recorded there is waited on by the launch's stream, or by the rule of the null
// stream (it and blocking streams wait for each other, non-blocking ones do
// not).
#include <cstdio>
#include <set>
#include <string>

#include "stream_join.h"

namespace {

struct Stream {
  bool blocking = true;
  bool busy = false;
};
Stream null_stream;
Stream* of(ps_stream_t s) { return s ? reinterpret_cast<Stream*>(s) : &null_stream; }

struct Event {
  Stream* recorded = nullptr;
};
std::set<std::pair<Stream*, Stream*>> waits;  // (waiting, awaited)
int live_events = 0;

bool ordered(Stream* launch, Stream* work) {
  if (launch == work || waits.count({launch, work})) return true;
  if (launch == &null_stream) return work->blocking;
  return work == &null_stream && launch->blocking;
}

}  // namespace

extern "C" {
const char* ps_last_error(void) { return ""; }
int ps_stream_idle(ps_stream_t s, int* idle) {
  *idle = !of(s)->busy;
  return PS_OK;
}
int ps_event_create(ps_event_t* e) {
  *e = reinterpret_cast<ps_event_t>(new Event);
  ++live_events;
  return PS_OK;
}
int ps_event_destroy(ps_event_t e) {
  delete reinterpret_cast<Event*>(e);
  --live_events;
  return PS_OK;
}
int ps_event_record(ps_event_t e, ps_stream_t s) {
  reinterpret_cast<Event*>(e)->recorded = of(s);
  return PS_OK;
}
int ps_stream_wait_event(ps_stream_t s, ps_event_t e) {
  waits.insert({of(s), reinterpret_cast<Event*>(e)->recorded});
  return PS_OK;
}
}

namespace PowerSparse {
void ThrowOnError(int status) {
  if (status != PS_OK) throw status;
}
}  // namespace PowerSparse

int main() {
  // per place: 0 null, 1-2 blocking idle / busy, 3-4 non-blocking idle / busy,
  // 5 the stream of the place before
  int wrong = 0, cases = 0;
  for (int null_busy = 0; null_busy < 2; ++null_busy)
    for (int mix = 0; mix < 6 * 6 * 6; ++mix) {
      Stream own[3];
      ps_stream_t given[3];
      std::string text = null_busy ? "null busy:" : "null idle:";
      int m = mix;
      for (int k = 0; k < 3; ++k, m /= 6) {
        const int kind = m % 6;
        own[k].blocking = kind < 3;
        own[k].busy = kind == 2 || kind == 4;
        given[k] = kind == 0                ? nullptr
                   : kind == 5 && k > 0     ? given[k - 1]
                                            : reinterpret_cast<ps_stream_t>(&own[k]);
        const char* const names[] = {" null",          " blocking",          " blocking+work",
                                     " non-blocking",  " non-blocking+work", " same"};
        text += names[kind];
      }
      null_stream.busy = null_busy;
      waits.clear();
      bool good = true;
      {
        const PowerSparse::StreamJoin join(3, given);
        Stream* const launch = of(join.Launch());
        if (null_stream.busy) good &= ordered(launch, &null_stream);
        for (ps_stream_t s : given)
          if (of(s)->busy) good &= ordered(launch, of(s));
      }
      good &= live_events == 0;
      ++cases;
      if (!good) {
        std::printf("not ordered: %s\n", text.c_str());
        ++wrong;
      }
    }
  std::printf("%d of %d not ordered\n", wrong, cases);
  return wrong ? 1 : 0;
}
