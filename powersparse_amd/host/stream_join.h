// The stream of a dispatcher's fused launch.
#pragma once

#include <algorithm>
#include <vector>

#include "matrix_utils.h"

namespace PowerSparse {

// The reference runs workset s on streams[s] (spmm_solution.cu:18-26,
// sddmm_solution.cu:24-26), so work a caller queued on streams[s] before the
// call runs before that workset; work queued on the null stream (the outputs'
// clearing, usually) runs before every workset on a blocking stream. The fused
// launch runs behind all of it, whatever the streams' kind:
// - no work left on the supplied streams: on the null stream, behind what is
//   queued there. Ordering a created stream behind the null stream costs about
//   36 us on MI355X (a 10 k-node SDDMM N = 32 after its clearing: 66 us a call
//   so, 25 us on the null stream), and asking whether the null stream has work
//   left about 20 (44 us a call). On the null stream the launch also runs behind
//   the process's other blocking streams; two threads with a matrix and streams
//   each lose nothing by it (C1 graphs of 10 k to 500 k nodes, a pair of calls:
//   40 / 145 / 334 / 1896 us, 53 / 147 / 343 / 1917 on streams[0]).
// - work left on a supplied stream: on streams[0], into which every other
//   stream with work left, the null stream included, is joined by an event
//   (released after the dispatcher's device synchronisation). A non-blocking
//   streams[0] would not wait for the null stream by itself.
class StreamJoin {
 public:
  StreamJoin(int count, const ps_stream_t* streams) {
    std::vector<ps_stream_t> busy;
    for (int s = 0; s < count; ++s)
      if (streams[s] && std::find(streams, streams + s, streams[s]) == streams + s &&
          Busy(streams[s]))
        busy.push_back(streams[s]);
    if (busy.empty()) return;
    launch_ = streams[0];
    if (launch_ && Busy(nullptr)) busy.push_back(nullptr);
    for (ps_stream_t s : busy) {
      if (s == launch_) continue;
      ps_event_t e = nullptr;
      ThrowOnError(ps_event_create(&e));
      events_.push_back(e);
      ThrowOnError(ps_event_record(e, s));
      ThrowOnError(ps_stream_wait_event(launch_, e));
    }
  }
  ~StreamJoin() {
    for (ps_event_t e : events_) ps_event_destroy(e);
  }
  StreamJoin(const StreamJoin&) = delete;
  StreamJoin& operator=(const StreamJoin&) = delete;

  // The stream of the fused launch.
  ps_stream_t Launch() const { return launch_; }

 private:
  static bool Busy(ps_stream_t s) {
    int idle = 1;
    ThrowOnError(ps_stream_idle(s, &idle));
    return !idle;
  }

  std::vector<ps_event_t> events_;
  ps_stream_t launch_ = nullptr;
};

}  // namespace PowerSparse
