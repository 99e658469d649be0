// A call of several launches whose first one takes something on the device that a later one gives back.
#pragma once

namespace ds41g {

// launch(i) enqueues launch i of `count` and returns its error, 0 if it was enqueued. At the first error
// nothing more of the call is enqueued; what launch 0 took is then given back by give_back(), whose own
// error is of no use to the caller. Returns the first error.
template <class Launch, class GiveBack>
int launch_sequence(int count, const Launch &launch, const GiveBack &give_back) {
  for (int i = 0; i < count; ++i)
    if (const int rc = launch(i)) {
      if (i > 0) give_back();
      return rc;
    }
  return 0;
}

}  // namespace ds41g
