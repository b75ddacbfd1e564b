// What the torch host layer uses of libsba.so besides the C ABI: a forward that prepares the schedule of the backward that
// follows it (tile lists, cursors, cleared flags), so that the backward needs no scheduler launch of its own; and which backward a call runs.
#pragma once
#include "../../include/sba.h"

namespace sba {

// Sizes: of the schedule, of the backward's workspace besides it, of what makes it faster behind that, and of `carry`; whether the schedule
// has parts per row and head (and not only per tile).
struct Prepared {
  size_t schedule, rest, laid, carry;
  bool row_parts;
};
int prepared_bytes(const SbaArgs* a, Prepared* out);
// sba_fwd with the schedule in a->workspace (`schedule` bytes of it).
int forward_prepared(const SbaArgs* a);
// sba_fwd for a call that no backward follows: a max_seqlen below the longest sequence then voids it only where the carry capacity does.
int forward_alone(const SbaArgs* a);
// Whether the backward these arguments describe can run on the schedule its forward prepared.
bool prepared_fits(const SbaArgs* a);
// sba_bwd on that schedule, with the rest in a->workspace.  The schedule serves ONE backward: its cursors are used up.
int backward_prepared(const SbaArgs* a, void* sched);

// What sba_bwd would run for these arguments on the current device, with this workspace: the form of its first pass (of its longer sequences,
// where those of up to 64 tokens are taken apart from them), and the heads that pass takes (all, unless they go through in groups or are split between two forms).
enum : int32_t { kBwdTwoKernels = 0, kBwdKeyTiles = 1, kBwdRowTiles = 2, kBwdTiny = 3 };
struct BackwardRoute {
  int32_t form, heads;
};
int backward_route(const SbaArgs* a, BackwardRoute* out);
// One pass of sba_bwd whose tiles wait for each other for so many polls only (a workspace for all heads).
int backward_with_polls(const SbaArgs* a, int32_t polls);

}  // namespace sba
