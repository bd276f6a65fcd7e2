// preprocess.h -- host-side preprocessing (split stencils, alias order,
// sweep dependency levels).
#pragma once

#include <vector>

namespace mfcfd {

// generate_connectivity.f90:12-246.  cnt[d] (N) and lists[d] (22*N + 32)
// for d = xpos, xneg, ypos, yneg, zpos, zneg; point numbers 1-based.
void generate_split_stencils(int n, const double* x, const double* y, const double* z,
                             const double* tan1, const double* tan2, const double* nor,
                             const int* status, const int* nbhs, const int* conn, int* const cnt[6],
                             int* const lists[6]);

// implicit_aliasing.f90:13-44
void aliasing(int n, const int* nbhs, const int* conn, int* alias, int* pwa);

// The LU-SGS sweeps as one plan per sweep direction, built on the host from
// the device-order lists.
//
// The reference visits points in a fixed order -- the alias order of
// point_with_alias (implicit_forward_and_reverse_sweeps.f90:26-85), or the
// type order wall, interior, outer, supersonic inlet, supersonic outlet of
// the alternative driver (implicit_forward_and_reverse_sweeps_backup.f90:
// 25-139) -- and each visited point reads its neighbours' delU in place.  An
// entry a point takes (alias smaller in the forward sweep, larger in the
// backward one) therefore reads this sweep's value of the neighbour when the
// neighbour was visited earlier ("wait" entry), and the value from before
// the sweep otherwise ("old" entry).  A supersonic point copies its nearest
// neighbour's delU under the same rule.
//
// Levels: a point's level is one more than the deepest of (a) the points its
// wait entries read and (b) the earlier-visited points that read it as an old
// entry (they must read before it writes).  Every order by level therefore
// reproduces the visiting order's results, in place (one launch per level) or
// with old values read from a snapshot (the sync-free sweep).
struct SweepDirPlan {
    std::vector<int> seq;             // visited points, device numbers, by level (stable)
    std::vector<int> level_ptr;       // level l covers seq[level_ptr[l] .. level_ptr[l+1])
    std::vector<long long> take_ptr;  // position u takes take[take_ptr[u] .. take_ptr[u+1])
    std::vector<unsigned> take;       // k << 4 | wait << 3 | direction (kTakeCopy: copy entry)
    std::vector<unsigned char> late;  // per position: its last entries, which read the wait
                                      // dependency that executes last (0..kMaxLate; 0: none)
    std::vector<int> slots;           // group g's wave w executes position slots[kSweepGroup*g + w] (-1: none)
    std::vector<unsigned char> late_src;  // per position: 1 + the wave that executes its late entries'
                                      // point when that is in the same group, else 0
    std::vector<int> old_pts;         // points some regular entry reads as old
    std::vector<int> old_src;         // copy sources read as old
    std::vector<int> wait_src;        // copy sources read as this sweep's value
};

constexpr unsigned kTakeWait = 8u;
// at most this many entries of a position are set apart as late (one lane each)
constexpr int kMaxLate = 4;
constexpr unsigned kTakeCopy = 7u;
// positions of a group: one per wave of the sweep kernel's workgroup
constexpr int kSweepGroup = 8;
// doubles from one published record of the sweep kernel to the next, five
// doubles or five floats a record: the kernel polls and publishes it in
// 16-byte pieces, and counts on each of its 64-bit words coming whole, so every
// record starts on a 16-byte boundary and stays within one 64-byte line
template <typename T>
constexpr int kRecord = sizeof(T) == 4 ? 4 : 8;
constexpr int kTakeShift = 4;

struct SweepPlanInputs {
    int n;                       // points (device numbering 0..n-1)
    const int* status;           // [n]
    const int* alias;            // [n] the reference's alias of each point
    const int* nbhs;             // [n]
    const int* conn;             // [27 n] device numbers
    const int* cnt;              // [6][n] direction lists as the flux stencils walk them
    const long long* off;        // [6][n]
    const int* lst;
    const double* x;             // [n] coordinates, device order (supersonic nearest neighbour)
    const double* y;
    const double* z;
    std::vector<int> visit_fwd;  // the reference's visiting order of each sweep (device numbers)
    std::vector<int> visit_bwd;
    bool backup;                 // the alternative driver: outer points swept, status /= 1 filter
};

struct SweepPlan {
    bool backup = false;
    SweepDirPlan fwd, bwd;
    int n_visited = 0;
    // builds both directions; returns 0, or -1 when a wait entry would not
    // precede its point in the execution order (never, by construction;
    // checked anyway because the sync-free sweep relies on it)
    int build(const SweepPlanInputs& in);
};

// Cuts the positions of a built direction into groups of kSweepGroup, which
// the sweep kernel's workgroups take in order, one position per wave (slots,
// late_src).  A position whose late dependency's group still has a free wave
// joins that group, up to max_chain positions in a row: the value then goes
// from wave to wave through LDS instead of through memory.  Of a position's
// candidates the one with the longest chain of dependents below it joins.
//
// Every position's dependencies lie in its own group or in earlier ones: a
// position starts a chain only when every position before it has a group, and
// joins one only when all of its dependencies have.  The lowest unfinished
// group therefore never waits for a later one, and inside it positions wait
// only for earlier positions, so groups taken in order always finish,
// however few of them run at a time.
void group_positions(SweepDirPlan& plan, int n, int max_chain);

// The same for several chain lengths: what they share, and a cut for each.  The
// plan outlives it; cuts may run side by side.
class SweepGrouper {
   public:
    SweepGrouper(const SweepDirPlan& plan, int n);
    void cut(int max_chain, std::vector<int>& slots, std::vector<unsigned char>& late_src) const;

   private:
    const SweepDirPlan& plan;
    std::vector<int> position;  // [n] of each point (-1: none)
    std::vector<int> joins;     // per position: of those whose late dependency it is, the one with the
                                // longest chain of dependents (-1: none)
};

// Longest chain of positions a sweep workgroup hands from wave to wave, from
// the waves resident on the chip and the plan's mean positions per dependency
// level.  A chain shortens the path through the levels, and holds all eight
// waves of its workgroup until its last position is done: with many levels in
// flight that costs nothing, with few it keeps ready positions waiting.  Sweep
// kernel times, in ms, with chains of 1 (late entries not set apart), 2 and 8:
//   1M FP64, 13.6 levels in flight    11.4   9.7   9.2
//   3M FP64, 6.8                      20.5  18.0  18.9
//   8M FP64, 4.1                      33.8  35.4  41.5
//   3M mixed, 13.6                    17.5  13.4  12.9
//   8M mixed, 8.2                     26.8  22.5  23.5
int chain_for(int resident_waves, double per_level);

// Chains of the two precisions (0: FP64, 1: mixed) of one bound context, which
// may change its precision at any time: each has its groups.
struct SweepChains {
    int chain[2] = {1, 1};
    // the precision whose groups precision m runs (its own, or the other's
    // when the chains are alike); -1: consecutive positions, no groups
    int grouping(int m) const { return chain[m] == 1 ? -1 : m == 1 && chain[0] == chain[1] ? 0 : m; }
};

// the list a sweep walks for point i and direction d (device numbers):
// the flux stencil's list, except that a wall point takes no ZPOS term and
// an outer point (alternative driver only) walks conn for ZPOS
// (implicit_LdelU_forward_sweep_outer.f90:346-347) and nothing for ZNEG
void sweep_list(const SweepPlanInputs& in, int i, int d, const int*& list, int& count);

// nearest neighbour of a supersonic point (implicit_forward_and_reverse_
// sweeps.f90:39-50; the alternative driver skips wall points, ..._backup.f90:
// 56): strict <, first hit in conn order, start distance as the reference
int nearest_neighbour(const SweepPlanInputs& in, int p, double start, bool skip_wall);

}  // namespace mfcfd
