// kernels_sweep.hip -- LU-SGS sweeps without level barriers.
//
// The forward sweep of implicit_forward_and_reverse_sweeps.f90:26-57 visits
// the swept points in alias order; point i reads delUp of every stencil
// neighbour with a smaller alias, already updated earlier in the same sweep
// (implicit_LdelU_forward_sweep_interior.f90:51-117).  The backward sweep
// (implicit_forward_and_reverse_sweeps.f90:58-85) mirrors it with delUn and
// larger aliases.  The alternative driver (implicit_forward_and_reverse_
// sweeps_backup.f90:25-139) visits wall, interior, outer and supersonic
// points in type order with the same alias tests, so a neighbour it visits
// later contributes its value from before the sweep.
//
// The host plan (preprocess.h, SweepPlan) lists, per execution position,
// the entries the point takes, each packed as k << 4 | wait << 3 | d:
// direction list d (kTakeCopy for a supersonic point's copy of its nearest
// neighbour), and whether the entry reads this sweep's value of k ("wait":
// k executes earlier) or the value from before the sweep ("old").  Every
// entry's least-squares weight w (1/dist**power times the Cramer cofactors of
// its list applied to the entry's offset) is computed once, at bind
// (k_sweep_weights).  A position's sweep term is sum_e (Gnew_e - Gold_e)*w_e,
// which equals the reference's Cramer solve of the summed products up to
// rounding.
//
// Per sweep:
//   k_sweep_snap   the values old entries read: prim(U_k + delU_k) of every
//                  point an entry reads as old (pold), and delU of every copy
//                  source read as old (dold), before anything is overwritten;
//   k_sweep_mark   marks pub (the published primitive states) and delU of
//                  every copy source read as this sweep's value with a
//                  signalling-NaN pattern that no arithmetic produces
//                  (kPending);
//   k_sweep_async  a persistent grid of workgroups of kSweepWaves waves; each
//                  round thread 0 takes the next group of the plan with one
//                  atomic and wave w works on the group's position w.
//                  Lane e of the wave takes entry e (longer lists go round
//                  again): Gold from the neighbour's state before the sweep
//                  first (it does not depend on the sweep, so its loads and
//                  arithmetic overlap the wait), then the neighbour's
//                  published primitive state -- polled until it is no
//                  longer pending for a wait entry, read from pold for an
//                  old one -- and Gnew from it.  The wave's sum is a
//                  fixed-order DPP reduction that leaves the sums in lane
//                  kTailLane.  The entries of the dependency that executes
//                  last (the plan puts them at the end, late[t] of them) sit
//                  on the wave's last lanes and are summed apart, by two row
//                  shifts, and added last.  With SPLIT the wave sums the
//                  others first and only then waits for that one point, so
//                  the full reduction is off the dependency chain; without,
//                  it waits for all of them together, which costs fewer
//                  instructions.  The sums are the same, bit for bit.
//                  Lane kTailLane publishes the point's state
//                  prim(U_i + delU_i), computed once here instead of once
//                  per entry that reads it, then stores its delU.  The
//                  mixed form publishes that state as five FP32 values in
//                  three 64-bit words: its consumers evaluate their fluxes
//                  in FP32, so three words per poll instead of five.
//
// What bounds it: the chain of dependent positions, one hop per level (977
// levels of 20 positions on a 20k cloud, 6.6k of 150 on a 1M one, 15.7k of
// 500 on an 8M one).  A hop through memory is the publication, the poll that
// sees it, one flux, a reduction and a conversion.  So, with SPLIT, a group
// holds chains (group_positions): a position whose late dependency has a
// place in the group joins it, the waves of the chain do everything up to
// their late entry side by side, and the late state goes from wave to wave
// through LDS.  That takes the memory round trip out of 60% of the hops.
// Polls are 16-byte loads of one aligned record in a loop of a dozen
// instructions, and publications 16-byte write-through stores: the record in
// five 8-byte atomics each way, in a loop that chose between loads and
// atomic adds word by word, cost 0.2 us more per hop.  Sweep kernel, before
// and after, in ms: 20k FP64 2.09 -> 1.28, mixed 1.56 -> 1.05; 1M FP64 12.6
// -> 9.0, mixed 9.6 -> 6.9; 8M FP64 (no chains, chain_for) 33.6 -> 33.8,
// mixed 26.2 -> 22.5.
//
// Memory model.  Inside k_sweep_async the memory other waves read while it
// runs is pub (and dsrc, the published delU of the copy sources), each 64-bit
// value written once.  These arrays are fine-grained device memory: hipMalloc's
// coarse-grained memory is coherent only at kernel boundaries, and on MI355X
// a value written there by one wave was measured still reading as pending,
// through agent-scope atomic loads on another CU, a second after its writer
// had finished.  A position publishes with write-through stores (copy sources
// with device-scope atomic swaps); a waiting lane reads with agent-scope loads
// and, should a value still read pending after kSpinAtomic polls, re-reads it
// with device-scope atomic adds of zero, which are performed at the device's
// coherence point (the zero comes from a kernel argument, so the compiler
// cannot turn the add into a load).  A non-pending value is the final one:
// the marks are written before the kernel starts and each location is
// written once while it runs.  Each value is checked on its own, so no
// ordering between locations is needed.  Everything else the kernel reads
// is not written while it runs, and delU, which the later kernels read, is
// ordered by the kernel boundary.
//
// Progress.  Every wait entry reads a point of the same group or of an
// earlier one (group_positions), so of a workgroup that is running.  The
// waves of a group run side by side and wait among themselves only for
// earlier positions; the lowest unfinished group never waits on another, and
// the barrier between a workgroup's rounds only delays its next group, which
// is later than every group taken, so every wait ends, however few
// workgroups are resident.  A wait that exceeds the spin limit is counted in
// the residual record and the host reports an error; the kernel still runs
// to completion.
//
// T is the arithmetic of the split fluxes and of the published state (float
// in the mixed form); the weights, the sums, D_inv and the new delU stay FP64.
// The FP64 flux evaluations take the sweep form of qlskum_math.h (flux_eval
// with SWEEP), and this unit is compiled with -ffp-contract=on (a*b + c
// fused within an expression): every Gold and Gnew of both sweeps is
// evaluated the same way, so an unchanged neighbour contributes exactly zero.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_common.h"
#include "device_state.h"
#include "kernels.h"
#include "preprocess.h"
#include "qlskum_math.h"



namespace mfcfd {

namespace {

// waves per workgroup: one point per wave, and one ticket counter atomic per
// workgroup and round for a group of kSweepWaves positions.  Same-address
// device-scope atomics serialise (~12 ns each), so a ticket per 4 positions
// capped the sweep near 330 positions per microsecond, less than the 8M mixed
// sweep needs (350): with 8 per ticket the first kernel's FP64 sweep took 35.3
// -> 33.6 ms and the mixed one 29.2 -> 26.3 ms.  8 waves of a workgroup
// still fit the FP64 kernel's 2 waves per SIMD.
constexpr int kSweepWaves = kSweepGroup;
constexpr int kSweepBlock = 64 * kSweepWaves;
// the late entries sit on lanes 64 - kMaxLate .. 63, which two row shifts sum
static_assert(kMaxLate >= 1 && kMaxLate <= 4, "late lanes must fit the last four lanes of a row");
// record j of pub (T of the kernel) or of dsrc (double)
template <typename T>
__device__ __forceinline__ double* record(double* base, long long j) {
    static_assert(kRecord<T> % 2 == 0 && 8 % kRecord<T> == 0, "records are polled in aligned 16-byte pieces");
    return base + kRecord<T> * j;
}
// about a second of polling; legitimate waits end within milliseconds
constexpr int kSpinLimit = 1 << 20;
// polls by atomic load before the atomic-add fallback
constexpr int kSpinAtomic = 4096;
// polls of a value in LDS: a round trip there is some 50 ns
constexpr int kSpinLimitLds = 1 << 24;

// a signalling NaN with a payload: arithmetic only ever produces quiet NaNs
constexpr unsigned long long kPending = 0x7FF4DEAD5EEDF00DULL;

// publish one value: a device-scope atomic swap, performed at the coherence
// point every XCD's atomics read
__device__ __forceinline__ void store_value(double* p, double v) {
    __hip_atomic_exchange(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v),
                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));

// one poll: the NW 64-bit words at w as agent-scope loads (sc1), 16 bytes at
// a time, waited for in the same block.  Each word is aligned and read whole;
// the words may be of different moments, and each is checked on its own.
template <int NW>
__device__ __forceinline__ void poll_words(const unsigned long long* w, unsigned long long out[NW]) {
    static_assert(NW == 3 || NW == 5, "three or five words");
    u64x2 a, b;
    unsigned long long c;
    if constexpr (NW == 5) {
        asm volatile(
            "global_load_dwordx4 %0, %3, off sc1\n\t"
            "global_load_dwordx4 %1, %3, off offset:16 sc1\n\t"
            "global_load_dwordx2 %2, %3, off offset:32 sc1\n\t"
            "s_waitcnt vmcnt(0)"
            : "=&v"(a), "=&v"(b), "=&v"(c)
            : "v"(w)
            : "memory");
        out[2] = b.x;
        out[3] = b.y;
    } else {
        asm volatile(
            "global_load_dwordx4 %0, %2, off sc1\n\t"
            "global_load_dwordx2 %1, %2, off offset:16 sc1\n\t"
            "s_waitcnt vmcnt(0)"
            : "=&v"(a), "=&v"(c)
            : "v"(w)
            : "memory");
    }
    out[0] = a.x;
    out[1] = a.y;
    out[NW - 1] = c;
}

// publish NW words: write-through stores (sc0 sc1), 16 bytes at a time.  (The
// s_nop keeps the data registers in place until the last store has read them.)
template <int NW>
__device__ __forceinline__ void publish_words(unsigned long long* p, const unsigned long long v[NW]) {
    const u64x2 a = {v[0], v[1]};
    if constexpr (NW == 5) {
        const u64x2 b = {v[2], v[3]};
        asm volatile(
            "global_store_dwordx4 %0, %1, off sc0 sc1\n\t"
            "global_store_dwordx4 %0, %2, off offset:16 sc0 sc1\n\t"
            "global_store_dwordx2 %0, %3, off offset:32 sc0 sc1\n\t"
            "s_nop 1"
            :
            : "v"(p), "v"(a), "v"(b), "v"(v[4])
            : "memory");
    } else {
        asm volatile(
            "global_store_dwordx4 %0, %1, off sc0 sc1\n\t"
            "global_store_dwordx2 %0, %2, off offset:16 sc0 sc1\n\t"
            "s_nop 1"
            :
            : "v"(p), "v"(a), "v"(v[2])
            : "memory");
    }
}

template <int NW>
__device__ __forceinline__ bool any_pending(const unsigned long long v[NW]) {
    bool p = false;
#pragma unroll
    for (int r = 0; r < NW; ++r) p = p || v[r] == kPending;
    return p;
}

// read NW 64-bit words written in this sweep, waiting until none is pending:
// agent-scope loads of all of them at every poll (polling one value and
// re-reading the others once it arrives costs a second memory round trip on
// the dependency chain: measured 21% slower sweeps), device-scope atomic adds
// of zero after kSpinAtomic polls.  Gives up after the spin limit, or at once
// when another wait of this sweep already gave up, so a broken schedule ends
// the kernel instead of stalling it point by point.
template <int NW>
__device__ __forceinline__ void wait_words(double* v, unsigned long long out[NW], int* stalls,
                                           unsigned long long zero) {
    unsigned long long* w = reinterpret_cast<unsigned long long*>(v);
    int left = kSpinAtomic;
    bool pending;
#pragma clang loop unroll(disable)
    do {
        poll_words<NW>(w, out);
        pending = any_pending<NW>(out);
    } while (pending && --left > 0);
    if (!pending) return;
#pragma clang loop unroll(disable)
    for (int spins = kSpinAtomic; spins < kSpinLimit; ++spins) {
        __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int r = 0; r < NW; ++r)
            out[r] = __hip_atomic_fetch_add(w + r, zero, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!any_pending<NW>(out)) return;
        if ((spins & 255) == 0 && __hip_atomic_load(stalls, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
            return;
    }
    __hip_atomic_fetch_add(stalls, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The mixed form publishes prim(U + delU) as five FP32 values in three 64-bit
// words (its consumers evaluate their fluxes in FP32 anyway): lo/hi halves
// p0/p1, p2/p3, p4/0.  A word with a zero high half never matches kPending;
// the other two would need a high half of 0x7FF4DEAD, a NaN payload that
// arithmetic does not produce (it yields the default NaN, or passes on the
// payload of a NaN operand, and no operand here carries that one).
__device__ __forceinline__ unsigned long long pack2(float lo, float hi) {
    return (unsigned long long)__float_as_uint(lo) | ((unsigned long long)__float_as_uint(hi) << 32);
}

// read the NW words a wave of the same workgroup publishes in LDS, waiting
// until none is pending; bounded as wait_words is
template <int NW>
__device__ __forceinline__ void wait_words_lds(const unsigned long long* w, unsigned long long out[NW], int* stalls) {
    int left = kSpinLimitLds;
    bool pending;
#pragma clang loop unroll(disable)
    do {
#pragma unroll
        for (int r = 0; r < NW; ++r) out[r] = __hip_atomic_load(w + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        pending = any_pending<NW>(out);
    } while (pending && --left > 0);
    if (pending) __hip_atomic_fetch_add(stalls, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the state of this sweep a wait entry reads: from the neighbour's words in
// LDS when its wave belongs to the workgroup (lds not null), else from pub
template <typename T>
__device__ __forceinline__ void wait_state(double* pub, const unsigned long long* lds, T out[5], int* stalls,
                                           unsigned long long zero) {
    constexpr int NW = sizeof(T) == 4 ? 3 : 5;
    unsigned long long b[NW];
    if (lds)
        wait_words_lds<NW>(lds, b, stalls);
    else
        wait_words<NW>(pub, b, stalls, zero);
    if constexpr (sizeof(T) == 4) {
        out[0] = __uint_as_float((unsigned)b[0]);
        out[1] = __uint_as_float((unsigned)(b[0] >> 32));
        out[2] = __uint_as_float((unsigned)b[1]);
        out[3] = __uint_as_float((unsigned)(b[1] >> 32));
        out[4] = __uint_as_float((unsigned)b[2]);
    } else {
#pragma unroll
        for (int r = 0; r < 5; ++r) out[r] = __longlong_as_double((long long)b[r]);
    }
}

// a 64-bit value every lane of the wave holds alike, in scalar registers
__device__ __forceinline__ long long uniform64(long long v) {
    const int lo = __builtin_amdgcn_readfirstlane((int)v);
    const int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
    return ((long long)hi << 32) | (long long)(unsigned)lo;
}

// one DPP move of a double (both 32-bit halves through v_mov_b32_dpp): a
// lane whose source lane lies outside its row, or whose row is masked off,
// reads 0
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROW_MASK, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROW_MASK, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// The lane that finishes a position.  The reduction below leaves the wave's
// sums in lane 63, so the point's own inputs are loaded into that lane too,
// and nothing crosses lanes between the reduction and the publication.
constexpr int kTailLane = 63;

// Sums over the 64 lanes of a wave (all active), in a fixed order, for five
// values at once, left in lane kTailLane.  Prefix sums within each row of 16
// lanes (row_shr 1, 2, 4, 8: lane 15 of a row holds the row's sum), row 0's
// sum into row 1 and row 2's into row 3 (row_bcast:15), then lane 31's into
// rows 2 and 3 (row_bcast:31): lane 63 ends with the total.  Each step is one
// VALU move per half, where a shuffle is a round trip through the LDS
// crossbar.  The five values take each step together, so five independent
// chains are in flight instead of one: the reduction sits on the sweep's
// dependency chain.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void sum_step5(double v[5]) {
#pragma unroll
    for (int r = 0; r < 5; ++r) v[r] = v[r] + dpp_move<CTRL, ROW_MASK>(v[r]);
}
__device__ __forceinline__ void wave_sum5(double v[5]) {
    sum_step5<0x111, 0xf>(v);
    sum_step5<0x112, 0xf>(v);
    sum_step5<0x114, 0xf>(v);
    sum_step5<0x118, 0xf>(v);
    sum_step5<0x142, 0xa>(v);
    sum_step5<0x143, 0xc>(v);
}

// The end of a position, on lane kTailLane: U_i + delU and its primitive
// state, published (FP64, or FP32 packed in three words in the mixed form),
// delU published too when the point is a copy source read in this sweep,
// then delU stored for the later kernels.  Called at the end of both kinds
// of position, so that no values merge between them before it.
template <typename T>
__device__ __forceinline__ void finish_position(const SweepAsync& a, double* dU, int i, const Frame<double>& f,
                                                const double res[5], const double Ui[5], int slot,
                                                unsigned long long* lds) {
    double U[5];
#pragma unroll
    for (int r = 0; r < 5; ++r) U[r] = res[r] + Ui[r];
    constexpr int NW = sizeof(T) == 4 ? 3 : 5;
    unsigned long long w[NW];
    if constexpr (sizeof(T) == 4) {
        const Frame<float> f32 = frame_as<float>(f);
        float U32[5], p32[5];
#pragma unroll
        for (int r = 0; r < 5; ++r) U32[r] = float(U[r]);
        conserved_to_prim(U32, f32, p32);
        w[0] = pack2(p32[0], p32[1]);
        w[1] = pack2(p32[2], p32[3]);
        w[2] = pack2(p32[4], 0.0f);
    } else {
        double pp[5];
        conserved_to_prim<double, true>(U, f, pp);
#pragma unroll
        for (int r = 0; r < 5; ++r) w[r] = (unsigned long long)__double_as_longlong(pp[r]);
    }
    // the next position of the chain first
#pragma unroll
    for (int r = 0; r < NW; ++r) __hip_atomic_store(lds + r, w[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    unsigned long long* pub = reinterpret_cast<unsigned long long*>(record<T>(a.pub, i));
    publish_words<NW>(pub, w);
    if (slot >= 0) {
#pragma unroll
        for (int r = 0; r < 5; ++r) store_value(record<double>(a.dsrc, slot) + r, res[r]);
    }
#pragma unroll
    for (int r = 0; r < 5; ++r) dU[5 * (long long)i + r] = res[r];
}

// the list a sweep walks for point i and direction d (SweepPlan's
// sweep_list): the flux stencil's list, except an outer point's z term,
// which walks conn (implicit_LdelU_forward_sweep_outer.f90:346-347)
__device__ __forceinline__ void sweep_list_dev(const DevGeom& g, int cls, int d, int i, const int*& list,
                                               int& count) {
    if (cls == 2 && d == ZPOS) {
        list = g.conn + kConnCols * (long long)i;
        count = g.nbhs[i];
        return;
    }
    list = g.lst + g.dir_off[(long long)d * g.n + i];
    count = g.dir_cnt[(long long)d * g.n + i];
}

// setup: the weight of every taken entry, one thread per position.  Entries
// come grouped by direction; each direction's Cramer cofactors are those of
// the whole list the reference walks (list_cofactors, the same arithmetic as
// the flux stencils' weights).
template <bool UW>
__global__ void __launch_bounds__(kBlock) k_sweep_weights(DevGeom g, SweepAsync a, double power) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= a.count) return;
    const int i = a.seq[u];
    const int cls = g.status[i];
    const Frame<double> f = load_frame(g.frame, i);
    const double4 pi4 = g.pos[i];
    double c[3] = {0.0, 0.0, 0.0};
    int cur = -1;
    for (long long e = a.take_ptr[u]; e < a.take_ptr[u + 1]; ++e) {
        const unsigned packed = a.take[e];
        const int d = (int)(packed & 7u);
        if (d == (int)kTakeCopy) {
            a.wgt[e] = 0.0;
            continue;
        }
        if (d != cur) {
            const int* list;
            int count;
            sweep_list_dev(g, cls, d, i, list, count);
            list_cofactors<UW>(g, i, f, list, count, d >> 1, power, c);
            cur = d;
        }
        const double4 pk = g.pos[packed >> kTakeShift];
        const double delx = pk.x - pi4.x, dely = pk.y - pi4.y, delz = pk.z - pi4.z;
        const double dels = delx * f.t1[0] + dely * f.t1[1] + delz * f.t1[2];
        const double delt = delx * f.t2[0] + dely * f.t2[1] + delz * f.t2[2];
        const double deln = delx * f.n[0] + dely * f.n[1] + delz * f.n[2];
        a.wgt[e] = wls_weight<UW>(dels, delt, deln, power) * (c[0] * dels + c[1] * delt + c[2] * deln);
    }
}

// the values old entries read, taken before the sweep overwrites anything:
// pold = prim(U + delU) (get_primitive_vector.f90:10-41) of the points
// regular entries read as old, dold = delU of the copy sources read as old
__global__ void __launch_bounds__(kBlock) k_sweep_snap(DevGeom g, DevState s, const double* dU, SweepAsync a) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < a.n_old) {
        const int k = a.old_pts[e];
        double U[5], prim[5];
#pragma unroll
        for (int r = 0; r < 5; ++r) U[r] = dU[5 * (long long)k + r] + s.U[5 * (long long)k + r];
        conserved_to_prim<double, true>(U, load_frame(g.frame, k), prim);
#pragma unroll
        for (int r = 0; r < 5; ++r) a.pold[5 * (long long)k + r] = prim[r];
    } else if (e < (long long)a.n_old + a.n_old_src) {
        const int q = a.old_src[e - a.n_old];
#pragma unroll
        for (int r = 0; r < 5; ++r) a.dold[5 * (long long)q + r] = dU[5 * (long long)q + r];
    }
}

// pending marks: all of pub and every slot of dsrc, 16 bytes a thread
__global__ void __launch_bounds__(kBlock) k_sweep_mark(SweepAsync a, long long pub_pairs) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < pub_pairs) {
        reinterpret_cast<u64x2*>(a.pub)[e] = u64x2{kPending, kPending};
    } else if (e < pub_pairs + kRecord<double> / 2 * (long long)a.n_wait_src) {
        reinterpret_cast<u64x2*>(a.dsrc)[e - pub_pairs] = u64x2{kPending, kPending};
    }
}

template <bool FORWARD, bool UW, typename T, bool SPLIT>
__global__ void __launch_bounds__(kSweepBlock, sizeof(T) == 4 ? 4 : 2) k_sweep_async(DevGeom g, DevState s, FlowParams fp,
                                                             SweepAsync a) {
    constexpr int NW = sizeof(T) == 4 ? 3 : 5;
    // double-buffered: round r uses slot r & 1 while a wave may still read the
    // other.  A group number is rewritten two rounds later, after a barrier
    // that every wave reaches only after reading it; a wave marks its words
    // of round r + 1 as pending in round r, after the barrier that ended the
    // reads of round r - 1 and before the one that starts round r + 1
    __shared__ unsigned sh_group[2];
    __shared__ unsigned long long sh_pub[2][kSweepWaves][8];
    const int lane = threadIdx.x & 63;
    const unsigned wave = threadIdx.x >> 6;
    double* dU = FORWARD ? s.delUp : s.delUn;
    if (lane < NW)
        __hip_atomic_store(&sh_pub[0][wave][lane], kPending, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    for (unsigned round = 0;; ++round) {
        // a position's work up to its waits is off the dependency chain
        __builtin_amdgcn_s_setprio(0);
        if (threadIdx.x == 0)
            sh_group[round & 1] = __hip_atomic_fetch_add(a.ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (lane < NW)
            __hip_atomic_store(&sh_pub[(round + 1) & 1][wave][lane], kPending, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        // wave-uniform values are moved to scalar registers (readfirstlane):
        // the position, the point and its entry range
        const unsigned group = __builtin_amdgcn_readfirstlane(sh_group[round & 1]);
        if (group >= (unsigned)a.groups) break;   // the same for the whole workgroup
        // without chains a group is kSweepWaves consecutive positions
        const unsigned own = kSweepWaves * group + wave;
        const int t = __builtin_amdgcn_readfirstlane(SPLIT ? a.slots[own] : own < (unsigned)a.count ? (int)own : -1);
        if (t < 0) continue;   // the last group's spare waves
        unsigned long long* mine = sh_pub[round & 1][wave];
        const int i = __builtin_amdgcn_readfirstlane(a.seq[t]);
        const long long tb = uniform64(a.take_ptr[t]), te = uniform64(a.take_ptr[t + 1]);
        const Frame<double> f = load_frame(g.frame, i);
        // the point's conserved state for the final update, loaded now so
        // that its latency stays off the path after the reduction
        double Ui[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        int slot = -1;   // the point's slot as a copy source read in this sweep
        if (lane == kTailLane) {
#pragma unroll
            for (int r = 0; r < 5; ++r) Ui[r] = s.U[5 * (long long)i + r];
            if (a.src_slot) slot = a.src_slot[i];
        }
        const unsigned first = te > tb ? __builtin_amdgcn_readfirstlane(a.take[tb]) : 0u;
        if (te > tb && (first & 7u) == kTakeCopy) {
            // supersonic point: the nearest neighbour's delU
            // (implicit_forward_and_reverse_sweeps.f90:38-52, 69-83)
            if (lane == kTailLane) {
                const long long q = (long long)(first >> kTakeShift);
                double res[5];
                if (first & kTakeWait) {
                    wait_state<double>(record<double>(a.dsrc, a.src_slot[q]), nullptr, res, a.stalls, a.zero);
                } else {
#pragma unroll
                    for (int r = 0; r < 5; ++r) res[r] = a.dold[5 * q + r];
                }
                finish_position<T>(a, dU, i, f, res, Ui, slot, mine);
            }
        } else {
            const int cls = __builtin_amdgcn_readfirstlane(g.status[i]);
            const Frame<T> ft = frame_as<T>(f);
            // the point's own inputs of the final update, read before the wait
            double D_inv = 0.0, own[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            if (lane == kTailLane) {
                D_inv = s.dinv[i];
#pragma unroll
                for (int r = 0; r < 5; ++r)
                    own[r] = FORWARD ? s.flux_res[5 * (long long)i + r] : s.delUp[5 * (long long)i + r];
            }
            // The entries of the wait dependency that executes last sit at the
            // end of the list, at most kMaxLate of them, on the wave's last
            // lanes; the others share the lanes below.
            const int n_late = __builtin_amdgcn_readfirstlane((int)a.late[t]);
            const int src = SPLIT ? __builtin_amdgcn_readfirstlane((int)a.late_src[t]) : 0;
            const unsigned long long* from = src ? sh_pub[round & 1][src - 1] : nullptr;
            const int stride = 64 - n_late;
            const bool late = lane >= stride;
            const long long tl = te - n_late;
            double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            T Gold[5] = {T(0), T(0), T(0), T(0), T(0)};
            double wgt = 0.0;
            long long k = 0;
            int d = 0;
            long long e = late ? te - (64 - lane) : tb + lane;
            if (late || e < tl) {
                for (;;) {
                    const unsigned packed = a.take[e];
                    k = (long long)(packed >> kTakeShift);
                    d = (int)(packed & 7u);
                    wgt = a.wgt[e];
                    // the flux of the neighbour's state before the sweep first:
                    // it does not depend on the sweep, so its loads and
                    // arithmetic overlap the wait for the state of this sweep,
                    // whose flux follows
                    T pt[5], Gnew[5];
#pragma unroll
                    for (int r = 0; r < 5; ++r) pt[r] = T(s.prim[5 * k + r]);
                    flux_eval<T, true>(dir_family(cls, d), d >> 1, (d & 1) ? -1 : 1, ft, pt, T(fp.pi), Gold);
                    if (SPLIT && late) break;
                    if (packed & kTakeWait) {
                        wait_state<T>(record<T>(a.pub, k), nullptr, pt, a.stalls, a.zero);
                    } else {
#pragma unroll
                        for (int r = 0; r < 5; ++r) pt[r] = T(a.pold[5 * k + r]);
                    }
                    // with no late entries set apart, the wave is on the dependency
                    // chain from here to the publication: its SIMD issues for it
                    // before a wave still working ahead of its waits
                    if (!SPLIT) __builtin_amdgcn_s_setprio(3);
                    flux_eval<T, true>(dir_family(cls, d), d >> 1, (d & 1) ? -1 : 1, ft, pt, T(fp.pi), Gnew);
#pragma unroll
                    for (int r = 0; r < 5; ++r) acc[r] = acc[r] + (double)(Gnew[r] - Gold[r]) * wgt;
                    e += stride;
                    if (late || e >= tl) break;
                }
            }
            if constexpr (SPLIT) {
                double c[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
                wave_sum5(acc);
                if (late) {
                    T pt[5], Gnew[5];
                    wait_state<T>(record<T>(a.pub, k), from, pt, a.stalls, a.zero);
                    // on the dependency chain from here to the publication
                    __builtin_amdgcn_s_setprio(3);
                    flux_eval<T, true>(dir_family(cls, d), d >> 1, (d & 1) ? -1 : 1, ft, pt, T(fp.pi), Gnew);
#pragma unroll
                    for (int r = 0; r < 5; ++r) c[r] = (double)(Gnew[r] - Gold[r]) * wgt;
                }
                sum_step5<0x111, 0xf>(c);
                sum_step5<0x112, 0xf>(c);
#pragma unroll
                for (int r = 0; r < 5; ++r) acc[r] = acc[r] + c[r];
            } else {
                // the same sums in the same order
                double c[5];
#pragma unroll
                for (int r = 0; r < 5; ++r) {
                    c[r] = late ? acc[r] : 0.0;
                    acc[r] = late ? 0.0 : acc[r];
                }
                sum_step5<0x111, 0xf>(c);
                sum_step5<0x112, 0xf>(c);
                wave_sum5(acc);
#pragma unroll
                for (int r = 0; r < 5; ++r) acc[r] = acc[r] + c[r];
            }
            if (lane == kTailLane) {
                // wall terms are doubled (implicit_LdelU_forward_sweep_wall.f90:405);
                // the product with 1 or 2 is exact
                const double twice = cls == 1 ? 2.0 : 1.0;
                double res[5];
#pragma unroll
                for (int r = 0; r < 5; ++r) {
                    const double term = twice * acc[r];
                    res[r] = FORWARD ? -(D_inv * (own[r] + term)) : own[r] - D_inv * term;
                }
                finish_position<T>(a, dU, i, f, res, Ui, slot, mine);
            }
        }
    }
    // the last workgroup out resets the counters for the next sweep
    if (threadIdx.x == 0) {
        const unsigned done = __hip_atomic_fetch_add(a.ctr + 1, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (done == gridDim.x - 1) {
            __hip_atomic_store(a.ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.ctr + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

__global__ void k_copy_sweep(double* dst, const double* src, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

template <bool FORWARD, bool UW, typename T, bool SPLIT>
int resident_grid(int count) {
    int dev = 0, per_cu = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k_sweep_async<FORWARD, UW, T, SPLIT>,
                                                     kSweepBlock, 0) != hipSuccess)
        return 0;
    if (per_cu < 1) per_cu = 1;
    const long long grid = (long long)per_cu * prop.multiProcessorCount;
    return (int)(grid < count ? grid : count);
}

template <bool UW, typename T, bool SPLIT>
int pair_grid(int count) {
    const int a = resident_grid<true, UW, T, SPLIT>(count);
    const int b = resident_grid<false, UW, T, SPLIT>(count);
    return a < b ? a : b;
}

template <bool FORWARD, bool UW, typename T>
void launch_one(const DevGeom& g, const DevState& s, const FlowParams& p, const SweepAsync& a, int grid,
                hipStream_t st, const hipEvent_t* ev) {
    double* dU = FORWARD ? s.delUp : s.delUn;
    const long long n_snap = (long long)a.n_old + a.n_old_src;
    if (n_snap > 0)
        hipLaunchKernelGGL(k_sweep_snap, dim3(grid_for(n_snap, kBlock)), dim3(kBlock), 0, st, g, s,
                           (const double*)dU, a);
    const long long pairs = kRecord<T> / 2 * (long long)g.n;
    const long long n_mark = pairs + kRecord<double> / 2 * (long long)a.n_wait_src;
    hipLaunchKernelGGL(k_sweep_mark, dim3(grid_for(n_mark, kBlock)), dim3(kBlock), 0, st, a, pairs);
    if (ev) (void)hipEventRecord(ev[0], st);
    if (a.split)
        hipLaunchKernelGGL((k_sweep_async<FORWARD, UW, T, true>), dim3(grid), dim3(kSweepBlock), 0, st, g, s, p, a);
    else
        hipLaunchKernelGGL((k_sweep_async<FORWARD, UW, T, false>), dim3(grid), dim3(kSweepBlock), 0, st, g, s, p, a);
    if (ev) (void)hipEventRecord(ev[1], st);
}

template <bool UW, typename T>
void launch_pair(const DevGeom& g, const DevState& s, const FlowParams& p, const SweepAsync& fwd,
                 const SweepAsync& bwd, int grid, hipStream_t st, const hipEvent_t* ev) {
    launch_one<true, UW, T>(g, s, p, fwd, grid, st, ev);
    launch_one<false, UW, T>(g, s, p, bwd, grid, st, ev ? ev + 2 : nullptr);
}

}  // namespace

int sweep_async_grid(int groups, bool unit_weight, bool mixed) {
    if (groups <= 0) return 0;
    const auto grid = [&](auto uw, auto t) {
        using T = decltype(t);
        constexpr bool UW = decltype(uw)::value;
        const int a = pair_grid<UW, T, true>(groups), b = pair_grid<UW, T, false>(groups);
        return a < b ? a : b;
    };
    using std::false_type;
    using std::true_type;
    if (mixed) return unit_weight ? grid(true_type{}, 0.0f) : grid(false_type{}, 0.0f);
    return unit_weight ? grid(true_type{}, 0.0) : grid(false_type{}, 0.0);
}

void launch_sweep_weights(const DevGeom& g, const SweepAsync& a, double power, hipStream_t st) {
    if (a.count <= 0) return;
    if (power == 0.0)
        hipLaunchKernelGGL(k_sweep_weights<true>, dim3(grid_for(a.count, kBlock)), dim3(kBlock), 0, st, g, a, power);
    else
        hipLaunchKernelGGL(k_sweep_weights<false>, dim3(grid_for(a.count, kBlock)), dim3(kBlock), 0, st, g, a, power);
}

void launch_sweeps_async(const DevGeom& g, const DevState& s, const FlowParams& p, const SweepAsync& fwd,
                         const SweepAsync& bwd, int grid, hipStream_t st, const hipEvent_t* ev) {
    if (fwd.count > 0 && grid > 0) {
        if (p.mixed) {
            if (p.power == 0.0)
                launch_pair<true, float>(g, s, p, fwd, bwd, grid, st, ev);
            else
                launch_pair<false, float>(g, s, p, fwd, bwd, grid, st, ev);
        } else {
            if (p.power == 0.0)
                launch_pair<true, double>(g, s, p, fwd, bwd, grid, st, ev);
            else
                launch_pair<false, double>(g, s, p, fwd, bwd, grid, st, ev);
        }
    }
    // implicit_forward_and_reverse_sweeps.f90:86-88; the alternative driver
    // leaves it to state_update_implicit.f90:98-100
    if (!p.backup)
        hipLaunchKernelGGL(k_copy_sweep, dim3(grid_for(5LL * g.n, kBlock)), dim3(kBlock), 0, st, s.delUp,
                           (const double*)s.delUn, 5LL * g.n);
}

}  // namespace mfcfd
