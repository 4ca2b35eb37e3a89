// Work planes of an operator: how many right-hand-side slots W1 and W2 hold,
// and when they may move.  Host arithmetic only (no HIP), so that it can be
// tested on its own.
#pragma once
#include <algorithm>
#include <cstdint>

namespace gla {

// A partitioned operator takes all partitions of a pass in one launch
// (run_matvec_parts: each source partition transformed once, the sum over them
// between the transforms) when its slots stay within kPartBytes; otherwise, or
// when only that much work memory is at hand, it runs the five passes once per
// (source, target) pair on one slot per right-hand side.  48^3 fine cells (8
// source partitions) on 24^3 coarse ones, ComplexF32: 211 us pair by pair (40
// launches of too few workgroups each, the forward and inverse transforms of
// pass 3 once per pair), 69 us in five launches.  The bound is on memory: it
// keeps the partitions' planes of one call within a hundredth of the GPU's.
constexpr int64_t kPartBytes = (int64_t)2 << 30;

struct Slots {
    int64_t w1, w2;
};

inline bool covers(Slots a, Slots b) { return a.w1 >= b.w1 && a.w2 >= b.w2; }

// Source and target partitions of an operator, and the bytes of one slot.
struct SlotCost {
    int64_t Ps, Pt, w1, w2;
};

// one slot per right-hand side: unpartitioned operators, and pair by pair
inline Slots pair_slots(int64_t nrhs) { return Slots{nrhs, nrhs}; }

// all partitions of nrhs right-hand sides in one launch
inline Slots part_slots(const SlotCost& c, int64_t nrhs)
{
    return Slots{nrhs * std::max(c.Ps, c.Pt), nrhs * (c.Ps + (c.Pt > 1 ? c.Pt : 0))};
}

// the largest count whose partitions are taken in one launch (0: none)
inline int64_t part_limit(const SlotCost& c)
{
    if (c.Ps * c.Pt == 1) return 0;
    const Slots one = part_slots(c, 1);
    return std::min((int64_t)65535 / one.w1, kPartBytes / (one.w1 * c.w1 + one.w2 * c.w2));
}

// The slots reserved for nrhs right-hand sides: enough for every count up to
// nrhs in the form it runs in, so they only grow with nrhs.
inline Slots want_slots(const SlotCost& c, int64_t nrhs)
{
    const Slots pair = pair_slots(nrhs), part = part_slots(c, std::min(nrhs, part_limit(c)));
    return Slots{std::max(pair.w1, part.w1), std::max(pair.w2, part.w2)};
}

struct WorkPlanes {
    void* w1 = nullptr;
    void* w2 = nullptr;
    Slots held{0, 0};
    int64_t nrhs = 0;   // the largest count they were ensured for
};

enum class Ensure { ok, capture, pinned, memory };

// Planes for nrhs right-hand sides, in the form of want_slots or, where that
// much memory cannot be had, pair by pair.  A count up to one ensured before
// moves nothing, whatever other counts ran in between: a graph captured over
// the planes stays valid until a larger count is applied or reserved.  Planes
// that hold the pair form are kept until larger ones exist; a size that was
// refused is not asked for again by the same or a smaller count.
//   may_grow  false under stream capture: no allocation, and the count is
//             kept from moving the planes later
//   pinned    a recorded batch uses the planes
//   mem       alloc(bytes) -> pointer or null, release(pointer)
template <typename Mem>
Ensure ensure_planes(WorkPlanes& p, const SlotCost& c, int64_t nrhs, bool may_grow, bool pinned, Mem& mem)
{
    if (nrhs <= p.nrhs) return Ensure::ok;
    const Slots want = want_slots(c, nrhs);
    const bool fits = covers(p.held, pair_slots(nrhs));
    if (covers(p.held, want) || (fits && !may_grow)) {
        p.nrhs = nrhs;
        return Ensure::ok;
    }
    if (!may_grow) return Ensure::capture;
    if (pinned) return fits ? Ensure::ok : Ensure::pinned;
    WorkPlanes n;
    auto grow = [&](Slots s) {
        n.w1 = mem.alloc(s.w1 * c.w1);
        n.w2 = n.w1 ? mem.alloc(s.w2 * c.w2) : nullptr;
        if (n.w1 && !n.w2) mem.release(n.w1);
        n.held = s;
        return n.w1 && n.w2;
    };
    auto drop = [&] {
        if (p.w1) mem.release(p.w1);
        if (p.w2) mem.release(p.w2);
        p = WorkPlanes();
    };
    if (fits) {
        if (grow(want)) {
            drop();
            p = n;
        }
    } else {
        drop();
        if (!grow(want) && (covers(pair_slots(nrhs), want) || !grow(pair_slots(nrhs)))) return Ensure::memory;
        p = n;
    }
    p.nrhs = nrhs;
    return Ensure::ok;
}

}  // namespace gla
