"""Work planes of an operator (csrc/gla_slots.hpp, the code the library runs)
on the CPU with a counting allocator: over many orders of eager, reserved,
captured and batch-pinned counts and with memory that runs out, planes hold
what every accepted count needs, a count up to one ensured before moves
nothing, and a refused size is not asked for again."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gilaelectromagnetics.jl_amd", "csrc")

SHIM = r"""
#include "gla_slots.hpp"
#include <map>
struct Mem {
    int64_t room, used = 0, allocs = 0, releases = 0, next = 0;
    std::map<void*, int64_t> live;
    void* alloc(int64_t bytes)
    {
        ++allocs;
        if (used + bytes > room) return nullptr;
        void* const p = (void*)(++next);
        live[p] = bytes;
        used += bytes;
        return p;
    }
    void release(void* p)
    {
        ++releases;
        used -= live.at(p);
        live.erase(p);
    }
};
struct Op { gla::SlotCost c; gla::WorkPlanes p; Mem m; };
extern "C" {
Op* op_new(int64_t Ps, int64_t Pt, int64_t b1, int64_t b2, int64_t room)
{
    Op* o = new Op;
    o->c = gla::SlotCost{Ps, Pt, b1, b2};
    o->m.room = room;
    return o;
}
void op_free(Op* o) { delete o; }
void op_room(Op* o, int64_t room) { o->m.room = room; }
// status 0 ok, 1 capture, 2 pinned, 3 memory; then w1, w2, slots, allocs, releases, bytes in use
void op_ensure(Op* o, int64_t nrhs, int may_grow, int pinned, int64_t* out)
{
    out[0] = (int64_t)gla::ensure_planes(o->p, o->c, nrhs, may_grow != 0, pinned != 0, o->m);
    out[1] = (int64_t)o->p.w1;
    out[2] = (int64_t)o->p.w2;
    out[3] = o->p.held.w1;
    out[4] = o->p.held.w2;
    out[5] = o->m.allocs;
    out[6] = o->m.releases;
    out[7] = o->m.used;
}
int64_t op_limit(Op* o) { return gla::part_limit(o->c); }
void op_part(Op* o, int64_t n, int64_t* out)
{
    const gla::Slots s = gla::part_slots(o->c, n);
    out[0] = s.w1;
    out[1] = s.w2;
}
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("slots")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-Werror", f"-I{CSRC}", str(d / "shim.cpp"),
                    "-o", str(d / "shim.so")], check=True)
    L = ctypes.CDLL(str(d / "shim.so"))
    i64 = ctypes.c_int64
    L.op_new.argtypes, L.op_new.restype = [i64] * 5, ctypes.c_void_p
    L.op_free.argtypes = [ctypes.c_void_p]
    L.op_room.argtypes = [ctypes.c_void_p, i64]
    L.op_ensure.argtypes = [ctypes.c_void_p, i64, ctypes.c_int, ctypes.c_int, ctypes.POINTER(i64)]
    L.op_limit.argtypes, L.op_limit.restype = [ctypes.c_void_p], i64
    L.op_part.argtypes = [ctypes.c_void_p, i64, ctypes.POINTER(i64)]
    return L


class Op:
    def __init__(self, L, Ps, Pt, b1, b2, room=1 << 60):
        self.L, self.h, self.b = L, L.op_new(Ps, Pt, b1, b2, room), (b1, b2)

    def __del__(self):
        self.L.op_free(self.h)

    def room(self, n):
        self.L.op_room(self.h, n)

    def limit(self):
        return self.L.op_limit(self.h)

    def part(self, n):
        o = (ctypes.c_int64 * 2)()
        self.L.op_part(self.h, n, o)
        return tuple(o)

    def ensure(self, nrhs, may_grow=True, pinned=False):
        o = (ctypes.c_int64 * 8)()
        self.L.op_ensure(self.h, nrhs, may_grow, pinned, o)
        self.status, self.ptr, self.held, self.calls, self.used = o[0], (o[1], o[2]), (o[3], o[4]), (o[5], o[6]), o[7]
        return self.status


OK, CAPTURE, PINNED, MEMORY = range(4)
MiB = 1 << 20


def test_a_smaller_count_moves_and_shrinks_nothing(shim):
    # 1 source, 2 target partitions of 128^3 ComplexF32: pair by pair at 5, in
    # one launch at 2, whose W1 is smaller and whose W2 is larger
    op = Op(shim, 1, 2, 128 * 128 * 256 * 3 * 8, 256 * 256 * 128 * 3 * 8)
    assert op.limit() == 2
    assert op.ensure(5) == OK
    ptr, held = op.ptr, op.held
    for n in (2, 1, 5, 3, 4, 2):
        assert op.ensure(n) == OK and op.ptr == ptr and op.held == held
    assert held[0] >= 5 and held[1] >= 6
    # reserved counts above the one-launch limit, then one eager right-hand side
    op = Op(shim, 8, 1, 60 * MiB, 100 * MiB)
    assert op.limit() == 1 and op.ensure(3) == OK
    ptr = op.ptr
    assert op.ensure(1) == OK and op.ptr == ptr
    op = Op(shim, 4, 4, 50 * MiB, 100 * MiB)
    assert op.ensure(6) == OK and op.ensure(1) == OK
    assert op.ensure(6, may_grow=False) == OK   # still reserved


def test_a_refused_size_is_asked_for_once(shim):
    op = Op(shim, 8, 1, 10 * MiB, 20 * MiB, room=100 * MiB)   # one launch takes 240 MiB, pair by pair 30
    assert op.ensure(1) == OK and op.held == (1, 1)
    ptr, calls = op.ptr, op.calls
    op.room(op.used)                                          # another allocator took the rest
    for _ in range(3):
        assert op.ensure(1) == OK and op.ptr == ptr and op.calls == calls
    # held planes that suffice are kept when larger ones cannot be had
    op = Op(shim, 8, 1, 10 * MiB, 20 * MiB, room=300 * MiB)
    assert op.ensure(1) == OK and op.held == (8, 8)
    ptr = op.ptr
    assert op.ensure(2) == OK and op.ptr == ptr
    calls = op.calls
    assert op.ensure(2) == OK and op.ensure(1) == OK and op.calls == calls


def test_capture_and_pinned(shim):
    op = Op(shim, 8, 1, MiB, MiB)
    assert op.ensure(1, may_grow=False) == CAPTURE and op.used == 0
    assert op.ensure(1) == OK
    ptr = op.ptr
    assert op.ensure(2, pinned=True) == OK and op.ptr == ptr      # 8 slots: pair by pair
    assert op.ensure(9, pinned=True) == PINNED and op.ptr == ptr
    assert op.ensure(9, may_grow=False) == CAPTURE and op.ptr == ptr
    assert op.ensure(3, may_grow=False) == OK and op.ptr == ptr   # captured: stays where it is
    assert op.ensure(3) == OK and op.ptr == ptr
    assert op.ensure(4) == OK and op.ptr != ptr and op.held == (32, 32)


@pytest.mark.parametrize("seed", range(40))
def test_random_orders(shim, seed):
    rng = random.Random(seed)
    Ps, Pt = rng.choice([(1, 1), (1, 2), (2, 1), (8, 1), (1, 27), (4, 4), (2, 3), (27, 1)])
    b1, b2 = (int(2 ** rng.uniform(10, 29)) for _ in range(2))
    need = lambda n: n * (b1 + b2)
    op = Op(shim, Ps, Pt, b1, b2, rng.choice([1 << 60, need(8), need(8 * Ps * Pt), 4 << 30]))
    most, fixed = 0, None          # the largest count ensured, and where its planes lie
    for _ in range(60):
        n, mode = int(2 ** rng.uniform(0, 6)), rng.choice(["eager", "eager", "capture", "pinned"])
        if rng.random() < 0.1:
            op.room(rng.choice([1 << 60, need(4), need(8 * Ps * Pt), 4 << 30]))
        before = getattr(op, "calls", (0, 0))
        st = op.ensure(n, may_grow=mode != "capture", pinned=mode == "pinned")
        assert op.used == op.held[0] * b1 + op.held[1] * b2      # nothing lost, nothing kept twice
        if st == OK:
            assert op.held[0] >= n and op.held[1] >= n
        if mode != "eager":
            assert op.calls == before
            assert st in (OK, CAPTURE if mode == "capture" else PINNED)
        if n <= most:
            assert st == OK and op.ptr == fixed and op.calls == before
        elif st == OK and mode != "pinned":
            most, fixed = n, op.ptr
        elif st == MEMORY:
            most, fixed = 0, None
        elif most:
            assert op.ptr == fixed


@pytest.mark.parametrize("Ps,Pt", [(8, 1), (1, 8), (2, 2), (3, 1)])
def test_every_count_up_to_the_ensured_one_has_its_form(shim, Ps, Pt):
    # with memory enough, each count the one-launch form takes finds its slots
    op = Op(shim, Ps, Pt, 40 * MiB, 70 * MiB)
    assert 1 <= op.limit() < 30
    assert op.ensure(30) == OK
    for n in range(1, op.limit() + 1):
        w1, w2 = op.part(n)
        assert op.held[0] >= w1 and op.held[1] >= w2
        assert w1 * 40 * MiB + w2 * 70 * MiB <= 2 << 30
    w1, w2 = op.part(op.limit() + 1)
    assert w1 * 40 * MiB + w2 * 70 * MiB > 2 << 30
