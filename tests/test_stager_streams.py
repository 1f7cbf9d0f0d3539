"""The stager's device backend over a model of HIP's streams and events (fake_hip_streams.cpp): no copy into a slot may start
before the reads and the copies in front of it are certain to be done, and no reader before the copy that it acquired."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "moe_gen_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    out = tmp_path_factory.mktemp("fake_hip")
    objs = []
    for src in (os.path.join(CSRC, "stage.cpp"), os.path.join(HERE, "fake_hip_streams.cpp")):
        objs.append(str(out / (os.path.basename(src) + ".o")))
        subprocess.check_call([HIPCC, "-O1", "-std=c++17", "-fPIC", "--offload-host-only", "--offload-arch=gfx950", "-x", "hip", "-c", src,
                               "-o", objs[-1]])
    so = str(out / "libstage.so")
    # (the runtime's names are bound to the model's, whatever else the process has loaded)
    subprocess.check_call(["g++", "-shared", "-Wl,-Bsymbolic", *objs, "-lpthread", "-o", so])
    return so


class Pool:
    """One module type of `slots` slots over the model; a module's bytes are its id.  Notes what every consumer stream read."""

    def __init__(self, library, slots, modules, pageable=(), on_demand=True, slot_bytes=64):
        self.slot_bytes = slot_bytes
        # a library of its own per pool: the model's streams and log are global
        so = f"{library}.{Pool.count}"
        Pool.count += 1
        os.link(library, so)
        L = self.L = ctypes.CDLL(so)
        for f in ("moe_last_error", "fake_clock", "fake_copies"):
            getattr(L, f).restype = ctypes.c_char_p
        L.fake_kernel.restype = ctypes.c_uint64
        for f in ("fake_kernel", "fake_clock"):
            getattr(L, f).argtypes = [ctypes.c_void_p]
        self.mem = (ctypes.c_uint8 * (slots * slot_bytes))()
        self.base = ctypes.addressof(self.mem)
        self.st = ctypes.c_void_p()
        self.ok(L.moe_stage_create(ctypes.byref(self.st), 1, (ctypes.c_size_t * 1)(slot_bytes), (ctypes.c_int32 * 1)(slots),
                                   (ctypes.c_void_p * 1)(self.base), 0))
        if pageable:
            self.ok(L.moe_stage_set_bounce(self.st, 2, ctypes.c_size_t(4096), 1))
        self.src = [(ctypes.c_uint8 * slot_bytes)(*([m] * slot_bytes)) for m in range(modules)]
        for m in range(modules):
            add = L.moe_stage_add_module_pageable if m in pageable else L.moe_stage_add_module
            assert add(self.st, 0, 1, (ctypes.c_void_p * 1)(ctypes.addressof(self.src[m])), (ctypes.c_size_t * 1)(slot_bytes),
                       (ctypes.c_size_t * 1)(0)) == m
        if on_demand:
            self.ok(L.moe_stage_set_policy(self.st, 0, 1))
        self.slots, self.held, self.reads = slots, {}, []

    count = 0

    def ok(self, rc):
        assert rc == 0, self.L.moe_last_error()

    def copies(self):
        """(slot, stream, number, clock) of every copy so far"""
        out = []
        for line in self.L.fake_copies().decode().splitlines():
            head, clock = line.split("|")
            dst, _, stream, number = map(int, head.split())
            out.append(((dst - self.base) // self.slot_bytes, stream, number, dict(map(int, c.split(":")) for c in clock.split())))
        return out

    def fetch(self, *ids):
        return self.L.moe_stage_fetch(self.st, (ctypes.c_int32 * len(ids))(*ids), len(ids), None)

    def acquire(self, m, stream):
        slot = ctypes.c_int32(-1)
        rc = self.L.moe_stage_acquire(self.st, m, ctypes.c_void_p(stream), ctypes.byref(slot))
        if rc != 0:
            return False
        s = slot.value
        into = [c for c in self.copies() if c[0] == s]
        clock = dict(map(int, c.split(":")) for c in self.L.fake_clock(stream).decode().split())
        assert all(clock.get(st, 0) >= number for _, st, number, _ in into), f"module {m}: read in front of its copy"
        assert bytes(self.mem[s * self.slot_bytes:(s + 1) * self.slot_bytes]) == bytes([m] * self.slot_bytes), f"module {m}: slot {s} holds other weights"
        self.held[m] = (s, stream, len(into))
        return True

    def release(self, m, stream=None):
        """of a held module, behind a kernel that reads it; or of a resident one that nobody acquired, on `stream`"""
        if m in self.held:
            s, stream, n = self.held.pop(m)
            number = self.L.fake_kernel(stream)
            into = [c for c in self.copies() if c[0] == s]
            assert len(into) == n, f"module {m}: slot {s} was overwritten while it was held"
            self.reads.append((s, stream, number, len(self.copies())))
        self.ok(self.L.moe_stage_release(self.st, m, ctypes.c_void_p(stream)))

    def check(self):
        log = self.copies()
        for s, stream, number, at in self.reads:
            for slot, _, _, clock in log[at:]:
                assert slot != s or clock.get(stream, 0) >= number, f"slot {s}: refilled before stream {stream:#x} has read it"
        for s in range(self.slots):
            into = [c for c in log if c[0] == s]
            for (_, stream, number, _), (_, _, _, clock) in zip(into, into[1:]):
                assert clock.get(stream, 0) >= number, f"slot {s}: two copies at once"

    def close(self):
        self.ok(self.L.moe_stage_destroy(self.st))


A, B, C = 0xa0, 0xb0, 0xc0


@pytest.mark.parametrize("pageable", [False, True])
def test_a_shared_release_event_outlives_the_next_release(library, pageable):
    """Slots 0 and 1 are let go on one stream, which takes one event; what refills slot 0 is dropped unread on another stream and the
    slot refilled again, which takes another event; slot 1's refill still waits for the first."""
    p = Pool(library, 2, 6, range(6) if pageable else ())
    assert p.acquire(0, A) and p.acquire(1, A)
    p.release(0)
    p.release(1)
    assert p.fetch(2) == 0                                   # into slot 0
    p.release(2, B)
    assert p.fetch(3) == 0                                   # into slot 0 again
    assert p.acquire(4, B) and p.acquire(3, B)               # 4 into slot 1, behind A's reads
    p.release(3)
    p.release(4)
    p.check()
    p.close()


def test_a_pinned_module_follows_a_queued_copy_into_its_slot(library):
    """A module of ordinary memory is dropped, or taken over, while the worker has still to copy it: a pinned module that gets its slot
    is copied behind it, not under it."""
    p = Pool(library, 1, 2, pageable=(0,), slot_bytes=1 << 18)               # (64 chunks: the worker is still at it)
    for i in range(6):
        assert p.fetch(0) == 0
        p.release(0, B)
        assert p.acquire(1, A)
        p.release(1)
    p.ok(p.L.moe_stage_sync(p.st))
    p.check()
    p.close()


@pytest.mark.parametrize("seed", range(24))
def test_random_calls_of_several_consumer_streams(library, seed):
    rng = random.Random(seed)
    modules = 9
    pageable = ((), range(modules), range(0, modules, 2))[seed % 3]
    p = Pool(library, rng.choice([1, 2, 3, 5]), modules, pageable, on_demand=seed % 4 != 0)
    for _ in range(120):
        what, m = rng.random(), rng.randrange(modules)
        if what < 0.35 and p.held:
            p.release(rng.choice(sorted(p.held)))
        elif what < 0.55:
            p.fetch(*rng.sample(range(modules), rng.choice([1, 1, 2])))       # (refused where no slot is free)
        elif what < 0.62:
            if m not in p.held and p.L.moe_stage_resident(p.st, m) == 1:
                p.release(m, rng.choice([A, B, C]))
        elif what < 0.66:
            assert p.L.moe_stage_pump(p.st) >= 0
        elif m not in p.held:
            p.acquire(m, rng.choice([A, B, C]))
    for m in sorted(p.held):
        p.release(m)
    p.ok(p.L.moe_stage_sync(p.st))
    p.check()
    p.close()
