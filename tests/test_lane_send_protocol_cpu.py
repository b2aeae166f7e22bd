"""CPU model of the inbox protocol's two wide paths, under random
interleavings (include/charming_detail/device_rt.h; the single-message paths
are modelled in test_inbox_protocol_cpu.py, whose ring and chares are used
here).

send_lanes: the lanes of a sender reserve, write and publish one message each,
in their own destinations; a lane without room waits, after the others have
published, then writes and publishes by itself (or gives up: a send to the
sender's own full inbox at once, else at the spin limit or when the run
stops).  poll_next: the consumer reads the ready words of its read position
and of the 15 granules after it, makes one acquire if the first is published,
and takes the messages found published with it without reading their words
again.  A message's bytes count as seen only if it was published before the
consumer's last acquire."""
import random

import pytest
from test_inbox_protocol_cpu import (ERR_SELF_RING_FULL, ERR_SPIN_LIMIT,
                                     GRANULE, Chare, Error, Inbox, alloc_size,
                                     defer, deliver_in_order, producer, run)

AHEAD = 16


def lane_sender(boxes, sends, me=None, spin_limit=0, stop=lambda: False,
                early_tag=False):
    """Generator: one PE making send_lanes calls; a send is a list of
    (destination, message).  early_tag plants a mistake: a late lane
    publishes before it writes."""
    for lanes in sends:
        st = []
        for dst, m in lanes:
            slot = -(-alloc_size(m["bytes"]) // GRANULE) * GRANULE
            box = boxes[dst]
            st.append(dict(dst=dst, box=box, m=dict(m, slot=slot), pos=box.tail,
                           slot=slot))
            box.tail += slot
            yield

        def room(s):
            return s["pos"] + s["slot"] - s["box"].head <= s["box"].R

        def write(s):
            s["box"].mem[s["pos"]] = s["m"]

        def publish(s):
            g = s["pos"] // GRANULE
            s["box"].ready[g % s["box"].NG] = g + 1

        for s in st:
            s["late"] = not room(s)
            if not s["late"]:
                write(s)
            yield
        for s in st:                 # after the barrier and the release
            if not s["late"]:
                publish(s)
                yield
        spins = 0
        while any(s["late"] for s in st):
            spins += 1
            for s in st:
                if not s["late"]:
                    continue
                if room(s):
                    steps = [write, publish]
                    for f in reversed(steps) if early_tag else steps:
                        f(s)
                        yield
                    s["late"] = False
                elif s["dst"] == me:
                    s["box"].raise_error(ERR_SELF_RING_FULL)
                elif stop():
                    s["late"] = False
                elif spin_limit and spins > spin_limit:
                    s["box"].raise_error(ERR_SPIN_LIMIT)
            yield


def wide_consumer(box, chare, deliver, n_total, keep_bits=False):
    """Generator: the scheduler loop with poll_next's look ahead.  keep_bits
    plants a mistake: bits read after the acquire count as acquired."""
    done, base, seen, acquired = 0, 0, 0, set()

    def published():
        return {p for p in box.mem
                if box.ready[p // GRANULE % box.NG] == p // GRANULE + 1}
    while done < n_total:
        revived = [d for d in box.deferred if d[3] == 2]
        if revived:
            d = min(revived, key=lambda e: e[4])
            if chare.gate(d[2]["refnum"]):
                box.deferred.remove(d)
                if not box.deferred:
                    box.arena_used = 0
                deliver(d[2], chare)
                done += 1
            else:
                d[3] = 1
            yield
            continue
        g = box.read_pos // GRANULE
        at = g - base
        if not (at < AHEAD and seen >> at & 1):
            found = 0
            for k in range(AHEAD):   # (no order among the lanes' loads)
                found |= (box.ready[(g + k) % box.NG] == g + k + 1) << k
                if k % 5 == 0:
                    yield
            if not found & 1:
                continue
            acquired = published()
            yield
            if keep_bits:
                for k in range(AHEAD):
                    found |= (box.ready[(g + k) % box.NG] == g + k + 1) << k
            base, seen = g, found
        assert box.read_pos in acquired, "read before it was acquired"
        m = box.mem.pop(box.read_pos)
        if chare.gate(m["refnum"]):
            deliver(m, chare)
            done += 1
        else:
            defer(box, m)
        yield
        box.read_pos += m["slot"]
        box.head = box.read_pos
        yield


def _msg(src, k, refnum, nbytes):
    return {"src": src, "k": k, "refnum": refnum, "bytes": nbytes,
            "payload": ("p", src, k, nbytes)}


def _setup(rng, ring_bytes, n_dst, n_lane_pes, per, n_single):
    """Refnums 0 .. N-1 of each destination, spread over senders by lanes (one
    message to every destination a send) and, for destination 0, single
    ones."""
    boxes = [Inbox(ring_bytes, 1 << 20) for _ in range(n_dst)]
    chares = [Chare(b) for b in boxes]
    refs = []
    for d in range(n_dst):
        n = n_lane_pes * per + (n_single if d == 0 else 0)
        refs.append(rng.sample(range(n), n))
    senders = []
    for p in range(n_lane_pes):
        senders.append([[(d, _msg(p, k, refs[d][p * per + k],
                                  rng.choice([0, 8, 24, 64])))
                         for d in rng.sample(range(n_dst), n_dst)]
                        for k in range(per)])
    single = [_msg(n_lane_pes, k, refs[0][n_lane_pes * per + k],
                   rng.choice([8, 100, 200])) for k in range(n_single)]
    return boxes, chares, refs, senders, single


@pytest.mark.parametrize("ring_bytes", [512, 1024, 4096])
@pytest.mark.parametrize("seed", range(8))
def test_exactly_once_in_refnum_order(seed, ring_bytes):
    # rings of 8, 16 and 64 granules: fewer than are looked ahead, as many,
    # more; hundreds of laps of the smallest, most sends with late lanes
    rng = random.Random(seed * 7 + ring_bytes)
    boxes, chares, refs, senders, single = _setup(rng, ring_bytes, 3, 3, 25, 20)
    gens = [lane_sender(boxes, s) for s in senders]
    gens.append(producer(boxes[0], 3, False, single, 0))
    gens += [wide_consumer(b, c, deliver_in_order, len(r))
             for b, c, r in zip(boxes, chares, refs)]
    run(gens, rng)
    for b, c, r in zip(boxes, chares, refs):
        assert c.got == list(range(len(r)))
        assert b.head == b.tail == b.read_pos and not b.mem and b.error == 0


def test_a_late_lane_holds_back_no_other():
    # destination 1's consumer never runs: destination 0 gets every message
    # that its lanes made before the wait
    rng = random.Random(5)
    boxes = [Inbox(1024, 1 << 20) for _ in range(2)]
    chare, got = Chare(boxes[0]), []
    fit = 1024 // GRANULE
    sends = [[(1, _msg(0, k, -1, 8)), (0, _msg(0, k, -1, 8))]
             for k in range(fit + 1)]
    stop = [False]
    gens = [lane_sender(boxes, sends, stop=lambda: stop[0]),
            wide_consumer(boxes[0], chare, lambda m, c: got.append(m["k"]),
                          fit + 1)]
    live = list(gens)
    for _ in range(20000):
        g = rng.choice(live)
        try:
            next(g)
        except StopIteration:
            live.remove(g)
        if len(got) == fit + 1:
            stop[0] = True
        if not live:
            break
    assert not live and got == list(range(fit + 1))
    assert len(boxes[1].mem) == fit


def test_full_inboxes_end_in_the_documented_errors():
    sends = [[(0, _msg(0, k, -1, 8)), (1, _msg(0, k, -1, 8))]
             for k in range(20)]
    boxes = [Inbox(1024, 1 << 20) for _ in range(2)]
    with pytest.raises(Error) as e:
        run([lane_sender(boxes, sends, spin_limit=50)], random.Random(1))
    assert e.value.code == ERR_SPIN_LIMIT
    boxes = [Inbox(1024, 1 << 20), Inbox(1 << 16, 1 << 20)]
    with pytest.raises(Error) as e:
        run([lane_sender(boxes, sends, me=0)], random.Random(2))
    assert e.value.code == ERR_SELF_RING_FULL


@pytest.mark.parametrize("mistake", ["early_tag", "keep_bits"])
def test_planted_mistakes_are_caught(mistake):
    caught = 0
    for seed in range(20):
        rng = random.Random(300 + seed)
        boxes, chares, refs, senders, single = _setup(rng, 512, 2, 3, 25, 10)
        gens = [lane_sender(boxes, s, early_tag=mistake == "early_tag")
                for s in senders]
        gens.append(producer(boxes[0], 3, False, single, 0))
        gens += [wide_consumer(b, c, deliver_in_order, len(r),
                               keep_bits=mistake == "keep_bits")
                 for b, c, r in zip(boxes, chares, refs)]
        try:
            run(gens, rng)
        except (AssertionError, KeyError):
            caught += 1
    assert caught > 0
