"""The marks of a hand-over inside a launch, as a model on the CPU: units that start at any time, values that carry the launch's number, waits
that are given up.  What a launch takes has to be of that launch, whatever became of the launches before it."""
import itertools

import pytest

UNITS, WAIT, STEP = 4, 3, 16


class Memory:
    """One slot per unit (value, tag), the word that the number is read from, the error word of a step."""

    def __init__(self):
        self.slots, self.word, self.err = [(None, 0)] * UNITS, 0, False


def unit(m, u, launch, delay, advances):
    """One unit of launch `launch`: starts `delay` turns late, reads the launch's number, stores its value with it, takes every unit's."""
    for _ in range(delay):
        yield
    tag = m.word + 1
    yield
    m.slots[u] = (launch, tag)
    yield
    for _ in range(WAIT):
        if all(t == tag for _, t in m.slots):
            taken = [v for v, _ in m.slots]
            assert all(v == launch for v in taken) or m.err, f"unit {u} of launch {launch} took {taken} and nothing was reported"
            break
        yield
    else:
        m.err = True
    if advances and u == 0:
        m.word += 1


def run_steps(advances):
    """Steps of one launch each: one with units that start when the others have left, then one with units that start a little late."""
    refused = 0
    for late in itertools.product((0, 3 * WAIT), repeat=UNITS):
        for behind in itertools.product((0, WAIT - 1), repeat=UNITS):
            m = Memory()
            for launch, delays in enumerate(((0,) * UNITS, late, behind)):
                m.err = False
                if not advances:
                    m.word += STEP                                      # the step's first kernel: before any launch that waits
                live = [unit(m, u, launch, delays[u], advances) for u in range(UNITS)]
                while live:                                             # (a launch ends when all of its units have)
                    live = [g for g in live if next(g, "left") != "left"]
                refused += m.err
    assert refused                                                      # (somebody gave up)


def test_a_number_of_the_step_stays_with_its_launch():
    """StepCtl.launch: advanced between launches only."""
    run_steps(advances=False)


def test_a_number_that_a_unit_advances_can_leave_its_launch():
    """The model sees the fault it is there for: unit 0 gives up and advances the word, a unit that starts later marks its value with
    the next launch's number, which the next launch takes for its own."""
    with pytest.raises(AssertionError, match="nothing was reported"):
        run_steps(advances=True)


@pytest.mark.parametrize("cleared_every,sound", [(4, True), (7, True), (None, False)])
def test_marks_that_come_round(cleared_every, sound):
    """Marks of 8 steps: blocks whose last units' slots lie unused for any number of steps and are then waited for.  A slot that was last written
    8 steps ago holds the present mark; cleared in less than that, no slot is that old."""
    around = 8 * STEP
    for idle in range(1, 20):
        m, since, taken = Memory(), 0, True
        for step in range(2 * idle + 2):
            if cleared_every and since + 1 > cleared_every:
                m.slots, since = [(None, 0)] * UNITS, 0
            since += 1
            tag = ((step + 1) * STEP + 1) % around              # (number + 1, as lg_tag has it)
            wide = step % (idle + 1) == 0
            taken &= not (wide and m.slots[UNITS - 1][1] == tag)  # there before the unit has stored it
            for u in range(UNITS if wide else UNITS - 1):
                m.slots[u] = (step, tag)
        if not sound and not taken:
            return
        assert taken
    assert sound


class Model:
    """A caller thread and its stream: steps that were launched and have not ended, True for one with launches that wait."""

    def __init__(self):
        self.launching = self.plain = self.recorded = False
        self.stream, self.mark = [], 0                          # mark: how many of the stream's steps lie ahead of the recorded event


def caller(models, me, turns, steps, checks_launching):
    """The calls of one model: begin (under the lock: one turn of the model here), then the launches, then the end."""
    for _ in range(steps):
        me.launching, me.plain = True, False
        last = turns[0]
        if last is not None and last is not me:
            if checks_launching and last.launching:
                me.plain = True
            else:
                if not last.recorded:
                    last.recorded, last.mark = True, len(last.stream)
                me.plain = last.mark > 0
        if not me.plain:
            turns[0], me.recorded = me, False
        yield
        me.stream.append(not me.plain)
        yield
        me.launching = False
        assert sum(any(m.stream) for m in models) <= 1, "two models have launches that wait"
        yield


@pytest.mark.parametrize("checks_launching", [True, False])
def test_one_model_at_a_time_has_launches_that_wait(checks_launching):
    """Threads and streams in any order: the latest model with such launches keeps them until its stream has ended them.  Without the look at a step that
    is still being launched the model sees the fault: the event lies ahead of it."""
    import random
    seen = False
    for seed in range(400):
        rng, turns, models = random.Random(seed), [None], [Model() for _ in range(3)]
        live = [caller(models, m, turns, 6, checks_launching) for m in models]
        try:
            while live:
                g = rng.choice(live)
                if next(g, "left") == "left":
                    live.remove(g)
                m = rng.choice(models)
                if m.stream and rng.random() < 0.4:             # the device ends a step
                    m.stream.pop(0)
                    m.mark = max(0, m.mark - 1)
        except AssertionError:
            seen = True
    assert seen is not checks_launching


class Device:
    """Streams of (kind, what has to have ended before) in order; an entry runs when it is at the front of its stream and nothing is left to wait for."""

    def __init__(self, n):
        self.streams, self.done = [[] for _ in range(n)], [0] * n

    def running(self):
        return [s[0][0] for s in self.streams if s and (s[0][1] is None or self.done[s[0][1][0]] >= s[0][1][1])]

    def end(self, i):
        s = self.streams[i]
        if s and (s[0][1] is None or self.done[s[0][1][0]] >= s[0][1][1]):
            s.pop(0)
            self.done[i] += 1


def server(dev, ms, me, turns, rng, checks_prompts):
    """The calls of one model: steps (as `caller` has them) and prompts, which the host waits for."""
    for _ in range(8):
        m = ms[me]
        if rng.random() < 0.4:
            dep = None
            if checks_prompts:
                m.prompting = True
                yield
                last = turns[0]
                while last is not None and last != me and ms[last].launching:
                    yield
                    last = turns[0]
                if last is not None and last != me:
                    dep = (last, dev.done[last] + len(dev.streams[last]))
            want = dev.done[me] + len(dev.streams[me]) + 2
            for _ in range(2):
                dev.streams[me].append(("prompt", dep))
                yield
            while dev.done[me] < want:
                yield
            m.prompting = False
        else:
            m.launching, m.plain = True, False
            last = turns[0]
            if checks_prompts and any(o.prompting for o in ms if o is not m):
                m.plain = True
            elif last is not None and last != me:
                m.plain = ms[last].launching or "waiting" in [k for k, _ in dev.streams[last]]
            if not m.plain:
                turns[0] = me
            yield
            dev.streams[me].append(("plain" if m.plain else "waiting", None))
            yield
            m.launching = False
        yield


@pytest.mark.parametrize("checks_prompts", [True, False])
def test_no_prompt_runs_beside_launches_that_wait(checks_prompts):
    """Threads and streams in any order: a prompt's blocks and launches that wait are never on the device together.  Without the count of prompts, and the wait
    of a prompt's stream for what was launched before it, the model sees them there."""
    import random
    together = twos = 0
    for seed in range(400):
        rng, turns, dev, ms = random.Random(seed), [None], Device(3), [Model() for _ in range(3)]
        for m in ms:
            m.prompting = False
        live = [server(dev, ms, i, turns, rng, checks_prompts) for i in range(3)]
        for _ in range(20000):
            if not live:
                break
            g = rng.choice(live)
            if next(g, "left") == "left":
                live.remove(g)
            if rng.random() < 0.5:
                dev.end(rng.randrange(3))
            on = dev.running()
            together += "prompt" in on and "waiting" in on
            twos += on.count("waiting") > 1
        assert not live, "a thread waits for ever"
    assert not twos and bool(together) is not checks_prompts


SHIM = """
#include "%s/lg_far.h"
struct U { unsigned x, y, z, w; };
extern "C" void put(const unsigned *xyz, unsigned tag, unsigned *u) { const U v = lg_far_unit<U>(xyz[0], xyz[1], xyz[2], lg_far_marks(tag)); u[0] = v.x; u[1] = v.y; u[2] = v.z; u[3] = v.w; }
extern "C" int take(const unsigned *u, unsigned tag, unsigned *xyz) {
    const U v = { u[0], u[1], u[2], u[3] };
    xyz[0] = v.x; xyz[1] = lg_far_y(v); xyz[2] = v.z;
    return lg_far_miss(v, lg_far_marks(tag)) == 0;
}
"""


@pytest.fixture(scope="module")
def far(tmp_path_factory):
    """put(three words, step, layer) -> a unit; take(unit, step, layer) -> its words, or None: the functions that the kernels call, built for the host."""
    import ctypes as C
    import os
    import subprocess
    d = tmp_path_factory.mktemp("far")
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "little-gemma_amd", "csrc")
    (d / "far.cpp").write_text(SHIM % csrc)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(d / "far.so"), str(d / "far.cpp")], check=True)
    L = C.CDLL(str(d / "far.so"))
    U3, U4 = C.c_uint * 3, C.c_uint * 4

    def tag(step, layer):
        return (step * 256 + layer + 1) << 4 & 0xFFFFFFFF               # (lg_far_tag(lg_tag(launch + layer)))

    def put(words, step, layer):
        u = U4()
        L.put(U3(*words), C.c_uint(tag(step, layer)), u)
        return list(u)

    def take(u, step, layer):
        w = U3()
        return list(w) if L.take(U4(*u), C.c_uint(tag(step, layer)), w) else None
    return put, take


def words(rng):
    """What rows hold, and what hides a mix of two of them best: zeros and equal words."""
    return rng.choice(([0, 0, 0], [w := rng.getrandbits(32), w, w], [rng.getrandbits(32) for _ in range(3)]))


@pytest.mark.parametrize("layers", [(0, 1), (3, 7, 11, 254), tuple(range(42))])
def test_a_unit_of_a_launch_is_whole_and_its_own(far, layers):
    """A unit in memory, written by the launches of steps of any width (some leave it alone), seen with either half of the present and the other of the launch before it at
    that place: taken only when both are the present launch's; nor is one of any earlier launch, or cleared memory, taken whole."""
    import random
    put, take = far
    rng = random.Random(len(layers))
    cell, step = [0, 0, 0, 0], rng.getrandbits(20)
    for _ in range(300):
        step = (step + rng.choice((1, 1, 2, 255, 256, 257, rng.randrange(1, 1 << 15)))) % (1 << 20)
        for layer in layers:
            w = words(rng)
            new = put(w, step, layer)
            assert take(cell, step, layer) is None
            assert take([0, 0, 0, 0], step, layer) is None
            assert take(new[:2] + cell[2:], step, layer) is None and take(cell[:2] + new[2:], step, layer) is None, (step, layer)
            assert take(new, step, layer) == w
            cell = new


def test_a_unit_of_the_only_layer_with_such_launches(far):
    """The same layer step after step: halves of steps up to 254 apart do not fit together, whole units up to 2^16 - 1 (they are cleared in half that)."""
    import random
    put, take = far
    rng = random.Random(1)
    for step in [rng.getrandbits(20) for _ in range(40)] + [255, 256, 65535, 65536, (1 << 20) - 1]:
        w = words(rng)
        new = put(w, step, 5)
        for back in list(range(1, 255)) + [255, 256, 511, 512, 65280, 65535] + [rng.randrange(255, 1 << 16) for _ in range(50)]:
            old = put(w, (step - back) % (1 << 20), 5)
            assert take(old, step, 5) is None
            if back < 255:
                assert take(new[:2] + old[2:], step, 5) is None and take(old[:2] + new[2:], step, 5) is None
