"""The forward scan's waits for its -W rows (csrc/gdn_fwd.hip, fwd_scan_kernel), on a model of a wave's
vector memory queue and on the built kernel.

A wave copies its 16 rows of -W of a chunk into an LDS ring four steps ahead and reads them back as
fragments.  It cannot wait for one copy: its operations retire in issue order and it can only wait until
at most N of them are in flight, so N must not exceed the operations that were surely issued after the
copy.  The compiler keeps an operation inside its window between two barriers and may reorder there, so
what counts is the operations of whole windows: those between the copy's window and the wait's.

The model issues the windows of a document of n chunks as the kernel does (the prologue, a peeled first
round, rounds of four steps, up to three last steps that request nothing) and checks every wait before the
rows are read; one operation more must be caught in each place.  The built kernel must have the model's
operations in its windows and no wait looser than the model's.
"""

import pytest

from kernel_windows import LIB, OBJDUMP, windows

DEPTH = 4
W_OPS = ["copy"] * 4 + ["u"]  # issue_w: four copies of four rows, and the U^T load
K_OPS = ["k"] * 4             # issue_k
LIMITS = {"start": 27, "first round": 19, "round": 27, "last 0": 19, "last 1": 12, "last 2": 5}


class ProtocolError(AssertionError):
    pass


def replay(n, limits=LIMITS):
    """Check the waits of a document of n > 0 chunks."""
    issued = []  # windows in order: (operations, the step whose -W is among them or None)

    def window(ops, copies=None):
        issued.append((ops, copies))

    def wait(step, limit):
        at = [i for i, (_, copies) in enumerate(issued) if copies == step]
        if not at:
            raise ProtocolError(f"-W of step {step} was never requested")
        after = sum(len(ops) for ops, _ in issued[at[-1] + 1:])
        if after < limit:
            raise ProtocolError(f"-W of step {step} may be in flight: {after} operations issued after it, {limit} left")

    for x in range(DEPTH):
        window(W_OPS + (K_OPS if x else []), copies=x)
    wait(0, limits["start"])
    tau = 0

    def step(name, more):
        nonlocal tau
        window((K_OPS if more else []) + ["store h"])  # up to the barrier between the contractions
        wait(tau + 1, limits[name])                    # read right after it, before the second's requests
        window((W_OPS if more else []) + ["store v"], copies=tau + DEPTH if more else None)
        tau += 1

    while tau + DEPTH <= n:
        name = "round" if tau else "first round"
        for _ in range(DEPTH):
            step(name, True)
    for i in range(n - tau):
        step(f"last {i}", False)
    return tau


@pytest.mark.parametrize("n", list(range(1, 14)) + [144])
def test_every_wait_covers_its_copies(n):
    assert replay(n) == n


@pytest.mark.parametrize("place", sorted(LIMITS))
def test_a_looser_wait_is_caught(place):
    """Each limit is tight, but the peeled round's: it leaves out its first step's own Kg^T loads."""
    slack = 4 if place == "first round" else 0
    with pytest.raises(ProtocolError, match="may be in flight"):
        for n in range(1, 14):
            replay(n, dict(LIMITS, **{place: LIMITS[place] + slack + 1}))
    for n in range(1, 14):
        replay(n, dict(LIMITS, **{place: LIMITS[place] + slack}))


@pytest.mark.skipif(not (LIB.exists() and OBJDUMP.exists()), reason="needs the built library and llvm-objdump")
@pytest.mark.parametrize("kernel", ["fwd_scan_kernelIDF16bLb0EE", "fwd_scan_kernelIDF16_Lb0EE",
                                    "fwd_scan_kernelIDF16bLb1EE", "fwd_scan_kernelIDF16_Lb1EE"])
def test_the_built_kernel_keeps_its_windows(kernel, tmp_path):
    ws = windows(kernel, str(tmp_path))
    waits = lambda w: [x[1] for x in w if isinstance(x, tuple)]

    def ring_wait(w):
        """The strictest wait ahead of the window's last four LDS reads, the ring's."""
        reads = [i for i, x in enumerate(w) if x == "read"]
        return min(waits(w[:reads[-4]]), default=63)

    # the prologue: 16 copies, 4 + 12 operand loads and the table's, then the first wait
    assert ws[0].count("copy") == 16 and ws[0].count("load") >= 16
    assert ring_wait(ws[0]) <= LIMITS["start"]
    # full steps: the peeled round, then the loop
    full = [i for i, w in enumerate(ws) if i and "copy" in w]
    assert len(full) == 2 * DEPTH
    for place, i in enumerate(full):
        first, second = ws[i - 1], ws[i]
        assert first.count("load") >= len(K_OPS) and first.count("store") == 1, first
        assert second.count("copy") == 4 and second.count("load") >= 1 and second.count("store") == 1, second
        assert ring_wait(second) <= LIMITS["first round" if place < DEPTH else "round"], second
    # the last steps that read another's -W: two of the three
    last = [w for w in ws[1:] if "copy" not in w and "load" not in w and w.count("read") >= 7]
    assert len(last) == 2
    for w, limit in zip(sorted(last, key=ring_wait), (LIMITS["last 1"], LIMITS["last 0"])):
        assert w.count("store") == 1 and ring_wait(w) <= limit, w
