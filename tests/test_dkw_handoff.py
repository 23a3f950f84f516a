"""The reverse scan's hand-off to a bwd_dkw running beside it (csrc/gdn_bwd.hip: bwd_scan_kernel's
announcements, bwd_dkw_kernel's wait), on a model of the four waves' vector memory queues and on the
built kernel.

Each wave of a value-slice workgroup stores a quarter of every step's dS and dVn.  A chunk is announced
(one atomic add, by wave 0) three steps later: at the end of a full step every wave waits until at most 36
of its operations are in flight, a barrier follows, and wave 0 announces.  A wave's operations retire in
issue order, so the wait covers a store once at least 36 operations were surely issued after it; the
compiler keeps an operation inside its window between two barriers and may reorder there, so what counts
is the operations of whole windows.  After the last step every wave waits for everything, and wave 0
announces the rest.

The model asserts that every announcement follows all stores of its step by all four waves, and that every
step is announced once, in the order in which the scan finishes them; a looser wait, an announcement a step
early and one without the barrier must fail.  The built kernel must have the model's operations in its
windows.
"""

import pytest

from kernel_windows import LIB, OBJDUMP, windows

DEPTH = 4
FIRST = 5    # -W^T's four loads and the store of dS, up to the barrier between the contractions
SECOND = 7   # kdec Kn's four loads, dv_local, X and the store of dVn
ANNOUNCE = 3
LIMIT = ANNOUNCE * (FIRST + SECOND)  # BWD_ANNOUNCE * BWD_STEP_OPS


class ProtocolError(AssertionError):
    pass


def replay(n, limit=LIMIT, announce=ANNOUNCE, barrier=True):
    """The steps of a document of n chunks announced, in order."""
    issued = []  # per window: (step, operations); every wave issues the same
    known = [0]  # windows surely retired when wave 0 announces, for the wave that knows least
    announced = []

    def retired(operations_left):
        """Windows whose every operation has retired once at most that many are in flight."""
        left = 0
        for i in range(len(issued) - 1, -1, -1):
            if left >= operations_left:
                return i + 1
            left += issued[i][1]
        return 0

    def publish(step):
        last = max(i for i, (s, _) in enumerate(issued) if s == step)
        if last >= known[0]:
            raise ProtocolError(f"step {step} announced while its stores may be in flight")
        announced.append(step)

    tau = 0
    while tau + DEPTH <= n:
        for _ in range(DEPTH):
            issued += [(tau, FIRST), (tau, SECOND)]
            now = retired(limit)
            if barrier:
                known[0] = now
            if tau >= announce:
                publish(tau - announce)
            known[0] = now  # without the barrier the other waves are a step behind wave 0
            tau += 1
    for _ in range(n - tau):
        issued += [(tau, 1), (tau, 1)]  # the stores alone
        tau += 1
    known[0] = len(issued)
    for step in range(len(announced), n):
        publish(step)
    return announced


@pytest.mark.parametrize("n", list(range(14)) + [144])
def test_reverse_scan_announcements_follow_their_stores(n):
    assert replay(n) == list(range(n))


def test_a_looser_wait_is_caught():
    with pytest.raises(ProtocolError, match="may be in flight"):
        replay(9, limit=LIMIT + 1)


def test_an_announcement_a_step_early_is_caught():
    with pytest.raises(ProtocolError, match="may be in flight"):
        replay(9, announce=ANNOUNCE - 1)


def test_an_announcement_without_the_barrier_is_caught():
    with pytest.raises(ProtocolError, match="may be in flight"):
        replay(9, barrier=False)


def test_chunk_counts_reach_eight_only_after_every_slice():
    """Eight value slices announce their steps; a chunk's count (chunk = last - step) reaches 8,
    bwd_dkw's condition, only once every slice has announced that step, each after its own stores."""
    n = 11
    counts = [0] * n
    for done, steps in enumerate(replay(n) for _ in range(8)):
        assert max(counts) <= done
        for step in steps:
            counts[n - 1 - step] += 1
    assert counts == [8] * n


@pytest.mark.skipif(not (LIB.exists() and OBJDUMP.exists()), reason="needs the built library and llvm-objdump")
@pytest.mark.parametrize("kernel", ["bwd_scan_kernelIDF16bLb1ELb0EE", "bwd_scan_kernelIDF16_Lb1ELb0EE"])
def test_the_built_kernel_keeps_its_windows(kernel, tmp_path):
    ws = windows(kernel, str(tmp_path))
    full = [i for i, w in enumerate(ws) if i and w.count("load") >= 6 and ws[i - 1].count("load") >= 4
            and w[-1] == ("wait", LIMIT)]
    assert len(full) == 2 * DEPTH  # the peeled round, then the loop
    for i in full:
        first, second = ws[i - 1], ws[i]
        assert first.count("load") >= 4 and first.count("store") == 1, first
        assert second.count("load") >= 6 and second.count("store") == 1, second
    # announcements: after the barrier behind the wait of the peeled round's last step and of every step of the loop
    atomics = [i for i, w in enumerate(ws) if i and "atomic" in w]
    assert [i + 1 for i in full[DEPTH - 1:]] == atomics[:DEPTH + 1]
    # the rest once nothing is in flight
    assert ("wait", 0) in [w[-1] for w in ws if w]
