"""CPU model of the panel kernel's units (panel_tile.h): the ticket order and
the publication by agent-scope stores.

Units: ticket 0 is the diagonal unit 0; then, for each block column c, the
diagonal unit c + 1 (blocks (c + 1, c) and (c + 1, c + 1)) and one unit for each
other block (t, c) below.  Block (t, c) needs L(t, i) and L(c, i) for i < c, and
D_c.  Checked for every small panel: each block of the panel belongs to exactly
one unit, and a unit needs only blocks of units with smaller tickets (so that a
unit waits only on workgroups that have started).

Publication: agent-scope stores travel to the coherence point on their own and
are acknowledged there; `s_waitcnt vmcnt(0)` in every wavefront waits for the
acknowledgements, a barrier follows, and the flag is stored.  Every interleaving
is explored; dropping the wait must lose the property."""
import pytest


def unit_of(ticket, P, R):
    """(t, c, diagonal unit) of a ticket, as the kernel decodes it."""
    if ticket == 0:
        return 0, 0, True
    c, u = 0, ticket - 1
    while c < P - 1 and u >= R - c - 1:
        u -= R - c - 1
        c += 1
    return c + 1 + u, c, u == 0 and c < P - 1


def units(P, R):
    return (P - 1) * (R - 1) - (P - 1) * (P - 2) // 2 + 1 + R - P


@pytest.mark.parametrize("P", range(1, 9))
def test_units_cover_the_panel_in_dependency_order(P):
    for R in list(range(P, P + 6)) + [40]:
        made = {}  # block -> ticket; ("D", c) for the inverse
        for ticket in range(units(P, R)):
            t, c, diag = unit_of(ticket, P, R)
            assert c < P and t < R
            blocks = [(t, t)] if ticket == 0 else [(t, c), (t, t)] if diag else [(t, c)]
            needs = [("D", c)] if ticket else []
            if ticket:
                needs += [(t, i) for i in range(c)] + [(c, i) for i in range(c)]
            for b in needs:
                assert b in made, (P, R, ticket, b)  # a smaller ticket's
            for b in blocks:
                assert b not in made
                made[b] = ticket
                if b[0] == b[1]:
                    made[("D", b[0])] = ticket
        want = {(t, c) for c in range(P) for t in range(c, R)} | {("D", c) for c in range(P)}
        assert set(made) == want


def outcomes(wait):
    """What a reader that saw the flag can read of two published words."""
    program = ["store0", "store1"] + (["wait"] if wait else []) + ["flag"]
    start = (0, frozenset(), (0, 0), 0, False)
    seen, stack, result = {start}, [start], set()
    while stack:
        pc, flying, memory, flag, flag_flying = stack.pop()
        if flag:
            result.add(memory)
        nxt = []
        if pc < len(program):
            op = program[pc]
            if op == "flag":
                nxt.append((pc + 1, flying, memory, flag, True))
            elif op != "wait":
                nxt.append((pc + 1, flying | {int(op[-1])}, memory, flag, flag_flying))
            elif not flying:
                nxt.append((pc + 1, flying, memory, flag, flag_flying))
        for w in flying:  # a store reaches the coherence point and is acknowledged
            nxt.append((pc, flying - {w}, tuple(1 if i == w else m for i, m in enumerate(memory)), flag, flag_flying))
        if flag_flying:
            nxt.append((pc, flying, memory, 1, False))
        for s in nxt:
            if s not in seen:
                seen.add(s)
                stack.append(s)
    return result


def test_publication_by_agent_scope_stores():
    assert outcomes(wait=True) == {(1, 1)}
    assert (0, 0) in outcomes(wait=False)
