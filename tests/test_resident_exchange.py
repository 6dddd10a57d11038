"""CPU model of the exchange of k_trd_wide (quack_amd/csrc/qk_trdres.hip): G workgroups that
meet once a column through two alternating buffers of words tagged with the column.

One step of a workgroup is one access in the kernel's order: publish row c-1 (its owner),
publish its y, store V's column c-1 (its owner), read everything of column c.  A
workgroup is held up at every one of its steps in turn while the others go as far as they
can; then it goes on.  Nobody may be left waiting for words that were overwritten, and every
reflector has to be stored once."""
import pytest


def program(n, G, g, leave):
    """The accesses of workgroup g: (kind, column).  leave: it goes after its last rows' y;
    else it stays to column 1 and stores V's column c-1 at c = g (mod G)."""
    last = 1 if g == 0 or not leave else g + 1
    for c in range(n - 1, last - 1, -1):
        if g == (c - 1) % G:
            yield "row", c
        if g < c:
            yield "y", c
        if g == ((c - 1) if leave else c) % G:
            yield "store", c
        if leave and g > 0 and c == last:
            return
        yield "read", c


class Run:
    def __init__(self, n, G, leave):
        self.n, self.G = n, G
        self.prog = [list(program(n, G, g, leave)) for g in range(G)]
        self.pc = [0] * G
        self.y = [[None] * n, [None] * n]  # tag of row r's y, by column parity
        self.row = [None, None]
        self.stored = []

    def step(self, g):
        """One access of workgroup g; False if it has to wait or is done."""
        if self.pc[g] == len(self.prog[g]):
            return False
        kind, c = self.prog[g][self.pc[g]]
        if kind == "read":
            if self.row[c & 1] != c or any(t != c for t in self.y[c & 1][:c]):
                return False
        elif kind == "row":
            self.row[c & 1] = c
        elif kind == "y":
            for r in range(g, c, self.G):
                self.y[c & 1][r] = c
        else:
            self.stored.append(c - 1)
        self.pc[g] += 1
        return True

    def go(self, groups):
        moved = True
        while moved:
            moved = False
            for g in groups:
                while self.step(g):
                    moved = True

    def stuck(self):
        return [g for g in range(self.G) if self.pc[g] < len(self.prog[g])]


def stuck_cases(n, G, leave):
    bad = []
    for slow in range(G):
        for at in range(len(Run(n, G, leave).prog[slow])):
            r = Run(n, G, leave)
            others = [g for g in range(G) if g != slow]
            while r.pc[slow] < at and (r.step(slow) or any([r.step(g) for g in others])):
                pass
            r.go(others)  # the slow one is held up here
            r.go(range(G))
            if r.stuck():
                bad.append((slow, at))
            else:
                assert sorted(r.stored) == list(range(n - 1))
    return bad


@pytest.mark.parametrize("n,G", [(17, 2), (24, 3), (40, 5), (64, 8), (61, 8)])
def test_every_delay_ends(n, G):
    assert stuck_cases(n, G, leave=True) == []


def test_the_model_sees_the_fault():
    """A workgroup that stays without a row is nobody's to wait for."""
    assert stuck_cases(64, 8, leave=False)
