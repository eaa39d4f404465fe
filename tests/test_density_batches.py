"""density(): its squares are taken in batches where memory allows and one by one where it does
not, with the same terms in the same order.  The tree calls are replaced by a stand-in that holds
a set number of trees, so no GPU is needed."""
import pytest


class _Device:
    """Trees as tuples of the orbitals summed; a call that would exceed `room` live trees fails."""

    def __init__(self, room):
        self.room, self.live, self.largest = room, 0, 0

    def attach(self, monkeypatch, X):
        dev = self

        class Tree:
            def __init__(self, mra):
                self.terms, self.held = (), False

            def make(self, terms):
                if dev.live == dev.room:
                    raise X.M.MwgError("device allocation failed")
                dev.live += 1
                self.terms, self.held = terms, True

            def __del__(self):
                dev.live -= self.held

        def multiply_batch(prec, outs, coefs, as_, bs):
            dev.largest = max(dev.largest, len(outs))
            for o, c, a, b in zip(outs, coefs, as_, bs):
                assert a is b
                if a == "empty":
                    raise X.M.MwgError("empty input tree")
                o.make(((c, a),))
            return outs

        def add_batch(outs, sums):
            for o, terms in zip(outs, sums):
                assert all(c == 1.0 for c, _ in terms)
                o.make(sum((t.terms for _, t in terms), ()))
            return outs

        for name, f in (("FunctionTree", Tree), ("multiply_batch", multiply_batch), ("add_batch", add_batch)):
            monkeypatch.setattr(X.M, name, f)


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 70])
@pytest.mark.parametrize("room", [3, 10, 32, 33, 34, 1000])
def test_every_square_once_whatever_fits(monkeypatch, n, room):
    from mrchem_amd import mrchem as X
    dev = _Device(room)
    dev.attach(monkeypatch, X)
    Phi = [X.Orbital("phi%d" % i, 1.0 + i, "p") for i in range(n)]
    rho = X.density(1e-4, Phi, None)
    assert rho.terms == tuple((p.occ, p.tree) for p in Phi)
    assert dev.largest == min(n, X.DENSITY_BATCH)
    del rho
    assert dev.live == 0


def test_other_errors_stay():
    from mrchem_amd import mrchem as X
    with pytest.MonkeyPatch.context() as mp:
        _Device(1000).attach(mp, X)
        with pytest.raises(X.M.MwgError, match="empty"):
            X.density(1e-4, [X.Orbital("a", 2.0, "p"), X.Orbital("empty", 2.0, "p"), X.Orbital("c", 2.0, "p")], None)
        assert X.density(1e-4, [], None) is None
