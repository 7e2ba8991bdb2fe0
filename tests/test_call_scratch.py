"""CPU: the scratch that the router's and the many-token MLP's launches hand each other belongs to one call.  Two host
threads may interleave their launches on one stream, and a captured call keeps its scratch's address for every replay, so
a buffer kept for the next call would be written by both."""
import pytest
import torch


class _Lib:
    """Stands for the library: notes the scratch of every call, and has a second call arrive within the first."""

    def __init__(self, name, scratch_arg):
        self.name, self.arg, self.seen, self.again = name, scratch_arg, [], None

    def __getattr__(self, attr):
        if attr == self.name:
            return self._call
        if attr == self.name + "_workspace":
            return lambda *a: 1 << 16
        raise AttributeError(attr)

    def _call(self, *args):
        self.seen.append(args[self.arg])
        if self.again is not None:
            again, self.again = self.again, None
            again()
        return 0


class _Kept:
    """Stands for the kept workspaces: one buffer per purpose."""

    def __init__(self):
        self.ws = {}

    def get(self, purpose, nbytes):
        return self.ws.setdefault(purpose, torch.zeros(nbytes, dtype=torch.uint8))


@pytest.fixture
def stand_in(pkg, monkeypatch):
    def use(name, scratch_arg):
        fake = _Lib(name, scratch_arg)
        monkeypatch.setattr(pkg.resident, "lib", lambda: fake)
        monkeypatch.setattr(pkg.resident, "_stream", lambda: 0)
        monkeypatch.setattr(pkg.resident, "WORKSPACES", _Kept())
        return fake
    return use


def _own_scratch(fake, call):
    fake.again = call
    call()
    assert len(fake.seen) == 2 and fake.seen[0] != fake.seen[1]


def test_route(pkg, stand_in):
    fake = stand_in("mi_moe_route", 11)
    x, rw = torch.zeros((3, 64), dtype=torch.bfloat16), torch.zeros((64, 8))
    _own_scratch(fake, lambda: pkg.route(x, rw, None, 2))


def test_many_token_mlp(pkg, stand_in):
    fake = stand_in("mi_mlp_many", 15)
    D, I = 256, 256
    x = torch.zeros((33, D), dtype=torch.bfloat16)
    leaves = [pkg.bf16_leaf(torch.zeros(s, dtype=torch.bfloat16), device="cpu") for s in ((D, I), (D, I), (I, D))]
    _own_scratch(fake, lambda: pkg.bf16_mlp(x, *leaves, 7.0))
