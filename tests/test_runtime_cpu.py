"""The copies of matrices that decode steps read (`Runtime.tile_for_decode`): asked for while a model is built, made
when it is whole, the ones every step reads first, within half of the memory that is free then."""
import contextlib

import torch

from fllm_amd.parts.runtime import PIECE, Runtime


class Matrix:
    """Stands for a matrix on the device: the runtime asks only where it is and how large."""
    is_cuda = True

    def __init__(self, name, mib):
        self.name, self.mib = name, mib

    def numel(self):
        return self.mib << 19

    def element_size(self):
        return 2


class Library:
    def __init__(self):
        self.made = []

    def tile_for_decode(self, w, gate_up=False):
        self.made.append((w.name, gate_up))
        return True


def build(rt):
    rt.collect_tile_requests()
    for layer in range(3):
        rt.tile_for_decode(Matrix(f"o{layer}", 32))
        rt.tile_for_decode(Matrix(f"qkv{layer}", 48), priority=1)
        rt.tile_for_decode(Matrix(f"down{layer}", 112))
        rt.tile_for_decode(Matrix(f"gate_up{layer}", 224), gate_up=True, priority=1)
    return rt.tiles_for_model()


def test_copies_are_made_by_priority_within_half_of_the_free_memory(monkeypatch):
    every = [(f"{kind}{layer}", False) for layer in range(3) for kind in ("o", "down")] + \
            [(f"{kind}{layer}", kind == "gate_up") for layer in range(3) for kind in ("qkv", "gate_up")]
    for free_mib, want in ((1 << 20, every),                       # plenty: all twelve, the first kind first
                           (2 * (3 * 144 + 48 + 224 + 48 + 10), every[:6] + [("qkv0", False), ("gate_up0", True), ("qkv1", False)]),
                           (2 * 300, [("o0", False), ("down0", False), ("o1", False), ("down1", False)]),
                           (2 * 40, [("o0", False)])):
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (free_mib << 20, 1 << 40))
        lib = Library()
        made = build(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles="auto"))
        assert lib.made == want, (free_mib, lib.made)
        assert made == sum(m << 20 for m in (dict(o=32, qkv=48, down=112, gate_up=224)[n.rstrip("012")] for n, _ in want))
    # switched on: no budget; switched off, or another precision: nothing
    lib = Library()
    build(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles=True))
    assert lib.made == every
    for rt in (Runtime(torch.device("cpu"), torch.bfloat16, Library(), 128, decode_weight_tiles=False),
               Runtime(torch.device("cpu"), torch.float32, Library(), 128)):
        assert build(rt) == 0 and rt.ops.made == []


def test_outside_a_model_a_copy_is_made_at_once(monkeypatch):
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (100 << 20, 1 << 40))
    lib = Library()
    rt = Runtime(torch.device("cpu"), torch.bfloat16, lib, 128)
    rt.tile_for_decode(Matrix("small", 4))
    rt.tile_for_decode(Matrix("large", 16))             # more than a twentieth of what is free
    rt.tile_for_decode(Matrix("pair", 2), gate_up=True)
    assert lib.made == [("small", False), ("pair", True)]


class LibraryWithExperts(Library):
    def tile_experts_supported(self, w):
        return not w.name.startswith("odd")

    def tile_experts(self, w):
        self.made.append(w.name)
        return True


def build_routed(rt, layers=3, kind=""):
    rt.collect_tile_requests()
    for layer in range(layers):
        rt.tile_experts(Matrix(f"up{layer}", 200), Matrix(f"{kind}down{layer}", 100))
        rt.tile_for_decode(Matrix(f"o{layer}", 32))
        rt.tile_for_decode(Matrix(f"qkv{layer}", 48), priority=1)
    rt.tile_for_decode(Matrix("vocabulary", 300), priority=2)
    return rt.tiles_for_model()


def test_experts_copies_come_last_in_pairs_and_within_an_eighth(monkeypatch):
    dense = [(f"{kind}{layer}", False) for kind in ("o", "qkv") for layer in range(3)] + [("vocabulary", False)]       # 540 MiB
    pairs = [name for layer in range(3) for name in (f"up{layer}", f"down{layer}")]                                    # 300 MiB a layer
    for free_mib, want in ((1 << 20, dense + pairs),
                           (8 * 650, dense + pairs[:4]),            # an eighth holds two layers' pairs
                           (8 * 290, dense),                        # and not one, though a single stack would fit
                           (2 * 560, dense),                        # what every step reads is not pushed out
                           (2 * 100, [("o0", False), ("o1", False), ("o2", False)])):
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (free_mib << 20, 1 << 40))
        lib = LibraryWithExperts()
        made = build_routed(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles="auto"))
        assert lib.made == want, (free_mib, lib.made)
        assert made == sum((540 if want[:7] == dense else 32 * len(want), 300 * sum(n in ("up0", "up1", "up2") for n in want))) << 20
    lib = LibraryWithExperts()
    build_routed(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles=True))
    assert lib.made == dense + pairs
    lib = LibraryWithExperts()                                      # a stack that has no copy: neither has the other
    build_routed(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles=True), kind="odd")
    assert lib.made == dense
    lib = LibraryWithExperts()                                      # outside of a model: at once, within a twentieth together
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (100 << 20, 1 << 40))
    rt = Runtime(torch.device("cpu"), torch.bfloat16, lib, 128)
    rt.tile_experts(Matrix("a", 3), Matrix("b", 3))
    rt.tile_experts(Matrix("c", 3), Matrix("d", 2))
    assert lib.made == ["c", "d"]


class LibraryWithPieces(LibraryWithExperts):
    """Counts the memory of copies: what is made inside `copies_together` lies in that piece as long as it has room."""

    def __init__(self, free=None):
        super().__init__()
        self.pieces, self.allocated, self.left, self.free, self.held = [], 0, 0, free, set()

    @contextlib.contextmanager
    def copies_together(self, nbytes):
        self.pieces.append(nbytes)
        self.left = nbytes if self._allocate(nbytes) else 0
        yield
        self.left = 0

    def _allocate(self, nbytes):
        fits = self.free is None or self.allocated + nbytes <= self.free
        self.allocated += nbytes if fits else 0
        return fits

    def _copy(self, w):
        size = w.mib << 20
        if size <= self.left:
            self.left -= size
        elif not self._allocate(size):
            raise torch.cuda.OutOfMemoryError("no room")
        self.held.add(w.name)
        return True

    def tile_for_decode(self, w, gate_up=False):
        return self._copy(w)

    def tile_experts(self, w):
        return self._copy(w)

    def forget_copy(self, w):
        self.held.discard(w.name)


def alternating(rt, layers=6):
    """Matrices of 50 and 235 MiB in turn, the vocabulary's, and a few small ones."""
    rt.collect_tile_requests()
    for layer in range(layers):
        rt.tile_for_decode(Matrix(f"qkv{layer}", 50), priority=1)
        rt.tile_for_decode(Matrix(f"gate_up{layer}", 235), gate_up=True, priority=1)
        rt.tile_for_decode(Matrix(f"o{layer}", 8))
    rt.tile_for_decode(Matrix("vocabulary", 1002), priority=2)
    return rt.tiles_for_model()


def test_copies_take_the_memory_that_the_budget_counts(monkeypatch):
    """Whatever the sizes and whatever is left out: the pieces hold what is made and nothing else, none beyond PIECE."""
    for free_mib, want in ((1 << 20, 6 * 293 + 1002), (2 * 700, 48 + 50 + 235 + 50 + 235 + 50), (2 * 60, 48), (300, 48 + 50 + 50), (2 * 20, 16)):
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (free_mib << 20, 1 << 40))
        lib = LibraryWithPieces()
        made = alternating(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles="auto"))
        assert lib.allocated == sum(lib.pieces) == made == want << 20, (free_mib, lib.pieces)
        assert made <= free_mib << 19
        assert all(p <= PIECE for p in lib.pieces)
    assert len(lib.pieces) == 1                              # small ones share one
    lib = LibraryWithPieces()
    build_routed(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles=True))
    assert lib.allocated == (540 + 900) << 20


def test_a_copy_without_memory_is_left_out(monkeypatch):
    """More was said to be free than there is: under "auto" the model is built with the copies there was room for, a pair of experts' stacks
    whole or not at all; where copies were asked for outright the error stands."""
    import pytest
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (1 << 40, 1 << 40))
    lib = LibraryWithPieces(free=500 << 20)
    made = alternating(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles="auto"))
    assert 0 < made == sum(dict(o=8, qkv=50, gate_up=235)[n[:-1]] for n in lib.held) << 20 and lib.allocated <= lib.free
    lib = LibraryWithPieces(free=(540 + 250) << 20)
    build_routed(Runtime(torch.device("cpu"), torch.bfloat16, lib, 128, decode_weight_tiles="auto"))
    assert not any(n.startswith(("up", "down")) for n in lib.held)
    with pytest.raises(torch.cuda.OutOfMemoryError):
        alternating(Runtime(torch.device("cpu"), torch.bfloat16, LibraryWithPieces(free=500 << 20), 128, decode_weight_tiles=True))
