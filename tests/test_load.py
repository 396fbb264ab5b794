"""Loading a layer without a GPU: what ``load_mlp_weights`` does around its conversions, with the
conversion and its check replaced by stand-ins."""
import weakref

import pytest
import torch

I, H = 512, 256


class _Source(torch.Tensor):
    """A checkpoint tensor whose device copy is a tensor of this process, kept in ``copies`` weakly."""

    copies = []

    def to(self, *args, **kwargs):
        t = torch.zeros(tuple(self.shape), dtype=torch.bfloat16)
        _Source.copies.append(weakref.ref(t))
        return t


class _Checkpoint(dict):
    """Makes a tensor at each access and keeps none, like a lazily read checkpoint."""

    def __getitem__(self, name):
        return torch.zeros(super().__getitem__(name)).as_subclass(_Source)


def _checkpoint():
    return _Checkpoint({"gate_proj.weight": (I, H), "up_proj.weight": (I, H), "down_proj.weight": (H, I)})


@pytest.fixture
def stand_ins(pkg, monkeypatch):
    from qwen_mlp_amd import mlp

    def begin(w, fmt, stream):
        return mlp.PackedWeight(torch.zeros(0, dtype=torch.uint8), *w.shape, fmt)

    monkeypatch.setattr(_Source, "copies", [])
    monkeypatch.setattr(mlp, "_pack_weight_begin", begin)
    monkeypatch.setattr(mlp, "_pack_weight_end", lambda pw, strict, stream: pw)
    return mlp


def test_sources_outlive_their_conversions(stand_ins, monkeypatch):
    """A matrix's bf16 source lives until the check that waits for its conversion: dropped before,
    memory that belongs to another stream could be handed out again while the conversion reads it."""
    mlp = stand_ins
    alive = []

    def end(pw, strict, stream):
        alive.append(_Source.copies[len(alive)]() is not None)
        return pw

    monkeypatch.setattr(mlp, "_pack_weight_end", end)
    mlp.load_mlp_weights("cuda", _checkpoint())
    assert alive == [True, True, True]


def test_a_later_failure_keeps_what_came_before(stand_ins, monkeypatch, tmp_path):
    """Matrices load in the order gate, down, up: where a later one is missing, those before it
    have been checked and cached, and where one of those is refused, that is the error."""
    mlp = stand_ins
    from qwen_mlp_amd import weight_cache

    saved = []
    monkeypatch.setattr(weight_cache, "save", lambda path, pw: saved.append((pw.rows, pw.cols)))
    sd = _checkpoint()
    del sd["up_proj.weight"]
    with pytest.raises(KeyError, match="up_proj"):
        mlp.load_mlp_weights("cuda", sd, tensor_cache_path=str(tmp_path))
    assert saved == [(I, H), (H, I)]

    def end(pw, strict, stream):
        raise ValueError("non-finite")

    monkeypatch.setattr(mlp, "_pack_weight_end", end)
    with pytest.raises(ValueError, match="non-finite"):
        mlp.load_mlp_weights("cuda", sd, tensor_cache_path=str(tmp_path))


def test_pool_refuses_a_device_that_is_not_a_gpu(pkg, monkeypatch):
    """Also where the current GPU's stream already holds a workspace."""
    from qwen_mlp_amd import _lib

    pool = pkg.WorkspacePool()
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(_lib, "raw_stream", lambda index=None: 0)
    pool._ws[pool._key("cuda", None)] = torch.zeros(64, dtype=torch.uint8)
    assert pool.reserve(64, "cuda:0").numel() == 64
    with pytest.raises(ValueError, match="cpu"):
        pool.reserve(64, "cpu")
