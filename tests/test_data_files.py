"""Hidden-state files: what the header says about a tensor's bytes is checked before they are read (no GPU needed)."""

import json

import pytest
import torch


def _write(path, hs_bytes=None, id_bytes=None, cut=0):
    """Two tensors of ``[4, 4, 8]`` bf16 and ``[4]`` int64; ``hs_bytes`` / ``id_bytes``: lengths the header states instead
    of the shapes' own (the file holds what the shapes ask for)."""
    hs, ids = torch.arange(128).bfloat16().view(4, 4, 8), torch.arange(4) + 1
    hs_len, id_len = 256 if hs_bytes is None else hs_bytes, 32 if id_bytes is None else id_bytes
    header = {"hidden_states": {"dtype": "BF16", "shape": [4, 4, 8], "data_offsets": [0, hs_len]},
              "token_ids": {"dtype": "I64", "shape": [4], "data_offsets": [hs_len, hs_len + id_len]}}
    text = json.dumps(header).encode()
    raw = (len(text).to_bytes(8, "little") + text + hs.view(torch.int16).numpy().tobytes() + ids.numpy().tobytes()
           + bytes(256))
    path.write_bytes(raw[:len(raw) - 256 - cut])
    return hs, ids


def test_offsets_point_at_the_tensors(tmp_path):
    from speculators_amd.data import HiddenStatesFile

    hs, ids = _write(tmp_path / "a.safetensors")
    f = HiddenStatesFile(tmp_path / "a.safetensors")
    raw = (tmp_path / "a.safetensors").read_bytes()
    assert raw[f.data_offset("token_ids"):] == ids.numpy().tobytes()
    assert raw[f.data_offset("hidden_states"):f.data_offset("token_ids")] == hs.view(torch.int16).numpy().tobytes()
    assert torch.equal(f.load()["hidden_states"], hs)


@pytest.mark.parametrize("lengths,name", [((192, 32), "hidden_states"), ((264, 32), "hidden_states"),
                                          ((256, 24), "token_ids"), ((256, 40), "token_ids"), ((256, -8), "token_ids")])
def test_a_byte_length_that_is_not_the_shapes_is_an_error(tmp_path, lengths, name):
    from speculators_amd.data import HiddenStatesFile

    _write(tmp_path / "a.safetensors", *lengths)
    f = HiddenStatesFile(tmp_path / "a.safetensors")
    with pytest.raises(ValueError, match=name):
        f.load()
    with pytest.raises(ValueError, match=name):
        f.data_offset(name)
