"""The distances between matrix and vector instructions that the streaming prefill loop keeps by construction (csrc/gen_prefill_stream.py,
check_distances), in the text of every form, and that the check sees an instruction that is moved too close (no GPU)."""

import importlib.util
import pathlib

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "tt-xla_amd" / "csrc"
_spec = importlib.util.spec_from_file_location("gen_prefill_stream", CSRC / "gen_prefill_stream.py")
G = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(G)


@pytest.mark.parametrize("form", G.FORMS, ids=lambda f: f.name)
def test_distances(form):
    lines = G.generate(form)
    assert G.check_distances(form, lines) == (2, {64: 5, 128: 12 if form.wide else 10, 256: 19}[form.d])
    # the first vector instruction of an iteration that reads its scores, put in front of the matrix instruction before it
    top = lines.index("L_it1%=:")
    reads = next(i for i in range(top, len(lines)) if lines[i].startswith("v_fma_f32") and f"v{form.S[1]}," in lines[i])
    moved = lines.copy()
    moved.insert(next(i for i in range(top, reads) if lines[i].startswith("v_mfma")), moved.pop(reads))
    with pytest.raises(AssertionError):
        G.check_distances(form, moved)
    # a probability written behind the matrix instruction that reads it
    reader = next(i for i in range(top, len(lines)) if lines[i].startswith("v_mfma") and G.vr(form.P[0], 4) in lines[i])
    moved = lines.copy()
    moved.insert(reader + 1, f"v_cvt_pk_bf16_f32 v{form.P[0]}, v{form.T[0]}, v{form.T[1]}")
    with pytest.raises(AssertionError):
        G.check_distances(form, moved)
