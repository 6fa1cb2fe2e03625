"""Latent prompts on either side of the lines between which their expansion takes 64 latent values per step (more than 256 workgroups, 480, 800): both layouts of
either weight, activations as slices, a last tile of one row block; one call against the operators in turn, as test_gpu_latent_prompt.py
has it."""

import pytest

import test_gpu_latent_prompt as L

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    L.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("joint,slices", [(None, False), ("latent first", True), ("heads first", False)])
@pytest.mark.parametrize("n,users,s", [
    (64, 1, 256), (65, 1, 256), (119, 1, 256), (120, 1, 256),  # 256 workgroups, 260, 476, 480
    (96, 1, 256), (95, 1, 256), (64, 3, 96), (64, 2, 160),  # 384 workgroups, 380, 384, 384
    (100, 1, 480), (99, 1, 512), (64, 7, 160), (128, 1, 512),  # 800 workgroups, 792, 1152, 1024
])
def test_either_step(n, users, s, joint, slices):
    L.test_one_call_equals_the_operators(n, users, s, 32, joint, slices)
