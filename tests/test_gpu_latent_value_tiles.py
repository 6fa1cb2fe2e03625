"""The value projection of a latent step where a workgroup takes several blocks of 32 users (128 heads: from 33 users on; 40 heads: three
blocks in two workgroups, the last one short) and users around a piece of four rows and a block: the step
against the operators in turn, as test_gpu_latent_step.py has it, for both layouts of the weights."""

import pytest

import test_gpu_latent_step as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    S.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("views", [False, True])
@pytest.mark.parametrize("users,n", [(4, 16), (5, 16), (29, 16), (64, 128), (65, 128), (100, 128), (97, 40), (161, 64)])
def test_several_blocks_of_users(users, n, views):
    S.test_step_equals_operators_in_turn(users, n, 16, 30, views)
