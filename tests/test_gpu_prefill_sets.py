"""Key-set prefill shapes (8- and 4-row workgroups, four key sets) against the
double oracle, at the edges of their tiles, 32-key blocks and splits. Criterion
and input construction as test_gpu_prefill.py."""
import pytest

from test_gpu_prefill import barrier_status_clear, run_prefill  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[8, 4], ids=["rows8", "rows4"])
def shape(kvm, request):
    prev = kvm.debug_prefill_key_sets(request.param)
    yield request.param
    kvm.debug_prefill_key_sets(prev)


@pytest.mark.parametrize("T,base", [(1, 0), (3, 0), (4, 28), (5, 31), (7, 32), (8, 120), (9, 127),
                                    (33, 5), (130, 100), (257, 0)])
def test_tile_and_block_edges(kvm, orc, dev, shape, T, base):
    """Rows around whole tiles, keys around one block, one iteration of all
    sets (128 keys) and sets without a block; 32- and 64-token pages."""
    for P in (32, 64):
        run_prefill(kvm, orc, dev, T, base, 1, P=P, seed=T + base)


@pytest.mark.parametrize("S", [2, 3, 8])
def test_splits(kvm, orc, dev, shape, S):
    """Key splits, some of them without keys (40 keys over 8 splits)."""
    run_prefill(kvm, orc, dev, 6, 34, S, seed=S)
    run_prefill(kvm, orc, dev, 50, 300, S, P=64, seed=S)


@pytest.mark.parametrize("P", [1, 16, 128])
def test_page_sizes(kvm, orc, dev, shape, P):
    """Pages smaller than a block (ids looked up per key) and larger."""
    run_prefill(kvm, orc, dev, 75, 29, 1, P=P, seed=P)


def test_moving_reference(kvm, orc, dev, shape):
    """Keys growing along the context: every set's reference max moves and the
    sets fold states of different references."""
    run_prefill(kvm, orc, dev, 60, 700, 1, P=64, seed=3, kgrow=9.0)


@pytest.mark.parametrize("T,S", [(384, 8), (385, 8), (777, 5), (1024, 1), (1025, 1)])
def test_automatic_choice(kvm, orc, dev, T, S):
    """Either side of the row counts where the automatic choice changes; S is
    the most splits the launch may use."""
    run_prefill(kvm, orc, dev, T, 70, S, P=64, seed=T)
