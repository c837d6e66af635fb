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


@pytest.mark.parametrize("T,base", [(1100, 60), (1500, 300), (2048, 100)])
def test_two_rounds_of_workgroups(kvm, orc, dev, shape, T, base):
    """1025 to 2048 rows, which a session runs on 8-row workgroups where the
    prefix is short: more workgroups than CUs, the heaviest tiles first."""
    run_prefill(kvm, orc, dev, T, base, 1, seed=T)


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


class _ShiftedPool:
    """The launcher on a copy of the pool that starts 8 bytes past a 16-byte
    boundary."""

    def __init__(self, kvm):
        self.kvm, self.KvLayout = kvm, kvm.KvLayout

    def launch_attn_prefill_flash(self, q, T, base, layer, pt, pool, *rest):
        import torch
        buf = torch.zeros(pool.numel() + 8, dtype=pool.dtype, device=pool.device)
        assert buf.data_ptr() % 16 == 0
        buf[4:4 + pool.numel()] = pool
        self.kvm.launch_attn_prefill_flash(q, T, base, layer, pt, buf[4:4 + pool.numel()], *rest)
        torch.cuda.synchronize()


@pytest.mark.parametrize("T,base,S", [(33, 100, 1), (50, 300, 8)])
def test_pool_at_an_8_byte_boundary(kvm, orc, dev, shape, T, base, S):
    """The key sets load K/V rows straight to LDS, 16 bytes a lane; a pool
    without that alignment runs on the tiles, forced or not."""
    run_prefill(_ShiftedPool(kvm), orc, dev, T, base, S, P=64, seed=T)
    kvm.debug_prefill_key_sets(0)
    run_prefill(_ShiftedPool(kvm), orc, dev, T, base, S, P=64, seed=T)
