"""What the autotuner chooses among: 2D chains in LDS run on bits with a plan of their own,
so it leaves their lds_block alone; the lines that the sizes give are among the
candidates."""
import pytest

import casmcode_monte_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge,block", [(24, 512), (60, 1024), (122, 256), (25, 1024),
                                        (123, 512)])
def test_block_of_chains_on_words_is_left(edge, block):
    print("autotune words", edge, block, flush=True)
    with M.Run([dict(shape=(edge, edge), temperature=1500.0, seed=i) for i in range(5)],
               mode=M.MODE_CHECKERBOARD, J1=0.1) as r:
        r.set_schedule(lds_block=block)
        chosen = r.autotune(16)
        assert chosen["lds_block"] == block and r.schedule()["lds_block"] == block
        assert chosen["trial_ms"] > 0.0
