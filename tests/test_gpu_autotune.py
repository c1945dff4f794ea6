"""What the autotuner chooses among: 2D chains in LDS run on bits with a plan of their own,
so it leaves their lds_block alone; schedules saved for other kernels do not reach chains
on bits; the lines that the sizes give are among the candidates."""
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


@pytest.mark.parametrize("J2,colours", [(0.0, 2), (-0.02, 4)])
def test_saved_schedule_of_the_byte_kernels(J2, colours, tmp_path, monkeypatch):
    """A file from a run that tuned the kernels on bytes (64 lines a band)."""
    f = tmp_path / "tuned"
    f.write_text(f"hbm:2:{colours}:18:2 256 1 1 0.5 64 0\n")
    monkeypatch.setenv("MCG_TUNE_CACHE", str(f))
    print("autotune saved", J2, flush=True)
    with M.Run([dict(shape=(512, 512), temperature=1500.0, seed=i) for i in range(3)],
               mode=M.MODE_CHECKERBOARD, J1=0.1, J2=J2) as r:
        chosen = r.autotune(16)
        assert chosen["band_lines"] != 64 and chosen["trial_ms"] != 0.5
        assert len(f.read_text().splitlines()) == 2  # the new one is saved beside it


def test_saved_schedule_of_the_path_is_used(tmp_path, monkeypatch):
    f = tmp_path / "tuned"
    f.write_text("hbm:2:2:20:1 256 2 8 0.25 0 0\n")
    monkeypatch.setenv("MCG_TUNE_CACHE", str(f))
    print("autotune saved, bytes", flush=True)
    with M.Run([dict(shape=(1000, 1000), temperature=1500.0, seed=i) for i in range(2)],
               mode=M.MODE_CHECKERBOARD, J1=0.1) as r:
        chosen = r.autotune(16)
        assert (chosen["units_per_thread"], chosen["graph_passes"], chosen["trial_ms"]) == (2, 8, 0.25)
