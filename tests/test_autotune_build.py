"""A tuning choice counts for the library build that it was timed with: the
same build finds it again, another build times its own candidates."""
from types import SimpleNamespace

import torch

from torch_de_solver_amd import autotune, mat_engine, native, nn_engine


class _Engine:
    def __init__(self, *args, **kwargs):
        pass

    def train_step(self, *args):
        pass

    backward = train_step


def test_choices_belong_to_a_build(tmp_path, monkeypatch):
    timed = []

    def time_ms(fn, reps):
        timed.append(1)
        return 1.0 + (len(timed) % 3)

    monkeypatch.setenv('TDX_TUNE_CACHE', str(tmp_path / 'tuning.json'))
    monkeypatch.setattr(nn_engine, 'NNEngine', _Engine)
    monkeypatch.setattr(mat_engine, 'MatEngine', _Engine)
    monkeypatch.setattr(autotune, '_time_ms', time_ms)
    nn = [SimpleNamespace(groups=[SimpleNamespace(n_entries=10, slot_base=[0, 1])])]
    arch = SimpleNamespace(d_in=2, width=32, n_layers=4, n_out=1)
    mat = SimpleNamespace(shape=(64, 64), n_eq=1, dp=2, dtype=torch.float32, equations=[])

    def tune():
        return (autotune.tune_nn(nn, arch, 'cpu', torch.zeros(4)),
                autotune.tune_mat(mat, 'cpu', torch.zeros(1, 64, 64)))

    builds = []
    for name in ('first', 'second'):
        lib = tmp_path / (name + '.so')
        lib.write_bytes(name.encode())
        builds.append(str(lib))
    monkeypatch.setattr(native, 'LIB_PATH', builds[0])
    first = tune()
    assert [r['cached'] for _, r in first] == [False, False]
    again = tune()
    assert [r['cached'] for _, r in again] == [True, True]
    assert [c for c, _ in again] == [c for c, _ in first]
    monkeypatch.setattr(native, 'LIB_PATH', builds[1])
    n = len(timed)
    assert [r['cached'] for _, r in tune()] == [False, False]
    assert len(timed) == n + len(autotune.NN_CHUNK_CANDIDATES) + len(autotune.MAT_ROW_CANDIDATES)
    monkeypatch.setattr(native, 'LIB_PATH', builds[0])
    assert [r['cached'] for _, r in tune()] == [True, True]
