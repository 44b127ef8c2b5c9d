"""The package is two compiled files: what uses them builds the one that is missing, and an
extension of another torch is not used."""
import sys
import types

import pytest

from qmoe_amd import _lib, build


@pytest.mark.parametrize('library,extension,built', [
    (True, True, []), (False, True, ['library']), (True, False, ['extension']), (False, False, ['library'])])
def test_what_is_missing_is_built_and_no_more(library, extension, built, tmp_path, monkeypatch):
    done = []
    monkeypatch.setattr(build, 'build_library', lambda: done.append('library'))     # (which builds both)
    monkeypatch.setattr(build, 'build_tensor_args', lambda: done.append('extension'))
    if not library:
        monkeypatch.setattr(build, 'LIB_PATH', str(tmp_path / 'library.so'))
    if not extension:
        monkeypatch.setattr(build, 'TENSOR_ARGS_PATH', str(tmp_path / 'extension.so'))
    build.build_what_is_missing()
    assert done == built


def test_an_extension_of_another_torch_is_built_again_and_not_loaded(monkeypatch):
    import torch
    import qmoe_amd
    assert build.tensor_args_fit() and _lib.tensor_args().built_against == build.torch_mark()
    monkeypatch.setattr(torch, '__version__', torch.__version__ + '.1')
    assert not build.tensor_args_fit()
    monkeypatch.setattr(torch, '__version__', torch.__version__[:-3])       # the beginning of the real one
    assert not build.tensor_args_fit()
    monkeypatch.undo()
    for other in (types.ModuleType('of no torch'), types.ModuleType('of another')):
        if other.__name__ == 'of another':
            other.built_against = 'qmoe_amd, built against torch 1.0'
        monkeypatch.setattr(_lib, '_tensor_args', None)
        monkeypatch.setitem(sys.modules, 'qmoe_amd._tensor_args', other)
        monkeypatch.setattr(qmoe_amd, '_tensor_args', other, raising=False)
        with pytest.raises(ImportError, match='of another torch'):
            _lib.tensor_args()


def test_a_kernels_limit_of_lds_is_the_same_for_all_its_launches():
    """Set to what a launch has, it can be another thread's by the time of that launch: it goes
    through a function that takes a constant."""
    import glob
    import os
    uses = {}
    for path in glob.glob(os.path.join(build.HERE, 'csrc', '*')):
        with open(path) as f:
            text = f.read()
        uses[os.path.basename(path)] = text.count('hipFuncSetAttribute'), text.count('allow_lds<')
    assert {name: n for name, (n, _) in uses.items() if n} == {'sub1_common.h': 1}
    assert uses['sub1_prepared.hip'][1] and uses['sub1_kernels.hip'][1]
