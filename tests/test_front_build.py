"""The build of the torch front end, without compiling: the C library needs
neither torch nor a host compiler, an older front end never stays beside a
newer library, and attention.py loads a front end only beside the library, for
the torch and Python, that it was built for."""
import json
import sys

import pytest

from redshift_amd import attention as A
from redshift_amd import build as B


@pytest.fixture
def tree(tmp_path, monkeypatch):
    """build() with stand-ins for the compilers, into an empty folder that
    holds an older build's front end."""
    lib = tmp_path / 'lib'
    lib.mkdir()
    for name in ('LIBRARY', 'PROBE_LIBRARY', 'FRONT_LIBRARY', 'BUILD_INFO'):
        monkeypatch.setattr(B, name, lib / getattr(B, name).name)
    monkeypatch.setattr(A, 'FRONT_LIBRARY', B.FRONT_LIBRARY)
    monkeypatch.setattr(A, 'BUILD_INFO', B.BUILD_INFO)
    monkeypatch.setattr(A, 'DEFAULT_LIBRARY', B.LIBRARY)
    monkeypatch.setattr(A, '_FRONT', None)
    monkeypatch.setattr(B, '_compile_all', lambda objdir, sources, extra, jobs: [(n, '') for n, _ in sources])

    def run(cmd):
        out = cmd[cmd.index('-o') + 1]
        with open(out, 'w') as f:
            f.write(f'built as {out}')
        return ''
    monkeypatch.setattr(B, '_run', run)
    monkeypatch.setattr(B, 'hipcc', lambda: 'hipcc')
    B.FRONT_LIBRARY.write_text('an older front end')
    return lib


def test_the_library_builds_without_torch(tree, monkeypatch, capsys):
    monkeypatch.setitem(sys.modules, 'torch', None)   # import torch raises ImportError
    assert B.build() == B.LIBRARY
    assert B.LIBRARY.exists() and B.PROBE_LIBRARY.exists() and not B.FRONT_LIBRARY.exists()
    assert set(json.loads(B.BUILD_INFO.read_text())) == {'git_head', 'library_sha256'}
    assert 'torch is not importable' in capsys.readouterr().err


def test_the_library_builds_without_a_host_compiler(tree, monkeypatch, capsys):
    monkeypatch.setattr(B.shutil, 'which', lambda name: None)
    assert B.build() == B.LIBRARY and not B.FRONT_LIBRARY.exists()
    assert 'no host compiler' in capsys.readouterr().err


def test_a_failed_front_end_leaves_the_library_and_no_older_one(tree, monkeypatch):
    run = B._run

    def failing(cmd):
        if str(B.FRONT_SOURCE) in cmd:
            raise RuntimeError('command failed')
        return run(cmd)
    monkeypatch.setattr(B, '_run', failing)
    with pytest.raises(RuntimeError, match='command failed'):
        B.build()
    assert B.LIBRARY.exists() and not B.FRONT_LIBRARY.exists()
    assert json.loads(B.BUILD_INFO.read_text())['library_sha256'] == B.file_sha256(B.LIBRARY)


def test_the_loader_takes_only_the_front_end_of_its_build(tree):
    B.build()
    assert A._front_mismatch() is None
    good = json.loads(B.BUILD_INFO.read_text())
    for changed, reason in (({'library_sha256': '0'}, 'not from one build'), ({'front_sha256': '0'}, 'not from one build'),
                            ({'torch': '0.0'}, 'was built for torch 0.0'), ({'python': 'x'}, 'was built for python x')):
        B.BUILD_INFO.write_text(json.dumps({**good, **changed}))
        assert reason in A._front_mismatch()
    B.BUILD_INFO.unlink()
    assert A._front_mismatch()
    B.BUILD_INFO.write_text(json.dumps(good))
    assert A._front_mismatch() is None
    B.FRONT_LIBRARY.unlink()
    with pytest.warns(RuntimeWarning, match='run from Python'):
        front = A._load_front()
    assert front.attention(1, 2) is None and front.attention_fused(1) is None
    assert A._FRONT is front
