"""Builds libqwix_hip.so (gfx950) from the .hip sources in this directory with hipcc, and the host module _plans.so from
plans.cpp with g++ against the installed torch.

Run directly (`python qwix_amd/csrc/build.py`) or through `__graft_entry__.build()`.
Each source is compiled to an object file in `build/`, then everything is linked into
`qwix_amd/libqwix_hip.so`, which the ctypes loader in `qwix_amd/_lib.py` opens.
"""
import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
OUT = os.path.join(PKG, 'libqwix_hip.so')
PLANS = os.path.join(PKG, '_plans.so')
OBJ_DIR = os.path.join(HERE, 'build')
HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
FLAGS = [
    '--offload-arch=gfx950', '-O3', '-std=c++17', '-fPIC', '-fvisibility=hidden',
    # No packed-FP32 VALU ops (v_pk_*_f32) in generated code.
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    '-Wno-unused-command-line-argument',
]


def sources():
  return sorted(f for f in os.listdir(HERE) if f.endswith('.hip'))


def _compile(src: str, force: bool) -> str:
  obj = os.path.join(OBJ_DIR, src[:-4] + '.o')
  deps = [os.path.join(HERE, f) for f in (src, 'common.h', 'qgemm_grouped.h', 'qgemm_strips.h', 'qgemm_tiles.h')]
  deps.append(os.path.join(os.path.dirname(PKG), 'include', 'qwix_hip.h'))
  if not force and os.path.exists(obj) and all(os.path.getmtime(obj) > os.path.getmtime(d) for d in deps):
    return obj
  cmd = [HIPCC, *FLAGS, '-c', os.path.join(HERE, src), '-o', obj]
  r = subprocess.run(cmd, capture_output=True, text=True)
  err = '\n'.join(l for l in r.stderr.splitlines() if 'packed-fp32-ops' not in l)
  if r.returncode != 0:
    raise RuntimeError(f'hipcc failed on {src}:\n{err}')
  if err.strip():
    print(err, file=sys.stderr)
  return obj


def _build_plans(force: bool) -> None:
  """The launch plans (host code only): a Python extension linked to libqwix_hip.so next to it."""
  import sysconfig
  import torch
  src = os.path.join(HERE, 'plans.cpp')
  deps = [src, os.path.join(os.path.dirname(PKG), 'include', 'qwix_hip.h')]
  if not force and os.path.exists(PLANS) and all(os.path.getmtime(PLANS) > os.path.getmtime(d) for d in deps):
    return
  t = os.path.dirname(torch.__file__)
  cmd = ['g++', '-O2', '-std=c++17', '-fPIC', '-shared', '-fvisibility=hidden',
         f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}', '-I' + os.path.join(t, 'include'),
         '-I' + os.path.join(t, 'include', 'torch', 'csrc', 'api', 'include'), '-I' + sysconfig.get_paths()['include'], src,
         '-o', PLANS, '-L' + PKG, '-lqwix_hip', '-L' + os.path.join(t, 'lib'), '-ltorch_python', '-ltorch_cpu', '-lc10',
         '-Wl,-rpath,$ORIGIN']
  r = subprocess.run(cmd, capture_output=True, text=True)
  if r.returncode != 0:
    raise RuntimeError(f'g++ failed on plans.cpp:\n{r.stderr}')


def build(force: bool = True, verbose: bool = True) -> str:
  os.makedirs(OBJ_DIR, exist_ok=True)
  srcs = sources()
  with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
    objs = list(ex.map(lambda s: _compile(s, force), srcs))
  cmd = [HIPCC, '--offload-arch=gfx950', '-shared', '-fPIC', *objs, '-o', OUT]
  r = subprocess.run(cmd, capture_output=True, text=True)
  if r.returncode != 0:
    raise RuntimeError(f'link failed:\n{r.stderr}')
  _build_plans(force)
  if verbose:
    print(f'built {OUT} from {len(srcs)} sources')
  return OUT


if __name__ == '__main__':
  build(force='--incremental' not in sys.argv)
