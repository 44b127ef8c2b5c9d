"""Compiles libsub1_hip.so for gfx950 with hipcc (cross-compiles without a GPU), and
the Python extension that takes tensors apart for it with g++."""
import os
import re
import subprocess
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB_PATH = os.path.join(HERE, 'libsub1_hip.so')
TENSOR_ARGS_PATH = os.path.join(HERE, '_tensor_args.so')
SOURCES = [os.path.join(HERE, 'csrc', 'sub1_kernels.hip'),
           os.path.join(HERE, 'csrc', 'sub1_pack.hip'),
           os.path.join(HERE, 'csrc', 'sub1_prepared.hip'),
           os.path.join(HERE, 'csrc', 'sub1_tiles.hip'),
           os.path.join(HERE, 'csrc', 'sub1_tables.cpp')]

HIPCC_FLAGS = [
    '-O3', '--offload-arch=gfx950', '-fPIC', '-shared', '-std=c++17',
    # keep the compiler from forming packed fp32 instructions
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    # registers and scratch memory per kernel, read back below
    '-Rpass-analysis=kernel-resource-usage',
    '-I' + os.path.join(ROOT, 'include'), '-I' + os.path.join(HERE, 'csrc'),
]


def kernels_with_scratch(compiler_output):
    """{kernel: bytes of scratch memory per lane} for the kernels that spill
    registers, from the compiler's resource-usage remarks."""
    found, name = {}, None
    for line in compiler_output.splitlines():
        m = re.search(r'remark: Function Name: (\S+)', line)
        if m:
            name = m.group(1)
        m = re.search(r'remark:\s+ScratchSize \[bytes/lane\]: (\d+)', line)
        if m and name and int(m.group(1)):
            found[name] = int(m.group(1))
    return found


# Kernels known to spill, and how many bytes per lane: the fused kernel's form for
# tokens grouped by expert keeps four tokens' sums per lane.
SPILLS_ACCEPTED = {'_ZN12_GLOBAL__N_125moe_prepared_fused_kernelILb1ELb0ELb0EEEvNS_12PreparedArgsE': 36}


def torch_mark():
    """What the extension says of the torch that it was built against, of the one installed."""
    import torch
    return 'qmoe_amd, built against torch ' + torch.__version__


def build_tensor_args():
    """Builds the extension module against the installed torch's headers."""
    import torch
    from torch.utils import cpp_extension
    cmd = [os.environ.get('CXX', 'g++'), '-O2', '-fPIC', '-shared', '-std=c++17', '-fvisibility=hidden',
           '-D_GLIBCXX_USE_CXX11_ABI=%d' % torch._C._GLIBCXX_USE_CXX11_ABI,
           '-DSUB1_TORCH_VERSION="%s"' % torch.__version__,
           os.path.join(HERE, 'csrc', 'tensor_args.cpp')]
    cmd += ['-isystem' + path for path in cpp_extension.include_paths() + [sysconfig.get_paths()['include']]]
    cmd += ['-L' + path for path in cpp_extension.library_paths()]
    cmd += ['-ltorch_python', '-ltorch_cpu', '-lc10', '-o', TENSOR_ARGS_PATH]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError('g++ failed:\n' + res.stdout)
    return TENSOR_ARGS_PATH


def build_library(verbose=False):
    """Builds the library and the extension; refuses a build in which a kernel spills registers
    to scratch memory beyond what SPILLS_ACCEPTED lists.  The kernels are
    written to fit their registers (72 to 96 of the 128 that 16 wavefronts per
    compute unit leave a lane), and a spill in a walk costs more than any of
    the tunings measured; one build of the one-token launch that spilled 12
    registers also gave results that differed from run to run (cause not
    established; the code was restructured to fit)."""
    build_tensor_args()
    hipcc = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
    cmd = [hipcc] + HIPCC_FLAGS + SOURCES + ['-o', LIB_PATH]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError('hipcc failed:\n' + res.stdout)
    spilling = {k: v for k, v in kernels_with_scratch(res.stdout).items()
                if v > SPILLS_ACCEPTED.get(k, 0)}
    if spilling:
        os.remove(LIB_PATH)
        raise RuntimeError('kernels that spill registers to scratch memory: %s' % spilling)
    if verbose:
        print('\n'.join(l for l in res.stdout.splitlines() if 'kernel-resource-usage' not in l
                        and not l.lstrip().startswith(('|', '^')) and '__global__' not in l))
    return LIB_PATH


def tensor_args_fit():
    """Whether the extension is there and of the installed torch (looked up in the file: a
    module that has been loaded cannot be loaded again once it is rebuilt)."""
    try:
        with open(TENSOR_ARGS_PATH, 'rb') as f:
            return torch_mark().encode() + b'\0' in f.read()
    except FileNotFoundError:
        return False


def build_what_is_missing():
    """For programs that use what is built: builds only what is not there."""
    if not os.path.exists(LIB_PATH):
        build_library()
    elif not tensor_args_fit():
        build_tensor_args()


if __name__ == '__main__':
    print(build_library(verbose=True))
