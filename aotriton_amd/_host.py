"""Loads _torch_host.so, the native host path between PyTorch and the library (csrc/torch/host.cpp).  If it is
missing or was built for another torch this raises instead of falling back to anything else."""
import os

PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), '_torch_host.so')


def load():
    import torch      # first: the extension links its libraries
    hint = 'build it with `python -m aotriton_amd.build`. There is no fallback path.'
    try:
        from . import _torch_host
    except ImportError as e:
        raise ImportError(f'{PATH} is missing or does not load with torch {torch.__version__}: {hint}') from e
    if _torch_host.torch_version != str(torch.__version__):      # its C++ ABI is another with every version
        raise ImportError(f'{PATH} was built for torch {_torch_host.torch_version}, this is {torch.__version__}: {hint}')
    return _torch_host


class _OnFirstUse:
    """Stands for the extension in a module that is also of use without torch."""

    def __getattr__(self, name):
        if name.startswith('__'):
            raise AttributeError(name)
        function = getattr(load(), name)
        setattr(self, name, function)
        return function


on_first_use = _OnFirstUse()
