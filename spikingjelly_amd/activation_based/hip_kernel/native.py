"""The native host path: ``spikingjelly_amd/_sjhip_torch.so`` (``csrc/torch_binding.cpp``), torch's C++ autograd in front of
the C ABI of ``libsjhip.so``.  Built in-tree by the same ``make``; a missing module raises, nothing falls back silently."""

from __future__ import annotations

from . import library

_module = None


def load():
    """The extension module (imported once); ``OSError`` when it or the library is not built."""
    global _module
    if _module is None:
        library.load()
        try:
            from spikingjelly_amd import _sjhip_torch
        except ImportError as e:
            raise OSError(f"spikingjelly_amd/_sjhip_torch.so cannot be imported ({e}); run `make -C spikingjelly_amd/csrc`") from e
        if _sjhip_torch.abi_version() != library.ABI_VERSION:
            raise OSError(f"_sjhip_torch.so: ABI version {_sjhip_torch.abi_version()} != {library.ABI_VERSION}")
        _module = _sjhip_torch
    return _module
