"""Lazy tensors backed by torch allocations (bindings/lazy_tensor/main.cc:25-34,
lazy_tensor_template.h:19-98): the buffer is created only if the chosen backend
asks for it and is dropped when the operator returns."""
import ctypes

from .. import _lib


class _Lazy:
    """Owns the ctypes struct plus the Python callbacks that keep it alive.  Both are made when the
    struct is asked for: the native host path allocates by itself and never does."""
    C = None
    ACQ = None
    DISP = None

    def __init__(self, like_view, device_index, dtype=None, eager=None):
        """``like_view``: the view whose shape the buffer takes, or a function that makes it when the
        struct is first needed."""
        self._like_view = like_view
        self._device = device_index
        self._eager = eager
        self._held = None
        self._c = None

    @property
    def on_demand(self):
        """Stands for a buffer that is allocated when the operator asks for it."""
        return self._eager is None

    @property
    def _like(self):
        if callable(self._like_view):
            self._like_view = self._like_view()
        return self._like_view

    @property
    def c(self):
        """The C struct; made, with its callbacks, on first use."""
        if self._c is None:
            self._c = self._make()
        return self._c

    def _make(self):
        import torch
        from . import DType
        c = self.C()
        c.cookie = None
        if self._eager is not None:
            c.eager = self._eager.to_c()
            self._acq = self.ACQ(0)
            self._disp = self.DISP(0)
        else:
            def acquire(self_ptr, out_ptr):
                try:
                    dev = torch.device('cuda', self._device) if self._device is not None else None
                    t = torch.empty(tuple(self._like.sizes), dtype=torch.float32, device=dev)
                    self._held = t
                    out = out_ptr.contents
                    out.ptr = t.data_ptr()
                    for i in range(len(self._like.sizes)):
                        out.sizes[i] = t.size(i)
                        out.strides[i] = t.stride(i)
                    out.dtype = int(DType.kFloat32)
                    self_ptr.contents.cookie = 1
                    return 0
                except Exception:
                    return 1

            def dispose(self_ptr):
                self._held = None
                self_ptr.contents.cookie = None

            self._acq = self.ACQ(acquire)
            self._disp = self.DISP(dispose)
        c.acquire = self._acq
        c.dispose = self._disp
        return c

    def __bool__(self):
        return True


class LazyTensor2(_Lazy):
    C = _lib.fa_lazy_tensor2
    ACQ = _lib.ACQUIRE2
    DISP = _lib.DISPOSE2


class LazyTensor4(_Lazy):
    C = _lib.fa_lazy_tensor4
    ACQ = _lib.ACQUIRE4
    DISP = _lib.DISPOSE4


def delta(L_view, device_index):
    """fp32 tensor shaped like L, allocated on demand."""
    return LazyTensor2(L_view, device_index)


def dq_acc(dq_view, device_index):
    """fp32 tensor shaped like dQ; this library never acquires it."""
    return LazyTensor4(dq_view, device_index)


def eager_delta(delta_view):
    return LazyTensor2(delta_view, None, eager=delta_view)


def eager_null_dq_acc():
    from . import T4, DType
    return LazyTensor4(T4(0, [0] * 4, [0] * 4, DType.kFloat32), None,
                       eager=T4(0, [0] * 4, [0] * 4, DType.kFloat32))
