"""The breakdown of a step's device time by class of kernel leaves no entry point out."""
import inspect
import types

from kv_cache_optimization_for_llm_amd.ops import kernels as K

# reads for measurements, the library's start-up timing, and what runs inside an entry point that has a class
APART = {"stream_read", "stream_reread", "stream_mixed", "gemm_vendor_tune", "_recurrent_chunks"}


def test_every_launching_entry_point_has_a_class():
    launching = {name for name, f in vars(K).items() if isinstance(f, types.FunctionType) and f.__module__ == K.__name__
                 and name != "_stream" and "_stream()" in inspect.getsource(f)}
    assert launching - APART <= set(K.KERNEL_CLASSES), launching - APART - set(K.KERNEL_CLASSES)
    assert all(callable(getattr(K, name)) for name in K.KERNEL_CLASSES)
