"""Host-side mirror of the rollback caches
(Sources/DFlash/RecurrentRollbackCache.swift) over the C handles of
include/dflash_cache.h.

The native handle does the bookkeeping and enqueues the kernels; these classes
keep the torch tensors alive (the handle only stores their device pointers) and
give the caches the reference's names.  ``cache[0]`` is the conv window
[B, keep, C], ``cache[1]`` the recurrent state [B, Hv, Dv, Dk].
"""

from __future__ import annotations

import ctypes as C
from typing import Optional

import torch

from . import _lib
from ._lib import native as _native
from .dflash_kernels import _stream


class _NativeCache:
    KIND = _lib.CACHE_MAMBA

    def __init__(self, conv_kernel_size: int = 4):
        self._h = C.c_void_p(_lib.load().dflash_cache_create(self.KIND, conv_kernel_size))
        if not self._h:
            raise _lib.DFlashError("cache_create: " + _lib.last_error())
        self._handle = self._h.value
        self._by_ptr = {}

    def __del__(self):
        h, self._h = getattr(self, "_h", None), None
        load = getattr(_lib, "load", None)          # None while the interpreter shuts down
        if h and load:
            load().dflash_cache_destroy(h)

    # slots -------------------------------------------------------------------
    def __getitem__(self, i: int) -> Optional[torch.Tensor]:
        return self._by_ptr.get(_native.cache_get_slot(self._handle, i))

    def __setitem__(self, i: int, t: Optional[torch.Tensor]) -> None:
        p = _native.cache_set_slot(self._handle, i, t)
        if t is not None:
            self._by_ptr[p] = t
        if not self._holds_snapshot():
            self._forget_dead()

    def _holds_snapshot(self) -> bool:
        return False

    def _forget_dead(self) -> None:
        held, h = self._by_ptr, self._handle
        self._by_ptr = {p: held[p] for p in (_native.cache_get_slot(h, 0), _native.cache_get_slot(h, 1)) if p in held}

    @property
    def offset(self) -> int:
        return int(_lib.load().dflash_cache_offset(self._h))

    @offset.setter
    def offset(self, v: int) -> None:
        _lib.check(_lib.load().dflash_cache_set_offset(self._h, int(v)), "cache_set_offset")

    def trim(self, n: int) -> int:
        return int(_lib.load().dflash_cache_trim(self._h, int(n)))

    @property
    def is_trimmable(self) -> bool:
        return False


class MambaCache(_NativeCache):
    """Plain recurrent cache without rollback (the reference's MambaCache lives in mlx-swift-lm;
    only its use at DFlashRuntime.swift:206-211 matters here)."""

    KIND = _lib.CACHE_MAMBA


class KVCacheSimple(_NativeCache):
    """Trimmable attention cache as seen by restoreTargetCacheAfterAcceptance
    (DFlashRuntime.swift:212-218): an offset that ``trim`` lowers."""

    KIND = _lib.CACHE_KV

    @property
    def is_trimmable(self) -> bool:
        return True


class _RollbackCache(_NativeCache):
    """``protocol DFlashRollbackCache`` (RecurrentRollbackCache.swift:12-18)."""

    @property
    def is_armed(self) -> bool:
        return _native.cache_is_armed(self._handle)

    def _holds_snapshot(self) -> bool:
        return _native.cache_is_armed(self._handle)

    def arm_rollback(self, prefix_len: int = 0) -> None:
        _native.cache_arm(self._handle, prefix_len)

    def record_tape(self, tape: torch.Tensor, k: torch.Tensor, g: torch.Tensor, qkv: Optional[torch.Tensor]) -> None:
        state = self[1]
        if state is None:
            raise _lib.DFlashError("record_tape: slot 1 (recurrent state) is empty")
        self._tape_refs = _native.cache_record_tape(self._handle, tape, k, g, qkv, state)

    def rollback(self, n_accepted: int) -> None:
        rc = _lib.load().dflash_cache_rollback(self._h, _stream(), int(n_accepted))
        self._after_rollback()
        _lib.check(rc, "rollback")

    def clear_transients(self) -> None:
        _lib.check(_lib.load().dflash_cache_clear_transients(self._h), "clear_transients")
        self._after_rollback()

    def _after_rollback(self) -> None:
        # tape tensors stay referenced until the next cycle records new ones: the replay
        # that reads them may still be queued on the stream.  A rollback that was refused leaves the cache
        # armed: the handle still points at the snapshot, whose tensors no slot holds any more.
        if not self._holds_snapshot():
            self._forget_dead()


class RecurrentRollbackCache(_RollbackCache):
    """``RecurrentRollbackCache`` (RecurrentRollbackCache.swift:34-182): tape-replay rollback."""

    KIND = _lib.CACHE_TAPE
    default_conv_kernel_size = 4            # :135


class MambaSnapshotCache(_RollbackCache):
    """``MambaSnapshotCache`` (RecurrentRollbackCache.swift:193-232): snapshot-only rollback."""

    KIND = _lib.CACHE_SNAPSHOT
