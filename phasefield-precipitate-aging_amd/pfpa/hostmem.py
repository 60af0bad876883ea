"""Host memory of batch read-backs, used again from one read to the next.

A read-back of a batch fills some ten to hundred MB of new host arrays.  From
malloc these are fresh pages whenever the C heap has given its top back to the
system in between, which depends on everything the process allocated before: a
page fault per 4 KiB, as long as the copy itself (twelve FP64 domains of 200 to
900 cells a side, 300 steps and their read-back: 12.4 ms a pass without faults,
17-25 ms with 13,800).  Blocks mapped here come back when the last array on them
is gone, and serve the next read of that size."""
import collections
import mmap
import threading
import weakref

import numpy as np


class BlockPool:
    """Blocks of anonymous memory by size class, at most `limit` bytes of them
    free; none are kept while the pool has no user (open / close)."""

    def __init__(self, limit):
        self.limit = limit
        self.users = set()
        self.free = collections.OrderedDict()   # size -> free blocks; last used class last
        self.free_bytes = 0
        # Finalizers run wherever an array dies, also inside this pool's own
        # code on the same thread, so they only put the block here and take the
        # lock if it is to be had; whoever holds it sorts the block in next time.
        self.returned = collections.deque()
        self.lock = threading.Lock()

    @staticmethod
    def size_class(nbytes):
        """`nbytes` rounded up to an eighth of its power of two (and to pages)."""
        step = max(mmap.PAGESIZE, 1 << max(0, nbytes.bit_length() - 4))
        return max(1, -(-nbytes // step)) * step

    def open(self, user):
        self.users.add(user)

    def close(self, user):
        self.users.discard(user)
        self._try_sort()

    def array(self, shape, dtype):
        """An uninitialised C-order array.  Its memory serves another array
        once it and every view of it are gone."""
        dtype = np.dtype(dtype)
        count = 1
        for n in shape:
            count *= int(n)
        size = self.size_class(count * dtype.itemsize)
        with self.lock:
            self._sort()
            block = None
            if size in self.free:
                self.free.move_to_end(size)
                block = self.free[size].pop()
                self.free_bytes -= size
                if not self.free[size]:
                    del self.free[size]
        if block is None:
            block = mmap.mmap(-1, size)
        # on a memoryview, so that views have this array for their base, not the block
        owner = np.frombuffer(block, dtype=dtype, count=count)
        weakref.finalize(owner, self._give_back, block).atexit = False
        return owner.reshape(shape)

    def _give_back(self, block):
        self.returned.append(block)
        self._try_sort()

    def _try_sort(self):
        if self.lock.acquire(blocking=False):
            try:
                self._sort()
            finally:
                self.lock.release()

    def _sort(self):
        while self.returned:
            block = self.returned.popleft()
            size = len(block)
            self.free.setdefault(size, []).append(block)
            self.free.move_to_end(size)
            self.free_bytes += size
        limit = self.limit if self.users else 0
        while self.free_bytes > limit:
            size = next(iter(self.free))
            self.free[size].pop(0)
            self.free_bytes -= size
            if not self.free[size]:
                del self.free[size]


# Read-backs of all batches of the process: two of some hundred MB alternate
# without a fault where a program holds one while it makes the next.
read_back = BlockPool(256 << 20)
