"""The dispatch rule of the fused gradient, restated for tests: whether the rows of one launch run two
a workgroup (csrc/nrc_grad_rows.hpp).  The workgroups go in order to the CU that is free first."""
import heapq


def rows_of(records, chunks):
    """Rows of a cache whose step has `records` records in rows of `chunks` chunks, and the chunks of one."""
    n = max(1, -(-records // 64))
    return -(-n // chunks), min(chunks, n)


def launch_end(rows, cus, per_group, base, per_chunk):
    free = [0] * cus
    for count, chunks in rows:
        for _ in range(-(-count // per_group)):
            heapq.heappush(free, heapq.heappop(free) + base + per_chunk * chunks)
    return max(free)


def in_pairs(sizes, cus=256):
    """sizes: (records, chunks) of each cache of one launch, a cache with several chunks a row among them."""
    rows = [rows_of(*s) for s in sizes]
    if sum(r for r, _ in rows) <= cus:
        return False
    return 10 * launch_end(rows, cus, 2, 10, 8) < 9 * launch_end(rows, cus, 1, 8, 5)
