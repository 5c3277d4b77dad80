"""The work queues of the large-tile GEMMs (csrc/chunks.hpp, csrc/combine.hpp) and the way a launch shares them out
(mx_gemm_kernel in csrc/bwmm_mx.hip, rows_per_piece in csrc/mx_tile.hpp), restated on the host: what a test of cut rounds needs
in order to know that its launch is cut."""

import numpy as np

CHUNK_ROWS, CHUNK_ROWS_MAX, FIXED_COST = 256, 320, 20
CLASSES, NO_CLASS = 12, 12


def chunks_of(tp2id, b2e, B, E, T, pad_row=False):
    """[(first slot, rows, expert)] of the tables' chunks; pad_row: with activation checkpoints."""
    real = np.asarray(tp2id).reshape(-1, B)
    real = (real >= 0) & (real < T)
    b2e = np.asarray(b2e).reshape(-1)
    valid = np.where(real.any(axis=1), B - np.argmax(real[:, ::-1], axis=1), 0)
    out, b = [], 0
    while b < len(b2e):
        e, j, end = b2e[b], b, -1
        while j < len(b2e) and b2e[j] == e:
            if valid[j]:
                end = j * B + valid[j]
            j += 1
        if pad_row:
            end = b * B + 1 if end < 0 else min(end + 1, j * B)
        n = end - b * B
        if 0 <= e < E and n > 0:
            pieces = 1 if n <= CHUNK_ROWS_MAX else -(-(n - CHUNK_ROWS_MAX) // CHUNK_ROWS) + 1
            out += [(b * B + i * CHUNK_ROWS, CHUNK_ROWS if i + 1 < pieces else int(n) - i * CHUNK_ROWS, int(e)) for i in range(pieces)]
        b = j
    return out


def row_tiles(rows):
    return 4 if rows <= 64 else 8 if rows <= 128 else 2 * ((rows + 31) // 32)


def chunk_class(rows, stream):
    t = row_tiles(rows)
    if not stream:
        return {20: 0, 18: 2}.get(t, 4 if t >= 10 else 9)
    return {20: 1, 18: 3, 16: 5, 14: 6, 12: 7, 10: 8, 8: 10, 4: 11}[t]


def queues_of(chunks, pad_row=False):
    """(interleave, one list of (class, chunk) in queue order for each of the eight XCDs)."""
    n, runs = len(chunks), 1 + sum(a[2] != b[2] for a, b in zip(chunks, chunks[1:]))
    avg = (n + runs // 2) // runs
    interleave = 1 if avg < 3 or n > 4096 else min(avg, 8)
    work = [row_tiles(r) + FIXED_COST for _, r, _ in chunks]
    total, before, out = sum(work), 0, [[] for _ in range(8)]
    for i, c in enumerate(chunks):
        stream = interleave == 1 and (i + 1 == n or chunks[i + 1][2] != c[2])
        cls = chunk_class(c[1], stream)
        if pad_row and row_tiles(c[1]) == 18:
            cls -= 2
        out[min(7, (2 * before + work[i]) * 8 // (2 * total))].append((cls, c))
        before += work[i]
    return interleave, [sorted(q, key=lambda x: x[0]) for q in out]


def workgroups_per_xcd(gx, max_chunks, cus=256):
    return min(cus // 8, (4 * gx * max_chunks + 7) // 8)


def cut_of(queue, interleave, gx, W):
    """(items that are whole, shift): the others are cut into 1 << shift pieces."""
    total = len(queue) * gx
    full, rest = divmod(total, W)
    shift = 0 if interleave > 1 or rest == 0 or 2 * rest > W else 1 if 4 * rest > W else 2
    if shift and queue[full * W // gx][0] > 8:
        shift = 0
    return (full * W if shift else total), shift


def launch_cuts(queues, gx, max_chunks):
    """The set of shifts of the XCDs that have a queue."""
    W = workgroups_per_xcd(gx, max_chunks)
    return {cut_of(q, queues[0], gx, W)[1] for q in queues[1] if q}


def pieces(rows, shift):
    per = (((rows + (1 << shift) - 1) >> shift) + 31) & ~31
    per = rows if rows <= 128 else max(per, 64)
    return [max(0, min(per, rows - i * per)) for i in range(1 << shift)]


def items_of(w, queue, interleave, gx, W):
    """What workgroup w does, in order: ("whole", item, class) and at last maybe ("piece", item, number, rows, class)."""
    total = len(queue) * gx
    whole, shift = cut_of(queue, interleave, gx, W)
    out, item, step = [], w, 2 * (W - 1 - w) + 1
    while item < whole:
        out.append(("whole", item, queue[item // gx][0]))
        item, step = item + step, 2 * W - step
    if shift:
        p = item - whole
        at = whole + (p >> shift)
        if at < total:
            rows = pieces(queue[at // gx][1][1], shift)[p & ((1 << shift) - 1)]
            if rows > 0:
                out.append(("piece", at, p & ((1 << shift) - 1), rows, chunk_class(rows, True)))
    return out
