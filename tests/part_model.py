"""The schedule of the part-wise triangular sweeps, restated: parts, windows of 64 slots and the
codes of a slot's entries (csrc/fcap_parts.hip), for a CSR structure with 0-based arrays."""
import numpy as np

PART_ROWS = 4096


def stencil(dims, steps):
    """(ioffset, ja, diag), 1-based, of a box of cells each coupled to the cells `steps` away, both ways."""
    idx = np.arange(np.prod(dims)).reshape(dims[::-1])   # [z, y, x]
    pairs = [np.stack([idx.ravel(), idx.ravel()])]
    for st in steps:
        st = st[::-1]
        lo = tuple(slice(max(0, -k), d - max(0, k)) for k, d in zip(st, idx.shape))
        hi = tuple(slice(max(0, k), d - max(0, -k)) for k, d in zip(st, idx.shape))
        p = np.stack([idx[lo].ravel(), idx[hi].ravel()])
        pairs += [p, p[::-1]]
    row, col = np.concatenate(pairs, axis=1)
    order = np.lexsort((col, row))
    row, col = row[order], col[order]
    ioffset = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=idx.size))])
    one = lambda x: np.ascontiguousarray(x + 1, np.int32)  # noqa: E731
    return one(ioffset), one(col), one(np.flatnonzero(row == col))


# six, then eight entries in a strict triangle (a row coupled to itself and 12 or 16 others)
STEPS6 = ((1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 0, 1), (0, 1, 1))
STEPS8 = STEPS6 + ((1, 1, 1), (2, 0, 0))


def _linked(start, ptr, ja, diag):
    """Whether row start[u] reads row start[u - 1]."""
    f = np.zeros(len(start), bool)
    for u in range(1, len(start)):
        r = start[u]
        f[u] = start[u - 1] in ja[ptr[r]:diag[r]]
    return f


def pencil_parts(ptr, ja, diag):
    """(part of each row, parts) where the numbering has the runs of structured blocks, else None."""
    n = len(diag)
    start = np.flatnonzero(~_linked(np.arange(n), ptr, ja, diag))
    lines = len(start)
    if 4 * lines > n:
        return None
    lf = _linked(start, ptr, ja, diag)
    sheet = np.flatnonzero(~lf)
    sheets = len(sheet)
    sf = _linked(start[sheet], ptr, ja, diag)
    nlines = np.diff(np.append(sheet, lines))
    part, nparts, s0 = np.zeros(lines, int), 0, 0
    while s0 < sheets:
        J, s1 = nlines[s0], s0 + 1
        while s1 < sheets and sf[s1] and nlines[s1] == J:
            s1 += 1
        K = s1 - s0
        bj = min(J, 64 // min(8, K))
        bk = min(K, 64 // bj)
        nj, nk = -(-J // bj), -(-K // bk)
        ids = {}
        for d in range(nj + nk - 1):
            for b in range(max(0, d - nj + 1), min(nk, d + 1)):
                ids[b, d - b] = nparts
                nparts += 1
        for k in range(K):
            for j in range(J):
                part[sheet[s0 + k] + j] = ids[k * nk // K, j * nj // J]
        s0 = s1
    if nparts * 512 > n + 64 * 512:
        return None
    return np.repeat(part, np.diff(np.append(start, n))), nparts


def run_parts(ptr, ja, diag, rows=PART_ROWS):
    n = len(diag)
    return np.arange(n) // rows, -(-n // rows)


class Schedule:
    """Packed slots of both sweeps: rows, step, win (first window of a part), win_part, slot_of."""

    def __init__(self, ptr, ja, diag, part, nparts):
        n = len(diag)
        self.csr = ptr, ja, diag
        lev = np.zeros(n, int)
        for i in range(n):
            if diag[i] > ptr[i]:
                lev[i] = lev[ja[ptr[i]:diag[i]]].max() + 1
        order = np.lexsort((np.arange(n), lev, part))
        rows, step, win, win_part, used, rank = [], [], [0], [], 64, 0

        def close():
            nonlocal used
            while used < 64:
                rows.append(rows[-1])
                step.append(step[-1])
                used += 1

        begin = np.searchsorted(part[order], np.arange(nparts + 1))
        for p in range(nparts):
            b = begin[p]
            while b < begin[p + 1]:
                e = b + 1
                while e < begin[p + 1] and lev[order[e]] == lev[order[b]]:
                    e += 1
                if used + (e - b) > 64:
                    close()
                else:
                    rank += 1
                for q in order[b:e]:
                    if used == 64:
                        used = rank = 0
                        win_part.append(p)
                    rows.append(q)
                    step.append(rank)
                    used += 1
                b = e
            close()
            win.append(len(win_part))
        self.rows, self.step = np.array(rows), np.array(step, np.uint8)
        self.win, self.win_part = np.array(win, np.int32), np.array(win_part)
        self.nparts, self.npk = nparts, len(rows)
        self.slot_of = np.zeros(n, int)
        self.slot_of[self.rows[::-1]] = np.arange(self.npk)[::-1]   # a row's first slot

    def entries(self, upper, width):
        """(slot x width) CSR positions of a slot's entries, -1 past its last."""
        ptr, ja, diag = self.csr
        s = diag[self.rows] + 1 if upper else ptr[self.rows]
        c = (ptr[self.rows + 1] if upper else diag[self.rows]) - s
        assert c.max(initial=0) <= width
        k = np.arange(width)
        return np.where(k < c[:, None], s[:, None] + k, -1)

    def codes(self, upper, width, ring):
        """(width + 1, slots): ring slot, packed slot | top bit, or `ring` (padding); then the row."""
        e = self.entries(upper, width)
        at = self.slot_of[self.csr[1][np.maximum(e, 0)]]
        q = np.arange(self.npk)[:, None]
        same = self.win_part[at >> 6] == self.win_part[q >> 6]
        inside = same & ((at < 64 * (q >> 6) + ring) if upper else (at + ring >= 64 * ((q >> 6) + 1)))
        own = self.slot_of[self.rows][:, None]
        assert np.all((e < 0) | ((at > own) if upper else (at < own)))
        code = np.where(inside, at & (ring - 1), at | 0x80000000)
        code = np.where(e < 0, ring, code)
        first = (np.arange(self.npk) == self.slot_of[self.rows])[:, None] & (e >= 0)
        self.inside = inside[first].mean() if first.any() else 0.0
        return np.vstack([code.T, self.rows[None]]).astype(np.uint32).view(np.int32)

    def values(self, upper, width, a, d, dtype):
        e = self.entries(upper, width)
        return np.vstack([np.where(e < 0, 0.0, a[np.maximum(e, 0)]).T, d[self.rows][None]]).astype(dtype)


def packed(x):
    """(entries, slots) in the kernels' layout: 16-byte blocks of entries, the rest one by one."""
    x = np.ascontiguousarray(x)
    v = 16 // x.itemsize
    b = x.shape[0] // v
    blocks = x[:b * v].reshape(b, v, -1).transpose(0, 2, 1).reshape(-1)
    return np.ascontiguousarray(np.concatenate([blocks, x[b * v:].reshape(-1)]))
