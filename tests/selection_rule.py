"""The one-wave selection's rule restated in numpy for one row of logits (at most 512, k <= 15): which list of candidates it ranks and
whether it accepts what it ranked, or leaves the row to the reference's rungs over the probabilities."""
import numpy as np

GAP, GAP_LAST, FLOOR = np.float32(2.0 ** -19), np.float32(2.0 ** -17), np.float32(-69.0)
FINITE = 0x00800000   # keys from here on are above -inf's


def keys(logits):
    b = np.ascontiguousarray(logits, np.float32).view(np.uint32)
    return np.where(b >> 31, ~b, b ^ np.uint32(0x80000000)).astype(np.int64)


def list_length(logits, k, wide=True):
    """Candidates: the keys not below the (k+1)-th largest of the best of sixteen groups (32 from k = 12 on).
    wide: the row lies eight logits to a lane, however short it is."""
    n = logits.size
    padded = np.full(512 if wide else max(64, 1 << (n - 1).bit_length()), FINITE - 1, np.int64)
    padded[:n] = keys(logits)
    heads = padded.reshape(-1, 16 if k < 12 or padded.size == 64 else 32).max(axis=0)
    exact = heads[(heads[:, None] < heads[None, :]).sum(axis=1) == k]
    return int((padded >= max(exact[0] if exact.size else 0, FINITE)).sum())


def select(logits, k, gap=GAP, gap_last=GAP_LAST, wide=True):
    """(accepted, ids): ids only if accepted."""
    key, n = keys(logits), logits.size
    if (key < FINITE - 1).any() or list_length(logits, k, wide) > 64:   # (NaN with its sign set)
        return False, None
    order = np.argsort(key, kind="stable")[::-1][:k + 1]
    slots = [int(e) for e in order if key[e] >= FINITE]
    if len(set(key[slots].tolist())) != len(slots) or len(slots) < min(k + 1, n):   # (equal keys leave an empty slot, whichever of them is in the other)
        return False, None
    l = logits[slots].astype(np.float32)
    with np.errstate(invalid="ignore"):
        d = (l - l[0]).astype(np.float32)
        fall = (d - np.append(d[1:], np.float32(-np.inf))).astype(np.float32)[:k]
        needed = np.full(k, gap, np.float32)
        needed[k - 1] = gap_last
        ok = (fall >= needed).all() and (d[:k] >= FLOOR).all()
    return bool(ok), np.array(slots[:k], np.int32) if ok else None


def crowded_rows(n, k, seed=0):
    """Rows whose favourites crowd into few residues modulo 16 or 64, so that the list comes out long: (its length, row)."""
    rng = np.random.default_rng(1000 * n + k + seed)
    for modulo, residues, each in [(16, 1, 32), (16, 2, 16), (16, 3, 12), (16, 4, 10), (16, 5, 16), (16, k, 8), (64, k, 8), (64, k - 1, 8), (16, 1, 14), (32, k, 4)]:
        row = rng.normal(0, 1, n).astype(np.float32)
        for r in rng.permutation(modulo)[:max(residues, 1)]:
            row[r::modulo][:each] += np.float32(8)
        yield list_length(row, k), row
