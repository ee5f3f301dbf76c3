"""Hand-made octrees for the traversal tests: every node form the word layout
allows the traversal to meet, at up to the full 23 levels."""
import numpy as np


def mixed_tree(seed, levels, fanout=2.2, loose=False):
    """Random tree with leaves, childless descriptors and far (two-word) child
    slots at every level; `levels` descriptor levels. Masks are as the
    reference writes them (a node's children are all descriptors or all
    leaves). One path always reaches the last level, whose descriptor there is
    childless when the seed is odd. loose: some one-word child blocks are
    followed by a word that their last child uses as its far word."""
    rng = np.random.default_rng(seed)

    def node(level, spine):
        # (valid mask, children or None for leaves, large)
        if level == levels - 1:
            if spine and seed % 2:
                return (0, [], False)
            return (int(rng.integers(1, 256)), None, False)
        if not spine and rng.random() < 0.15:
            return (0, [], False)
        if not spine and rng.random() < (0.3 if level < 6 else 0.6):
            return (int(rng.integers(1, 256)), None, False)
        p = min(1.0, fanout / 8.0) if level > 2 else 0.6
        valid = 0
        for c in range(8):
            if rng.random() < p:
                valid |= 1 << c
        keep = int(rng.integers(0, 8))
        if spine or not valid:
            valid |= 1 << keep
        kids = [node(level + 1, spine and c == keep) for c in range(8) if valid >> c & 1]
        return (valid, kids, bool(rng.random() < 0.4) or size(kids) > 0x2000)

    def size(kids):
        return sum(2 + (bin(k[0]).count("1") if k[1] is None else size(k[1])) for k in kids)

    words = []

    def emit(n, at, far):
        # descriptor of n at words[at]; its child block goes at the end of the array
        valid, kids, large = n
        start = len(words)
        off = start - at
        d = (valid << 8) | (valid if kids else 0) | (0x10000 if large else 0)
        if far:
            words[at] = d | 0x20000
            words[at + 1] = off
        else:
            assert off <= 0x3FFF, "child block too far for a one-word slot"
            words[at] = d | (off << 18)
        if kids is None:
            words.extend(int(x) | 1 for x in rng.integers(0, 1 << 32, bin(valid).count("1")))
            return
        per = 2 if large else 1
        spare = loose and not large and rng.random() < 0.5
        words.extend([0] * (per * len(kids) + spare))
        for i, k in enumerate(kids):
            emit(k, start + i * per, large or (spare and i == len(kids) - 1))

    root = node(0, True)
    words.append(0)
    root_far = seed % 3 == 0
    if root_far:
        words.append(0)
    emit(root, 0, root_far)
    return np.array(words, np.uint64).astype(np.uint32)
