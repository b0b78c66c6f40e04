"""The coders' forms that guess and correct, restated on Python integers and checked on the CPU: the float32
search of decode_float_kernel with its walks in both directions (decoder.hpp: decode_symbol<..., FLOAT>),
the decoder of four symbols between two looks (decode_few_symbol, decode_few_lane) and the encoder of
four symbols without a branch (encoder_few.hpp: FewEncoder).  The float search is compared with the exact one,
the coders with the bit-serial coder of tests/pycoder.py."""
import random

import numpy as np
import pytest

import pycoder
from test_kernel_arithmetic_model import M32, random_table, step_count

M64 = (1 << 64) - 1


def mulhi(a, b):
    return (a * b) >> 32


def f32(x):
    """x rounded to float32, as an integer (x < 2^33: the result is a whole number or x itself)."""
    return int(np.float32(x))


# ---- the float search ----------------------------------------------------------------------------
def below_off(c, span, off):
    """The sign of fma(c * 2^-149, float32(span) * 2^95, -float32(off) * 2^-38): one rounding, which keeps the sign."""
    return c * f32(span) < f32(off) << 16


def float_search(cdf, log2, skip, span, off):
    """The guess: steps on held entries, then two a round trip, as decode_symbol takes them."""
    steps = log2 - skip
    held_steps = 3 if steps >= 5 else steps - 2
    apart = 1 << (steps - held_steps)
    left = [None] + [cdf[k * apart] for k in range(1, 1 << held_steps)]
    at = 0
    for h in range(held_steps - 1, -1, -1):
        up = below_off(left[1 << h], span, off)
        at |= up << (steps - held_steps + h)
        for k in range(1, 1 << h):
            left[k] = left[(1 << h) + k] if up else left[k]
    k = steps - held_steps - 1
    if k % 2 == 0:
        at |= below_off(cdf[at + (1 << k)], span, off) << k
        k -= 1
    while k >= 1:
        c1, c2, c3 = cdf[at + (1 << k - 1)], cdf[at + (1 << k)], cdf[at + 3 * (1 << k - 1)]
        up = below_off(c2, span, off)
        at |= up << k
        at |= below_off(c3 if up else c1, span, off) << k - 1
        k -= 2
    return at


def corrected(cdf, log2, skip, safe, span, off, p):
    """decode_symbol's test and walks from the guess p (span not the full range): (symbol, T(lower), width, walked)."""
    plast, end = len(cdf) - 2, (1 << log2 - skip) - 1
    lo, hi = cdf[p] << 16, cdf[p + 1] << 16
    t_lo = mulhi(span, lo)
    width = ((span if safe and p == plast else mulhi(span, hi)) - t_lo) & M32
    rel, walked = (off - t_lo) & M32, 0
    if rel >= width:
        top = safe and p == plast
        while t_lo > off:
            p, hi, top, walked = p - 1, lo, False, walked - 1
            lo = cdf[p] << 16
            t_lo = mulhi(span, lo)
        width = ((span if top else mulhi(span, hi)) - t_lo) & M32
        while (off - t_lo) & M32 >= width and p < end:
            p, walked = p + 1, walked + 1
            t_lo = mulhi(span, cdf[p] << 16)
            width = ((span if safe and p == plast else mulhi(span, cdf[p + 1] << 16)) - t_lo) & M32
    return p, t_lo, width, walked


def table(rng, nsym, skew=3):
    return random_table(rng, nsym, skew)


@pytest.mark.parametrize("log2", [3, 4, 5, 6])
@pytest.mark.parametrize("skip", [0, 1])
def test_float_search_is_corrected_to_the_exact_symbol(log2, skip):
    """Every symbol that is searched, code values at its ends and around them, spans from the smallest to the largest: the
    guess is off by at most one and the walks end at the exact symbol, at the last entry of a half table (skip 1), at the
    last symbol (safe, skip 0) and next to it."""
    rng = random.Random(10 * log2 + skip)
    nsym, short, over = 1 << log2, set(), set()
    last = (1 << log2 - skip) - 1
    for trial in range(60):
        cdf = table(rng, nsym, rng.choice([0.5, 1, 3, 8]))
        for span in [M32, (1 << 30) + 1, 0x80000001, rng.randrange((1 << 30) + 1, 1 << 32), rng.randrange((1 << 30) + 1, 1 << 32)]:
            safe = not skip and rng.random() < 0.5
            for m in range(last + 1 if skip or safe else last):            # not safe: the last symbol does not occur
                t_lo = mulhi(span, cdf[m] << 16)
                t_hi = span if safe and m == nsym - 1 else mulhi(span, cdf[m + 1] << 16)
                for off in {t_lo, t_lo + 1, t_lo + 100, t_hi - 1, t_hi - 2, t_hi - 100, rng.randrange(t_lo, t_hi)}:
                    if not t_lo <= off < t_hi:
                        continue
                    guess = float_search(cdf, log2, skip, span, off)
                    assert abs(guess - m) <= 1
                    p, lo, width, walked = corrected(cdf, log2, skip, safe, span, off, guess)
                    assert (p, lo, width) == (m, t_lo, t_hi - t_lo) and walked == m - guess
                    if guess < m:
                        short.add((m, safe))
                    elif guess > m:
                        over.add((m, safe))
    for s in ([False] if skip else [False, True]):
        most = last if skip or s else last - 1                             # the symbol at the search's end, or next to the last one
        assert {(m, s) for m in range(1, most + 1)} <= short               # fallen short of each
        assert {(m, s) for m in range(0, last)} <= over                    # and overshot from each


# ---- the decoder of four symbols between two looks ------------------------------------------------
class Reader:
    """BitReader on a stream that begins `skip` bytes after an aligned word; zeros behind it."""

    def __init__(self, data, skip):
        data = b"\xAA" * skip + data + b"\0" * (-(len(data) + skip) % 4)
        self.words = [int.from_bytes(data[i:i + 4], "big") for i in range(0, len(data), 4)]
        b0, b1, b2, self.nextw = (self.word(i) for i in range(4))
        s = 8 * skip
        self.off = (((b0 << 32 | b1) << s) & M64) >> 32
        self.win = ((b1 << 32 | b2) << s) & M64
        self.bits, self.pos = 64 - s, 4                        # bits: spare + kSymbolBits

    def word(self, i):
        return self.words[i] if i < len(self.words) else 0

    def top_up(self):
        if self.bits <= 32:
            self.win |= self.nextw << 32 >> self.bits
            self.bits += 32
            self.nextw = self.word(self.pos)
            self.pos += 1


def few_symbol(cdf, log2, skip, safe, exact, span, off):
    """decode_few_symbol's search: (symbol, T(lower), T(upper))."""
    def scaled(c):
        return (c << 16) & M32 if exact and span == 0 else mulhi(span, c << 16)
    held = 1 << (log2 - skip - 2)
    left, m, h = [cdf[4 * k] for k in range(held)], 0, held >> 1
    while h >= 1:
        up = scaled(left[h]) <= off
        m = 2 * m + up
        left = [left[h + k] if up else left[k] for k in range(h)]
        h >>= 1
    c = cdf[4 * m:4 * m + 5]
    up2 = scaled(c[2]) <= off
    t = scaled(c[3] if up2 else c[1])
    up = t <= off
    t_lo = t if up else scaled(c[2] if up2 else c[0])
    t_hi = scaled(c[4] if up2 else c[2]) if up else t
    m = 4 * m + 2 * up2 + up
    return m, t_lo, span if safe and m == (1 << log2) - 1 else t_hi


def few_decode(cdf, log2, data, n, at, skip=0, safe=True):
    """decode_few_lane: (symbols, groups decoded a second time one by one)."""
    rd, low, span, out, redone = Reader(data, at), 0, 0, [], 0
    off = rd.off

    def symbol(exact):
        nonlocal low, span, off
        m, t_lo, t_hi = few_symbol(cdf, log2, skip, safe, exact, span, off)
        low, off, width = (low + t_lo) & M32, (off - t_lo) & M32, (t_hi - t_lo) & M32
        d = (width - 1) & M32
        k = step_count(low, (low + d) & M32, d)
        interval = (low << 32 | width) << k & M64
        low, span = interval >> 32, interval & M32
        off = ((off << 32 | rd.win >> 32) << k & M64) >> 32
        rd.win = rd.win << k & M64
        rd.bits -= k
        return m

    def one_by_one():
        nonlocal low
        rd.top_up()
        assert rd.bits >= 18
        if span == 0:
            low = 0
        return symbol(True)

    while len(out) + 4 <= n:
        rd.top_up()
        kept = off, low, span, rd.bits, rd.win
        four = [symbol(False) for _ in range(4)]
        if span == 0 or rd.bits < 0:
            off, low, span, rd.bits, rd.win = kept
            four = [one_by_one() for _ in range(4)]
            redone += 1
        out += four
    while len(out) < n:
        out.append(one_by_one())
    return out, redone


# ---- the encoder of four symbols without a branch ------------------------------------------------
class FewEncoder:
    def __init__(self, cdf):
        self.cdf, self.redone, self.fours = cdf, 0, 0
        self.span = self.tail = self.out = self.waiting = self.cache = self.ones = 0
        self.words = None                                      # None: the empty held-back word is still to come

    def store(self, word):
        if self.words is None:
            assert word == 0
            self.words = []
        else:
            assert 0 <= word <= M32
            self.words.append(word)

    def release(self, carry):
        self.store(self.cache + carry)
        for _ in range(self.ones):
            self.store(0 if carry else M32)
        self.ones = 0

    def take_words(self):
        if self.waiting < 32:
            return
        self.waiting -= 32
        first = self.out >> self.waiting
        word, carry = first & M32, first >> 32
        assert carry in (0, 1) and self.waiting < 32
        self.out &= (1 << self.waiting) - 1
        if word != M32 and self.ones == 0:
            self.store(self.cache + carry)
            self.cache = word
        elif not carry and word == M32:
            self.ones += 1
        else:
            self.release(carry)
            self.cache = word

    def keep(self, k):
        self.out = (self.out << k) + (self.tail >> 32)
        self.waiting += k
        self.tail &= M32
        assert self.out < 1 << 64 and self.waiting <= 63

    def narrow(self, t_lo, t_hi):
        self.tail = (self.tail + t_lo) & M64
        width = (t_hi - t_lo) & M32
        d, low = (width - 1) & M32, self.tail & M32
        n = step_count(low, (low + d) & M32, d)
        self.tail = self.tail << n & M64
        self.span = width << n & M32
        return n

    def bounds(self, s, exact):
        def t(c):
            return c << 16 if exact and self.span == 0 else mulhi(self.span, c << 16)
        return t(self.cdf[s]), self.span if s == len(self.cdf) - 2 else t(self.cdf[s + 1])

    def put_one(self, s):
        assert self.waiting <= 31
        self.keep(self.narrow(*self.bounds(s, True)))
        self.take_words()

    def put_four(self, symbols):
        kept, most, k = (self.tail, self.span), min(63 - self.waiting, 31), 0
        for s in symbols:
            k += self.narrow(*self.bounds(s, False))
        self.fours += 1
        if self.span == 0 or k > most:
            self.tail, self.span = kept
            self.take_words()
            for s in symbols:
                self.put_one(s)
            self.redone += 1
            k = 0
        self.keep(k)

    def encode(self, symbols):
        full = len(symbols) // 8 * 8
        for i in range(0, full, 8):
            self.put_four(symbols[i:i + 4])
            self.put_four(symbols[i + 4:i + 8])
            self.take_words()
        for s in symbols[full:]:
            self.put_one(s)
        self.tail = self.tail + 0x40000000 << 2
        self.keep(2)
        self.take_words()
        nbits = self.waiting & 31
        self.release(self.out >> nbits)
        part = (self.out & (1 << nbits) - 1) << 32 - nbits & M32 if nbits else 0
        return b"".join(w.to_bytes(4, "big") for w in self.words) + part.to_bytes(4, "big")[:(nbits + 7) // 8]


def streams(rng, nsym):
    """(table, symbols): likely and rare symbols, the last one, full ranges again and again, runs of carries."""
    kind = rng.randrange(5)
    n = rng.choice([1, 3, 4, 5, 8, 11, 64, 100, 256])
    if kind == 0:                                              # every interval scales back to the full range
        step = 65536 // nsym
        cdf = [i * step for i in range(nsym)] + [65535]
        return cdf, [rng.randrange(nsym) for _ in range(n)]
    cdf = random_table(rng, nsym, rng.choice([0.5, 1, 3, 8]) if kind != 1 else 200)
    hot = max(range(nsym), key=lambda s: cdf[s + 1] - cdf[s])
    if kind == 1:                                              # next to no bits, then 16 a symbol
        return cdf, [hot if rng.random() < 0.9 else rng.randrange(nsym) for _ in range(n)]
    if kind == 2:
        return cdf, [rng.randrange(nsym) for _ in range(n)]
    if kind == 3:
        return cdf, [nsym - 1 if rng.random() < 0.5 else rng.randrange(nsym) for _ in range(n)]
    return cdf, [rng.choice([0, nsym // 2, nsym // 2, nsym - 1]) for _ in range(n)]


@pytest.mark.parametrize("log2", [4, 5, 6])
def test_four_at_a_time_equals_the_bit_serial_coder(log2):
    rng = random.Random(log2)
    fours = enc_redone = dec_redone = groups = 0
    for _ in range(300):
        cdf, symbols = streams(rng, 1 << log2)
        want, _ = pycoder.encode(cdf, symbols)
        enc = FewEncoder(cdf)
        assert enc.encode(symbols) == want
        got, redone = few_decode(cdf, log2, want, len(symbols), rng.randrange(4))
        assert got == symbols
        fours, enc_redone = fours + enc.fours, enc_redone + enc.redone
        dec_redone, groups = dec_redone + redone, groups + len(symbols) // 4
    assert 100 < enc_redone < fours - 100 and 100 < dec_redone < groups - 100          # both ways are taken


@pytest.mark.parametrize("log2", [4, 5, 6])
def test_four_at_a_time_in_the_lower_half(log2):
    """The search over the lower half of the table, the last symbol's bound left out."""
    rng = random.Random(7 * log2)
    half = 1 << log2 - 1
    for _ in range(100):
        low = random_table(rng, half + 1, rng.choice([1, 3, 8]))
        cdf = [min(c, 65535 - half) for c in low[:-1]] + list(range(65536 - half, 65536))
        if any(b <= a for a, b in zip(cdf, cdf[1:])):
            continue
        symbols = [rng.randrange(half) for _ in range(rng.choice([4, 9, 64, 256]))]
        want, _ = pycoder.encode(cdf, symbols)
        assert FewEncoder(cdf).encode(symbols) == want
        assert few_decode(cdf, log2, want, len(symbols), rng.randrange(4), skip=1, safe=False)[0] == symbols
