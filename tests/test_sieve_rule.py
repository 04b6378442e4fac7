"""The rule by which the sieve path's finish (rs_sieve.h: other_threshold, shift_of) takes a token that it picked with an approximate total, in whole
numbers of any size: whenever it says that the token is certain, every total within the error picks the same one."""
import random


def _pick(weights, order, top_k, P, u_num, u_den):
    """(token, above, n_gt, n_eq, w_thr, w_tie, r, run, own): threshold, tie weight and pick of one row for the mass P, as the oracle has them."""
    mass, count, i = 0, 0, 0
    while True:
        w = weights[order[i]]
        j = i
        while j < len(order) and weights[order[j]] == w:
            j += 1
        if count + (j - i) >= top_k or mass + w * (j - i) >= P or j == len(order):
            break
        mass += w * (j - i)
        count += j - i
        i = j
    n_gt, n_eq = count, j - i
    w_tie = min(w, max(P - mass, 0) // n_eq, w * max(top_k - n_gt, 0) // n_eq)
    if w_tie == 0 and mass == 0:
        w_tie = 1
    S = mass + n_eq * w_tie
    r = S * u_num // u_den + 1 if u_num < u_den else S
    run = 0
    for t, x in enumerate(weights):
        own = x if x > w else w_tie if x == w else 0
        if run < r <= run + own:
            return t, mass, n_gt, n_eq, w, w_tie, r, run, own
        run += own
    raise AssertionError


def _certain(pick, err, least, most, top_k, n):
    t, above, n_gt, n_eq, w, w_tie, r, run, own = pick
    down = above + w * n_eq
    other = (n_gt > 0 and not above < least) or (n_gt + n_eq < top_k and not down >= most)
    if other:
        shift = err + 2 * n + 2
    elif least >= above + w_tie * n_eq + n_eq or (w_tie == w and least >= down):
        shift = 0
    else:
        shift = err + n_eq + 2
    return min(r - run - 1, run + own - r) >= shift, other


def test_a_token_that_is_called_certain_is_picked_by_every_total():
    rng = random.Random(5)
    certain = others = moved = 0
    for row in range(3000):
        n = rng.choice([1, 2, 3, 5, 9, 20, 40])
        scale = rng.choice([30, 1000, 10 ** 6, 10 ** 9])
        weights = [max(1, int(scale * 2.0 ** rng.uniform(-rng.choice([0, 3, 12, 25]), 0))) for _ in range(n)]
        if rng.random() < 0.4:
            weights = [rng.choice(weights[: 1 + n // 4]) for _ in weights]                 # ties
        order = sorted(range(n), key=lambda t: -weights[t])
        total = sum(weights)
        for _ in range(12):
            top_k = rng.choice([1, 2, n, n, max(1, n // 2)])
            P = max(1, min(total, int(total * rng.choice([rng.random(), 1 - rng.random() ** 4 / 100, 1.0]))))
            err = max(1, int(total * 2.0 ** -rng.uniform(1, 30)))
            u_den = 1 << 64
            u_num = rng.choice([0, u_den, u_den - 1, rng.randrange(u_den), rng.randrange(u_den)])
            picks = [(_pick(weights, order, top_k, P, u_num, u_den), err, max(P - err, 0), P + err)]
            # (lists of more than 64 tokens: the threshold of the largest P, which the exact one is below by less than twice the error)
            top = _pick(weights, order, top_k, P + err, u_num, u_den)
            if top[2] and top[1] >= max(P - err, 0):
                picks.append((top, 2 * err, max(P - err, 0), P + err))
            for pick, e, least, most in picks:
                sure, other = _certain(pick, e, least, most, top_k, n)
                certain += sure
                others += sure and other
                for q in [P, max(1, P - err + 1), P + err - 1] + [rng.randint(max(1, P - err + 1), P + err - 1) for _ in range(4)]:
                    got = _pick(weights, order, top_k, q, u_num, u_den)[0]
                    moved += got != pick[0]
                    assert not sure or got == pick[0], (weights, top_k, P, err, u_num, q)
    print("certain %d, of them with another threshold possible %d; totals that pick another token %d" % (certain, others, moved))
    assert certain > 1000 and others > 300 and moved > 1000
