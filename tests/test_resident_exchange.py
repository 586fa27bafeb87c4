"""A host model of the resident solver's exchange (wot_amd/csrc/resident.hip): every
workgroup is the list of its loads and stores of exchanged words, in program order, and a
scheduler delays workgroups at will.  A load of an empty word waits, a load of a word that
another step left is an error, and a schedule in which everybody waits is a stall."""
import random

import pytest

KSUMS = 8


class Rules:
    """What the kernel does; the defects the model has to see are variants of it."""
    words_emptied = staticmethod(lambda n: KSUMS)   # of the next check's sums, at a check of n values
    read_all = False        # workgroups without rows on a side take the other side's potentials too
    flag_buffers = 3        # of the tau check's maxima


class NarrowSums(Rules):
    words_emptied = staticmethod(lambda n: n)


class ReadAll(Rules):
    read_all = True


class TwoFlagBuffers(Rules):
    flag_buffers = 2


def program(wg, own, steps, rules):
    """Loads ('r', word, tag) and stores ('w', word, tag or None: emptied) of one workgroup."""
    n_wg = len(own)
    f_own, g_own = [w for w in range(n_wg) if own[w][0]], [w for w in range(n_wg) if own[w][1]]
    has_f, has_g = own[wg]
    ops = []
    it = chk = published = 0
    flags_open = False
    tau = any(s != 'iterate' for s in steps)  # the duality-gap schedule

    def sums(n):
        nonlocal chk
        chk += 1
        for q in range(rules.words_emptied(n)):
            ops.append(('w', ('s', (chk + 1) % 3, wg, q), None))
        for q in range(n):
            ops.append(('w', ('s', chk % 3, wg, q), chk))
        for q in range(n):
            for b in range(n_wg):
                ops.append(('r', ('s', chk % 3, b, q), chk))

    def absorb():
        nonlocal flags_open
        if flags_open:
            for b in range(n_wg):
                ops.append(('r', ('t', published % rules.flag_buffers, b), published))
        flags_open = False

    for step in steps:
        if step == 'iterate':
            it += 1
            p, old = it % 2, (it - 1) % 2
            if it > 1 and (has_f or rules.read_all):
                for b in g_own:
                    ops.append(('r', ('g', old, b), it - 1))
            absorb()
            if has_f:
                if it > 1:
                    ops.append(('w', ('f', old, wg), None))
                ops.append(('w', ('f', p, wg), it))
            if has_g or rules.read_all:
                for b in f_own:
                    ops.append(('r', ('f', p, b), it))
            if has_g and it > 1:
                ops.append(('w', ('g', old, wg), None))
            if rules.flag_buffers == 2 and tau and it > 1:
                ops.append(('w', ('t', old, wg), None))
            if has_g:
                ops.append(('w', ('g', p, wg), it))
            if tau:
                if rules.flag_buffers == 3:
                    ops.append(('w', ('t', (it + 1) % 3, wg), None))
                ops.append(('w', ('t', it % rules.flag_buffers, wg), it))
                flags_open, published = True, it
        elif step == 'duality':
            absorb()
            for b in g_own:
                ops.append(('r', ('g', it % 2, b), it))
            for b in f_own:
                ops.append(('r', ('f', it % 2, b), it))
            sums(7)
        else:  # a check of so many sums
            absorb()
            sums(step)
    return ops


def run(progs, pick):
    """None when every workgroup ends; else what went wrong.  pick(runnable) names the next one."""
    mem, at = {}, [0] * len(progs)
    waiting = set()
    while True:
        live = [w for w in range(len(progs)) if at[w] < len(progs[w])]
        if not live:
            return None
        runnable = [w for w in live if w not in waiting]
        if not runnable:
            return 'stall'
        w = pick(runnable)
        kind, word, tag = progs[w][at[w]]
        if kind == 'w':
            mem[word] = tag
            waiting = {v for v in waiting if progs[v][at[v]][1] != word}
        else:
            seen = mem.get(word)
            if seen is None:
                waiting.add(w)
                continue
            if seen != tag:
                return 'stale'
        at[w] += 1


def outcomes(own, steps, rules):
    progs = [program(w, own, steps, rules) for w in range(len(own))]
    bad = set()
    for late in range(len(own)):
        # a workgroup that only moves when nobody else can, from each of its steps on
        for start in range(0, len(progs[late]), 3):
            ahead = [0]

            def pick(runnable):
                others = [w for w in runnable if w != late]
                if late in runnable and (not others or ahead[0] < start):
                    ahead[0] += 1
                    return late
                return others[ahead[0] % len(others)]
            bad.add(run(progs, pick))
    rng = random.Random(5)
    for _ in range(200):
        weight = [rng.choice((1, 1, 40)) for _ in own]
        bad.add(run(progs, lambda r: rng.choices(r, [weight[w] for w in r])[0]))
    return bad - {None}


# two evolution checks, the sum of K-tilde, two duality checks
GAP = (['iterate'] * 3 + [4]) * 2 + [1] + ['iterate'] * 2 + ['duality'] + ['iterate'] * 2 + ['duality']


FIXED = ['iterate'] * 7
# workgroups 2 and 3 without rows of C (300 x 400, 900 x 8000), without rows of C^T
WIDE = [(True, True)] * 2 + [(False, True)] * 2
TALL = [(True, True)] * 2 + [(True, False)] * 2


def test_sums_of_checks_of_different_widths():
    own = [(True, True)] * 4
    assert outcomes(own, GAP, Rules) == set()
    assert 'stale' in outcomes(own, GAP, NarrowSums)


@pytest.mark.parametrize('own', [WIDE, TALL, [(True, True), (False, True)], [(True, False), (True, True)]])
@pytest.mark.parametrize('steps', [FIXED, GAP])
def test_workgroups_without_rows_on_a_side(own, steps):
    assert outcomes(own, steps, Rules) == set()


@pytest.mark.parametrize('own,steps', [(WIDE, FIXED), (WIDE, GAP), (TALL, FIXED)])
def test_reading_what_one_does_not_need_stalls(own, steps):
    assert 'stall' in outcomes(own, steps, ReadAll)


def test_two_buffers_of_maxima_stall():
    assert 'stall' in outcomes(WIDE, GAP, TwoFlagBuffers)
