"""The PMM model of one tree evaluated state by state in long double, whose range
(1e-4932) holds the likelihood of a site of a few hundred leaves without
scaling: posteriors of every node, expected counts of every branch, likelihoods
of the sites."""
import numpy as np

LD = np.longdouble


def evaluate(t, Q, codes, lengths, nu, phi):
    """(post0, postS [node, site], counts [node, 5], log-likelihood [site]) by
    post-order nodes; codes: rows of the leaves in post-order, 0 unedited, 1..m
    edits, -1 missing, -2 silenced."""
    N, K = len(t.parent), codes.shape[1]
    row = {int(v): i for i, v in enumerate(np.nonzero(np.asarray(t.c0) < 0)[0])}
    x, nu, phi = np.asarray(lengths, dtype=LD), LD(nu), LD(phi)
    stay, keep = np.exp(-(1 + nu) * x), np.exp(-nu * x)
    edit, sil = -np.expm1(-x) * keep, -np.expm1(-nu * x)
    post0, postS, counts, llh = np.zeros((N, K), LD), np.zeros((N, K), LD), np.zeros((N, 5), LD), np.zeros(K, LD)
    for k in range(K):
        m = len(Q[k])
        q = np.array([Q[k][j + 1] for j in range(m)], dtype=LD)
        below, edge, top = np.zeros((N, m + 2), LD), np.zeros((N, m + 2), LD), np.zeros((N, m + 2), LD)
        for v in range(N):
            b = below[v]
            if t.c0[v] < 0:
                c = codes[row[v], k]
                if c >= 0:
                    b[c] = 1 - phi
                else:
                    b[m + 1] = 1
                    if c == -1:
                        b[:m + 1] = phi
            else:
                b[:] = edge[t.c0[v]] * edge[t.c1[v]]
            edge[v, 0] = stay[v] * b[0] + edit[v] * (q * b[1:m + 1]).sum() + sil[v] * b[m + 1]
            edge[v, 1:m + 1] = keep[v] * b[1:m + 1] + sil[v] * b[m + 1]
            edge[v, m + 1] = b[m + 1]
        llh[k] = np.log(edge[N - 1, 0])
        top[N - 1, 0] = 1 / edge[N - 1, 0]
        for v in range(N - 1, -1, -1):
            b, a = below[v], top[v]
            counts[v] += [a[0] * stay[v] * b[0], a[0] * edit[v] * (q * b[1:m + 1]).sum(), a[0] * sil[v] * b[m + 1],
                          keep[v] * (a[1:m + 1] * b[1:m + 1]).sum(), sil[v] * a[1:m + 1].sum() * b[m + 1]]
            here = np.zeros(m + 2, LD)
            here[0] = a[0] * stay[v]
            here[1:m + 1] = a[1:m + 1] * keep[v] + a[0] * edit[v] * q
            here[m + 1] = a[m + 1] + sil[v] * a[:m + 1].sum()
            post0[v, k], postS[v, k] = here[0] * b[0], here[m + 1] * b[m + 1]
            if t.c0[v] >= 0:
                top[t.c0[v]], top[t.c1[v]] = here * edge[t.c1[v]], here * edge[t.c0[v]]
    return post0, postS, counts, llh
