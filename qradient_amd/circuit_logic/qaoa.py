"""QAOA circuit on the GPU (reference qradient/circuit_logic/qaoa.py:8-70).

|+>^n, then per layer exp(-i gamma_i C) and RX(beta_i) on every qubit, with C
the z / zz part of the observable (state.py:261-297).  ``grad_run(betas,
gammas)`` returns (E, grad[p, 2]), column 0 = dE/d beta_i, column 1 =
dE/d gamma_i.  Unlike the reference, an ``ini_state`` array is copied, never
mutated.
"""
import ctypes
import warnings

import numpy as np

from .. import _native
from ..physical_components import Gates
from .base import ParametrizedCircuit, draw_uniforms, sample_projectors

# Shots of shifted circuits that are in memory at once (20 bytes each on the
# host): with more, the circuits are drawn and run in groups.
SHOT_GROUP = 1 << 24


class Qaoa(ParametrizedCircuit):
    def __init__(self, qubit_number, observable, layer_number, **kwargs):
        backend = ParametrizedCircuit.split_backend(kwargs)
        if kwargs:
            raise TypeError('unexpected keyword arguments: {}'.format(sorted(kwargs)))
        ParametrizedCircuit.init(self, qubit_number, observable, False, backend)
        self._gates = Gates(self.qnum).add_xrots().add_x_summed() \
            .add_classical_ham(self.observable, include_individual_components=True)
        self.lnum = int(layer_number)
        self.state_history = None
        self.has_loaded_eigensystem = False

    def _init_state(self, st):
        st.reset('+')  # uniform superposition (qaoa.py:17)

    def __check_parameters(self, betas, gammas):
        """qaoa.py:186-191."""
        betas = np.asarray(betas, dtype=np.float64)
        gammas = np.asarray(gammas, dtype=np.float64)
        if (betas.size != self.lnum) or (gammas.size != self.lnum):
            raise ValueError(('Wrong amount of parameters. Expected {} and {},'.format(self.lnum, self.lnum),
                              ' found {} and {}.'.format(betas.size, gammas.size)))
        return np.ascontiguousarray(betas.ravel()), np.ascontiguousarray(gammas.ravel())

    def _get_plan(self):
        if self._plan is None:
            h = ctypes.c_void_p()
            _native.call('qg_qaoa_plan', self.context().handle, self.qnum, self.lnum,
                         _native.DTYPES[self.dtype], 1, ctypes.byref(h))
            self._plan = h
        return self._plan

    def _terms(self):
        terms = self.observable.classical_terms()
        arr, k = _native.terms_array(terms)
        off = np.array([0, k], dtype=np.int32)
        return arr, off

    def grad_run(self, betas, gammas, hide_progbar=True, ini_state=None):
        """(E, grad[p, 2]): qaoa.py:40-70."""
        betas, gammas = self.__check_parameters(betas, gammas)
        arr, off = self._terms()
        E = np.empty(1)
        grad = np.empty((self.lnum, 2), dtype='double')
        if ini_state is None:
            _native.call('qg_qaoa_grad_run', self._get_plan(), 1, arr, _native.iptr(off), _native.dptr(betas),
                         _native.dptr(gammas), _native.dptr(E), _native.dptr(grad))
        else:
            # the library only reads ini_state (the reference scales it in place)
            _keep, ini = self._ini(ini_state, self.qnum)
            _native.call('qg_qaoa_grad_run_ini', self._get_plan(), 1, arr, _native.iptr(off), _native.dptr(betas),
                         _native.dptr(gammas), ini, _native.dptr(E), _native.dptr(grad))
        self._plan_state = False
        return np.float64(E[0]), grad

    def sample_grad(self, betas, gammas, shot_num=1, hide_progbar=True, exact_expec_val=True, ini_state=None):
        """Not implemented in the reference either (qaoa.py:72-81): warns and
        returns None."""
        warnings.warn('Not implemented yet.')

    def sample_grad_dense(self, betas, gammas, shot_num=1, hide_progbar=True, exact_expec_val=True,
                          ini_state=None):
        """(E, grad[p, 2]) from finite-shot measurements of shifted circuits
        in the computational basis (qaoa.py:83-158).

        For layer i: each classical-Hamiltonian component C_j phase-shifted by
        exp(-+i pi/4 C_j) after the cost phase gives grad[i, 1] = sum_j
        (o_plus_j - o_minus_j); each qubit's mixer rotation shifted by +-pi/2
        gives grad[i, 0] = sum_q (o_plus_q - o_minus_q) / 2.  An estimate o is
        the mean of C(x) over shot_num basis draws of the shifted circuit's
        final state.  The reference carries each suffix circuit as a dense
        left-hand-side matrix; here the shifted copies of a layer's stored
        states run the rest of the circuit on the device together, and are
        sampled there by the inverse CDF at uniforms drawn on the host in the
        reference's order.  E is <C> (or, with exact_expec_val=False, the
        shot estimate of the whole observable).  The reference mutates
        ``ini_state``; it is only read here."""
        betas, gammas = self.__check_parameters(betas, gammas)
        n, L = self.qnum, self.lnum
        cterms = self.observable.classical_terms()
        arr, k = _native.terms_array(cterms)
        C = self._classical_values(cterms)
        _keep, ini = self._ini(ini_state, n)
        terms = cterms if exact_expec_val else self.observable.terms
        w = np.array([t[3] for t in terms])
        shots = int(shot_num)
        # draws in the reference's order: E's shots, then per layer each
        # component's two circuits and each qubit's
        u_E = None if exact_expec_val else draw_uniforms(len(terms), shots)
        m_arr, m = _native.terms_array(terms)
        expec = np.empty(m + 1)
        total = L * 2 * (k + n)
        o = np.empty(total)
        group = max(1, SHOT_GROUP // max(1, shots))
        for first in range(0, total, group):
            u = draw_uniforms(min(group, total - first), shots)
            if shots == 0:
                u = np.zeros((u.shape[0], 1))  # no shots: E alone, the estimates are nan
            idx = np.empty(u.shape, dtype=np.int32)
            _native.call('qg_qaoa_shift_sample_part', self._get_plan(), arr, k, _native.dptr(betas),
                         _native.dptr(gammas), ini, m_arr, m, None if first else _native.dptr(expec), first,
                         u.shape[0], u.shape[1], _native.dptr(u), _native.iptr(idx))
            o[first:first + u.shape[0]] = C[idx[:, :shots]].mean(axis=1)
        if exact_expec_val:
            E = np.float64((w * expec[:m]).sum())
        else:
            E = sample_projectors(.5 * (expec[m] + expec[:m]), w, shots, uniforms=u_E)
        o = o.reshape(L, k + n, 2)
        diff = o[:, :, 0] - o[:, :, 1]
        grad = np.empty((L, 2), dtype='double')
        for i in range(L):
            # summed component by component and qubit by qubit, in order
            grad[i, 0] = .5 * sum(diff[i, k:].tolist(), 0.)
            grad[i, 1] = sum(diff[i, :k].tolist(), 0.)
        return E, grad

    def _classical_values(self, cterms):
        """C(x) in natural order, summed in term order (state.py:273-294)."""
        n = self.qnum
        x = np.arange(2 ** n, dtype=np.int64)
        C = np.zeros(2 ** n)
        for kind, i, j, w in cterms:
            s = 1.0 - 2.0 * ((x >> (n - 1 - i)) & 1)
            if kind == _native.TERM_ZZ:
                s = s * (1.0 - 2.0 * ((x >> (n - 1 - j)) & 1))
            C = C + w * s
        return C

    def run_expec_val(self, betas, gammas, hide_progbar=True, exact_expec_val=True, shot_num=1, ini_state=None):
        """Forward circuit, then the exact expectation or, with
        exact_expec_val=False, its shot_num-shot estimate (qaoa.py:23-38)."""
        betas, gammas = self.__check_parameters(betas, gammas)
        arr, off = self._terms()
        E = np.empty(1)
        if ini_state is None:
            _native.call('qg_qaoa_expec_val', self._get_plan(), 1, arr, _native.iptr(off), _native.dptr(betas),
                         _native.dptr(gammas), _native.dptr(E))
        else:
            _keep, ini = self._ini(ini_state, self.qnum)
            _native.call('qg_qaoa_expec_val_ini', self._get_plan(), 1, arr, _native.iptr(off), _native.dptr(betas),
                         _native.dptr(gammas), ini, _native.dptr(E))
        self._plan_state = True
        if not exact_expec_val:
            return self.sample_expec_val(shot_num)
        return np.float64(E[0])
