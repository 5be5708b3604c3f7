"""Deferred epilogues: dot() holds its launch back and the add_col_vec / activation / sample calls
that follow it on its own target run in the product's epilogue; an in-place mult_by_scalar is held
back likewise and the add_mult / add_mult_sign calls of a parameter update (deepnet/parameter.py:80-106)
are folded into one pass.  Every sequence here is run with
the deferral switched off (each call its own launch) and on, and must leave the same bits in every
matrix it touches and the same generator state; sequences that must NOT be folded (another
matrix in between, a second bias, operands that change between the calls, reads, frees) are
checked the same way."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _f(a):
    return np.asarray(a, dtype=np.float32, order='F')


def _bits(m):
    return m.asarray().view(np.uint32).copy()


SHAPES = [(500, 784, 100, True), (784, 500, 100, False), (1024, 784, 128, True), (10, 1024, 128, True), (33, 17, 5, False),
          (2048, 128, 2048, True), (64, 4096, 64, True), (3, 2, 2, False),       # m, k, n, first operand transposed
          (1409, 705, 1537, True)]                                               # (k_gemm_split: tests/test_ring_plans.py)


def _run(cm, deferred, seq, shape, seed):
    m, k, n, ta = shape
    rng = np.random.default_rng(seed)
    cm.set_deferred_epilogues(deferred)
    cm.CUDAMatrix.init_random(7)
    A = cm.CUDAMatrix(_f(rng.standard_normal((k, m) if ta else (m, k)) * 0.1))
    B = cm.CUDAMatrix(_f(rng.standard_normal((k, n))))
    bias = cm.CUDAMatrix(_f(rng.standard_normal((m, 1))))
    other = cm.CUDAMatrix(_f(rng.standard_normal((m, n))))
    T, S = cm.empty((m, n)), cm.empty((m, n))
    T.assign(-3.0); S.assign(-4.0)
    a = A.T if ta else A
    out = seq(cm, a, B, bias, other, T, S)
    after = cm.empty((64, 48)); after.fill_with_rand()            # the generator's state shows in its next draws
    res = [_bits(x) for x in (T, S, other, bias, after)] + ([out] if out is not None else [])
    cm.set_deferred_epilogues(True)
    return res


def seq_sigmoid(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.apply_sigmoid()


def seq_sigmoid_sample(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.apply_sigmoid(); T.sample_bernoulli(target=S)


def seq_relu(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.lower_bound(0)


def seq_tanh(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); cm.tanh(T)


def seq_no_bias(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.apply_sigmoid(); T.sample_bernoulli(target=S)


def seq_bias_only_then_read(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias)
    return T.asarray().view(np.uint32).copy()                   # the read launches what is held back


def seq_dot_alone_then_other_work(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); other.mult(T); T.apply_sigmoid()     # the sigmoid is an ordinary launch


def seq_bias_on_another_matrix(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); other.add_col_vec(bias); T.add_col_vec(bias); T.apply_sigmoid()


def seq_two_biases(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.add_col_vec(bias); T.apply_sigmoid(); T.apply_sigmoid()


def seq_bias_changes_in_between(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); bias.mult(2.0); T.apply_sigmoid(); bias.add(1.0); T.sample_bernoulli(target=S)


def seq_operand_changes_in_between(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); B.mult(0.5); T.add_col_vec(bias); cm.tanh(T)


def seq_sigmoid_into_another_target(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.apply_sigmoid(target=S); S.sample_bernoulli(target=other)


def seq_sample_in_place(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.apply_sigmoid(); T.sample_bernoulli()      # target = self: not folded


def seq_scaled_and_accumulating_products(cm, a, B, bias, other, T, S):
    cm.dot(a, B, mult=0.5, target=T); T.add_col_vec(bias); T.apply_sigmoid()             # alpha != 1: launched at once
    S.add_dot(a, B); S.add_col_vec(bias); S.lower_bound(0)


def seq_two_products_in_a_row(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); cm.dot(a, B, target=S); S.add_col_vec(bias); S.apply_sigmoid(); T.add_col_vec(bias); T.lower_bound(0)


def seq_free_while_held_back(cm, a, B, bias, other, T, S):
    tmp = cm.empty(T.shape)
    cm.dot(a, B, target=tmp); tmp.add_col_vec(bias)
    tmp.free_device_memory()                                     # launches (into memory that is then given back)
    again = cm.empty(T.shape); again.assign(1.5); T.add(again)


def seq_lower_bound_not_zero(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.lower_bound(0.25)


# ---- the parameter update of deepnet/parameter.py:80-106 (w = T, w_delta = S, gradient = other)

def _params(T, S, other):
    T.assign(0.25); S.assign(-0.5)                      # (the harness fills them with constants: make them vary)
    T.add(other); S.subtract(other)
    return T, S, other


def seq_update_plain(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); wd.add_mult(g); w.add_mult(wd, -0.01)


def seq_update_with_reset(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); wd.add_mult(g); w.add_mult(wd, -0.01); g.assign(0)


def seq_update_l2_l1_reset(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.5); wd.add_mult(w, 0.001); wd.add_mult_sign(w, 0.0005); wd.add_mult(g); w.add_mult(wd, -0.1); g.assign(0)


def seq_update_l2_only(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.5); wd.add_mult(w, 0.001); wd.add_mult(g); w.add_mult(wd, -0.1); g.assign(1.0)     # (not a reset)


def seq_update_l1_only_twice(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    for _ in range(2):
        wd.mult(0.5); wd.add_mult_sign(w, 0.0005); wd.add_mult(g); w.add_mult(wd, -0.1)


def seq_update_not_spelled_scaled_gradient(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); wd.add_mult(g, 0.5); w.add_mult(wd, -0.01); g.assign(0)


def seq_update_not_spelled_wrong_order(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); wd.add_mult(g); wd.add_mult(w, 0.001); w.add_mult(wd, -0.01)


def seq_update_not_spelled_no_gradient(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); wd.add_mult(w, 0.001); w.add_mult(wd, -0.01)


def seq_update_interrupted(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); g.mult(2.0); wd.add_mult(g); w.add_mult(wd, -0.01); wd.mult(0.5); bias.mult(3.0); wd.add_mult(g)


def seq_update_reads_another_matrix(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); wd.add_mult(g); w.add_mult(g, -0.01); w.add_mult(wd, -0.01)


def seq_update_too_many_terms(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); wd.add_mult(w, 0.001); wd.add_mult_sign(w, 0.0005); wd.add_mult(g); wd.add_mult(g); w.add_mult(wd, -0.01)


def seq_update_then_product(cm, a, B, bias, other, T, S):
    w, wd, g = _params(T, S, other)
    wd.mult(0.9); wd.add_mult(g); w.add_mult(wd, -0.01)
    cm.dot(a, B, target=g); g.add_col_vec(bias); g.apply_sigmoid(); wd.mult(0.5); wd.add_mult(g); w.add_mult(wd, 0.3); g.assign(0)


def seq_scale_alone_then_read(cm, a, B, bias, other, T, S):
    T.assign(2.0); T.add(other); T.mult(0.5)
    return T.asarray().view(np.uint32).copy()


# ---- the dropout mask of deepnet/neuralnet.py:194-198 (mask = S, state = T)

def seq_dropout(cm, a, B, bias, other, T, S):
    T.add(other); S.fill_with_rand(); S.greater_than(0.5); T.mult(S)


def seq_dropout_after_a_layer(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.lower_bound(0); S.fill_with_rand(); S.greater_than(0.3); T.mult(S)
    other.fill_with_rand(); other.greater_than(0.7); T.mult(other)


def seq_layer_mask_for_another_matrix(cm, a, B, bias, other, T, S):
    # the mask that follows the layer is meant for another matrix: the layer comes first, then the masking
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.lower_bound(0); S.fill_with_rand(); S.greater_than(0.3); other.mult(S); other.add(T)


def seq_layer_mask_unfinished(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.lower_bound(0); S.fill_with_rand(); other.add(T); S.greater_than(0.5); T.mult(S)


def seq_layer_mask_is_an_operand(cm, a, B, bias, other, T, S):
    # the mask is drawn into the matrix the product reads: the product must see the old values
    cm.dot(a, B, target=T); T.lower_bound(0); B.fill_with_rand(); B.greater_than(0.5); cm.dot(a, B, target=S)


def seq_layer_mask_then_sample(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.lower_bound(0); S.fill_with_rand(); S.greater_than(0.5); T.mult(S)
    T.apply_sigmoid(); T.sample_bernoulli(target=other)


def seq_two_layers_with_masks(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.lower_bound(0); S.fill_with_rand(); S.greater_than(0.5); T.mult(S)
    cm.dot(a, B, target=other); other.lower_bound(0); S.fill_with_rand(); S.greater_than(0.25); other.mult(S)


def seq_layer_without_mask_then_draw(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.lower_bound(0); other.fill_with_randn(); S.fill_with_rand()


# the hidden sample as cudamat/examples/rbm_cudamat.py:63-65 spells it: r.fill_with_rand(); r.less_than(h, target=h)
def seq_sample_by_uniforms(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.apply_sigmoid(); S.fill_with_rand(); S.less_than(T, target=T)


def seq_sample_by_uniforms_into_another_target(cm, a, B, bias, other, T, S):
    T.apply_sigmoid(); S.fill_with_rand(); S.less_than(T, target=other); S.fill_with_rand(); T.less_than(S, target=S)


def seq_sample_by_uniforms_behind_a_relu_layer(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.lower_bound(0); S.fill_with_rand(); S.less_than(T, target=T); other.fill_with_rand()


def seq_sample_by_uniforms_of_itself(cm, a, B, bias, other, T, S):
    S.fill_with_rand(); S.less_than(S, target=S); T.fill_with_rand(); T.less_than(other)


def seq_dropout_mask_then_read(cm, a, B, bias, other, T, S):
    S.fill_with_rand(); S.greater_than(0.25)
    return S.asarray().view(np.uint32).copy()


def seq_dropout_into_another_target(cm, a, B, bias, other, T, S):
    T.add(other); S.fill_with_rand(); S.greater_than(0.5); T.mult(S, target=other)


def seq_dropout_threshold_into_another_target(cm, a, B, bias, other, T, S):
    T.add(other); S.fill_with_rand(); S.greater_than(0.5, target=other); T.mult(S)


def seq_dropout_mask_times_itself(cm, a, B, bias, other, T, S):
    S.fill_with_rand(); S.greater_than(0.5); S.mult(S); T.fill_with_rand(); T.mult(T)


def seq_dropout_roles_exchanged(cm, a, B, bias, other, T, S):
    T.add(other); S.fill_with_rand(); S.greater_than(0.5); S.mult(T)


def seq_fill_then_other_work(cm, a, B, bias, other, T, S):
    S.fill_with_rand(); T.add(S); S.greater_than(0.5); T.mult(S)


def seq_dropout_of_special_values(cm, a, B, bias, other, T, S):
    T.assign(-0.0); other.assign(float('inf')); T.add_mult(other, -1.0)        # -inf everywhere: times a zero of the mask is NaN
    S.fill_with_rand(); S.greater_than(0.5); T.mult(S)


def seq_fill_then_another_draw(cm, a, B, bias, other, T, S):
    # the generator's state moves to its other buffer in large calls: the second call must see the first one's
    S.fill_with_rand(); T.assign(0.5); T.sample_bernoulli(target=other); S.fill_with_rand(); T.fill_with_randn()
    S.fill_with_rand(); S.greater_than(0.5); other.sample_bernoulli()


# the backward pass of a layer of rectified linear units: deriv = dot(w, deriv_above);
# deriv.apply_rectified_linear_deriv(state)  (deepnet/neuralnet.py:203-222, layer.py:168-172)
def seq_relu_deriv(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.apply_rectified_linear_deriv(other)


def seq_masked_relu_deriv(cm, a, B, bias, other, T, S):
    # ... of a layer with dropout: deriv.mult(mask) in between (neuralnet.py:212-213)
    S.fill_with_rand(); S.greater_than(0.5); cm.dot(a, B, target=T); T.mult(S); T.apply_rectified_linear_deriv(other)


def seq_masked_deriv_without_activation(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.mult(other); S.add(T)


def seq_factor_then_bias(cm, a, B, bias, other, T, S):
    # a bias behind the factor is not the layer's sequence: nothing may be reordered
    cm.dot(a, B, target=T); T.mult(other); T.add_col_vec(bias); T.apply_sigmoid()


def seq_factor_twice(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.mult(other); T.mult(other); T.apply_rectified_linear_deriv(S)


def seq_factor_is_the_target(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.mult(T); T.apply_rectified_linear_deriv(other)


def seq_factor_into_another_target(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.mult(other, target=S); T.apply_rectified_linear_deriv(S)


def seq_factor_then_lower_bound(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.mult(other); T.lower_bound(0); S.fill_with_rand(); S.greater_than(0.5); T.mult(S)


def seq_relu_deriv_then_other_work(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.apply_rectified_linear_deriv(other); T.mult(0.5); other.add(T)


def seq_relu_deriv_into_another_target(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.apply_rectified_linear_deriv(other, target=S)


def seq_relu_deriv_by_itself(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.apply_rectified_linear_deriv(T)


def seq_relu_deriv_after_a_bias(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.apply_rectified_linear_deriv(other)


def seq_relu_deriv_of_another_matrix(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); S.apply_rectified_linear_deriv(T); other.apply_rectified_linear_deriv(S)


def seq_relu_deriv_with_special_values(cm, a, B, bias, other, T, S):
    other.assign(0.0); S.assign(-0.0); other.subtract(S)                  # zeros of both signs in the gate
    cm.dot(a, B, target=T); T.apply_rectified_linear_deriv(other)
    S.assign(np.inf); cm.dot(a, B, target=T); T.apply_rectified_linear_deriv(S)


# a softmax layer and its loss: state.apply_softmax(); state.get_softmax_cross_entropy(labels, loss);
# state.apply_softmax_grad(labels, target=deriv)  (deepnet/softmax_layer.py:25-62)
def _labels(cm, T, shift=0):
    m, n = T.shape
    return cm.CUDAMatrix(_f(((np.arange(n) * 7 + shift) % m).reshape(1, n))), cm.empty((1, n))


def seq_softmax_loss_grad(cm, a, B, bias, other, T, S):
    lab, loss = _labels(cm, T)
    cm.dot(a, B, target=T); T.add_col_vec(bias); T.apply_softmax(); T.get_softmax_cross_entropy(lab, loss); T.apply_softmax_grad(lab, target=S)
    return _bits(loss)


def seq_softmax_grad_only(cm, a, B, bias, other, T, S):
    lab, loss = _labels(cm, T)
    cm.dot(a, B, target=T); T.apply_softmax(); T.apply_softmax_grad(lab, target=S)


def seq_softmax_loss_only_then_read(cm, a, B, bias, other, T, S):
    lab, loss = _labels(cm, T)
    cm.dot(a, B, target=T); T.apply_softmax(); T.get_softmax_cross_entropy(lab, loss, tiny=1e-6)
    return _bits(loss)


def seq_softmax_alone_then_other_work(cm, a, B, bias, other, T, S):
    cm.dot(a, B, target=T); T.apply_softmax(); other.add(T)


def seq_softmax_grad_in_place(cm, a, B, bias, other, T, S):
    lab, loss = _labels(cm, T)
    cm.dot(a, B, target=T); T.apply_softmax(); T.get_softmax_cross_entropy(lab, loss); T.apply_softmax_grad(lab)
    return _bits(loss)


def seq_softmax_into_another_target(cm, a, B, bias, other, T, S):
    lab, loss = _labels(cm, T)
    cm.dot(a, B, target=T); T.apply_softmax(target=other); other.get_softmax_cross_entropy(lab, loss); other.apply_softmax_grad(lab, target=S)
    return _bits(loss)


def seq_softmax_loss_of_the_logits(cm, a, B, bias, other, T, S):
    # the loss and the gradient are asked of the matrix the softmax read, not of its result: nothing joins
    lab, loss = _labels(cm, T)
    cm.dot(a, B, target=T); T.apply_sigmoid(); T.apply_softmax(target=other); T.get_softmax_cross_entropy(lab, loss); T.apply_softmax_grad(lab, target=S)
    return _bits(loss)


def seq_softmax_two_label_vectors(cm, a, B, bias, other, T, S):
    lab, loss = _labels(cm, T)
    lab2, _ = _labels(cm, T, shift=1)
    cm.dot(a, B, target=T); T.apply_softmax(); T.get_softmax_cross_entropy(lab, loss); T.apply_softmax_grad(lab2, target=S)
    return _bits(loss)


def seq_softmax_correct_in_between(cm, a, B, bias, other, T, S):
    lab, loss = _labels(cm, T)
    hit = cm.empty(loss.shape)
    cm.dot(a, B, target=T); T.apply_softmax(); T.get_softmax_correct(lab, hit); T.get_softmax_cross_entropy(lab, loss); T.apply_softmax_grad(lab, target=S)
    return np.concatenate([_bits(loss).ravel(), _bits(hit).ravel()])


def seq_softmax_then_scale_in_place(cm, a, B, bias, other, T, S):
    # an in-place scale is held back itself and launches what waits before it
    cm.dot(a, B, target=T); T.apply_softmax(); T.mult(0.9); other.mult(0.5); other.add_mult(T)


def seq_softmax_gradient_over_the_logits_of_another(cm, a, B, bias, other, T, S):
    # the gradient's target is the matrix a second softmax reads
    lab, loss = _labels(cm, T)
    cm.dot(a, B, target=T); T.apply_softmax(target=other); other.apply_softmax_grad(lab, target=T); T.apply_softmax(target=S)
    S.get_softmax_cross_entropy(lab, loss)
    return _bits(loss)


SEQS = [seq_sample_by_uniforms, seq_sample_by_uniforms_into_another_target, seq_sample_by_uniforms_behind_a_relu_layer,
        seq_sample_by_uniforms_of_itself, seq_masked_relu_deriv, seq_masked_deriv_without_activation, seq_factor_then_bias, seq_factor_twice, seq_factor_is_the_target,
        seq_factor_into_another_target, seq_factor_then_lower_bound, seq_layer_mask_for_another_matrix, seq_layer_mask_unfinished, seq_layer_mask_is_an_operand, seq_layer_mask_then_sample,
        seq_two_layers_with_masks, seq_layer_without_mask_then_draw, seq_softmax_loss_grad, seq_softmax_grad_only, seq_softmax_loss_only_then_read, seq_softmax_alone_then_other_work,
        seq_softmax_grad_in_place, seq_softmax_into_another_target, seq_softmax_loss_of_the_logits, seq_softmax_two_label_vectors,
        seq_softmax_correct_in_between, seq_softmax_then_scale_in_place, seq_softmax_gradient_over_the_logits_of_another, seq_relu_deriv, seq_relu_deriv_then_other_work, seq_relu_deriv_into_another_target, seq_relu_deriv_by_itself,
        seq_relu_deriv_after_a_bias, seq_relu_deriv_of_another_matrix, seq_relu_deriv_with_special_values, seq_fill_then_another_draw, seq_dropout, seq_dropout_after_a_layer, seq_dropout_mask_then_read, seq_dropout_into_another_target,
        seq_dropout_threshold_into_another_target, seq_dropout_mask_times_itself, seq_dropout_roles_exchanged,
        seq_fill_then_other_work, seq_dropout_of_special_values, seq_update_plain, seq_update_with_reset, seq_update_l2_l1_reset, seq_update_l2_only, seq_update_l1_only_twice,
        seq_update_not_spelled_scaled_gradient, seq_update_not_spelled_wrong_order, seq_update_not_spelled_no_gradient,
        seq_update_interrupted, seq_update_reads_another_matrix, seq_update_too_many_terms, seq_update_then_product,
        seq_scale_alone_then_read, seq_sigmoid, seq_sigmoid_sample, seq_relu, seq_tanh, seq_no_bias, seq_bias_only_then_read, seq_dot_alone_then_other_work,
        seq_bias_on_another_matrix, seq_two_biases, seq_bias_changes_in_between, seq_operand_changes_in_between,
        seq_sigmoid_into_another_target, seq_sample_in_place, seq_scaled_and_accumulating_products, seq_two_products_in_a_row,
        seq_free_while_held_back, seq_lower_bound_not_zero]


@pytest.mark.parametrize("seq", SEQS, ids=lambda f: f.__name__)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%dx%d%s" % (s[0], s[1], s[2], 't' if s[3] else 'n'))
def test_same_bits_with_and_without_deferral(cm, seq, shape):
    want = _run(cm, False, seq, shape, 5)
    got = _run(cm, True, seq, shape, 5)
    for i, (g, w) in enumerate(zip(got, want)):
        assert np.array_equal(g, w), "matrix %d differs" % i
    cm.CUDAMatrix.init_random(1)


# ---- accumulating products and row sums (the statistics of a contrastive-divergence step,
# cudamat/examples/rbm_cudamat.py:73-86): W nv x nh, v / v2 nv x B, h / h2 nh x B, bv nv x 1, bh nh x 1

STAT_SHAPES = [(784, 500, 100), (500, 784, 100), (33, 17, 5), (1024, 1024, 128), (100, 60, 128), (2048, 64, 16), (256, 512, 200),
               (36, 40, 7), (4, 4, 2), (784, 1024, 128), (1024, 10, 128), (1280, 640, 64), (1022, 10, 128), (66, 130, 31)]          # nv, nh, batch


def stat_cd(cm, o):
    eps = 0.01
    o.W.add_dot(o.v, o.h.T, mult=eps); o.W.add_dot(o.v2, o.h2.T, mult=-eps)
    o.bv.add_sums(o.v, axis=1, mult=eps); o.bv.add_sums(o.v2, axis=1, mult=-eps)
    o.bh.add_sums(o.h, axis=1, mult=eps); o.bh.add_sums(o.h2, axis=1, mult=-eps)


def stat_cd_subtract_dot(cm, o):
    o.W.add_dot(o.v, o.h.T); o.W.subtract_dot(o.v2, o.h2.T)
    o.bh.add_sums(o.h, axis=1); o.bv.add_sums(o.v, axis=1, mult=0.5); o.bh.add_sums(o.h2, axis=1, mult=-1.0); o.bv.add_sums(o.v2, axis=1, mult=-0.5)


def stat_pair_then_read(cm, o):
    o.W.add_dot(o.v, o.h.T, mult=0.25); o.W.add_dot(o.v2, o.h2.T, mult=-0.75)
    return o.W.asarray().view(np.uint32).copy()


def stat_single_then_read(cm, o):
    o.W.add_dot(o.v, o.h.T, mult=0.25)
    return o.W.asarray().view(np.uint32).copy()


def stat_three_products(cm, o):
    o.W.add_dot(o.v, o.h.T, mult=0.25); o.W.add_dot(o.v2, o.h2.T, mult=-0.75); o.W.add_dot(o.v, o.h2.T, mult=0.125)


def stat_products_into_two_targets(cm, o):
    o.W.add_dot(o.v, o.h.T, mult=0.25); o.W2.add_dot(o.v2, o.h2.T, mult=-0.75); o.W.add_dot(o.v2, o.h.T); o.W2.add_dot(o.v, o.h2.T)


def stat_second_product_reads_the_target(cm, o):
    # the visible states are overwritten by a product of the weights, then used: nothing may be reordered
    o.W.add_dot(o.v, o.h.T, mult=0.25); cm.dot(o.W, o.h, target=o.v2); o.W.add_dot(o.v2, o.h2.T, mult=-0.75)


def stat_overwriting_product_after_accumulating(cm, o):
    o.W.add_dot(o.v, o.h.T, mult=0.25); cm.dot(o.v2, o.h2.T, target=o.W); o.W.add_dot(o.v, o.h2.T); o.W.add_dot(o.v2, o.h.T, mult=2.0)


def stat_transposed_operands(cm, o):
    # the same statistics with the roles exchanged: W2t is nh x nv
    o.W2t.add_dot(o.h, o.v.T, mult=0.5); o.W2t.add_dot(o.h2, o.v2.T, mult=-0.5)


def stat_three_sums_on_one_vector(cm, o):
    o.bv.add_sums(o.v, axis=1, mult=0.5); o.bv.add_sums(o.v2, axis=1, mult=-0.25); o.bv.add_sums(o.v, axis=1, mult=2.0)


def stat_sums_on_three_vectors(cm, o):
    o.bv.add_sums(o.v, axis=1); o.bh.add_sums(o.h, axis=1); o.bv2.add_sums(o.v2, axis=1); o.bv.add_sums(o.v2, axis=1, mult=-1.0)


def stat_sum_of_a_queued_result(cm, o):
    o.bv.add_sums(o.v, axis=1, mult=0.5); o.bv2.add_sums(o.bv, axis=1); o.bv.add_sums(o.v2, axis=1)


def stat_sum_into_a_queued_source(cm, o):
    col = o.v.slice(0, 1)                      # the first column of v as an nv x 1 vector
    o.bv.add_sums(o.v, axis=1, mult=0.5); col.add_sums(o.v2, axis=1); o.bv.add_sums(o.v, axis=1)


def stat_sums_other_axis_in_between(cm, o):
    o.bv.add_sums(o.v, axis=1, mult=0.5); o.row.add_sums(o.v, axis=0); o.bv.add_sums(o.v2, axis=1)


def stat_sums_then_read(cm, o):
    o.bh.add_sums(o.h, axis=1, mult=0.5); o.bh.add_sums(o.h2, axis=1, mult=-0.5)
    return o.bh.asarray().view(np.uint32).copy()


def stat_sum_with_assignment(cm, o):
    o.bv.assign(0); o.bv.add_sums(o.v, axis=1); o.bh.assign(1.0); o.bh.add_sums(o.h, axis=1, mult=3.0); o.bh.mult(0.5)


def stat_sums_of_transposed_views(cm, o):
    o.bh.add_sums(o.hT.T, axis=1, mult=0.5); o.bh.add_sums(o.h2, axis=1, mult=-0.5)      # hT is B x nh


# a weight gradient and the bias gradient of the same layer (deepnet/edge.py:236-242, layer.py:206-211): one
# product with the sums that follow it
def stat_gradient(cm, o):
    o.W.add_dot(o.v, o.h.T); o.bh.add_sums(o.h, axis=1)


def stat_gradient_two_sums(cm, o):
    o.W.add_dot(o.v, o.h.T, mult=0.5); o.bv.add_sums(o.v, axis=1); o.bh.add_sums(o.h, axis=1, mult=0.25)


def stat_gradient_sum_reads_the_target(cm, o):
    o.W.add_dot(o.v, o.h.T, mult=0.5); o.bv.add_sums(o.W, axis=1)


def stat_gradient_sum_into_an_operand(cm, o):
    col = o.v.slice(0, 1)
    o.W.add_dot(o.v, o.h.T, mult=0.5); col.add_sums(o.v2, axis=1); o.W.add_dot(o.v, o.h2.T)


def stat_gradient_then_second_product(cm, o):
    o.W.add_dot(o.v, o.h.T, mult=0.5); o.bh.add_sums(o.h, axis=1); o.W.add_dot(o.v2, o.h2.T, mult=-0.5); o.bh.add_sums(o.h2, axis=1)


def stat_gradients_of_two_layers(cm, o):
    o.W.add_dot(o.v, o.h.T); o.bh.add_sums(o.h, axis=1); o.W2t.add_dot(o.h2, o.v2.T); o.bv.add_sums(o.v2, axis=1)
    return o.bv.asarray().view(np.uint32).copy()


STATS = [stat_gradient, stat_gradient_two_sums, stat_gradient_sum_reads_the_target, stat_gradient_sum_into_an_operand,
         stat_gradient_then_second_product, stat_gradients_of_two_layers, stat_cd, stat_cd_subtract_dot, stat_pair_then_read, stat_single_then_read, stat_three_products, stat_products_into_two_targets,
         stat_second_product_reads_the_target, stat_overwriting_product_after_accumulating, stat_transposed_operands,
         stat_three_sums_on_one_vector, stat_sums_on_three_vectors, stat_sum_of_a_queued_result, stat_sum_into_a_queued_source,
         stat_sums_other_axis_in_between, stat_sums_then_read, stat_sum_with_assignment, stat_sums_of_transposed_views]


class _Stat(object):
    def __init__(self, cm, shape, seed):
        nv, nh, B = shape
        rng = np.random.default_rng(seed)
        g = lambda *d: cm.CUDAMatrix(_f(rng.standard_normal(d)))
        self.W, self.W2, self.W2t = g(nv, nh), g(nv, nh), g(nh, nv)
        self.v, self.v2, self.h, self.h2, self.hT = g(nv, B), g(nv, B), g(nh, B), g(nh, B), g(B, nh)
        self.bv, self.bv2, self.bh, self.row = g(nv, 1), g(nv, 1), g(nh, 1), g(1, B)

    def all(self):
        return [self.W, self.W2, self.W2t, self.v, self.v2, self.h, self.h2, self.bv, self.bv2, self.bh, self.row]


@pytest.mark.parametrize("seq", STATS, ids=lambda f: f.__name__)
@pytest.mark.parametrize("shape", STAT_SHAPES, ids=lambda s: "%dx%dx%d" % s)
def test_statistics_keep_their_bits(cm, seq, shape):
    res = []
    for deferred in (False, True):
        cm.set_deferred_epilogues(deferred)
        o = _Stat(cm, shape, 11)
        out = seq(cm, o)
        res.append([_bits(x) for x in o.all()] + ([out] if out is not None else []))
    cm.set_deferred_epilogues(True)
    for i, (w, g) in enumerate(zip(*res)):
        assert np.array_equal(g, w), "matrix %d differs" % i


def test_statistics_are_the_float64_definition(cm):
    o = _Stat(cm, (784, 500, 100), 12)
    w0, bv0, bh0 = o.W.asarray().astype(np.float64), o.bv.asarray().astype(np.float64), o.bh.asarray().astype(np.float64)
    v, v2, h, h2 = (x.asarray().astype(np.float64) for x in (o.v, o.v2, o.h, o.h2))
    stat_cd(cm, o)
    eps = np.float64(np.float32(0.01))
    assert np.allclose(o.W.asarray(), w0 + eps * (v @ h.T - v2 @ h2.T), rtol=1e-5, atol=1e-5)
    assert np.allclose(o.bv.asarray(), bv0 + eps * (v.sum(1, keepdims=True) - v2.sum(1, keepdims=True)), rtol=1e-5, atol=1e-5)
    assert np.allclose(o.bh.asarray(), bh0 + eps * (h.sum(1, keepdims=True) - h2.sum(1, keepdims=True)), rtol=1e-5, atol=1e-5)


# ---- consecutive parameter updates (deepnet updates every edge and layer of a net in turn, neuralnet.py:300-312)

def _upd(p, d, g, mom=0.9, lr=0.01, l2=None, l1=None, reset=True):
    d.mult(mom)
    if l2 is not None:
        d.add_mult(p, l2)
    if l1 is not None:
        d.add_mult_sign(p, l1)
    d.add_mult(g); p.add_mult(d, -lr)
    if reset:
        g.assign(0)


def upd_six_in_a_row(cm, P):
    for i in range(6):
        _upd(*P[i])


def upd_without_resets(cm, P):
    for i in range(4):
        _upd(*P[i], reset=False)


def upd_mixed_decays_and_resets(cm, P):
    _upd(*P[0], l2=0.001); _upd(*P[1], reset=False); _upd(*P[2], l1=0.002, l2=0.0005); _upd(*P[3], mom=0.5, lr=0.1, l1=0.01)


def upd_eleven(cm, P):
    for i in range(11):
        _upd(*P[i % 6], mom=0.9 - 0.05 * i)              # more than one launch holds; the same parameter again: in order


def upd_tied(cm, P):
    # the second update reads what the first wrote, the third writes what the second read (both are 1024 x 1)
    _upd(*P[1]); _upd(P[3][0], P[3][1], P[1][0], reset=False); _upd(P[1][0], P[1][1], P[3][2])


def upd_gradient_is_another_delta(cm, P):
    _upd(*P[0]); _upd(P[1][0], P[1][1], P[1][2]); _upd(P[0][0], P[0][2], P[0][1])     # roles exchanged on the same arrays


def upd_then_scale_that_is_no_update(cm, P):
    _upd(*P[0]); _upd(*P[1]); P[2][0].mult(0.5); P[2][0].add_mult(P[2][2], 2.0); P[2][1].add(P[2][0])


def upd_then_read(cm, P):
    _upd(*P[0]); _upd(*P[1], reset=False)
    return P[1][0].asarray().view(np.uint32).copy()


def upd_interleaved_with_a_product(cm, P):
    _upd(*P[0]); cm.dot(P[0][0], P[0][0].T, target=P[6]); _upd(*P[1]); _upd(*P[2])


def upd_reset_of_another_gradient(cm, P):
    P[0][1].mult(0.9); P[0][1].add_mult(P[0][2]); P[0][0].add_mult(P[0][1], -0.01); P[1][2].assign(0); _upd(*P[1])


def upd_sums_between(cm, P):
    # a layer's weights, its biases behind a sum of their gradient (twice: the sums and the updates of a net in turn)
    _upd(*P[0]); P[1][2].add_sums(P[2][2], axis=1, mult=0.01); _upd(*P[1])
    P[3][2].add_sums(P[2][1], axis=1, mult=0.02); P[3][2].add_sums(P[2][2], axis=1, mult=0.5); _upd(*P[3]); _upd(*P[4], l2=0.001)


def upd_sums_of_what_waits(cm, P):
    _upd(*P[2]); P[1][2].add_sums(P[2][0], axis=1, mult=0.01); _upd(*P[1])           # reads the weights
    _upd(*P[2], reset=False); P[3][2].add_sums(P[2][2], axis=1, mult=0.01); _upd(*P[3])          # reads the gradient
    _upd(*P[2]); P[1][0].add_sums(P[2][1], axis=1, mult=0.01); _upd(*P[1])           # reads the step


def upd_sums_into_what_waits(cm, P):
    for i in range(3):
        _upd(*P[1], reset=i != 1); P[1][i].add_sums(P[2][0], axis=1, mult=0.01); _upd(*P[2])


def upd_sums_that_join_and_do_not(cm, P):
    _upd(*P[1]); P[3][2].add_sums(P[2][0], axis=1); P[1][0].add_sums(P[2][0], axis=1); _upd(*P[3])
    _upd(*P[0]); P[1][2].add_sums(P[2][0], axis=1); P[1][2].add_sums(P[2][1], axis=1); P[3][2].add_sums(P[2][2], axis=1)
    P[3][2].add_sums(P[2][1], axis=1); _upd(*P[3]); _upd(*P[2])                     # four sums are launched at once


def upd_sum_then_read(cm, P):
    _upd(*P[0]); P[1][2].add_sums(P[2][2], axis=1, mult=0.01)
    return P[0][0].asarray().view(np.uint32).copy()


# Products that updates wait behind, and their late operands.  X, Y, Z: 300 x 300, updates (X[0], X[1], X[2]); b: 300 x 1; A, B, T, U:
# products of 300 terms (k_gemm_ring); late_*: the operand comes when the product waits, or has left for the products that share a launch

def late_bias_of_an_update(cm, o):
    for i in range(3):
        _upd(*o.b, reset=i != 2); cm.dot(o.A, o.B, target=o.T); o.T.add_col_vec(o.b[i]); o.T.apply_sigmoid(); o.U.add(o.T)


def late_bias_beside_an_update(cm, o):
    _upd(*o.X); cm.dot(o.A, o.B, target=o.T); o.T.add_col_vec(o.b[0]); o.T.lower_bound(0); _upd(*o.b)


def late_factor_of_an_update(cm, o):
    for i in range(3):
        _upd(*o.X, reset=i != 2); cm.dot(o.A, o.B, target=o.T); o.T.mult(o.X[i]); o.T.apply_rectified_linear_deriv(o.Y[0]); o.U.add(o.T)


def late_factor_and_gate_of_updates(cm, o):
    _upd(*o.X); _upd(*o.Y, reset=False); cm.dot(o.A, o.B, target=o.T); o.T.mult(o.X[0]); o.T.apply_rectified_linear_deriv(o.Y[0])


def late_gate_of_an_update(cm, o):
    for i in range(3):
        _upd(*o.X, reset=i != 2); cm.dot(o.A, o.B, target=o.T); o.T.apply_rectified_linear_deriv(o.X[i]); o.U.add(o.T)


def late_second_product_of_an_update(cm, o):
    for i in range(3):
        _upd(*o.X, reset=i != 2); o.T.add_dot(o.A, o.B, mult=0.1); o.T.add_dot(o.X[i], o.B, mult=-0.1)
        _upd(*o.X, reset=i != 2); o.T.add_dot(o.A, o.B, mult=0.1); o.T.add_dot(o.A, o.X[i], mult=-0.1); o.b[2].add_sums(o.T, axis=1, mult=0.01)


def late_gate_behind_updates(cm, o):
    # the layer's order of deepnet: input gradient, weight gradient, its update, the sums and update of the biases, the gate
    cm.dot(o.A, o.B, target=o.T); o.X[2].add_dot(o.A, o.Y[0]); _upd(*o.X); o.b[2].add_sums(o.A, axis=1); _upd(*o.b)
    o.T.apply_rectified_linear_deriv(o.Y[0]); o.U.add(o.T)


def late_gate_that_an_update_writes(cm, o):
    for i in range(3):
        cm.dot(o.A, o.B, target=o.T); _upd(*o.X, reset=i != 2); o.T.apply_rectified_linear_deriv(o.X[i]); o.U.add(o.T)


def late_gate_that_a_grouped_product_writes(cm, o):
    cm.dot(o.A, o.B, target=o.T); o.Y[2].add_dot(o.A, o.B, mult=-0.1); _upd(*o.X); o.T.apply_rectified_linear_deriv(o.Y[2])


def late_gate_that_a_grouped_sum_writes(cm, o):
    cm.dot(o.A, o.B, target=o.T); o.col.add_sums(o.A, axis=1, mult=0.1); _upd(*o.X); o.T.apply_rectified_linear_deriv(o.over_col)


def late_gate_of_a_target_that_a_grouped_product_reads(cm, o):
    cm.dot(o.A, o.B, target=o.T); o.Y[2].add_dot(o.T, o.B, mult=0.1); _upd(*o.X); o.T.apply_rectified_linear_deriv(o.Y[0])


def late_gate_of_a_target_that_a_grouped_sum_reads(cm, o):
    cm.dot(o.A, o.B, target=o.T); o.b[2].add_sums(o.T, axis=1, mult=0.1); _upd(*o.X); o.T.apply_rectified_linear_deriv(o.Y[0])


def late_gate_of_an_update_of_the_target(cm, o):
    cm.dot(o.A, o.B, target=o.T); _upd(o.X[0], o.X[1], o.T); o.T.apply_rectified_linear_deriv(o.Y[0])
    cm.dot(o.A, o.B, target=o.X[0]); _upd(*o.X); o.X[0].apply_rectified_linear_deriv(o.Y[0])


def late_gate_of_an_accumulating_product(cm, o):
    o.T.add_dot(o.A, o.B, mult=0.1); _upd(*o.X); o.T.apply_rectified_linear_deriv(o.Y[0])
    o.T.add_dot(o.A, o.B, mult=0.1); o.T.add_dot(o.A, o.Y[1], mult=0.1); _upd(*o.X); o.T.apply_rectified_linear_deriv(o.Y[0])


def late_gate_twice_and_into_another_target(cm, o):
    cm.dot(o.A, o.B, target=o.T); _upd(*o.X); o.T.apply_rectified_linear_deriv(o.Y[0]); o.T.apply_rectified_linear_deriv(o.Y[1])
    cm.dot(o.A, o.B, target=o.T); _upd(*o.X); o.T.apply_rectified_linear_deriv(o.Y[0], target=o.U)


def late_gate_behind_an_unfinished_update(cm, o):
    cm.dot(o.A, o.B, target=o.T); o.X[1].mult(0.9); o.X[1].add_mult(o.X[2]); o.T.apply_rectified_linear_deriv(o.X[1])
    cm.dot(o.A, o.B, target=o.T); o.Y[0].mult(0.9); o.T.apply_rectified_linear_deriv(o.Y[0])


LATE = [f for n, f in sorted(globals().items()) if n.startswith('late_')]


class _Late:
    def __init__(self, cm, seed, side):
        rng = np.random.default_rng(seed)
        g = lambda *d: cm.CUDAMatrix(_f(rng.standard_normal(d)))
        n = side
        self.X, self.Y, self.b = ([g(*d) for _ in range(3)] for d in ((n, n), (n, n), (n, 1)))
        self.A, self.B, self.T, self.U, self.over_col = (g(n, n) for _ in range(5))
        self.col = self.over_col.slice(n - 1, n)              # (its last column)

    def all(self):
        return self.X + self.Y + self.b + [self.A, self.B, self.T, self.U, self.over_col]


@pytest.mark.parametrize("seq", LATE, ids=lambda f: f.__name__)
@pytest.mark.parametrize("side", [300, 60, 640])
def test_late_operands_of_products_keep_the_order_of_calls(cm, seq, side):
    """(60: on the kernels of 16 x 16 blocks; 640: another tile)"""
    res = []
    for deferred in (False, True):
        cm.set_deferred_epilogues(deferred)
        o = _Late(cm, 31, side)
        for _ in range(2):
            seq(cm, o)
        res.append([_bits(x) for x in o.all()])
    cm.set_deferred_epilogues(True)
    for i, (w, g) in enumerate(zip(*res)):
        assert np.array_equal(g, w), "matrix %d differs" % i


UPDS = [upd_sums_between, upd_sums_of_what_waits, upd_sums_into_what_waits, upd_sums_that_join_and_do_not, upd_sum_then_read, upd_six_in_a_row, upd_without_resets, upd_mixed_decays_and_resets, upd_eleven, upd_tied, upd_gradient_is_another_delta,
        upd_then_scale_that_is_no_update, upd_then_read, upd_interleaved_with_a_product, upd_reset_of_another_gradient]


def _params_of_a_net(cm, seed):
    rng = np.random.default_rng(seed)
    g = lambda *d: cm.CUDAMatrix(_f(rng.standard_normal(d)))
    shapes = [(784, 1024), (1024, 1), (1024, 1024), (1024, 1), (37, 10), (10, 1)]
    P = [(g(*sh), g(*sh), g(*sh)) for sh in shapes]
    P.append(cm.empty((784, 784)))
    return P


@pytest.mark.parametrize("seq", UPDS, ids=lambda f: f.__name__)
def test_consecutive_updates_keep_their_bits(cm, seq):
    res = []
    for deferred in (False, True):
        cm.set_deferred_epilogues(deferred)
        P = _params_of_a_net(cm, 21)
        out = seq(cm, P)
        res.append([_bits(x) for t in P[:6] for x in t] + [_bits(P[6])] + ([out] if out is not None else []))
    cm.set_deferred_epilogues(True)
    for i, (w, g) in enumerate(zip(*res)):
        assert np.array_equal(g, w), "matrix %d differs" % i


def test_the_folded_sequence_is_the_float64_definition(cm, rng):
    m, k, n = 500, 784, 100
    w, x, b = _f(0.05 * rng.standard_normal((k, m))), _f(rng.random((k, n))), _f(rng.standard_normal((m, 1)))
    W, X, Bv, T = cm.CUDAMatrix(w), cm.CUDAMatrix(x), cm.CUDAMatrix(b), cm.empty((m, n))
    cm.dot(W.T, X, target=T); T.add_col_vec(Bv); T.apply_sigmoid()
    want = 1.0 / (1.0 + np.exp(-(w.astype(np.float64).T @ x.astype(np.float64) + b)))
    assert np.allclose(T.asarray(), want, rtol=1e-5, atol=1e-6)


def test_training_steps_of_the_bench_keep_their_bits(cm):
    import bench
    for cls, seed, params in ((bench.RBM, 1, lambda o: [o.W, o.bv, o.bh, o.h, o.hs, o.v2, o.h2]),
                              (bench.MLP, 3, lambda o: o.W + o.b + o.dW + [o.loss] + o.mask),
                              (bench.RBMExample, 1, lambda o: [o.w_vh, o.w_v, o.w_h, o.wu_vh, o.wu_v, o.wu_h, o.v, o.h, o.r])):
        res = []
        for deferred in (False, True):
            cm.set_deferred_epilogues(deferred)
            cm.CUDAMatrix.init_random(seed)
            obj = cls(cm)
            for _ in range(3):
                obj.step()
            res.append([_bits(p) for p in params(obj)])
        cm.set_deferred_epilogues(True)
        for a, b in zip(*res):
            assert np.array_equal(a, b)
    cm.CUDAMatrix.init_random(1)


def test_the_switch_reports_its_previous_setting(cm):
    assert cm.set_deferred_epilogues(False) is True
    assert cm.set_deferred_epilogues(True) is False
    assert cm.set_deferred_epilogues(True) is True


def test_launch_deferred_queues_what_is_held_back(cm, rng):
    """A caller that goes on with its own work on the NULL stream (here: a plain hipMemcpy through the
    runtime, which the library does not see) finds the results of every call it has made."""
    import ctypes as ct
    hip = ct.CDLL('libamdhip64.so')
    hip.hipMemcpy.argtypes = [ct.c_void_p, ct.c_void_p, ct.c_size_t, ct.c_int]
    a, b = _f(rng.standard_normal((96, 64)) * 0.1), _f(rng.standard_normal((64, 40)))
    bias = _f(rng.standard_normal((96, 1)))
    A, B, bv = cm.CUDAMatrix(a), cm.CUDAMatrix(b), cm.CUDAMatrix(bias)
    T = cm.empty((96, 40)); T.assign(-3.0)
    cm.cuda_sync_threads()
    cm.dot(A, B, target=T)
    T.add_col_vec(bv)                         # both calls are held back now
    cm.launch_deferred()
    got = np.empty((96, 40), dtype=np.float32, order='F')
    assert hip.hipMemcpy(got.ctypes.data, ct.cast(T.p_mat.contents.data_device, ct.c_void_p), got.nbytes, 2) == 0
    want = a.astype(np.float64) @ b.astype(np.float64) + bias
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-5)
    T.apply_sigmoid()                         # and the library goes on from there
    np.testing.assert_allclose(T.asarray(), 1.0 / (1.0 + np.exp(-want)), rtol=1e-5, atol=1e-6)
    cm.launch_deferred()                      # nothing held back: no effect


@pytest.mark.parametrize("shape", [(1003, 700, 250), (784, 500, 100)], ids=lambda s: "%dx%dx%d" % s)
def test_the_statistics_of_a_step_are_queued_with_its_last_sum(cm, shape):
    """With two products and four sums nothing more can join: they are on their way when the last call returns (mid-sized products, of
    more than 128 terms, share a launch with others, smaller ones do not)."""
    import ctypes as ct
    hip = ct.CDLL('libamdhip64.so')
    hip.hipMemcpy.argtypes = [ct.c_void_p, ct.c_void_p, ct.c_size_t, ct.c_int]
    res = []
    for deferred in (False, True):
        cm.set_deferred_epilogues(deferred)
        o = _Stat(cm, shape, 13)
        stat_cd(cm, o)
        out = []
        for m in (o.W, o.bv, o.bh):
            got = np.empty(m.shape, dtype=np.float32, order='F')
            assert hip.hipMemcpy(got.ctypes.data, ct.cast(m.p_mat.contents.data_device, ct.c_void_p), got.nbytes, 2) == 0
            out.append(got.view(np.uint32))
        res.append(out)
    cm.set_deferred_epilogues(True)
    for w, g in zip(*res):
        assert np.array_equal(g, w)


def _launches(cm, run):
    """Kernels that the calls of run() queue (recorded on a stream of the test's own)."""
    import ctypes as ct
    hip = ct.CDLL('libamdhip64.so')
    stream, graph, nodes = ct.c_void_p(), ct.c_void_p(), ct.c_size_t()
    run()
    cm.cuda_sync_threads()
    assert hip.hipStreamCreateWithFlags(ct.byref(stream), 1) == 0
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    cm._cudamat.graph_set_stream(stream, 1)
    run()
    cm.launch_deferred()
    cm._cudamat.graph_set_stream(None, 0)
    assert hip.hipStreamEndCapture(stream, ct.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ct.byref(nodes)) == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
    return nodes.value


@pytest.mark.parametrize("inputs,outputs,batch", [(279, 681, 103), (734, 123, 116), (107, 531, 124)])
def test_sums_go_with_their_product_where_others_wait(cm, inputs, outputs, batch):
    """A gradient of at most 128 terms takes the sums of its layer along: also behind products that wait to share a launch and read or write
    what the sums do, or have sums of their own."""
    g = lambda *d: cm.CUDAMatrix(_f(0.1 * np.random.default_rng(d[0]).standard_normal(d)))
    W, X, Y, D, DX, G, G2, b, b2 = (g(inputs, outputs), g(inputs, batch), g(outputs, batch), g(outputs, batch), g(inputs, batch), g(inputs, outputs),
                                    g(inputs, outputs), g(outputs, 1), g(outputs, 1))
    # (at most as many as the gradients and the other products)
    assert _launches(cm, lambda: (G.add_dot(X, D.T), b.add_sums(D, axis=1))) == 1
    assert _launches(cm, lambda: (cm.dot(W.T, X, target=Y), Y.add_col_vec(b), cm.dot(W, D, target=DX), G.add_dot(X, D.T), b.add_sums(D, axis=1))) <= 3
    assert _launches(cm, lambda: (G.add_dot(X, D.T), b.add_sums(D, axis=1), G2.add_dot(X, D.T), b2.add_sums(D, axis=1))) <= 2


# ---- random call sequences: whatever is held back, every matrix ends with the bits of the separate launches

def _random_sequence(cm, rng_ops, pool, vecs, rows, n_ops):
    """n_ops library calls on randomly chosen matrices of one shape family (m x n matrices, m x 1 and
    1 x n vectors, a k x m and a k x n operand pair per product): the operand choice includes every
    kind of aliasing the calls accept."""
    M = lambda: pool[rng_ops.integers(len(pool))]
    V = lambda: vecs[rng_ops.integers(len(vecs))]
    scal = lambda: float(np.float32(rng_ops.choice([0.0, 1.0, -1.0, 0.5, 0.9, -0.01, 2.0, 0.3])))
    m_, n_ = pool[0].shape
    lab, loss = cm.CUDAMatrix(_f(((np.arange(n_) * 5) % m_).reshape(1, n_))), cm.empty((1, n_))
    loss.assign(0)
    reads = []
    for _ in range(n_ops):
        op = rng_ops.integers(31)
        a, b, c = M(), M(), M()
        if op == 0: cm.dot(pool.A.T, pool.B, target=a)
        elif op == 1: a.add_dot(pool.A.T, pool.B, mult=scal())
        elif op == 2: a.add_dot(pool.A2.T, pool.B2, mult=scal())
        elif op == 3: a.subtract_dot(pool.A.T, pool.B2)
        elif op == 4: a.add_col_vec(V())
        elif op == 5: a.apply_sigmoid()
        elif op == 6: a.lower_bound(0)
        elif op == 7: a.sample_bernoulli(target=b)
        elif op == 8: a.mult(scal())
        elif op == 9: a.add_mult(b, scal())
        elif op == 10: a.add_mult_sign(b, scal())
        elif op == 11: a.assign(scal())
        elif op == 12: a.fill_with_rand()
        elif op == 13: a.greater_than(scal())
        elif op == 14: a.mult(b)
        elif op == 15: V().add_sums(a, axis=1, mult=scal())
        elif op == 16: rows[rng_ops.integers(len(rows))].add_sums(a, axis=0, mult=scal())
        elif op == 17: a.add(b, target=c)
        elif op == 18: cm.tanh(a)
        elif op == 19: reads.append(_bits(a))
        elif op == 20: a.add_mult(b)               # factor 1: the gradient of an update
        elif op == 22: a.apply_rectified_linear_deriv(b)
        elif op == 23: a.apply_rectified_linear_deriv(b, target=c)
        elif op == 24: a.apply_softmax() if rng_ops.integers(2) else a.apply_softmax(target=b)
        elif op == 25: a.get_softmax_cross_entropy(lab, loss)
        elif op == 26: a.apply_softmax_grad(lab, target=b)
        elif op == 27:      # a layer as deepnet spells it, with the variations that do and do not fold
            cm.dot(pool.A.T, pool.B, target=a)
            if rng_ops.integers(2): a.add_col_vec(V())
            kind = rng_ops.integers(4)
            if kind == 0: a.apply_sigmoid()
            elif kind == 1: a.lower_bound(0)
            elif kind == 2: cm.tanh(a)
            if rng_ops.integers(2):
                b.fill_with_rand()
                if rng_ops.integers(4): b.greater_than(scal())
                (a if rng_ops.integers(2) else c).mult(b)
            elif rng_ops.integers(2): a.sample_bernoulli(target=b)
        elif op == 29: a.less_than(b, target=b if rng_ops.integers(2) else c)
        elif op == 30: a.fill_with_rand(); a.less_than(b, target=b)
        elif op == 28:      # an output layer and its loss
            a.apply_softmax() if rng_ops.integers(2) else a.apply_softmax(target=b)
            src = a if rng_ops.integers(4) else b
            if rng_ops.integers(2): src.get_softmax_cross_entropy(lab, loss)
            if rng_ops.integers(4): src.apply_softmax_grad(lab, target=c)
        else: V().add_sums(a, axis=1)
    reads.append(_bits(loss))
    return reads


class _Pool(list):
    pass


@pytest.mark.parametrize("shape", [(500, 100, 784), (64, 128, 96), (33, 7, 20), (1024, 128, 128), (784, 500, 100)],
                         ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("seed", range(12))
def test_random_sequences_keep_their_bits(cm, shape, seed):
    m, n, k = shape
    res = []
    for deferred in (False, True):
        cm.set_deferred_epilogues(deferred)
        cm.CUDAMatrix.init_random(3 + seed)
        rng = np.random.default_rng(100 + seed)
        g = lambda *d: cm.CUDAMatrix(_f(rng.standard_normal(d) * 0.5))
        pool = _Pool(g(m, n) for _ in range(4))
        pool.A, pool.A2, pool.B, pool.B2 = g(k, m), g(k, m), g(k, n), g(k, n)
        vecs, rows = [g(m, 1) for _ in range(2)], [g(1, n) for _ in range(2)]
        reads = _random_sequence(cm, np.random.default_rng(5100 + seed), pool, vecs, rows, 60)
        after = cm.empty((64, 48)); after.fill_with_rand()
        res.append([_bits(x) for x in list(pool) + vecs + rows + [after]] + reads)
    cm.set_deferred_epilogues(True)
    cm.CUDAMatrix.init_random(1)
    assert len(res[0]) == len(res[1])
    for i, (w, gt) in enumerate(zip(*res)):
        assert np.array_equal(gt, w), "result %d differs" % i


# ---- elementwise calls that wait for each other and run as one pass

def _ew_call(cm, kind, x, y, t, vecs, s):
    col, row = vecs
    calls = {'mult': lambda: x.mult(y, target=t), 'add': lambda: x.add(y, target=t), 'subtract': lambda: x.subtract(y, target=t),
             'divide': lambda: x.divide(y, target=t), 'sigmoid': lambda: x.apply_sigmoid(target=t), 'tanh': lambda: cm.tanh(x, target=t),
             'exp': lambda: cm.exp(x, target=t), 'add_mult': lambda: t.add_mult(y, s), 'scale': lambda: x.mult(s, target=t),
             'shift': lambda: x.add(s, target=t), 'gate': lambda: x.apply_rectified_linear_deriv(y, target=t),
             'lower': lambda: x.lower_bound(s, target=t), 'col': lambda: x.mult_by_col(col, target=t), 'row': lambda: x.add_row_vec(row, target=t),
             'add_col': lambda: x.add_col_vec(col, target=t), 'col_mult': lambda: x.add_col_mult(col, s, target=t),
             'sum': lambda: x.sum(axis=0, target=row), 'assign': lambda: t.assign(x)}
    calls[kind]()


# sides of products on every tile of k_gemm_ring and on the kernels beside it (one of 128 terms at most is not on the ring)
GROUP_SIDES = [[64, 130, 301, 700], [100, 200, 784, 1024], [129, 250, 1003, 1500], [16, 33, 520, 2100]]


@pytest.mark.parametrize("sides", GROUP_SIDES, ids=lambda s: "-".join(map(str, s)))
@pytest.mark.parametrize("seed", range(6))
def test_products_that_share_a_launch_keep_their_bits(cm, sides, seed):
    """Products in a row, independent ones and others (a target that the next reads or writes, an operand that the next writes, two
    into one target), with biases, activations, gates, factors and row sums between them: the bits of one launch each."""
    init = np.random.default_rng(99)
    first = {(a, b, i): _f(0.1 * init.standard_normal((a, b))) for a in sides for b in sides for i in range(2)}
    cols = {a: _f(init.standard_normal((a, 1))) for a in sides}

    def run(deferred):
        rng = np.random.default_rng(seed)
        cm.set_deferred_epilogues(deferred)
        mats = {k: cm.CUDAMatrix(v) for k, v in first.items()}
        vecs = {k: cm.CUDAMatrix(v) for k, v in cols.items()}
        pick = lambda a, b: (a, b, int(rng.integers(2)))
        view = lambda key, trans: mats[key].T if trans else mats[key]
        for _ in range(60):
            m, n, k = (sides[int(i)] for i in rng.integers(0, len(sides), 3))
            ta, tb, kind, tail = (int(rng.integers(x)) for x in (2, 2, 8, 5))
            A, B, C = pick(k, m) if ta else pick(m, k), pick(n, k) if tb else pick(k, n), pick(m, n)
            A2, gate, rows = pick(k, m) if ta else pick(m, k), pick(m, n), pick(m, n)
            if kind < 7 and (C in (A, B) or (kind == 4 and C == A2) or (kind < 3 and tail == 2 and C == gate)):
                continue                                     # (a product into one of its operands is no product)
            T = mats[C]
            if kind < 3:
                cm.dot(view(A, ta), view(B, tb), target=T)
                if tail == 1:
                    T.add_col_vec(vecs[m]); T.apply_sigmoid()
                elif tail == 2:
                    T.apply_rectified_linear_deriv(mats[gate])
                elif tail == 3:
                    T.add_col_vec(vecs[m]); T.lower_bound(0)
            elif kind < 6:
                T.add_dot(view(A, ta), view(B, tb), mult=0.01)
                if kind == 4:                                # ... and a second one into it
                    T.add_dot(view(A2, ta), view(B, tb), mult=-0.01)
                if tail < 3:
                    vecs[m].add_sums(mats[rows], axis=1, mult=0.01)
            elif kind == 6:
                cm.dot(view(A, ta), view(B, tb), mult=0.5, target=T)
            else:
                mats[rows].mult(0.01)
        out = [_bits(mats[k]) for k in sorted(mats)] + [_bits(vecs[k]) for k in sorted(vecs)]
        cm.set_deferred_epilogues(True)
        return out

    for want, got in zip(run(False), run(True)):
        assert np.array_equal(want, got)


# (from 2^23 elements on calls without a common input do not wait for each other)
@pytest.mark.parametrize("h,w", [(1, 1), (3, 1), (1, 7), (64, 33), (65, 33), (130, 127), (1001, 37), (2052, 2049), (2897, 2897)])
@pytest.mark.parametrize("seed", range(4))
def test_elementwise_calls_that_wait_keep_their_bits(cm, h, w, seed):
    """Random programs over few matrices (in place, reading what the call before wrote, through column views that overlap
    and start at any 4-byte boundary) give the bits of the calls one by one."""
    kinds = ['mult', 'add', 'subtract', 'divide', 'sigmoid', 'tanh', 'exp', 'add_mult', 'scale', 'shift', 'gate', 'lower', 'col', 'row',
             'add_col', 'col_mult', 'sum', 'assign']
    rng = np.random.default_rng([seed, h, w])
    start = [np.asarray(rng.standard_normal((h, w + 2)), dtype=np.float32, order='F') for _ in range(5)]
    vec = [np.asarray(rng.standard_normal(shape), dtype=np.float32, order='F') for shape in ((h, 1), (1, w))]
    # in half of the programs the calls fit together: sources from one half of the matrices, targets in the other
    apart = seed % 2 == 0
    program = []
    for _ in range(40):
        src = rng.integers(0, 2 if apart and rng.random() < 0.8 else 5, 2)
        dst = rng.integers(2, 5) if apart else rng.integers(0, 5)
        offs = rng.integers(0, 3, 3) if rng.random() < 0.3 else [1, 1, 1]
        program.append((kinds[rng.integers(0, len(kinds))], src, dst, offs, float(np.float32(rng.standard_normal()))))
    got = []
    for defer in (True, False):
        cm.set_deferred_epilogues(defer)
        try:
            mats = [cm.CUDAMatrix(a) for a in start]
            vecs = [cm.CUDAMatrix(v) for v in vec]
            for kind, src, dst, offs, s in program:
                x, y, t = (mats[i].slice(int(o), int(o) + w) for i, o in zip((src[0], src[1], dst), offs))
                # (views of one matrix that overlap in part are not defined: such a call takes its input in place)
                x, y = ((t if (i == dst and o != offs[2]) else v) for v, i, o in ((x, src[0], offs[0]), (y, src[1], offs[1])))
                _ew_call(cm, kind, x, y, t, vecs, s)
            got.append([np.array(m.asarray()) for m in mats + vecs])
        finally:
            cm.set_deferred_epilogues(True)
    for a, b in zip(*got):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("h,w", [(1, 1), (3, 1), (65, 33), (1001, 37), (2052, 2049)])
@pytest.mark.parametrize("seed", range(4))
def test_elementwise_calls_that_go_on_in_place_keep_their_bits(cm, h, w, seed):
    """Chains of calls on one matrix, with others between them and with the matrix itself as the other operand."""
    kinds = ['mult', 'add', 'subtract', 'sigmoid', 'tanh', 'add_mult', 'scale', 'shift', 'gate', 'lower', 'col', 'row', 'add_col', 'col_mult']
    rng = np.random.default_rng([seed, h, w, 1])
    start = [np.asarray(rng.standard_normal((h, w + 1)), dtype=np.float32, order='F') for _ in range(5)]
    vec = [np.asarray(rng.standard_normal(shape), dtype=np.float32, order='F') for shape in ((h, 1), (1, w))]
    program, at = [], 0
    for _ in range(40):
        if rng.random() < 0.3:
            at = int(rng.integers(0, 5))
        x, y = (at, int(rng.integers(0, 5))) if rng.random() < 0.8 else rng.integers(0, 5, 2)
        program.append((kinds[rng.integers(0, len(kinds))], int(x), int(y), at, float(np.float32(rng.standard_normal()))))
    got = []
    for defer in (True, False):
        cm.set_deferred_epilogues(defer)
        try:
            mats = [cm.CUDAMatrix(a) for a in start]
            views = [m.slice(seed % 2, seed % 2 + w) for m in mats]
            vecs = [cm.CUDAMatrix(v) for v in vec]
            for kind, x, y, t, s in program:
                _ew_call(cm, kind, views[x], views[y], views[t], vecs, s)
            got.append([np.array(m.asarray()) for m in mats + vecs])
        finally:
            cm.set_deferred_epilogues(True)
    for a, b in zip(*got):
        assert np.array_equal(a, b, equal_nan=True)


def test_a_waiting_elementwise_call_is_seen_by_what_follows(cm, rng):
    a = cm.CUDAMatrix(np.asarray(rng.standard_normal((130, 70)), dtype=np.float32, order='F'))
    want = a.asarray() * 2
    t = cm.empty((130, 70))
    a.mult(2.0, target=t)
    assert np.array_equal(t.asarray(), want)                     # a copy to the host
    t2, s = cm.empty((130, 70)), cm.empty((1, 70))
    a.mult(2.0, target=t2)
    a.add(1.0, target=t)
    t2.sum(axis=0, target=s)                                     # a reduction
    assert np.allclose(s.asarray(), want.sum(axis=0, keepdims=True), atol=1e-4)
    b = cm.empty((130, 70))
    a.mult(2.0, target=b)
    a.free_device_memory()                                       # the operand's memory goes away
    assert np.array_equal(b.asarray(), want)


# ---- sums and maxima of one matrix that wait for each other

# k_col_sum_max on a wavefront and on a workgroup per column; k_colblock on 2 and 4 columns, streams and not; k_rows_one with one
# slice (of 64, 128, 256 and more columns, streams and not) and with several; few rows, whose row sums and maxima do not wait
RED_SHAPES = [(1, 1), (3, 5), (4, 3), (5, 130), (67, 1), (130, 70), (1001, 2047), (4097, 33), (1024, 2048), (1028, 1030), (2052, 1500), (16384, 200),
              (16390, 260), (1024, 16640), (4100, 4100), (65540, 260), (7, 9000)]


@pytest.mark.parametrize("h,w", RED_SHAPES)
def test_sums_and_maxima_that_wait_keep_their_bits(cm, h, w):
    rng = np.random.default_rng([h, w])
    a = np.asarray(rng.standard_normal((h, w), dtype=np.float32), order='F')
    a[rng.integers(0, h), rng.integers(0, w)] = np.inf
    a[rng.integers(0, h), rng.integers(0, w)] = -np.inf
    a[rng.integers(0, h), :] = -np.finfo(np.float32).max
    a[rng.integers(0, h), rng.integers(0, w)] = np.nan
    m = cm.CUDAMatrix(a)
    got = []
    for order in ('sSmM', 'MmSs', 'sm', 'MS'):
        for defer in (True, False):
            cm.set_deferred_epilogues(defer)
            try:
                out = {'s': cm.empty((1, w)), 'S': cm.empty((h, 1)), 'm': cm.empty((1, w)), 'M': cm.empty((h, 1))}
                for k in order:
                    (m.sum if k in 'sS' else m.max)(axis=int(k in 'SM'), target=out[k])
                got.append({k: np.array(out[k].asarray()) for k in order})
            finally:
                cm.set_deferred_epilogues(True)
        for k in order:
            assert np.array_equal(got[-2][k], got[-1][k], equal_nan=True), (order, k)
    # (comparisons that NaN fails, from the lowest finite value along a column and from -infinity along a row)
    assert np.array_equal(got[0]['m'], np.fmax.reduce(a, axis=0, keepdims=True, initial=-np.finfo(np.float32).max))
    assert np.array_equal(got[0]['M'], np.fmax.reduce(a, axis=1, keepdims=True, initial=-np.inf))


def test_sums_and_maxima_that_do_not_go_together(cm, rng):
    """One result twice, results that share memory with the matrix or with each other, other matrices and what reads a result."""
    a, b = (np.asarray(rng.standard_normal((64, 48)), dtype=np.float32, order='F') for _ in range(2))
    x, y = cm.CUDAMatrix(a), cm.CUDAMatrix(b)
    row = cm.empty((1, 48))
    x.sum(axis=0, target=row)
    x.max(axis=0, target=row)                                    # over the sum
    assert np.array_equal(row.asarray(), a.max(axis=0, keepdims=True))
    r1, r2, col = cm.empty((1, 48)), cm.empty((1, 48)), cm.empty((64, 1))
    x.max(axis=0, target=r1)
    x.max(axis=0, target=r2)                                     # again, elsewhere
    y.max(axis=1, target=col)
    x.sum(axis=1, target=x.slice(0, 1))                          # into the matrix's first column
    x.max(axis=0, target=row)
    want = a.copy()
    want[:, 0] = a.astype(np.float64).sum(axis=1)
    assert np.array_equal(r1.asarray(), a.max(axis=0, keepdims=True)) and np.array_equal(r2.asarray(), r1.asarray())
    assert np.array_equal(col.asarray(), b.max(axis=1, keepdims=True))
    # (48 terms of about 1: rounding of each of the 48 additions, sums below 32)
    assert np.allclose(row.asarray(), want.max(axis=0, keepdims=True), rtol=0, atol=48 * 32 * 2.0 ** -24)
    x.max(axis=1, target=col)
    x.mult(2.0)                                                  # the matrix changes behind a maximum that waits
    y.sum(axis=1, target=col)
    y.add_col_vec(col)                                           # reads what waits
    assert np.allclose(y.asarray(), b + b.astype(np.float64).sum(axis=1, keepdims=True), rtol=0, atol=48 * 32 * 2.0 ** -24)


COLUMN_RESULTS = """
import ctypes as ct, sys
import numpy as np
from deepnet_amd import cudamat as cm
hip = ct.CDLL('libamdhip64.so')
def free():
    a, b = ct.c_size_t(), ct.c_size_t()
    cm.cuda_sync_threads()
    assert hip.hipMemGetInfo(ct.byref(a), ct.byref(b)) == 0
    return a.value
cm.cublas_init()
x = cm.CUDAMatrix(np.ones((16448, 4096), dtype=np.float32, order='F'))
col, row = cm.empty((16448, 1)), cm.empty((1, 4096))
small, r3 = cm.CUDAMatrix(np.ones((3, 4096), dtype=np.float32, order='F')), cm.empty((1, 4096))
small.sum(axis=0, target=r3); small.max(axis=0, target=r3); r3.asarray()      # (kernels are loaded)
before = free()
x.sum(axis=0, target=row); x.max(axis=0, target=r3)
columns = before - free()
assert row.asarray()[0, 5] == 16448 and r3.asarray()[0, 7] == 1
x.sum(axis=1, target=col); x.max(axis=1, target=col)
print(columns, before - free())
"""


def test_results_along_the_columns_take_no_workspace():
    """In a process of its own (another one's workspace has grown): sums and maxima of columns leave the device memory as it
    is, those of rows take their partial sums (16 slices of 16448 rows, two results: 2 MiB)."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, '-c', COLUMN_RESULTS], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    columns, rows = map(int, r.stdout.split()[-2:])
    assert columns == 0 and rows > 0


# ---- the kinds of calls that wait, in any order

def _mixed_sequence(cm, rng, pool, vecs, rows, params, n_ops):
    M, V, R = (lambda l=l: l[rng.integers(len(l))] for l in (pool, vecs, rows))
    scal = lambda: float(np.float32(rng.choice([0.0, 1.0, 0.5, 0.9, -0.01, 2.0])))
    n, reads = pool[0].shape[1], []

    def update():
        w, wd, g = params[rng.integers(len(params))]
        wd.mult(0.9); wd.add_mult(g); w.add_mult(wd, -0.01)
        if rng.integers(2):
            g.assign(0)

    def look():
        for q in rng.permutation(4)[:rng.integers(1, 5)]:
            (a.sum if q < 2 else a.max)(axis=int(q % 2), target=V() if q % 2 else R())

    def temporary():
        t = cm.empty(a.shape)
        a.add(b, target=t); t.sum(axis=0, target=R()); t.free_device_memory()

    kinds = [look, look, update, update, temporary,
             lambda: params[1][rng.integers(3)].add_sums(a, axis=1, mult=scal()), lambda: V().add_sums(a, axis=1),
             lambda: cm.dot(pool.A.T, pool.B, target=a), lambda: a.add_dot(pool.A.T, pool.B, mult=scal()),
             lambda: a.add_col_vec(V()), lambda: a.add_row_vec(R()), lambda: a.mult_by_col(V(), target=b), lambda: a.apply_sigmoid(target=b),
             lambda: a.lower_bound(0), lambda: a.mult(b, target=c), lambda: a.add_mult(b, scal()), lambda: a.mult(scal()),
             lambda: a.apply_rectified_linear_deriv(b), lambda: a.assign(b), lambda: a.apply_softmax(target=b), lambda: a.fill_with_rand(),
             lambda: a.slice(0, 1).add_mult(V(), 0.5), lambda: a.slice(1, n).mult(0.5, target=(b if b is not a else c).slice(0, n - 1)) if c is not a else None,
             lambda: V().mult(V(), target=V()), lambda: R().add(scal()), lambda: reads.append(_bits(R())), lambda: reads.append(_bits(a))]
    hot = rng.integers(0, len(kinds), 10)                         # (every sequence favours some)
    for _ in range(n_ops):
        a, b, c = M(), M(), M()
        kinds[hot[rng.integers(10)] if rng.random() < 0.7 else rng.integers(len(kinds))]()
    return reads


@pytest.mark.parametrize("shape", [(500, 100, 784), (33, 7, 20), (1024, 300, 64)], ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("seed", range(8))
def test_sums_maxima_updates_and_the_rest_keep_their_bits(cm, shape, seed):
    m, n, k = shape
    res = []
    for deferred in (False, True):
        cm.set_deferred_epilogues(deferred)
        cm.CUDAMatrix.init_random(3 + seed)
        rng = np.random.default_rng([seed, m])
        g = lambda *d: cm.CUDAMatrix(_f(rng.standard_normal(d) * 0.5))
        pool = _Pool(g(m, n) for _ in range(4))
        pool.A, pool.B = g(k, m), g(k, n)
        vecs, rows = [g(m, 1) for _ in range(3)], [g(1, n) for _ in range(3)]
        params = [tuple(g(*d) for _ in range(3)) for d in ((m, n), (m, 1), (37, 10))]
        reads = _mixed_sequence(cm, np.random.default_rng([seed, m, 9]), pool, vecs, rows, params, 60)
        res.append([_bits(x) for x in list(pool) + vecs + rows + [x for t in params for x in t]] + reads)
    cm.set_deferred_epilogues(True)
    cm.CUDAMatrix.init_random(1)
    assert len(res[0]) == len(res[1])
    for i, (w, gt) in enumerate(zip(*res)):
        nan = np.isnan(w.view(np.float32))                        # (of either sign)
        assert np.array_equal(nan, np.isnan(gt.view(np.float32))) and np.array_equal(gt[~nan], w[~nan]), "result %d differs" % i
