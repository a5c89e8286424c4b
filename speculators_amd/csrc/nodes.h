// Autograd nodes (nodes.cpp) as functions of the binding module (binding.cpp).
#pragma once
#include <Python.h>

PyObject* spx_error_class();  // SpxError
// attention(q, k, v, lo, hi, block_lo, block_hi, context_keys, ttt_step, scaling) -> out [1, NQ, Hq, D]
PyObject* spx_node_attention(PyObject*, PyObject* const* args, Py_ssize_t n);
// row_loss(op, logits [..., V], targets) -> float32 [...]
PyObject* spx_node_row_loss(PyObject*, PyObject* const* args, Py_ssize_t n);

// wanted(ctx of a Python node) -> for each of the tensors it was applied to, whether the running backward pass asks for its gradient
PyObject* spx_node_wanted(PyObject*, PyObject* const* args, Py_ssize_t n);

// The launches of a decoder layer in sequence (layer_host.cpp), called by layer.py; arguments positional, as read there.
PyObject* spx_layer_product(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_tail_forward(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_tail_backward(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_ttt_forward(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_ttt_backward(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_normed_forward(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_normed_backward(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_product_tn(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_products_tn(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_loss_step(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_loss_terms(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_loss_steps_begin(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_loss_steps_pass(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_loss_steps_end(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_cat_bf16(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* spx_layer_gain_sums(PyObject*, PyObject* const* args, Py_ssize_t n);
