// Autograd nodes (nodes.cpp) as functions of the binding module (binding.cpp).
#pragma once
#include <Python.h>

PyObject* spx_error_class();  // SpxError
// attention(q, k, v, lo, hi, block_lo, block_hi, context_keys, ttt_step, scaling) -> out [1, NQ, Hq, D]
PyObject* spx_node_attention(PyObject*, PyObject* const* args, Py_ssize_t n);
// row_loss(op, logits [..., V], targets) -> float32 [...]
PyObject* spx_node_row_loss(PyObject*, PyObject* const* args, Py_ssize_t n);
