// The entry points of layer_core.cpp and mixed_core.cpp in the module of step_core.cpp.
#pragma once
#include <Python.h>

PyObject* natsl_make_layer(PyObject*, PyObject* args);
PyObject* natsl_layer_train(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* natsl_layer_backward(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* natsl_layer_prompt_front(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* natsl_layer_prompt_rest(PyObject*, PyObject* const* a, Py_ssize_t n);

PyObject* natsl_make_entries(PyObject*, PyObject* args);
PyObject* natsl_mixed_plain(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* natsl_hard_select_plain(PyObject*, PyObject* const* a, Py_ssize_t n);
