// One question to autograd that Python cannot ask: whether anything but the
// next node's backward sees the gradient that a node sends along one of its
// edges.  A backward that would leave that gradient out (its consumer's work
// done in the same pass) may do so only if nothing does.
#include <Python.h>
#include <torch/csrc/autograd/engine.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/python_function.h>

namespace {
bool observed(PyObject *ctx, int input) {
    if (!THPFunction_Check(ctx)) return true;
    const auto self = reinterpret_cast<THPFunction *>(ctx)->cdata.lock();
    if (!self || input < 0 || (size_t)input >= self->num_outputs()) return true;
    const torch::autograd::Edge &edge = self->next_edge((size_t)input);
    if (!edge.is_valid()) return true;
    torch::autograd::Node *fn = edge.function.get();
    // hooks of the tensor (its gradient's, retain_grad's) live on the node that made it, beside the node's own
    if (!fn->tensor_pre_hooks().empty() || !fn->retains_grad_hooks().empty() || !fn->pre_hooks().empty() ||
        !fn->post_hooks().empty())
        return true;
    // the running pass: what grad() or backward(inputs=...) was asked for
    const auto *info = torch::autograd::get_current_graph_task_exec_info();
    if (!info) return true;  // not inside a pass that can be asked
    const auto it = info->find(fn);
    return it != info->end() && it->second.captures_ && !it->second.captures_->empty();
}
}  // namespace

// ctx: the context of a torch.autograd.Function inside its backward; input: the
// position of a tensor among its tensor arguments.  0 when only the node that
// made that tensor will see the gradient returned for it; 1 otherwise, and
// whenever that cannot be told.
extern "C" int drp_grad_observed(PyObject *ctx, int input) {
    try {
        return observed(ctx, input) ? 1 : 0;
    } catch (...) {
        return 1;
    }
}
