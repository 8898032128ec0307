// The autograd functions of the Python modules: one call into a native module, forward and backward, as nodes of PyTorch's
// graph. They stand in for the reference's autograd function (dpcpp_bindings/tiny_dpcpp_nn/modules.py:65-136), which pads, scales,
// converts and slices with PyTorch operations around the native calls; a training step on a small batch then spends
// its time in Python and in a dozen launches. Here the step is one entry into C++ each way, and what surrounds the passes is
// part of them (tnn::Module::forward_rows / backward_rows).
#pragma once

#include <ATen/TracerMode.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/torch.h>

#include "tnn/tnn_api.h"

namespace tnn_binding {

using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// The interpreter's lock is released before a module's is waited for, here and in every binding: a thread that holds a module's
// may need the interpreter's for a moment (dropping the last reference to a tensor that Python has seen).
typedef std::lock_guard<std::recursive_mutex> ModuleLock;
typedef std::scoped_lock<std::recursive_mutex, std::recursive_mutex> ModulePairLock;

/// A network or an encoding: gradients of its input (a network's) and of its parameters.
struct ModuleBackward : public torch::autograd::Node {
    std::shared_ptr<tnn::Module> module;
    tnn::Module::RowsPass pass; // its input tensor is in `input`
    SavedVariable input, params;
    double loss_scale = 1.0;
    bool released = false;

    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        TORCH_CHECK(!released, torch::autograd::ERR_BACKWARD_TWICE);
        const torch::Tensor x = input.unpack(), p = params.unpack();
        if (!grads[0].defined()) return {torch::Tensor(), torch::Tensor()};
        const torch::AutoGradMode no_grad(false);
        tnn::Module::RowsPass kept = pass;
        kept.input = x;
        const ModuleLock pass_lock(module->pass_mutex());
        auto [dx, dparams] = module->backward_rows(grads[0], kept, loss_scale, task_should_compute_output(0), p);
        return {dx, dparams};
    }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        input.reset_data();
        params.reset_data();
        pass.hidden.reset();
        pass.output.reset();
        pass.order.reset();
        released = true;
    }
    std::string name() const override { return "TnnModuleBackward"; }
};

/// A grid encoding and its network as one call: gradients of the network's parameters and of the table.
struct EncodedNetworkBackward : public torch::autograd::Node {
    std::shared_ptr<tnn::Module> network, encoding;
    tnn::Module::RowsPass pass; // the encoded batch
    SavedVariable positions, params, table;
    double loss_scale = 1.0;

    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const torch::Tensor x = positions.unpack(), p = params.unpack(), t = table.unpack();
        if (!grads[0].defined()) return {torch::Tensor(), torch::Tensor()};
        const torch::AutoGradMode no_grad(false);
        const ModulePairLock pass_lock(network->pass_mutex(), encoding->pass_mutex());
        auto [dparams, dtable] = network->backward_rows_with_encoding(*encoding, x, grads[0], pass, loss_scale, p, t);
        return {dparams, dtable};
    }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        positions.reset_data();
        params.reset_data();
        table.reset_data();
        pass.levels.reset();
        pass.order.reset();
    }
    std::string name() const override { return "TnnEncodedNetworkBackward"; }
};

/// The nodes here have no forward-mode derivative: a tangent is refused, as PyTorch refuses it for a function without a jvp, not dropped.
inline void refuse_tangents(std::initializer_list<torch::Tensor> inputs) {
    for (const torch::Tensor &t : inputs)
        TORCH_CHECK_NOT_IMPLEMENTED(!torch::autograd::isFwGradDefined(t), "tiny_dpcpp_nn modules have no forward-mode derivative");
}

/// y = module(x), recorded for autograd when that is on and anything asks for gradients. Nothing while torch.jit.trace records: it
/// sees PyTorch's operators, of a call here the allocation of the result alone (modules.py then makes the call an operator).
inline std::optional<torch::Tensor> call(const std::shared_ptr<tnn::Module> &module, const torch::Tensor &x, const torch::Tensor &params, bool push, bool training,
                          double loss_scale) {
    if (at::tracer::impl::is_dispatch_enabled()) return std::nullopt;
    refuse_tangents({x, params});
    const torch::Tensor in = module->input_rows(x); // (PyTorch operations where any are needed: autograd sees them)
    const bool record = torch::autograd::compute_requires_grad(in, params);
    tnn::Module::RowsPass pass;
    torch::Tensor y;
    {
        const torch::AutoGradMode no_grad(false);
        const ModuleLock pass_lock(module->pass_mutex());
        y = module->forward_rows(in, push && module->n_params() ? params : torch::Tensor(), record, training, pass);
    }
    if (!record) return y;
    auto node = std::shared_ptr<ModuleBackward>(new ModuleBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(in, params));
    node->module = module;
    node->input = SavedVariable(pass.input, false);
    pass.input.reset();
    node->pass = std::move(pass);
    node->params = SavedVariable(params, false);
    node->loss_scale = loss_scale;
    torch::autograd::set_history(y, node);
    return y;
}

/// y = network(encoding(positions)) for a pair that can_train_with_encoding (or, without autograd, can_fuse_encoding) accepts. Nothing
/// for no positions, and while torch.jit.trace records.
inline std::optional<torch::Tensor> call_with_encoding(const std::shared_ptr<tnn::Module> &network, const std::shared_ptr<tnn::Module> &encoding, const torch::Tensor &x,
                                        const torch::Tensor &params, const torch::Tensor &table, bool push_network, bool push_table, double loss_scale) {
    if (at::tracer::impl::is_dispatch_enabled() || (x.dim() > 0 && x.size(0) == 0)) return std::nullopt;
    refuse_tangents({x, params, table});
    const torch::Tensor positions = x.detach().to(torch::kFloat32).contiguous();
    const bool record = torch::autograd::compute_requires_grad(params, table);
    tnn::Module::RowsPass pass;
    torch::Tensor y;
    {
        const torch::AutoGradMode no_grad(false);
        const ModulePairLock pass_lock(network->pass_mutex(), encoding->pass_mutex());
        if (push_table) encoding->push_params(table);
        y = network->forward_rows_with_encoding(*encoding, positions, push_network ? params : torch::Tensor(), record, pass);
    }
    if (!record) return y;
    auto node = std::shared_ptr<EncodedNetworkBackward>(new EncodedNetworkBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(params, table));
    node->network = network;
    node->encoding = encoding;
    node->pass = std::move(pass);
    node->positions = SavedVariable(positions, false);
    node->params = SavedVariable(params, false);
    node->table = SavedVariable(table, false);
    node->loss_scale = loss_scale;
    torch::autograd::set_history(y, node);
    return y;
}

} // namespace tnn_binding
