// A program's own module: the methods of the reference's tnn::Module (include/tnn_api.h:62-303 there) are all it has to have.
// Compiled, not run (tests/test_cpp_host_api.py).
#include "tnn/tnn_api.h"

class Identity : public tnn::Module {
  public:
    torch::Tensor initialize_params() override { return {}; }
    torch::Tensor initialize_params(const torch::Tensor &) override { return {}; }
    void set_params(const torch::Tensor &, bool) override {}
    torch::Tensor get_params() override { return {}; }
    torch::Tensor forward_pass(const torch::Tensor &x) override { return x; }
    std::tuple<torch::Tensor, torch::Tensor> backward_pass(const torch::Tensor &g, const torch::Tensor &, bool, bool) override { return {g, {}}; }
    std::tuple<torch::Tensor, torch::Tensor> backward_pass(const torch::Tensor &g, bool, bool) override { return {g, {}}; }
    torch::Tensor inference(const torch::Tensor &x) override { return x; }
    size_t n_params() override { return 0; }
    size_t n_output_dims() override { return 1; }

  protected:
    void FreeWorkspace() override {}
    void AllocateWorkspace(const size_t) override {}
};

tnn::Module *make() { return new Identity; }
