// The operators with a gradient as autograd nodes in C++, included by points_cuda.cpp inside its unnamed namespace:
// a call from Python enters the extension once, and the backward pass runs on the engine's thread without taking the
// interpreter's lock (a torch.autograd.Function in Python costs about 15 us a pass more than its kernels' launches).
// Where nothing records, the forward function is called directly and no node is made.
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

inline bool records(const at::Tensor& t)
{
    return at::GradMode::is_enabled() && t.requires_grad();
}

struct GriddingBatch : torch::autograd::Function<GriddingBatch>
{
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& ptcloud, double scale)
    {
        ctx->save_for_backward({ptcloud});
        ctx->saved_data["scale"] = scale;
        return gridding_batch_forward(ptcloud, scale);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const at::Tensor ptcloud = ctx->get_saved_variables()[0];
        return {gridding_batch_backward(ptcloud, ctx->saved_data["scale"].toDouble(), grads[0].contiguous()), at::Tensor()};
    }
};

at::Tensor gridding_batch(const at::Tensor& ptcloud, double scale)
{
    const at::Tensor points = ptcloud.contiguous();
    return records(points) ? GriddingBatch::apply(points, scale) : gridding_batch_forward(points, scale);
}
