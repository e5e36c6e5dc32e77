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

struct CubicSampling : torch::autograd::Function<CubicSampling>
{
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& ptcloud, const at::Tensor& cubic_features, int64_t neighborhood_size)
    {
        const int scale = as_int(cubic_features.size(2), "scale"), size = as_int(neighborhood_size, "neighborhood_size");
        const std::vector<at::Tensor> sampled = sample_cubes(scale, size, ptcloud, cubic_features, true);
        ctx->save_for_backward({sampled[1]});
        ctx->saved_data["scale"] = static_cast<int64_t>(scale);
        ctx->saved_data["neighborhood_size"] = neighborhood_size;
        return sampled[0];
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const at::Tensor vertices = ctx->get_saved_variables()[0];
        const std::vector<at::Tensor> out =
            sample_cubes_grad(static_cast<int>(ctx->saved_data["scale"].toInt()), static_cast<int>(ctx->saved_data["neighborhood_size"].toInt()),
                              grads[0].contiguous(), vertices, ctx->needs_input_grad(0));
        return {out[0], out[1], at::Tensor()};
    }
};

at::Tensor cubic_sampling(const at::Tensor& ptcloud, const at::Tensor& cubic_features, int64_t neighborhood_size)
{
    TORCH_CHECK(cubic_features.dim() == 5, "cubic_features must have shape (B, c, scale, scale, scale)");
    const at::Tensor points = ptcloud.contiguous(), maps = cubic_features.contiguous();
    if (records(points) || records(maps))
        return CubicSampling::apply(points, maps, neighborhood_size);
    return sample_cubes(as_int(maps.size(2), "scale"), as_int(neighborhood_size, "neighborhood_size"), points, maps, true)[0];
}
