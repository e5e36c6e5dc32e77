// The operators with a gradient as autograd nodes in C++, included by points_cuda.cpp inside its unnamed namespace:
// a call from Python enters the extension once, and the backward pass runs on the engine's thread without taking the
// interpreter's lock (a torch.autograd.Function in Python costs about 15 us a pass more than its kernels' launches).
// Where nothing records, the forward function is called directly and no node is made.
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Whether a call has to go through its node.  (With a forward-mode tangent too, whether or not gradients are recorded:
// none of the nodes has a forward mode, and the node says so, where the kernels alone would lose the tangent in silence.)
inline bool records(const at::Tensor& t)
{
    return (at::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(/*level=*/0).defined();
}

// (The backward pass needs the points; it gets a copy that the forward kernel makes, so that the caller's may be changed in place.)
struct GriddingBatch : torch::autograd::Function<GriddingBatch>
{
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& ptcloud, double scale)
    {
        at::Tensor kept;
        at::Tensor grid = gridding_batch_forward(ptcloud, scale, &kept);
        ctx->save_for_backward({kept});
        ctx->saved_data["scale"] = scale;
        return grid;
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

// The gradient of an interpolation (three_interpolate) or grouping walks lists of (index, weight) inverted per target;
// they are built with the forward pass, and several backward passes share them.  (idx and weight are kept outside the
// saved variables: as in the Python functions, they may be changed in place once the lists exist.)
struct InterpolateFeatures : torch::autograd::Function<InterpolateFeatures>
{
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& features, const at::Tensor& idx, const at::Tensor& weight)
    {
        TORCH_CHECK(features.dim() == 3, "features must have shape (B, c, m)");
        ctx->saved_data["m"] = features.size(2);
        if (!features.requires_grad())
            return three_interpolate(features, idx, weight);
        const at::Tensor places = idx.contiguous(), weights = weight.contiguous();
        std::pair<at::Tensor, at::Tensor> out = three_interpolate_recording(features.contiguous(), places, weights);
        if (out.second.numel())
            ctx->saved_data["lists"] = out.second;
        else
        {
            ctx->saved_data["idx"] = places;
            ctx->saved_data["weight"] = weights;
        }
        return out.first;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        if (!ctx->needs_input_grad(0))
            return {at::Tensor(), at::Tensor(), at::Tensor()};
        const at::Tensor grad = grads[0].contiguous();
        const int m = static_cast<int>(ctx->saved_data["m"].toInt());
        const auto lists = ctx->saved_data.find("lists");
        return {lists != ctx->saved_data.end() ? three_interpolate_grad_lists(grad, lists->second.toTensor(), m)
                                               : three_interpolate_grad(grad, ctx->saved_data["idx"].toTensor(), ctx->saved_data["weight"].toTensor(), m),
                at::Tensor(), at::Tensor()};
    }
};

at::Tensor interpolate_features(const at::Tensor& features, const at::Tensor& idx, const at::Tensor& weight)
{
    return records(features) || records(weight) ? InterpolateFeatures::apply(features, idx, weight) : three_interpolate(features, idx, weight);
}

struct GroupFeatures : torch::autograd::Function<GroupFeatures>
{
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& features, const at::Tensor& idx)
    {
        const at::Tensor places = idx.contiguous();
        std::pair<at::Tensor, at::Tensor> out = grouping_operation_recording(features.contiguous(), places);
        ctx->saved_data["n"] = features.size(2);
        if (out.second.numel())
            ctx->saved_data["lists"] = out.second;
        else
            ctx->saved_data["idx"] = places;
        return out.first;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const at::Tensor grad = grads[0].contiguous();
        const int n = static_cast<int>(ctx->saved_data["n"].toInt());
        const auto lists = ctx->saved_data.find("lists");
        return {lists != ctx->saved_data.end() ? grouping_operation_grad_lists(grad, lists->second.toTensor(), n)
                                               : grouping_operation_grad(grad, ctx->saved_data["idx"].toTensor(), n),
                at::Tensor()};
    }
};

at::Tensor group_features(const at::Tensor& features, const at::Tensor& idx)
{
    return records(features) ? GroupFeatures::apply(features, idx) : grouping_operation(features.contiguous(), idx.contiguous());
}

// The Chamfer loss as one node: the means with the search, and a backward pass that takes the loss's gradient as the
// one number it is, where a node for the distances alone is handed two arrays of equal numbers to be written and read.
struct ChamferLoss : torch::autograd::Function<ChamferLoss>
{
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& xyz1, const at::Tensor& xyz2)
    {
        const at::Tensor a = xyz1.contiguous(), b = xyz2.contiguous();
        const std::vector<at::Tensor> out = chamfer_loss_forward(a, b);
        ctx->save_for_backward({a, b, out[1]});
        return out[0];
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const std::vector<at::Tensor> out = chamfer_loss_backward(saved[0], saved[1], saved[2], grads[0]);
        return {out[0], out[1]};
    }
};

at::Tensor chamfer_loss(const at::Tensor& xyz1, const at::Tensor& xyz2)
{
    return records(xyz1) || records(xyz2) ? ChamferLoss::apply(xyz1, xyz2) : chamfer_loss_forward(xyz1.contiguous(), xyz2.contiguous())[0];
}
