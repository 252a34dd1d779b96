// CLIP text encoder on the HIP kernels: token ids [B, 77] -> last hidden state [B, 77, 768].
//
// Replaces the reference's LiteRT text encoder (VulkanUnetPipeline.kt:48-53: int[77] ->
// [1, 77, 768], the UNet's cross-attention context), an export of SD1.5's text_encoder
// (CLIP ViT-L/14 text tower: 12 pre-LayerNorm layers of width 768, 12 heads, quick-GELU MLP
// of 3072, causal self-attention, final LayerNorm).  Per layer:
//   qkv = LN1(x) Wqkv^T + b                     (one GEMM over the fused q/k/v weight)
//   x += out_proj(causal_attention(q, k, v))
//   x += fc2(quick_gelu(fc1(LN2(x))))           (quick-GELU in fc1's epilogue)
// with the residual adds in the GEMM epilogues (in place on x), activations fp16.  LN1 and LN2
// run inside the GEMMs around them: the one that writes x keeps its row statistics, the one
// that reads it has the affine folded into its weight (as separate launches they took 113 of
// 554 us for two prompts).
#include "graph.h"

namespace sdu {

static const int kSeq = 77, kHid = 768, kLayers = 12, kHeads = 12, kFfn = 3072, kVocab = 49408;
static const float kLnEps = 1e-5f;
static const std::string kPf = "text_model.";

static std::string layer(int i) { return kPf + "encoder.layers." + std::to_string(i); }

static void clip_register(AuxNet& n) {
    n.add(kPf + "embeddings.token_embedding.weight", {kVocab, kHid}, WK_EMBED);
    n.add(kPf + "embeddings.position_embedding.weight", {kSeq, kHid}, WK_EMBED);
    for (int i = 0; i < kLayers; ++i) {
        const std::string a = layer(i) + ".self_attn.";
        // q, k, v weights and biases each contiguous: one [3C, C] weight, one [3C] bias
        n.add(a + "q_proj.weight", {kHid, kHid}, WK_LINEAR);
        n.add(a + "k_proj.weight", {kHid, kHid}, WK_LINEAR, GL_PLAIN, 0, true);
        n.add(a + "v_proj.weight", {kHid, kHid}, WK_LINEAR, GL_PLAIN, 0, true);
        n.add(a + "q_proj.bias", {kHid}, WK_BIAS);
        n.add(a + "k_proj.bias", {kHid}, WK_BIAS, GL_PLAIN, 0, true);
        n.add(a + "v_proj.bias", {kHid}, WK_BIAS, GL_PLAIN, 0, true);
        n.add(a + "out_proj.weight", {kHid, kHid}, WK_LINEAR);
        n.add(a + "out_proj.bias", {kHid}, WK_BIAS);
        n.add(layer(i) + ".layer_norm1.weight", {kHid}, WK_NORM_W);
        n.add(layer(i) + ".layer_norm1.bias", {kHid}, WK_NORM_B);
        n.add(layer(i) + ".mlp.fc1.weight", {kFfn, kHid}, WK_LINEAR);
        n.add(layer(i) + ".mlp.fc1.bias", {kFfn}, WK_BIAS);
        n.add(layer(i) + ".mlp.fc2.weight", {kHid, kFfn}, WK_LINEAR);
        n.add(layer(i) + ".mlp.fc2.bias", {kHid}, WK_BIAS);
        n.add(layer(i) + ".layer_norm2.weight", {kHid}, WK_NORM_W);
        n.add(layer(i) + ".layer_norm2.bias", {kHid}, WK_NORM_B);
    }
    n.add(kPf + "final_layer_norm.weight", {kHid}, WK_NORM_W);
    n.add(kPf + "final_layer_norm.bias", {kHid}, WK_NORM_B);
}

int clip_create(Ctx& c, const char* weights_dir, uint64_t seed, int flags) {
    AuxNet* n = new AuxNet();
    n->kind = AUX_CLIP;
    clip_register(*n);
    // folded projections, each [N, C] weight, then [N] bias and [N] column sums (fp32)
    const int lnN[2] = {3 * kHid, kFfn};
    const auto fold_bytes = [](int N) { return (size_t)N * (kHid * sizeof(f16) + 2 * sizeof(float)); };
    const size_t extra = kLayers * (fold_bytes(lnN[0]) + fold_bytes(lnN[1]));
    int st = aux_alloc(c, *n, extra);
    if (st) { aux_free(n); return st; }
    const bool affine = (flags & SDU_INIT_RANDOM_AFFINE) != 0;
    for (const WeightRec& r : n->weights) {
        st = weights_dir ? load_weight_file(c, r, weights_dir) : gen_weight(c, r, seed, affine, 0.02);
        if (st) { aux_free(n); return st; }
    }
    char* p = (char*)n->pool + n->pool_bytes - extra;
    hipError_t e = hipSuccess;
    for (int i = 0; i < 2 * kLayers && e == hipSuccess; ++i) {
        const std::string pf = layer(i / 2), w = i % 2 ? ".mlp.fc1" : ".self_attn.q_proj", g = i % 2 ? ".layer_norm2" : ".layer_norm1";
        const int N = lnN[i % 2];
        AuxNet::LnLinear l;
        l.w = (f16*)p;
        l.b = (float*)(l.w + (size_t)N * kHid);
        l.s = l.b + N;
        p += fold_bytes(N);
        n->ln.push_back(l);
        e = fold_ln_launch(n->wd(pf + w + ".weight"), n->wd(pf + w + ".bias"), n->wd(pf + g + ".weight"), n->wd(pf + g + ".bias"),
                           l.w, l.b, l.s, N, kHid, c.stream);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(c.stream);
    if (e != hipSuccess) { aux_free(n); return hip_fail(c, e, "clip weights"); }
    aux_free(c.clip);
    c.clip = n;
    return SDU_OK;
}

static void clip_body(Exec& E, AuxNet& n, AuxState& S) {
    const int B = S.key[0], T = B * kSeq, C = kHid;
    f16* x = E.alloc<f16>((size_t)T * C);
    f16* h = E.alloc<f16>((size_t)T * C);
    f16* qkv = E.alloc<f16>((size_t)T * 3 * C);
    f16* at = E.alloc<f16>((size_t)T * C);
    f16* f = E.alloc<f16>((size_t)T * kFfn);
    // row statistics of x before each layer's LayerNorms (GemmArgs::row_part)
    float* rp1 = E.alloc<float>((size_t)(C / 64) * T * 2);
    float* rp2 = E.alloc<float>((size_t)(C / 64) * T * 2);
    E.run("clip_embed", [&] {
        return embed_launch((const int32_t*)S.in, n.wd(kPf + "embeddings.token_embedding.weight"),
                            n.wd(kPf + "embeddings.position_embedding.weight"), x, rp1, B, kSeq, C, kVocab, E.s);
    });
    // a projection of LayerNorm(x), the LayerNorm inside the GEMM
    auto ln_gemm = [&](const AuxNet::LnLinear& l, int N, const float* part, f16* out) {
        GemmArgs g = dense_args(x, C, T, N, C, l.w, out, N);
        g.bias2 = l.b;
        g.ln_part = part;
        g.ln_colsum = l.s;
        g.ln_eps = kLnEps;
        return g;
    };
    for (int i = 0; i < kLayers; ++i) {
        const std::string pf = layer(i), a = pf + ".self_attn.";
        gemm(E, "clip_linear", ln_gemm(n.ln[2 * i], 3 * C, rp1, qkv));
        AttnArgs aa{qkv, qkv + C, qkv + 2 * C, at, B, kHeads, kSeq, kSeq, C / kHeads, 3 * C, 3 * C, 3 * C, C,
                    1.0f / sqrtf((float)(C / kHeads)), 1};
        E.run("clip_attn", [&] { return attention_launch(aa, E.s); });
        {
            GemmArgs g = dense_args(at, C, T, C, C, n.wd(a + "out_proj.weight"), x, C);
            g.bias = n.wd(a + "out_proj.bias");
            g.res = x;
            g.ldr = C;
            g.row_part = rp2;
            gemm(E, "clip_linear", g);
        }
        {
            GemmArgs g = ln_gemm(n.ln[2 * i + 1], kFfn, rp2, f);
            g.act = ACT_QUICK_GELU;
            gemm(E, "clip_linear", g);
        }
        {
            GemmArgs g = dense_args(f, kFfn, T, C, kFfn, n.wd(pf + ".mlp.fc2.weight"), x, C);
            g.bias = n.wd(pf + ".mlp.fc2.bias");
            g.res = x;
            g.ldr = C;
            g.row_part = rp1;
            gemm(E, "clip_linear", g);
        }
    }
    E.run("clip_ln", [&] {
        return layernorm_launch(x, n.wd(kPf + "final_layer_norm.weight"), n.wd(kPf + "final_layer_norm.bias"), h, T, C, kLnEps, E.s);
    });
    E.run("clip_io", [&] { return f16_to_f32_launch(h, (float*)S.out, (int64_t)T * C, E.s); });
}

int clip_encode_device(Ctx& c, const int32_t* d_ids, int B, float* d_out) {
    if (!c.clip) return set_err(&c, SDU_ERR_WEIGHT, "no CLIP text encoder (sdu_clip_init)");
    if (B < 1 || B > 64) return set_err(&c, SDU_ERR_ARG, "CLIP encode: B in 1..64");
    const size_t in_b = (size_t)B * kSeq * 4, out_b = (size_t)B * kSeq * kHid * 4;
    int st = 0;
    AuxState* S = aux_state(c, *c.clip, {B}, B, in_b, out_b, clip_body, &st);
    if (!S) return st;
    hipError_t e;
    if ((e = hipMemcpyAsync(S->in, d_ids, in_b, hipMemcpyDeviceToDevice, c.stream)) ||
        (e = hipGraphLaunch(S->exec, c.stream)) ||
        (e = hipMemcpyAsync(d_out, S->out, out_b, hipMemcpyDeviceToDevice, c.stream)))
        return hip_fail(c, e, "clip encode");
    return SDU_OK;
}

}  // namespace sdu
