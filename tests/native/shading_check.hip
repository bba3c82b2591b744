// Test entry points around the library's device arithmetic (exact_math.h,
// shading.h): the short forms as they are, and the shading functions beside the
// same formulas with plain square roots and divisions.  All pointers are device
// memory; every call returns once its kernel has ended (0, or the HIP error).
#include "shading.h"

using namespace snkpt;

namespace {

__global__ void k_unary(int op, const float* a, float* out, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = op == 0 ? rcp_exact(a[i]) : sqrt_exact(a[i]);
}
__global__ void k_quotient(const float* x, const float* d, float* out, float* out_signed, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = div_exact(x[i], d[i]);
    out_signed[i] = div_signed(x[i], fabsf(d[i]), rcp_exact(fabsf(d[i])));
}

V3 __device__ ref_normalize(V3 a) {
    const float l = sqrtf(dot(a, a));
    return l > 0.0f ? V3{a.x / l, a.y / l, a.z / l} : a;
}
V3 __device__ ref_eval(const Mat& m, V3 n, V3 wo, V3 wi) {
    if (m.flags & 2u) return m.albedo * (1.0f / kRefPi);
    const V3 f0{0.04f + (m.albedo.x - 0.04f) * m.metallic, 0.04f + (m.albedo.y - 0.04f) * m.metallic,
                0.04f + (m.albedo.z - 0.04f) * m.metallic};
    const V3 h = ref_normalize(wo + wi);
    const float hv = fmaxf(dot(h, wo), 0.0f);
    const float c1 = fminf(fmaxf(1.0f - hv, 0.0f), 1.0f), c2 = c1 * c1, fw = (c2 * c2) * c1;
    const V3 F{f0.x + (1.0f - f0.x) * fw, f0.y + (1.0f - f0.y) * fw, f0.z + (1.0f - f0.z) * fw};
    const float a = m.roughness * m.roughness, r = m.roughness + 1.0f, k = (r * r) / 8.0f;
    const float nv = fmaxf(dot(n, wo), 0.0f), nl = fmaxf(dot(n, wi), 0.0f);
    const float G = g1_schlick(nv, k) * g1_schlick(nl, k);
    const V3 spec = F * (ggx_d(fmaxf(dot(n, h), 0.0f), a * a) * G / (4.0f * nv * nl + 0.0001f));
    const float kdm = 1.0f - m.metallic;
    return V3{(1.0f - F.x) * kdm * m.albedo.x, (1.0f - F.y) * kdm * m.albedo.y, (1.0f - F.z) * kdm * m.albedo.z} *
               (1.0f / kRefPi) +
           spec;
}
float __device__ ref_pdf(const Mat& m, V3 n, V3 wo, V3 wi) {
    const float ci = dot(n, wi);
    if (ci <= 0.0f) return 0.0f;
    const float ps = spec_prob(m);
    float pdf = (1.0f - ps) * ci * (1.0f / kPi);
    if (ps > 0.0f) {
        const V3 h = ref_normalize(wo + wi);
        const float a = m.roughness * m.roughness, a2 = a * a;
        const float nh = fmaxf(dot(n, h), 0.0f), d = nh * nh * (a2 - 1.0f) + 1.0f;
        const float D = a2 / (kPi * d * d), wh = fabsf(dot(wo, h));
        if (wh > 0.0f) pdf += ps * D * nh / (4.0f * wh);
    }
    return pdf;
}
bool __device__ ref_sample(const Mat& m, V3 n, V3 wo, float ul, float u1, float u2, V3& wi) {
    const float s = copysignf(1.0f, n.z), q = -1.0f / (s + n.z), bb = n.x * n.y * q;
    const V3 t{1.0f + s * n.x * n.x * q, s * bb, -s * n.x}, b{bb, s + n.y * n.y * q, -n.y};
    const float ph = 2.0f * kPi * u2;
    if (ul < spec_prob(m)) {
        const float a = m.roughness * m.roughness, a2 = a * a;
        const float c2 = (1.0f - u1) / (1.0f + (a2 - 1.0f) * u1);
        const float ct = sqrtf(fmaxf(c2, 0.0f)), st = sqrtf(fmaxf(1.0f - c2, 0.0f));
        const V3 h = t * (st * cosf(ph)) + b * (st * sinf(ph)) + n * ct;
        wi = h * (2.0f * dot(wo, h)) - wo;
    } else {
        const float r = sqrtf(u1), z = sqrtf(fmaxf(1.0f - u1, 0.0f));
        wi = t * (r * cosf(ph)) + b * (r * sinf(ph)) + n * z;
    }
    return dot(n, wi) > 0.0f;
}
float __device__ ref_heuristic(float a, float b) {
    const float a2 = a * a, b2 = b * b;
    return a2 + b2 > 0.0f ? a2 / (a2 + b2) : 0.0f;
}

// in: 20 floats a case (normal, wo, wi, albedo, roughness, metallic, three uniforms,
// two pdfs, Lambert flag); out, ref: 15 floats a case.
__global__ void k_shading(const float* in, float* out, float* ref, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float* p = in + 20 * (size_t)i;
    const V3 nn{p[0], p[1], p[2]}, wo{p[3], p[4], p[5]}, wi{p[6], p[7], p[8]};
    Mat m{};
    m.albedo = V3{p[9], p[10], p[11]};
    m.roughness = p[12];
    m.metallic = p[13];
    m.flags = p[19] != 0.0f ? 2u : 0u;
    for (int k = 0; k < 2; ++k) {
        float* o = (k ? ref : out) + 15 * (size_t)i;
        const V3 u = k ? ref_normalize(nn) : normalize(nn);
        V3 f, fs, w{0.0f, 0.0f, 0.0f};
        float pdf, ph;
        bool ok;
        if (k) {
            f = fs = ref_eval(m, nn, wo, wi);
            pdf = ref_pdf(m, nn, wo, wi);
            ok = ref_sample(m, nn, wo, p[14], p[15], p[16], w);
            ph = ref_heuristic(p[17], p[18]);
        } else {
            const V3 h = brdf_half(m, wo, wi);
            f = brdf_eval(m, brdf_view(m, nn, wo), nn, wo, wi, h);
            fs = brdf_eval<true>(m, brdf_view(m, nn, wo), nn, wo, wi, h);
            pdf = brdf_pdf(m, nn, wo, wi, h);
            ok = brdf_sample(m, nn, wo, p[14], p[15], p[16], w);
            ph = power_heuristic(p[17], p[18]);
        }
        o[0] = u.x, o[1] = u.y, o[2] = u.z;
        o[3] = f.x, o[4] = f.y, o[5] = f.z;
        o[6] = pdf, o[7] = ph;
        o[8] = w.x, o[9] = w.y, o[10] = w.z;
        o[11] = ok ? 1.0f : 0.0f;
        o[12] = fs.x, o[13] = fs.y, o[14] = fs.z;
    }
}

int finish() {
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? (int)e : (int)hipDeviceSynchronize();
}
constexpr uint32_t kBlock = 256;
uint32_t grid(uint32_t n) { return (n + kBlock - 1) / kBlock; }

}  // namespace

extern "C" {
int check_unary(int op, const float* a, float* out, uint32_t n) {
    if (!n || !a || !out) return -1;
    k_unary<<<grid(n), kBlock>>>(op, a, out, n);
    return finish();
}
int check_quotient(const float* x, const float* d, float* out, float* out_signed, uint32_t n) {
    if (!n || !x || !d || !out || !out_signed) return -1;
    k_quotient<<<grid(n), kBlock>>>(x, d, out, out_signed, n);
    return finish();
}
int check_shading(const float* in, float* out, float* ref, uint32_t n) {
    if (!n || !in || !out || !ref) return -1;
    k_shading<<<grid(n), kBlock>>>(in, out, ref, n);
    return finish();
}
}
