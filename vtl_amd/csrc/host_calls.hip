// Whole calls on host tensors: upload, kernels and download behind one entry point.
//
// A program that keeps its tensors on the host pays, per call, for every step between the
// kernels: 64 x 784 -> 256 is 10 us of kernels.  Made from the host language step by step,
// the same call took 41 us, 18 of them outside the library.
#include "common.hpp"

namespace vtlhip {
namespace {

// Device memory for the length of a call.  Released while its kernels may still run: the pool hands
// it out again behind them.
struct Scratch {
    void *ptr = nullptr;
    ~Scratch() { release(); }
    Scratch() = default;
    Scratch(const Scratch &) = delete;
    Scratch &operator=(const Scratch &) = delete;
    int take(size_t bytes)
    {
        release();
        return bytes ? vtl_hip_malloc(&ptr, bytes) : VTL_HIP_OK;
    }
    void release()
    {
        if (ptr)
            (void)vtl_hip_free(ptr);
        ptr = nullptr;
    }
    void swap(Scratch &o)
    {
        void *p = ptr;
        ptr = o.ptr;
        o.ptr = p;
    }
    template <typename T>
    T *as() { return static_cast<T *>(ptr); }
};

#define VTL_STEP(expr)            \
    do {                          \
        const int rc_ = (expr);   \
        if (rc_ != VTL_HIP_OK)    \
            return rc_;           \
    } while (0)

// Up to this many rows the linear on f32 rows quantizes them inside its own launch, so the
// activations stay f32 between layers (1 row through 4096 -> 11008 -> 4096 -> 1024: 23.4 against
// 28.0 us); with more rows per-row codes go from layer to layer.  The bits are the same.
constexpr int kFewRows = 32;

// Up to how many bytes of codes the first product reads over the link: each XCD fetches them, which from here on takes what a launch that carries
// them up does (us, carried and read: 7 x 128 x 128 17.3 and 14.1, 64 x 256 x 128 20.8 and 18.1, 200 x 300 x 64 23.3 and 20.0, 32 x 512 x 512 22.2 and 20.7, 20 x 500 x
// 1100 21.9 and 22.4, 64 x 256 x 784 24.2 and 29.3).
constexpr size_t kCodesOverLink = (size_t)16 << 10;

// Not two to eight dense rows with one scale that are no whole vectors: the product's matrix-vector kernel reads those in every workgroup, in parts, and from so many codes
// on that is slower over the link than a quantizer's launch that reads f32 there once (us, quantized by a launch and read as codes: 3 x 80 x 251 17.2 and 15.7, but 7 x 48 x
// 309 19.3 and 24.2, 5 x 126 x 422 18.6 and 21.0, 8 x 61 x 1372 23.7 and 36.3; 2 x 48 x 907 18.4 and 17.4, 2 x 48 x 1187 17.8 and 18.9).  Carried up they are 1 to 8 % behind
// that launch as well, up to kCodesOverLink; once a stream has been named that launch has an upload in front, and codes are 1 to 10 % ahead (5 x 48 x 1162 39.1 and 35.0).
bool few_ragged_rows(int rows, int cols, int row)
{
    return vtlhip::single_stream() && rows <= 8 && row % 16 != 0 && cols >= (rows == 2 ? 1024 : 256) && (size_t)rows * (size_t)row <= kCodesOverLink;
}

// Whether activations beyond that are made codes of by the host, where rows_long_enough says so too.  On the null stream alone the launch that quantizes them
// reads up to 1 MiB of them over the link itself, where weights are uploaded first, so the host is behind it for longer (us, by the device and by the host, rows x
// values: scales per row 130 x 256 25.2 and 26.3, 98 x 200 21.6 and 23.1, but 106 x 363 24.0 and 23.1, 766 x 240 49.5 and 43.2; one scale 763 x 36 25.7 and 27.3, 1437 x
// 35 39.2 and 40.8, but 400 x 67 25.6 and 24.9).
bool activations_long_enough(const vtl_hip_layer &l, int rows, int cols)
{
    const size_t codes = (size_t)rows * (size_t)cols;
    if (!vtlhip::rows_long_enough(rows, cols, l.per_channel))
        return false;
    if (!vtlhip::single_stream() || codes * sizeof(float) > (size_t)1 << 20 || vtlhip::tuning().host_quantize == 1)
        return true;
    return l.per_channel ? cols > 256 || codes >= (size_t)64 << 10 : cols >= 64;
}

int check_layers(const vtl_hip_layer *layers, int count, int cols, int &out_cols)
{
    for (int i = 0; i < count; i++) {
        const vtl_hip_layer &l = layers[i];
        if (l.kind == VTL_HIP_LAYER_RELU)
            continue;
        if (l.kind != VTL_HIP_LAYER_LINEAR || l.in_features != cols || l.out_features < 0 || !l.wq || !l.sw)
            return VTL_HIP_ERR_INVALID_ARG;
        cols = l.out_features;
    }
    out_cols = cols;
    return VTL_HIP_OK;
}

// Whether one row of the caller's, against weights with one scale, is quantized in the launch of the product.  That every workgroup
// reads a long row over the link, or that it is uploaded first (20 to 32 KiB), is more than a second launch behind one that reads it once; rows
// that start anywhere are read twice there and hold out longer (us, in two launches and in one: 64 x 4096 15.9 and 15.8, 48 x 5120 15.9
// and 16.4, 16 x 5120 15.6 and 14.3, 64 x 6000 16.3 and 17.2, 600 x 8192 18.4 and 18.0, 64 x 10000 18.0 and 20.4, 2500 x 10000 22.8 and 24.9, 16 x 10000 17.8
// and 16.1, 64 x 14336 19.6 and 24.1, 16 x 14336 19.1 and 18.7; 64 x 6001 19.5 and 17.2, 64 x 11001 21.1 and 21.1, 5500 x 11001 29.6 and 28.6, 64 x 14001 21.6
// and 23.8, 32 x 14001 21.2 and 20.1).  Beyond 14336 both take two.
bool row_in_one(int n, int k)
{
    if (k % 16 != 0)
        return k <= 11008 || n <= 32 || k > 14336;
    return k <= 4096 || ((k <= 5120 || k > 8192) && n <= 16) || k > 14336;
}

int forward_layers(const float *x_host, int rows, int cols, const vtl_hip_layer *layers, int count, float *y_host)
{
    int out_cols = 0;
    VTL_STEP(check_layers(layers, count, cols, out_cols));
    if (rows == 0 || cols == 0 || out_cols == 0)
        return count == 0 ? VTL_HIP_OK : VTL_HIP_ERR_INVALID_ARG;
    const size_t in_bytes = (size_t)rows * (size_t)cols * sizeof(float);
    Scratch cur, next;                     // f32 rows
    Scratch work;                          // of layers on f32 rows, to the call's last launch: once a stream has been named a release waits
    size_t work_bytes = 0;
    Scratch codes, scales, next_codes, next_scales;
    const float *x = nullptr;              // the f32 rows, or null while the activations are codes
    int i = 0;
    // the last layer writes y itself, unless a ReLU of its own comes behind it
    HostResult result;
    const size_t out_bytes = (size_t)rows * (size_t)out_cols * sizeof(float);
    const bool ends_linear = count > 0 && (layers[count - 1].kind == VTL_HIP_LAYER_LINEAR ||
                                           (count > 1 && layers[count - 2].kind == VTL_HIP_LAYER_LINEAR));
    // Written over the link as it is computed, with rows that end where lines do, 4 MiB is no slower than a copy behind the
    // launch (256 x 4096 126 -> 121 us; 256 x 5000 145 and 158, 256 x 8000 205 and 222).  Other rows leave lines to two
    // workgroups: 100 x 6001 76 -> 74, but 96 x 8191 90 and 92, 200 x 4999 117 and 126, 200 x 6001 133 and 151, 192 x 10000 186 and 236.
    const size_t most = out_cols % 32 == 0 ? (size_t)4 << 20 : (size_t)5 << 19;
    float *const y = ends_linear ? static_cast<float *>(result.begin(y_host, out_bytes, most)) : nullptr;
    HostInput input;
    vtlhip::CallScratch own;
    // (32 KiB is what the kernels that quantize in every workgroup take at most; near it the eight XCDs' transfers
    // cost what an upload does)
    // One row has one scale either way: a layer with one for all of its weights takes it as one with a scale per row does, in one
    // launch instead of two (us, per tensor: 1 x 832 x 448 17.4 -> 15.9, 1 x 3000 x 513 20.9 -> 17.3, 1 x 576 x 238 18.4 -> 16.9; a second layer of
    // 64 x 256 20.9 -> 17.0, of 2500 x 11008 29.3 -> 24.6).
    const auto by_row = [&](const vtl_hip_layer &l) { return l.per_channel || rows == 1; };
    const bool first_by_row = count > 0 && by_row(layers[0]) && (layers[0].per_channel || row_in_one(layers[0].out_features, cols));
    // Rows that a launch would only make codes of are made codes of by the host: few bytes of them are read over the link by the product's launch,
    // more go up.
    const int8_t *in = nullptr;            // the activations where they are codes, and their scales
    const float *in_scales = nullptr;
    bool padded = false;                   // whether the codes lie in rows of l.row_bytes
    if (count > 0 && layers[0].kind == VTL_HIP_LAYER_LINEAR &&
        (rows > kFewRows || (rows > 1 && !layers[0].per_channel) || (rows > 8 && !layer_takes_input(layers[0], rows)))) {
        const vtl_hip_layer &l = layers[0];
        const int row = l.row_bytes > cols ? l.row_bytes : cols;
        if (few_ragged_rows(rows, cols, row) && vtlhip::tuning().host_quantize != 1) {
            // (by the device, below)
        } else if ((size_t)rows * (size_t)row <= kCodesOverLink && input.stage_codes(x_host, rows, cols, l.per_channel, row)) {
            in = static_cast<const int8_t *>(input.data);
            in_scales = input.scales;
        } else if (activations_long_enough(l, rows, cols) && host_makes_codes(rows, cols, row)) {
            VTL_STEP(codes.take((size_t)rows * (size_t)row));
            VTL_STEP(scales.take((l.per_channel ? (size_t)rows : 1) * sizeof(float)));
            int status = VTL_HIP_OK;
            if (upload_codes(x_host, rows, cols, l.per_channel, codes.as<int8_t>(), row, scales.as<float>(), nullptr, nullptr, 0, status)) {
                VTL_STEP(status);
                in = codes.as<int8_t>();
                in_scales = scales.as<float>();
            } else {
                codes.release();
                scales.release();
            }
        }
        padded = in && l.row_bytes != 0;
    }
    const bool upload_first = rows <= 8 && in_bytes > ((size_t)20 << 10) && in_bytes <= ((size_t)32 << 10);
    if (!in && count > 0 && layers[0].kind == VTL_HIP_LAYER_LINEAR && !(upload_first && first_by_row) &&
        input.stage(x_host, in_bytes)) {
        // The first launch takes the input over the link itself: 64 x 784, per tensor, 4 us less than behind an
        // upload.  Rows that are no whole vectors are read twice, which still is no slower (forward of 200 x 1001
        // 56.9 against 61.4 us, 64 x 1023 37.9 and 39.3, 64 x 2047 and 64 x 4095 level).  The launches for
        // a few rows read them in every workgroup, out of the L2 but for the first of each XCD: 0 to 2.6 us more than from
        // device memory for a row of up to 4096, 10 for 32 such rows (read once), where the upload takes 3 and 13 and a
        // launch of its own.
        x = static_cast<const float *>(input.data);
        if (!first_by_row || rows > kFewRows) {
            VTL_STEP(codes.take((size_t)rows * (size_t)cols));
            VTL_STEP(scales.take((layers[0].per_channel ? (size_t)rows : 1) * sizeof(float)));
            VTL_STEP(vtl_hip_quantize_f32_i8(x, rows, cols, layers[0].per_channel, codes.as<int8_t>(), scales.as<float>()));
            x = nullptr;
            in = codes.as<int8_t>();
            in_scales = scales.as<float>();
            input.release();
        }
    }
    if (!in && !x) {
        VTL_STEP(cur.take(in_bytes));
        VTL_STEP(vtl_hip_upload(cur.ptr, x_host, in_bytes));
        x = cur.as<float>();
    }
    while (i < count) {
        const vtl_hip_layer &l = layers[i];
        if (l.kind == VTL_HIP_LAYER_RELU) {
            VTL_STEP(vtl_hip_relu_f32(cur.as<float>(), (int64_t)rows * cols));
            i++;
            continue;
        }
        const int n = l.out_features;
        const bool relu = i + 1 < count && layers[i + 1].kind == VTL_HIP_LAYER_RELU;
        i += relu ? 2 : 1;
        const bool last = y && i == count;
        // the next layer takes codes as well, and does not make them in its own launch
        const bool feeds = l.per_channel && rows > kFewRows && i < count && layers[i].kind == VTL_HIP_LAYER_LINEAR &&
                           layers[i].per_channel && !layer_takes_rows(layers[i], rows);
        if (x && by_row(l) && !feeds) {
            if (!last)
                VTL_STEP(next.take((size_t)rows * (size_t)n * sizeof(float)));
            const size_t need = vtl_hip_linear_f32_dynquant_workspace(rows, cols);
            if (need > work_bytes) {
                VTL_STEP(work.take(need));
                work_bytes = need;
            }
            VTL_STEP(layer_f32(l, x, last ? y : next.as<float>(), rows, relu, work.ptr, need, last ? &result : nullptr,
                               input.data != nullptr));
            if (input.data) {
                input.release();
                if (result.attached())
                    result.input_released();
            }
            cur.swap(next);
            x = cur.as<float>();
            cols = n;
            continue;
        }
        if (x) {
            VTL_STEP(codes.take((size_t)rows * (size_t)cols));
            VTL_STEP(scales.take((l.per_channel ? (size_t)rows : 1) * sizeof(float)));
            VTL_STEP(vtl_hip_quantize_f32_i8(x, rows, cols, l.per_channel, codes.as<int8_t>(), scales.as<float>()));
            x = nullptr;
            in = codes.as<int8_t>();
            in_scales = scales.as<float>();
        }
        if (feeds) {
            VTL_STEP(next_codes.take((size_t)rows * (size_t)n));
            VTL_STEP(next_scales.take((size_t)rows * sizeof(float)));
            VTL_STEP(layer_linear_i8_requant(l, in, in_scales, next_codes.as<int8_t>(),
                                             next_scales.as<float>(), rows, relu, padded));
            codes.swap(next_codes);
            scales.swap(next_scales);
            in = codes.as<int8_t>();
            in_scales = scales.as<float>();
        } else {
            if (!last)
                VTL_STEP(cur.take((size_t)rows * (size_t)n * sizeof(float)));
            VTL_STEP(layer_linear_i8_f32(l, in, in_scales, last ? y : cur.as<float>(), rows, relu,
                                         last ? &result : nullptr, padded));
            x = cur.as<float>();
        }
        if (input.data) {
            input.release();
            if (result.attached())
                result.input_released();
        }
        padded = false;
        cols = n;
    }
    if (!y)
        return vtl_hip_memcpy_d2h(y_host, cur.ptr, out_bytes);
    if (result.attached() || !single_stream()) {   // nothing more to launch: what a release waits for is what the results are waited for
        for (Scratch *s : {&work, &cur, &next, &codes, &scales, &next_codes, &next_scales})
            s->release();
    }
    return result.finish();
}

int colsum(const float *x, int64_t rows, int64_t cols, float *out) { return vtl_hip_colsum_f32(x, rows, cols, out); }
int colsum(const double *x, int64_t rows, int64_t cols, double *out) { return vtl_hip_colsum_f64(x, rows, cols, out); }

template <typename T>
int upload(Scratch &to, const T *host, size_t count)
{
    VTL_STEP(to.take(count * sizeof(T)));
    return vtl_hip_upload(to.ptr, host, count * sizeof(T));
}

template <typename T>
int upload_both(Scratch &to0, const T *host0, size_t count0, Scratch &to1, const T *host1, size_t count1)
{
    VTL_STEP(to0.take(count0 * sizeof(T)));
    VTL_STEP(to1.take(count1 * sizeof(T)));
    int status = VTL_HIP_OK;
    if (upload_two(to0.ptr, host0, count0 * sizeof(T), to1.ptr, host1, count1 * sizeof(T), status))
        return status;
    VTL_STEP(vtl_hip_upload(to0.ptr, host0, count0 * sizeof(T)));
    return vtl_hip_upload(to1.ptr, host1, count1 * sizeof(T));
}

constexpr size_t kResultMost = (size_t)8 << 20;

// How many bytes a product writes over the link as it is computed.  Rows that do not end where lines do leave lines to two
// workgroups, which the link takes apart: a copy behind the launch is faster unless there is little to write (us,
// copied and written over the link: f32 700 x 1001 x 200 122 and 136, 1024 x 1001 x 64 117 and 128, x 320 184 and
// 195, 256 x 1000 x 800 level, 256 x 700 x 16 38 and 36; whole lines 1024 x 1024 x 16 107 and 102, x 400 200 and 198).
template <typename T>
size_t direct_most(int m, int n)
{
    const bool whole_lines = (size_t)n * sizeof(T) % 128 == 0;
    return whole_lines || (int64_t)m * n <= 196608 ? kResultMost : 0;
}

template <typename T>
int matmul_host(const T *a, const T *b, T *c, int m, int n, int k)
{
    if (m < 0 || n < 0 || k < 0)
        return VTL_HIP_ERR_INVALID_ARG;
    if (m == 0 || n == 0)
        return VTL_HIP_OK;
    if (!c || (k > 0 && (!a || !b)))
        return VTL_HIP_ERR_INVALID_ARG;
    Scratch da, db, dc;
    VTL_STEP(upload_both(da, a, (size_t)m * (size_t)k, db, b, (size_t)k * (size_t)n));
    const size_t bytes = (size_t)m * (size_t)n * sizeof(T);
    HostResult result;
    vtlhip::CallScratch own;
    if (T *out = static_cast<T *>(result.begin(c, bytes, direct_most<T>(m, n)))) {
        VTL_STEP(matmul_to(&result, da.as<T>(), db.as<T>(), out, m, n, k, 0));
        return result.finish();
    }
    VTL_STEP(dc.take(bytes));
    VTL_STEP(matmul_to(nullptr, da.as<T>(), db.as<T>(), dc.as<T>(), m, n, k, 0));
    return vtl_hip_memcpy_d2h(c, dc.ptr, bytes);
}

// Up to how many rows of dW one launch writes all gradients over the link.  What a launch writes there as it computes goes as it is
// stored, a row of a few bytes by itself; dW by a launch of its own is gathered to lines in the cache, and crosses while W comes up
// (us, launch by launch and in one: f32 10 x 778 x 2 30 and 73, 64 x 1500 x 3 40 and 171, 5 x 100 x 3 24 and 31, 5 x 40 x 3 24 and 22; 10 x 1000 x 9
// 30 and 42, 150 x 300 x 9 35 and 33; 10 x 1000 x 8 30 and 28, 3 x 2000 x 8 33 and 36, 3 x 5000 x 16 57 and 76; 3 x 2000 x 33 49 and 48, 3 x 4500 x 33 81
// and 89; f64 10 x 778 x 2 29 and 43, 10 x 1000 x 4 30 and 27, 3 x 2000 x 4 32 and 36).
int64_t rows_over_link(size_t row_bytes)
{
    if (row_bytes >= 128)
        return 2048;
    if (row_bytes >= 48 || row_bytes == 32)
        return 1024;
    if (row_bytes > 32)
        return 400;
    return row_bytes >= 16 && row_bytes % 8 == 0 ? 128 : 48;
}

template <typename T>
int linear_backward_host(const T *grad, const T *x, const T *w, T *dx, T *dw, T *db, int m, int n, int k)
{
    if (m < 0 || n < 0 || k < 0 || !grad || (dx && !w) || (dw && !x))
        return VTL_HIP_ERR_INVALID_ARG;
    const size_t mn = (size_t)m * (size_t)n, mk = (size_t)m * (size_t)k, nk = (size_t)n * (size_t)k;
    Scratch dev_grad, dev_x, dev_w, dev_dx, dev_dw, dev_db;
    if (mn == 0)
        return VTL_HIP_ERR_INVALID_ARG;
    // dW and db are computed, and on their way to the host, while the host copies W for the upload behind them.  What
    // shares memory with W waits in device memory until that is done (`late`).
    struct Gradient {
        T *host;
        size_t bytes;
        Scratch &dev;
        bool late;
        T *out = nullptr;
        bool direct = false;
        int take(HostResult &result)
        {
            if (!host || bytes == 0)
                return VTL_HIP_OK;
            out = static_cast<T *>(result.begin(host, bytes, late ? 0 : kResultMost));
            direct = out != nullptr;
            if (!direct) {
                VTL_STEP(dev.take(bytes));
                out = dev.as<T>();
            }
            return VTL_HIP_OK;
        }
    };
    HostResult result;
    vtlhip::CallScratch own;
    const size_t dw_bytes = nk * sizeof(T), db_bytes = (size_t)n * sizeof(T);
    Gradient gw = {dw, dw_bytes, dev_dw, dx && meet(dw, dw_bytes, w, dw_bytes)}, gx = {dx, mk * sizeof(T), dev_dx, false},
             gb = {db, db_bytes, dev_db, dx && meet(db, db_bytes, w, dw_bytes)};
    VTL_STEP(gw.take(result));
    VTL_STEP(gx.take(result));
    VTL_STEP(gb.take(result));
    // Every operand in one upload and all gradients in one launch, where there is less to copy than two more launches take (us, in two
    // and in one: 64 x 64 x 64 30.6 and 25.2, 256 x 64 x 64 36.0 and 28.6, 64 x 256 x 256 46.4 and 40.9, 64 x 256 x 400
    // 56.7 and 53.8; f64 64 x 128 x 128 42.7 and 36.1, 16 x 256 x 256 53.9 and 51.5).
    if (single_stream() && gw.direct && gx.direct && (!gb.out || gb.direct) && (mn + mk + nk) * sizeof(T) <= kUploadTogether &&
        n <= rows_over_link(k * sizeof(T))) {
        VTL_STEP(dev_grad.take(mn * sizeof(T)));
        VTL_STEP(dev_x.take(mk * sizeof(T)));
        VTL_STEP(dev_w.take(nk * sizeof(T)));
        const HostUpload operands[3] = {{dev_grad.ptr, grad, mn * sizeof(T)}, {dev_x.ptr, x, mk * sizeof(T)}, {dev_w.ptr, w, nk * sizeof(T)}};
        int status = VTL_HIP_OK;
        if (upload_together(operands, 3, status)) {
            VTL_STEP(status);
            if (!gradients_in_one(&result, dev_grad.as<T>(), dev_x.as<T>(), dev_w.as<T>(), gx.out, gw.out, gb.out, m, n, k, status)) {
                VTL_STEP(weight_gradients_to(nullptr, dev_grad.as<T>(), dev_x.as<T>(), gw.out, gb.out, m, n, k));
                status = matmul_to(&result, dev_grad.as<T>(), dev_w.as<T>(), gx.out, m, k, n, 0);
            }
            VTL_STEP(status);
            return result.finish();
        }
    }
    if (gw.out)
        VTL_STEP(upload_both(dev_grad, grad, mn, dev_x, x, mk));
    else
        VTL_STEP(upload(dev_grad, grad, mn));
    if (gw.out)     // [N,K] = grad^T[N,M] . x[M,K], and the column sums
        VTL_STEP(weight_gradients_to(gw.direct && !gx.out ? &result : nullptr, dev_grad.as<T>(), dev_x.as<T>(), gw.out, gb.out, m, n, k));
    else if (gb.out)
        VTL_STEP(colsum(dev_grad.as<T>(), m, n, gb.out));
    if (gx.out) {   // [M,K] = grad[M,N] . W[N,K]
        VTL_STEP(upload(dev_w, w, nk));
        VTL_STEP(matmul_to(gx.direct ? &result : nullptr, dev_grad.as<T>(), dev_w.as<T>(), gx.out, m, k, n, 0));
    }
    const Gradient *all[3] = {&gw, &gx, &gb};
    void *host[3];
    const void *dev[3];
    size_t bytes[3];
    int count = 0;
    bool direct = false;
    for (const Gradient *g : all) {
        direct = direct || g->direct;
        if (g->out && !g->direct) {
            host[count] = g->host;
            dev[count] = g->out;
            bytes[count++] = g->bytes;
        }
    }
    VTL_STEP(vtl_hip_download(count, host, dev, bytes));
    return direct ? result.finish() : VTL_HIP_OK;
}

}  // namespace
}  // namespace vtlhip

using namespace vtlhip;

extern "C" {

int vtl_hip_forward_i8_host(const float *x_host, int rows, int cols, const vtl_hip_layer *layers, int count,
                            float *y_host)
{
    if (rows < 0 || cols < 0 || count < 0 || (count > 0 && !layers) || !x_host || !y_host)
        return VTL_HIP_ERR_INVALID_ARG;
    return forward_layers(x_host, rows, cols, layers, count, y_host);
}

int vtl_hip_upload_two(void *dst0, const void *src0, size_t bytes0, void *dst1, const void *src1, size_t bytes1)
{
    if ((bytes0 && (!dst0 || !src0)) || (bytes1 && (!dst1 || !src1)))
        return VTL_HIP_ERR_INVALID_ARG;
    int status = VTL_HIP_OK;
    if (upload_two(dst0, src0, bytes0, dst1, src1, bytes1, status))
        return status;
    if (bytes0)
        VTL_STEP(vtl_hip_upload(dst0, src0, bytes0));
    return bytes1 ? vtl_hip_upload(dst1, src1, bytes1) : VTL_HIP_OK;
}

int vtl_hip_upload_quantized(const float *src_host, int64_t rows, int64_t cols, int per_row, int8_t *q, float *scale,
                             void *extra_device, const void *extra_host, size_t extra_bytes)
{
    if (rows < 0 || cols < 0 || (rows > 0 && cols > 0 && (!src_host || !q)) || (extra_bytes && (!extra_device || !extra_host)))
        return VTL_HIP_ERR_INVALID_ARG;
    int status = VTL_HIP_OK;
    // (once a stream has been named, a release of the f32 memory would wait for the device: 868 x 64 with a small forward 80 us, as codes 56)
    if (scale && rows > 0 && cols > 0 && (!single_stream() || rows_long_enough(rows, cols, per_row)) &&
        upload_codes(src_host, rows, cols, per_row, q, cols, scale, extra_device, extra_host, extra_bytes, status))
        return status;
    if (per_row && scale && rows > 0 && cols > 0 &&
        upload_rows(src_host, rows, cols, q, scale, extra_device, extra_host, extra_bytes, status))
        return status;
    const size_t bytes = (size_t)rows * (size_t)cols * sizeof(float);
    Scratch x;
    VTL_STEP(x.take(bytes));
    VTL_STEP(vtl_hip_upload_two(x.ptr, src_host, bytes, extra_device, extra_host, extra_bytes));
    return vtl_hip_quantize_f32_i8(x.as<float>(), rows, cols, per_row, q, scale);
}

int vtl_hip_matmul_host_f32(const float *a, const float *b, float *c, int m, int n, int k)
{
    return matmul_host<float>(a, b, c, m, n, k);
}

int vtl_hip_matmul_host_f64(const double *a, const double *b, double *c, int m, int n, int k)
{
    return matmul_host<double>(a, b, c, m, n, k);
}

int vtl_hip_linear_backward_host_f32(const float *grad, const float *x, const float *W, float *dx, float *dw,
                                     float *db, int m, int n, int k)
{
    return linear_backward_host<float>(grad, x, W, dx, dw, db, m, n, k);
}

int vtl_hip_linear_backward_host_f64(const double *grad, const double *x, const double *W, double *dx, double *dw,
                                     double *db, int m, int n, int k)
{
    return linear_backward_host<double>(grad, x, W, dx, dw, db, m, n, k);
}

}  // extern "C"
