/*
 * Host staging object of the sensor-feature boundary, in C11 over the HIP
 * runtime C API.  Behaviour follows the reference host object
 * src/cuda/features.cu:9-88: a handle owns one non-blocking stream and
 * staging buffers for up to max_batch (<= 1024) environments; extraction
 * copies the caller's host arrays in, runs the device entry, copies the 142
 * features out and waits.  Failures record "<stage>: <runtime message>" in
 * the handle; argument errors return 0 and leave the text untouched.
 *
 * Batches of up to FB_STAGE_MAX environments go through pinned memory of the
 * handle instead: the call copies FB_STAGE_ROWS environments at a time into
 * it and launches the extraction on them, which reads the rows over PCIe and
 * writes its features there, while the next rows, if any, are copied.  That
 * leaves out four copy-engine transfers and the runtime's own staging of
 * pageable memory.  Handles of up to FB_STAGE_MAX environments hold no device
 * buffers.
 */
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "turbinator/training/cuda_features.h"

enum {
    FB_OBS = 4148,
    FB_MISSION = 10,
    FB_CAMERA = 16384,
    FB_FEATURES = 142,
    FB_MAX_BATCH = 1024,
    /* Pageable copies -> pinned rows, 32 at a time, us on one box with the
     * arrays in the host's caches: 1 environment 38.9 -> 19.1, 16 65.7 ->
     * 33.8, 32 80.0 -> 51.9, 64 119.6 -> 76.7, 128 180.8 -> 124.9, 256 295.6
     * -> 237.2 (8 rows at a time 327.8, 64 240.8, all at once 331.4).  Larger
     * batches gain a tenth (1,024: 1,177 -> 1,038), which 26 MB more of
     * pinned memory per handle are not spent on. */
    FB_STAGE_MAX = 256,
    FB_STAGE_ROWS = 32
};

struct tb_cuda_feature_batch {
    int device_id;
    size_t max_batch;
    hipStream_t stream;
    float *obs;
    float *mission;
    unsigned char *cameras;
    float *features;
    /* Pinned rows of up to stage_max environments (staged_rows) and their
     * device address; stage_max 0 when there are none.  The device buffers
     * above are NULL when stage_max is max_batch. */
    size_t stage_max;
    unsigned char *staged, *staged_device;
    char error[192];
};

/* Byte offsets of the pinned rows' sections for n environments: obs at 0, and
 * each section on 16 bytes. */
typedef struct {
    size_t cameras, features, mission, end;
} fb_sections;

static fb_sections staged_rows(size_t n) {
    fb_sections s;
    s.cameras = n * FB_OBS * sizeof(float);
    s.features = s.cameras + n * FB_CAMERA;
    s.mission = (s.features + n * FB_FEATURES * sizeof(float) + 15) & ~(size_t)15;
    s.end = s.mission + n * FB_MISSION * sizeof(float);
    return s;
}

/* The device entry reads (and so clears) the launch error itself; a refused
 * launch whose error is already cleared is reported as a launch failure
 * rather than as "no error". */
static hipError_t launch_status(void) {
    const hipError_t status = hipGetLastError();
    return status == hipSuccess ? hipErrorLaunchFailure : status;
}

static int fb_fail(tb_cuda_feature_batch *batch, const char *stage, hipError_t status) {
    snprintf(batch->error, sizeof(batch->error), "%s: %s", stage, hipGetErrorString(status));
    return 0;
}

tb_cuda_feature_batch *tb_cuda_feature_batch_create(int device_id, size_t max_batch) {
    if (max_batch == 0 || max_batch > FB_MAX_BATCH) return NULL;
    if (hipSetDevice(device_id) != hipSuccess) return NULL;
    tb_cuda_feature_batch *batch = (tb_cuda_feature_batch *)calloc(1, sizeof(*batch));
    if (!batch) return NULL;
    batch->device_id = device_id;
    batch->max_batch = max_batch;
    if (hipStreamCreateWithFlags(&batch->stream, hipStreamNonBlocking) != hipSuccess) {
        batch->stream = NULL;
        tb_cuda_feature_batch_destroy(batch);
        return NULL;
    }
    batch->stage_max = max_batch < FB_STAGE_MAX ? max_batch : FB_STAGE_MAX;
    if (hipHostMalloc((void **)&batch->staged, staged_rows(batch->stage_max).end,
                      hipHostMallocDefault) != hipSuccess) {
        batch->staged = NULL;
        batch->stage_max = 0;
        (void)hipGetLastError();
    } else if (hipHostGetDevicePointer((void **)&batch->staged_device, batch->staged, 0) !=
               hipSuccess) {
        (void)hipHostFree(batch->staged);
        batch->staged = NULL;
        batch->stage_max = 0;
        (void)hipGetLastError();
    }
    /* Only batches above the pinned rows take the copies; without pinned
     * memory every batch does. */
    if (max_batch > batch->stage_max &&
        (hipMalloc((void **)&batch->obs, max_batch * FB_OBS * sizeof(float)) != hipSuccess ||
         hipMalloc((void **)&batch->mission, max_batch * FB_MISSION * sizeof(float)) != hipSuccess ||
         hipMalloc((void **)&batch->cameras, max_batch * FB_CAMERA) != hipSuccess ||
         hipMalloc((void **)&batch->features, max_batch * FB_FEATURES * sizeof(float)) !=
             hipSuccess)) {
        tb_cuda_feature_batch_destroy(batch);
        return NULL;
    }
    return batch;
}

void tb_cuda_feature_batch_destroy(tb_cuda_feature_batch *batch) {
    if (!batch) return;
    (void)hipSetDevice(batch->device_id);
    if (batch->stream) (void)hipStreamSynchronize(batch->stream);
    if (batch->obs) (void)hipFree(batch->obs);
    if (batch->mission) (void)hipFree(batch->mission);
    if (batch->cameras) (void)hipFree(batch->cameras);
    if (batch->features) (void)hipFree(batch->features);
    if (batch->staged) (void)hipHostFree(batch->staged);
    if (batch->stream) (void)hipStreamDestroy(batch->stream);
    free(batch);
}

const char *tb_cuda_feature_batch_error(const tb_cuda_feature_batch *batch) {
    return batch ? batch->error : "CUDA feature batch unavailable";
}

static int extract_staged(tb_cuda_feature_batch *batch, const float *obs, const float *mission,
                          const unsigned char *cameras, size_t count, float *out_features) {
    const fb_sections at = staged_rows(batch->stage_max);
    unsigned char *const host = batch->staged, *const device = batch->staged_device;
    hipError_t launch = hipSuccess;
    for (size_t first = 0; first < count && launch == hipSuccess; first += FB_STAGE_ROWS) {
        const size_t rows = count - first < FB_STAGE_ROWS ? count - first : FB_STAGE_ROWS;
        const size_t o = first * FB_OBS, m = first * FB_MISSION, c = first * FB_CAMERA;
        memcpy(host + o * sizeof(float), obs + o, rows * FB_OBS * sizeof(float));
        memcpy(host + at.mission + m * sizeof(float), mission + m,
               rows * FB_MISSION * sizeof(float));
        memcpy(host + at.cameras + c, cameras + c, rows * FB_CAMERA);
        if (!tb_cuda_extract_features_device(
                (const float *)device + o, (const float *)(device + at.mission) + m,
                device + at.cameras + c,
                (float *)(device + at.features) + first * FB_FEATURES, rows, batch->stream))
            launch = launch_status();
    }
    /* Also after a refused launch: the rows launched before it are read from
     * memory that the next call writes. */
    const hipError_t status = hipStreamSynchronize(batch->stream);
    if (launch != hipSuccess) return fb_fail(batch, "extract features", launch);
    if (status != hipSuccess) return fb_fail(batch, "synchronize features", status);
    memcpy(out_features, host + at.features, count * FB_FEATURES * sizeof(float));
    return 1;
}

int tb_cuda_extract_features_host(tb_cuda_feature_batch *batch, const float *obs,
                                  const float *mission, const unsigned char *cameras,
                                  size_t count, float *out_features) {
    if (!batch || !obs || !mission || !cameras || !out_features || count == 0 ||
        count > batch->max_batch)
        return 0;
    batch->error[0] = 0;
    hipError_t status = hipSetDevice(batch->device_id);
    if (status != hipSuccess) return fb_fail(batch, "select device", status);
    if (count <= batch->stage_max)
        return extract_staged(batch, obs, mission, cameras, count, out_features);
    status = hipMemcpyAsync(batch->obs, obs, count * FB_OBS * sizeof(float),
                            hipMemcpyHostToDevice, batch->stream);
    if (status != hipSuccess) return fb_fail(batch, "copy observations", status);
    status = hipMemcpyAsync(batch->mission, mission, count * FB_MISSION * sizeof(float),
                            hipMemcpyHostToDevice, batch->stream);
    if (status != hipSuccess) return fb_fail(batch, "copy mission", status);
    status = hipMemcpyAsync(batch->cameras, cameras, count * FB_CAMERA, hipMemcpyHostToDevice,
                            batch->stream);
    if (status != hipSuccess) return fb_fail(batch, "copy cameras", status);
    if (!tb_cuda_extract_features_device(batch->obs, batch->mission, batch->cameras,
                                         batch->features, count, batch->stream))
        return fb_fail(batch, "extract features", launch_status());
    status = hipMemcpyAsync(out_features, batch->features, count * FB_FEATURES * sizeof(float),
                            hipMemcpyDeviceToHost, batch->stream);
    if (status != hipSuccess) return fb_fail(batch, "copy features", status);
    status = hipStreamSynchronize(batch->stream);
    return status == hipSuccess ? 1 : fb_fail(batch, "synchronize features", status);
}
