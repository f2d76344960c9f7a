/* The few HIP calls of side.hip as host stubs that record what was asked for (tests only). */
#pragma once
#include <stddef.h>
typedef struct stub_stream* hipStream_t;
typedef struct stub_event* hipEvent_t;
typedef int hipError_t;
enum { hipSuccess = 0, hipStreamNonBlocking = 1, hipEventDisableTiming = 2, hipDeviceAttributeMultiprocessorCount = 0 };
typedef int hipStreamCaptureStatus;
enum { hipStreamCaptureStatusNone = 0 };
hipError_t hipGetDevice(int*);
hipError_t hipDeviceGetAttribute(int*, int, int);
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus*);
hipError_t hipStreamCreateWithFlags(hipStream_t*, unsigned);
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned);
hipError_t hipEventRecord(hipEvent_t, hipStream_t);
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned);
