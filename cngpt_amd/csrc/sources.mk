# The library's translation units (one list, for its Makefile and the sanitizer
# build of tests/asan).
HIP_SRC := rowops.hip gemm.hip split.hip split_train.hip attn_split.hip attention.hip decode.hip sample.hip persist.hip loss.hip train.hip attn_bwd.hip
CPP_SRC := cngpt_hip.cpp train_host.cpp
C_SRC   := fast.c model_host.c
