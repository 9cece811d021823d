// Generated by gen_bindings.py from ramvamp_amd/build.py; do not edit by hand.
// Compiles the HIP sources for gfx950 with hipcc (no cmake, no CUDA, no other
// backend) into OUT_DIR/libramvamp_attn.so and links it. RAMVAMP_AMD_DIR
// points at the repository that holds ramvamp_amd/csrc and include/.
use std::{env, path::PathBuf, process::Command};

const SOURCES: &[&str] = &[
        "rv_abi.cpp",
        "rv_prologue.hip",
        "rv_decode.hip",
        "rv_prefill.hip",
        "rv_quant.hip",
        "rv_batched.hip",
        "rv_gemv_abi.cpp",
        "rv_block_abi.cpp",
        "rv_router.hip",
        "rv_floors.hip",
];
const FLAGS: &[&str] = &["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"];
const EXTRA: &[(&str, &[&str])] = &[
        ("rv_prefill.hip", &["-mllvm", "-amdgpu-mfma-vgpr-form"]),
];

fn main() {
    let root = PathBuf::from(env::var("RAMVAMP_AMD_DIR").unwrap_or_else(|_| "../..".into()));
    let csrc = root.join("ramvamp_amd/csrc");
    let out = PathBuf::from(env::var("OUT_DIR").unwrap());
    let hipcc = env::var("HIPCC").unwrap_or_else(|_| "/opt/rocm/bin/hipcc".into());
    let mut objs = Vec::new();
    for src in SOURCES {
        let obj = out.join(format!("{src}.o"));
        let mut cmd = Command::new(&hipcc);
        cmd.args(FLAGS);
        if let Some((_, more)) = EXTRA.iter().find(|(s, _)| s == src) {
            cmd.args(*more);
        }
        let status = cmd.arg("-c").arg("-o").arg(&obj).arg(csrc.join(src)).status().expect("hipcc");
        assert!(status.success(), "hipcc failed on {src}");
        objs.push(obj);
    }
    let status = Command::new(&hipcc)
        .args(["--offload-arch=gfx950", "-shared", "-fPIC", "-o"])
        .arg(out.join("libramvamp_attn.so"))
        .args(&objs)
        .status()
        .expect("hipcc link");
    assert!(status.success(), "hipcc link failed");
    println!("cargo:rustc-link-search=native={}", out.display());
    println!("cargo:rustc-link-lib=dylib=ramvamp_attn");
    println!("cargo:rerun-if-changed={}", csrc.display());
    println!("cargo:rerun-if-changed={}", root.join("include").display());
}
